"""The F16 neck kernels (fp16-MFMA implicit GEMM in 64-deep stages of two
32-channel slices) at the edges of their tiles: odd slice counts (Cin % 64 ==
32, where a stage crosses taps or ends half empty), one-slice maps, ragged
pixel counts and output channels, K splits.

Bound against float64 over the fp16-rounded operands: exact products, one fp32
accumulation per 32 of K plus the K split's, each rounding by at most 2^-23 of
S = sum |w x|, and the bias add's rounding."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _close(got, ref, s, b, K):
    bound = (K // 32 + 20) * 2.0 ** -23 * s + 2.0 ** -23 * (np.abs(ref) + np.abs(b))
    err = np.abs(got.astype(np.float64) - (ref + b))
    assert (err <= bound).all(), float((err / bound).max())


@pytest.mark.parametrize("H,W,Cin,Cout", [(3, 5, 32, 4), (16, 8, 64, 128), (19, 13, 96, 132), (23, 17, 160, 68), (40, 37, 224, 260),
                                          (9, 9, 1024, 36)])
@pytest.mark.parametrize("k", [1, 3])
def test_conv_f16_tiles(mi, ctx, H, W, Cin, Cout, k):
    rng = np.random.default_rng(H * W + Cin + k)
    w = rng.standard_normal((Cout, Cin, k, k)).astype(np.float16)
    b = rng.standard_normal(Cout).astype(np.float32)
    x = rng.standard_normal((H, W, Cin)).astype(np.float32)
    wd, bd, xd = torch.from_numpy(w.view(np.int16)).cuda(), torch.from_numpy(b).cuda(), torch.from_numpy(x).cuda()
    y = torch.full((H * W, Cout), float("nan"), dtype=torch.float32, device="cuda")
    ctx.neck_conv(mi.from_torch(wd, mi.F16, [k, k, Cin, Cout]), bd.data_ptr(), xd.data_ptr(), H, W, y.data_ptr())
    ctx.synchronize()
    pad = np.zeros((H + k - 1, W + k - 1, Cin))
    pad[k // 2:k // 2 + H, k // 2:k // 2 + W] = x.astype(np.float16)
    ref, s = np.zeros((H * W, Cout)), np.zeros((H * W, Cout))
    for i in range(k):
        for j in range(k):
            a, t = pad[i:i + H, j:j + W].reshape(H * W, Cin), w[:, :, i, j].astype(np.float64)
            ref += a @ t.T
            s += np.abs(a) @ np.abs(t).T
    _close(y.cpu().numpy(), ref, s, b, Cin * k * k)


@pytest.mark.parametrize("H,W,Cin,Cout", [(3, 5, 32, 4), (16, 8, 64, 32), (13, 11, 96, 36), (21, 10, 160, 68)])
def test_deconv_f16_tiles(mi, ctx, H, W, Cin, Cout):
    rng = np.random.default_rng(H * W + Cin)
    w = rng.standard_normal((Cin, Cout, 2, 2)).astype(np.float32)
    b = rng.standard_normal(Cout).astype(np.float32)
    x = rng.standard_normal((H * W, Cin)).astype(np.float32)
    wd, bd, xd = torch.from_numpy(w).cuda(), torch.from_numpy(b).cuda(), torch.from_numpy(x).cuda()
    y = torch.full((4 * H * W, Cout), float("nan"), dtype=torch.float32, device="cuda")
    ctx.neck_deconv(mi.from_torch(wd, mi.F32, [2, 2, Cout, Cin]), bd.data_ptr(), xd.data_ptr(), H, W, False, y.data_ptr())
    ctx.synchronize()
    a, t = x.astype(np.float16).astype(np.float64), w.astype(np.float16).astype(np.float64).reshape(Cin, -1)
    place = lambda v: v.reshape(H, W, Cout, 2, 2).transpose(0, 3, 1, 4, 2).reshape(4 * H * W, Cout)
    _close(y.cpu().numpy(), place(a @ t), place(np.abs(a) @ np.abs(t)), b, Cin)


def test_conv_f16_ranges_of_odd_length(mi, ctx):
    """A K split keeps its ranges where they are odd: 36 x 36 of 256 channels sums 72 slices of 32 in
    ranges of seven, and longer ones would round more. 2^24 in slice 6, 1 in slice 7 and -2^24 in
    slice 8 come out as 1 exactly, since a new range begins with slice 7 (with it in the first
    range 2^24 + 1 rounds to 2^24)."""
    H, C, N = 36, 256, 256
    w = np.zeros((N, C, 3, 3), np.float16)
    w[:, 200, 0, 0], w[:, 230, 0, 0], w[:, 5, 0, 1] = 4096, 1, -4096
    x = np.zeros((H, H, C), np.float32)
    x[..., 200], x[..., 230], x[..., 5] = 4096, 1, 4096
    wd, bd, xd = torch.from_numpy(w.view(np.int16)).cuda(), torch.zeros(N, device="cuda"), torch.from_numpy(x).cuda()
    y = torch.full((H, H, N), float("nan"), dtype=torch.float32, device="cuda")
    ctx.neck_conv(mi.from_torch(wd, mi.F16, [3, 3, C, N]), bd.data_ptr(), xd.data_ptr(), H, H, y.data_ptr())
    ctx.synchronize()
    assert bool((y[1:, 1:] == 1).all()), y[1:, 1:].unique()


@pytest.mark.parametrize("Cin,Cout", [(672, 20), (704, 96)])
@pytest.mark.parametrize("gelu", [False, True])
def test_deconv_f16_large_map_few_columns(mi, ctx, Cin, Cout, gelu):
    """A conv-transpose of few output channels over a large F32 map reads it without a pass before:
    bit for bit its two halves by themselves, which take the pass (no output pixel sees both)."""
    H, W = 124, 131
    rng = np.random.default_rng(Cin)
    wd = torch.from_numpy(rng.standard_normal((Cin, Cout, 2, 2)).astype(np.float16).view(np.int16)).cuda()
    bd = torch.from_numpy(rng.standard_normal(Cout).astype(np.float32)).cuda()
    xd = torch.from_numpy(rng.standard_normal((H * W, Cin)).astype(np.float32)).cuda()
    assert H * W * Cin > 10 ** 7 > H * W * Cin // 2
    y = torch.full((2, 4 * H * W, Cout), float("nan"), dtype=torch.float32, device="cuda")
    wt = mi.from_torch(wd, mi.F16, [2, 2, Cout, Cin])
    ctx.neck_deconv(wt, bd.data_ptr(), xd.data_ptr(), H, W, gelu, y[0].data_ptr())
    for i in range(2):
        ctx.neck_deconv(wt, bd.data_ptr(), xd[i * H * W // 2:].data_ptr(), H // 2, W, gelu, y[1, i * 2 * H * W:].data_ptr())
    ctx.synchronize()
    assert torch.isfinite(y).all() and torch.equal(y[0], y[1])

"""F32 MUL_MATs (fp32 MFMAs) and neck convolutions on the bf16-MFMA kernel (each
fp32 value as three bf16 ones, six products): against float64, at the edges of
their tiles (128 x 128, 32 of K), K remainders and K split, and with infinities
and NaN.

Bound, of the bf16-MFMA kernel, which the fp32 sums stay below too: an output adds six products per 32 of K into an fp32 accumulator, each
addition rounding by at most 2^-23 of a running sum that stays below
S = sum |w x|, and drops three products of at most 2^-24 S each:
(6 ceil(K / 32) + 4) 2^-23 S; a K split adds one rounding per range."""
from time import perf_counter

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _mul_mat(mi, ctx, w, x, noalloc=False):
    wd, xd = torch.from_numpy(w).cuda(), torch.from_numpy(x).cuda()
    out = torch.full((x.shape[0], w.shape[0]), float("nan"), dtype=torch.float32, device="cuda")
    call = ctx.mul_mat_noalloc if noalloc else ctx.mul_mat
    K = w.shape[1]
    call(mi.from_torch(wd, mi.F32, [K, w.shape[0]]), mi.from_torch(xd, mi.F32, [K, x.shape[0]]),
         mi.from_torch(out, mi.F32, [w.shape[0], x.shape[0]]))
    ctx.synchronize()
    return out.cpu().numpy()


def _bound(K, s, extra=0):
    return (6 * -(-K // 32) + 4 + extra) * 2.0 ** -23 * s + 1e-37


@pytest.mark.parametrize("M,N,K", [(1, 1, 128), (128, 128, 128), (129, 127, 132), (127, 130, 160), (33, 17, 588),
                                   (300, 257, 1020), (5, 260, 2304)])
@pytest.mark.parametrize("noalloc", [False, True])
def test_mul_mat_f32_split(mi, ctx, M, N, K, noalloc):
    rng = np.random.default_rng(M * 7 + N + K)
    w = (rng.standard_normal((N, K)) * np.exp(rng.uniform(-3, 3, (N, 1)))).astype(np.float32)
    x = (rng.standard_normal((M, K)) * np.exp(rng.uniform(-8, 8, (M, K)))).astype(np.float32)
    got = _mul_mat(mi, ctx, w, x, noalloc).astype(np.float64)
    ref, s = x.astype(np.float64) @ w.astype(np.float64).T, np.abs(x).astype(np.float64) @ np.abs(w).astype(np.float64).T
    assert (np.abs(got - ref) <= _bound(K, s)).all(), float((np.abs(got - ref) / s).max())


def test_mul_mat_f32_split_exact_integers(mi, ctx):
    """Whole numbers whose sums stay below 2^24 come out exact (24-bit operands use all three planes)."""
    rng = np.random.default_rng(3)
    x = np.zeros((70, 256), np.float32)
    x[np.arange(70), rng.integers(0, 256, 70)] = rng.integers(-(2 ** 24) + 1, 2 ** 24, 70)
    w = rng.integers(-1, 2, (90, 256)).astype(np.float32)
    assert np.array_equal(_mul_mat(mi, ctx, w, x), x @ w.T)


def test_mul_mat_f32_split_non_finite(mi, ctx):
    """Infinities, NaN, and activations that round up to an infinite bf16 give what fp32 products
    and sums give: weights of one significant bit have two zero planes."""
    M, N, K = 140, 150, 192
    rng = np.random.default_rng(5)
    w = np.exp2(rng.integers(-3, 4, (N, K))).astype(np.float32) * rng.choice([-1, 1], (N, K)).astype(np.float32)
    x = rng.standard_normal((M, K)).astype(np.float32)
    inf, top = np.float32(np.inf), np.float32(3.4e38)
    x[3, 5], x[9, 7], x[9, 100] = inf, inf, -inf
    x[77, 191], x[139, 0] = np.nan, -inf
    w[20, 7] = 0.0           # 0 * inf
    w[:, 33] = np.abs(w[:, 33]) * 0 + 0.5
    x[50, 33] = top          # finite: its bf16 rounds to infinity
    x[50, :33] = x[50, 34:] = 0
    w[149, 64], w[0, 191] = inf, np.nan
    got = _mul_mat(mi, ctx, w, x)
    with np.errstate(all="ignore"):
        ref = np.zeros((M, N), np.float32)
        for k in range(K):
            ref = ref + x[:, k:k + 1] * w[:, k][None, :]
    assert np.array_equal(np.isnan(got), np.isnan(ref))
    assert np.array_equal(np.isinf(got), np.isinf(ref)) and np.array_equal(got[np.isinf(ref)], ref[np.isinf(ref)])
    ok = np.isfinite(ref)
    with np.errstate(all="ignore"):
        s = np.abs(x.astype(np.float64)) @ np.abs(w.astype(np.float64)).T
    assert (np.abs(got[ok].astype(np.float64) - ref[ok]) <= 4 * _bound(K, s[ok])).all()


@pytest.mark.parametrize("H,W,Cin,Cout,k", [(8, 8, 32, 32, 3), (17, 11, 64, 36, 3), (23, 20, 256, 256, 3), (9, 13, 36, 20, 1),
                                            (40, 33, 160, 132, 1)])
@pytest.mark.parametrize("special", [False, True])
def test_neck_conv_f32_split(mi, ctx, H, W, Cin, Cout, k, special):
    rng = np.random.default_rng(H * W + Cin + k)
    w = rng.standard_normal((Cout, Cin, k, k)).astype(np.float32)
    b = rng.standard_normal(Cout).astype(np.float32)
    x = rng.standard_normal((H, W, Cin)).astype(np.float32)
    if special:  # one infinite pixel channel: the outputs its taps reach are infinite, the others untouched
        x[H // 2, W // 2, Cin - 1] = np.inf
    wd, bd, xd = (torch.from_numpy(a).cuda() for a in (w, b, x))
    y = torch.full((H * W, Cout), float("nan"), dtype=torch.float32, device="cuda")
    ctx.neck_conv(mi.from_torch(wd, mi.F32, [k, k, Cin, Cout]), bd.data_ptr(), xd.data_ptr(), H, W, y.data_ptr())
    ctx.synchronize()
    pad = np.zeros((H + k - 1, W + k - 1, Cin))
    pad[k // 2:k // 2 + H, k // 2:k // 2 + W] = x
    ref, s = np.zeros((H * W, Cout)), np.zeros((H * W, Cout))
    with np.errstate(all="ignore"):
        for i in range(k):
            for j in range(k):
                a, t = pad[i:i + H, j:j + W].reshape(H * W, Cin), w[:, :, i, j].astype(np.float64)
                ref += a @ t.T
                s += np.abs(a) @ np.abs(t).T
    got = y.cpu().numpy().astype(np.float64)
    fin = np.isfinite(ref)
    assert fin.all() != special
    assert np.array_equal(np.isinf(got), np.isinf(ref)) and np.array_equal(got[~fin], ref[~fin])
    err = np.abs(got[fin] - (ref + b)[fin])
    assert (err <= _bound(Cin * k * k, s[fin], 20) + 2.0 ** -23 * (np.abs(ref[fin]) + np.abs(np.broadcast_to(b, ref.shape)[fin]))).all()


@pytest.mark.parametrize("value", [float("inf"), float("nan")])
def test_neck_conv_f32_non_finite_takes_no_hundredfold(mi, ctx, value):
    """Outputs that are not finite are summed again by the whole wavefront: one infinite pixel makes
    a 72 x 72 call some three times as long (the other wavefronts wait), not a hundred times."""
    H, C = 72, 256
    g = torch.Generator(device="cuda").manual_seed(1)
    w, b = torch.randn((C, C, 3, 3), generator=g, device="cuda"), torch.zeros(C, device="cuda")
    x, y = torch.randn((H * H, C), generator=g, device="cuda"), torch.empty((H * H, C), device="cuda")

    def time():
        best = float("inf")
        for _ in range(5):
            ctx.synchronize()
            t = perf_counter()
            for _ in range(4):
                ctx.neck_conv(mi.from_torch(w, mi.F32, [3, 3, C, C]), b.data_ptr(), x.data_ptr(), H, H, y.data_ptr())
            ctx.synchronize()
            best = min(best, perf_counter() - t)
        return best

    finite = time()
    x[H * H // 2 + 5, 3] = value
    assert time() <= 15 * finite
    assert int((~torch.isfinite(y)).sum()) == 9 * C


@pytest.mark.parametrize("xs,ws", [(1.0, 1.0), (1e-36, 1.0), (1.0, 1e-36), (2e-38, 64.0), (1e-42, 1e6), (1e6, 1e-42), (1e-20, 1e-13),
                                   (1e30, 1e-30), (1e33, 1e-3), (1e-3, 1e33), (1e20, 1e10)])
@pytest.mark.parametrize("k,Cin,Cout", [(1, 588, 140), (3, 64, 36)])
def test_neck_conv_f32_error_at_every_magnitude(mi, ctx, k, Cin, Cout, xs, ws):
    """rms error of sqrt(K) roundings of 2^-24 each, from subnormal operands to outputs of 1e33."""
    H, W, K = 13, 11, k * k * Cin
    rng = np.random.default_rng(17)
    w = (rng.standard_normal((Cout, Cin, k, k)) * ws).astype(np.float32)
    x = (rng.standard_normal((H, W, Cin)) * xs).astype(np.float32)
    wd, bd, xd = torch.from_numpy(w).cuda(), torch.zeros(Cout, device="cuda"), torch.from_numpy(x).cuda()
    y = torch.full((H * W, Cout), float("nan"), dtype=torch.float32, device="cuda")
    ctx.neck_conv(mi.from_torch(wd, mi.F32, [k, k, Cin, Cout]), bd.data_ptr(), xd.data_ptr(), H, W, y.data_ptr())
    ctx.synchronize()
    pad = np.zeros((H + k - 1, W + k - 1, Cin))
    pad[k // 2:k // 2 + H, k // 2:k // 2 + W] = x
    ref = np.zeros((H * W, Cout))
    for i in range(k):
        for j in range(k):
            ref += pad[i:i + H, j:j + W].reshape(H * W, Cin) @ w[:, :, i, j].astype(np.float64).T
    err = np.sqrt(np.mean((y.cpu().numpy() - ref) ** 2) / np.mean(ref ** 2))
    assert err <= K ** 0.5 * 2.0 ** -24, err


def _whole(rng, shape, bits):
    """Odd whole numbers of up to `bits` bits, either sign."""
    return ((rng.integers(0, 2 ** (bits - 1), shape) * 2 + 1) * rng.choice([-1, 1], shape)).astype(np.float32)


def _exact_case(rng, planes, H, W, Cin, Cout, k):
    """A map [H, W, Cin] and a kernel [Cout, Cin, k, k] of which every output is one product, exact in
    fp32: whole numbers of 24 bits (all three planes) on one side and +-1 on the other, or of 12 bits
    (two planes each, of which the product of the lower ones counts) on both."""
    x, w = np.zeros((H, W, Cin), np.float32), np.zeros((Cout, Cin, k, k), np.float32)
    bits = {"kernel": (1, 24), "map": (24, 1), "both": (12, 12)}[planes]
    if planes == "map":  # one tap of one channel per output
        x = _whole(rng, x.shape, bits[0])
        w[np.arange(Cout), rng.integers(0, Cin, Cout), rng.integers(0, k, Cout), rng.integers(0, k, Cout)] = _whole(rng, Cout, 1)
    else:                # one channel of pixels three apart
        at = np.ix_(range(0, H, 3), range(0, W, 3))
        c = rng.integers(0, Cin, x[at].shape[:2])
        x[at[0], at[1], c] = _whole(rng, c.shape, bits[0])
        w = _whole(rng, w.shape, bits[1])
    return x, w


def _conv64(x, w):
    H, W, Cin = x.shape
    Cout, k = w.shape[0], w.shape[2]
    pad = np.zeros((H + k - 1, W + k - 1, Cin))
    pad[k // 2:k // 2 + H, k // 2:k // 2 + W] = x
    return sum(pad[i:i + H, j:j + W].reshape(H * W, Cin) @ w[:, :, i, j].astype(np.float64).T for i in range(k) for j in range(k))


@pytest.mark.parametrize("H,W,Cin,Cout,k", [(1, 1, 128, 4, 1), (16, 8, 128, 128, 1), (43, 3, 132, 124, 1), (127, 1, 160, 132, 1),
                                            (11, 3, 588, 16, 1), (20, 15, 1020, 260, 1), (5, 1, 2304, 260, 1), (9, 13, 36, 20, 1),
                                            (17, 11, 64, 36, 3), (16, 8, 32, 128, 3), (43, 3, 96, 124, 3), (23, 20, 256, 256, 3)])
@pytest.mark.parametrize("planes", ["kernel", "map", "both"])
@pytest.mark.parametrize("offset", [0, 1])
def test_neck_conv_f32_exact_integers(mi, ctx, H, W, Cin, Cout, k, planes, offset):
    """Equality where an error bound cannot tell a missing plane or product; also with rows that
    float4 stores cannot reach (offset: floats by which the output misses 16 bytes)."""
    x, w = _exact_case(np.random.default_rng(H * W + Cin + k), planes, H, W, Cin, Cout, k)
    wd, bd, xd = torch.from_numpy(w).cuda(), torch.zeros(Cout, device="cuda"), torch.from_numpy(x).cuda()
    y = torch.full((H * W * Cout + 2,), float("nan"), dtype=torch.float32, device="cuda")
    ctx.neck_conv(mi.from_torch(wd, mi.F32, [k, k, Cin, Cout]), bd.data_ptr(), xd.data_ptr(), H, W, y.data_ptr() + 4 * offset)
    ctx.synchronize()
    got = y.cpu().numpy()
    assert np.isnan(got[:offset]).all() and np.isnan(got[offset + H * W * Cout:]).all()
    assert np.array_equal(got[offset:offset + H * W * Cout].reshape(H * W, Cout), _conv64(x, w))


@pytest.mark.parametrize("planes", ["kernel", "map", "both"])
@pytest.mark.parametrize("at", ["conv1x1", "conv3x3"])
def test_sam3_neck_f32_exact_integers(mi, ctx, planes, at):
    """The same through the fused neck's scale 2 (1x1, then 3x3), whose kernels one launch repacks;
    the other convolution passes its map on."""
    E, G, C1, D = 160, 12, 64, 96
    rng = np.random.default_rng(5)
    one, three = np.zeros((D, E, 1, 1), np.float32), np.zeros((D, D, 3, 3), np.float32)
    one[np.arange(D), np.arange(D), 0, 0] = three[np.arange(D), np.arange(D), 1, 1] = 1
    x = np.zeros((G, G, E), np.float32)
    if at == "conv1x1":
        x, one = _exact_case(rng, planes, G, G, E, D, 1)
    else:
        x[..., :D], three = _exact_case(rng, planes, G, G, D, D, 3)
    ref = _conv64(_conv64(x, one).reshape(G, G, D), three)
    keep, scales = [], []
    for shapes in ([("deconv1", E, C1), ("deconv2", C1, D), ("conv1x1", D, D), ("conv3x3", D, D)],
                   [("deconv1", E, C1), ("conv1x1", D, C1), ("conv3x3", D, D)], [("conv1x1", D, E), ("conv3x3", D, D)],
                   [("conv1x1", D, E), ("conv3x3", D, D)]):
        s = {}
        for n, a, b in shapes:
            k = {"deconv1": 2, "deconv2": 2, "conv1x1": 1, "conv3x3": 3}[n]
            w = torch.zeros((a, b, k, k)) if len(scales) != 2 else torch.from_numpy(one if n == "conv1x1" else three)
            bias = torch.zeros(b if k == 2 else a, device="cuda")
            keep += [w.cuda(), bias]
            s[n + "_w"] = mi.from_torch(keep[-2], mi.F32, [k, k, b, a])
            s[n + "_b"] = bias.data_ptr()
        scales.append(s)
    out = [torch.full((h * h, D), float("nan"), dtype=torch.float32, device="cuda") for h in (4 * G, 2 * G, G, G // 2)]
    xd = torch.from_numpy(x).cuda()
    ctx.sam3_neck(xd.data_ptr(), E, G, scales, [o.data_ptr() for o in out])
    ctx.synchronize()
    assert np.array_equal(out[2].cpu().numpy(), ref)

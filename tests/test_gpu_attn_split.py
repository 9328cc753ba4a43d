"""FLASH_ATTN_EXT over key ranges: ragged last ranges, ranges of two key tiles,
both staging paths, one range and several to a workgroup, and every count of
ranges from 4 to 16, against softmax in float64.

A workgroup takes the reference of its probabilities anew at each of its
ranges, also when the second half's scores lie far below or above the first's.
Probabilities are rounded to fp16 (2^-11 relative), so an output is off by at
most 2^-10 sum p |v| plus the fp32 sums' share: 1.5e-3 of it here."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D", [64, 96, 128])
@pytest.mark.parametrize("H,nq,nkv", [(1, 1, 512), (1, 100, 5000), (2, 130, 1111), (4, 1021, 3999), (16, 576, 640), (13, 1000, 700)])
@pytest.mark.parametrize("pad", [0, 4])
@pytest.mark.parametrize("shift", [0.0, 30.0, -30.0])
def test_flash_attn_key_ranges(mi, ctx, D, H, nq, nkv, pad, shift):
    g = torch.Generator(device="cuda").manual_seed(nq + nkv + D)
    q, k, v = (torch.randn((H, n, D + pad), generator=g, device="cuda") for n in (nq, nkv, nkv))
    q[..., 0] = D ** 0.5 / 4  # key component 0 raises or lowers the second half's scores by `shift`
    k[:, nkv // 2:, 0] += shift * 4 / D ** 0.5 * D ** 0.5 / 4
    q, k, v = q.half(), k.half(), v.half()
    out = torch.full((nq, H, D), float("nan"), device="cuda")
    s = 2 * (D + pad)
    t = lambda a: mi.from_torch(a, mi.F16, [D, a.shape[1], H, 1], [2, s, s * a.shape[1], s * a.shape[1] * H])
    ctx.flash_attn_ext(t(q), t(k), t(v), mi.from_torch(out, mi.F32, [D, H, nq, 1]), D ** -0.5)
    ctx.synchronize()
    qd, kd, vd = (a[..., :D].double() for a in (q, k, v))
    for h in range(H):
        p = torch.softmax(torch.mm(qd[h], kd[h].T.contiguous()) * D ** -0.5, -1)
        ref, w = torch.mm(p, vd[h]), torch.mm(p, vd[h].abs())
        err = (out[:, h].double() - ref).abs()
        assert bool((err <= 1.5e-3 * w).all()), float((err / w).max())


@pytest.mark.parametrize("ntile", range(8, 34, 2))
def test_flash_attn_every_range_count(mi, ctx, ntile):
    """One workgroup's queries: ntile / 2 ranges of two key tiles (at most 16)."""
    nq, nkv, D = 5, 64 * ntile - 7, 64
    g = torch.Generator(device="cuda").manual_seed(ntile)
    q, k, v = (torch.randn((n, D), generator=g, device="cuda").half() for n in (nq, nkv, nkv))
    out = torch.full((nq, 1, D), float("nan"), device="cuda")
    ctx.flash_attn_ext(*(mi.from_torch(a, mi.F16, [D, a.shape[0], 1, 1]) for a in (q, k, v)),
                       mi.from_torch(out, mi.F32, [D, 1, nq, 1]), D ** -0.5)
    ctx.synchronize()
    qd, kd, vd = (a.double() for a in (q, k, v))
    p = torch.softmax(torch.mm(qd, kd.T.contiguous()) * D ** -0.5, -1)
    err = (out[:, 0].double() - torch.mm(p, vd)).abs()
    assert bool((err <= 1.5e-3 * torch.mm(p, vd.abs())).all())


@pytest.mark.parametrize("H,nq,nkv", [(4, 1021, 3999), (12, 256, 4096), (16, 640, 512), (8, 1024, 1024), (8, 1150, 1020)])
@pytest.mark.parametrize("D,pad", [(64, 0), (96, 0), (128, 0), (96, 4)])
@pytest.mark.parametrize("shift", [0.0, 20.0, -20.0, -60.0])
def test_flash_attn_ranges_do_not_depend_on_the_grid(mi, ctx, D, pad, H, nq, nkv, shift):
    """All heads at once give a workgroup two or three ranges, one head at a time one; the ranges
    are the same, and so is every probability's fp16 rounding: what is left are the fp32 roundings
    of rescaling a workgroup's sums (at most two per range of 2^-24 each, and the combine's)."""
    g = torch.Generator(device="cuda").manual_seed(nq + nkv + D)
    q, k, v = (torch.randn((H, n, D + pad), generator=g, device="cuda") for n in (nq, nkv, nkv))
    q[..., 0] = D ** 0.5 / 4  # key component 0 raises or lowers the second half's scores by `shift`
    k[:, nkv // 2:, 0] += shift
    q, k, v = q.half(), k.half(), v.half()
    s = 2 * (D + pad)
    t = lambda a: mi.from_torch(a, mi.F16, [D, a.shape[1], a.shape[0], 1], [2, s, s * a.shape[1], s * a.shape[1] * a.shape[0]])
    both = []
    for heads in (H, 1):
        out = torch.full((H // heads, nq, heads, D), float("nan"), device="cuda")
        for i in range(H // heads):
            a = slice(i * heads, (i + 1) * heads)
            ctx.flash_attn_ext(t(q[a]), t(k[a]), t(v[a]), mi.from_torch(out[i], mi.F32, [D, heads, nq, 1]), D ** -0.5)
        ctx.synchronize()
        both.append((out[0] if heads == H else out[:, :, 0].transpose(0, 1)).double())
    assert torch.isfinite(both[0]).all()
    assert float((both[0] - both[1]).norm() / both[1].norm()) <= 1e-6

"""FLASH_ATTN_EXT over key ranges: every count of ranges the launcher picks
(2 to 16, ragged last ranges, ranges of two key tiles), both staging paths,
against softmax in float64.

A workgroup takes the reference of its probabilities anew halfway through its
range, also when the second half's scores lie far below or above the first's.
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

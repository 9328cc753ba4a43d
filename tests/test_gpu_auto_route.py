"""The default route of MUL_MATs with file-layout quantized weights, on both
sides of each line of its rule: it must give the bits of both forced routes."""
import numpy as np
import pytest
import torch

from gpu_helpers import dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tname", ["q8_0", "q4_0", "q4_1"])
@pytest.mark.parametrize("M,N,K", [(64, 548, 480), (65, 548, 480), (64, 548, 448), (64, 547, 480), (1, 256, 1024), (1, 252, 1024),
                                   (4096, 36, 128), (4095, 36, 128), (4096, 35, 160), (1793, 1667, 64), (1793, 1537, 96),
                                   (1792, 1668, 64)])
def test_auto_matches_both_routes(mi, ctx, orc, tname, M, N, K):
    t = orc.NAME_TYPE[tname]
    wd = dev(orc.quantize_weights(t, orc.normal(N * K, M + K, 1, std=0.02).reshape(N, K)).view(np.uint8))
    xd = dev(orc.normal(M * K, N, 2).reshape(M, K))
    wt, xt = mi.from_torch(wd, t, [K, N]), mi.from_torch(xd, mi.F32, [K, M])
    outs = []
    try:
        for kernel in (mi.MMQ_AUTO, mi.MMQ_F16, mi.MMQ_INT8):
            out = torch.full((M, N), float("nan"), dtype=torch.float32, device="cuda")
            ctx.set_mmq_kernel(kernel)
            ctx.mul_mat(wt, xt, mi.from_torch(out, mi.F32, [N, M]))
            ctx.synchronize()
            outs.append(out)
    finally:
        ctx.set_mmq_kernel(mi.MMQ_AUTO)
    assert torch.isfinite(outs[0]).all()
    assert torch.equal(outs[0], outs[1]) and torch.equal(outs[0], outs[2])

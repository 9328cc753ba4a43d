"""The default route of MUL_MATs with file-layout quantized weights, on both
sides of each line of its rule: it must give the bits of both forced routes."""
from time import perf_counter

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


@pytest.mark.parametrize("M,N,K", [(64, 256, 512), (64, 256, 544), (65, 320, 416), (64, 320, 416), (128, 32, 768), (129, 32, 768),
                                   (128, 4096, 768), (65, 81, 128), (65, 81, 160), (1297, 1540, 1856), (1297, 1540, 1888),
                                   (16300, 512, 1888)])
def test_auto_matches_both_routes_q4_1(mi, ctx, orc, M, N, K):
    test_auto_matches_both_routes(mi, ctx, orc, "q4_1", M, N, K)


@pytest.mark.parametrize("tname,M,N,K,kernel", [("q8_0", 9, 2540, 480, 1), ("q8_0", 36, 3604, 4512, 1), ("q4_0", 26, 164, 4640, 1),
                                                ("q4_1", 158, 260, 64, 0), ("q4_1", 68, 81, 64, 0)])
def test_auto_is_no_slower_than_the_types_own_route(mi, ctx, orc, tname, M, N, K, kernel):
    """Shapes at which the int8 route serves Q8_0 and Q4_0 (kernel 1), the fp16 route Q4_1 (0), in
    20 to 40 percent less time than the other: the default route is that one, within the clock's noise."""
    t = orc.NAME_TYPE[tname]
    wd = dev(orc.quantize_weights(t, orc.normal(N * K, 1, 1, std=0.02).reshape(N, K)).view(np.uint8))
    xd, out = dev(orc.normal(M * K, 2, 2).reshape(M, K)), torch.empty((M, N), device="cuda")
    args = mi.from_torch(wd, t, [K, N]), mi.from_torch(xd, mi.F32, [K, M]), mi.from_torch(out, mi.F32, [N, M])
    best = {}
    try:
        for _ in range(6):
            for k in (mi.MMQ_AUTO, kernel):
                ctx.set_mmq_kernel(k)
                for _ in range(3):
                    ctx.mul_mat(*args)
                ctx.synchronize()
                t0 = perf_counter()
                for _ in range(60):
                    ctx.mul_mat(*args)
                ctx.synchronize()
                best[k] = min(best.get(k, float("inf")), perf_counter() - t0)
    finally:
        ctx.set_mmq_kernel(mi.MMQ_AUTO)
    assert best[mi.MMQ_AUTO] <= 1.15 * best[kernel], best

"""MUL_MAT with F16 weights around the depth where the kernel changes (K = 640),
at row, column and K remainders, for aligned and unaligned destinations: the
results leave through LDS, as float4 or one column per lane.

Reference: float64 sums of the products of the fp16 operands. Each product is
exact in fp32; K additions of fp32 (rounded or truncated) err by at most
K * 2^-23 of the sum of the products' absolute values."""
import numpy as np
import pytest
import torch

from gpu_helpers import dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,N,K", [(1, 1, 640), (5, 3, 608), (127, 130, 632), (129, 127, 640), (64, 65, 648), (63, 191, 704),
                                   (200, 132, 712), (257, 258, 768), (130, 36, 4512)])
@pytest.mark.parametrize("off", [0, 1])
def test_f16_depths_and_remainders(mi, ctx, orc, M, N, K, off):
    w = orc.normal(N * K, M + K, 1, std=0.05).reshape(N, K).astype(np.float16)
    x = orc.normal(M * K, N, 2).reshape(M, K)
    wd, xd = dev(w), dev(x)
    buf = torch.full((M * N + 2,), float("nan"), dtype=torch.float32, device="cuda")
    out = buf[off:off + M * N]
    ctx.mul_mat(mi.from_torch(wd, mi.F16, [K, N]), mi.from_torch(xd, mi.F32, [K, M]), mi.from_torch(out, mi.F32, [N, M]))
    torch.cuda.synchronize()
    got = buf.cpu().numpy()
    assert np.isnan(got[:off]).all() and np.isnan(got[off + M * N:]).all()
    a, b = x.astype(np.float16).astype(np.float64), w.astype(np.float64)
    err = np.abs(got[off:off + M * N].reshape(M, N) - a @ b.T)
    assert (err <= K * 2.0 ** -23 * (np.abs(a) @ np.abs(b).T)).all()


@pytest.mark.parametrize("M,N,K", [(255, 129, 1000), (256, 129, 1000), (256, 129, 1024), (300, 259, 648), (16300, 257, 712),
                                   (16500, 257, 712)])
def test_f16_unsplit_rows_that_begin_within_lines(mi, ctx, orc, M, N, K):
    """Both sides of the rule by which ragged shapes of one workgroup per CU take the other kernel."""
    test_f16_depths_and_remainders(mi, ctx, orc, M, N, K, 0)

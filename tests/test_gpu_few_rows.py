"""MUL_MATs of few activation rows (at most 64, K <= 512) take one kernel that
quantizes the rows itself; it must give the bits of the quantize pass and the
tiled kernel (mi355_context_set_skinny off), K split included, at row, column
and block remainders, for padded activation rows, zero and special rows."""
import numpy as np
import pytest
import torch

from gpu_helpers import dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tname", ["q8_0", "q4_0", "q4_1"])
@pytest.mark.parametrize("M,N,K", [(1, 1, 32), (1, 4736, 512), (9, 256, 256), (31, 129, 96), (32, 100, 224), (33, 771, 480),
                                   (64, 1024, 512), (64, 36, 352), (2, 128, 64)])
@pytest.mark.parametrize("prepared", [True, False])
@pytest.mark.parametrize("pad", [0, 12])
def test_few_rows_bit_identical(mi, ctx, orc, tname, M, N, K, prepared, pad):
    t = orc.NAME_TYPE[tname]
    w = orc.quantize_weights(t, orc.normal(N * K, M + K, 1, std=0.02).reshape(N, K))
    x = orc.normal(M * (K + pad), N, 2).reshape(M, K + pad)
    x[0, :32] = 0.0
    if M > 1:
        x[1, :K] *= np.float32(1e-30)
        x[-1, K // 2] = 3e38
    wd, xd = dev(w.view(np.uint8)), dev(x)
    wt = mi.from_torch(wd, t, [K, N])
    if prepared:
        n = mi.weight_prepared_nbytes(wt)
        buf = torch.empty(n + 256, dtype=torch.uint8, device="cuda")
        wt = ctx.weight_prepare(wt, buf.data_ptr() + (-buf.data_ptr()) % 256, n)
    p = 4 * (K + pad)
    xt = mi.from_torch(xd, mi.F32, [K, M], [4, p, p * M, p * M])
    outs = []
    ctx.set_mmq_kernel(mi.MMQ_INT8)
    try:
        for few in (True, False):
            out = torch.full((M, N), float("nan"), dtype=torch.float32, device="cuda")
            ctx.set_skinny(few)
            ctx.mul_mat(wt, xt, mi.from_torch(out, mi.F32, [N, M]))
            ctx.synchronize()
            outs.append(out.cpu().numpy().view(np.uint32))
    finally:
        ctx.set_skinny(True)
        ctx.set_mmq_kernel(mi.MMQ_AUTO)
    assert np.array_equal(outs[0], outs[1])

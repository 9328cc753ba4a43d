"""F32 MUL_MATs run on the fp32 MFMA kernels from every entry point: no
workspace, no scratch, one result per operands, and fp32's precision at every
magnitude fp32 holds."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _tensors(mi, w, x):
    (N, K), M = w.shape, x.shape[0]
    out = torch.full((M, N), float("nan"), dtype=torch.float32, device="cuda")
    return mi.from_torch(w, mi.F32, [K, N]), mi.from_torch(x, mi.F32, [K, M]), mi.from_torch(out, mi.F32, [N, M]), out


@pytest.mark.parametrize("M,N,K", [(5, 96, 160), (3, 3500, 3200), (5, 4096, 4096)])
def test_same_bits_with_and_without_allocation(mi, ctx, M, N, K):
    """Weights up to and past what three 16-bit planes in the fixed 64 MiB scratch could hold."""
    g = torch.Generator(device="cuda").manual_seed(N)
    w, x = torch.randn((N, K), generator=g, device="cuda"), torch.randn((M, K), generator=g, device="cuda")
    s0, s1, d, a = _tensors(mi, w, x)
    ctx.mul_mat(s0, s1, d)
    _, _, d, b = _tensors(mi, w, x)
    ctx.mul_mat_noalloc(s0, s1, d)
    ctx.synchronize()
    assert torch.isfinite(a).all() and torch.equal(a, b)


def test_captured_call_outlives_the_workspace(mi):
    """A captured F32 call holds no library memory: replays give the eager bits, also after a
    quantized MUL_MAT has replaced the context's workspace by a larger one."""
    stream = torch.cuda.Stream()
    ctx = mi.Context(0, stream.cuda_stream)
    try:
        with torch.cuda.stream(stream):
            g = torch.Generator(device="cuda").manual_seed(11)
            w, x = torch.randn((300, 588), generator=g, device="cuda"), torch.randn((70, 588), generator=g, device="cuda")
            s0, s1, d, out = _tensors(mi, w, x)
            ctx.mul_mat(s0, s1, d)
            eager = out.clone()
            ctx.synchronize()
            graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(graph, stream=stream):
                ctx.mul_mat(s0, s1, d)
            rows = torch.zeros((512, 34 * 32), dtype=torch.uint8, device="cuda")
            y, r = torch.randn((900, 1024), device="cuda"), torch.empty((900, 512), device="cuda")
            for step in range(4):
                out.fill_(float("nan"))
                graph.replay()
                ctx.synchronize()
                assert torch.equal(out, eager), step
                n = 300 * (step + 1) - 300  # no rows, then growing operands in the workspace
                if n:
                    ctx.mul_mat(mi.from_torch(rows, mi.Q8_0, [1024, 512]), mi.from_torch(y, mi.F32, [1024, n]),
                                mi.from_torch(r, mi.F32, [512, n]))
                    ctx.synchronize()
    finally:
        ctx.close()


@pytest.mark.parametrize("xs,ws", [(1.0, 1.0), (1e-36, 1.0), (1.0, 1e-36), (2e-38, 64.0), (1e-20, 1e-13)])
def test_error_at_every_magnitude(mi, ctx, xs, ws):
    """The fp32 sums of K terms: rms error of sqrt(K) roundings of 2^-24 each."""
    M, N, K = 130, 140, 588
    rng = np.random.default_rng(17)
    w = (rng.standard_normal((N, K)) * ws).astype(np.float32)
    x = (rng.standard_normal((M, K)) * xs).astype(np.float32)
    s0, s1, d, out = _tensors(mi, torch.from_numpy(w).cuda(), torch.from_numpy(x).cuda())
    ctx.mul_mat(s0, s1, d)
    ctx.synchronize()
    ref = x.astype(np.float64) @ w.astype(np.float64).T
    err = np.sqrt(np.mean((out.cpu().numpy() - ref) ** 2) / np.mean(ref ** 2))
    assert err <= K ** 0.5 * 2.0 ** -24, err

"""GPU parity of the SAM3 ViT encoder path (sam3.cpp:3714-3853): each fused
node group against the oracle's ggml node sequence, the F32 mul_mat of the
patch embedding, the prefix, and whole blocks against the oracle's
composition of sam3_vit_block_forward.

Bars: bias/residual/win_part/win_unpart/RoPE passes are bit-exact (each ggml
node rounds to fp32 and so do the fused passes); LayerNorm is within 1 ulp
(mean and variance are reduced in double in another order); GELU-erf within
4 ulp plus the 1 + erf(x) cancellation term 1.2e-7*|x| (device erff vs the
host's).  A whole block is compared with the oracle run twice (the
fp16-rounded Q/K/V the GPU attention uses, evaluated exactly; ggml-cpu's F32
attention) at the bars of tests/block_refs.block_bars: within the two runs'
own spread (max 1.5x, RMS 1.25x, never tighter than 1e-2 / 5e-4; 1e-2 is the
CPU-vs-GPU block bound of the reference's tests/test_metal_overhead.cpp:
240-246) and no line of the difference with a mean beyond 6 standard errors.
Activation-quantization roundings flipped by upstream differences reach the
output; a wiring mistake gives errors of order 0.05-1.
"""
import ctypes as C

import numpy as np
import pytest
import torch

from gpu_helpers import dev

pytestmark = pytest.mark.gpu


def _p(t):
    return C.c_void_p(t.data_ptr())


def _ulp_diff(a, b):
    ai = a.view(np.int32).astype(np.int64)
    bi = b.view(np.int32).astype(np.int64)
    ai = np.where(ai < 0, -(ai & 0x7fffffff), ai)
    bi = np.where(bi < 0, -(bi & 0x7fffffff), bi)
    return np.abs(ai - bi)


from block_refs import axial_cis, block_bars, gelu_ref, ln_ref, rope_ref, vit_block_ref, win_part, win_unpart  # noqa: E402


# ---------------------------------------------------------------- fused passes
# E = 256 and 1024 take the grouped kernel (64 lanes x 1 or 4 float4 per row),
# E = 1152 (V = 9 float4 per lane) the one-wavefront-per-row kernel
@pytest.mark.parametrize("window,add_grid,E", [(0, 0, 256), (24, 0, 256), (0, 24, 256), (24, 0, 1024), (0, 0, 1152)])
def test_layer_norm(mi, ctx, orc, window, add_grid, E):
    grid = 48
    M = grid * grid
    x = orc.normal(M * E, 1, 1).reshape(M, E) * np.float32(3.0) + np.float32(0.5)
    w = orc.normal(E, 1, 2) * np.float32(0.2) + np.float32(1.0)
    b = orc.normal(E, 1, 3) * np.float32(0.1)
    pos = orc.normal(add_grid * add_grid * E, 1, 4).reshape(-1, E) if add_grid else None
    xd, wd, bd = dev(x), dev(w), dev(b)
    posd = dev(pos) if add_grid else None
    y = torch.empty_like(xd)
    ctx.vit_layer_norm(_p(xd), _p(posd) if add_grid else None, add_grid, _p(wd), _p(bd), _p(y), M, E, grid, window)
    ctx.synchronize()
    got = y.cpu().numpy()
    xin = x
    if add_grid:
        r = np.arange(M)
        pr = (r // grid % add_grid) * add_grid + (r % grid) % add_grid
        xin = (x + pos[pr]).astype(np.float32)
    ref = ln_ref(orc, xin, w, b)
    if window:
        ref = win_part(orc, ref, grid, window)
    assert _ulp_diff(got, ref).max() <= 1


def test_qkv_rope_bit_exact(mi, ctx, orc):
    NH, HD, ws, B = 4, 64, 24, 4
    E, N = NH * HD, ws * ws
    M = N * B
    qkv = orc.normal(M * 3 * E, 2, 1).reshape(M, 3 * E)
    bias = orc.normal(3 * E, 2, 2) * np.float32(0.1)
    freqs = axial_cis(orc, HD, ws, 1.0)
    qkvd, bd, fd = dev(qkv), dev(bias), dev(freqs)
    q = torch.empty((B, NH, N, HD), dtype=torch.float16, device="cuda")
    k, v = torch.empty_like(q), torch.empty_like(q)
    ctx.vit_qkv_rope(_p(qkvd), _p(bd), _p(fd), _p(q), _p(k), _p(v), M, N, NH, HD)
    ctx.synchronize()
    t = (qkv + bias).astype(np.float32)  # ggml_add(qkv, qkv_b)
    parts = [t[:, i * E:(i + 1) * E].reshape(B, N, NH, HD).transpose(0, 2, 1, 3) for i in range(3)]
    qr = rope_ref(orc, parts[0], freqs, HD, N).reshape(B, NH, N, HD)
    kr = rope_ref(orc, parts[1], freqs, HD, N).reshape(B, NH, N, HD)
    assert np.array_equal(q.cpu().numpy(), qr.astype(np.float16))
    assert np.array_equal(k.cpu().numpy(), kr.astype(np.float16))
    assert np.array_equal(v.cpu().numpy(), parts[2].astype(np.float16))


@pytest.mark.parametrize("window", [0, 24])
def test_proj_residual_bit_exact(mi, ctx, orc, window):
    grid, E = 48, 256
    M = grid * grid
    x = orc.normal(M * E, 3, 1).reshape(M, E)
    p = orc.normal(M * E, 3, 2).reshape(M, E)
    b = orc.normal(E, 3, 3)
    xd, pd, bd = dev(x), dev(p), dev(b)
    ctx.vit_proj_residual(_p(xd), _p(pd), _p(bd), M, E, grid, window)
    ctx.synchronize()
    t = (p + b).astype(np.float32)
    if window:
        t = win_unpart(orc, t, grid, window)
    assert np.array_equal(xd.cpu().numpy(), (x + t).astype(np.float32))


def test_bias_gelu_and_residual(mi, ctx, orc):
    rows, n = 300, 4736
    h = orc.normal(rows * n, 4, 1).reshape(rows, n) * np.float32(2.0)
    b = orc.normal(n, 4, 2)
    hd_, bd = dev(h), dev(b)
    ctx.vit_bias_gelu(_p(hd_), _p(bd), rows, n)
    ctx.synchronize()
    u = (h + b).astype(np.float32)
    ref = gelu_ref(orc, u)
    got = hd_.cpu().numpy()
    # 4 ulp of the result, plus the cancellation in 1 + erf(x) for negative x:
    # one ulp of 1 (1.19e-7) times 0.5*|u|
    bound = 4 * np.spacing(np.abs(ref)) + 1.2e-7 * np.abs(u)
    assert (np.abs(got - ref) <= bound).all()
    x = orc.normal(rows * n, 4, 3).reshape(rows, n)
    xd, fd = dev(x), dev(h)
    ctx.vit_bias_residual(_p(xd), _p(fd), _p(bd), rows, n)
    ctx.synchronize()
    assert np.array_equal(xd.cpu().numpy(), (x + (h + b).astype(np.float32)).astype(np.float32))


def test_gelu_erf_against_exact(mi, ctx):
    """The device GELU's erf (a fitted polynomial-and-exp2 form) against
    0.5 u (1 + erf(u / sqrt(2))) in double, on 4M evenly spaced u in [-9, 9] and on every
    float around the erf pieces' boundary (u = +-sqrt(2)) and clamp (u = +-4 sqrt(2)).  The
    erf error (< 9e-8), the rounding of u / sqrt(2) (through erf's slope, < 4e-8) and the
    rounding of 1 + erf (1.2e-7) bound |got - exact| by 1.3e-7 |u|, plus one ulp of the
    result for its own rounding."""
    from scipy.special import erf
    parts = [np.linspace(-9, 9, 1 << 22, dtype=np.float32)]
    for c in (np.sqrt(2.0), 4 * np.sqrt(2.0)):
        m = int(np.float32(c).view(np.uint32))
        near = np.arange(m - 100000, m + 100000, dtype=np.uint32).view(np.float32)
        parts += [near, -near]
    u = np.concatenate(parts)
    n = 4096
    u = np.concatenate([u, np.zeros((-len(u)) % n, np.float32)])
    rows = len(u) // n
    hd_, bd = dev(u.reshape(rows, n)), dev(np.zeros(n, np.float32))
    ctx.vit_bias_gelu(_p(hd_), _p(bd), rows, n)
    ctx.synchronize()
    got = hd_.cpu().numpy().reshape(-1).astype(np.float64)
    u64 = u.astype(np.float64)
    exact = 0.5 * u64 * (1.0 + erf(u64 / np.sqrt(2.0)))
    bound = 1.3e-7 * np.abs(u64) + np.spacing(np.abs(exact).astype(np.float32)).astype(np.float64)
    err = np.abs(got - exact)
    assert (err <= bound).all(), (float(u[np.argmax(err - bound)]), float((err - bound).max()))


@pytest.mark.parametrize("M,N,K", [(1, 1, 1), (70, 33, 588), (5184, 1024, 588)])
def test_mul_mat_f32(mi, ctx, orc, M, N, K):
    """F32 x F32 mul_mat (patch embedding): |gpu - exact| <= 1e-5 * sum|w x|."""
    w = orc.normal(N * K, 5, 1, std=0.02).reshape(N, K)
    x = orc.normal(M * K, 5, 2).reshape(M, K)
    wd, xd = dev(w), dev(x)
    dst = torch.empty((M, N), dtype=torch.float32, device="cuda")
    ctx.mul_mat(mi.from_torch(wd, mi.F32, [K, N]), mi.from_torch(xd, mi.F32, [K, M]), mi.from_torch(dst, mi.F32, [N, M]))
    ctx.synchronize()
    rows = np.arange(M) if M <= 256 else np.linspace(0, M - 1, 128).astype(int)
    ref = x[rows].astype(np.float64) @ w.T.astype(np.float64)
    absterm = np.abs(x[rows]).astype(np.float64) @ np.abs(w.T).astype(np.float64)
    assert (np.abs(dst.cpu().numpy()[rows] - ref) <= 1e-5 * absterm + 1e-30).all()


# ---------------------------------------------------------------- prefix and blocks
def _hp(mi, E, NH, MLP, ws, grid, P=14, pos_grid=24):
    hp = mi.VitHparams()
    hp.embed_dim, hp.num_heads, hp.mlp_dim, hp.window_size = E, NH, MLP, ws
    hp.grid, hp.patch_size, hp.pos_grid, hp.eps = grid, P, pos_grid, 1e-5
    return hp


def test_vit_prefix(mi, ctx, orc):
    E, grid, P, pg = 256, 48, 14, 24
    img = orc.uniform(3 * (grid * P) ** 2, 6, 1).reshape(3, grid * P, grid * P)
    pw = orc.normal(E * 3 * P * P, 6, 2, std=0.02).reshape(E, 3, P, P)  # ggml [P, P, 3, E]
    pos = orc.normal(pg * pg * E, 6, 3).reshape(pg * pg, E)
    lw = orc.normal(E, 6, 4) * np.float32(0.2) + np.float32(1.0)
    lb = orc.normal(E, 6, 5) * np.float32(0.1)
    hp = _hp(mi, E, 4, 1024, 24, grid, P, pg)
    imgd, pwd, posd, lwd, lbd = dev(img), dev(pw), dev(pos), dev(lw), dev(lb)
    x = torch.empty((grid * grid, E), dtype=torch.float32, device="cuda")
    ctx.vit_prefix(hp, _p(imgd), mi.from_torch(pwd, mi.F32, [P, P, 3, E]), _p(posd), _p(lwd), _p(lbd), _p(x))
    ctx.synchronize()
    # oracle: im2col + F32 mul_mat (ggml_conv_2d_sk_p0), + tiled pos, ln_pre
    cols = img.reshape(3, grid, P, grid, P).transpose(1, 3, 0, 2, 4).reshape(grid * grid, 3 * P * P)
    conv = orc.mul_mat(pw.reshape(E, -1), orc.F32, 3 * P * P, E, np.ascontiguousarray(cols))
    conv = conv.reshape(grid * grid, E)
    r = np.arange(grid * grid)
    pr = (r // grid % pg) * pg + (r % grid) % pg
    ref = ln_ref(orc, (conv + pos[pr]).astype(np.float32), lw, lb)
    assert np.abs(x.cpu().numpy() - ref).max() <= 1e-4


def _block_weights(mi, orc, t, E, MLP, seed):
    shapes = {"qkv": (3 * E, E), "proj": (E, E), "fc1": (MLP, E), "fc2": (E, MLP)}
    host, devs = {}, {}
    for i, (name, (N, K)) in enumerate(shapes.items()):
        w = orc.normal(N * K, seed, 10 + i, std=0.02).reshape(N, K)
        q = orc.quantize_weights(t, w)
        host[name] = (q, N, K)
        devs[name] = dev(q.view(np.uint8) if q.dtype != np.float32 else q)
    vec = {}
    for i, (name, n, s, m) in enumerate([("norm1_w", E, 0.2, 1.0), ("norm1_b", E, 0.1, 0.0), ("qkv_b", 3 * E, 0.05, 0.0),
                                          ("proj_b", E, 0.05, 0.0), ("norm2_w", E, 0.2, 1.0), ("norm2_b", E, 0.1, 0.0),
                                          ("fc1_b", MLP, 0.05, 0.0), ("fc2_b", E, 0.05, 0.0)]):
        vec[name] = orc.normal(n, seed, 20 + i) * np.float32(s) + np.float32(m)
    return host, devs, vec


@pytest.mark.parametrize("is_global", [0, 1])
@pytest.mark.parametrize("tname", ["q8_0", "q4_0"])
def test_vit_block(mi, ctx, orc, is_global, tname):
    t = orc.NAME_TYPE[tname]
    E, NH, MLP, grid, ws = 256, 4, 1024, 48, 24
    HD = E // NH
    M = grid * grid
    host, devs, vec = _block_weights(mi, orc, t, E, MLP, seed=7 + is_global)
    freqs = axial_cis(orc, HD, grid, ws / grid) if is_global else axial_cis(orc, HD, ws, 1.0)
    x0 = orc.normal(M * E, 8, 1).reshape(M, E)
    vd = {k: dev(v) for k, v in vec.items()}
    fd = dev(freqs)
    blk = mi.VitBlock()
    for name in ("qkv", "proj", "fc1", "fc2"):
        _, N, K = host[name]
        setattr(blk, name + "_w", mi.from_torch(devs[name], t, [K, N]))
    for k, v in vd.items():
        setattr(blk, k, v.data_ptr())
    blk.freqs_cis = fd.data_ptr()
    blk.is_global = is_global
    hp = _hp(mi, E, NH, MLP, ws, grid)
    x = dev(x0)
    ctx.vit_block_forward(hp, blk, _p(x))
    ctx.synchronize()
    got = x.cpu().numpy()
    assert np.isfinite(got).all()
    # each stage is pinned tightly by the tests above; here activation-quantization
    # roundings flipped by ~1e-4 upstream differences reach the output
    ref16 = vit_block_ref(orc, t, x0, host, vec, E, NH, MLP, grid, 0 if is_global else ws, freqs, True)
    ref32 = vit_block_ref(orc, t, x0, host, vec, E, NH, MLP, grid, 0 if is_global else ws, freqs, False)
    block_bars(got, ref16, ref32, f"vit block {tname} global={is_global}")


@pytest.mark.parametrize("is_global", [0, 1])
@pytest.mark.parametrize("tname", ["f16", "q8_0", "q4_0", "q4_1"])
def test_vit_block_fusion_bit_exact(mi, ctx, orc, is_global, tname):
    """The fused LN / GELU producers write exactly the operand mul_mat would
    make from their f32 rows: fused and unfused blocks agree bit for bit."""
    t = orc.NAME_TYPE[tname]
    E, NH, MLP, grid, ws = 256, 4, 1024, 48, 24
    HD = E // NH
    M = grid * grid
    host, devs, vec = _block_weights(mi, orc, t, E, MLP, seed=17 + is_global)
    freqs = axial_cis(orc, HD, grid, ws / grid) if is_global else axial_cis(orc, HD, ws, 1.0)
    x0 = orc.normal(M * E, 9, 1).reshape(M, E)
    vd = {k: dev(v) for k, v in vec.items()}
    fd = dev(freqs)
    blk = mi.VitBlock()
    for name in ("qkv", "proj", "fc1", "fc2"):
        _, N, K = host[name]
        setattr(blk, name + "_w", mi.from_torch(devs[name], t, [K, N]))
    for k, v in vd.items():
        setattr(blk, k, v.data_ptr())
    blk.freqs_cis = fd.data_ptr()
    blk.is_global = is_global
    hp = _hp(mi, E, NH, MLP, ws, grid)
    outs = []
    try:
        for fuse in (False, True):
            ctx.set_fusion(fuse)
            x = dev(x0)
            ctx.vit_block_forward(hp, blk, _p(x))
            ctx.synchronize()
            outs.append(x.cpu().numpy())
    finally:
        ctx.set_fusion(True)
    assert np.isfinite(outs[0]).all()
    assert np.array_equal(outs[0], outs[1]), f"max diff {np.abs(outs[0] - outs[1]).max():.3e}"


@pytest.mark.parametrize("tname", ["f16", "q8_0"])
def test_vit_block_attention_keeps_a_workgroup_per_range(mi, ctx, orc, tname):
    """A global block at a grid whose FLASH_ATTN_EXT call gives workgroups several key ranges (8 heads
    of 1024 tokens) equals the block composed of its ops with attention one head at a time, where
    each range has its own: no fp32 rounding differs, which a quantizer would make another quant of."""
    t = orc.NAME_TYPE[tname]
    E, NH, MLP, grid = 512, 8, 512, 32
    HD, M = E // NH, grid * grid
    host, devs, vec = _block_weights(mi, orc, t, E, MLP, seed=27)
    x0 = orc.normal(M * E, 28, 1).reshape(M, E)
    vd = {k: dev(v) for k, v in vec.items()}
    fd = dev(axial_cis(orc, HD, grid, 24 / grid))
    w = {n: mi.from_torch(devs[n], t, [host[n][2], host[n][1]]) for n in host}
    blk = mi.VitBlock()
    for n in w:
        setattr(blk, n + "_w", w[n])
    for k, v in vd.items():
        setattr(blk, k, v.data_ptr())
    blk.freqs_cis, blk.is_global = fd.data_ptr(), 1
    got = dev(x0)
    ctx.vit_block_forward(_hp(mi, E, NH, MLP, 16, grid, pos_grid=16), blk, _p(got))

    rows = lambda n: torch.empty((M, n), dtype=torch.float32, device="cuda")
    mm = lambda n, a, o: ctx.mul_mat(w[n], mi.from_torch(a, mi.F32, [a.shape[1], M]), mi.from_torch(o, mi.F32, [o.shape[1], M]))
    x, y, qkv, attn, h = dev(x0), rows(E), rows(3 * E), rows(E), rows(MLP)
    q, k, v = (torch.empty((NH, M, HD), dtype=torch.float16, device="cuda") for _ in range(3))
    ctx.vit_layer_norm(_p(x), None, 0, _p(vd["norm1_w"]), _p(vd["norm1_b"]), _p(y), M, E, grid)
    mm("qkv", y, qkv)
    ctx.vit_qkv_rope(_p(qkv), _p(vd["qkv_b"]), _p(fd), _p(q), _p(k), _p(v), M, M, NH, HD)
    for i in range(NH):
        o = rows(HD)
        ctx.flash_attn_ext(*(mi.from_torch(a[i], mi.F16, [HD, M, 1, 1]) for a in (q, k, v)),
                           mi.from_torch(o, mi.F32, [HD, 1, M, 1]), HD ** -0.5)
        ctx.synchronize()
        attn[:, i * HD:(i + 1) * HD] = o
    torch.cuda.synchronize()
    mm("proj", attn, y)
    ctx.vit_proj_residual(_p(x), _p(y), _p(vd["proj_b"]), M, E, grid)
    ctx.vit_layer_norm(_p(x), None, 0, _p(vd["norm2_w"]), _p(vd["norm2_b"]), _p(y), M, E, grid)
    mm("fc1", y, h)
    ctx.vit_bias_gelu(_p(h), _p(vd["fc1_b"]), M, MLP)
    mm("fc2", h, y)
    ctx.vit_bias_residual(_p(x), _p(y), _p(vd["fc2_b"]), M, E)
    ctx.synchronize()
    assert torch.isfinite(got).all() and torch.equal(got, x)

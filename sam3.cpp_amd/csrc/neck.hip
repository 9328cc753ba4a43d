// SAM3 SimpleFPN neck kernels (sam3_build_neck_graph, sam3.cpp:3867-3925) on
// token-major activations [H*W][C] (ggml [C, W, H]).  conv_f16_dma_kernel (over
// fp16 maps; conv_f32map_kernel for a 1x1 or conv-transpose over an F32 one, and conv_f16_kernel,
// register-staged, for the rest and operands beyond 32-bit buffer offsets) is the fp16-MFMA implicit GEMM of the F16-kernel convolutions (3x3,
// 1x1 and the 2x2 / stride-2 conv-transpose with its scatter, bias and GELU in
// the epilogue; the 3x3 and 1x1 split K on grids smaller than the CU count, the
// partial sums added by gemm_f32.hip's reduce); F32-kernel convolutions run on
// gemm_f32.hip.  The rest are
// HBM-bound passes: the conv-transpose kernel repack + F16 cast, the 3x3
// kernel repacks for the implicit GEMMs (one launch for all of a neck's), and, for maps the implicit GEMMs do
// not take, im2col, the conv-transpose scatter and bias adds; the 2x2
// max-pool.
#include "common.cuh"
#include "kernels.h"
#include "pack.cuh"

namespace mi355 {

namespace {
unsigned nblk(int64_t n) { return (unsigned)((n + 255) / 256); }
}

// a conv-transpose kernel's F16 GEMM rows (deconv_pack_block). Alone it is latency: 672 ->
// 4 x 32 with sixteen wavefronts a block 4.8 us, with four 7.6.
__global__ __launch_bounds__(1024) void deconv_pack_kernel(const void* __restrict__ w, int wtype, int Cin, int Cout,
                                                          uint16_t* __restrict__ out) {
    __shared__ uint16_t t[PACK_LDS];
    deconv_pack_block<16>(blockIdx.x, w, wtype, Cin, Cout, out, t);
}

// Every kernel of a neck repacked in one launch. Alone each of the seven to eleven repacks moves a few
// MB in 4 to 17 us, most of it the launch and the latency of one pass of scattered reads; together
// they overlap. A block serves one repack: the first whose end lies past it.
namespace {
struct NeckPacks {
    NeckPack j[NECK_PACKS];
    unsigned end[NECK_PACKS];  // block after the repack's last
    int n;
};
}  // namespace
__global__ __launch_bounds__(256) void neck_pack_kernel(const NeckPacks p) {
    __shared__ uint16_t t[PACK_LDS];
    int i = 0;
    while (i + 1 < p.n && blockIdx.x >= p.end[i]) ++i;
    const NeckPack& j = p.j[i];
    const int64_t blk = blockIdx.x - (i ? p.end[i - 1] : 0), it = blk * 256 + threadIdx.x;
    if (j.k == 2) {
        deconv_pack_block<4>(blk, j.w, j.type, j.Cin, j.Cout, j.out, t);
    } else if (j.type == T_F16) {
        conv3x3_pack_f16_item(it, static_cast<const uint16_t*>(j.w), j.Cin, j.Cout, j.out);
    } else {
        const int taps = j.k * j.k, K = taps * j.Cin;
        split_w_item(it, static_cast<const float*>(j.w), taps, j.Cout, K, (K + 31) / 32 * 32, j.out);
    }
}

// y[(2py + kh)(2W) + 2px + kw][co] = D[py*W + px][(kh*2 + kw)*Cout + co] + b[co]
// (then GELU-erf, or not).  Four channels per thread; Cout % 4 == 0.
__global__ __launch_bounds__(256) void deconv_scatter_kernel(const float* __restrict__ D, const float* __restrict__ b,
                                                             int H, int W, int Cout, int gelu, float* __restrict__ y) {
    const int c4 = Cout / 4;
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= 4LL * H * W * c4) return;
    const int co = (int)(i % c4) * 4;
    const int64_t pix = i / c4;
    const int W2 = 2 * W;
    const int oy = (int)(pix / W2), ox = (int)(pix % W2);
    const int64_t p = (int64_t)(oy >> 1) * W + (ox >> 1);
    const int t = (oy & 1) * 2 + (ox & 1);
    v4f v = *reinterpret_cast<const v4f*>(&D[p * 4 * Cout + (int64_t)t * Cout + co]);
    const v4f bb = *reinterpret_cast<const v4f*>(&b[co]);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const float s = v[j] + bb[j];
        v[j] = gelu ? gelu_erf(s) : s;
    }
    *reinterpret_cast<v4f*>(&y[pix * Cout + co]) = v;
}

// ggml_im2col for a 3x3 / stride 1 / pad 1 convolution on token-major input:
// cols[p][(ic*3 + kh)*3 + kw] = x[(oy + kh - 1)*W + ox + kw - 1][ic], zero
// outside the image; F32, or F16 rounded to nearest even (im2col in the
// kernel's type).
template <bool F16>
__global__ __launch_bounds__(256) void im2col3x3_kernel(const float* __restrict__ x, int H, int W, int C,
                                                        void* __restrict__ cols) {
    const int64_t K = 9LL * C;
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (int64_t)H * W * K) return;
    const int64_t p = i / K;
    const int k = (int)(i - p * K);
    const int ic = k / 9, tap = k - ic * 9;
    const int oy = (int)(p / W) + tap / 3 - 1, ox = (int)(p % W) + tap % 3 - 1;
    const float v = oy >= 0 && oy < H && ox >= 0 && ox < W ? x[((int64_t)oy * W + ox) * C + ic] : 0.0f;
    if (F16) static_cast<uint16_t*>(cols)[i] = f2h(v);
    else static_cast<float*>(cols)[i] = v;
}

// F32 3x3 kernel [Cout][Cin][3][3] (ggml [3, 3, Cin, Cout]) -> rows [Cout][tap][Cin],
// tap = kh*3 + kw: the K order of the implicit-GEMM convolution
__global__ __launch_bounds__(256) void conv3x3_pack_kernel(const float* __restrict__ w, int Cin, int Cout,
                                                           float* __restrict__ out) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= 9LL * Cin * Cout) return;
    const int ci = (int)(i % Cin);
    const int64_t r = i / Cin;
    const int tap = (int)(r % 9), co = (int)(r / 9);
    out[i] = w[((int64_t)co * Cin + ci) * 9 + tap];
}

// F16 3x3 kernel [Cout][Cin][3][3] -> rows [Cout][tap][Cin] (the implicit GEMM's K order)
__global__ __launch_bounds__(256) void conv3x3_pack_f16_kernel(const uint16_t* __restrict__ w, int Cin, int Cout,
                                                               uint16_t* __restrict__ out) {
    conv3x3_pack_f16_item((int64_t)blockIdx.x * blockDim.x + threadIdx.x, w, Cin, Cout, out);
}

// ggml_conv_2d_s1_ph (TAPS = 9) or ggml_conv_2d_sk_p0 1x1 (TAPS = 1) with an F16
// kernel as an implicit GEMM: y[p][n] = bias[n] + sum_{tap, c} f16(x[p + tap
// offset][c]) * w[n][tap][c] over a token-major map (C % 32 == 0), zero outside
// the image.  TAPS = 4 is conv_transpose_2d_p0 (kernel 2, stride 2): the GEMM
// of the map with the deconv_pack rows [4*Cout][C], each column n = t*Cout + co
// stored to pixel (2py + t/2, 2px + t%2) of the 2x map as bias[co] + sum (then
// GELU-erf if gelu), the scatter of deconv_scatter_kernel done in registers.  The activations are rounded to fp16
// (RNE) as they are loaded, exactly as ggml's F16 im2col rounds them, so the
// products are those of im2col + F16 MUL_MAT; fp32 accumulation.
// Workgroup 128(m) x 128(n), four wavefronts of 64 x 64 (2 x 2
// v_mfma_f32_32x32x16_f16 tiles), K staged KST = 32 at a time (one tap's
// channel slice) through two LDS buffers.  The next
// stage's map values are held raw (fp32) in registers and rounded to fp16 as
// they are parked in LDS after the current stage's MFMAs, so their global
// latency overlaps the MFMAs.  Tile rows are KST halves (KST / 8 16-byte
// chunks), unpadded; chunk c of row r sits in slot c ^ csw(r), which spreads
// the rows of one ds_read_b128 pass over all 64 banks.
namespace {
constexpr int CT = 128;
template <int CH>
__device__ __forceinline__ int csw(int r) {
    return CH == 8 ? ((r & 7) ^ ((r >> 3) & 1)) : (((r >> 1) & 3) ^ ((r >> 3) & 1));
}
}
template <int TAPS, int KST>
__global__ __launch_bounds__(256, 2) void conv_f16_kernel(const float* __restrict__ x, const uint16_t* __restrict__ w,
                                                          const float* __restrict__ bias, int H, int W, int C, int N,
                                                          int gelu, float* __restrict__ y) {
    constexpr int CH = KST / 8, HC = CH / 2;  // chunks per row; chunks per loading thread
    __shared__ __attribute__((aligned(16))) _Float16 sA[2][CT * KST];
    __shared__ __attribute__((aligned(16))) _Float16 sB[2][CT * KST];
    const int M = H * W, K = TAPS == 9 ? 9 * C : C;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wv & 1, wn = wv >> 1;
    const int lr = lane & 31, g = lane >> 5;
    // XCD-aware tile order (each XCD a contiguous band of tiles)
    const int tiles_n = (N + CT - 1) / CT, tiles = ((M + CT - 1) / CT) * tiles_n;
    const int per_xcd = (tiles + 7) / 8;
    const int tl = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
    if (tl >= tiles) return;
    const int m0 = (tl / tiles_n) * CT, n0 = (tl % tiles_n) * CT;
    // loader: thread t fills row t/2 of both tiles, chunks HC*(t%2) .. +HC-1 of the stage
    const int lrow = tid >> 1, lc = HC * (tid & 1);
    const int am = m0 + lrow, bn = n0 + lrow;
    const int oy = am / W, ox = am - (am / W) * W;
    v4f ra[2 * HC];
    uint4 rb[HC];
    auto load = [&](int k0) {
        const int tap = TAPS == 9 ? k0 / C : 0, c0 = k0 - tap * C;
        const int iy = TAPS == 9 ? oy + tap / 3 - 1 : oy, ix = TAPS == 9 ? ox + tap % 3 - 1 : ox;
        const bool in = am < M && iy >= 0 && iy < H && ix >= 0 && ix < W;
        const float* src = x + ((int64_t)iy * W + ix) * C + c0 + 8 * lc;
#pragma unroll
        for (int h = 0; h < 2 * HC; ++h) ra[h] = in ? *reinterpret_cast<const v4f*>(src + 4 * h) : v4f{0, 0, 0, 0};
        const uint4* ws = reinterpret_cast<const uint4*>(w + (int64_t)bn * K + k0 + 8 * lc);
#pragma unroll
        for (int h = 0; h < HC; ++h) rb[h] = bn < N ? ws[h] : uint4{0, 0, 0, 0};
    };
    auto park = [&](int buf) {
#pragma unroll
        for (int h = 0; h < HC; ++h) {
            const int slot = ((lc + h) ^ csw<CH>(lrow)) << 3;
            const v4f a = ra[2 * h], b = ra[2 * h + 1];
            const uint4 q = {(uint32_t)f2h(a[0]) | ((uint32_t)f2h(a[1]) << 16), (uint32_t)f2h(a[2]) | ((uint32_t)f2h(a[3]) << 16),
                             (uint32_t)f2h(b[0]) | ((uint32_t)f2h(b[1]) << 16), (uint32_t)f2h(b[2]) | ((uint32_t)f2h(b[3]) << 16)};
            *reinterpret_cast<uint4*>(&sA[buf][lrow * KST + slot]) = q;
            *reinterpret_cast<uint4*>(&sB[buf][lrow * KST + slot]) = rb[h];
        }
    };
    const v16f zf = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
    v16f acc[2][2] = {{zf, zf}, {zf, zf}};
    const int nst = K / KST;
    load(0);
    park(0);
    __syncthreads();
    for (int s = 0; s < nst; ++s) {
        const int buf = s & 1;
        if (s + 1 < nst) load((s + 1) * KST);
#pragma unroll
        for (int kk = 0; kk < KST / 16; ++kk) {
            v8h a[2], b[2];
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const int ra_ = wm * 64 + i * 32 + lr, rb_ = wn * 64 + i * 32 + lr, c = 2 * kk + g;
                a[i] = *reinterpret_cast<const v8h*>(&sA[buf][ra_ * KST + ((c ^ csw<CH>(ra_)) << 3)]);
                b[i] = *reinterpret_cast<const v8h*>(&sB[buf][rb_ * KST + ((c ^ csw<CH>(rb_)) << 3)]);
            }
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[i], b[j], acc[i][j], 0, 0, 0);
        }
        if (s + 1 < nst) park(buf ^ 1);
        __syncthreads();
    }
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const int n = n0 + wn * 64 + j * 32 + lr;
        if (n >= N) continue;
        if (TAPS == 4) {
            const int Cout = N >> 2, t = n / Cout, co = n - t * Cout;
            const float bv = bias[co];
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const int m = m0 + wm * 64 + i * 32 + 8 * (r >> 2) + 4 * g + (r & 3);
                    if (m >= M) continue;
                    const int py = m / W, px = m - (m / W) * W;
                    const int64_t pix = (int64_t)(2 * py + (t >> 1)) * (2 * W) + 2 * px + (t & 1);
                    const float s = acc[i][j][r] + bv;
                    y[pix * Cout + co] = gelu ? gelu_erf(s) : s;
                }
        } else {
            const float bv = bias[n];
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const int m = m0 + wm * 64 + i * 32 + 8 * (r >> 2) + 4 * g + (r & 3);
                    if (m < M) y[(int64_t)m * N + n] = acc[i][j][r] + bv;
                }
        }
    }
}

// conv_f16_kernel's implicit GEMM over an fp16 map, both operands staged by LDS DMA
// (buffer_load ... lds) in 64-deep K stages, two slices of 32 channels of a tap: rows of 128 bytes
// per output pixel (zero by the buffer's range check outside the image or past M) and per weight
// row: whole lines, which the L2 feeds to the LDS at 35 TB/s, twice the rate of 64-byte rows.
// What bounds it: the 288 x 288 3x3 convolution of 256 channels takes 121 us (810 TFLOP/s; 152 with
// 32-deep stages, 32 x 32 x 16 MFMAs and offsets worked out per stage), 81 without its MFMAs and 78
// without its DMA. Three and five stages in flight (32-deep) or 256-row workgroups were no faster.
// The 72 x 72 conv-transpose 1024 -> 4 x 512 62 -> 40 us, 144 x 144 512 -> 4 x 256 64 -> 47 us.
// Two stage buffers, 64 KB: two workgroups per CU, four wavefronts of 64 x 64.
// v_mfma_f32_16x16x32_f16 with the operands swapped (A = weight rows, B = pixels): a lane holds
// four consecutive channels of one pixel, which leave in one store, and the chip runs this form
// faster at its power limit than 32 x 32 x 16 (1.89 against 1.64 PFLOP/s on random data).
// A slice's fragments are read while the slice before it is multiplied (two register sets). The
// barrier lies before a stage's second half: by then both halves are in registers everywhere, so
// the buffer takes stage s + 2, and stage s + 1 is readable.
// LDS rows of eight 16-byte chunks, chunk c of row r in slot c ^ (r >> 1 & 7): the 16 rows of a
// ds_read_b128 quarter (two to a line of the 64 banks) cover all of them.
namespace {
constexpr int CONV_OOB = 0x7ffffff0;  // a buffer offset past every operand the launcher admits
struct ConvStage {
    uint16_t A[CT * 64];  // map rows (pixels) x two slices of 32 channels
    uint16_t B[CT * 64];  // weight rows x 64 K
};
__device__ __forceinline__ int hswz(int r) { return (r >> 1) & 7; }
}  // namespace

// OH: the output is fp16 (the f32 result rounded, RNE), for a map only another of these kernels reads.
// PAIR: C % 64 == 0, so both slices of a stage lie in one tap: the lanes' map offsets change only
// with the tap, and a stage's DMA is eight loads with a scalar offset. (Working the offsets out
// for every stage took as many cycles as the stage's MFMAs.)
template <int TAPS, bool OH, bool PAIR>
__global__ __launch_bounds__(256, 2) void conv_f16_dma_kernel(const uint16_t* __restrict__ x, const uint16_t* __restrict__ w,
                                                              const float* __restrict__ bias, int H, int W, int C, int N,
                                                              int gelu, void* __restrict__ yv, int ksplit, int sps,
                                                              float* __restrict__ part) {
    constexpr int NL = 8;  // DMA instructions per wavefront and stage: 4 map, 4 weight
    __shared__ __attribute__((aligned(16))) ConvStage sb[2];
    const int M = H * W, K = TAPS == 9 ? 9 * C : C, cps = C / 32, nsl = K / 32;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wv >> 1, wn = wv & 1;
    const int r16 = lane & 15, kg = lane >> 4;
    // XCD-aware tile order (each XCD a contiguous band of tiles); with a K split (taps 1 and
    // 9) the split is the slowest index: slot (split, tile) runs slices [split * sps, + sps)
    const int tiles_n = (N + CT - 1) / CT, tiles = ((M + CT - 1) / CT) * tiles_n;
    const int TT = tiles * ksplit, per_xcd = (TT + 7) / 8;
    const int tls = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
    if (tls >= TT) return;
    const int split = tls / tiles, tl = tls - split * tiles;
    const int m0 = (tl / tiles_n) * CT, n0 = (tl % tiles_n) * CT;
    // this split's slices and stages (PAIR: stages begin at even slices, so a range of odd bounds has
    // a first or last stage of one slice)
    const int sl0 = split * sps, sl1 = min(nsl, sl0 + sps), nst = PAIR ? (sl1 + 1) / 2 - sl0 / 2 : (sl1 - sl0 + 1) / 2;

    // DMA instruction j moves rows 8 (4 wv + j) + lane / 8: LDS slot lane % 8, global chunk
    // slot ^ hswz(row), slice chunk / 4. Per lane the byte offset of its chunk within the slice at
    // the pixel itself and, for the 3x3, which taps lie inside
    const v4i xr = make_rsrc(x, (int64_t)M * C * 2), wr = make_rsrc(w, (int64_t)N * K * 2);
    int xoff[4], tmask[4], woff[4], half[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int row = 8 * (4 * wv + j) + (lane >> 3), p = m0 + row, n = n0 + row;
        const int c = (lane & 7) ^ hswz(row), py = p / W, px = p - py * W;
        half[j] = c >> 2;
        xoff[j] = p < M ? p * C * 2 + ((c & 3) << 4) : CONV_OOB;
        woff[j] = n < N ? n * K * 2 + (c << 4) : CONV_OOB;
        tmask[j] = 0;
        if (TAPS == 9 && p < M)
            for (int t = 0; t < 9; ++t) {
                const int iy = py + t / 3 - 1, ix = px + t % 3 - 1;
                tmask[j] |= (iy >= 0 && iy < H && ix >= 0 && ix < W) << t;
            }
    }
    const uint32_t lb[2] = {(uint32_t)__builtin_amdgcn_readfirstlane(lds_addr(&sb[0])),
                            (uint32_t)__builtin_amdgcn_readfirstlane(lds_addr(&sb[1]))};
    // the next stage to load, in order: its first slice, that slice's tap and channel slice
    int dsl = PAIR ? sl0 & ~1 : sl0, dtap = TAPS == 9 ? dsl / cps : 0, dcs = dsl - dtap * cps;
    int voff[4];  // PAIR: the lanes' map offsets of tap dtap
    auto at_tap = [&]() __attribute__((always_inline)) {
        const int off = TAPS == 9 ? ((dtap / 3 - 1) * W + dtap % 3 - 1) * C * 2 : 0;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const bool in = TAPS != 9 || ((tmask[j] >> dtap) & 1);
            voff[j] = in && xoff[j] != CONV_OOB ? xoff[j] + off + 64 * half[j] : CONV_OOB;
        }
    };
    if (PAIR) at_tap();
    auto dma = [&](uint32_t base) __attribute__((always_inline)) {
        if (PAIR) {
            if (dsl + 1 >= sl1) {  // the range ends within the stage: its second slice reads zero
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    if (half[j]) voff[j] = woff[j] = CONV_OOB;
            }
#pragma unroll
            for (int j = 0; j < 4; ++j)
                dma_b128_so(xr, base + (uint32_t)offsetof(ConvStage, A) + 1024u * (4 * wv + j), voff[j], dcs * 64);
#pragma unroll
            for (int j = 0; j < 4; ++j)
                dma_b128_so(wr, base + (uint32_t)offsetof(ConvStage, B) + 1024u * (4 * wv + j), woff[j], dsl * 64);
            dsl += 2;
            dcs += 2;
            if (TAPS == 9 && dcs == cps) {
                dcs = 0;
                ++dtap;
                at_tap();
            }
            return;
        }
        // byte offset of each of the two slices' map rows from the pixel's own row
        int tap[2], off[2];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            tap[h] = dtap;
            off[h] = (TAPS == 9 ? ((dtap / 3 - 1) * W + dtap % 3 - 1) * C * 2 : 0) + dcs * 64;
            if (TAPS == 9 && ++dcs == cps) {
                dcs = 0;
                ++dtap;
            } else if (TAPS != 9) {
                ++dcs;
            }
        }
        const bool odd = dsl + 1 >= sl1;  // no second slice (the last stage of an odd count)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const bool in = !(odd && half[j]) && (TAPS != 9 || ((tmask[j] >> (half[j] ? tap[1] : tap[0])) & 1));
            const int o = in && xoff[j] != CONV_OOB ? xoff[j] + (half[j] ? off[1] : off[0]) : CONV_OOB;
            dma_b128_so(xr, base + (uint32_t)offsetof(ConvStage, A) + 1024u * (4 * wv + j), o, 0);
        }
#pragma unroll
        for (int j = 0; j < 4; ++j)
            dma_b128_so(wr, base + (uint32_t)offsetof(ConvStage, B) + 1024u * (4 * wv + j), odd && half[j] ? CONV_OOB : woff[j],
                        dsl * 64);
        dsl += 2;
    };

    v4f acc[4][4];  // [pixel tile][channel tile]
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = v4f{0, 0, 0, 0};
    struct Frag {
        v8h a[4], b[4];
    };
    auto read = [&](Frag& f, const ConvStage& st, int h) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int ra = 64 * wm + 16 * i + r16, rb = 64 * wn + 16 * i + r16;
            f.a[i] = *reinterpret_cast<const v8h*>(&st.A[ra * 64 + (((4 * h + kg) ^ hswz(ra)) << 3)]);
            f.b[i] = *reinterpret_cast<const v8h*>(&st.B[rb * 64 + (((4 * h + kg) ^ hswz(rb)) << 3)]);
        }
    };
    auto mul = [&](const Frag& f) __attribute__((always_inline)) {
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(f.b[j], f.a[i], acc[i][j], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
    };

    if (PAIR && (sl0 & 1)) {  // the range begins within its first stage, whose first slice reads zero
        int w0[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            w0[j] = woff[j];
            if (!half[j]) voff[j] = woff[j] = CONV_OOB;
        }
        dma(lb[0]);
#pragma unroll
        for (int j = 0; j < 4; ++j) woff[j] = w0[j];
        at_tap();
    } else {
        dma(lb[0]);
    }
    if (nst > 1) {
        dma(lb[1]);
        wait_vmcnt<NL>();
    } else {
        wait_vmcnt<0>();
    }
    __syncthreads();
    Frag f0, f1;
    read(f0, sb[0], 0);
    for (int s = 0; s < nst; ++s) {
        read(f1, sb[s & 1], 1);
        mul(f0);
        __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): both halves are in registers (a wait the compiler sees)
        if (s + 1 < nst) {
            wait_vmcnt<0>();  // stage s + 1 has landed
            asm volatile("s_barrier" ::: "memory");
            if (s + 2 < nst) dma(lb[s & 1]);
            read(f0, sb[(s + 1) & 1], 0);
        }
        mul(f1);
    }

    if (TAPS != 4 && ksplit > 1) {  // this split's partial sums, no bias: part [split][M][N] (N % 4 == 0)
        float* P = part + (int64_t)split * M * N;
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int m = m0 + 64 * wm + 16 * i + r16, n = n0 + 64 * wn + 16 * j + 4 * kg;
                if (m < M && n < N) *reinterpret_cast<v4f*>(&P[(int64_t)m * N + n]) = acc[i][j];
            }
        return;
    }
    // four channels n .. n + 3 of one pixel per lane and tile: one store where the rows allow it
    // (they lie in one tap of a conv-transpose: Cout % 4 == 0)
    const int Cout = TAPS == 4 ? N >> 2 : N;
    const bool v4 = Cout % 4 == 0 && (reinterpret_cast<uintptr_t>(yv) & (OH ? 7 : 15)) == 0;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int n = n0 + 64 * wn + 16 * j + 4 * kg;
        if (n >= N) continue;
        const int t = TAPS == 4 ? n / Cout : 0, co = n - t * Cout;
        float bv[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) bv[r] = n + r < N ? bias[co + r] : 0.0f;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int m = m0 + 64 * wm + 16 * i + r16;
            if (m >= M) continue;
            int64_t pix = m;
            if (TAPS == 4) {
                const int qy = m / W, qx = m - (m / W) * W;
                pix = (int64_t)(2 * qy + (t >> 1)) * (2 * W) + 2 * qx + (t & 1);
            }
            v4f o;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const float sv = acc[i][j][r] + bv[r];
                o[r] = TAPS == 4 && gelu ? gelu_erf(sv) : sv;
            }
            const int64_t at = pix * Cout + co;
            if (v4) {
                if (OH)
                    *reinterpret_cast<uint2*>(static_cast<uint16_t*>(yv) + at) =
                        make_uint2((uint32_t)f2h(o[0]) | ((uint32_t)f2h(o[1]) << 16), (uint32_t)f2h(o[2]) | ((uint32_t)f2h(o[3]) << 16));
                else *reinterpret_cast<v4f*>(static_cast<float*>(yv) + at) = o;
            } else {
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    if (n + r < N) {
                        if (OH) static_cast<uint16_t*>(yv)[at + r] = f2h(o[r]);
                        else static_cast<float*>(yv)[at + r] = o[r];
                    }
            }
        }
    }
}

// The 1x1 and the conv-transpose over an F32 map: the same GEMM with the map staged as it is (128
// bytes per pixel and 32-deep stage) and rounded to fp16 (RNE, f2h) as the fragments are read, so no
// pass over the map goes before it: 1x1, 288 x 288, 256 -> 256 channels 36 us, against 25 for that
// pass and 30 for conv_f16_dma_kernel. The same operands, products and order over K: the same bits.
// Map rows of 8 chunks of 16 bytes, chunk c of row r in slot c ^ (r >> 1 & 7); weight rows of
// four, csw<4>.
namespace {
struct Map32Stage {
    float A[CT * 32];     // 128 map rows x 32 channels, fp32
    uint16_t B[CT * 32];  // 128 weight rows x 32 K, fp16
};
}  // namespace
template <int TAPS>
__global__ __launch_bounds__(256, 3) void conv_f32map_kernel(const float* __restrict__ x, const uint16_t* __restrict__ w,
                                                             const float* __restrict__ bias, int H, int W, int C, int N, int gelu,
                                                             float* __restrict__ y, int ksplit, int sps,
                                                             float* __restrict__ part) {
    __shared__ __attribute__((aligned(16))) Map32Stage sb[2];
    const int M = H * W;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wv & 1, wn = wv >> 1;
    const int lr = lane & 31, g = lane >> 5;
    const int tiles_n = (N + CT - 1) / CT, tiles = ((M + CT - 1) / CT) * tiles_n;
    const int TT = tiles * ksplit, per_xcd = (TT + 7) / 8;
    const int tls = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
    if (tls >= TT) return;
    const int split = tls / tiles, tl = tls - split * tiles;
    const int m0 = (tl / tiles_n) * CT, n0 = (tl % tiles_n) * CT;
    const int s0 = split * sps, nst = min(C / 32 - s0, sps);
    // map DMA instruction j of wavefront wv: rows 8 (4 wv + j) + lane / 8; weights: rows
    // 16 (2 wv + j) + lane / 4; the stage is the loads' scalar offset
    const v4i xr = make_rsrc(x, (int64_t)M * C * 4), wr = make_rsrc(w, (int64_t)N * C * 2);
    int xoff[4], woff[2];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int row = 8 * (4 * wv + j) + (lane >> 3), p = m0 + row;
        xoff[j] = p < M ? p * C * 4 + (((lane & 7) ^ hswz(row)) << 4) : CONV_OOB;
    }
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const int row = 16 * (2 * wv + j) + (lane >> 2), n = n0 + row;
        woff[j] = n < N ? n * C * 2 + (((lane & 3) ^ csw<4>(row)) << 4) : CONV_OOB;
    }
    const uint32_t lb[2] = {(uint32_t)__builtin_amdgcn_readfirstlane(lds_addr(&sb[0])),
                            (uint32_t)__builtin_amdgcn_readfirstlane(lds_addr(&sb[1]))};
    auto dma = [&](int s, uint32_t base) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < 4; ++j)
            dma_b128_so(xr, base + (uint32_t)offsetof(Map32Stage, A) + 1024u * (4 * wv + j), xoff[j], s * 128);
#pragma unroll
        for (int j = 0; j < 2; ++j)
            dma_b128_so(wr, base + (uint32_t)offsetof(Map32Stage, B) + 1024u * (2 * wv + j), woff[j], s * 64);
    };
    const v16f zf = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
    v16f acc[2][2] = {{zf, zf}, {zf, zf}};
    auto compute = [&](const Map32Stage& b) __attribute__((always_inline)) {
#pragma unroll
        for (int kk = 0; kk < 2; ++kk) {
            v8h a[2], bf[2];
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const int ra = wm * 64 + i * 32 + lr, rb = wn * 64 + i * 32 + lr, c = 4 * kk + 2 * g;
                const v4f lo = *reinterpret_cast<const v4f*>(&b.A[ra * 32 + ((c ^ hswz(ra)) << 2)]);
                const v4f hi = *reinterpret_cast<const v4f*>(&b.A[ra * 32 + (((c + 1) ^ hswz(ra)) << 2)]);
                const uint4 q = {(uint32_t)f2h(lo[0]) | ((uint32_t)f2h(lo[1]) << 16), (uint32_t)f2h(lo[2]) | ((uint32_t)f2h(lo[3]) << 16),
                                 (uint32_t)f2h(hi[0]) | ((uint32_t)f2h(hi[1]) << 16), (uint32_t)f2h(hi[2]) | ((uint32_t)f2h(hi[3]) << 16)};
                a[i] = __builtin_bit_cast(v8h, q);
                bf[i] = *reinterpret_cast<const v8h*>(&b.B[rb * 32 + (((2 * kk + g) ^ csw<4>(rb)) << 3)]);
            }
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[i], bf[j], acc[i][j], 0, 0, 0);
        }
    };
    dma(s0, lb[0]);
    if (nst > 1) {
        dma(s0 + 1, lb[1]);
        wait_vmcnt<6>();
    } else {
        wait_vmcnt<0>();
    }
    __syncthreads();
    for (int s = 0; s < nst; ++s) {
        compute(sb[s & 1]);
        if (s + 1 < nst) {
            wait_vmcnt<0>();  // stage s + 1 has landed
            asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");  // and stage s's buffer is read
            if (s + 2 < nst) dma(s0 + s + 2, lb[s & 1]);
        }
    }
    if (TAPS == 4) {  // + bias (+ GELU), each tap to its pixel of the 2x map
        const int Cout = N >> 2;
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int n = n0 + wn * 64 + j * 32 + lr;
            if (n >= N) continue;
            const int t = n / Cout, co = n - t * Cout;
            const float bv = bias[co];
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const int m = m0 + wm * 64 + i * 32 + 8 * (r >> 2) + 4 * g + (r & 3);
                    if (m >= M) continue;
                    const int qy = m / W, qx = m - qy * W;
                    const int64_t pix = (int64_t)(2 * qy + (t >> 1)) * (2 * W) + 2 * qx + (t & 1);
                    const float v = acc[i][j][r] + bv;
                    y[pix * Cout + co] = gelu ? gelu_erf(v) : v;
                }
        }
        return;
    }
    // a split's partial sums go without bias, in a branch of their own: its load, also where it is
    // only skipped, makes a store wait for the one before (9 x 9, 256 -> 52 channels 8.8 us, 13.9 so)
    auto store = [&](float* D, bool plain, const float (&bv)[2]) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int n = n0 + wn * 64 + j * 32 + lr;
            if (n >= N) continue;
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const int m = m0 + wm * 64 + i * 32 + 8 * (r >> 2) + 4 * g + (r & 3);
                    if (m < M) D[(int64_t)m * N + n] = plain ? acc[i][j][r] : acc[i][j][r] + bv[j];
                }
        }
    };
    if (ksplit > 1) {
        store(part + (int64_t)split * M * N, true, {0.0f, 0.0f});
        return;
    }
    float bv[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) bv[j] = n0 + wn * 64 + j * 32 + lr < N ? bias[n0 + wn * 64 + j * 32 + lr] : 0.0f;
    store(y, false, bv);
}

// y[r][c] += b[c], four channels per thread (C % 4 == 0)
__global__ __launch_bounds__(256) void bias_rows_kernel(float* __restrict__ y, const float* __restrict__ b, int64_t rows,
                                                        int C) {
    const int c4 = C / 4;
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= rows * c4) return;
    const int c = (int)(i % c4) * 4;
    v4f v = *reinterpret_cast<const v4f*>(&y[i * 4]);
    const v4f bb = *reinterpret_cast<const v4f*>(&b[c]);
    *reinterpret_cast<v4f*>(&y[i * 4]) = v + bb;
}

// ggml_pool_2d MAX, 2x2 window, stride 2, no padding: four channels per thread
// (F16: an fp16 map in and out)
template <bool F16>
__global__ __launch_bounds__(256) void maxpool2_kernel(const void* __restrict__ x, int H, int W, int C, void* __restrict__ y) {
    const int c4 = C / 4, H2 = H / 2, W2 = W / 2;
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (int64_t)H2 * W2 * c4) return;
    const int c = (int)(i % c4) * 4;
    const int64_t q = i / c4;
    const int py = (int)(q / W2), px = (int)(q % W2);
    const int64_t at = ((int64_t)(2 * py) * W + 2 * px) * C + c;
    auto load = [&](int64_t o) -> v4f {
        if (!F16) return *reinterpret_cast<const v4f*>(static_cast<const float*>(x) + o);
        const uint2 u = *reinterpret_cast<const uint2*>(static_cast<const uint16_t*>(x) + o);
        return v4f{h2f(u.x & 0xffff), h2f(u.x >> 16), h2f(u.y & 0xffff), h2f(u.y >> 16)};
    };
    const v4f a = load(at), b = load(at + C), d = load(at + (int64_t)W * C), e = load(at + (int64_t)W * C + C);
    v4f m;
#pragma unroll
    for (int j = 0; j < 4; ++j) m[j] = fmaxf(fmaxf(a[j], b[j]), fmaxf(d[j], e[j]));
    if (F16)
        *reinterpret_cast<uint2*>(static_cast<uint16_t*>(y) + q * C + c) =
            make_uint2((uint32_t)f2h(m[0]) | ((uint32_t)f2h(m[1]) << 16), (uint32_t)f2h(m[2]) | ((uint32_t)f2h(m[3]) << 16));
    else *reinterpret_cast<v4f*>(static_cast<float*>(y) + q * C + c) = m;
}

hipError_t launch_deconv_pack(const void* w, int wtype, int Cin, int Cout, uint16_t* out, hipStream_t st) {
    const int64_t n = deconv_pack_blocks(Cin, Cout);
    if (n > 0) deconv_pack_kernel<<<(unsigned)n, 1024, 0, st>>>(w, wtype, Cin, Cout, out);
    return hipGetLastError();
}

hipError_t launch_neck_pack(const NeckPack* jobs, int n, hipStream_t st) {
    if (n <= 0) return hipSuccess;
    if (n > NECK_PACKS) return hipErrorInvalidValue;
    NeckPacks p{};
    int64_t end = 0;
    for (int i = 0; i < n; ++i) {
        const NeckPack& j = jobs[i];
        const int64_t K = (int64_t)j.k * j.k * j.Cin;
        const int64_t items = j.type == T_F16 ? K * j.Cout : (K + 31) / 32 * 4 * j.Cout;
        end += j.k == 2 ? deconv_pack_blocks(j.Cin, j.Cout) : (items + 255) / 256;
        p.j[i] = j;
        p.end[i] = (unsigned)end;
    }
    p.n = n;
    if (end > 0x7fffffff) return hipErrorInvalidValue;
    neck_pack_kernel<<<(unsigned)end, 256, 0, st>>>(p);
    return hipGetLastError();
}

hipError_t launch_deconv_scatter(const float* D, const float* b, int H, int W, int Cout, bool gelu, float* y,
                                 hipStream_t st) {
    if (Cout % 4 != 0) return hipErrorInvalidValue;
    const int64_t n = 4LL * H * W * (Cout / 4);
    if (n > 0) deconv_scatter_kernel<<<nblk(n), 256, 0, st>>>(D, b, H, W, Cout, gelu ? 1 : 0, y);
    return hipGetLastError();
}

hipError_t launch_im2col3x3(const float* x, int H, int W, int C, bool f16, void* cols, hipStream_t st) {
    const int64_t n = (int64_t)H * W * 9 * C;
    if (n <= 0) return hipSuccess;
    if (f16) im2col3x3_kernel<true><<<nblk(n), 256, 0, st>>>(x, H, W, C, cols);
    else im2col3x3_kernel<false><<<nblk(n), 256, 0, st>>>(x, H, W, C, cols);
    return hipGetLastError();
}

hipError_t launch_conv3x3_pack(const float* w, int Cin, int Cout, float* out, hipStream_t st) {
    const int64_t n = 9LL * Cin * Cout;
    if (n > 0) conv3x3_pack_kernel<<<nblk(n), 256, 0, st>>>(w, Cin, Cout, out);
    return hipGetLastError();
}

hipError_t launch_conv3x3_pack_f16(const uint16_t* w, int Cin, int Cout, uint16_t* out, hipStream_t st) {
    const int64_t n = 9LL * Cin * Cout;
    if (n > 0) conv3x3_pack_f16_kernel<<<nblk(n), 256, 0, st>>>(w, Cin, Cout, out);
    return hipGetLastError();
}

// operands the DMA kernel's 32-bit buffer offsets reach (with the out-of-range offset above)
bool conv_f16_dma_fits(int taps, int64_t M, int64_t C, int64_t N) {
    return M * C * 4 < CONV_OOB - 4096 && N * (taps == 9 ? 9 : 1) * C * 2 < CONV_OOB - 4096;
}
namespace {
// K split of the DMA kernel (taps 1 and 9), in 32-deep slices: grids below one tile per CU; a
// slice of a tile counts 0.9 us.
int conv_f16_ksplit(int taps, int64_t M, int64_t C, int64_t N, int64_t* sps) {
    const int64_t nsl = (taps == 9 ? 9 : 1) * C / 32;
    *sps = nsl;
    if (taps == 4 || !conv_f16_dma_fits(taps, M, C, N)) return 1;
    const int64_t tiles = ((M + CT - 1) / CT) * ((N + CT - 1) / CT);
    const int S = gemm_ksplit(tiles, 256, M, N, nsl, 0.9);
    *sps = (nsl + S - 1) / S;
    return S;
}
}  // namespace

size_t conv_f16_part_bytes(int taps, int64_t M, int64_t C, int64_t N) {
    int64_t sps;
    const int S = conv_f16_ksplit(taps, M, C, N, &sps);
    return S > 1 ? (size_t)S * (size_t)M * (size_t)N * 4 : 0;
}

hipError_t launch_conv_f16(int taps, const void* x, bool x16, const uint16_t* w, const float* bias, int H, int W, int C,
                           int N, bool gelu, void* y, bool y16, hipStream_t st, float* part, size_t part_bytes) {
    if ((taps != 1 && taps != 4 && taps != 9) || C % 32 != 0 || (reinterpret_cast<uintptr_t>(x) & 15) ||
        (reinterpret_cast<uintptr_t>(w) & 15) || (taps == 4 && N % 16 != 0))
        return hipErrorInvalidValue;
    const int64_t M = (int64_t)H * W;
    if (M <= 0 || N <= 0) return hipSuccess;
    const int tiles = (int)(((M + CT - 1) / CT) * ((N + CT - 1) / CT));
    const unsigned grid = (unsigned)((tiles + 7) / 8 * 8);
    const int gl = gelu ? 1 : 0;
    if (x16 && !conv_f16_dma_fits(taps, M, C, N)) return hipErrorInvalidValue;
    const bool map32 = taps != 9 && !x16 && !y16 && conv_f16_dma_fits(taps, M, C, N);
    if (x16 || map32) {
        // the K split, when the caller gave room for its partial sums
        // (the reduce stores float4 rows: y and part on 16 bytes; N % 4 == 0 in the split choice)
        const bool a16 = ((reinterpret_cast<uintptr_t>(y) | reinterpret_cast<uintptr_t>(part) |
                           reinterpret_cast<uintptr_t>(bias)) & 15) == 0;
        int64_t sps64;
        int S = conv_f16_ksplit(taps, M, C, N, &sps64);
        if (!part || !a16 || (size_t)S * (size_t)M * (size_t)N * 4 > part_bytes) S = 1;
        const int sps = S > 1 ? (int)sps64 : (taps == 9 ? 9 : 1) * C / 32;
        const unsigned gs = (unsigned)((tiles * S + 7) / 8 * 8);
        const uint16_t* xh = static_cast<const uint16_t*>(x);
        const bool pair = C % 64 == 0;
        auto go = [&](auto even, auto any) {
            if (pair) even<<<gs, 256, 0, st>>>(xh, w, bias, H, W, C, N, gl, y, S, sps, part);
            else any<<<gs, 256, 0, st>>>(xh, w, bias, H, W, C, N, gl, y, S, sps, part);
        };
        const float* xf = static_cast<const float*>(x);
        float* yf = static_cast<float*>(y);
        if (map32 && taps == 1) conv_f32map_kernel<1><<<gs, 256, 0, st>>>(xf, w, bias, H, W, C, N, 0, yf, S, sps, part);
        else if (map32) conv_f32map_kernel<4><<<gs, 256, 0, st>>>(xf, w, bias, H, W, C, N, gl, yf, S, sps, part);
        else if (taps == 9 && !y16) go(conv_f16_dma_kernel<9, false, true>, conv_f16_dma_kernel<9, false, false>);
        else if (taps == 4 && y16) go(conv_f16_dma_kernel<4, true, true>, conv_f16_dma_kernel<4, true, false>);
        else if (taps == 4) go(conv_f16_dma_kernel<4, false, true>, conv_f16_dma_kernel<4, false, false>);
        else if (taps == 1 && y16) go(conv_f16_dma_kernel<1, true, true>, conv_f16_dma_kernel<1, true, false>);
        else return hipErrorInvalidValue;
        const hipError_t e = hipGetLastError();
        if (S == 1 || e != hipSuccess) return e;
        return launch_split_reduce(part, S, (int)M, N, bias, static_cast<float*>(y), (y16 ? 2LL : 4LL) * N, st, y16);
    }
    // K step 32: 64-deep steps, staged through registers here, measured slower
    if (y16) return hipErrorInvalidValue;  // fp16 maps: the DMA kernel only
    const float* xf = static_cast<const float*>(x);
    float* yf = static_cast<float*>(y);
    if (taps == 9)
        conv_f16_kernel<9, 32><<<grid, 256, 0, st>>>(xf, w, bias, H, W, C, N, gl, yf);
    else if (taps == 4)
        conv_f16_kernel<4, 32><<<grid, 256, 0, st>>>(xf, w, bias, H, W, C, N, gl, yf);
    else
        conv_f16_kernel<1, 32><<<grid, 256, 0, st>>>(xf, w, bias, H, W, C, N, gl, yf);
    return hipGetLastError();
}

hipError_t launch_bias_rows(float* y, const float* b, int64_t rows, int C, hipStream_t st) {
    if (C % 4 != 0) return hipErrorInvalidValue;
    const int64_t n = rows * (C / 4);
    if (n > 0) bias_rows_kernel<<<nblk(n), 256, 0, st>>>(y, b, rows, C);
    return hipGetLastError();
}

hipError_t launch_maxpool2(const void* x, int H, int W, int C, void* y, hipStream_t st, bool f16) {
    if (C % 4 != 0) return hipErrorInvalidValue;
    const int64_t n = (int64_t)(H / 2) * (W / 2) * (C / 4);
    if (n > 0 && f16) maxpool2_kernel<true><<<nblk(n), 256, 0, st>>>(x, H, W, C, y);
    else if (n > 0) maxpool2_kernel<false><<<nblk(n), 256, 0, st>>>(x, H, W, C, y);
    return hipGetLastError();
}

}  // namespace mi355

// Weight repacks as device functions, one item (what one thread writes) per call: each has a kernel
// of its own, and the neck makes those of all its kernels in one launch.
#pragma once
#include "common.cuh"
#include "kernels.h"

namespace mi355 {

typedef __bf16 v2b __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint32_t pk_bf16(float a, float b) {
    const v2f v = {a, b};
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, v2b));
}

// The factor, exact in fp32, by which both operands of the split GEMM are multiplied before they are
// split: the lowest plane of the smallest fp32 values is then a normal bf16.
constexpr float SPLIT_UP = 16777216.0f;

// item i of the planes of SPLIT_UP times the rows of an F32 kernel [N][K] (taps == 9: a 3x3 one
// [N][C][3][3] read in (tap, channel) order) -> [N][KP / 32][3][32] bf16, zero past K: eight
// consecutive K
__device__ __forceinline__ void split_w_item(int64_t i, const float* __restrict__ w, int taps, int N, int K, int KP,
                                             uint16_t* __restrict__ out) {
    const int k8 = KP / 8;
    if (i >= (int64_t)N * k8) return;
    const int n = (int)(i / k8), k0 = (int)(i - (int64_t)n * k8) * 8;
    const int C = K / taps;
    uint16_t h[8], m[8], l[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        const int k = k0 + j;
        float x = 0.0f;
        if (k < K) {
            const int64_t e = taps == 1 ? k : (int64_t)(k % C) * taps + k / C;
            x = w[(int64_t)n * K + e];
        }
        x *= SPLIT_UP;
        const uint32_t a = pk_bf16(x, 0.0f) & 0xffffu;
        const float r = x - __uint_as_float(a << 16);
        const uint32_t b = pk_bf16(r, 0.0f) & 0xffffu;
        h[j] = (uint16_t)a;
        m[j] = (uint16_t)b;
        l[j] = (uint16_t)(pk_bf16(r - __uint_as_float(b << 16), 0.0f) & 0xffffu);
    }
    uint16_t* o = out + (int64_t)n * KP * 3 + (k0 >> 5) * 96 + (k0 & 31);
    auto put = [&](uint16_t* d, const uint16_t (&v)[8]) {
        *reinterpret_cast<uint4*>(d) = make_uint4(v[0] | (uint32_t)v[1] << 16, v[2] | (uint32_t)v[3] << 16,
                                                  v[4] | (uint32_t)v[5] << 16, v[6] | (uint32_t)v[7] << 16);
    };
    put(o, h);
    put(o + 32, m);
    put(o + 64, l);
}

// A conv-transpose kernel [kW=2, kH=2, Cout, Cin] (memory [ci][co][kh][kw]), F32 or F16, -> F16
// MUL_MAT weight rows [4*Cout][Cin], row n = (kh*2 + kw)*Cout + co. The F32 -> F16 cast rounds to
// nearest even, as ggml_cast does (sam3_conv_transpose_weight, sam3.cpp:1087-1090). Block b of WV
// wavefronts transposes 64 channels ci by 64 elements (co, tap) through LDS (8 KB): whole segments
// are read and written. One thread per element read 64 lines per wavefront, each line again for
// every other element of it. t: PACK_LDS halves.
constexpr int PACK_LDS = 64 * 66;
__host__ __device__ inline int64_t deconv_pack_blocks(int Cin, int Cout) { return (int64_t)((Cin + 63) / 64) * ((4LL * Cout + 63) / 64); }
template <int WV>
__device__ __forceinline__ void deconv_pack_block(int64_t b, const void* __restrict__ w, int wtype, int Cin, int Cout,
                                                  uint16_t* __restrict__ out, uint16_t* t) {
    constexpr int NR = 64 / WV;  // rows per wavefront
    const int nci = (Cin + 63) / 64, lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int ci0 = (int)(b % nci) * 64, e0 = (int)(b / nci) * 64, ne = 4 * Cout;
    uint16_t v[NR];
#pragma unroll
    for (int k = 0; k < NR; ++k) {
        const int ci = ci0 + WV * k + wv, e = e0 + lane;
        const int64_t src = (int64_t)ci * ne + e;
        v[k] = 0;
        if (ci < Cin && e < ne) v[k] = wtype == T_F16 ? static_cast<const uint16_t*>(w)[src] : f2h(static_cast<const float*>(w)[src]);
    }
#pragma unroll
    for (int k = 0; k < NR; ++k) t[66 * lane + WV * k + wv] = v[k];
    __syncthreads();
#pragma unroll
    for (int k = 0; k < NR; ++k) {
        const int r = WV * k + wv, e = e0 + r, ci = ci0 + lane;  // e = co * 4 + tap
        if (ci < Cin && e < ne) out[((int64_t)(e & 3) * Cout + (e >> 2)) * Cin + ci] = t[66 * r + lane];
    }
}

// item i of an F16 3x3 kernel [Cout][Cin][3][3] -> rows in (tap, channel) order: one element
__device__ __forceinline__ void conv3x3_pack_f16_item(int64_t i, const uint16_t* __restrict__ w, int Cin, int Cout,
                                                      uint16_t* __restrict__ out) {
    if (i >= 9LL * Cin * Cout) return;
    const int ci = (int)(i % Cin);
    const int64_t r = i / Cin;
    const int tap = (int)(r % 9), co = (int)(r / 9);
    out[i] = w[((int64_t)co * Cin + ci) * 9 + tap];
}

}  // namespace mi355

// Products of a few rows with a large matrix -- gfx950.
//
//   trimkv_linear_rows   out[m][n] = sum_k x[m][k] w[n][k] (+ bias[n]), up to 64 rows x (a decode step's tokens), w in nn.Linear's
//                        layout, 16-bit operands, fp32 sums, one rounding
//
// The launch is bound by the stream of weights: every byte of w is read once and used for at most 64 rows.
#include "common.hip.h"

namespace trimkv {

typedef __bf16 lr_bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 lr_f16x8 __attribute__((ext_vector_type(8)));
typedef float lr_f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t lr_u32x4 __attribute__((ext_vector_type(4)));

struct LinearRowsArgs {
    const uint16_t* x; int64_t xs;
    const uint16_t* w; int64_t ws;
    const uint16_t* bias;
    uint16_t* out; int64_t os;
    int m, n, k;
};

template <bool F16>
__device__ __forceinline__ lr_f32x4 lr_mfma(lr_u32x4 a, lr_u32x4 b, lr_f32x4 c) {
    if constexpr (F16) return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(lr_f16x8, a), __builtin_bit_cast(lr_f16x8, b), c, 0, 0, 0);
    else return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(lr_bf16x8, a), __builtin_bit_cast(lr_bf16x8, b), c, 0, 0, 0);
}
template <bool F16> __device__ __forceinline__ float lr_load(uint16_t b) { return F16 ? f16_bits_to_f32(b) : bf16_bits_to_f32(b); }
template <bool F16> __device__ __forceinline__ uint16_t lr_bits(float f) { return F16 ? f32_to_f16_bits(f) : f32_to_bf16_bits(f); }

// A workgroup computes 16 NT outputs of all 16 MT rows; its KS wavefronts take turns on the 64-element steps of k (so that
// together they read runs of KS x 128 bytes of every row of w) and add their sums up in LDS.  A wavefront keeps one to two
// groups of U steps in flight, straight into operand registers: lane l holds row l % 16, elements 8 (l / 16) .. + 7 of 32.
template <bool F16, int MT, int NT, int KS, int U>
__global__ __launch_bounds__(KS * 64) void linear_rows_kernel(LinearRowsArgs a) {
    __shared__ lr_f32x4 part[KS][NT * MT][64];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), r = lane & 15, g = lane >> 4;
    const int n0 = blockIdx.x * NT * 16, steps = a.k >> 6;
    const uint16_t* wp[NT]; const uint16_t* xp[MT];
#pragma unroll
    for (int t = 0; t < NT; ++t) wp[t] = a.w + (int64_t)min(n0 + 16 * t + r, a.n - 1) * a.ws + 8 * g;
#pragma unroll
    for (int t = 0; t < MT; ++t) xp[t] = a.x + (int64_t)min(16 * t + r, a.m - 1) * a.xs + 8 * g;
    lr_f32x4 acc[NT][MT];
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int y = 0; y < MT; ++y) acc[t][y] = lr_f32x4{0.f, 0.f, 0.f, 0.f};
    lr_u32x4 wf[2][U][2][NT], xf[2][U][2][MT];
    auto request = [&](int s0, int b) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int at = min(s0 + u * KS, steps - 1) * 64;      // past the end: re-read, never used
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int t = 0; t < NT; ++t) wf[b][u][h][t] = __builtin_nontemporal_load((const lr_u32x4*)(wp[t] + at + 32 * h));
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int t = 0; t < MT; ++t) xf[b][u][h][t] = *(const lr_u32x4*)(xp[t] + at + 32 * h);
        }
    };
    auto multiply = [&](int s0, int b) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (s0 + u * KS >= steps) break;
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int t = 0; t < NT; ++t)
#pragma unroll
                    for (int y = 0; y < MT; ++y) acc[t][y] = lr_mfma<F16>(wf[b][u][h][t], xf[b][u][h][y], acc[t][y]);
        }
    };
    constexpr int STEP = KS * U;
    request(wave, 0);
    for (int s = wave; s < steps; s += 2 * STEP) {
        request(s + STEP, 1);
        __builtin_amdgcn_sched_barrier(0);
        multiply(s, 0);
        __builtin_amdgcn_sched_barrier(0);
        request(s + 2 * STEP, 0);
        __builtin_amdgcn_sched_barrier(0);
        multiply(s + STEP, 1);
        __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int y = 0; y < MT; ++y) part[wave][t * MT + y][lane] = acc[t][y];
    __syncthreads();
    // a lane of tile (t, y) holds outputs n0 + 16 t + 4 g .. + 3 of row 16 y + r
    for (int i = threadIdx.x; i < NT * MT * 64; i += KS * 64) {
        const int tile = i >> 6, l = i & 63, m = (tile % MT) * 16 + (l & 15), n = n0 + (tile / MT) * 16 + (l >> 4) * 4;
        lr_f32x4 f = part[0][tile][l];
#pragma unroll
        for (int w = 1; w < KS; ++w) f += part[w][tile][l];
        if (m >= a.m) continue;
        uint16_t* o = a.out + (int64_t)m * a.os + n;
        uint16_t v[4];
#pragma unroll
        for (int c = 0; c < 4; ++c) v[c] = lr_bits<F16>(f[c] + (a.bias && n + c < a.n ? lr_load<F16>(a.bias[n + c]) : 0.0f));
        if (n + 3 < a.n && a.os % 4 == 0) {
            *(uint2*)o = make_uint2(v[0] | (uint32_t)v[1] << 16, v[2] | (uint32_t)v[3] << 16);
            continue;
        }
#pragma unroll
        for (int c = 0; c < 4; ++c)
            if (n + c < a.n) o[c] = v[c];
    }
}

template <bool F16, int MT, int NT, int KS, int U>
static void launch_rows(const LinearRowsArgs& a, hipStream_t s) {
    hipLaunchKernelGGL((linear_rows_kernel<F16, MT, NT, KS, U>), dim3((a.n + 16 * NT - 1) / (16 * NT)), dim3(KS * 64), 0, s, a);
}
template <bool F16>
static void launch_rows_by_size(const LinearRowsArgs& a, int variant, hipStream_t s) {
    const int mt = (a.m + 15) / 16;
#define V(id, NT, KS, U1, U2, U4) case id: \
    if (mt == 1) launch_rows<F16, 1, NT, KS, U1>(a, s); else if (mt == 2) launch_rows<F16, 2, NT, KS, U2>(a, s); else launch_rows<F16, 4, NT, KS, U4>(a, s); break;
    switch (variant) {
        V(0, 1, 8, 4, 2, 1)
        V(1, 1, 16, 2, 1, 1)
        V(2, 2, 8, 2, 2, 1)
        V(3, 2, 16, 1, 1, 1)
        V(4, 4, 8, 1, 1, 1)
        V(5, 1, 16, 1, 1, 1)
        V(6, 1, 8, 2, 1, 1)
        V(7, 1, 4, 4, 2, 1)
        V(8, 2, 4, 2, 2, 1)
        V(9, 4, 4, 2, 1, 1)
    }
#undef V
}
}  // namespace trimkv
using namespace trimkv;
extern "C" int trimkv_linear_rows(const void* x, int64_t x_stride, const void* w, int64_t w_stride, const void* bias, void* out, int64_t out_stride, int rows, int n, int k,
                                  int dtype, int variant, void* stream) {
    LinearRowsArgs a{(const uint16_t*)x, x_stride, (const uint16_t*)w, w_stride, (const uint16_t*)bias, (uint16_t*)out, out_stride, rows, n, k};
    if (dtype == TRIMKV_F16) launch_rows_by_size<true>(a, variant, (hipStream_t)stream); else launch_rows_by_size<false>(a, variant, (hipStream_t)stream);
    return launch_status("trimkv_linear_rows");
}

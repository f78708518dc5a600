// Products of a few rows with a large matrix (the tokens of a decode step and a linear layer) -- gfx950.
//
//   trimkv_linear_rows        out[m][n] = sum_k x[m][k] w[n][k] (+ bias[n]), up to 64 rows x, w as nn.Linear keeps it
//   trimkv_linear_rows_add    the same plus a residual, with sums of the squares of the result for the norm behind it
//   trimkv_linear_rows_norm   either of the others of the RMS norm of x
//   trimkv_linear_rows_silu   out[m][n] = silu(gate) * up with gate = x . w[n] and up = x . w[inter + n]: a gated feed-forward's
//                             first two matrices and the product of their outputs
//
// 16-bit operands, fp32 sums in a fixed order.
//
// What bounds it: the stream of weights, each byte of which is used for at most 64 rows, and on its way the rate at which one
// compute unit takes operands in (57-60 GB/s measured, whatever the mix of w and x and however much is in flight), because every
// workgroup also reads all of x.  Hence
//  * operands travel through LDS.  In operand layout neighbouring lanes hold neighbouring rows, and a load of 64 lanes in 64 (or
//    8 x 8) different lines is served one lane at a time: 16 B/clk per compute unit.  LDS-direct loads whose lanes run along
//    the rows (8 rows x 128 bytes each) take in 28 B/clk; ds_read_b128 does the regrouping.  12288 x 2048 with 16 rows: 19 us
//    with operand-layout loads, 11.4 here; 4096 x 4096 with 64 rows: 23.4 and 13.7;
//  * a workgroup takes 8 NG rows of w, NG chosen so that the busiest compute unit takes in least (rows_plan below);
//  * the wavefronts of a workgroup take turns on k, 64 elements at a time, each with a ring of its own, so that the main loop
//    has no barrier; their sums meet in LDS at the end of a tile while the next tile's loads are already under way.
//
// Measured in a graph of launches over matrices that no cache holds, us here | the vendor library's product:
//            n x k      1 row        16 rows      32 rows      64 rows
//      2048 x 2048    3.8 | 10.9    4.7 | 11.1    6.0 | 11.2    7.2 | 11.8
//     12288 x 2048   10.1 | 16.6   10.5 | 16.7   11.1 | 16.9   13.9 | 18.2
//      2048 x 6144    6.6 | 11.1    8.5 | 11.3   11.5 | 16.6   16.4 | 19.5
//      4096 x 4096    7.5 | 15.7    8.6 | 15.5   11.1 | 13.4   13.1 | 15.2
//     10240 x 4096   15.0 | 26.6   15.6 | 27.8   16.8 | 23.6   21.3 | 29.6
//     24576 x 4096   32.7 | 45.2   32.7 | 45.5   35.1 | 50.2   40.8 | 50.1
//      4096 x 12288  18.9 | 23.1   21.1 | 23.5   26.8 | 29.1   36.1 | 39.1
#include "common.hip.h"

namespace trimkv {

typedef __bf16 lr_bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 lr_f16x8 __attribute__((ext_vector_type(8)));
typedef float lr_f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t lr_u32x4 __attribute__((ext_vector_type(4)));
#define LR_LDS __attribute__((address_space(3)))

struct LinearRowsArgs {
    const uint16_t* x; int64_t x_stride;
    const uint16_t* w; int64_t w_stride;
    const uint16_t* bias;
    uint16_t* out; int64_t out_stride;
    int m, n, k;        // n: columns of out
    int vec;            // four columns of out can be stored at once
    int round_all;      // silu: the two products and silu(gate) are rounded before they are used, as modules do
    // a residual added to the product: the sums of the squares of what is stored, 8 columns at a time, go to squares [m][n / 8]
    const uint16_t* res; int64_t res_stride;
    // an RMS norm of x in front of the product: its weight; squares [m][k / 8] as above
    const uint16_t* norm_w; float eps;
    float* squares;
};

template <bool F16>
__device__ __forceinline__ lr_f32x4 lr_mfma(lr_u32x4 a, lr_u32x4 b, lr_f32x4 c) {
    if constexpr (F16) return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(lr_f16x8, a), __builtin_bit_cast(lr_f16x8, b), c, 0, 0, 0);
    else return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(lr_bf16x8, a), __builtin_bit_cast(lr_bf16x8, b), c, 0, 0, 0);
}
constexpr int LR_NORM_K = 8192, LR_NORM_ROWS = 32;        // longest and most rows with a norm in front of the product
__device__ __forceinline__ float lr_lo(uint32_t p) { return __uint_as_float(p << 16); }
__device__ __forceinline__ float lr_hi(uint32_t p) { return __uint_as_float(p & 0xffff0000u); }
__device__ __forceinline__ uint32_t lr_pack(float lo, float hi) {
    typedef float f32x2 __attribute__((ext_vector_type(2)));
    typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{lo, hi}, bf16x2));
}
template <bool F16> __device__ __forceinline__ float lr_load(uint16_t b) { return F16 ? f16_bits_to_f32(b) : bf16_bits_to_f32(b); }
template <bool F16> __device__ __forceinline__ uint16_t lr_bits(float f) { return F16 ? f32_to_f16_bits(f) : f32_to_bf16_bits(f); }

// 64 lanes x 16 bytes from base + off to LDS at lds + 16 * lane (base and lds wavefront-uniform).  The compiler neither counts
// nor waits for these loads: whoever reads the LDS waits with an explicit s_waitcnt first.  ONCE: nobody reads the line again.
template <bool ONCE>
__device__ __forceinline__ void lr_load_to_lds(const uint16_t* base, uint32_t off, uint32_t lds) {
    uint32_t saved;
    if constexpr (ONCE)
        asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %3\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2 nt\n\ts_mov_b32 m0, %0"
                     : "=&s"(saved) : "v"(off), "s"(base), "s"(lds) : "memory");
    else
        asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %3\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2\n\ts_mov_b32 m0, %0"
                     : "=&s"(saved) : "v"(off), "s"(base), "s"(lds) : "memory");
}

// XG groups of 8 rows of x, NG groups of 8 rows of w, two to a block of the matrix cores (SILU: 8 of gate and 8 of up; of an odd number the last block repeats
// its half), W wavefronts, D steps of 64 elements of k in flight per wavefront.  A step in LDS: row r of a block holds its eight 16-byte pieces rotated by r / 2,
// which spreads the 16 rows of an operand read over all banks (the rotation is in the lanes' source addresses).
// A decoder's residual add and RMS norm have no launch of their own (4.6 us, most of it latency): the product in front of them (ADD)
// adds the residual where it rounds and leaves sums of squares, a few KB that the product behind them (NORM) adds up while its first
// operands are on their way; x becomes round(round(x / rms) * weight), as modules round, on its way from LDS to the matrix cores.
// A layer's four products with adds and norms, 16 rows: 43.6 -> 40.2 us at 2048 features and 6144, 92.0 -> 83.5 at 4096 and 12288; 1 row
// 38.9 -> 35.9 and 84.7 -> 79.7; 32 rows 49.8 -> 48.0 and 107 -> 102 (both sides while tiles were blocks of 16).  With more rows the arithmetic on the way no longer hides.
enum { LR_PLAIN = 0, LR_ADD = 1, LR_NORM = 2 };
template <bool F16, bool SILU, int MODE, int XG, int NG, int W, int D>
__global__ __launch_bounds__(64 * W) void linear_rows_kernel(LinearRowsArgs a) {
    constexpr bool NORM = MODE == LR_NORM, ADD = MODE == LR_ADD;
    static_assert(MODE == LR_PLAIN || !F16, "bf16 only");
    static_assert(!SILU || NG % 2 == 0, "gate and up");
    constexpr int NT = (NG + 1) / 2, MT = (XG + 1) / 2, L = NG + XG, STEP = L * 1024, U = NT * MT, CG = SILU ? NG / 2 : NG;     // CG: groups of 8 columns of a tile
    static_assert((D - 1) * L < 64, "the wait counts at most 63 loads");
    __shared__ __attribute__((aligned(1024))) char ring[W * D * STEP];
    __shared__ lr_f32x4 part[U * (W - 1)][64];
    __shared__ __attribute__((aligned(16))) uint16_t norm_w[NORM ? LR_NORM_K : 8];
    __shared__ float scale[NORM ? LR_NORM_ROWS : 1];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), r = lane & 15, g = lane >> 4;
    const uint32_t ring_at = (uint32_t)(uintptr_t)(LR_LDS char*)ring + wave * D * STEP;
    const char* mine = ring + wave * D * STEP;
    // a load brings 8 rows, position lane % 8 of row lane / 8; rows that are not there repeat the last one
    uint32_t w_off[2], x_off[XG];
#pragma unroll
    for (int j = 0; j < 2; ++j) w_off[j] = (uint32_t)(min(lane >> 3, a.n - 1) * a.w_stride * 2) + (((lane & 7) - (8 * j + (lane >> 3)) / 2) & 7) * 16;
#pragma unroll
    for (int j = 0; j < XG; ++j) {
        const int row = 8 * j + (lane >> 3);
        x_off[j] = (uint32_t)(min(row, a.m - 1) * a.x_stride * 2) + (((lane & 7) - (row >> 1)) & 7) * 16;
    }
    const int steps = a.k >> 6, first = wave, per_tile = (steps - wave + W - 1) / W, tiles = (a.n + 8 * CG - 1) / (8 * CG);
    // the first column of group c of a tile: the last one of out is moved back so that all its rows exist (it stores the columns that are its own)
    auto column_at = [&](int tile, int c) __attribute__((always_inline)) { return min((tile * CG + c) * 8, max(a.n - 8, 0)); };
    // where a tile begins along k: eight neighbours, one on each XCD, at the same place, the next eight elsewhere (multiples of the golden section, spread evenly)
    auto first_of = [&](int tile) __attribute__((always_inline)) { return first + (int)__umulhi(((uint32_t)tile >> 3) * 0x9e3779b9u, (uint32_t)per_tile) * W; };
    int ask_tile = blockIdx.x, ask_step = first_of(blockIdx.x), ask_left = per_tile, ask_slot = 0;
    int left = per_tile * ((tiles - (int)blockIdx.x + (int)gridDim.x - 1) / (int)gridDim.x);
    auto request = [&]() __attribute__((always_inline)) {       // left: steps that have not been requested; below 0 fewer than D are on their way
        if (--left < 0) return;
        const uint32_t to = ring_at + ask_slot * STEP;
#pragma unroll
        for (int j = 0; j < NG; ++j) {
            const int64_t row = SILU ? column_at(ask_tile, j / 2) + (j % 2 ? a.n : 0) : column_at(ask_tile, j);
            lr_load_to_lds<true>(a.w + row * a.w_stride + ask_step * 64, w_off[j % 2], to + j * 1024);
        }
#pragma unroll
        for (int j = 0; j < XG; ++j) lr_load_to_lds<false>(a.x + ask_step * 64, x_off[j], to + (NG + j) * 1024);
        ask_step = ask_step + W < steps ? ask_step + W : first;
        if (--ask_left == 0) {
            ask_left = per_tile;
            ask_tile += (int)gridDim.x;
            ask_step = first_of(ask_tile);
        }
        ask_slot = ask_slot + 1 == D ? 0 : ask_slot + 1;
    };
    float inv[MT], sum = 0.f;
    constexpr int ROW_THREADS = 64 * W / (8 * XG);        // that add up the squares of one row
    if constexpr (NORM) {       // the weight of the norm: 512 elements a load, of a last one with fewer the last 8 again
        const uint32_t at = (uint32_t)(uintptr_t)(LR_LDS uint16_t*)norm_w;
        for (int p = wave; p * 512 < a.k; p += W) lr_load_to_lds<false>(a.norm_w, (uint32_t)min(p * 512 + lane * 8, a.k - 8) * 2, at + p * 1024);
        const float* from = a.squares + (int64_t)min((int)threadIdx.x / ROW_THREADS, a.m - 1) * (a.k >> 3);
        for (int c = (threadIdx.x % ROW_THREADS) * 4; c < a.k >> 3; c += ROW_THREADS * 4) {
            const lr_f32x4 f = *(const lr_f32x4*)(from + c);
            sum += (f[0] + f[1]) + (f[2] + f[3]);
        }
    }
#pragma unroll
    for (int d = 0; d < D; ++d) request();
    if constexpr (NORM) {
#pragma unroll
        for (int d = 1; d < ROW_THREADS; d <<= 1) sum += __shfl_xor(sum, d, 64);
        if (threadIdx.x % ROW_THREADS == 0) scale[threadIdx.x / ROW_THREADS] = rsqrtf(sum / (float)a.k + a.eps);
        // weight and scales are there for all wavefronts
        if (left >= 0) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(D * L) : "memory");
        else asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
#pragma unroll
        for (int t = 0; t < MT; ++t) inv[t] = scale[XG == 1 ? r & 7 : t * 16 + r];
    }
    lr_f32x4 acc[U];
    int slot = 0;
    for (int tile = blockIdx.x; tile < tiles; tile += gridDim.x) {
#pragma unroll
        for (int u = 0; u < U; ++u) acc[u] = lr_f32x4{0.f, 0.f, 0.f, 0.f};
        int step = first_of(tile);
        for (int s = 0; s < per_tile; ++s) {
            if (left >= 0) asm volatile("s_waitcnt vmcnt(%0)" ::"n"((D - 1) * L) : "memory");
            else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            const char* p = mine + slot * STEP;
            lr_u32x4 wf[2][NT], xf[2][MT], nf[2];
#pragma unroll
            for (int h = 0; h < 2; ++h) {
#pragma unroll
                for (int b = 0; b < NT; ++b) {
                    const int row = 2 * b + 1 == NG ? r & 7 : r;        // half a block: rows 8 .. 15 repeat it
                    wf[h][b] = *(const lr_u32x4*)(p + (b * 16 + row) * 128 + ((h * 4 + g + (row >> 1)) & 7) * 16);
                }
#pragma unroll
                for (int t = 0; t < MT; ++t) {
                    const int row = XG == 1 ? r & 7 : t * 16 + r;       // 8 rows: columns 8 .. 15 repeat them
                    xf[h][t] = *(const lr_u32x4*)(p + (NG * 8 + row) * 128 + ((h * 4 + g + (row >> 1)) & 7) * 16);
                }
                if constexpr (NORM) nf[h] = *(const lr_u32x4*)(norm_w + step * 64 + (h * 4 + g) * 8);
            }
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");          // the step has been read: its room is free
            __builtin_amdgcn_sched_barrier(0);
            request();
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (NORM) {
#pragma unroll
                for (int h = 0; h < 2; ++h)
#pragma unroll
                    for (int t = 0; t < MT; ++t)
#pragma unroll
                        for (int i = 0; i < 4; ++i) {
                            const uint32_t y = lr_pack(lr_lo(xf[h][t][i]) * inv[t], lr_hi(xf[h][t][i]) * inv[t]);
                            xf[h][t][i] = lr_pack(lr_lo(y) * lr_lo(nf[h][i]), lr_hi(y) * lr_hi(nf[h][i]));
                        }
            }
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int b = 0; b < NT; ++b)
#pragma unroll
                    for (int t = 0; t < MT; ++t) acc[b * MT + t] = lr_mfma<F16>(wf[h][b], xf[h][t], acc[b * MT + t]);
            slot = slot + 1 == D ? 0 : slot + 1;
            step = step + W < steps ? step + W : first;
        }
        // the sums of a block and 16 rows go to the wavefront they belong to
        if (tile != (int)blockIdx.x) asm volatile("s_barrier" ::: "memory");        // the sums of the tile before have been read
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (u % W != wave) part[u * (W - 1) + (wave - u % W + W) % W - 1][lane] = acc[u];
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (u % W != wave || (u / MT * 2 + 1 == NG && g >= 2)) continue;
            // this lane: columns n .. n + 3 of row m (SILU: lanes 32 .. 63 have up of what lanes 0 .. 31 have gate of)
            const int c8 = SILU ? u / MT : u / MT * 2 + (g >> 1), m = u % MT * 16 + r, n = column_at(tile, c8) + 4 * (g & 1);
            // Columns below `own` are the group's before, whose sums may have begun elsewhere along k: a column has one writer
            const int own = (tile * CG + c8) * 8;
            if (own >= a.n || n >= a.n || n + 4 <= own || (m >= a.m && !ADD)) continue;       // no such columns, another group's, or no such row
            lr_f32x4 f = acc[u];
#pragma unroll
            for (int o = 0; o < W - 1; ++o) f += part[u * (W - 1) + o][lane];
            uint16_t v[4];
#pragma unroll
            for (int c = 0; c < 4; ++c)
                if (a.bias && n + c < a.n) f[c] += lr_load<F16>(a.bias[(SILU && g >= 2 ? a.n : 0) + n + c]);
            if constexpr (SILU) {
                lr_f32x4 e;
#pragma unroll
                for (int c = 0; c < 4; ++c) e[c] = __shfl_xor(f[c], 32, 64);
                if (g >= 2) continue;
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    if (a.round_all) {
                        const float x = lr_load<F16>(lr_bits<F16>(f[c]));
                        v[c] = lr_bits<F16>(lr_load<F16>(lr_bits<F16>(x / (1.0f + expf(-x)))) * lr_load<F16>(lr_bits<F16>(e[c])));
                    } else v[c] = lr_bits<F16>(f[c] / (1.0f + expf(-f[c])) * e[c]);
                }
            } else {
#pragma unroll
                for (int c = 0; c < 4; ++c) v[c] = lr_bits<F16>(f[c]);
            }
            if constexpr (ADD) {            // n is a multiple of 16: eight columns are there or none
                const uint2 y = *(const uint2*)(a.res + (int64_t)min(m, a.m - 1) * a.res_stride + n);
                const float old[4] = {lr_lo(y.x), lr_hi(y.x), lr_lo(y.y), lr_hi(y.y)};
                float sq = 0.f;
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    v[c] = lr_bits<F16>(lr_load<F16>(v[c]) + old[c]);
                    const float x = lr_load<F16>(v[c]);
                    sq = fmaf(x, x, sq);
                }
                sq += __shfl_xor(sq, 16, 64);
                if (m >= a.m) continue;
                if ((g & 1) == 0) a.squares[(int64_t)m * (a.n >> 3) + (n >> 3)] = sq;
            }
            uint16_t* o = a.out + (int64_t)m * a.out_stride + n;
            if (a.vec) *(uint2*)o = make_uint2(v[0] | (uint32_t)v[1] << 16, v[2] | (uint32_t)v[3] << 16);
            else
#pragma unroll
                for (int c = 0; c < 4; ++c)
                    if (n + c >= own && n + c < a.n) o[c] = v[c];
        }
    }
}

constexpr int LR_CUS = 256;

// Groups of 8 rows of w per tile.  A compute unit that runs `rounds` tiles takes in rounds * (rows of w + rows of x) * k elements;
// the least of that is the fastest (12288 x 4096, 64 rows: 5, 6, 8 groups 2 x 104, 112, 128: 28.5, 22.4, 25.4 us; 4608 x 2048, 16 rows: 2, 3, 4, 5 groups 2 x 32,
// 40, 48, 56: 7.6, 6.9, 7.2, 7.9).  Among equals the smaller one.  In blocks of 16 only, and gate and up in blocks of their own, a tile often had more than its
// compute unit's share while others had none.  Blocks of 16, all beginning at the first k -> groups of 8, eight tiles at each beginning, us, 16 rows if not said: norm and silu
// 2 x 6144 x 2048 12.6 -> 11.2 (4 rows 12.6 -> 11.4, 32 rows 14.7 -> 12.6), norm 4608 x 2048 7.6 -> 6.9 (9.0 -> 8.4), 6656 x 4096 14.5 -> 12.6, add 4096 x 4096 8.9 -> 8.2, 64 rows: 10240 x
// 4096 22.0 -> 20.8, 6144 x 2048 10.3 -> 9.6, 12288 x 4096 23.3 -> 22.4, silu 2 x 12288 x 4096 44.3 -> 40.0.  The beginnings alone: 0 .. 7 % of these (2048 x 6144 8.6 -> 8.5, 64
// rows of 2 x 12288 x 4096 46.0 -> 40.0): tiles that begin together otherwise ask the same few channels of memory for the same k.
static int rows_plan(int n, int x_rows, bool silu) {
    static const int plain[] = {1, 2, 3, 4, 5, 6, 8, 12}, paired[] = {2, 4, 6, 8, 12};
    const int* sizes = silu ? paired : plain;
    const int most = x_rows < 64 ? (silu ? 4 : 6) : (silu ? 5 : 8);     // fewer rows of x: more than that was not faster at any size measured
    int best = sizes[0];
    int64_t least = INT64_MAX;
    for (int i = 0; i < most; ++i) {
        const int ng = sizes[i];
        const int64_t cols = 8 * (silu ? ng / 2 : ng), tiles = (n + cols - 1) / cols, cost = (tiles + LR_CUS - 1) / LR_CUS * (8 * ng + x_rows);
        if (cost < least) { least = cost; best = ng; }
    }
    return best;
}

template <bool F16, bool SILU, int XG, int NG, int W, int D, int MODE>
static void rows_launch(const LinearRowsArgs& a, hipStream_t s) {
    constexpr int CG = SILU ? NG / 2 : NG, SUMS = (W - 1) * ((NG + 1) / 2) * ((XG + 1) / 2) * 1024;
    constexpr int LDS = W * D * (NG + XG) * 1024 + SUMS + (MODE == LR_NORM ? LR_NORM_K * 2 + LR_NORM_ROWS * 4 : 32);
    static_assert(LDS <= 160 * 1024, "LDS of a compute unit");
    const int tiles = (a.n + 8 * CG - 1) / (8 * CG), most = LR_CUS * (160 * 1024 / LDS);
    hipLaunchKernelGGL((linear_rows_kernel<F16, SILU, MODE, XG, NG, W, D>), dim3(tiles < most ? tiles : most), dim3(64 * W), 0, s, a);
}
// Wavefronts and depth: the fastest of 2, 4, 8 and 1 .. 4 over the shapes above, as far as LDS reaches.  Eight wavefronts up to 32 rows: each has half as many steps
// of four, one behind the other, and up to 8 KB of a step of all are asked for before the first one is used; with 64 rows their sums take the room of a second step.
template <bool F16, int XG, int MODE = LR_PLAIN>
static void rows_by_groups(const LinearRowsArgs& a, bool silu, hipStream_t s) {
    const int ng = rows_plan(a.n, 8 * XG, silu);
    constexpr bool MANY = XG == 8, SOME = XG == 4;
    if constexpr (MODE != LR_ADD)
        if (silu) {
            if constexpr (MANY)
                if (ng == 12) return rows_launch<F16, true, XG, 12, 4, 1, MODE>(a, s);
            if (ng == 8) return rows_launch<F16, true, XG, 8, MANY ? 2 : SOME ? 4 : 8, MANY || SOME ? 2 : 1, MODE>(a, s);
            if (ng == 6) return rows_launch<F16, true, XG, 6, MANY ? 4 : 8, MANY ? 2 : 1, MODE>(a, s);
            if (ng == 4) return rows_launch<F16, true, XG, 4, MANY ? 4 : 8, MANY || XG == 1 ? 2 : 1, MODE>(a, s);
            return rows_launch<F16, true, XG, 2, MANY ? 4 : 8, MANY ? 2 : 1, MODE>(a, s);
        }
    if constexpr (MANY) {
        if (ng == 12) return rows_launch<F16, false, XG, 12, 4, 1, MODE>(a, s);
        if (ng == 8) return rows_launch<F16, false, XG, 8, 4, 1, MODE>(a, s);
    }
    constexpr int W = MANY ? 4 : 8, D = SOME ? 1 : 2;
    switch (ng) {
        case 1: return rows_launch<F16, false, XG, 1, W, XG == 1 ? 4 : 2, MODE>(a, s);
        case 2: return rows_launch<F16, false, XG, 2, W, 2, MODE>(a, s);
        case 3: return rows_launch<F16, false, XG, 3, W, D, MODE>(a, s);
        case 4: return rows_launch<F16, false, XG, 4, W, D, MODE>(a, s);
        case 5: return rows_launch<F16, false, XG, 5, W, XG == 2 ? 1 : D, MODE>(a, s);
        default: return rows_launch<F16, false, XG, 6, W, XG == 2 && MODE == LR_NORM ? 1 : D, MODE>(a, s);
    }
}
template <bool F16>
static void rows_by_rows(const LinearRowsArgs& a, bool silu, hipStream_t s) {
    if (a.m <= 8) rows_by_groups<F16, 1>(a, silu, s);
    else if (a.m <= 16) rows_by_groups<F16, 2>(a, silu, s);
    else if (a.m <= 32) rows_by_groups<F16, 4>(a, silu, s);
    else rows_by_groups<F16, 8>(a, silu, s);
}

template <int MODE>
static void norm_by_rows(const LinearRowsArgs& a, bool silu, hipStream_t s) {
    if (a.m <= 8) rows_by_groups<false, 1, MODE>(a, silu, s);
    else if (a.m <= 16) rows_by_groups<false, 2, MODE>(a, silu, s);
    else rows_by_groups<false, 4, MODE>(a, silu, s);
}

}  // namespace trimkv

using namespace trimkv;

static int rows_check_and_launch(const char* fn, LinearRowsArgs a, bool silu, int dtype, void* stream) {
    if (!a.x || !a.w || !a.out) return fail(TRIMKV_ERR_NULL, "%s: null pointer argument", fn);
    if (dtype != TRIMKV_BF16 && dtype != TRIMKV_F16) return fail(TRIMKV_ERR_DTYPE, "%s: bf16 or fp16 only (dtype=%d)", fn, dtype);
    if (a.m <= 0 || a.m > 64 || a.n <= 0 || a.n > (1 << 29) || a.k <= 0 || a.k % 64)
        return fail(TRIMKV_ERR_SHAPE, "%s: bad sizes rows=%d (1 .. 64) n=%d k=%d (a multiple of 64)", fn, a.m, a.n, a.k);
    if (a.x_stride < a.k || a.w_stride < a.k || a.out_stride < a.n || a.x_stride % 8 || a.w_stride % 8 || a.x_stride > (1 << 24) || a.w_stride > (1 << 24))
        return fail(TRIMKV_ERR_SHAPE, "%s: strides %lld %lld (>= k, multiples of 8, at most 2^24) %lld (>= n)", fn, (long long)a.x_stride, (long long)a.w_stride, (long long)a.out_stride);
    if (((uintptr_t)a.x | (uintptr_t)a.w) & 15) return fail(TRIMKV_ERR_SHAPE, "%s: x and w must be 16-byte aligned", fn);
    a.vec = a.n % 4 == 0 && a.out_stride % 4 == 0 && !((uintptr_t)a.out & 7);
    if (a.norm_w) norm_by_rows<LR_NORM>(a, silu, (hipStream_t)stream);
    else if (a.res) norm_by_rows<LR_ADD>(a, silu, (hipStream_t)stream);
    else if (dtype == TRIMKV_F16) rows_by_rows<true>(a, silu, (hipStream_t)stream);
    else rows_by_rows<false>(a, silu, (hipStream_t)stream);
    return launch_status(fn);
}

extern "C" int trimkv_linear_rows(const void* x, int64_t x_stride, const void* w, int64_t w_stride, const void* bias, void* out, int64_t out_stride,
                                  int rows, int n, int k, int dtype, void* stream) {
    return rows_check_and_launch("trimkv_linear_rows",
                                 LinearRowsArgs{(const uint16_t*)x, x_stride, (const uint16_t*)w, w_stride, (const uint16_t*)bias, (uint16_t*)out, out_stride, rows, n, k, 0, 0}, false, dtype, stream);
}

extern "C" int trimkv_linear_rows_silu(const void* x, int64_t x_stride, const void* w, int64_t w_stride, const void* bias, void* out, int64_t out_stride,
                                       int rows, int inter, int k, int round_all, int dtype, void* stream) {
    return rows_check_and_launch("trimkv_linear_rows_silu",
                                 LinearRowsArgs{(const uint16_t*)x, x_stride, (const uint16_t*)w, w_stride, (const uint16_t*)bias, (uint16_t*)out, out_stride, rows, inter, k, 0, round_all}, true, dtype, stream);
}

extern "C" int trimkv_linear_rows_add(const void* x, int64_t x_stride, const void* w, int64_t w_stride, const void* bias, const void* residual, int64_t residual_stride,
                                      void* out, int64_t out_stride, float* squares, int rows, int n, int k, int dtype, void* stream) {
    const char* fn = "trimkv_linear_rows_add";
    if (!residual || !squares) return fail(TRIMKV_ERR_NULL, "%s: null pointer argument", fn);
    if (dtype != TRIMKV_BF16) return fail(TRIMKV_ERR_DTYPE, "%s: bf16 only (dtype=%d)", fn, dtype);
    if (rows > LR_NORM_ROWS || n % 16) return fail(TRIMKV_ERR_SHAPE, "%s: at most %d rows, n a multiple of 16 (got %d, %d)", fn, LR_NORM_ROWS, rows, n);
    if (residual_stride < n || residual_stride % 4 || out_stride % 4 || ((uintptr_t)residual | (uintptr_t)out) & 7)
        return fail(TRIMKV_ERR_SHAPE, "%s: residual and out must be 8-byte aligned, their strides multiples of 4 and at least n (%lld)", fn, (long long)residual_stride);
    LinearRowsArgs a{(const uint16_t*)x, x_stride, (const uint16_t*)w, w_stride, (const uint16_t*)bias, (uint16_t*)out, out_stride, rows, n, k, 0, 0};
    a.res = (const uint16_t*)residual; a.res_stride = residual_stride; a.squares = squares;
    return rows_check_and_launch(fn, a, false, dtype, stream);
}

extern "C" int trimkv_linear_rows_norm(const void* x, int64_t x_stride, const float* squares, const void* norm_weight, float eps, const void* w, int64_t w_stride,
                                       const void* bias, void* out, int64_t out_stride, int rows, int n, int k, int silu, int round_all, int dtype, void* stream) {
    const char* fn = "trimkv_linear_rows_norm";
    if (!squares || !norm_weight) return fail(TRIMKV_ERR_NULL, "%s: null pointer argument", fn);
    if (dtype != TRIMKV_BF16) return fail(TRIMKV_ERR_DTYPE, "%s: bf16 only (dtype=%d)", fn, dtype);
    if (rows > LR_NORM_ROWS || k > LR_NORM_K) return fail(TRIMKV_ERR_SHAPE, "%s: at most %d rows of %d (got %d of %d)", fn, LR_NORM_ROWS, LR_NORM_K, rows, k);
    if (((uintptr_t)norm_weight | (uintptr_t)squares) & 15) return fail(TRIMKV_ERR_SHAPE, "%s: squares and norm_weight must be 16-byte aligned", fn);
    LinearRowsArgs a{(const uint16_t*)x, x_stride, (const uint16_t*)w, w_stride, (const uint16_t*)bias, (uint16_t*)out, out_stride, rows, n, k, 0, round_all};
    a.norm_w = (const uint16_t*)norm_weight; a.eps = eps; a.squares = const_cast<float*>(squares);
    return rows_check_and_launch(fn, a, silu != 0, dtype, stream);
}

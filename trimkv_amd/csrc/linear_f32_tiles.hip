// Products of many rows with a matrix in fp32 (the tokens of a prompt and a linear layer of a decoder that runs in fp32) -- gfx950.
//
//   trimkv_linear_f32_tiles        out[m][n] = sum_k x[m][k] w[n][k], w as nn.Linear keeps it
//   trimkv_linear_f32_tiles_form   how it is cut by sizes
//
// What bounds it: the matrix cores.  Their fp32 instructions do 157 TFLOP/s at most (the vendor library's product 97 - 120 at the sizes below); three
// bf16 terms hold all 24 bits of an fp32 number from 2^-103 on, and six of the nine products of two such sums (those above 2^-24 of the largest; the others are 3 * 2^-25 of
// |x w| at most) on the bf16 instructions take 2.7 times fewer cycles.  The operands come as fp32 and are split on their way, once for every tile that they are in: beside 6 MU NU
// matrix instructions for MU x NU blocks of 16 x 16 x 32 stand 32 (MU + NU) vector instructions, eight for a pair of numbers: v_cvt_pk_bf16_f32 takes a term of both,
// v_dot2_f32_bf16 what is left of one, exactly (with masks, subtractions and packs four more: 5 % slower), and v_max3_f32 follows the largest.  Matrix and vector instructions of one wavefront follow one another (spread between one
// another, v_dot2 waits for the matrix cores and the others gain nothing measurable), so that the tiles run at 178 - 189 TFLOP/s of fp32 product.  Hence
//  * all four wavefronts of a workgroup have the same tile and take turns on k, 32 at a time, each with LDS of its own: nothing is split twice and the main
//    loop has no barrier; their sums meet in LDS at the end;
//  * a tile may have any number of blocks of 16 either way, so that a launch can be cut into what fills the compute units (f32_tiles_form);
//  * x is held, w streams past it: 16 rows of w are requested, one period of k later read, split, and multiplied, all while their neighbours are.
// Error against 64 bits (2-norm, relative; numbers of a normal distribution): 3.5e-7 for k = 2048, 5.0e-7 for 4096, that of the sums (the vendor library's
// product 8.1e-7, 1.1e-6; fp32 matrix instructions in this file's order 4.1e-7).
// What bf16 terms do not hold is done by fp32 matrix instructions.  Infinities, NaN and numbers that round to infinity end as results that are not finite: blocks with such
// results are done again.  Numbers below 2^-103 lose up to 2^-125 each.  That is nothing beside a result of 2^-97 k times the largest number and more; a tile with a smaller
// result looks through its rows, and blocks with a row that has such a number are done again (rows 2^-118 times a normal distribution, against a matrix 2^100 times, without it:
// error 8.8e-6, 2^-126 2.3e-3, 2^-134 0.6; now 4.1e-7).  Following the largest costs 3 - 5 % of a launch, 7 % in the smallest tiles, a row of zeros in each tile 40 %: 811 x 6144 x 2048 117 -> 122 us, 160 with
// such rows (the vendor library's 205), 900 if all of x is below 2^-103.  With the smallest number followed instead, single zeros sent tiles to look.
//
// Measured (rows x n x k, us here | the vendor library's product): 811 x 6144 x 2048 122 | 205, 811 x 2048 x 2048 45 | 58, 811 x 1024 x 2048 27 | 35, 300 x 6144 x
// 2048 46 | 64, 300 x 2048 x 2048 23 | 28, 100 x 2048 x 2048 15 | 21, 30 x 6144 x 2048 17 | 21, 1700 x 6144 x 2048 242 | 373, 811 x 4096 x 4096 166 | 248.
#include "hybrid.hip.h"

namespace trimkv {

struct F32TilesArgs {
    const float* x; int64_t xs;
    const float* w; int64_t ws;
    float* y; int64_t ys;
    int m, n, k, vec;
};

// 16 rows x 128 bytes to LDS at lds, the first 8 from base + off0, the others from low + 1024 + off1 (the offset in the instruction moves both addresses).
// The compiler neither counts nor waits for these loads: the reader waits with an explicit s_waitcnt first.
__device__ __forceinline__ void ft_load_unit(const char* base, const char* low, uint32_t off0, uint32_t off1, uint32_t lds) {
    uint32_t saved;
    asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %5\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %3\n\tglobal_load_lds_dwordx4 %2, %4 offset:1024\n\ts_mov_b32 m0, %0"
                 : "=&s"(saved) : "v"(off0), "v"(off1), "s"(base), "s"(low), "s"(lds) : "memory");
}

struct Terms { hy_u32x4 t[3]; };      // eight numbers as sums of three bf16 each

// f less one of the two bf16 numbers in p, exactly.  minus: -1 for that one and 0 for the other, in a register: as an instruction's constant the compiler writes
// the pair (-1, 0) as the number -1.0, which the instruction takes for (0, -1)
__device__ __forceinline__ float ft_rest(uint32_t p, uint32_t minus, float f) {
    return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(hy_bf16x2, p), __builtin_bit_cast(hy_bf16x2, minus), f, false);
}

// Three bf16 terms hold the 24 bits of numbers from 2^-103 on (and 0): below, what the last ones stand for is under 2^-126 and may be lost
constexpr uint32_t FT_LEAST = (127u - 103u) << 23;       // bits of 2^-103
__device__ __forceinline__ float ft_most(float most, float a, float b) {
    asm("v_max3_f32 %0, %0, |%1|, |%2|" : "+v"(most) : "v"(a), "v"(b));
    return most;
}

__device__ __forceinline__ void split8(const hy_f32x4 (&v)[2], Terms& o, float& most) {
    uint32_t low, high;
    asm("s_mov_b32 %0, 0xbf80" : "=s"(low));
    asm("s_mov_b32 %0, 0xbf800000" : "=s"(high));
#pragma unroll
    for (int p = 0; p < 4; ++p) {
        float a = v[p >> 1][2 * (p & 1)], b = v[p >> 1][2 * (p & 1) + 1];
        most = ft_most(most, a, b);
#pragma unroll
        for (int t = 0; t < 3; ++t) {
            const uint32_t u = pack2(a, b);
            o.t[t][p] = u;
            if (t < 2) { a = ft_rest(u, low, a); b = ft_rest(u, high, b); }
        }
    }
}

// the wavefronts' rings, or their sums and eight words behind these
constexpr int ft_lds(int MU, int NU, int D) { return D * (MU + NU) * 8 > MU * NU * 3 ? D * (MU + NU) * 8192 : MU * NU * 3072 + 32; }

// 16 x 16 results by fp32 matrix instructions, for a whole wavefront.  Four sums of k / 4 products: one of all errs by 8.1e-7 for k = 2048
__device__ __forceinline__ hy_f32x4 f32_block(const F32TilesArgs& a, int m0, int n0) {
    const int lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
    const float* const x = a.x + (int64_t)min(m0 + r, a.m - 1) * a.xs + 4 * g;
    const float* const w = a.w + (int64_t)min(n0 + r, a.n - 1) * a.ws + 4 * g;
    hy_f32x4 acc[4] = {};
    for (int k = 0; k < a.k; k += 16) {
        const hy_f32x4 xf = *(const hy_f32x4*)(x + k), wf = *(const hy_f32x4*)(w + k);
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[i] = mfma16_f32(wf[i], xf[i], acc[i]);
    }
    return (acc[0] + acc[1]) + (acc[2] + acc[3]);
}

// MU x NU blocks of 16 x 16 to a tile, D periods of k in LDS.  Two workgroups to a compute unit where registers and LDS (80 KB) allow it.
template <int MU, int NU, int D>
__global__ __launch_bounds__(256, (MU + NU) * D <= 10 ? 2 : 1) void linear_f32_tiles_kernel(F32TilesArgs a) {
    constexpr int L = MU + NU, U = MU * NU, R1 = (MU + 2) / 2, R2 = MU + 2 - R1;
    static_assert(NU >= 3 && 2 * (L * D - 1) < 64, "the wait counts at most 63 loads");
    extern __shared__ __attribute__((aligned(1024))) char lds[];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), r = lane & 15, g = lane >> 4;
    const int mt = (a.m + 16 * MU - 1) / (16 * MU), nt = (a.n + 16 * NU - 1) / (16 * NU), whole = mt * nt, share = (whole + 7) / 8;
    const int at = (blockIdx.x & 7) * share + (blockIdx.x >> 3);
    if ((int)(blockIdx.x >> 3) >= share || at >= whole) return;
    const int m0 = at % mt * 16 * MU, n0 = at / mt * 16 * NU;
    const uint32_t ring_at = (uint32_t)(uintptr_t)(HY_LDS char*)lds + wave * D * L * 2048;
    const char* const mine = lds + wave * D * L * 2048;
    // units 0 .. MU - 1: 16 rows of x each; MU .. L - 1: 16 rows of w.  A load brings 8 rows x 128 bytes
    uint32_t off[L][2];
#pragma unroll
    for (int j = 0; j < L; ++j)
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int row = 8 * h + (lane >> 3), piece = ((lane & 7) - (row >> 1)) & 7;
            off[j][h] = j < MU ? (uint32_t)min(16 * j + row, a.m - 1 - m0) * (uint32_t)(a.xs * 4) + piece * 16
                               : (uint32_t)min(16 * (j - MU) + row, a.n - 1 - n0) * (uint32_t)(a.ws * 4) + piece * 16;
        }
    const char* const xb = (const char*)(a.x + (int64_t)m0 * a.xs);
    const char* const wb = (const char*)(a.w + (int64_t)n0 * a.ws);
    const int total = a.k >> 5, periods = (total - wave + 3) >> 2;
    auto request = [&](int j, int p, int slot) __attribute__((always_inline)) {       // behind the last period: that one again, never read
        const char* const from = (j < MU ? xb : wb) + (int64_t)(wave + 4 * min(p, periods - 1)) * 128;
        ft_load_unit(from, from - 1024, off[j][0], off[j][1], ring_at + (slot * L + j) * 2048);
    };
    hy_f32x4 acc[U];
    float most = 0.f;        // of the numbers this lane has split
#pragma unroll
    for (int u = 0; u < U; ++u) acc[u] = hy_f32x4{0.f, 0.f, 0.f, 0.f};
    struct Raw { hy_f32x4 v[2]; };
    auto read = [&](int j, int slot) __attribute__((always_inline)) {
        Raw o;
#pragma unroll
        for (int h = 0; h < 2; ++h) o.v[h] = *(const hy_f32x4*)(mine + (slot * L + j) * 2048 + r * 128 + ((h * 4 + g + (r >> 1)) & 7) * 16);
        return o;
    };
    // Order of the units: 0 and the held ones, 1 of w, then 2 .. NU - 1 of w; a period later again
    auto tail = [](int i) { return i == 0 ? MU : i <= MU ? i - 1 : MU + 1; };
    if (periods > 0) {
#pragma unroll
        for (int d = 0; d < D; ++d) {
#pragma unroll
            for (int i = 0; i < MU + 2; ++i) request(tail(i), d, d);
#pragma unroll
            for (int j = 2; j < NU; ++j) request(MU + j, d, d);
        }
        Raw hraw[MU], first, coming;
        Terms held[MU], cur, nxt;
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * (L * D - MU - 2)) : "memory");
        first = read(MU, 0);
#pragma unroll
        for (int i = 0; i < MU; ++i) hraw[i] = read(i, 0);
        coming = read(MU + 1, 0);
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
        for (int i = 0; i < R1; ++i) request(tail(i), D, 0);
        int slot = 0, after = D > 1 ? 1 : 0;
        split8(first.v, cur, most);
        for (int p = 0; p < periods; ++p) {
#pragma unroll
            for (int i = 0; i < MU; ++i) split8(hraw[i].v, held[i], most);
#pragma unroll
            for (int j = 0; j < NU; ++j) {
                asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
                if (j == 0) {
#pragma unroll
                    for (int i = R1; i < MU + 2; ++i) request(tail(i), p + D, slot);
                } else if (j == NU - 1) {
#pragma unroll
                    for (int i = 0; i < R1; ++i) request(tail(i), p + 1 + D, after);
                } else request(MU + j + 1, p + D, slot);
                const Raw now = coming;
                if (j < NU - 2) {
                    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * (L * D - 1)) : "memory");
                    coming = read(MU + j + 2, slot);
                } else if (j == NU - 2) {
                    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * (L * D - R1)) : "memory");
                    coming = read(MU, after);
#pragma unroll
                    for (int i = 1; i < R1; ++i) hraw[i - 1] = read(i - 1, after);
                } else {
                    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * (L * D - R2)) : "memory");
#pragma unroll
                    for (int i = R1; i <= MU; ++i) hraw[i - 1] = read(i - 1, after);
                    coming = read(MU + 1, after);
                }
                __builtin_amdgcn_sched_barrier(0);
                split8(now.v, nxt, most);
                constexpr int X[6] = {0, 2, 1, 0, 1, 0}, W[6] = {2, 0, 1, 1, 0, 0};
#pragma unroll
                for (int q = 0; q < 6; ++q)
#pragma unroll
                    for (int i = 0; i < MU; ++i)
                        acc[i * NU + j] = mfma16(__builtin_bit_cast(hy_bf16x8, cur.t[W[q]]), __builtin_bit_cast(hy_bf16x8, held[i].t[X[q]]), acc[i * NU + j]);
                cur = nxt;
                __builtin_amdgcn_sched_barrier(0);
            }
            slot = after;
            after = after + 1 == D ? 0 : after + 1;
        }
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
    }
    // sums of the four wavefronts meet in LDS; unit u belongs to wavefront u % 4
    __syncthreads();
    hy_f32x4(*part)[64] = (hy_f32x4(*)[64])lds;
    int* const words = (int*)(lds + U * 3072);
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) most = fmaxf(most, __shfl_xor(most, d, 64));
    if (lane == 0) words[wave] = __float_as_int(most);
#pragma unroll
    for (int u = 0; u < U; ++u)
        if (u % 4 != wave) part[u * 3 + (wave - u % 4 + 4) % 4 - 1][lane] = acc[u];
    __syncthreads();
    auto store = [&](int u, hy_f32x4 s) __attribute__((always_inline)) {
        const int m = m0 + u / NU * 16 + r, n = n0 + u % NU * 16 + 4 * g;
        if (m >= a.m || n >= a.n) return;
        float* const y = a.y + (int64_t)m * a.ys + n;
        if (a.vec && n + 3 < a.n) *(hy_f32x4*)y = s;
        else
#pragma unroll
            for (int c = 0; c < 4; ++c)
                if (n + c < a.n) y[c] = s[c];
    };
    // 2^-125 of up to k numbers, times as many as large as any here, may be lost: less than 2^-27 of a result of `sure` or more
    most = fmaxf(fmaxf(__int_as_float(words[0]), __int_as_float(words[1])), fmaxf(__int_as_float(words[2]), __int_as_float(words[3])));
    const float sure = most * 0x1p-97f * (float)a.k;
    uint32_t again = 0;
    bool unsure = false;
#pragma unroll
    for (int u = 0; u < U; ++u) {
        if (u % 4 != wave) continue;
        hy_f32x4 s = acc[u];
#pragma unroll
        for (int o = 0; o < 3; ++o) s += part[u * 3 + o][lane];
        unsure |= fminf(fminf(fabsf(s[0]), fabsf(s[1])), fminf(fabsf(s[2]), fabsf(s[3]))) < sure;
        if (__any(!finite_bits(__builtin_bit_cast(hy_u32x4, s)))) again |= 1u << (u / 4);
        else store(u, s);
    }
    // Smaller results, rows of zeros above all: blocks with a row of x or of w that has a number of less than 2^-103 are done again as well
    unsure = __any(unsure);
    if (lane == 0) words[4 + wave] = unsure;
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    if (words[4] | words[5] | words[6] | words[7]) {
        uint32_t rows = 0;        // bit j: unit j has such a row
        for (int p = 0; p < periods; ++p)
#pragma unroll
            for (int j = 0; j < L; ++j)
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const hy_u32x4 v = *(const hy_u32x4*)((j < MU ? xb : wb) + (int64_t)(wave + 4 * p) * 128 + off[j][h]);
#pragma unroll
                    for (int i = 0; i < 4; ++i) rows |= (v[i] & 0x7fffffffu) - 1u < FT_LEAST - 1u ? 1u << j : 0u;
                }
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) rows |= __shfl_xor(rows, d, 64);
        if (lane == 0) words[wave] = (int)rows;
        __syncthreads();
        rows = (uint32_t)__builtin_amdgcn_readfirstlane(words[0] | words[1] | words[2] | words[3]);
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (u % 4 == wave && (rows >> (u / NU) & 1 || rows >> (MU + u % NU) & 1)) again |= 1u << (u / 4);
    }
    for (int i = 0; again >> i; ++i)
        if (again >> i & 1) store(4 * i + wave, f32_block(a, m0 + (4 * i + wave) / NU * 16, n0 + (4 * i + wave) % NU * 16));
}

struct F32Form { int mu, nu, d; bool pairs; float begin, period; };      // pairs: two workgroups to a compute unit

// A form takes begin + period * periods of 128 k (us) for a round of a tile per compute unit; with two workgroups to each, the beginnings of later
// rounds pass unseen.  Measured with 128 .. 1024 tiles of k = 512, 2048 and 4096, without the largest number followed: as it is 3 - 5 % more, of the first two 7 %.
constexpr F32Form F32_FORMS[] = {{1, 4, 2, true, 4.2f, 0.69f}, {2, 3, 2, true, 3.6f, 0.80f}, {2, 6, 1, true, 3.8f, 1.34f}, {3, 4, 1, true, 3.9f, 1.20f}, {4, 4, 1, true, 4.8f, 1.43f},
                                 {3, 6, 1, true, 4.6f, 1.68f}, {4, 5, 1, true, 5.2f, 1.72f}, {4, 6, 1, true, 5.2f, 2.05f}, {5, 6, 1, false, 6.8f, 2.34f}, {3, 9, 1, false, 7.0f, 2.37f},
                                 {4, 8, 1, false, 7.4f, 2.50f}, {4, 10, 1, false, 8.0f, 3.10f}, {6, 8, 1, false, 9.0f, 3.50f}};
constexpr int F32_FORM_COUNT = sizeof(F32_FORMS) / sizeof(F32_FORMS[0]);

static int f32_tiles_form(int m, int n, int k, float* cost) {
    int best = 0;
    for (int i = 0; i < F32_FORM_COUNT; ++i) {
        const F32Form& f = F32_FORMS[i];
        const int64_t tiles = (int64_t)((m + 16 * f.mu - 1) / (16 * f.mu)) * ((n + 16 * f.nu - 1) / (16 * f.nu)), rounds = (tiles + 255) / 256;
        const float c = (f.pairs ? 1.f : (float)rounds) * f.begin + (float)rounds * f.period * (float)((k + 127) / 128);
        if (!best || c < *cost) { *cost = c; best = i + 1; }
    }
    return best;
}

template <int I>
static int f32_tiles_launch(const F32TilesArgs& a, hipStream_t s) {
    constexpr F32Form F = F32_FORMS[I];
    constexpr int LDS = ft_lds(F.mu, F.nu, F.d);
    static_assert(LDS <= (F.pairs ? 80 : 160) * 1024, "LDS of a compute unit");
    static bool opted_in[64] = {};
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) dev = -1;
    if (dev < 0 || !opted_in[dev]) {
        hipError_t e = hipFuncSetAttribute((const void*)linear_f32_tiles_kernel<F.mu, F.nu, F.d>, hipFuncAttributeMaxDynamicSharedMemorySize, LDS);
        if (e != hipSuccess) return (int)e;
        if (dev >= 0) opted_in[dev] = true;
    }
    const int64_t tiles = (int64_t)((a.m + 16 * F.mu - 1) / (16 * F.mu)) * ((a.n + 16 * F.nu - 1) / (16 * F.nu));
    hipLaunchKernelGGL((linear_f32_tiles_kernel<F.mu, F.nu, F.d>), dim3((unsigned)(8 * ((tiles + 7) / 8))), dim3(256), LDS, s, a);
    return 0;
}

template <int I>
static int f32_tiles_by_form(int form, const F32TilesArgs& a, hipStream_t s) {
    if (form == I + 1) return f32_tiles_launch<I>(a, s);
    if constexpr (I + 1 < F32_FORM_COUNT) return f32_tiles_by_form<I + 1>(form, a, s);
    return -1;
}

}  // namespace trimkv

using namespace trimkv;

extern "C" int trimkv_linear_f32_tiles(const float* x, int64_t x_stride, const float* w, int64_t w_stride, float* out, int64_t out_stride, int rows, int n, int k, int form, void* stream) {
    const char* fn = "trimkv_linear_f32_tiles";
    F32TilesArgs a{x, x_stride, w, w_stride, out, out_stride, rows, n, k, 0};
    if (!x || !w || !out) return fail(TRIMKV_ERR_NULL, "%s: null pointer argument", fn);
    if (rows <= 0 || n <= 0 || k <= 0 || k % 32 || rows > (1 << 22) || n > (1 << 22) || x_stride < k || w_stride < k || x_stride > (1 << 20) || w_stride > (1 << 20) || x_stride % 4 || w_stride % 4 ||
        out_stride < n)
        return fail(TRIMKV_ERR_SHAPE, "%s: bad sizes rows=%d n=%d k=%d (a multiple of 32) strides %lld %lld %lld", fn, rows, n, k, (long long)x_stride, (long long)w_stride, (long long)out_stride);
    if (((uintptr_t)x | (uintptr_t)w) & 15 || (uintptr_t)out & 3) return fail(TRIMKV_ERR_SHAPE, "%s: x and w must be 16-byte aligned", fn);
    if (form < 0 || form > F32_FORM_COUNT) return fail(TRIMKV_ERR_SHAPE, "%s: no form %d", fn, form);
    float cost;
    if (!form) form = f32_tiles_form(rows, n, k, &cost);
    a.vec = out_stride % 4 == 0 && !((uintptr_t)out & 15);
    const int rc = f32_tiles_by_form<0>(form, a, (hipStream_t)stream);
    if (rc) return fail(rc, "%s: hipFuncSetAttribute failed (%d)", fn, rc);
    return launch_status(fn);
}

// Products that the tiles take at less than RATE (by the estimate) have too few of them: the vendor's library divides their k further.
extern "C" int trimkv_linear_f32_tiles_form(int rows, int n, int k) {
    constexpr float RATE = 95e6f;        // operations in a us
    if (rows <= 0 || n <= 0 || k <= 0 || k % 32) return 0;
    float cost;
    const int form = f32_tiles_form(rows, n, k, &cost);
    return 2.f * (float)rows * (float)n * (float)k >= RATE * cost ? form : 0;
}

// Products of many rows with a matrix (the tokens of a prompt and a linear layer) in bf16 -- gfx950.
//
//   trimkv_linear_tiles       out[m][n] = sum_k x[m][k] w[n][k], w as nn.Linear keeps it
//   trimkv_linear_tiles_silu  out[m][n] = silu(gate) * up with gate = x . w[n] and up = x . w[inter + n]: a gated feed-forward's first two
//                             matrices and the product of their outputs
//
// Tiles as tiles.hip.h multiplies them, of 256, 192 or 128 rows x 256 outputs (silu: 128 of the gate and 128 of up, which meet in one
// lane's accumulators), and of 128 x 128.  What bounds a launch: while the tiles fill the chip, the clock that the matrix cores leave it (1.7 - 1.8 GHz, matrix pipes
// busy 88 % of a tile's time: 1.5 PFLOP/s); before that, the last round of tiles, which the compute units do not share evenly.  So a launch is cut by sizes
// (tiles_cost): the height of its tiles, and whether the rows and columns that fill no whole tile go in small ones.  8286 x 6144 x 2048
// (rows x n x k): 33 x 24 tiles of 256 in four rounds 209 us, 32 x 24 and the last 94 rows in small ones 164; the vendor library's product 220 - 240.
#include "tiles.hip.h"
#include <math.h>

namespace trimkv {

struct TilesArgs {
    const uint16_t* x; int64_t xs;
    const uint16_t* w; int64_t ws;
    uint16_t* y; int64_t ys;
    int m, n, k;            // n: columns of y
    int round_all;          // silu: the two products and silu(gate) are rounded before they are used, as modules do
    int mt, nt;             // row and column tiles that are taken whole; what lies behind them goes in tiles of 128 x 128
};

__device__ __forceinline__ float rounded(float f) { return bf16_bits_to_f32(f32_to_bf16_bits(f)); }
__device__ __forceinline__ float silu(float f) { return f * sigmoid_fast(f); }

template <int XH, int WH, int R, bool SILU>
__device__ __forceinline__ void linear_tile(const TilesArgs& a, HY_LDS char* lds3, int m0, int n0) {
    const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6), j = lane & 15, hl = lane >> 4, wm = w >> 2, wn = w & 3;
    // rows that are not there are the last one again
    uint32_t xo[XH][2], wo[WH][2];
    const char* const xb = (const char*)(a.x + (int64_t)m0 * a.xs);
    const char* wb[2] = {(const char*)(a.w + (int64_t)n0 * a.ws), (const char*)(a.w + ((int64_t)a.n + n0) * a.ws)};
    if (!SILU) wb[1] = wb[0];
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const int rx = tile_x_load<R>(w, i) * 8 + (lane >> 3), rw = (2 * w + i) * 8 + (lane >> 3);
            if (h < XH) xo[h % XH][i] = (uint32_t)min(h * 32 * R + rx, a.m - 1 - m0) * (uint32_t)(a.xs * 2) + (((lane & 7) ^ tile_swizzle_x(rx)) << 4);
            if (h < WH) wo[h % WH][i] = (uint32_t)min((SILU ? 0 : h * 128) + rw, a.n - 1 - n0) * (uint32_t)(a.ws * 2) + (((lane & 7) ^ tile_swizzle_w(rw)) << 4);
        }
    hy_f32x4 acc[XH][WH][R][2];
    walk_tile<XH, WH, R, false>(lds3, a.k >> 6, [&](int h, int i, int step, uint32_t dst) __attribute__((always_inline)) { load_to_lds16_at(xb + step * 128, xo[h][i], dst); },
        [&](int h, int i, int step, uint32_t dst) __attribute__((always_inline)) { load_to_lds16_at(wb[h] + step * 128, wo[h][i], dst); }, acc);
    const bool wide = a.ys % 8 == 0 && ((uintptr_t)a.y & 15) == 0;
#pragma unroll
    for (int xh = 0; xh < XH; ++xh)
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const int i = m0 + xh * 32 * R + wm * 16 * R + r * 16 + j;
            if (i >= a.m) continue;
            uint16_t* const y = a.y + (int64_t)i * a.ys;
#pragma unroll
            for (int wh = 0; wh < (SILU ? 1 : WH); ++wh) {
                const int n = n0 + wh * 128 + wn * 32 + hl * 8;
                float f[8];
#pragma unroll
                for (int v = 0; v < 8; ++v) {
                    f[v] = acc[xh][wh][r][v >> 2][v & 3];
                    if constexpr (SILU) {
                        const float up = acc[xh][WH - 1][r][v >> 2][v & 3];
                        if (a.round_all) f[v] = rounded(silu(rounded(f[v]))) * rounded(up);
                        else f[v] = silu(f[v]) * up;
                    }
                }
                if (wide && n + 7 < a.n) { *(uint4*)(y + n) = make_uint4(pack2(f[0], f[1]), pack2(f[2], f[3]), pack2(f[4], f[5]), pack2(f[6], f[7])); continue; }
#pragma unroll
                for (int v = 0; v < 8; ++v)
                    if (n + v < a.n) y[n + v] = f32_to_bf16_bits(f[v]);
            }
        }
}

// XH, R: halves of a whole tile and their height.  Whole tiles come first, in blocks of 4 row tiles x all columns, row tiles fastest, cut into
// eight equal runs, one for each XCD: the rows and the weights that neighbouring workgroups read stay in its L2.
template <int XH, int R, bool SILU>
__global__ __launch_bounds__(512) void linear_tiles_kernel(TilesArgs a) {
    extern __shared__ __attribute__((aligned(16))) char lt_lds[];
    HY_LDS char* const lds3 = (HY_LDS char*)lt_lds;
    constexpr int TM = XH * 32 * R, TN = SILU ? 128 : 256;
    const int whole = a.mt * a.nt, share = (whole + 7) / 8;
    int at = blockIdx.x;
    if (at < 8 * share) {
        const int turn = at >> 3;
        at = (at & 7) * share + turn;
        if (at >= whole) return;
        const int blk = at / (4 * a.nt), in = at - blk * 4 * a.nt, high = min(4, a.mt - 4 * blk);
        linear_tile<XH, 2, R, SILU>(a, lds3, (4 * blk + in % high) * TM, in / high * TN);
        return;
    }
    if constexpr (!SILU) {
        at -= 8 * share;
        const int m2 = a.mt * TM, n2 = a.nt * TN, below = max(a.m - m2, 0), cols = (a.n + 127) / 128, under = (below + 127) / 128 * cols;
        if (at < under) { linear_tile<1, 1, 4, false>(a, lds3, m2 + at / cols * 128, at % cols * 128); return; }
        at -= under;
        const int rows = (min(a.m, m2) + 127) / 128, beside = (max(a.n - n2, 0) + 127) / 128;
        if (at < rows * beside) linear_tile<1, 1, 4, false>(a, lds3, at % rows * 128, n2 + at / rows * 128);
    }
}

struct TilesPlan { int mt, nt, tm, blocks; };

// form: tile height (TILES_256, _192, _128, or TILES_SMALL: 128 x 128 everywhere) + TILES_ROWS_APART, + TILES_COLS_APART: rows, columns behind whole tiles
// go in tiles of 128 x 128
constexpr int TILES_256 = 1, TILES_192 = 2, TILES_128 = 3, TILES_SMALL = 4, TILES_HEIGHT = 7, TILES_ROWS_APART = 8, TILES_COLS_APART = 16;

static TilesPlan tiles_layout(int m, int n, int form, bool silu) {
    const int h = form & TILES_HEIGHT, tn = silu ? 128 : 256, tm = h == TILES_128 ? 128 : h == TILES_192 ? 192 : 256;
    int mt = form & TILES_ROWS_APART ? m / tm : (m + tm - 1) / tm, nt = form & TILES_COLS_APART ? n / tn : (n + tn - 1) / tn;
    if (h == TILES_SMALL) mt = nt = 0;
    const int below = m > mt * tm ? (m - mt * tm + 127) / 128 * ((n + 127) / 128) : 0;
    const int beside = n > nt * tn ? ((m < mt * tm ? m : mt * tm) + 127) / 128 * ((n - nt * tn + 127) / 128) : 0;
    return {mt, nt, tm, 8 * ((mt * nt + 7) / 8) + below + beside};
}

// What a launch is taken to need (us): tiles in rounds of one per compute unit, the small ones behind the whole ones, one for each unit that the last round of
// those leaves idle (the dispatcher hands workgroups to shader engines in turn and waits for a busy one) and then in rounds of their own; and, as units
// drift apart and an emptier chip clocks higher, a part of it by work alone.  Fitted to 180 products of 65 .. 24000 rows with 64 .. 34816 outputs
// of 512 .. 17408 k, each in every form: the form it chooses takes 0.8 % longer than the best one on average.
static float tiles_cost(int m, int n, int k, int form, bool silu) {
    constexpr float CUS = 256, BY_WORK = 0.23f;
    const int h = form & TILES_HEIGHT;
    const TilesPlan p = tiles_layout(m, n, form, silu);
    const float steps = (float)(k / 64), big = h == TILES_256 ? 5.5f + 1.21f * steps : h == TILES_192 ? 1.0f + 1.01f * steps : 2.4f + 0.83f * steps, small = 1.0f + 0.49f * steps;
    const float whole = (float)p.mt * p.nt, rest = (float)p.blocks - 8 * ceilf(whole / 8), rounds = ceilf(whole / CUS), behind = rest - (rounds * CUS - whole);
    return (1 - BY_WORK) * (rounds * big + (behind > 0 ? ceilf(behind / CUS) * small : 0)) + BY_WORK * (whole * big + rest * small) / CUS;
}

// the form that is done first, and when
static int tiles_form(int m, int n, int k, bool silu, float* cost) {
    int best = 0;
    for (int form = 1; form < 32; ++form) {
        const int h = form & TILES_HEIGHT;
        if (h < TILES_256 || h > (silu ? TILES_128 : TILES_SMALL) || (form > TILES_HEIGHT && (silu || h == TILES_SMALL))) continue;
        const float c = tiles_cost(m, n, k, form, silu);
        if (!best || c < *cost) { *cost = c; best = form; }
    }
    return best;
}

template <int XH, int R, bool SILU>
static int tiles_launch(const TilesArgs& a, int blocks, hipStream_t s) {
    constexpr int LDS = tile_lds(XH, 2, R) > tile_lds(1, 1) || SILU ? tile_lds(XH, 2, R) : tile_lds(1, 1);
    static bool opted_in[64] = {};
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) dev = -1;
    if (dev < 0 || !opted_in[dev]) {
        hipError_t e = hipFuncSetAttribute((const void*)linear_tiles_kernel<XH, R, SILU>, hipFuncAttributeMaxDynamicSharedMemorySize, LDS);
        if (e != hipSuccess) return (int)e;
        if (dev >= 0) opted_in[dev] = true;
    }
    hipLaunchKernelGGL((linear_tiles_kernel<XH, R, SILU>), dim3(blocks), dim3(512), LDS, s, a);
    return 0;
}

static int tiles_check_and_launch(const char* fn, const TilesArgs& args, int form, bool silu, int dtype, void* stream) {
    TilesArgs a = args;
    if (!a.x || !a.w || !a.y) return fail(TRIMKV_ERR_NULL, "%s: null pointer argument", fn);
    if (dtype != TRIMKV_BF16) return fail(TRIMKV_ERR_DTYPE, "%s: dtype must be bf16 (dtype=%d)", fn, dtype);
    if (a.m <= 0 || a.n <= 0 || a.k <= 0 || a.k % 64 || a.m > (1 << 24) || a.n > (1 << 24) || a.xs < a.k || a.ws < a.k || a.xs > (1 << 20) || a.ws > (1 << 20) || a.xs % 8 || a.ws % 8 || a.ys < a.n)
        return fail(TRIMKV_ERR_SHAPE, "%s: bad sizes rows=%d n=%d k=%d strides %lld %lld %lld", fn, a.m, a.n, a.k, (long long)a.xs, (long long)a.ws, (long long)a.ys);
    if (((uintptr_t)a.x | (uintptr_t)a.w) & 15) return fail(TRIMKV_ERR_SHAPE, "%s: x and w must be 16-byte aligned", fn);
    if (form < 0 || form >= 32 || (form && (form & TILES_HEIGHT) < 1) || (form & TILES_HEIGHT) > (silu ? TILES_128 : TILES_SMALL) || (silu && form > TILES_HEIGHT)) return fail(TRIMKV_ERR_SHAPE, "%s: no form %d", fn, form);
    float cost;
    if (!form) form = tiles_form(a.m, a.n, a.k, silu, &cost);
    const TilesPlan p = tiles_layout(a.m, a.n, form, silu);
    a.mt = p.mt; a.nt = p.nt;
    hipStream_t s = (hipStream_t)stream;
    const int rc = p.tm == 128 ? silu ? tiles_launch<1, 4, true>(a, p.blocks, s) : tiles_launch<1, 4, false>(a, p.blocks, s)
                 : p.tm == 192 ? silu ? tiles_launch<2, 3, true>(a, p.blocks, s) : tiles_launch<2, 3, false>(a, p.blocks, s)
                               : silu ? tiles_launch<2, 4, true>(a, p.blocks, s) : tiles_launch<2, 4, false>(a, p.blocks, s);
    if (rc) return fail(rc, "%s: hipFuncSetAttribute failed (%d)", fn, rc);
    return launch_status(fn);
}

}  // namespace trimkv

using namespace trimkv;

extern "C" int trimkv_linear_tiles(const void* x, int64_t x_stride, const void* w, int64_t w_stride, void* out, int64_t out_stride, int rows, int n, int k, int form,
                                   int dtype, void* stream) {
    return tiles_check_and_launch("trimkv_linear_tiles", {(const uint16_t*)x, x_stride, (const uint16_t*)w, w_stride, (uint16_t*)out, out_stride, rows, n, k, 0}, form, false, dtype, stream);
}

extern "C" int trimkv_linear_tiles_silu(const void* x, int64_t x_stride, const void* w, int64_t w_stride, void* out, int64_t out_stride, int rows, int inter, int k,
                                        int round_all, int form, int dtype, void* stream) {
    return tiles_check_and_launch("trimkv_linear_tiles_silu", {(const uint16_t*)x, x_stride, (const uint16_t*)w, w_stride, (uint16_t*)out, out_stride, rows, inter, k, round_all}, form, true, dtype, stream);
}

// Products that the tiles take at less than RATE (by the estimate) have too few of them to fill the chip.  The vendor's library divides long k where outputs are
// few, so that the line is higher there.  Of 930 products of 70 .. 10000 rows, 512 .. 151936 outputs and k up to 17408: above the line 480, 1.14 times as fast on
// average, 29 of them slower by 3 % and more (15 by 8 %); with silu, a launch less, 415, 1.15, 14 (3).  Between RATE for short k and for long, where
// k is longer than 2048: 164, 0.98, 90; with silu 38, 0.93, 29.  us here | general (rows x n x k): 82 x 2048 x 2048 16 | 8, 613 x 4112 x 2048 20 | 21, 2252 x
// 4112 x 2048 35 | 43, 8286 x 6144 x 2048 164 | 230, 8286 x 2048 x 2048 64 | 69, 680 x 6144 x 4096 50 | 46, 1599 x 3072 x 8192 94 | 77, 1656 x
// 4096 x 4096 52 | 56, 8192 x 6176 x 4096 293 | 380, 8192 x 4096 x 4096 180 | 178, 8192 x 4096 x 12288 521 | 521; with silu 177 rows of 12288 x
// 2048 27 | 27, 412 29 | 34, 206 of 8192 x 3072 43 | 36, 8192 of 12288 x 4096 1058 | 1140.
extern "C" int trimkv_linear_tiles_form(int rows, int n, int k, int silu) {
    const float rate = k <= 2048 ? (silu ? 0.55e9f : 0.65e9f) : silu ? 0.8e9f : 1.0e9f;      // RATE: operations per us
    if (rows <= 0 || n <= 0 || k < 64) return 0;
    float cost;
    const int form = tiles_form(rows, n, k, silu != 0, &cost);
    return 2.0f * rows * n * k * (silu ? 2 : 1) >= rate * cost ? form : 0;
}

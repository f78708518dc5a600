// Tiles of a bf16 product x w^T on the matrix cores -- gfx950.
#pragma once

#include "hybrid.hip.h"

namespace trimkv {

// A workgroup of 8 wavefronts multiplies XH halves of 32 R rows of x (R = 4 or 3) with WH halves of 128 rows of w ("outputs") in steps of 64 k,
// which rotate through tile_buffers() LDS buffers filled by LDS-direct loads.  In a buffer, half h of x (4 R KiB) lies at h 4 R KiB,
// half h of w (16 KiB) behind those of x.
//
// A step has XH WH phases, one for each pair of halves, and each phase two parts: reading the fragments that it needs (and
// requesting as much of a later step), then 4 R products of 16x16x32 per wavefront.  The wavefronts of the first 16 R rows of a half and
// those of the others, one of each on every SIMD, are half a phase apart: while one multiplies, the other reads.  The
// barrier between the parts keeps them so, and with it the matrix cores never wait for LDS (16 fragments of 1 KiB are 4 x 8 KiB
// or 256 of a compute unit's cycles, as long as the products take); it also guards the buffers: what a part has read is requested anew
// two parts later at the earliest, what it reads has landed in the whole workgroup two parts before.
//
// 16x16x32 and not 32x32x16: the same schedule with 32x32x16 reached 1.15 against 1.36 PFLOP/s (8192 x 8192 x 8192).  Fragments of the first half of
// w read a phase ahead: 1.37 -> 1.44 at 32768 x 4608 x 4096 (12, 4, 8 and no fragments of a phase become 8, 4, 8 and 4).  A barrier before the last two or four products of a
// phase instead of behind them: 1.33.
constexpr int tile_buffers(int xh, int wh) { return xh + wh == 4 ? 2 : xh + wh == 3 ? 3 : 4; }
constexpr int tile_lds(int xh, int wh, int r = 4) { return tile_buffers(xh, wh) * (xh * r * 4096 + wh * 16384); }

// Where a fragment's outputs lie among the 32 of a wavefront: fragment c, MFMA row i <-> output 8 (i / 4) + 4 c + i % 4, so that a lane's
// accumulators of both fragments are eight outputs in a row.
__device__ __forceinline__ int tile_output(int c, int i) { return 8 * (i >> 2) + 4 * c + (i & 3); }

// The 16-byte pieces of row r (8 of them) lie at piece ^ tile_swizzle: rows r .. r + 15 of x, and the rows that a fragment of w takes, read at
// one piece fall on different banks.
__device__ __forceinline__ int tile_swizzle_x(int r) { return (r >> 1) & 7; }
__device__ __forceinline__ int tile_swizzle_w(int r) { return ((r >> 1) & 1) | (((r >> 3) & 3) << 1); }
// w in blocks of 32 outputs x 16 k (two halves of 8 k): place p of a block in LDS is taken from this place in memory
__device__ __forceinline__ int tile_packed_source(int p) { return (p & 32) + tile_output((p >> 4) & 1, p & 15); }

// KiB (8 rows) of a half of x that wavefront w requests as its load i; of 12 KiB the last wavefronts request one twice
template <int R> __device__ __forceinline__ int tile_x_load(int w, int i) { return R == 4 ? 2 * w + i : i && w < 4 ? 8 + w : w; }

__device__ __forceinline__ void tile_meet() {
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_barrier" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
}
// meet when this wavefront's fragments have been read and all but its last N requests have landed
template <int N> __device__ __forceinline__ void tile_meet_landed() {
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" :: "n"(N) : "memory");
    __builtin_amdgcn_sched_barrier(0);
}

// acc[xh][wh][r][c][v]: row 32 R xh + 16 R (w / 4) + 16 r + lane % 16, output 128 wh + 32 (w % 4) + 8 (lane / 16) + 4 c + v for wavefront w.
// request_x(h, i, step, lds_addr), request_w(...): the wavefront's LDS-direct load i (of 2) of half h of that step: 1 KiB each, of x KiB tile_x_load<R>(w, i)
// of the half, of w KiB 2 w + i; x and row-major w: 8 rows of 128 bytes; packed w: block 2 w + i, of 32 outputs x 16 k (outputs
// 32 ((2 w + i) / 4), k 16 ((2 w + i) % 4)).
template <int XH, int WH, int R, bool PACKED, class RequestX, class RequestW>
__device__ __forceinline__ void walk_tile(HY_LDS char* lds3, int steps, RequestX request_x, RequestW request_w, hy_f32x4 (&acc)[XH][WH][R][2]) {
    constexpr int B = tile_buffers(XH, WH), HALF = R * 4096, XB = XH * HALF, BUF = XB + WH * 16384;
    const uint32_t lds0 = (uint32_t)(uintptr_t)lds3;
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), j = lane & 15, hl = lane >> 4, wm = w >> 2, wn = w & 3;
    auto x_of = [&](int step, int buf, int h) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 2; ++i) request_x(h, i, min(step, steps - 1), lds0 + buf * BUF + h * HALF + tile_x_load<R>(w, i) * 1024);      // past the end: read again, never used
    };
    auto w_of = [&](int step, int buf, int h) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 2; ++i) request_w(h, i, min(step, steps - 1), lds0 + buf * BUF + XB + h * 16384 + (2 * w + i) * 1024);
    };
#pragma unroll
    for (int xh = 0; xh < XH; ++xh)
#pragma unroll
        for (int wh = 0; wh < WH; ++wh)
#pragma unroll
            for (int i = 0; i < 2 * R; ++i) acc[xh][wh][i >> 1][i & 1] = hy_f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    hy_bf16x8 xf[R][2], wf[3][2][2];
    HY_LDS char* const xr = lds3 + (wm * 16 * R + j) * 128;
    HY_LDS char* const wr = lds3 + XB + (PACKED ? wn * 4096 + (hl >> 1) * 1024 + (hl & 1) * 512 + j * 16 : (wn * 32 + tile_output(0, j)) * 128);
    const int xsw = tile_swizzle_x(j), wsw = tile_swizzle_w(tile_output(0, j));
    auto read_x = [&](int buf, int h) __attribute__((always_inline)) {
#pragma unroll
        for (int r = 0; r < R; ++r)
#pragma unroll
            for (int q = 0; q < 2; ++q) xf[r][q] = *(const HY_LDS hy_bf16x8*)(xr + buf * BUF + h * HALF + r * 2048 + (((4 * q + hl) ^ xsw) << 4));
    };
    auto read_w = [&](int buf, int h, int to) __attribute__((always_inline)) {
#pragma unroll
        for (int c = 0; c < 2; ++c)
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                if (PACKED) wf[to][c][q] = *(const HY_LDS hy_bf16x8*)(wr + buf * BUF + h * 16384 + q * 2048 + c * 256);
                else wf[to][c][q] = *(const HY_LDS hy_bf16x8*)(wr + buf * BUF + h * 16384 + c * 512 + (((4 * q + hl) ^ wsw) << 4));
            }
    };
    auto multiply = [&](int xh, int wh, int from) __attribute__((always_inline)) {
        __builtin_amdgcn_s_setprio(1);
#pragma unroll
        for (int i = 0; i < 4 * R; ++i) {
            const int q = i / (2 * R), r = i / 2 % R, c = i & 1;
            acc[xh][wh][r][c] = mfma16(wf[from][c][q], xf[r][q], acc[xh][wh][r][c]);
        }
        __builtin_amdgcn_s_setprio(0);
        tile_meet();
    };
    int buf = 0, last = B - 1;                      // of this step and of the one before
    auto turn = [&]() __attribute__((always_inline)) { last = buf; buf = buf == B - 1 ? 0 : buf + 1; };
    auto next = [&]() __attribute__((always_inline)) { return buf == B - 1 ? 0 : buf + 1; };
    // The first half of w is read a phase ahead where there are two, into another place than the present one's
    auto step = [&](int s, int here, int there) __attribute__((always_inline)) {
        if constexpr (XH == 2 && WH == 2) {
            constexpr int N = 12;
            read_x(buf, 0); w_of(s + B, buf, 0);
            tile_meet_landed<N>(); multiply(0, 0, here);
            read_w(buf, 1, 1); x_of(s + B, buf, 0);
            tile_meet_landed<N>(); multiply(0, 1, 1);
            read_x(buf, 1); w_of(s + B, buf, 1);
            tile_meet_landed<N>(); multiply(1, 1, 1);
            read_w(next(), 0, there); x_of(s + B, buf, 1);
            tile_meet_landed<N>(); multiply(1, 0, here);
        } else if constexpr (WH == 2) {
            constexpr int N = 6 * (B - 1);
            read_x(buf, 0); w_of(s + B - 1, last, 1); w_of(s + B, buf, 0);
            tile_meet_landed<N>(); multiply(0, 0, here);
            read_w(buf, 1, 1); read_w(next(), 0, there); x_of(s + B, buf, 0);
            tile_meet_landed<N>(); multiply(0, 1, 1);
        } else {
            constexpr int N = 4 * (B - 2);
            read_x(buf, 0); read_w(buf, 0, 0); x_of(s + B - 1, last, 0); w_of(s + B - 1, last, 0);
            tile_meet_landed<N>(); multiply(0, 0, 0);
        }
        turn();
    };
    // requested here, in the order in which the steps wait for them: what the steps up to the first one's turn do not request
    if constexpr (XH == 2 && WH == 2) {
#pragma unroll
        for (int p = 0; p < B; ++p) { w_of(p, p, 0); x_of(p, p, 0); w_of(p, p, 1); x_of(p, p, 1); }
        asm volatile("s_waitcnt vmcnt(12)" ::: "memory");
    } else if constexpr (WH == 2) {
#pragma unroll
        for (int p = 0; p < B; ++p) { if (p) w_of(p - 1, p - 1, 1); w_of(p, p, 0); x_of(p, p, 0); }
        asm volatile("s_waitcnt vmcnt(%0)" :: "n"(6 * (B - 1)) : "memory");
    } else {
#pragma unroll
        for (int p = 0; p + 1 < B; ++p) { x_of(p, p, 0); w_of(p, p, 0); }
        asm volatile("s_waitcnt vmcnt(%0)" :: "n"(4 * (B - 2)) : "memory");
    }
    tile_meet();
    if constexpr (WH == 2) {
        read_w(0, 0, 0);
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        tile_meet();                               // the first step requests this half anew
    }
    if (wm) tile_meet();                           // half a phase behind from here on
    int s = 0;
    for (; s + 1 < steps; s += 2) { step(s, 0, 2); step(s + 1, 2, 0); }
    if (s < steps) step(s, 0, 2);
    if (!wm) tile_meet();
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");       // nothing may land in LDS after the workgroup has gone
}

}  // namespace trimkv

// Mixture of experts with squared-ReLU experts -- gfx950.
//
//   trimkv_moe_route   sigmoid scores, choice scores with a correction, groups of neighbouring experts of which the best are
//                      open (a group's score: its two largest choice scores), top-k; weights are the plain scores
//   trimkv_moe_plan    (token, choice) rows ordered by expert, and the list of row tiles of the grouped products
//   trimkv_moe_gemm    one product per expert over its rows: up (rows gathered by token, squared ReLU) or down (rows
//                      scattered back to (token, choice) order)
//
// Expert weights are stored in the order in which the matrix cores take them: blocks of 32 outputs x 16 k, in a block first
// k 0..7 of the 32 outputs, then k 8..15 (lane l of a wavefront: output l % 32, k 8 (l / 32) .. + 7), so that a load
// instruction reads 1 KiB in one piece: [E][n padded / 32][k padded / 16][2][32][8].  n and k are padded with zeros to
// multiples of 64, activations are rows of k padded elements: no kernel has a tail along k.
#include "tiles.hip.h"
#include <algorithm>
#include <type_traits>

namespace trimkv {

constexpr int ROUTE_MAX_E = 1024;

// NE: 64-expert slices, rounded up
template <int NE>
__global__ __launch_bounds__(256) void route_kernel(const float* z, const float* correction, int32_t* ids, float* weights, int tokens, int E, int top, int count, int keep) {
    extern __shared__ float rt[];                 // per wavefront: choice [E], group [count]
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int t = blockIdx.x * 4 + w;
    float* choice = rt + w * (E + count);
    float* group = choice + E;
    const bool live = t < tokens;
    const float* zr = z + (int64_t)min(t, tokens - 1) * E;
    for (int e = lane; e < E; e += 64) choice[e] = sigmoid_f(zr[e]) + correction[e];
    __syncthreads();
    const int per = E / count;
    for (int g = lane; g < count; g += 64) {
        float a = -INFINITY, b = -INFINITY;
        for (int e = g * per; e < (g + 1) * per; ++e) {
            const float c = choice[e];
            if (c > a) { b = a; a = c; } else if (c > b) b = c;
        }
        group[g] = per > 1 ? a + b : a;
    }
    __syncthreads();
    float c[NE];
#pragma unroll
    for (int i = 0; i < NE; ++i) {
        const int e = i * 64 + lane;
        c[i] = -INFINITY;
        if (e < E) {
            const int g = e / per;
            int better = 0;
            for (int o = 0; o < count; ++o) better += group[o] > group[g] || (group[o] == group[g] && o < g);
            if (better < keep) c[i] = choice[e];
        }
    }
    for (int j = 0; j < top; ++j) {
        float best = -INFINITY;
        int at = 0x7fffffff;
#pragma unroll
        for (int i = 0; i < NE; ++i)
            if (c[i] > best) { best = c[i]; at = i * 64 + lane; }
#pragma unroll
        for (int d = 32; d > 0; d >>= 1) {
            const float bo = __shfl_xor(best, d, 64);
            const int ao = __shfl_xor(at, d, 64);
            if (bo > best || (bo == best && ao < at)) { best = bo; at = ao; }
        }
        at = min(at, E - 1);                      // non-finite logits: stay in bounds
#pragma unroll
        for (int i = 0; i < NE; ++i)
            if (i * 64 + lane == at) c[i] = -INFINITY;
        if (live && lane == 0) {
            ids[(int64_t)t * top + j] = at;
            weights[(int64_t)t * top + j] = sigmoid_f(zr[at]);
        }
    }
}

// Every workgroup counts all rows in LDS, those in front of its own apart, and scatters its own 2048 or more.  Bound by the LDS atomics of the
// count and, with one workgroup, by the scattered stores of a single compute unit: 32768 rows of 32 experts 17.0 us with one, 7.1 with
// sixteen, 8192 of 128 7.6 and 5.0, 524288 325 and 67.
constexpr int PLAN_CHUNK = 2048, PLAN_MOST = 16;
__global__ __launch_bounds__(1024) void plan_kernel(const int32_t* ids, int rows, int E, int tile, int32_t* order, int32_t* offsets, int32_t* tiles) {
    extern __shared__ int32_t pl[];               // of an expert: rows in front of this workgroup's [E], its others [E]; then first row, first tile
    int32_t* cursor = pl; int32_t* tcur = pl + E;
    const int tid = threadIdx.x, per = (rows + gridDim.x - 1) / gridDim.x, mine = blockIdx.x * per, end = min(rows, mine + per);
    for (int e = tid; e < 2 * E; e += 1024) pl[e] = 0;
    __syncthreads();
    auto each = [&](int from, int to, auto&& f) __attribute__((always_inline)) {
        auto some = [&](auto count) __attribute__((always_inline)) {      // so many experts requested together
            constexpr int U = decltype(count)::value;
            for (int i0 = from + tid; i0 < to; i0 += U * 1024) {
                int id[U];
#pragma unroll
                for (int u = 0; u < U; ++u) id[u] = ids[min(i0 + u * 1024, to - 1)];
#pragma unroll
                for (int u = 0; u < U; ++u)
                    if (i0 + u * 1024 < to) f(i0 + u * 1024, id[u]);
            }
        };
        if (to - from <= 2048) some(std::integral_constant<int, 2>{});      // 2048 rows: eight each, of which six are none, take 4.2 us for 3.7
        else some(std::integral_constant<int, 8>{});
    };
    each(0, rows, [&](int i, int e) __attribute__((always_inline)) { atomicAdd(&pl[i < mine ? e : E + e], 1); });
    __syncthreads();
    if (tid < 64) {                               // exclusive sums over experts, 64 at a time
        int base = 0, tbase = 0;
        for (int e0 = 0; e0 < E; e0 += 64) {
            const int e = e0 + tid, front = e < E ? cursor[e] : 0, c = e < E ? front + tcur[e] : 0, nt = (c + tile - 1) / tile;
            int s = c, ts = nt;
#pragma unroll
            for (int d = 1; d < 64; d <<= 1) {
                const int o = __shfl_up(s, d, 64), to = __shfl_up(ts, d, 64);
                if (tid >= d) { s += o; ts += to; }
            }
            if (e < E) {
                cursor[e] = base + s - c + front;
                tcur[e] = tbase + ts - nt;
                if (blockIdx.x == 0) offsets[e] = base + s - c;
            }
            base += __shfl(s, 63, 64);
            tbase += __shfl(ts, 63, 64);
        }
        if (blockIdx.x == 0 && tid == 0) { offsets[E] = base; tiles[0] = tbase; }
    }
    __syncthreads();
    // tiles[1 + 2 i] = expert, tiles[2 + 2 i] = first row of tile i; workgroup 0 has no rows in front of its own
    if (blockIdx.x == 0) {
        for (int e = tid; e < E; e += 1024) {
            const int first = cursor[e], c = (e + 1 < E ? cursor[e + 1] : rows) - first;
            for (int x = 0; x * tile < c; ++x) {
                const int i = tcur[e] + x;
                tiles[1 + 2 * i] = e;
                tiles[2 + 2 * i] = first + x * tile;
            }
        }
        __syncthreads();
    }
    each(mine, end, [&](int i, int e) __attribute__((always_inline)) { order[atomicAdd(&cursor[e], 1)] = i; });
}

struct GroupedArgs {
    const void* x; int64_t xs;                    // activations; up: row = order[i] / top, down: row = i
    const void* w;                                // [E][np][kp]
    void* y; int64_t ys;                          // up: row i; down: row order[i]
    const int32_t* order; const int32_t* offsets; const int32_t* tiles;
    int top, n, np, kp;
};
// squared ReLU of the up product; the down product passes
template <bool UP> __device__ __forceinline__ float expert_act(float f) { return UP ? (f > 0.0f ? f * f : 0.0f) : f; }

// element (n, k) of an expert's matrix
__device__ __forceinline__ int64_t packed_at(int n, int k, int kp) { return ((int64_t)(n >> 5) * (kp >> 4) + (k >> 4)) * 512 + ((k >> 3) & 1) * 256 + (n & 31) * 8 + (k & 7); }

// fp32: 16 rows x 64 outputs per workgroup.
template <bool UP>
__global__ __launch_bounds__(256) void grouped_f32_kernel(GroupedArgs a) {
    __shared__ float xs[16][17];
    __shared__ float wsm[64][17];
    if ((int)blockIdx.x >= a.tiles[0]) return;
    const int e = a.tiles[1 + 2 * blockIdx.x], m0 = a.tiles[2 + 2 * blockIdx.x], mend = a.offsets[e + 1];
    const int tid = threadIdx.x, n0 = blockIdx.y * 64;
    const int tn = tid & 63, tm = tid >> 6;
    const float* w = (const float*)a.w + (int64_t)e * a.np * a.kp;
    float acc[4] = {0.f, 0.f, 0.f, 0.f};
    for (int k0 = 0; k0 < a.kp; k0 += 16) {
        {
            const int r = tid >> 4, c = tid & 15, i = min(m0 + r, mend - 1);
            const int64_t row = UP ? a.order[i] / a.top : i;
            xs[r][c] = ((const float*)a.x)[row * a.xs + k0 + c];
        }
        for (int x = tid; x < 1024; x += 256) wsm[x >> 4][x & 15] = w[packed_at(n0 + (x >> 4), k0 + (x & 15), a.kp)];
        __syncthreads();
#pragma unroll
        for (int c = 0; c < 16; ++c)
#pragma unroll
            for (int y = 0; y < 4; ++y) acc[y] = fmaf(xs[tm * 4 + y][c], wsm[tn][c], acc[y]);
        __syncthreads();
    }
#pragma unroll
    for (int y = 0; y < 4; ++y) {
        const int i = m0 + tm * 4 + y;
        if (i < mend && n0 + tn < a.n) ((float*)a.y)[(UP ? (int64_t)i : (int64_t)a.order[i]) * a.ys + n0 + tn] = expert_act<UP>(acc[y]);
    }
}

// four consecutive outputs from n on
template <bool UP>
__device__ __forceinline__ void store_outputs(const GroupedArgs& a, uint16_t* yr, int n, float f0, float f1, float f2, float f3) {
    f0 = expert_act<UP>(f0); f1 = expert_act<UP>(f1); f2 = expert_act<UP>(f2); f3 = expert_act<UP>(f3);
    if (n + 3 < a.n && a.ys % 4 == 0) { *(uint2*)(yr + n) = make_uint2(pack2(f0, f1), pack2(f2, f3)); return; }
    if (n < a.n) yr[n] = f32_to_bf16_bits(f0);
    if (n + 1 < a.n) yr[n + 1] = f32_to_bf16_bits(f1);
    if (n + 2 < a.n) yr[n + 2] = f32_to_bf16_bits(f2);
    if (n + 3 < a.n) yr[n + 3] = f32_to_bf16_bits(f3);
}

// bf16, a handful of rows per expert (decode): 32 rows x 32 outputs per workgroup, whose KS wavefronts share the k of them;
// operands straight from memory.  The launch is bound by the stream of weights; UNROLL loads of them are in flight per lane.
template <bool UP, int KS>
__global__ __launch_bounds__(KS * 64) void grouped_skinny_kernel(GroupedArgs a) {
    constexpr int UNROLL = 8;
    __shared__ hy_f32x4 part[KS - 1][4][64];
    if ((int)blockIdx.x >= a.tiles[0]) return;
    const int e = a.tiles[1 + 2 * blockIdx.x], m0 = a.tiles[2 + 2 * blockIdx.x], mend = a.offsets[e + 1];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, j = lane & 31, hl = lane >> 5;
    const int nb = blockIdx.y, kb16 = a.kp >> 4, span = (kb16 + KS - 1) / KS, s0 = w * span, s1 = min(kb16, s0 + span);
    const int i = min(m0 + j, mend - 1);
    const uint16_t* xr = (const uint16_t*)a.x + (UP ? (int64_t)(a.order[i] / a.top) : (int64_t)i) * a.xs + hl * 8;
    const uint16_t* wr = (const uint16_t*)a.w + ((int64_t)e * (a.np >> 5) + nb) * kb16 * 512 + lane * 8;
    hy_f32x16 acc;
#pragma unroll
    for (int v = 0; v < 16; ++v) acc[v] = 0.0f;
    for (int s = s0; s < s1; s += UNROLL) {
        hy_u32x4 wf[UNROLL], xf[UNROLL];
#pragma unroll
        for (int u = 0; u < UNROLL; ++u) wf[u] = __builtin_nontemporal_load((const hy_u32x4*)(wr + (int64_t)min(s + u, s1 - 1) * 512));
#pragma unroll
        for (int u = 0; u < UNROLL; ++u) {
            xf[u] = *(const hy_u32x4*)(xr + min(s + u, s1 - 1) * 16);
            if (s + u >= s1) xf[u] = hy_u32x4{0u, 0u, 0u, 0u};
        }
#pragma unroll
        for (int u = 0; u < UNROLL; ++u) acc = mfma32(__builtin_bit_cast(hy_bf16x8, wf[u]), __builtin_bit_cast(hy_bf16x8, xf[u]), acc);
    }
    if (w) {
#pragma unroll
        for (int c = 0; c < 4; ++c) part[w - 1][c][lane] = hy_f32x4{acc[4 * c], acc[4 * c + 1], acc[4 * c + 2], acc[4 * c + 3]};
    }
    __syncthreads();
    if (w || m0 + j >= mend) return;
    // lane holds outputs 32 nb + 8 (v / 4) + 4 hl + v % 4 of row j
    uint16_t* y = (uint16_t*)a.y + (UP ? (int64_t)(m0 + j) : (int64_t)a.order[m0 + j]) * a.ys;
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        hy_f32x4 f = {acc[4 * c], acc[4 * c + 1], acc[4 * c + 2], acc[4 * c + 3]};
#pragma unroll
        for (int x = 0; x < KS - 1; ++x) f += part[x][c][lane];
        store_outputs<UP>(a, y, nb * 32 + 8 * c + 4 * hl, f[0], f[1], f[2], f[3]);
    }
}

// bf16, more than a few rows per expert (prompts): 256 rows x 256 outputs per workgroup (tiles.hip.h), or 192 or 128 rows of the
// last tile of an expert that holds no more.  It is bound by the matrix cores at the clock that they leave the chip (1.7 GHz): 8192 tokens x 4 of 32
// experts of 4096 x 4608 take 875 us where every expert has 1024 rows (1.42 PFLOP/s; rows in any order, the gather costs nothing) and 1020 where
// counts differ by a factor of 4 (143 row tiles, 32 of them part empty: 870 us of work for 256 compute units; the rest are units that wait
// for the next workgroup of their shader engine, 5 %, and the last tiles, 6 %).
// With the tiles that are not full last, as the shorter work to end on, the same took 1158: each of them reads its expert's weights
// alone then, 2 MB of w for 128 rows, and 128 rows last 87 us instead of 61.  A kernel that fed 32x32x16 products from five
// buffers of 32 k, all wavefronts in step, took 1300.
template <bool UP>
__global__ __launch_bounds__(512) void grouped_big_kernel(GroupedArgs a, int n_tiles, int experts) {
    extern __shared__ __attribute__((aligned(16))) char gb_lds[];
    HY_LDS char* const lds3 = (HY_LDS char*)gb_lds;
    const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6), j = lane & 15, hl = lane >> 4, wm = w >> 2, wn = w & 3;
    // The tiles of an expert stay together, for the weights that they share in an XCD's L2: in blocks of up to 4 of them x all columns of outputs,
    // row tiles fastest.  The whole is cut at columns of blocks into eight runs, one for each XCD, that cost the same: 6, 5 and 4
    // for a tile of 256, 192 and 128 rows (90, 74 and 61 us at 4096 k).  Equal numbers of tiles instead: 1107 us for 1020.
    int e = 0, m0 = 0, nt = 0;
    {
        auto cost_of = [](int c) __attribute__((always_inline)) { const int p = c & 255; return 6 * (c >> 8) + (p > 192 ? 6 : p > 128 ? 5 : p ? 4 : 0); };
        const int c0 = lane < experts ? a.offsets[lane + 1] - a.offsets[lane] : 0;
        auto rows_of = [&](int e0) __attribute__((always_inline)) { return e0 == 0 ? c0 : e0 + lane < experts ? a.offsets[e0 + lane + 1] - a.offsets[e0 + lane] : 0; };
        auto scan = [&](int v) __attribute__((always_inline)) {
#pragma unroll
            for (int d = 1; d < 64; d <<= 1) { const int o = __shfl_up(v, d, 64); if (lane >= d) v += o; }
            return v;
        };
        int total = 0;
        for (int e0 = 0; e0 < experts; e0 += 64) total += __builtin_amdgcn_readlane(scan(cost_of(rows_of(e0))), 63);
        const int xcd = blockIdx.x & 7, k = blockIdx.x >> 3;
        int from = 0, until = 0, found = 0;
        for (int end = 0; end < 2; ++end) {
            const int t = (int)((int64_t)total * n_tiles * (xcd + end) / 8);
            int cost = 0, tiles = 0, at = -1;
            for (int e0 = 0; e0 < experts && at < 0; e0 += 64) {
                const int c = rows_of(e0), mine = cost_of(c), n = (c + 255) >> 8, cs = cost + scan(mine), ts = tiles + scan(n);
                const unsigned long long in = __ballot(cs * n_tiles > t);
                if (in) {
                    const int l = __builtin_ctzll(in), of = __builtin_amdgcn_readlane(n, l), whole = __builtin_amdgcn_readlane(mine, l);
                    int rest = t - (__builtin_amdgcn_readlane(cs, l) - whole) * n_tiles;
                    const int b = rest / (24 * n_tiles), high = min(4, of - 4 * b);
                    rest -= b * 24 * n_tiles;
                    at = (__builtin_amdgcn_readlane(ts, l) - of + 4 * b) * n_tiles + rest / min(24, whole - 24 * b) * high;
                }
                cost = __builtin_amdgcn_readlane(cs, 63);
                tiles = __builtin_amdgcn_readlane(ts, 63);
            }
            (end ? until : from) = at < 0 ? tiles * n_tiles : at;
        }
        const int at = from + k;
        if (at >= until) return;
        int tiles = 0;
        for (int e0 = 0; e0 < experts && !found; e0 += 64) {
            const int n = (rows_of(e0) + 255) >> 8, ts = tiles + scan(n);
            const unsigned long long in = __ballot(ts * n_tiles > at);
            if (in) {
                const int l = __builtin_ctzll(in), of = __builtin_amdgcn_readlane(n, l), i = at - (__builtin_amdgcn_readlane(ts, l) - of) * n_tiles;
                const int b = i / (4 * n_tiles), j = i - b * 4 * n_tiles, high = min(4, of - 4 * b);
                nt = j / high;
                e = e0 + l;
                m0 = a.offsets[e] + (4 * b + j % high) * 256;
                found = 1;
            }
            tiles = __builtin_amdgcn_readlane(ts, 63);
        }
    }
    const int rows = __builtin_amdgcn_readfirstlane(a.offsets[e + 1] - m0), n0 = nt * 256, kb16 = a.kp >> 4;
    HY_LDS int32_t* const to = (HY_LDS int32_t*)(lds3 + tile_lds(1, 2));      // rows of y; the barriers of the walk lie between here and the stores
    if (!UP && tid < 256) to[tid] = a.order[m0 + min(tid, rows - 1)];
    const uint32_t source = tile_packed_source(lane) * 16;
    const int nb0 = n0 >> 5, nbs = a.np >> 5;
    const char* const wb = (const char*)a.w + (int64_t)e * nbs * kb16 * 1024;
    auto go = [&](auto halves, auto blocks) __attribute__((always_inline)) {
        constexpr int XH = decltype(halves)::value, R = decltype(blocks)::value;
        const uint16_t* xp[XH][2];
#pragma unroll
        for (int h = 0; h < XH; ++h)
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const int r = h * 32 * R + tile_x_load<R>(w, i) * 8 + (lane >> 3), x = m0 + min(r, rows - 1);
                xp[h][i] = (const uint16_t*)a.x + (UP ? (int64_t)(a.order[x] / a.top) : (int64_t)x) * a.xs + (((lane & 7) ^ tile_swizzle_x(r)) << 3);
            }
        hy_f32x4 acc[XH][2][R][2];
        walk_tile<XH, 2, R, true>(lds3, a.kp >> 6, [&](int h, int i, int step, uint32_t dst) __attribute__((always_inline)) { load_to_lds16(xp[h][i] + step * 64, dst); },
            [&](int h, int i, int step, uint32_t dst) __attribute__((always_inline)) {
                const int b = 2 * w + i, nb = min(nb0 + h * 4 + (b >> 2), nbs - 1);
                load_to_lds16_at(wb + ((int64_t)nb * kb16 + step * 4 + (b & 3)) * 1024, source, dst);
            }, acc);
#pragma unroll
        for (int xh = 0; xh < XH; ++xh)
#pragma unroll
            for (int r = 0; r < R; ++r) {
                const int i = xh * 32 * R + wm * 16 * R + r * 16 + j;
                if (i >= rows) continue;
                uint16_t* const y = (uint16_t*)a.y + (UP ? (int64_t)(m0 + i) : (int64_t)to[i]) * a.ys;
#pragma unroll
                for (int wh = 0; wh < 2; ++wh) {
                    const int n = n0 + wh * 128 + wn * 32 + hl * 8;
                    float f[8];
#pragma unroll
                    for (int v = 0; v < 8; ++v) f[v] = expert_act<UP>(acc[xh][wh][r][v >> 2][v & 3]);
                    if (n + 7 < a.n && a.ys % 8 == 0) { *(uint4*)(y + n) = make_uint4(pack2(f[0], f[1]), pack2(f[2], f[3]), pack2(f[4], f[5]), pack2(f[6], f[7])); continue; }
#pragma unroll
                    for (int v = 0; v < 8; ++v)
                        if (n + v < a.n) y[n + v] = f32_to_bf16_bits(f[v]);
                }
            }
    };
    const std::integral_constant<int, 1> one; const std::integral_constant<int, 2> two; const std::integral_constant<int, 3> three; const std::integral_constant<int, 4> four;
    if (rows > 192) go(two, four);
    else if (rows > 128) go(two, three);
    else go(one, four);
}

template <bool UP>
static int launch_big(const GroupedArgs& a, int rows, int experts, hipStream_t s) {
    constexpr int LDS = tile_lds(1, 2) + 1024;
    static_assert(tile_lds(2, 2) <= tile_lds(1, 2) && LDS <= 163840, "both forms fit");
    static bool opted_in[64] = {};
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) dev = -1;
    if (dev < 0 || !opted_in[dev]) {
        hipError_t e = hipFuncSetAttribute((const void*)grouped_big_kernel<UP>, hipFuncAttributeMaxDynamicSharedMemorySize, LDS);
        if (e != hipSuccess) return (int)e;
        if (dev >= 0) opted_in[dev] = true;
    }
    // A run has no more workgroups than its cost / 4 and the tiles of a column; the cost of all is at most 6 per 256 rows and 4 per expert.
    const int n_tiles = (a.np + 255) / 256, blocks = 8 * ((int)((int64_t)(6 * (rows / 256) + 4 * (experts < rows ? experts : rows) + 6) * n_tiles / 32) + 8);
    hipLaunchKernelGGL((grouped_big_kernel<UP>), dim3(blocks), dim3(512), LDS, s, a, n_tiles, experts);
    return 0;
}

}  // namespace trimkv

using namespace trimkv;

extern "C" const char* trimkv_moe_last_error(void) { return err_buf(); }

extern "C" int trimkv_moe_route(const float* logits, const float* correction, int32_t* ids, float* weights, int tokens, int experts, int top, int groups,
                                int keep_groups, void* stream) {
    const char* fn = "trimkv_moe_route";
    if (!logits || !correction || !ids || !weights) return fail(TRIMKV_ERR_NULL, "%s: null pointer argument", fn);
    if (tokens <= 0 || experts <= 0 || experts > ROUTE_MAX_E || groups <= 0 || experts % groups || keep_groups < 1 || keep_groups > groups || top < 1 ||
        top > keep_groups * (experts / groups))
        return fail(TRIMKV_ERR_SHAPE, "%s: bad sizes tokens=%d experts=%d top=%d groups=%d keep=%d", fn, tokens, experts, top, groups, keep_groups);
    auto go = [&](auto ne) {
        hipLaunchKernelGGL((route_kernel<decltype(ne)::value>), dim3((tokens + 3) / 4), dim3(256), 4 * (experts + groups) * sizeof(float), (hipStream_t)stream,
                           logits, correction, ids, weights, tokens, experts, top, groups, keep_groups);
    };
    if (experts <= 64) go(std::integral_constant<int, 1>{});
    else if (experts <= 128) go(std::integral_constant<int, 2>{});
    else if (experts <= 256) go(std::integral_constant<int, 4>{});
    else go(std::integral_constant<int, ROUTE_MAX_E / 64>{});
    return launch_status(fn);
}

extern "C" int trimkv_moe_plan(const int32_t* ids, int rows, int experts, int tile, int32_t* order, int32_t* offsets, int32_t* tiles, void* stream) {
    const char* fn = "trimkv_moe_plan";
    if (!ids || !order || !offsets || !tiles) return fail(TRIMKV_ERR_NULL, "%s: null pointer argument", fn);
    if (rows <= 0 || experts <= 0 || experts > ROUTE_MAX_E || tile <= 0) return fail(TRIMKV_ERR_SHAPE, "%s: bad sizes rows=%d experts=%d tile=%d", fn, rows, experts, tile);
    const int groups = std::min((rows + PLAN_CHUNK - 1) / PLAN_CHUNK, PLAN_MOST);
    hipLaunchKernelGGL(plan_kernel, dim3(groups), dim3(1024), 2 * experts * sizeof(int32_t), (hipStream_t)stream, ids, rows, experts, tile, order, offsets, tiles);
    return launch_status(fn);
}

extern "C" int trimkv_moe_gemm(const void* x, int64_t x_stride, const void* w, void* y, int64_t y_stride, const int32_t* order, const int32_t* offsets,
                               const int32_t* tiles, int rows, int experts, int tile, int top, int n, int n_padded, int k_padded, int up, int dtype, void* stream) {
    const char* fn = "trimkv_moe_gemm";
    if (!x || !w || !y || !order || !offsets || !tiles) return fail(TRIMKV_ERR_NULL, "%s: null pointer argument", fn);
    HY_CHECK_DTYPE(fn, dtype);
    if (rows <= 0 || experts <= 0 || top <= 0 || n <= 0 || n > n_padded || n_padded % 64 || k_padded <= 0 || k_padded % 64 || x_stride < k_padded || y_stride < n)
        return fail(TRIMKV_ERR_SHAPE, "%s: bad sizes rows=%d experts=%d n=%d/%d k=%d", fn, rows, experts, n, n_padded, k_padded);
    if (dtype == TRIMKV_F32 ? tile != 16 : tile != 32 && tile != 256) return fail(TRIMKV_ERR_SHAPE, "%s: row tiles of 16 in fp32, of 32 or 256 in bf16 (got %d)", fn, tile);
    if (((uintptr_t)x | (uintptr_t)w | (uintptr_t)y) & 15 || x_stride % 8) return fail(TRIMKV_ERR_SHAPE, "%s: x, w and y must be 16-byte aligned", fn);
    GroupedArgs a{x, x_stride, w, y, y_stride, order, offsets, tiles, top, n, n_padded, k_padded};
    hipStream_t s = (hipStream_t)stream;
    const int most = rows < experts ? rows : (rows - experts) / tile + experts;     // no more row tiles than this
    const dim3 grid(most, n_padded / 64);
    if (tile == 256) {
        const int rc = up ? launch_big<true>(a, rows, experts, s) : launch_big<false>(a, rows, experts, s);
        if (rc) return fail(rc, "%s: hipFuncSetAttribute failed (%d)", fn, rc);
    } else if (dtype == TRIMKV_BF16) {
        const dim3 g(most, n_padded / 32);
        if ((int64_t)most * n_padded / 32 < 2048) {
            if (up) hipLaunchKernelGGL((grouped_skinny_kernel<true, 8>), g, dim3(512), 0, s, a);
            else hipLaunchKernelGGL((grouped_skinny_kernel<false, 8>), g, dim3(512), 0, s, a);
        } else {
            if (up) hipLaunchKernelGGL((grouped_skinny_kernel<true, 4>), g, dim3(256), 0, s, a);
            else hipLaunchKernelGGL((grouped_skinny_kernel<false, 4>), g, dim3(256), 0, s, a);
        }
    } else {
        if (up) hipLaunchKernelGGL((grouped_f32_kernel<true>), grid, dim3(256), 0, s, a);
        else hipLaunchKernelGGL((grouped_f32_kernel<false>), grid, dim3(256), 0, s, a);
    }
    return launch_status(fn);
}

// Sliding-window attention of prompts and their portions -- gfx950 (masks, ring and arithmetic: window.hip.h).
//
//   window_prefill_kernel  on the matrix cores (bf16): keys are the ring (what earlier portions left) and then the portion's own
//                          rows; tiles that no query of the workgroup sees are skipped
//   window_prefill_f32_kernel  the same in fp32
//   window_rows_kernel     head sizes beyond the tiles: one wavefront per query
//
// In the prefill kernel the probabilities enter the second product as two bf16 terms each (17 bits).
#include "window.hip.h"
#include <algorithm>

namespace trimkv {

// ---- general form: one wavefront per (token, query head) ---------------------------------------
template <typename T>
__global__ __launch_bounds__(256) void window_rows_kernel(WindowArgs a) {
    const int b = blockIdx.y, lane = threadIdx.x & 63;
    const int t0 = a.cu[b], len = a.cu[b + 1] - t0;
    const int unit = blockIdx.x * 4 + (threadIdx.x >> 6);
    const int t = unit / a.H, h = unit - t * a.H;
    if (t >= len) return;
    const int g = h / (a.H / a.G), slot = a.slots[b], past = a.seen[2 * slot], i = past + t;
    const int cap = a.keep + a.size, nring = min(past, cap), nkeys = nring + t + 1;
    const T* q = (const T*)a.q + ((int64_t)(t0 + t) * a.H + h) * a.Dp;
    const T* rk = (const T*)a.rk + ((int64_t)slot * a.G + g) * cap * a.Dp;
    const T* rv = (const T*)a.rv + ((int64_t)slot * a.G + g) * cap * a.Dvp;
    const T* pk = (const T*)a.k + ((int64_t)t0 * a.G + g) * a.Dp;
    const T* pv = (const T*)a.v + ((int64_t)t0 * a.G + g) * a.Dvp;
    float m = WA_NEG, l = 0.0f, acc[8];
#pragma unroll
    for (int c = 0; c < 8; ++c) acc[c] = 0.0f;
    for (int base = 0; base < nkeys; base += 64) {
        const int x = base + lane;
        const int pos = x < nring ? ring_position(x, past, a.keep, a.size) : past + x - nring;
        const bool see = x < nkeys && (i - pos < a.size || pos < a.keep);
        if (__builtin_amdgcn_ballot_w64(see) == 0) continue;
        float s = WA_NEG;
        if (see) {
            const T* kr = x < nring ? rk + (int64_t)x * a.Dp : pk + (int64_t)(x - nring) * a.G * a.Dp;
            float d = 0.0f;
            for (int e = 0; e < a.D; ++e) d += ld(q + e) * ld(kr + e);
            s = d * a.scale_log2;
        }
        const float mn = fmaxf(m, wave_max_f(s)), alpha = exp2f(m - mn);
        const float p = see ? exp2f(s - mn) : 0.0f;
        m = mn;
        l = l * alpha + wave_sum_f(p);
#pragma unroll
        for (int c = 0; c < 8; ++c) acc[c] *= alpha;
        const int cnt = min(64, nkeys - base);
        for (int y = 0; y < cnt; ++y) {
            const float py = __shfl(p, y, 64);
            if (py == 0.0f) continue;                 // wavefront-uniform
            const int xx = base + y;
            const T* vr = xx < nring ? rv + (int64_t)xx * a.Dvp : pv + (int64_t)(xx - nring) * a.G * a.Dvp;
#pragma unroll
            for (int c = 0; c < 8; ++c)
                if (c * 64 + lane < a.Dv) acc[c] += py * ld(vr + c * 64 + lane);
        }
    }
    const float inv = 1.0f / (l + window_sink(a, m));
    T* o = (T*)a.out + ((int64_t)(t0 + t) * a.H + h) * a.Dv;
#pragma unroll
    for (int c = 0; c < 8; ++c) {
        const int d = c * 64 + lane;
        if (d < a.Dv) st(o + d, acc[c] * inv * window_gate<T>(a, t0 + t, h, d));
    }
}

// ---- fp32 prompts on the matrix cores --------------------------------------------------------------
// A workgroup owns 64 rows (consecutive query times x the query heads of one KV head), 16 per wavefront, and walks tiles of 64
// keys; or 32 rows, with half of every tile for two wavefronts each, whose sums are put together at the end.  Both products run on 16x16x4 fp32 MFMAs,
// transposed: S^T = K . Q^T, O^T += V^T . P^T, so a row is a column of the accumulators (lane % 16) and the probabilities a lane
// holds behind the first product are its operand of the second.  With g = lane / 16, A and B hold k = g of row / column lane % 16
// and register r of C row 4 g + r; the sums take features in the order 16 x + 4 g + r and keys likewise, so that a lane reads
// four consecutive floats of K.  LDS rows are DT + 4 floats apart: reads of either product fall on different banks.  The next
// tile waits in registers; a tile is all of the ring or all of the portion, so that its rows are one base and a stride.
//
// Bound by the matrix cores' fp32 rate (a sixteenth of bf16), 1.75 us a tile of 32 rows, and as much again of other vector instructions.  The longest
// rows of all heads go first: with a head's workgroups one behind the other the launch ended on long ones, 16 heads of 128 (8 KV heads): three
// prompts of 1000 tokens 300 us for 165, one of 4000 730 for 585.  300 + 511 tokens: 72 us with 64 rows in that order, 51 with 32; a
// wavefront per query row, which this replaces for head sizes up to 128, took 1060 us there, bound by its row-wise loads.  Rows that are not there come last
// (row_tile_at): in between, where every eighth workgroup has work, those all go to a few compute units.  Prompts of 2238, 25, 3, 14, 35, 2, 40 and 40 tokens, 8 heads
// of 96 (2 KV heads) 107 us for 499, of 2128 and 296, 16 of 128 295 for 428; finding the place takes 0.7 us.
// NaNs and infinities of keys that a row does not see must not reach it through 0 x inf: tiles with such values in V take their
// second product one key at a time.

// Place `at` among the tiles of bt rows of all sequences (up to `tiles` of each), the last ones first: those of tile t stand behind those of all later
// ones.  64 candidates for t at once: how many stand in front of the end of t is a sum over the sequences.
struct RowTile { int b, tile, t0, len, slot; };      // b = -1: there are not as many
__device__ __forceinline__ RowTile row_tile_at(const WindowArgs& a, int batch, int tiles, int bt, int at) {
    const int lane = threadIdx.x & 63;
    int start = 0, len = 0, slot = 0, own = 0;
    auto take = [&](int b0) __attribute__((always_inline)) {      // sequences b0 .. b0 + 63, one to a lane
        const int b = min(b0 + lane, batch - 1);
        start = a.cu[b]; len = a.cu[b + 1] - start; slot = a.slots[b];
        own = b0 + lane < batch ? min((max(len, 0) + bt - 1) / bt, tiles) : 0;
    };
    take(0);
    if (batch == 1) {                                             // every lane has the sequence, the first one its number of tiles
        own = __builtin_amdgcn_readfirstlane(own);
        return {at < own ? 0 : -1, own - 1 - at, start, len, slot};
    }
    int lo = 0, span = tiles, upto;                               // t is in lo .. lo + span - 1; places up to the end of lo
    do {
        const int step = (span + 63) / 64, t = lo + lane * step;
        int n = 0;
        for (int b0 = 0; b0 < batch; b0 += 64) {
            if (batch > 64) take(b0);
            for (int j = 0; j < min(64, batch - b0); ++j) n += max(__builtin_amdgcn_readlane(own, j) - t, 0);
        }
        const unsigned long long behind = __ballot(n > at && lane * step < span);
        if (!behind) return {-1, 0, 0, 0, 0};                     // in the first round only
        const int l = 63 - __builtin_clzll(behind);
        lo += l * step;
        span = min(step, span - l * step);
        upto = __builtin_amdgcn_readlane(n, l);
    } while (span > 1);
    int k = upto - at;                                            // from the last sequence that has the tile
    for (int b0 = (batch - 1) / 64 * 64; b0 >= 0; b0 -= 64) {
        if (batch > 64) take(b0);
        const unsigned long long has = __ballot(own > lo);
        const int n = __popcll(has);
        if (k <= n) {
            const int l = __builtin_ctzll(__ballot(own > lo && __popcll(has >> lane) == k));
            return {b0 + l, lo, __builtin_amdgcn_readlane(start, l), __builtin_amdgcn_readlane(len, l), __builtin_amdgcn_readlane(slot, l)};
        }
        k -= n;
    }
    return {-1, 0, 0, 0, 0};
}

template <int DT, int ROWS>
__global__ __launch_bounds__(256) void window_prefill_f32_kernel(WindowArgs a, int batch, int tiles) {      // grid: KV heads x tiles of rows of all sequences (in z what y does not hold)
    constexpr int LD = DT + 4, DB = DT / 16, PIECES = DT / 4, LOADS = 64 * PIECES / 256, RW = ROWS / 16, KS = 4 / RW, KB = 4 / KS;
    extern __shared__ __attribute__((aligned(16))) char wf_lds[];
    float* const kt = (float*)wf_lds; float* const vt = kt + 64 * LD;
    int* const where = (int*)(vt + 64 * LD);          // position of every key of the tile; past the end: beyond all queries
    int* const odd = where + 64;                      // number of tiles + 1 whose V held something that is not finite
    // later times of all heads first: they walk the most tiles
    const int per = a.H / a.G, bt = ROWS / per, g = blockIdx.x;
    const RowTile mine = row_tile_at(a, batch, tiles, bt, (int)min(blockIdx.z * gridDim.y + blockIdx.y, 0x7fffffffu));
    if (mine.b < 0) return;                           // workgroup-uniform, before any barrier
    const int t0 = __builtin_amdgcn_readfirstlane(mine.t0), len = __builtin_amdgcn_readfirstlane(mine.len), slot = __builtin_amdgcn_readfirstlane(mine.slot);
    const int first = __builtin_amdgcn_readfirstlane(mine.tile) * bt;
    const int past = a.seen[2 * slot], cap = a.keep + a.size, nring = min(past, cap), last = min(first + bt, len) - 1;
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, c = lane & 15, gr = lane >> 4;
    const int kb0 = w / RW * KB, row = w % RW * 16 + c, t = min(first + row / per, last), h = g * per + row % per, i = past + t;
    const bool live = row < bt * per && first + row / per < len;
    const float* rk = (const float*)a.rk + ((int64_t)slot * a.G + g) * cap * a.Dp;
    const float* rv = (const float*)a.rv + ((int64_t)slot * a.G + g) * cap * a.Dvp;
    const float* pk = (const float*)a.k + ((int64_t)t0 * a.G + g) * a.Dp;
    const float* pv = (const float*)a.v + ((int64_t)t0 * a.G + g) * a.Dvp;
    float4 q[DB];
    {
        const float* qr = (const float*)a.q + ((int64_t)(t0 + t) * a.H + h) * a.Dp;
#pragma unroll
        for (int x = 0; x < DB; ++x) q[x] = *(const float4*)(qr + min(16 * x + 4 * gr, a.Dp - 4));
#pragma unroll
        for (int x = 0; x < DB; ++x) q[x] = __builtin_bit_cast(float4, kept4(__builtin_bit_cast(hy_u32x4, q[x]), 16 * x + 4 * gr < a.Dp));
    }
    // tiles of the ring, then tiles of the portion; one of the portion that no row sees is skipped
    const int rtiles = (nring + 63) / 64, ntiles = rtiles + (last + 64) / 64;
    auto next_tile = [&](int x) {
        for (; x < ntiles; ++x) {
            const int lo = past + (x - rtiles) * 64, hi = lo + 63;   // positions, if the tile is of the portion
            if (x < rtiles || hi > past + first - a.size || lo < a.keep) break;
        }
        return x;
    };
    auto keys_of = [&](int x) { return min(64, x < rtiles ? nring - x * 64 : last + 1 - (x - rtiles) * 64); };
    hy_u32x4 kn[LOADS], vn[LOADS];
    int where_n = 0;
    const int piece = tid % PIECES * 4, ek = min(piece, a.Dp - 4), ev = min(piece, a.Dvp - 4), r0 = tid / PIECES;
    auto fetch = [&](int x) __attribute__((always_inline)) {
        const bool ring = x < rtiles;
        const int from = ring ? x * 64 : (x - rtiles) * 64, step = ring ? 1 : a.G, end = keys_of(x) - 1;
        const float* kb = (ring ? rk : pk) + (int64_t)from * step * a.Dp; const float* vb = (ring ? rv : pv) + (int64_t)from * step * a.Dvp;
#pragma unroll
        for (int y = 0; y < LOADS; ++y) {
            const int r = min(y * (256 / PIECES) + r0, end);        // loads are unconditional (a load under a branch is waited for on the spot)
            kn[y] = *(const hy_u32x4*)(kb + (uint32_t)(r * (step * a.Dp) + ek));
            vn[y] = *(const hy_u32x4*)(vb + (uint32_t)(r * (step * a.Dvp) + ev));
        }
        where_n = lane > end ? 0x7fffffff : ring ? ring_position(from + lane, past, a.keep, a.size) : past + from + lane;
    };
    hy_f32x4 o[DB];
#pragma unroll
    for (int x = 0; x < DB; ++x) o[x] = hy_f32x4{0.f, 0.f, 0.f, 0.f};
    float m = WA_NEG, l = 0.0f;
    if (tid == 0) *odd = 0;
    int tile = next_tile(0);
    if (tile < ntiles) fetch(tile);
    while (tile < ntiles) {
        __syncthreads();                              // the last tile is done with
        bool fine = true;
        const int here = keys_of(tile);
#pragma unroll
        for (int y = 0; y < LOADS; ++y) {             // what is not there becomes zero
            const int r = y * (256 / PIECES) + r0;
            const hy_u32x4 vv = kept4(vn[y], r < here && piece < a.Dvp);
            *(hy_u32x4*)(kt + r * LD + piece) = kept4(kn[y], r < here && piece < a.Dp);
            *(hy_u32x4*)(vt + r * LD + piece) = vv;
            fine = fine && finite_bits(vv);
        }
        if (tid < 64) where[tid] = where_n;
        if (!fine) *odd = tile + 1;
        __syncthreads();
        const int now = tile;
        tile = next_tile(tile + 1);
        if (tile < ntiles) fetch(tile);
        hy_f32x4 s[KB];
        float top = WA_NEG;
        {                                             // fragments of K are read one step of 16 features ahead
            const float* kr = kt + (kb0 * 16 + c) * LD + 4 * gr;
            float4 f[2][KB];
#pragma unroll
            for (int kb = 0; kb < KB; ++kb) {
                s[kb] = hy_f32x4{0.f, 0.f, 0.f, 0.f};
                f[0][kb] = *(const float4*)(kr + kb * 16 * LD);
            }
#pragma unroll
            for (int x = 0; x < DB; ++x) {
                if (x + 1 < DB) {
#pragma unroll
                    for (int kb = 0; kb < KB; ++kb) f[~x & 1][kb] = *(const float4*)(kr + kb * 16 * LD + 16 * (x + 1));
                }
#pragma unroll
                for (int y = 0; y < 4; ++y)
#pragma unroll
                    for (int kb = 0; kb < KB; ++kb) {
                        const float4 g4 = f[x & 1][kb];
                        s[kb] = mfma16_f32(y == 0 ? g4.x : y == 1 ? g4.y : y == 2 ? g4.z : g4.w, y == 0 ? q[x].x : y == 1 ? q[x].y : y == 2 ? q[x].z : q[x].w, s[kb]);
                    }
                __builtin_amdgcn_sched_barrier(0);
            }
        }
#pragma unroll
        for (int kb = 0; kb < KB; ++kb) {
            const int4 at = *(const int4*)(where + (kb0 + kb) * 16 + 4 * gr);
            const int pos[4] = {at.x, at.y, at.z, at.w};
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                s[kb][r] = pos[r] <= i && (i - pos[r] < a.size || pos[r] < a.keep) ? s[kb][r] * a.scale_log2 : -INFINITY;
                top = fmaxf(top, s[kb][r]);
            }
        }
        top = fmaxf(top, __shfl_xor(top, 16, 64));
        top = fmaxf(top, __shfl_xor(top, 32, 64));
        const float mn = fmaxf(m, top), alpha = exp2f(m - mn);
        m = mn;
        l *= alpha;
#pragma unroll
        for (int kb = 0; kb < KB; ++kb)
#pragma unroll
            for (int r = 0; r < 4; ++r) { s[kb][r] = exp2f(s[kb][r] - mn); l += s[kb][r]; }
#pragma unroll
        for (int x = 0; x < DB; ++x) o[x] *= alpha;
        if (*odd != now + 1) {
            const float* vr = vt + (kb0 * 16 + 4 * gr) * LD + c;       // one key ahead, as above
            float f[2][DB];
#pragma unroll
            for (int x = 0; x < DB; ++x) f[0][x] = vr[16 * x];
#pragma unroll
            for (int y = 0; y < 4 * KB; ++y) {
                if (y + 1 < 4 * KB) {
#pragma unroll
                    for (int x = 0; x < DB; ++x) f[~y & 1][x] = vr[((y + 1) / 4 * 16 + (y + 1) % 4) * LD + 16 * x];
                }
#pragma unroll
                for (int x = 0; x < DB; ++x) o[x] = mfma16_f32(f[y & 1][x], s[y / 4][y % 4], o[x]);
                __builtin_amdgcn_sched_barrier(0);
            }
        } else {                                      // workgroup-uniform: the keys' place takes the probabilities
            __syncthreads();
            float* const ps = kt + w * (KB * 256);    // [key][row]
#pragma unroll
            for (int kb = 0; kb < KB; ++kb)
#pragma unroll
                for (int r = 0; r < 4; ++r) ps[(kb * 16 + 4 * gr + r) * 16 + c] = s[kb][r];
            __syncthreads();
#pragma unroll 1
            for (int key = 0; key < KB * 16; ++key) {
                const float p = ps[key * 16 + c];
#pragma unroll
                for (int x = 0; x < DB; ++x) {
                    const float4 f = *(const float4*)(vt + (kb0 * 16 + key) * LD + 16 * x + 4 * gr);
                    o[x][0] += p == 0.0f ? 0.0f : p * f.x;
                    o[x][1] += p == 0.0f ? 0.0f : p * f.y;
                    o[x][2] += p == 0.0f ? 0.0f : p * f.z;
                    o[x][3] += p == 0.0f ? 0.0f : p * f.w;
                }
            }
        }
    }
    l += __shfl_xor(l, 16, 64);
    l += __shfl_xor(l, 32, 64);
    if constexpr (KS == 2) {                          // the wavefronts of the first keys take the others' sums
        hy_f32x4* const po = (hy_f32x4*)kt + w % RW * (DB * 64) + lane;
        float2* const pm = (float2*)vt + w % RW * 64 + lane;
        __syncthreads();
        if (w >= RW) {
#pragma unroll
            for (int x = 0; x < DB; ++x) po[x * 64] = o[x];
            *pm = make_float2(m, l);
        }
        __syncthreads();
        if (w >= RW) return;
        const float2 other = *pm;
        const float mn = fmaxf(m, other.x), ours = exp2f(m - mn), theirs = exp2f(other.x - mn);
        m = mn;
        l = (ours == 0.0f ? 0.0f : l * ours) + (theirs == 0.0f ? 0.0f : other.y * theirs);
#pragma unroll
        for (int x = 0; x < DB; ++x) {
            const hy_f32x4 f = po[x * 64];
#pragma unroll
            for (int r = 0; r < 4; ++r) o[x][r] = (ours == 0.0f ? 0.0f : o[x][r] * ours) + (theirs == 0.0f ? 0.0f : f[r] * theirs);
        }
    }
    if (!live) return;
    const float inv = 1.0f / (l + window_sink(a, m));
    float* out = (float*)a.out + ((int64_t)(t0 + t) * a.H + h) * a.Dv;
    float gate[DB][4];
#pragma unroll
    for (int x = 0; x < DB; ++x)
#pragma unroll
        for (int r = 0; r < 4; ++r) gate[x][r] = window_gate<float>(a, t0 + t, h, min(16 * x + 4 * gr + r, a.Dv - 1));
#pragma unroll
    for (int x = 0; x < DB; ++x)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int d = 16 * x + 4 * gr + r;
            if (d < a.Dv) out[d] = o[x][r] * inv * gate[x][r];
        }
}

// ---- prompts on the matrix cores -------------------------------------------------------------------
// A workgroup owns 128 rows = consecutive query times x the query heads of one KV head, 32 rows per wavefront.  Per tile of
// 64 keys a wavefront computes S^T[key][row] = K . Q^T and O^T[d][row] += V^T . P^T on 32x32x16 MFMAs: the row is the MFMA
// column (lane % 32), so maxima and sums live in the lane that needs them and the probabilities a lane holds after the first
// product are its operand of the second.  Layout (half hl = lane / 32): A, B hold k = 8 hl + 0..7 of row / column lane % 32;
// register v of C holds row 8 (v / 4) + 4 hl + v % 4.  Tiles come by LDS-direct loads, two buffers in turn.
//   K: 16-byte piece c of row r sits at c ^ swz(r), so that the rows of a fragment read fall on different banks
//   V: row-major too, read with ds_read_b64_tr_b16 (4 keys of one d per lane); its 32-byte pairs are swizzled by row
template <int D>
struct WindowTile {
    static constexpr int BN = 64, PIECES = D / 8, TILE = BN * D * 2, LOADS = BN * PIECES / 256;
    static __device__ __forceinline__ int kswz(int r) { return D == 64 ? (r >> 1) & 7 : r & 15; }
    static __device__ __forceinline__ int vswz(int r) { return D == 64 ? 4 * ((r >> 1) & 1) : 4 * (r & 3); }   // in 16-byte pieces
};

// Tiles are laid out for D features; products stop at USED of them.
template <int D, int USED>
__global__ __launch_bounds__(256, D <= 128 ? 2 : 1) void window_prefill_kernel(WindowArgs a) {
    using W = WindowTile<D>;
    constexpr int KS = USED / 16, DB = USED / 32;
    extern __shared__ __attribute__((aligned(16))) char wa_lds[];
    HY_LDS char* const lds3 = (HY_LDS char*)wa_lds;
    const uint32_t lds0 = (uint32_t)(uintptr_t)lds3;
    const int tid = threadIdx.x, lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int j = lane & 31, hl = lane >> 5;
    // workgroups go to the 8 XCDs in turn; the tiles of one (sequence, KV head) read the same keys, so they share an XCD
    int pair = blockIdx.y, tile = (int)gridDim.x - 1 - (int)blockIdx.x;
    if ((gridDim.y & 7) == 0) {
        const int lin = (int)blockIdx.y * (int)gridDim.x + (int)blockIdx.x, turn = lin >> 3;
        pair = (lin & 7) + 8 * (turn / (int)gridDim.x);
        tile = (int)gridDim.x - 1 - turn % (int)gridDim.x;
    }
    const int b = pair / a.G, g = pair - b * a.G;
    const int tok0 = a.cu[b], len = a.cu[b + 1] - tok0;
    const int per = a.H / a.G, BT = 128 / per, q0 = tile * BT;
    if (q0 >= len) return;                                        // workgroup-uniform, before any barrier
    const int slot = a.slots[b], past = a.seen[2 * slot], cap = a.keep + a.size, nring = min(past, cap);
    const int r = w * 32 + j, t = q0 + r / per, h = g * per + r % per;
    const bool ok = r < BT * per && t < len;
    const int tc = min(t, len - 1), i = past + tc;
    const int q1 = min(len - 1, q0 + BT - 1);                     // the workgroup's last query time
    const int tw0 = min(q0 + (w * 32) / per, len - 1), tw1 = min(q0 + (w * 32 + 31) / per, q1);

    const bf16_t* Q = (const bf16_t*)a.q + ((int64_t)(tok0 + tc) * a.H + h) * a.Dp;
    hy_bf16x8 qf[KS];
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
        const int e0 = ks * 16 + hl * 8;
        const hy_u32x4 raw = *(const hy_u32x4*)(Q + min(e0, a.Dp - 8));
        qf[ks] = __builtin_bit_cast(hy_bf16x8, e0 < a.Dp ? raw : hy_u32x4{0u, 0u, 0u, 0u});
    }
    hy_f32x16 o[DB];
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
        for (int v = 0; v < 16; ++v) o[db][v] = 0.0f;
    float m = WA_NEG, l = 0.0f;

    const char* rk = (const char*)a.rk + ((int64_t)slot * a.G + g) * cap * a.Dp * 2;
    const char* rv = (const char*)a.rv + ((int64_t)slot * a.G + g) * cap * a.Dvp * 2;
    const char* pk = (const char*)a.k + ((int64_t)tok0 * a.G + g) * a.Dp * 2;
    const char* pv = (const char*)a.v + ((int64_t)tok0 * a.G + g) * a.Dvp * 2;

    // tiles: the ring, then the portion's kept rows, then its window
    const int nr = (nring + 63) / 64;
    const int nkept = (max(0, min(a.keep - past, q1 + 1)) + 63) / 64;
    const int wt0 = max(nkept, max(0, q0 - a.size + 1) / 64);
    const int total = nr + nkept + max(0, q1 / 64 + 1 - wt0);
    // a load instruction of the workgroup covers RL rows; what a lane fetches of them does not depend on the tile, so a tile
    // whose rows all exist needs scalar addresses only
    constexpr int RL = 256 / W::PIECES;
    const int lrow = tid / W::PIECES, lpos = tid % W::PIECES;
    int kcol[2], vcol[2];                                  // swizzles repeat after 16 rows
#pragma unroll
    for (int x = 0; x < 2; ++x) {
        kcol[x] = min((lpos ^ W::kswz(lrow + x * RL)) * 16, a.Dp * 2 - 16);
        vcol[x] = min((lpos ^ W::vswz(lrow + x * RL)) * 16, a.Dvp * 2 - 16);
    }
    auto request = [&](int n, int buf) __attribute__((always_inline)) {
        const bool ring = n < nr;
        const int k0 = 64 * (ring ? n : n - nr < nkept ? n - nr : wt0 + n - nr - nkept);
        const int last = ring ? nring - 1 : len - 1;
        const char* kb = ring ? rk : pk;
        const char* vb = ring ? rv : pv;
        const int ks = ring ? a.Dp * 2 : a.G * a.Dp * 2, vs = ring ? a.Dvp * 2 : a.G * a.Dvp * 2;
        const uint32_t dst = lds0 + buf * 2 * W::TILE + w * 1024;
        if (k0 + 63 <= last) {
            const char* kt = kb + (int64_t)k0 * ks;
            const char* vt = vb + (int64_t)k0 * vs;
            const uint32_t ko = lrow * ks, vo = lrow * vs;
#pragma unroll
            for (int x = 0; x < W::LOADS; ++x) {
                load_to_lds16_at(kt + x * RL * ks, ko + kcol[x & 1], dst + x * 4096);
                load_to_lds16_at(vt + x * RL * vs, vo + vcol[x & 1], dst + W::TILE + x * 4096);
            }
        } else {
#pragma unroll
            for (int x = 0; x < W::LOADS; ++x) {
                const int64_t key = min(k0 + x * RL + lrow, last);
                load_to_lds16(kb + key * ks + kcol[x & 1], dst + x * 4096);
                load_to_lds16(vb + key * vs + vcol[x & 1], dst + W::TILE + x * 4096);
            }
        }
    };
    const int kx = 4 * hl + ((lane & 15) >> 2), jh = (lane >> 4) & 1;   // the transposing read: key of this lane, half of the 32 d
    auto k_frag = [&](int off, int blk, int ks) __attribute__((always_inline)) {
        const int row = blk * 32 + j;
        return *(const HY_LDS hy_bf16x8*)(lds3 + off + row * (D * 2) + (((2 * ks + hl) ^ W::kswz(j)) << 4));
    };
    auto v_frag = [&](int off, int st_, int db) __attribute__((always_inline)) {
        HY_LDS char* p = lds3 + off + W::TILE + (st_ * 16 + kx) * (D * 2) + ((((2 * db + jh) * 2) ^ W::vswz(kx)) << 4) + (lane & 3) * 8;
        const hy_s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((HY_LDS hy_s16x4*)p);
        const hy_s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((HY_LDS hy_s16x4*)(p + 8 * D * 2));
        return __builtin_bit_cast(hy_bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
    };

    request(0, 0);
    for (int n = 0; n < total; ++n) {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();                                   // tile n is complete, tile n - 1 is no longer read
        if (n + 1 < total) request(n + 1, (n + 1) & 1);
        const bool ring = n < nr;
        const int k0 = 64 * (ring ? n : n - nr < nkept ? n - nr : wt0 + n - nr - nkept);
        if (!ring && k0 > tw1) continue;                   // wavefront-uniform: nothing of the tile is visible yet
        if (!ring && k0 + 63 <= tw0 - a.size && past + k0 >= a.keep) continue;   // ... or any more
        const int off = (n & 1) * 2 * W::TILE;
        // operands are requested AHEAD steps before the MFMA that takes them; the fences keep the compiler from moving them back
        constexpr int AHEAD = 3;
        __builtin_amdgcn_s_setprio(1);                     // the wavefront that can feed the matrix cores goes first
        hy_f32x16 s[2];
#pragma unroll
        for (int v = 0; v < 16; ++v) s[0][v] = s[1][v] = 0.0f;
        {
            hy_bf16x8 kf[2 * KS];
#pragma unroll
            for (int x = 0; x < AHEAD; ++x) kf[x] = k_frag(off, x & 1, x >> 1);
#pragma unroll
            for (int x = 0; x < 2 * KS; ++x) {
                if (x + AHEAD < 2 * KS) kf[x + AHEAD] = k_frag(off, (x + AHEAD) & 1, (x + AHEAD) >> 1);
                s[x & 1] = mfma32(kf[x], qf[x >> 1], s[x & 1]);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        hy_bf16x8 vf[4 * DB];
#pragma unroll
        for (int x = 0; x < AHEAD; ++x) vf[x] = v_frag(off, x / DB, x % DB);
        __builtin_amdgcn_s_setprio(0);
        const bool whole = !ring && k0 + 63 <= tw0 && (k0 > tw1 - a.size || past + k0 + 63 < a.keep);
        if (!whole) {
            asm volatile("" :::);                          // keeps this a branch
            if (ring) {
#pragma unroll 1
                for (int v = 0; v < 16; ++v) {
                    // (rarely taken: a loop over registers through a compare, not 32 copies of the slot arithmetic)
                    const int x = k0 + 8 * (v >> 2) + 4 * hl + (v & 3);
                    bool see[2];
#pragma unroll
                    for (int blk = 0; blk < 2; ++blk) {
                        const int slot_ = x + 32 * blk, pos = ring_position(slot_, past, a.keep, a.size);
                        see[blk] = slot_ < nring && (i - pos < a.size || pos < a.keep);
                    }
#pragma unroll
                    for (int u = 0; u < 16; ++u) {
                        s[0][u] = u == v && !see[0] ? WA_NEG : s[0][u];
                        s[1][u] = u == v && !see[1] ? WA_NEG : s[1][u];
                    }
                }
            } else {
                const int x1 = i - past, x0 = x1 - a.size, xk = a.keep - past;    // rows up to x1 and beyond x0 or below xk
#pragma unroll
                for (int blk = 0; blk < 2; ++blk)
#pragma unroll
                    for (int v = 0; v < 16; ++v) {
                        const int x = k0 + blk * 32 + 8 * (v >> 2) + 4 * hl + (v & 3);
                        const bool see = (x <= x1) & ((x > x0) | (x < xk));
                        s[blk][v] = see ? s[blk][v] : WA_NEG;
                    }
            }
        }
        float tm = s[0][0];
#pragma unroll
        for (int v = 0; v < 16; ++v) tm = fmaxf(tm, fmaxf(s[0][v], s[1][v]));
        tm = tm > 0.5f * WA_NEG ? tm * a.scale_log2 : WA_NEG;
        // the reference moves only when some row outgrows it by 2^6 (or has none yet)
        if (__builtin_amdgcn_ballot_w64(tm > m + 6.0f) != 0) {
            const float mn = fmaxf(m, fmaxf(tm, __shfl_xor(tm, 32, 64)));
            const float alpha = __builtin_amdgcn_exp2f(m - mn);
            m = mn;
            l *= alpha;
#pragma unroll
            for (int db = 0; db < DB; ++db)
#pragma unroll
                for (int v = 0; v < 16; ++v) o[db][v] *= alpha;
        }
        const float ref = m > 0.5f * WA_NEG ? m : 0.0f;    // a row that has seen nothing: its scores give exp2(-huge) = 0
        const float sc = a.scale_log2;
        // the exponentials of the next 16 keys run between the MFMAs of these
        hy_u32x4 hi[2], lo[2];
        auto weigh = [&](int st_, int x) __attribute__((always_inline)) {
            const int v = (st_ & 1) * 8 + 2 * x;
            const float p0 = __builtin_amdgcn_exp2f(fmaf(s[st_ >> 1][v], sc, -ref)), p1 = __builtin_amdgcn_exp2f(fmaf(s[st_ >> 1][v + 1], sc, -ref));
            l += p0 + p1;
            uint32_t tw[2];
            split2<2>(p0, p1, tw);
            hi[st_ & 1][x] = tw[0]; lo[st_ & 1][x] = tw[1];
        };
#pragma unroll
        for (int x = 0; x < 4; ++x) weigh(0, x);
        __builtin_amdgcn_s_setprio(1);
#pragma unroll
        for (int st_ = 0; st_ < 4; ++st_) {
#pragma unroll
            for (int db = 0; db < DB; ++db) {
                const int x = st_ * DB + db;
                if (x + AHEAD < 4 * DB) vf[x + AHEAD] = v_frag(off, (x + AHEAD) / DB, (x + AHEAD) % DB);
                o[db] = mfma32(vf[x], __builtin_bit_cast(hy_bf16x8, hi[st_ & 1]), o[db]);
                if (st_ < 3 && db < 2) weigh(st_ + 1, db);
                __builtin_amdgcn_sched_barrier(0);
            }
#pragma unroll
            for (int db = 0; db < DB; ++db) {
                o[db] = mfma32(vf[st_ * DB + db], __builtin_bit_cast(hy_bf16x8, lo[st_ & 1]), o[db]);
                if (st_ < 3 && db < 2) weigh(st_ + 1, 2 + db);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        __builtin_amdgcn_s_setprio(0);
    }
    l += __shfl_xor(l, 32, 64);                            // the halves of a row hold disjoint keys
    if (!ok) return;
    float inv = 1.0f / (l + window_sink(a, m));
    const bf16_t* gr = (const bf16_t*)a.gate + (int64_t)(tok0 + t) * a.gate_stride + h * a.Dv;
    if (a.head_gate) inv *= window_gate<bf16_t>(a, tok0 + t, h, 0);
    bf16_t* orow = (bf16_t*)a.out + ((int64_t)(tok0 + t) * a.H + h) * a.Dv;
#pragma unroll
    for (int db = 0; db < DB; ++db) {
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const int d = db * 32 + 8 * c + 4 * hl;
            if (a.vec) {
                if (d >= a.Dv) continue;
                if (a.head_gate) st4(orow + d, make_float4(o[db][4 * c] * inv, o[db][4 * c + 1] * inv, o[db][4 * c + 2] * inv, o[db][4 * c + 3] * inv));
                else {
                    const float4 gt = ld4(gr + d);
                    st4(orow + d, make_float4(o[db][4 * c] * inv * sigmoid_fast(gt.x), o[db][4 * c + 1] * inv * sigmoid_fast(gt.y),
                                              o[db][4 * c + 2] * inv * sigmoid_fast(gt.z), o[db][4 * c + 3] * inv * sigmoid_fast(gt.w)));
                }
            } else {
#pragma unroll
                for (int x = 0; x < 4; ++x)
                    if (d + x < a.Dv) st(orow + d + x, o[db][4 * c + x] * inv * (a.head_gate ? 1.0f : sigmoid_fast(ld(gr + d + x))));
            }
        }
    }
}

template <int D, int USED = D>
static int launch_window_prefill(const WindowArgs& a, int batch, int max_len, hipStream_t s) {
    constexpr int LDS = 4 * WindowTile<D>::TILE;
    static bool opted_in[64] = {};
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) dev = -1;
    if (dev < 0 || !opted_in[dev]) {
        hipError_t e = hipFuncSetAttribute((const void*)window_prefill_kernel<D, USED>, hipFuncAttributeMaxDynamicSharedMemorySize, LDS);
        if (e != hipSuccess) return (int)e;
        if (dev >= 0) opted_in[dev] = true;
    }
    const int bt = 128 / (a.H / a.G);
    hipLaunchKernelGGL((window_prefill_kernel<D, USED>), dim3((max_len + bt - 1) / bt, batch * a.G), dim3(256), LDS, s, a);
    return 0;
}

template <int DT, int ROWS>
static int launch_window_rows_f32(const WindowArgs& a, int batch, int max_len, hipStream_t s) {
    constexpr int LDS = (2 * 64 * (DT + 4) + 64 + 4) * 4;
    static bool opted_in[64] = {};
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) dev = -1;
    if (dev < 0 || !opted_in[dev]) {
        hipError_t e = hipFuncSetAttribute((const void*)window_prefill_f32_kernel<DT, ROWS>, hipFuncAttributeMaxDynamicSharedMemorySize, LDS);
        if (e != hipSuccess) return (int)e;
        if (dev >= 0) opted_in[dev] = true;
    }
    const int bt = ROWS / (a.H / a.G);
    const int tiles = (max_len + bt - 1) / bt;
    const int64_t all = (int64_t)tiles * batch, y = std::min<int64_t>(all, 65535);
    hipLaunchKernelGGL((window_prefill_f32_kernel<DT, ROWS>), dim3(a.G, (unsigned)y, (unsigned)((all + y - 1) / y)), dim3(256), LDS, s, a, batch, tiles);
    return 0;
}

// 32 rows to a workgroup while 64 would leave compute units without a second one.  us with 32 | 64 rows, 8 KV heads of 128 with two
// query heads each: 600 tokens (152 workgroups of 64 rows) 55 | 73, 300 + 511 (256) 51 | 64, three times 600 (456) 85 | 94, three times 1000 (768) 187 | 165,
// three times 2000 627 | 552.
constexpr int F32_HALF_ROWS = 512;
template <int DT>
static int launch_window_prefill_f32(const WindowArgs& a, int batch, int max_len, hipStream_t s) {
    const int per = a.H / a.G;
    const int64_t wgs = (int64_t)((max_len + 64 / per - 1) / (64 / per)) * batch * a.G;
    return per <= 32 && wgs <= F32_HALF_ROWS ? launch_window_rows_f32<DT, 32>(a, batch, max_len, s) : launch_window_rows_f32<DT, 64>(a, batch, max_len, s);
}

}  // namespace trimkv

using namespace trimkv;

extern "C" int trimkv_window_prefill(const void* q, const void* k, const void* v, const void* ring_k, const void* ring_v, const int32_t* cu,
                                     const int32_t* slots, const int32_t* seen, const void* gate, int64_t gate_stride, void* out, int batch, int max_len,
                                     int heads, int kv_heads, int dim, int vdim, int dim_stride, int vdim_stride, int keep_first, int window,
                                     float scale, int head_gate, int sink, int dtype, void* stream) {
    const char* fn = "trimkv_window_prefill";
    WindowArgs a{};
    a.q = q; a.k = k; a.v = v; a.rk = ring_k; a.rv = ring_v; a.cu = cu; a.slots = slots; a.seen = seen; a.gate = gate; a.gate_stride = gate_stride; a.out = out;
    a.H = heads; a.G = kv_heads; a.D = dim; a.Dv = vdim; a.Dp = dim_stride; a.Dvp = vdim_stride; a.keep = keep_first; a.size = window;
    a.scale_log2 = scale * 1.4426950408889634f; a.splits = 1; a.head_gate = head_gate; a.sink = sink;
    if (int rc = window_common(fn, a, batch, dtype)) return rc;
    if (!k || !v || !cu) return fail(TRIMKV_ERR_NULL, "%s: null pointer argument", fn);
    if (max_len <= 0 || (int64_t)batch * kv_heads > 65535) return fail(TRIMKV_ERR_SHAPE, "%s: bad sizes max_len=%d batch*kv_heads=%lld", fn, max_len, (long long)batch * kv_heads);
    hipStream_t s = (hipStream_t)stream;
    const int per = heads / kv_heads, big = dim_stride > vdim_stride ? dim_stride : vdim_stride;
    const bool aligned = !(((uintptr_t)k | (uintptr_t)v) & 15);
    if (dtype == TRIMKV_BF16 && big <= 256 && per <= 128 && aligned && scale > 0.0f) {
        a.vec = vdim % 4 == 0 && !((uintptr_t)out & 7) && (head_gate || (gate_stride % 4 == 0 && !((uintptr_t)gate & 7)));
        const int rc = big <= 64 ? launch_window_prefill<64>(a, batch, max_len, s) : big <= 96 ? launch_window_prefill<128, 96>(a, batch, max_len, s) : big <= 128 ? launch_window_prefill<128>(a, batch, max_len, s)
                                                                                               : launch_window_prefill<256>(a, batch, max_len, s);
        if (rc) return fail(rc, "%s: hipFuncSetAttribute failed (%d)", fn, rc);
        return launch_status(fn);
    }
    if (dtype == TRIMKV_F32 && big <= 128 && per <= 64 && aligned) {
        const int rc = big <= 64 ? launch_window_prefill_f32<64>(a, batch, max_len, s) : launch_window_prefill_f32<128>(a, batch, max_len, s);
        if (rc) return fail(rc, "%s: hipFuncSetAttribute failed (%d)", fn, rc);
        return launch_status(fn);
    }
    const int64_t units = (int64_t)max_len * heads;
    HY_BY_DTYPE(dtype, T, hipLaunchKernelGGL((window_rows_kernel<T>), dim3((unsigned)((units + 3) / 4), batch), dim3(256), 0, s, a));
    return launch_status(fn);
}

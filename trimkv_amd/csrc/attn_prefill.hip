// Multi-query (prompt chunk) GQA attention over ragged per-segment K/V with the bottom-right
// causal mask, on MFMA -- gfx950.
//
// Replaces flash_attn_varlen_func at Q_LEN > 1 with causal=True
// (src/trimkv/attn/flash_attn.py:61-71, 135-145) and HF flash_attention_2 on the dense cache during
// prefill (src/trimkv/attn/__init__.py:15-26): query t of the chunk sees every older cached token
// plus the chunk's own tokens <= t, i.e. keys j <= n - Q_LEN + t.
//
// The kernels share the formulation below.
//   prefill_small_kernel    chunks of fewer than 64 queries: 16 queries to a wavefront, 32-key tiles, 16x16x32 MFMAs, running row maxima
//   prefill_attn_kernel     longer ones whose query tiles fill the chip: 32 queries to a wavefront, two groups of MFMA columns, on 64-key tiles that LDS-direct
//                           loads rotate through four LDS buffers, 16x16x32 MFMAs, wavefronts half a block apart; fp16 keeps row maxima, bf16 none (ATTEND_SUMS)
//   prefill_shares_kernel   the same loop over equal shares of all keys, whose outputs prefill_merge_kernel puts together (trimkv_prefill_attn_shares)
//   few::prefill_few_kernel little work, or keys divided by sizes (trimkv_prefill_attn_split): 32 queries to a wavefront, 32x32x16 MFMAs, all
//                           wavefronts in step, row maxima (attn_prefill_few.hip.h)
// Which of them takes a call: launch_prefill, trimkv_prefill_split_tiles and trimkv_prefill_equal_shares.
//
// A workgroup owns BT consecutive query times of one segment for all G query heads of its KV head,
// one wavefront per (head, 16 or 32 times), so a K/V tile staged in LDS is shared by the whole group.
// Per tile a wavefront computes
//     S^T[key][query] = K . Q^T           (A = K rows from LDS, B = Q rows held in registers)
//     O^T[d][query]  += V^T . P^T         (A = V columns gathered from LDS, B = P^T)
// Both products put the query on the MFMA column index, which is the lane index modulo 16 (32 for 32x32x16): every
// per-query quantity (running max, sum, rescale factor) lives in the lane that needs it, and the
// probabilities a lane holds after the first product are exactly the keys its B operand of the
// second product wants -- P never crosses lanes.  V is row-major in memory, so its A operand
// (8 keys at one d) needs a transposition: the large kernel reads it with the transposing LDS read
// (ds_read_b64_tr_b16); the small kernel gathers 8 dwords (d, d+1) per lane and splits them into an
// even-d and an odd-d operand.
#include "common.hip.h"
#include <algorithm>
#include <type_traits>

namespace trimkv {

typedef __bf16 pf_bf16x8 __attribute__((ext_vector_type(8)));
typedef float pf_f32x4 __attribute__((ext_vector_type(4)));
typedef float pf_f32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 pf_bf16x2 __attribute__((ext_vector_type(2)));
typedef uint32_t pf_u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t pf_u32x2 __attribute__((ext_vector_type(2)));

constexpr int PF_D = 128;                  // head_dim the tiles are built for; 64 and 96 run zero-padded to it (q = 0 there)
constexpr int PF_BN = 32;                  // keys per tile
constexpr int PF_ROW = 272;                // LDS bytes per K/V row: 256 + 16 keeps b128 alignment and spreads banks
constexpr float PF_NEG = -1.0e30f;

struct PrefillArgs {
    const uint16_t* q; int64_t q_sb, q_sh, q_st;   // element strides of [B][Hq][Q][D]
    uint16_t* out;                                  // [B][Q][Hq][D] contiguous
    const char* k; const char* v;
    const int32_t* seg_len; const int32_t* seg_start;
    int kv_heads, group, q_len, cap, max_len;
    int hd;                                         // real head_dim: rows of K, V, q and out hold hd elements
    float scale_log2;
    int split_tiles; float* part; float* part_ml;   // keys split over workgroups: tiles of keys apiece, unfinished outputs, their references and sums
    int* plan; int query_tiles, items;              // equal shares: [0] units of a share, [1 + i] first unit of query tile i; query tiles of a segment, in all
};

template <int G>
struct SmallCfg {
    static constexpr int TT = G >= 4 ? 1 : (G == 3 ? 1 : 4 / G);  // 16-query time tiles per workgroup
    static constexpr int WAVES = G * TT;
    static constexpr int THREADS = WAVES * 64;
    static constexpr int BT = 16 * TT;
    static constexpr int PIECES = (2 * PF_BN * 16 + THREADS - 1) / THREADS;  // 16-byte pieces per thread per tile (K and V)
};

typedef _Float16 pf_f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 pf_f16x2 __attribute__((ext_vector_type(2)));
// K, V, q and P travel as raw 16-bit pairs (the bf16 vector types are only carriers); F16 selects how the matrix and dot
// instructions read them and how fp32 results are rounded.
template <bool F16>
__device__ __forceinline__ pf_f32x4 mfma_16x16x32(pf_bf16x8 a, pf_bf16x8 b, pf_f32x4 c) {
    if constexpr (F16) return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(pf_f16x8, a), __builtin_bit_cast(pf_f16x8, b), c, 0, 0, 0);
    else return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ uint32_t pack_f16(float lo, float hi) {
    pf_f32x2 f = {lo, hi};
    pf_f16x2 b = __builtin_convertvector(f, pf_f16x2);
    return __builtin_bit_cast(uint32_t, b);
}
__device__ __forceinline__ uint32_t pack_bf16(float lo, float hi);
template <bool F16>
__device__ __forceinline__ uint32_t pack_kv(float lo, float hi) { return F16 ? pack_f16(lo, hi) : pack_bf16(lo, hi); }
// l + p.lo + p.hi for a packed pair of probabilities (a dot product with a pair of ones)
template <bool F16>
__device__ __forceinline__ float add_pair(uint32_t pw, float l) {
    if constexpr (F16) return __builtin_amdgcn_fdot2(__builtin_bit_cast(pf_f16x2, pw), __builtin_bit_cast(pf_f16x2, 0x3C003C00u), l, false);
    else return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(pf_bf16x2, pw), __builtin_bit_cast(pf_bf16x2, 0x3F803F80u), l, false);
}

__device__ __forceinline__ uint32_t pack_bf16(float lo, float hi) {
    pf_f32x2 f = {lo, hi};
    pf_bf16x2 b = __builtin_convertvector(f, pf_bf16x2);
    return __builtin_bit_cast(uint32_t, b);
}

// SPLIT: blockIdx.z takes split_tiles * 64 keys (see prefill_attn_kernel); the unfinished rows lie one behind the other, 128 floats each
template <int G, bool F16, bool SPLIT>
__global__ __launch_bounds__(SmallCfg<G>::THREADS) void prefill_small_kernel(PrefillArgs a) {
    using C = SmallCfg<G>;
    __shared__ __attribute__((aligned(16))) char lds_k[PF_BN * PF_ROW];
    __shared__ __attribute__((aligned(16))) char lds_v[PF_BN * PF_ROW];

    const int seg = blockIdx.y;
    const int tile = (int)gridDim.x - 1 - (int)blockIdx.x;  // later times see more keys: dispatch them first
    const int b = seg / a.kv_heads, h = seg - b * a.kv_heads;
    int n = a.seg_len ? a.seg_len[seg] : a.max_len;
    n = max(0, min(n, a.max_len));
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const int g = w % G, tt = w / G;
    const int j = lane & 15, ig = lane >> 4;   // MFMA column (query) and row group
    const int Q = a.q_len;
    const int t_wg0 = tile * C::BT;
    const int t_q = t_wg0 + tt * 16 + j;        // this lane's query time
    const bool q_ok = t_q < Q;
    const int64_t row0 = a.seg_start ? (int64_t)a.seg_start[seg] : (int64_t)seg * a.cap;

    // Q fragments: B operand of S^T = K.Q^T; lane (query j, k-group ig) holds bytes [ig*64 + ks*16, +16) of its row
    pf_bf16x8 qf[4];
    {
        const uint16_t* qrow = a.q + (int64_t)b * a.q_sb + (int64_t)(h * G + g) * a.q_sh + (int64_t)min(t_q, Q - 1) * a.q_st;
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) {
            const int e0 = ig * 32 + ks * 8;
            qf[ks] = *(const pf_bf16x8*)(qrow + min(e0, a.hd - 8));
            if (e0 >= a.hd) qf[ks] = pf_bf16x8{0, 0, 0, 0, 0, 0, 0, 0};   // padded features: whatever K holds there counts for nothing
        }
    }

    pf_f32x4 oe[4], oo[4];  // O^T accumulators: d = 2*(pb*16 + 4*ig + v) (even) and +1 (odd), query j
#pragma unroll
    for (int pb = 0; pb < 4; ++pb) { oe[pb] = {0.f, 0.f, 0.f, 0.f}; oo[pb] = {0.f, 0.f, 0.f, 0.f}; }
    float m_run = PF_NEG, l_run = 0.0f;

    // keys the workgroup has to visit: everything its last query may see
    const int t_last = min(Q - 1, t_wg0 + C::BT - 1);
    const int all_keys = max(0, min(n, n - Q + t_last + 1));
    const int k_first = SPLIT ? (int)blockIdx.z * a.split_tiles * 64 : 0;
    if (SPLIT && k_first > 0 && k_first >= all_keys) return;
    const int k_end = SPLIT ? min(all_keys, k_first + a.split_tiles * 64) : all_keys;
    const int vis_j = n - Q + t_q;              // last key visible to this lane's query
    const int vis_wave_max = n - Q + min(Q - 1, t_wg0 + tt * 16 + 15);

    // cooperative tile load: piece p of 2*32*16 (K rows then V rows), 16 bytes each
    pf_u32x4 stage[C::PIECES];
    auto fetch = [&](int kbase) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < C::PIECES; ++i) {
            const int p = tid + i * C::THREADS;
            if (p < 2 * PF_BN * 16) {
                const int isv = p >= PF_BN * 16, q16 = p & 15, key = (p >> 4) & (PF_BN - 1);
                const int row = min(kbase + key, max(n - 1, 0));
                const char* src = (isv ? a.v : a.k) + (row0 + row) * (int64_t)(a.hd * 2) + min(q16 * 16, a.hd * 2 - 16);
                stage[i] = *(const pf_u32x4*)src;
            }
        }
    };
    auto publish = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < C::PIECES; ++i) {
            const int p = tid + i * C::THREADS;
            if (p < 2 * PF_BN * 16) {
                const int isv = p >= PF_BN * 16, q16 = p & 15, key = (p >> 4) & (PF_BN - 1);
                *(pf_u32x4*)((isv ? lds_v : lds_k) + key * PF_ROW + q16 * 16) = stage[i];
            }
        }
    };

    if (k_end > k_first) fetch(k_first);
    for (int kbase = k_first; kbase < k_end; kbase += PF_BN) {
        __syncthreads();   // everyone is done reading the previous tile
        publish();
        __syncthreads();   // the tile is visible
        if (kbase + PF_BN < k_end) fetch(kbase + PF_BN);   // next tile in flight during the arithmetic

        if (kbase <= vis_wave_max) {   // wave-uniform: some query of this wavefront sees part of the tile
            // ---- S^T = K . Q^T for the two 16-key blocks ----
            pf_f32x4 s[2];
#pragma unroll
            for (int kb = 0; kb < 2; ++kb) {
                s[kb] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int ks = 0; ks < 4; ++ks) {
                    const pf_bf16x8 kf = *(const pf_bf16x8*)(lds_k + (kb * 16 + j) * PF_ROW + ig * 64 + ks * 16);
                    s[kb] = mfma_16x16x32<F16>(kf, qf[ks], s[kb]);
                }
            }
            // lane holds keys kbase + kb*16 + 4*ig + v of query j
            float tmax = PF_NEG;
#pragma unroll
            for (int kb = 0; kb < 2; ++kb) {
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    const int key = kbase + kb * 16 + 4 * ig + v;
                    const float x = (key <= vis_j && q_ok) ? s[kb][v] * a.scale_log2 : PF_NEG;
                    s[kb][v] = x;
                    tmax = fmaxf(tmax, x);
                }
            }
            tmax = fmaxf(tmax, __shfl_xor(tmax, 16, 64));
            tmax = fmaxf(tmax, __shfl_xor(tmax, 32, 64));
            const float m_new = fmaxf(m_run, tmax);
            const float alpha = __builtin_amdgcn_exp2f(m_run - m_new);
            m_run = m_new;
            float psum = 0.0f;
            float p[2][4];
#pragma unroll
            for (int kb = 0; kb < 2; ++kb) {
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    // a row that sees nothing keeps m == PF_NEG: exp2(0) would be 1, so mask explicitly
                    p[kb][v] = s[kb][v] > 0.5f * PF_NEG ? __builtin_amdgcn_exp2f(s[kb][v] - m_new) : 0.0f;
                    psum += p[kb][v];
                }
            }
            l_run = l_run * alpha + psum;
#pragma unroll
            for (int pb = 0; pb < 4; ++pb) {
#pragma unroll
                for (int v = 0; v < 4; ++v) { oe[pb][v] *= alpha; oo[pb][v] *= alpha; }
            }
            // P^T operand: k index e <-> key (e < 4 ? 4*ig + e : 16 + 4*ig + e - 4), all in this lane
            const uint4 pw = make_uint4(pack_kv<F16>(p[0][0], p[0][1]), pack_kv<F16>(p[0][2], p[0][3]),
                                        pack_kv<F16>(p[1][0], p[1][1]), pack_kv<F16>(p[1][2], p[1][3]));
            const pf_bf16x8 pfrag = __builtin_bit_cast(pf_bf16x8, pw);
            // ---- O^T += V^T . P^T: A = 8 keys at d pair (pb*16 + j): dwords (d, d+1), split even/odd ----
#pragma unroll
            for (int pb = 0; pb < 4; ++pb) {
                uint32_t dw[8];
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const int key = (e < 4) ? (4 * ig + e) : (16 + 4 * ig + e - 4);
                    dw[e] = *(const uint32_t*)(lds_v + key * PF_ROW + (pb * 16 + j) * 4);
                }
                uint32_t ev[4], od[4];
#pragma unroll
                for (int x = 0; x < 4; ++x) {
                    ev[x] = __builtin_amdgcn_perm(dw[2 * x + 1], dw[2 * x], 0x05040100u);
                    od[x] = __builtin_amdgcn_perm(dw[2 * x + 1], dw[2 * x], 0x07060302u);
                }
                const uint4 evq = make_uint4(ev[0], ev[1], ev[2], ev[3]), odq = make_uint4(od[0], od[1], od[2], od[3]);
                oe[pb] = mfma_16x16x32<F16>(__builtin_bit_cast(pf_bf16x8, evq), pfrag, oe[pb]);
                oo[pb] = mfma_16x16x32<F16>(__builtin_bit_cast(pf_bf16x8, odq), pfrag, oo[pb]);
            }
        }
    }

    // the four row groups of a query hold disjoint keys: add their sums, then normalise and store
    l_run += __shfl_xor(l_run, 16, 64);
    l_run += __shfl_xor(l_run, 32, 64);
    if (SPLIT && all_keys > a.split_tiles * 64) {
        const int64_t row = ((((int64_t)blockIdx.z * gridDim.y + seg) * gridDim.x + tile) * C::WAVES + w) * 16 + j;
        if (ig == 0) *(float2*)(a.part_ml + row * 2) = make_float2(m_run, l_run);
        float* po = a.part + row * PF_D + 8 * ig;
#pragma unroll
        for (int pb = 0; pb < 4; ++pb)
#pragma unroll
            for (int v = 0; v < 4; v += 2) *(float4*)(po + pb * 32 + 2 * v) = make_float4(oe[pb][v], oo[pb][v], oe[pb][v + 1], oo[pb][v + 1]);
        return;
    }
    if (q_ok) {
        const float inv = l_run > 0.0f ? 1.0f / l_run : 0.0f;
        uint32_t* orow = (uint32_t*)(a.out + (((int64_t)b * Q + t_q) * (a.kv_heads * G) + (h * G + g)) * a.hd);
#pragma unroll
        for (int pb = 0; pb < 4; ++pb) {
#pragma unroll
            for (int v = 0; v < 4; ++v)
                if (2 * (pb * 16 + 4 * ig + v) < a.hd) orow[pb * 16 + 4 * ig + v] = pack_kv<F16>(oe[pb][v] * inv, oo[pb][v] * inv);
        }
    }
}


// The shares of the keys put together: a workgroup per wavefront of prefill_small_kernel (16 rows), 8 features per thread.  A share
// that a row saw nothing of has sum 0 and is left out.
template <int G, bool F16>
__global__ __launch_bounds__(256) void prefill_small_merge_kernel(PrefillArgs a) {
    using C = SmallCfg<G>;
    const int seg = blockIdx.y, tile = (int)blockIdx.x / C::WAVES, w = (int)blockIdx.x % C::WAVES, tiles = (int)gridDim.x / C::WAVES;
    const int b = seg / a.kv_heads, h = seg - b * a.kv_heads, Q = a.q_len;
    int n = a.seg_len ? a.seg_len[seg] : a.max_len;
    n = max(0, min(n, a.max_len));
    const int all_keys = max(0, min(n, n - Q + min(Q - 1, tile * C::BT + C::BT - 1) + 1));
    const int share = a.split_tiles * 64, shares = (all_keys + share - 1) / share;
    if (shares <= 1) return;                     // one share: its workgroup wrote the result
    const int j = threadIdx.x >> 4, d = (threadIdx.x & 15) * 8, t_q = tile * C::BT + w / G * 16 + j;
    if (t_q >= Q || d >= a.hd) return;
    const int64_t row = (((int64_t)seg * tiles + tile) * C::WAVES + w) * 16 + j, per_share = (int64_t)gridDim.y * gridDim.x * 16;
    float m = -3.0e38f;
    for (int z = 0; z < shares; ++z) {
        const float2 x = *(const float2*)(a.part_ml + (row + z * per_share) * 2);
        if ((__float_as_uint(x.y) << 1) != 0) m = __builtin_fmaxf(m, x.x);
    }
    float l = 0.0f, o[8] = {};
#pragma unroll 4
    for (int z = 0; z < shares; ++z) {
        const float2 x = *(const float2*)(a.part_ml + (row + z * per_share) * 2);
        const float* po = a.part + (row + z * per_share) * PF_D + d;
        const float4 lo = *(const float4*)po, hi = *(const float4*)(po + 4);
        const float f = (__float_as_uint(x.y) << 1) != 0 ? __builtin_amdgcn_exp2f(x.x - m) : 0.0f;
        l += x.y * f;
        o[0] += lo.x * f; o[1] += lo.y * f; o[2] += lo.z * f; o[3] += lo.w * f;
        o[4] += hi.x * f; o[5] += hi.y * f; o[6] += hi.z * f; o[7] += hi.w * f;
    }
    const float inv = l > 0.0f ? 1.0f / l : 0.0f;
    uint16_t* out = a.out + (((int64_t)b * Q + t_q) * (a.kv_heads * G) + h * G + w % G) * a.hd + d;
    *(uint4*)out = make_uint4(pack_kv<F16>(o[0] * inv, o[1] * inv), pack_kv<F16>(o[2] * inv, o[3] * inv),
                              pack_kv<F16>(o[4] * inv, o[5] * inv), pack_kv<F16>(o[6] * inv, o[7] * inv));
}

// ---------------------------------------------------------------------------------------------
// Large-chunk kernel: 32 queries per wavefront, 64-key tiles, v_mfma_f32_16x16x32_bf16.
//
// MFMA 16x16x32 register layout (lane l, row group ig = l / 16):
//   A (16 x 32): row l % 16, k = 8 * ig + 0..7          B (32 x 16): column l % 16, k = 8 * ig + 0..7
//   C (16 x 16): column l % 16, register v holds row 4 * ig + v
// S^T = K . Q^T per 32-key block, two groups of 16 keys by two of 16 queries: after it a lane holds, for its query of either group,
// keys 4 ig + 0..3 and 16 + 4 ig + 0..3.  The second product consumes 32 keys per MFMA; its k index 8 ig + e stands for key 4 ig + e (e < 4) or
// 16 + 4 ig + e - 4, so that a lane's probabilities are its B operand.
//
// For launches that fill the chip; the others, and keys in shares by sizes, are attn_prefill_few.hip.h's.
// What bounds it is the clock that the chip holds under matrix load, and beside it the issue of vector instructions: matrix cores and vector ALU of a SIMD
// take turns when two wavefronts want both.  16x16x32 products cost less of the clock than 32x32x16 (registers only, random operands: 2.06 against 1.80 PFLOP/s at
// 2.02 and 1.76 GHz), but leave less room beside them (with two and four vector instructions per 32 cycles of product 1.85 | 1.66 and 1.64 | 1.55).  Hence
// the parts of a block in which one wavefront of a SIMD only multiplies while the other does the rest (`block` below), and in bf16 no row
// maxima (ATTEND_SUMS): 16 exponentials, 8 packs and 8 row sums per 32 products are left.
// 16 segments of 12288 keys, 4096 queries of 5 heads: 1.17 PFLOP/s with 32x32x16, exponentials between the products and matrix pipes busy
// 73 % at 1.58 GHz; the same with 16x16x32 1.16, 59 % at 1.88; in two parts 1.22; without maxima 1.28 PFLOP/s, 69 % at 1.77.  Row sums on the matrix cores as well
// (32 more cycles of them, 8 vector instructions less): +1 %, and -1 % where shares are equal; packs and row sums in the part that multiplies:
// 0.97; V read in the part that does not: 1.19.
//
// K and V tiles are staged by LDS-direct loads (global_load_lds_dwordx4): a tile never passes through registers and
// no VALU instruction takes part in staging.
// LDS: four K tiles [64 rows][256 B] in the low 64 KB, four V tiles (also row-major) in the next 64 KB.  A wavefront's
// load instruction fills 1 KB (lane l lands at +16 l), i.e. four whole rows; which 16-byte piece of global memory a
// lane fetches is free, and that is where the bank swizzle comes from:
//   K: piece c of row r sits at position c ^ (r & 15): the 16 rows a b128 fragment read touches (one piece index,
//      consecutive rows) fall on all 64 banks.
//   V: the 32-byte pair p of row r sits at pair position p ^ pf2_v_swizzle(r).  The A operand of O^T += V^T.P^T (8 keys at
//      one d per lane) is read with two ds_read_b64_tr_b16: within 16 lanes, lane i supplies 8 bytes (4 d of one key,
//      key = base + i / 4, d = d0 + 4 (i % 4) ..) and receives the four keys base .. base + 3 at d = d0 + i.
// The compiler does not see the LDS-direct loads (inline assembly: the builtin would make it wait for all of them before
// every LDS read), so it neither counts them nor waits for them: every wait is written out in the kernel, including
// the one before the wavefront ends.
// ---------------------------------------------------------------------------------------------
typedef float pf_f32x16 __attribute__((ext_vector_type(16)));
typedef short pf_s16x4 __attribute__((ext_vector_type(4)));
#define PF_LDS3 __attribute__((address_space(3)))

constexpr int PF2_BN = 64;                          // keys per tile (two 32-key blocks)
constexpr int PF2_NBUF = 4;                         // tiles in rotation: two being read, two on their way
constexpr int PF2_TILE = PF2_BN * PF_D * 2;         // bytes of one K (or V) tile: rows of 256 bytes
constexpr int PF2_VBASE = PF2_NBUF * PF2_TILE;      // 65536: K tiles below, V tiles above
constexpr int PF2_LDS = 2 * PF2_NBUF * PF2_TILE;    // 131072
constexpr float PF2_LAZY = 6.0f;                    // O is rescaled only when a row maximum grows by more than 2^6

// A workgroup is always 8 wavefronts (two per SIMD, 256 registers each) and owns 256 / G consecutive query times
// for all G heads: MFMA column c of wavefront w is row r = 32w + c of the workgroup, time r / G, head r % G.
// Every per-query quantity is per lane, so a wavefront may mix heads freely; time-major rows keep the
// spread of a wavefront's causal limits small.
constexpr float PF2_MOST = 1.0e12f;                 // without maxima: 2^40, the row sum from which on O is rescaled

constexpr int PF2_WAVES = 8;
constexpr int PF2_THREADS = PF2_WAVES * 64;
static_assert(PF2_THREADS * 2 * 16 == PF2_TILE, "a thread stages two 16-byte pieces of K and two of V per tile");

// One LDS-direct load of 16 bytes per lane: lane l's bytes land at LDS address lds_addr + 16 l.
__device__ __forceinline__ void pf2_load_to_lds(const char* sbase, uint32_t voff, uint32_t lds_addr) {
    uint32_t saved;
    asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %3\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2\n\ts_mov_b32 m0, %0"
                 : "=&s"(saved) : "v"(voff), "s"(sbase), "s"(lds_addr) : "memory");
}

// V: where the 32-byte pairs of row r lie (pair p at p ^ this): the rows that 32 lanes of a transposing read touch fall on different banks
__device__ __forceinline__ int pf2_v_swizzle(int r) { return 2 * (r & 3) + ((r >> 2) & 1); }

// tiles of keys that the last query of a query tile sees
__device__ __forceinline__ int tiles_seen(const PrefillArgs& a, int seg, int tile) {
    int n = a.seg_len ? a.seg_len[seg] : a.max_len;
    n = max(0, min(n, a.max_len));
    const int BT = (PF2_WAVES * 32) / a.group, t_last = min(a.q_len - 1, tile * BT + BT - 1);
    return (max(0, min(n, n - a.q_len + t_last + 1)) + PF2_BN - 1) / PF2_BN;
}
// units of query tile i of the launch where shares are equal: its key tiles, one if it sees nothing (its output is written all the same)
__device__ __forceinline__ int units_of(const PrefillArgs& a, int i) {
    const int seg = i / a.query_tiles;
    return max(1, tiles_seen(a, seg, i - seg * a.query_tiles));
}
constexpr int PF2_GROUPS = 256;                     // one workgroup per CU
constexpr int PF2_LEAST = 4;                        // units of a share at least

}  // namespace trimkv
#include "attn_prefill_few.hip.h"
namespace trimkv {

// One query tile against `count` tiles of keys from tile t_first on (PART; else against all of them).  Where that is not all that the
// query tile sees, unnormalised outputs with their exponent references and row sums (fp32) are left in `slot` for a merge kernel.
//
// HOW: what keeps the exponentials in range.  ATTEND_MAXIMA (fp16): the exponent reference of a row stays within 2^PF2_LAZY of its largest score.  ATTEND_SUMS (bf16,
// whose P has fp32's exponents): once set it moves only where the row's sum has grown beyond PF2_MOST, which takes no maxima; a score that exceeds the
// reference by 2^7 within a block overflows then, and whatever is not finite at the end (an input that is not among it) sets *again (0 before), for
// the caller to have it done again with ATTEND_MAXIMA over what it has written.
// What that costs falls on query tiles with a row that holds a score more than 88 nats above the first block's largest, or a value that is not finite.  16 segments of
// 6000 keys, 2048 queries of 4 heads: 246 us without (272 for the loop of few::, which has maxima always), 387 where one query tile of 32 of each segment has such
// a row, 444 where each one has, 497 where all rows are such.
enum { ATTEND_MAXIMA, ATTEND_SUMS };
template <bool F16, bool PART, int HOW>
__device__ __forceinline__ void attend_query_tile(const PrefillArgs& a, int seg, int tile, int t_first, int count, int64_t slot, PF_LDS3 int* again) {
    constexpr bool MAXIMA = HOW != ATTEND_SUMS;
    extern __shared__ __attribute__((aligned(16))) char pf2_lds[];
    PF_LDS3 char* const lds3 = (PF_LDS3 char*)pf2_lds;
    const uint32_t lds0 = (uint32_t)(uintptr_t)lds3;
    const int b = seg / a.kv_heads, h = seg - b * a.kv_heads;
    int n = a.seg_len ? a.seg_len[seg] : a.max_len;
    n = max(0, min(n, a.max_len));
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));                             // nothing of a query tile is worth a register during the one before it
    const int lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);   // wave-uniform by construction; saying so keeps what derives from it in scalar registers
    const int j = lane & 15, ig = lane >> 4;    // MFMA column (query, of either group of 16) and row group
    const int G = a.group, Q = a.q_len;
    const int BT = (PF2_WAVES * 32) / G;        // query times per workgroup; rows BT * G .. 255 are padding
    const int t_wg0 = tile * BT;
    const int t_w_first = t_wg0 + (w * 32) / G;
    const int64_t row0 = a.seg_start ? (int64_t)a.seg_start[seg] : (int64_t)seg * a.cap;

    // The rows of Q are asked for in front of the first keys and turned into fragments behind them: one memory round trip for both.
    pf_u32x4 qraw[2][4];
    int vis_j[2];                               // last key that this lane's query of either group sees
#pragma unroll
    for (int qg = 0; qg < 2; ++qg) {
        const int r = w * 32 + qg * 16 + j, t_q = t_wg0 + r / G;
        vis_j[qg] = n - Q + t_q;
        const uint16_t* qrow = a.q + (int64_t)b * a.q_sb + (int64_t)(h * G + r % G) * a.q_sh + (int64_t)min(t_q, Q - 1) * a.q_st;
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) qraw[qg][ks] = *(const pf_u32x4*)(qrow + min(ks * 32 + ig * 8, a.hd - 8));
    }

    // O^T: o[dg / 2][8 (dg % 2) + 4 qg + v] = d (16 dg + 4 ig + v) of query 16 qg + j.  Blocks of 16 and not of 4: the compiler gives a block of 4 other
    // registers with every MFMA and copies all of them back where the rescaling branch joins, a part of a larger block stays where it is.
    pf_f32x16 o[4];
#pragma unroll
    for (int db = 0; db < 4; ++db)
#pragma unroll
        for (int v = 0; v < 16; ++v) o[db][v] = 0.0f;
    auto o_of = [&](int dg, int qg, int v) __attribute__((always_inline)) { return o[dg >> 1][8 * (dg & 1) + 4 * qg + v]; };
    // Exponent references (log2 units) and this lane's shares of the row sums.  The score MFMAs start from -m_ref in their
    // accumulator (negm, all 4 registers alike: a lane is one query), so what they deliver is already s - m_ref.  The
    // reference starts at 0 and is moved onto the row maximum by the first block.  A query that sees no key at all
    // (segment shorter than the chunk) keeps reference 0: its masked scores give exp2(-huge) = 0, never exp2(0).
    float m_ref[2] = {0.0f, 0.0f}, l_run[2] = {0.0f, 0.0f};
    pf_f32x4 negm[2] = {{0.0f, 0.0f, 0.0f, 0.0f}, {0.0f, 0.0f, 0.0f, 0.0f}};

    const int t_last = min(Q - 1, t_wg0 + BT - 1);
    const int k_end = max(0, min(n, n - Q + t_last + 1));     // keys the query tile sees
    const int all_tiles = (k_end + PF2_BN - 1) / PF2_BN;
    const int vis_lo = n - Q + t_w_first;                     // last key that the wavefront's first query sees
    const int last_row = max(n - 1, 0);

    // ---- staging: global -> LDS ----
    // Thread tid fetches, for K and for V, one 16-byte piece of row tid / 16 and one of row 32 + tid / 16 of the tile; the
    // piece it fetches is the one whose swizzled position is tid % 16 (hd < 128: pieces past the row re-read its last one,
    // q is zero there and those columns of O are not stored).
    const uint32_t row_bytes = (uint32_t)a.hd * 2u;
    const char* kseg = a.k + row0 * (int64_t)row_bytes;
    const char* vseg = a.v + row0 * (int64_t)row_bytes;
    const int st_row = tid >> 4, st_pos = tid & 15;
    const uint32_t st_kcol = min((uint32_t)(st_pos ^ (st_row & 15)) * 16u, row_bytes - 16u);
    const uint32_t st_vcol = min((uint32_t)((((st_pos >> 1) ^ pf2_v_swizzle(st_row)) << 1) | (st_pos & 1)) * 16u, row_bytes - 16u);
    const uint32_t st_koff = (uint32_t)st_row * row_bytes + st_kcol;     // offsets inside a tile whose 64 rows all exist
    const uint32_t st_voff = (uint32_t)st_row * row_bytes + st_vcol;
    auto request_tile = [&](int tt, int buf) __attribute__((always_inline)) {
        const int kbase = (t_first + tt) * PF2_BN;
        const uint32_t dk = lds0 + buf * PF2_TILE + w * 1024, dv = dk + PF2_VBASE;
        if (kbase + PF2_BN <= n) {   // wave-uniform; the tile's base goes into the scalar base address
            const char* kt = kseg + (uint32_t)kbase * row_bytes;
            const char* vt = vseg + (uint32_t)kbase * row_bytes;
            pf2_load_to_lds(kt, st_koff, dk);
            pf2_load_to_lds(kt + 32 * row_bytes, st_koff, dk + PF2_TILE / 2);
            pf2_load_to_lds(vt, st_voff, dv);
            pf2_load_to_lds(vt + 32 * row_bytes, st_voff, dv + PF2_TILE / 2);
        } else {                     // rows past the segment's end are replaced by its last row (finite values, masked keys)
            const uint32_t r0 = (uint32_t)min(kbase + st_row, last_row) * row_bytes;
            const uint32_t r1 = (uint32_t)min(kbase + st_row + 32, last_row) * row_bytes;
            pf2_load_to_lds(kseg, r0 + st_kcol, dk);
            pf2_load_to_lds(kseg, r1 + st_kcol, dk + PF2_TILE / 2);
            pf2_load_to_lds(vseg, r0 + st_vcol, dv);
            pf2_load_to_lds(vseg, r1 + st_vcol, dv + PF2_TILE / 2);
        }
    };

    const int ntiles = PART ? min(all_tiles - t_first, count) : all_tiles;
    if (ntiles > 0) {
        request_tile(0, 0);
        request_tile(1, 1);
    }
    // Q fragments (B operand of S^T): 8 d of step ks at d = ks * 32 + ig * 8, multiplied by scale * log2(e) and rounded back
    // to 16 bits once, here: the score MFMAs then deliver exponents of two directly and the loop never multiplies a score.
    pf_bf16x8 qf[2][4];
#pragma unroll
    for (int qg = 0; qg < 2; ++qg)
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) {
            pf_u32x4 sc;
#pragma unroll
            for (int x = 0; x < 4; ++x) {
                const uint32_t raw = qraw[qg][ks][x];
                float lo, hi;
                if (F16) { lo = f16_bits_to_f32((uint16_t)(raw & 0xffffu)); hi = f16_bits_to_f32((uint16_t)(raw >> 16)); }
                else { lo = __uint_as_float(raw << 16); hi = __uint_as_float(raw & 0xffff0000u); }
                sc[x] = pack_kv<F16>(lo * a.scale_log2, hi * a.scale_log2);
            }
            if (ks * 32 + ig * 8 >= a.hd) sc = pf_u32x4{0u, 0u, 0u, 0u};   // padded features: whatever K holds there counts for nothing
            qf[qg][ks] = __builtin_bit_cast(pf_bf16x8, sc);
        }

    // per-lane LDS read offsets; the buffer, the 32-key block, the key group and the step are immediates on top of them
    PF_LDS3 char* k_ptr[4];
    PF_LDS3 char* v_ptr[8];
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
        k_ptr[ks] = lds3 + (j * 256 + (((4 * ks + ig) ^ j) << 4));
        asm volatile("" : "+v"(k_ptr[ks]));          // a value in a register from here on, not an expression to recompute in the loop
    }
    {
        const int kx = 4 * ig + (j >> 2);            // key (within its group of 16) this lane supplies to the transposing read
#pragma unroll
        for (int dg = 0; dg < 8; ++dg) {
            v_ptr[dg] = lds3 + (PF2_VBASE + kx * 256 + ((dg ^ pf2_v_swizzle(kx)) << 5) + (j & 3) * 8);
            asm volatile("" : "+v"(v_ptr[dg]));
        }
    }
    // fragment m of a block's keys: step m / 2, keys 16 (m % 2) ..
    auto k_frag = [&](int imm, int m) __attribute__((always_inline)) {
        return *(const PF_LDS3 pf_bf16x8*)(k_ptr[m >> 1] + imm + (m & 1) * 16 * 256);
    };
    auto v_frag = [&](int imm, int dg) __attribute__((always_inline)) {
        PF_LDS3 char* p = v_ptr[dg] + imm;
        const pf_s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((PF_LDS3 pf_s16x4*)p);                 // keys 4 ig + 0..3
        const pf_s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((PF_LDS3 pf_s16x4*)(p + 16 * 256));    // ... + 16
        return __builtin_bit_cast(pf_bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
    };
    struct Scores { pf_f32x4 g[2][2]; };             // g[kg][qg][v]: key 16 kg + 4 ig + v of the block, query 16 qg + j
    struct Pair { float x[2]; };                     // of the lane's two queries

    // Mask (diagonal blocks only), row maximum, and the lazy move of the exponent reference: O and l are
    // rescaled only when some row of the wavefront outgrows its reference by 2^PF2_LAZY.  FIRST: the wavefront's first
    // block puts the reference on the row maximum wherever it lies (O and l are still zero: nothing to rescale).
    // tmax: the maximum of s before masking, as the step computed it under its P.V MFMAs (ignored by FIRST).
    auto max8 = [&](const Scores& s, int qg) __attribute__((always_inline)) {
        float t = s.g[0][qg][0];
#pragma unroll
        for (int v = 1; v < 8; ++v) t = __builtin_fmaxf(t, s.g[v >> 2][qg][v & 3]);
        return t;
    };
    auto prepare = [&](Scores& s, int blk, Pair tmax, auto first_c, auto look_c) __attribute__((always_inline)) {
        constexpr bool FIRST = decltype(first_c)::value, LOOK = FIRST || MAXIMA || decltype(look_c)::value;     // sums are looked at now and then
        const int key0 = (blk + 2 * t_first) * 32;
        if (key0 + 31 > vis_lo) {   // wave-uniform: some query of the wavefront does not see the whole block
            // (the empty volatile statement keeps this a branch: as 48 speculated selects it would run for every block)
            asm volatile("" ::: );
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                const int key = key0 + 16 * (v >> 3) + 4 * ig + (v & 3), qg = (v >> 2) & 1;
                s.g[v >> 3][qg][v & 3] = key <= vis_j[qg] ? s.g[v >> 3][qg][v & 3] : PF_NEG;
            }
            if (MAXIMA && !FIRST) tmax = Pair{{max8(s, 0), max8(s, 1)}};
        }
        if (FIRST) tmax = Pair{{max8(s, 0), max8(s, 1)}};
        if (!FIRST && !MAXIMA) tmax = Pair{{l_run[0], l_run[1]}};
        if (FIRST || (LOOK && __builtin_amdgcn_ballot_w64(__builtin_fmaxf(tmax.x[0], tmax.x[1]) > (MAXIMA ? PF2_LAZY : PF2_MOST)) != 0)) {
#pragma unroll
            for (int qg = 0; qg < 2; ++qg) {
                float t2 = __builtin_fmaxf(tmax.x[qg], __shfl_xor(tmax.x[qg], 16, 64));   // the four row groups of a query agree on the reference
                t2 = __builtin_fmaxf(t2, __shfl_xor(t2, 32, 64));
                // how far the reference moves: onto the maximum (first block; not at all for a row that sees nothing), else up only; without maxima by the
                // exponent of the largest sum (0 of what is not finite)
                const float d = FIRST ? (t2 > 0.5f * PF_NEG ? t2 : 0.0f) : MAXIMA ? __builtin_fmaxf(t2, 0.0f) : __builtin_fmaxf((float)__builtin_amdgcn_frexp_expf(t2), 0.0f);
                m_ref[qg] += d;
#pragma unroll
                for (int v = 0; v < 4; ++v) { s.g[0][qg][v] -= d; s.g[1][qg][v] -= d; negm[qg][v] = -m_ref[qg]; }
                if (!FIRST) {
                    // Sums of 2^126 and more move the reference by 127 or 128, and v_exp_f32 gives 0 there instead of the denormal number: they are scaled by their
                    // exponent.  What a maximum that far away does not leave is nothing to the new one.
                    const float alpha = MAXIMA ? __builtin_amdgcn_exp2f(-d) : 0.0f;
                    auto moved = [&](float x) __attribute__((always_inline)) { return MAXIMA ? x * alpha : __builtin_ldexpf(x, -(int)d); };
                    l_run[qg] = moved(l_run[qg]);
#pragma unroll
                    for (int dg = 0; dg < 8; ++dg)
#pragma unroll
                        for (int v = 0; v < 4; ++v) o[dg >> 1][8 * (dg & 1) + 4 * qg + v] = moved(o[dg >> 1][8 * (dg & 1) + 4 * qg + v]);
                }
            }
        }
    };
    // P = exp2(s - ref) as bf16 (two scores -> one dword) and the row sum of the rounded P; pair x = 4 qg + 2 kg + half: in the order in
    // which the P operand takes them
    auto p_pair = [&](const Scores& s, int x) __attribute__((always_inline)) {
        const int qg = x >> 2, kg = (x >> 1) & 1, v = 2 * (x & 1);
        const float p0 = __builtin_amdgcn_exp2f(s.g[kg][qg][v]);
        const float p1 = __builtin_amdgcn_exp2f(s.g[kg][qg][v + 1]);
        const uint32_t pw = pack_kv<F16>(p0, p1);
        l_run[qg] = add_pair<F16>(pw, l_run[qg]);
        return pw;
    };
    auto meet = [&]() __attribute__((always_inline)) {
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("s_barrier" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
    };
    // A block of 32 keys has two parts: the exponentials of its scores while the LDS operands of what follows are read, then 32 MFMAs, P.V of the
    // block and the scores of the next one.  The wavefronts 4 .. 7 are one part behind the others, so that on every SIMD one
    // wavefront multiplies while the other one does everything else; the barrier between the parts keeps them so.
    //   vimm, kimm: byte offsets of this block's V and of the next block's K; LAND: the tile after this one has landed behind this part
    auto max3 = [](float x, float y, float z) __attribute__((always_inline)) { return __builtin_fmaxf(__builtin_fmaxf(x, y), z); };
    auto block = [&](Scores& s, auto vimm, auto kimm, auto land) __attribute__((always_inline)) -> Pair {
        pf_bf16x8 kf[8], vf[8];
#pragma unroll
        for (int m = 0; m < 8; ++m) kf[m] = k_frag(kimm, m);
        pf_bf16x8 pfrag[2];
        uint32_t pw[8];
#pragma unroll
        for (int x = 0; x < 8; ++x) pw[x] = p_pair(s, x);
#pragma unroll
        for (int qg = 0; qg < 2; ++qg) {
            const pf_u32x4 pq = {pw[4 * qg], pw[4 * qg + 1], pw[4 * qg + 2], pw[4 * qg + 3]};
            pfrag[qg] = __builtin_bit_cast(pf_bf16x8, pq);
        }
        asm volatile("" : "+v"(pfrag[0]), "+v"(pfrag[1]), "+v"(l_run[0]), "+v"(l_run[1]));
        __builtin_amdgcn_sched_barrier(0);
        if (decltype(land)::value) asm volatile("s_waitcnt vmcnt(4)\n\ts_barrier" ::: "memory");      // (the four loads of the tile after it may still be in flight)
        else asm volatile("s_barrier" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_setprio(1);
#pragma unroll
        for (int m = 0; m < 8; ++m) {
            vf[m] = v_frag(vimm, m);
#pragma unroll
            for (int qg = 0; qg < 2; ++qg) s.g[m & 1][qg] = mfma_16x16x32<F16>(kf[m], qf[qg][m >> 1], m < 2 ? negm[qg] : s.g[m & 1][qg]);
            __builtin_amdgcn_sched_barrier(0);
        }
        float mt[2][3];
        Pair mx = {{0.0f, 0.0f}};
#pragma unroll
        for (int m = 0; m < 8; ++m) {
#pragma unroll
            for (int qg = 0; qg < 2; ++qg) {
                pf_f32x16& all = o[m >> 1];
                const int at = 8 * (m & 1) + 4 * qg;
                const pf_f32x4 r = mfma_16x16x32<F16>(vf[m], pfrag[qg], pf_f32x4{all[at], all[at + 1], all[at + 2], all[at + 3]});
#pragma unroll
                for (int v = 0; v < 4; ++v) all[at + v] = r[v];
            }
            if (MAXIMA && m >= 2) {          // trees of three-input maxima (the last score MFMA has landed by then)
                const int qg = m & 1;
                const pf_f32x4 lo = s.g[0][qg], hi = s.g[1][qg];
                if (m < 4) { mt[qg][0] = max3(lo[0], lo[1], lo[2]); asm volatile("" : "+v"(mt[qg][0])); }
                else if (m < 6) { mt[qg][1] = max3(hi[0], hi[1], hi[2]); asm volatile("" : "+v"(mt[qg][1])); }
                else {
                    mt[qg][2] = max3(lo[3], hi[3], mt[qg][0]);
                    mx.x[qg] = __builtin_fmaxf(mt[qg][1], mt[qg][2]);
                    asm volatile("" : "+v"(mx.x[qg]));
                }
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        __builtin_amdgcn_s_setprio(0);
        meet();
        return mx;
    };

    // Every wavefront walks all blocks of the workgroup's tiles: the blocks that
    // lie wholly above a wavefront's diagonal (at most two of up to several hundred, the workgroup spans BT query times)
    // are masked like the diagonal ones and contribute zeros, which keeps the loop free of per-wavefront branches.
    if (ntiles > 0) {
        Scores s;
        asm volatile("s_waitcnt vmcnt(4)" ::: "memory");
        __syncthreads();
#pragma unroll
        for (int m = 0; m < 8; ++m)
#pragma unroll
            for (int qg = 0; qg < 2; ++qg) s.g[m & 1][qg] = mfma_16x16x32<F16>(k_frag(0, m), qf[qg][m >> 1], m < 2 ? negm[qg] : s.g[m & 1][qg]);
        prepare(s, 0, Pair{{0.0f, 0.0f}}, std::true_type{}, std::true_type{});
        if (w >= PF2_WAVES / 2) meet();
        // Iteration t (tile t in the buffer at off0, tile t + 1 at off1): blocks 2t and 2t + 1, and the scores of block 2t + 2.
        // Tile t + 2 is requested first, into the buffer tile t - 2 used (every wavefront has left it).  Behind the first part of block 2t tile t + 1 has landed
        // everywhere, in time for the K that the second block's first part reads.
        auto iteration = [&](int t, int b2, auto off0, auto off1, auto look) __attribute__((always_inline)) {
            constexpr std::integral_constant<int, PF2_TILE / 2> half{};
            request_tile(t + 2, b2);          // unconditional (rows clamped): the count of loads in flight stays fixed
            const Pair ma = block(s, off0, off0 + half, std::true_type{});
            prepare(s, 2 * t + 1, ma, std::false_type{}, std::false_type{});
            const Pair mb = block(s, off0 + half, off1, std::false_type{});
            prepare(s, 2 * t + 2, mb, std::false_type{}, look);
        };
        using I0 = std::integral_constant<int, 0>; using I1 = std::integral_constant<int, PF2_TILE>;
        using I2 = std::integral_constant<int, 2 * PF2_TILE>; using I3 = std::integral_constant<int, 3 * PF2_TILE>;
        int t = 0;
        for (; t + 4 < ntiles; t += 4) {      // four tiles per turn: buffer offsets are immediates of the LDS reads
            iteration(t, 2, I0{}, I1{}, std::false_type{});
            iteration(t + 1, 3, I1{}, I2{}, std::false_type{});
            iteration(t + 2, 0, I2{}, I3{}, std::false_type{});
            iteration(t + 3, 1, I3{}, I0{}, std::true_type{});
        }
        // up to four more, offsets computed; the scores that the last block leaves are of keys that are not there, and nobody reads them
        for (; t < ntiles; ++t) iteration(t, (t + 2) & 3, (t & 3) * PF2_TILE, ((t + 1) & 3) * PF2_TILE, std::true_type{});
        if (w < PF2_WAVES / 2) meet();
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // the look-ahead tiles were requested too: nothing may land after the wavefront has gone
    }

    if (HOW == ATTEND_SUMS) {
        float sign = l_run[0] * 0.0f + l_run[1] * 0.0f;       // 0, or not a number
#pragma unroll
        for (int db = 0; db < 4; ++db)
#pragma unroll
            for (int v = 0; v < 16; ++v) sign = fmaf(o[db][v], 0.0f, sign);
        if (!(sign == 0.0f)) *again = 1;
    }
    // the four row groups of a query hold disjoint keys: add their sums, then normalise and store
#pragma unroll
    for (int qg = 0; qg < 2; ++qg) {
        l_run[qg] += __shfl_xor(l_run[qg], 16, 64);
        l_run[qg] += __shfl_xor(l_run[qg], 32, 64);
    }
    if (PART && all_tiles > ntiles) {
#pragma unroll
        for (int qg = 0; qg < 2; ++qg)
            if (ig == 0) *(float2*)(a.part_ml + (slot * (PF2_WAVES * 32) + w * 32 + qg * 16 + j) * 2) = make_float2(m_ref[qg], l_run[qg]);
        float4* po = (float4*)a.part + (slot * PF2_WAVES + w) * (16 * 64) + lane;   // in register order: 1 KB per store
#pragma unroll
        for (int dg = 0; dg < 8; ++dg)
#pragma unroll
            for (int qg = 0; qg < 2; ++qg) po[(qg * 8 + dg) * 64] = make_float4(o_of(dg, qg, 0), o_of(dg, qg, 1), o_of(dg, qg, 2), o_of(dg, qg, 3));
        return;
    }
    // A lane holds four features of a row at a time: stored from there, a row of 256 bytes would leave in 16 pieces.  The wavefront's
    // 32 rows take the way through LDS instead (8 KB of its own; the 16-byte piece c of row j at c ^ (j % 16)) and leave whole.
    PF_LDS3 char* const mine = lds3 + w * 8192;
    __syncthreads();                             // every wavefront has left the tiles
#pragma unroll
    for (int qg = 0; qg < 2; ++qg) {
        const float inv = l_run[qg] > 0.0f ? 1.0f / l_run[qg] : 0.0f;
#pragma unroll
        for (int dg = 0; dg < 8; ++dg)
            *(PF_LDS3 pf_u32x2*)(mine + (qg * 16 + j) * 256 + (((dg * 2 + (ig >> 1)) ^ j) << 4) + (ig & 1) * 8) =
                pf_u32x2{pack_kv<F16>(o_of(dg, qg, 0) * inv, o_of(dg, qg, 1) * inv), pack_kv<F16>(o_of(dg, qg, 2) * inv, o_of(dg, qg, 3) * inv)};
    }
    const int piece = lane & 15;
#pragma unroll
    for (int x = 0; x < 8; ++x) {
        const int row = 4 * x + (lane >> 4), rr = w * 32 + row, t = t_wg0 + rr / G;
        const pf_u32x4 v = *(const PF_LDS3 pf_u32x4*)(mine + row * 256 + ((piece ^ (row & 15)) << 4));
        if (rr < BT * G && t < Q && piece * 8 < a.hd)
            *(pf_u32x4*)(a.out + (((int64_t)b * Q + t) * (a.kv_heads * G) + (h * G + rr % G)) * a.hd + piece * 8) = v;
    }
}

// ends with every wavefront having left the LDS tiles; `again` is 0 then, as it is in front
template <bool F16, bool PART>
__device__ __forceinline__ void attend_query_tile_once(const PrefillArgs& a, int seg, int tile, int t_first, int count, int64_t slot, PF_LDS3 int* again) {
    attend_query_tile<F16, PART, F16 ? ATTEND_MAXIMA : ATTEND_SUMS>(a, seg, tile, t_first, count, slot, again);
    if (F16 && !PART) return;              // a workgroup of PART has another query tile behind this one
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");       // for LDS: nobody waits for the stores
    if (!F16 && __builtin_amdgcn_readfirstlane(*again)) {
        __syncthreads();                         // everyone has read it
        if (threadIdx.x == 0) *again = 0;
        attend_query_tile<F16, PART, ATTEND_MAXIMA>(a, seg, tile, t_first, count, slot, again);
        __syncthreads();
    }
}

// A workgroup per query tile.
template <bool F16>
__global__ __launch_bounds__(PF2_THREADS) void prefill_attn_kernel(PrefillArgs a) {
    // Workgroups are handed to the 8 XCDs round robin in dispatch order (x fastest), and each XCD has its own L2.  All
    // query tiles of a segment read the same K/V, so they are mapped to one XCD (segment s on XCD s % 8, its tiles in
    // consecutive turns of that XCD, later times first: they see more keys): the K/V tiles that several of them walk at
    // about the same time are then fetched into one L2 instead of eight.
    int seg = blockIdx.y, tile = (int)gridDim.x - 1 - (int)blockIdx.x;
    if ((gridDim.y & 7) == 0) {
        const int lin = (int)blockIdx.y * (int)gridDim.x + (int)blockIdx.x;
        const int turn = lin >> 3;
        seg = (lin & 7) + 8 * (turn / (int)gridDim.x);
        tile = (int)gridDim.x - 1 - turn % (int)gridDim.x;
    }
    __shared__ int again;
    if (threadIdx.x == 0) again = 0;             // a barrier lies between this and whoever looks at it
    attend_query_tile_once<F16, false>(a, seg, tile, 0, 0, 0, (PF_LDS3 int*)&again);
}

// Equal shares (gridDim.x workgroups, one per CU): the key tiles of all query tiles, one query tile after the other, are cut into
// runs of equal length whatever the segments' lengths are.  A run ends one query tile, takes some whole ones and begins another, so
// a workgroup leaves at most two unfinished outputs: slot 2 wg of the query tile it found begun, 2 wg + 1 of the one it leaves.
// Runs that follow each other lie on one XCD: they read the same segment.
// What it costs beyond the keys' 1.6 us per 64 of them: about 11 us per query tile begun (Q, the first keys, the pipeline's fill, the
// rows on their way out) and the unfinished outputs.  Eight layers of 24 segments of 0.69 x 4100 keys, 777 queries of 2 heads each,
// with appends and eviction 1451 -> 1317 us; sizes on either side of the rule at trimkv_prefill_equal_shares.
template <bool F16>
__global__ __launch_bounds__(PF2_THREADS) void prefill_shares_kernel(PrefillArgs a) {
    __shared__ int sums[PF2_WAVES], found[2], again;
    const int tid = threadIdx.x, lane = tid & 63, groups = (int)gridDim.x;
    const int wg = (groups & 7) ? (int)blockIdx.x : ((int)blockIdx.x & 7) * (groups >> 3) + ((int)blockIdx.x >> 3);
    // first units of all query tiles: a thread sums the ones it has, a scan over the threads says where they begin
    const int each = (a.items + PF2_THREADS - 1) / PF2_THREADS, i0 = min(tid * each, a.items), i1 = min(i0 + each, a.items);
    const int first = i0 < i1 ? units_of(a, i0) : 0;         // all there is up to 512 query tiles
    int own = first;
    for (int i = i0 + 1; i < i1; ++i) own += units_of(a, i);
    int incl = own;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const int o = __shfl_up(incl, d, 64);
        if (lane >= d) incl += o;
    }
    if (lane == 63) sums[tid >> 6] = incl;
    __syncthreads();
    int before = incl - own, total = 0;
#pragma unroll
    for (int x = 0; x < PF2_WAVES; ++x) {
        if (x < (tid >> 6)) before += sums[x];
        total += sums[x];
    }
    const int per = max((total + groups - 1) / groups, PF2_LEAST);
    const int u0 = wg * per, u1 = min(u0 + per, total);
    for (int i = i0, at = before; i < i1; ++i) {
        const int c = i == i0 ? first : units_of(a, i);
        if (wg == 0) a.plan[1 + i] = at;
        if (u0 >= at && u0 < at + c) { found[0] = i; found[1] = u0 - at; }
        at += c;
    }
    if (tid == 0) again = 0;
    if (wg == 0 && tid == 0) a.plan[0] = per;
    if (u0 >= u1) return;                        // the whole workgroup: nothing was left for it
    __syncthreads();
    int i = __builtin_amdgcn_readfirstlane(found[0]), t_first = __builtin_amdgcn_readfirstlane(found[1]);
    for (int u = u0; u < u1; ++i, t_first = 0) {
        const int seg = i / a.query_tiles, count = min(units_of(a, i) - t_first, u1 - u);
        attend_query_tile_once<F16, true>(a, seg, i - seg * a.query_tiles, t_first, count, 2 * wg + (t_first == 0), (PF_LDS3 int*)&again);
        u += count;
    }
}

// The shares of the keys put together: one wavefront per (query tile, 16 of its rows, 64 features), lanes as they wrote.
// A share that a row saw nothing of has sum 0 and a reference of no meaning: it is left out.
// Shares as prefill_shares_kernel cut them, of which the first is in its workgroup's second slot.
template <bool F16>
__global__ __launch_bounds__(256) void prefill_merge_kernel(PrefillArgs a) {
    const int seg = blockIdx.y, tile = (int)blockIdx.x >> 3, w = (int)blockIdx.x & 7, tiles = (int)gridDim.x >> 3;
    const int b = seg / a.kv_heads, h = seg - b * a.kv_heads;
    int n = a.seg_len ? a.seg_len[seg] : a.max_len;
    n = max(0, min(n, a.max_len));
    const int half = threadIdx.x >> 6, lane = threadIdx.x & 63, j = lane & 15, ig = lane >> 4;       // half / 2: of the features, half % 2: of the rows
    const int G = a.group, Q = a.q_len, BT = (PF2_WAVES * 32) / G;
    const int t_last = min(Q - 1, tile * BT + BT - 1);
    const int all_tiles = (max(0, min(n, n - Q + t_last + 1)) + PF2_BN - 1) / PF2_BN;
    const int per = a.plan[0], at = a.plan[1 + seg * tiles + tile], first = at / per, shares = (at + max(all_tiles, 1) - 1) / per - first + 1;
    if (shares <= 1) return;                  // its workgroup wrote the result
    const int r = w * 32 + (half & 1) * 16 + j, g = r % G, t_q = tile * BT + r / G;
    if (r >= BT * G || t_q >= Q) return;
    auto slot = [&](int z) -> int64_t { return 2 * (first + z) + (z == 0); };
    const float2* ml = (const float2*)a.part_ml + r;
    const float4* po = (const float4*)a.part + w * (16 * 64) + ((half & 1) * 8 + (half >> 1) * 4) * 64 + lane;
    float m = -3.0e38f;
    for (int z = 0; z < shares; ++z) {
        const float2 x = ml[slot(z) * (PF2_WAVES * 32)];
        if ((__float_as_uint(x.y) << 1) != 0) m = __builtin_fmaxf(m, x.x);
    }
    float l = 0.0f;
    float4 o[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) o[c] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
#pragma unroll 2
    for (int z = 0; z < shares; ++z) {
        const float2 x = ml[slot(z) * (PF2_WAVES * 32)];
        float4 v[4];
#pragma unroll
        for (int c = 0; c < 4; ++c) v[c] = po[slot(z) * (PF2_WAVES * 16 * 64) + c * 64];
        const float f = (__float_as_uint(x.y) << 1) != 0 ? __builtin_amdgcn_exp2f(x.x - m) : 0.0f;
        l += x.y * f;
#pragma unroll
        for (int c = 0; c < 4; ++c) { o[c].x += v[c].x * f; o[c].y += v[c].y * f; o[c].z += v[c].z * f; o[c].w += v[c].w * f; }
    }
    const float inv = l > 0.0f ? 1.0f / l : 0.0f;
    char* orow = (char*)(a.out + (((int64_t)b * Q + t_q) * (a.kv_heads * G) + (h * G + g)) * a.hd);
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        const int d = (half >> 1) * 64 + 16 * c + 4 * ig;
        if (d < a.hd) *(uint2*)(orow + d * 2) = make_uint2(pack_kv<F16>(o[c].x * inv, o[c].y * inv), pack_kv<F16>(o[c].z * inv, o[c].w * inv));
    }
}

constexpr int PF_PART_ROW = (PF_D + 2) * 4;   // bytes that a row of a workgroup leaves for the merge

// > 64 KB of dynamic LDS needs the attribute once per device (the flag is only ever set, so a race repeats the call at worst)
template <auto KERNEL>
static int opt_in_lds() {
    static bool done[64] = {};
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) dev = -1;
    if (dev < 0 || !done[dev]) {
        hipError_t e = hipFuncSetAttribute((const void*)KERNEL, hipFuncAttributeMaxDynamicSharedMemorySize, PF2_LDS);
        if (e != hipSuccess) return (int)e;
        if (dev >= 0) done[dev] = true;
    }
    return 0;
}

// query tiles of a chunk and rows of each
static void query_tiles(int group, int q_len, int64_t* tiles, int64_t* rows) {
    const int tt = group >= 3 ? 1 : 4 / group;               // SmallCfg
    const int bt = q_len < 64 ? 16 * tt : (PF2_WAVES * 32) / group;
    *tiles = (q_len + bt - 1) / bt;
    *rows = q_len < 64 ? group * tt * 16 : PF2_WAVES * 32;
}

template <bool F16>
static int launch_prefill_split(const PrefillArgs& a, int nseg, hipStream_t st) {
    if (a.q_len < 64) {
        auto go = [&](auto g) {
            using C = SmallCfg<decltype(g)::value>;
            const int tiles = (a.q_len + C::BT - 1) / C::BT, share = a.split_tiles * 64;
            hipLaunchKernelGGL((prefill_small_kernel<decltype(g)::value, F16, true>), dim3(tiles, nseg, (a.max_len + share - 1) / share), dim3(C::THREADS), 0, st, a);
            hipLaunchKernelGGL((prefill_small_merge_kernel<decltype(g)::value, F16>), dim3(tiles * C::WAVES, nseg), dim3(256), 0, st, a);
        };
        switch (a.group) {
            case 1: go(std::integral_constant<int, 1>{}); break;
            case 2: go(std::integral_constant<int, 2>{}); break;
            case 3: go(std::integral_constant<int, 3>{}); break;
            case 4: go(std::integral_constant<int, 4>{}); break;
            case 5: go(std::integral_constant<int, 5>{}); break;
            case 6: go(std::integral_constant<int, 6>{}); break;
            case 7: go(std::integral_constant<int, 7>{}); break;
            default: go(std::integral_constant<int, 8>{}); break;
        }
        return 0;
    }
    if (int rc = opt_in_lds<few::prefill_few_kernel<F16, true>>()) return rc;
    const int bt = (PF2_WAVES * 32) / a.group, tiles = (a.q_len + bt - 1) / bt;
    const int key_tiles = (a.max_len + PF2_BN - 1) / PF2_BN, shares = (key_tiles + a.split_tiles - 1) / a.split_tiles;
    hipLaunchKernelGGL((few::prefill_few_kernel<F16, true>), dim3(tiles, nseg, shares), dim3(PF2_THREADS), PF2_LDS, st, a);
    hipLaunchKernelGGL((few::prefill_few_merge_kernel<F16>), dim3(tiles * PF2_WAVES, nseg), dim3(256), 0, st, a);
    return 0;
}

template <bool F16>
static int launch_prefill_shares(const PrefillArgs& a, int nseg, hipStream_t st) {
    if (int rc = opt_in_lds<prefill_shares_kernel<F16>>()) return rc;
    hipLaunchKernelGGL(prefill_shares_kernel<F16>, dim3(PF2_GROUPS), dim3(PF2_THREADS), PF2_LDS, st, a);
    hipLaunchKernelGGL((prefill_merge_kernel<F16>), dim3(a.query_tiles * PF2_WAVES, nseg), dim3(256), 0, st, a);
    return 0;
}

template <int G, bool F16>
static int launch_prefill(const PrefillArgs& a, int nseg, hipStream_t st) {
    // short chunks: 16 queries per wavefront waste fewer MFMA columns
    if (a.q_len < 64) {
        using C = SmallCfg<G>;
        const int tiles = (a.q_len + C::BT - 1) / C::BT;
        hipLaunchKernelGGL((prefill_small_kernel<G, F16, false>), dim3(tiles, nseg), dim3(C::THREADS), 0, st, a);
        return 0;
    }
    const int bt = (PF2_WAVES * 32) / G, tiles = (a.q_len + bt - 1) / bt;
    // Less work than takes the clock down, in query tiles x keys: all wavefronts in step.  us in step | in two parts, tiles x keys: bf16 64 x 2048 46 | 48, 128 x
    // 4096 83.7 | 85.8, 320 x 600 44 | 46, 192 x 4000 90 | 86, 512 x 4096 178 | 163, 1024 x 1500 144 | 139; fp16 128 x 4096 83 | 94, 256 x 2100 52 | 56, 192 x 4000
    // 94 | 96, 256 x 8192 226 | 218, 1024 x 1500 151 | 151.  Nor do long keys take it down where a third of the compute units has no tile: bf16 128 x 9000 167 |
    // 177, 136 x 5395 107 | 111, 160 x 8000 155 | 159, 168 x 5395 111 | 111, 192 x 6000 128 | 123; fp16 160 x 8000 167 | 180, 168 x 8000 168 | 176, 192 x
    // 8000 180 | 179 (beyond 16000 keys not measured).
    const int64_t items = (int64_t)tiles * nseg;
    if (items * a.max_len < (F16 ? 1200000 : 600000) || (items <= 168 && a.max_len <= 65536)) {
        if (int rc = opt_in_lds<few::prefill_few_kernel<F16, false>>()) return rc;
        hipLaunchKernelGGL((few::prefill_few_kernel<F16, false>), dim3(tiles, nseg), dim3(PF2_THREADS), PF2_LDS, st, a);
        return 0;
    }
    if (int rc = opt_in_lds<prefill_attn_kernel<F16>>()) return rc;
    hipLaunchKernelGGL((prefill_attn_kernel<F16>), dim3(tiles, nseg), dim3(PF2_THREADS), PF2_LDS, st, a);
    return 0;
}

}  // namespace trimkv

using namespace trimkv;

// Checks what both entry points take, and fills the arguments.
static int prefill_args(const char* fn, PrefillArgs& a, const void* q, int64_t q_stride_b, int64_t q_stride_h, int64_t q_stride_t, void* out,
                                   const void* k_slab, const void* v_slab, const int32_t* seg_len, const int32_t* seg_start,
                                   int batch, int kv_heads, int group, int q_len, int cap, int head_dim, int dtype, float scale,
                                   int max_len) {
    if (!q || !out || !k_slab || !v_slab) return fail(TRIMKV_ERR_NULL, "%s: null pointer argument", fn);
    if (dtype != TRIMKV_BF16 && dtype != TRIMKV_F16) return fail(TRIMKV_ERR_DTYPE, "%s: K/V/q must be bf16 or fp16 (dtype=%d)", fn, dtype);
    if (head_dim != 128 && head_dim != 96 && head_dim != 64) return fail(TRIMKV_ERR_UNSUPPORTED, "%s: head_dim must be 64, 96 or 128 (got %d)", fn, head_dim);
    if (group < 1 || group > 8) return fail(TRIMKV_ERR_UNSUPPORTED, "%s: group must be in [1, 8] (got %d)", fn, group);
    if (batch <= 0 || kv_heads <= 0 || q_len <= 0 || cap <= 0 || max_len <= 0)
        return fail(TRIMKV_ERR_SHAPE, "%s: bad sizes batch=%d kv_heads=%d q_len=%d cap=%d max_len=%d", fn, batch, kv_heads, q_len, cap, max_len);
    const int64_t nseg = (int64_t)batch * kv_heads;
    if (nseg > 65535) return fail(TRIMKV_ERR_SHAPE, "%s: batch*kv_heads=%lld exceeds the grid limit 65535", fn, (long long)nseg);
    if (!seg_start && max_len > cap) return fail(TRIMKV_ERR_CAPACITY, "%s: max_len %d exceeds capacity %d", fn, max_len, cap);
    if (((uintptr_t)q | (uintptr_t)out | (uintptr_t)k_slab | (uintptr_t)v_slab) & 15 || ((q_stride_b | q_stride_h | q_stride_t) & 7))
        return fail(TRIMKV_ERR_SHAPE, "%s: q/out/K/V must be 16-byte aligned and q strides multiples of 8 elements", fn);
    a.q = (const uint16_t*)q; a.q_sb = q_stride_b; a.q_sh = q_stride_h; a.q_st = q_stride_t; a.out = (uint16_t*)out;
    a.k = (const char*)k_slab; a.v = (const char*)v_slab; a.seg_len = seg_len; a.seg_start = seg_start;
    a.kv_heads = kv_heads; a.group = group; a.q_len = q_len; a.cap = cap; a.max_len = max_len; a.hd = head_dim; a.scale_log2 = scale * 1.4426950408889634f;
    a.split_tiles = 0; a.part = nullptr; a.part_ml = nullptr; a.plan = nullptr; a.query_tiles = 0; a.items = 0;
    return 0;
}

extern "C" int trimkv_prefill_attn(const void* q, int64_t q_stride_b, int64_t q_stride_h, int64_t q_stride_t, void* out,
                                   const void* k_slab, const void* v_slab, const int32_t* seg_len, const int32_t* seg_start,
                                   int batch, int kv_heads, int group, int q_len, int cap, int head_dim, int dtype, float scale,
                                   int max_len, void* stream) {
    const char* fn = "trimkv_prefill_attn";
    PrefillArgs a;
    if (int bad = prefill_args(fn, a, q, q_stride_b, q_stride_h, q_stride_t, out, k_slab, v_slab, seg_len, seg_start, batch, kv_heads,
                               group, q_len, cap, head_dim, dtype, scale, max_len)) return bad;
    const int nseg = batch * kv_heads;
    hipStream_t st = (hipStream_t)stream;
    const bool f16 = dtype == TRIMKV_F16;
    int rc = 0;
    switch (group) {
        case 1: rc = f16 ? launch_prefill<1, true>(a, nseg, st) : launch_prefill<1, false>(a, nseg, st); break;
        case 2: rc = f16 ? launch_prefill<2, true>(a, nseg, st) : launch_prefill<2, false>(a, nseg, st); break;
        case 3: rc = f16 ? launch_prefill<3, true>(a, nseg, st) : launch_prefill<3, false>(a, nseg, st); break;
        case 4: rc = f16 ? launch_prefill<4, true>(a, nseg, st) : launch_prefill<4, false>(a, nseg, st); break;
        case 5: rc = f16 ? launch_prefill<5, true>(a, nseg, st) : launch_prefill<5, false>(a, nseg, st); break;
        case 6: rc = f16 ? launch_prefill<6, true>(a, nseg, st) : launch_prefill<6, false>(a, nseg, st); break;
        case 7: rc = f16 ? launch_prefill<7, true>(a, nseg, st) : launch_prefill<7, false>(a, nseg, st); break;
        default: rc = f16 ? launch_prefill<8, true>(a, nseg, st) : launch_prefill<8, false>(a, nseg, st); break;
    }
    if (rc) return fail(rc, "%s: hipFuncSetAttribute failed (%d)", fn, rc);
    return launch_status(fn);
}

// ---- keys of a query tile split over several workgroups ----
// A query tile (256 / group times of one segment) is one workgroup, and a CU holds one: a chunk of few segments leaves CUs idle
// for as long as its longest segment takes (1.15 us per 64 keys).  Up to 128 query tiles the keys go to S workgroups of a query
// tile, all of them on the chip at once (tiles * S <= 256).  What S costs was fitted to tiles 8 .. 128, 512 .. 65536 keys: 3 us
// for the merge's launch, 0.8 us per share that a row's merge walks, 0.045 us per workgroup for its 130 KB written and read.
// Measured (us, D 128, whole -> split): 8 tiles of 2048 keys 44 -> 21, of 8192 keys 150 -> 31; 32 of 4096 79 -> 35; 56 of 2954
// 64 -> 37; 96 of 4096 80 -> 57; 128 of 8192 155 -> 107; left whole: 96 of 2048 44 -> 40, of 1024 27 -> 30, 40 of 1024 27 -> 25.
// Between 128 and 256 tiles: for callers that do not take equal shares (below), which are faster there.  Of unlike segments the longest
// one holds up the rest, and three shares let the others' CUs help: 160 and 168 tiles, mean length / longest 0.60 of 4100 keys 83 -> 79,
// 0.68 of 8192 151 -> 136; 192 tiles, 0.53 of 8192 153 -> 131; 224, 0.52 of 10000 194 -> 166, but 0.57 of 8192 166 -> 177.
extern "C" int trimkv_prefill_split_tiles(int batch, int kv_heads, int group, int q_len, int max_len, int uneven) {
    if (batch <= 0 || kv_heads <= 0 || group < 1 || group > 8 || q_len <= 0 || max_len <= 0) return 0;
    int64_t tiles, rows;
    query_tiles(group, q_len, &tiles, &rows);
    const int64_t items = tiles * batch * kv_heads;
    const int64_t key_tiles = ((int64_t)max_len + PF2_BN - 1) / PF2_BN;
    if (q_len < 64) {
        // Short chunks: a workgroup walks 64 keys in 2.2 us, two or more fit on a CU.  Whole -> split, us: 8 query tiles of 2048 keys
        // 72 -> 19, of 8192 278 -> 32; 32 of 2048 72 -> 20, of 8192 281 -> 40; 128 of 2048 73 -> 34, of 8192 281 -> 104; left whole:
        // 512 keys (20 -> 13 for a second launch), 512 query tiles (2048 keys 99 -> 109).
        float best = 2.2f * (float)key_tiles - 8.0f;
        int64_t take = 0;
        for (int64_t s = 2; s <= 32 && items * s <= 512; ++s) {
            const int64_t each = (key_tiles + s - 1) / s;
            const float us = 2.2f * (float)each + 3.0f + (0.8f + 0.02f * (float)items) * (float)s;
            if (us < best) { best = us; take = each; }
        }
        return (int)take;
    }
    if (items >= 256) return 0;
    if (items > 128) {
        const bool pays = uneven > 0 && key_tiles >= 64 && (items <= 170 ? uneven <= 75 : uneven <= 55 && items <= 224 && key_tiles <= 160);
        return pays ? (int)((key_tiles + 2) / 3) : 0;
    }
    float best = 1.15f * (float)key_tiles - 8.0f;   // below that the second launch costs a caller whose queue runs dry as much
    int64_t take = 0;
    for (int64_t s = 2; s <= 32 && items * s <= 256; ++s) {
        const int64_t each = (key_tiles + s - 1) / s;
        const float us = 1.15f * (float)each + 3.0f + (0.8f + 0.045f * (float)items) * (float)s;
        if (us < best) { best = us; take = each; }
    }
    return (int)take;
}

extern "C" int64_t trimkv_prefill_split_workspace(int batch, int kv_heads, int group, int q_len, int max_len, int split_tiles) {
    if (batch <= 0 || kv_heads <= 0 || group < 1 || group > 8 || q_len <= 0 || max_len <= 0 || split_tiles <= 0) return 0;
    int64_t tiles, rows;
    query_tiles(group, q_len, &tiles, &rows);
    const int64_t key_tiles = ((int64_t)max_len + PF2_BN - 1) / PF2_BN, shares = (key_tiles + split_tiles - 1) / split_tiles;
    return tiles * batch * kv_heads * shares * rows * PF_PART_ROW;
}

extern "C" int trimkv_prefill_attn_split(const void* q, int64_t q_stride_b, int64_t q_stride_h, int64_t q_stride_t, void* out,
                                         const void* k_slab, const void* v_slab, const int32_t* seg_len, const int32_t* seg_start,
                                         int batch, int kv_heads, int group, int q_len, int cap, int head_dim, int dtype, float scale,
                                         int max_len, int split_tiles, void* workspace, int64_t workspace_bytes, void* stream) {
    const char* fn = "trimkv_prefill_attn_split";
    PrefillArgs a;
    if (int bad = prefill_args(fn, a, q, q_stride_b, q_stride_h, q_stride_t, out, k_slab, v_slab, seg_len, seg_start, batch, kv_heads,
                               group, q_len, cap, head_dim, dtype, scale, max_len)) return bad;
    if (split_tiles <= 0) return fail(TRIMKV_ERR_SHAPE, "%s: split_tiles must be positive (got %d)", fn, split_tiles);
    const int64_t need = trimkv_prefill_split_workspace(batch, kv_heads, group, q_len, max_len, split_tiles);
    const int64_t shares = (((int64_t)max_len + PF2_BN - 1) / PF2_BN + split_tiles - 1) / split_tiles;
    if (shares > 65535) return fail(TRIMKV_ERR_SHAPE, "%s: %lld shares of the keys exceed the grid limit 65535", fn, (long long)shares);
    if (!workspace || workspace_bytes < need || (uintptr_t)workspace & 15)
        return fail(TRIMKV_ERR_CAPACITY, "%s: needs a 16-byte aligned workspace of %lld bytes (got %lld)", fn, (long long)need, (long long)workspace_bytes);
    a.split_tiles = split_tiles;
    a.part = (float*)workspace;
    a.part_ml = (float*)workspace + need / PF_PART_ROW * PF_D;
    hipStream_t st = (hipStream_t)stream;
    const int rc = dtype == TRIMKV_F16 ? launch_prefill_split<true>(a, batch * kv_heads, st) : launch_prefill_split<false>(a, batch * kv_heads, st);
    if (rc) return fail(rc, "%s: hipFuncSetAttribute failed (%d)", fn, rc);
    return launch_status(fn);
}

// ---- equal shares of all keys of a launch ----
// More than 128 query tiles.  Whole, the chip is done when its longest query tile is, or a last round that fills part of it: 1.2 us per
// 64 keys where a CU has little company, 1.6 where all are busy.  Equal shares take the mean of all CUs and pay for it with up to
// 67 MB of unfinished outputs written and read, about 26 us.  Estimates fitted to 80 launches (136 .. 1104 query tiles of 2500,
// 5000 and 9000 keys, mean length 52 .. 100 % of the longest) and compared with 340 more (168 .. 8192 query tiles of 8 .. 128 segments, 3100 .. 40000 keys,
// mean length 55 .. 100 %, chunks of 300 .. 8192): where they differ by 3 % the choice is the faster one, but from 512 query tiles of 32 segments on, where
// lengths average out and the workgroups of an XCD no longer walk the same keys at about the same time, shares lost by up to 15 % (1312
// tiles, 32 segments of 40000 keys 5761 -> 6228 us, 1056 tiles, 96 of 7000 814 -> 854).  11 % and more with the rows held there leave nothing that is
// slower by 3 %, and give up 2 .. 12 % at 13 of the 340 (most: 512 tiles, 64 segments of 0.55 x 11000 keys, 427 -> 382).  Beyond 8192 tiles or 40960 keys nothing
// was measured.  Whole -> shares, us: 168 tiles, 0.78 of 4100 keys 88 -> 83, 0.65 of 9000 170 -> 122; 264 tiles of 9000 377 -> 269, of 5000 167 -> 149;
// 288, 0.52 of 9000 289 -> 185; 352 of 5000 220 -> 204; 1296 of 12000 1407 -> 1369, of 32000 4263 -> 4051; 2576, 0.7 of 16000 2722 -> 2221; left
// whole: 216 of 2500 59 -> 67, 512 of 5000 174 -> 204, 704 of 9000 478 -> 495, 2048 of 8704 1381 -> 1485, 8192 of 16000 11355 -> 13595.
extern "C" int trimkv_prefill_equal_shares(int batch, int kv_heads, int group, int q_len, int max_len, int uneven) {
    if (batch <= 0 || kv_heads <= 0 || group < 1 || group > 8 || q_len < 64 || max_len <= 0) return 0;
    int64_t tiles, rows;
    query_tiles(group, q_len, &tiles, &rows);
    const int64_t items = tiles * batch * kv_heads;
    if (items <= 128 || items > 8192 || max_len > 40960 || (uneven && max_len < 3072)) return 0;
    // in tiles of 64 keys: the longest segment, the mean query tile, the first one of a mean segment
    const float even = uneven <= 0 ? 1.0f : uneven == 1 ? 0.6f : 0.01f * (float)uneven, all = (float)items / 256.0f;
    const float longest = (float)max_len / 64.0f, keys = (float)max_len * even, bt = 256.0f / (float)group;
    const float mean = std::max(1.0f, (keys - 0.5f * (float)q_len) / 64.0f + 0.5f + bt / 128.0f), least = std::max(1.0f, (keys - (float)q_len) / 64.0f);
    const float shares = 26.0f + 25.0f * (1.0f - even) + 0.03f * (float)items + 1.6f * mean * all;
    float whole;
    if (items <= 256) whole = std::max(1.6f * mean * all + 20.0f, 1.2f * longest + 12.0f);
    else {
        const float rounds = (float)(items / 256), rest = (float)(items % 256), last = least + (mean - least) * rest / (float)items;
        whole = rounds * (1.6f * mean + 8.0f) + (rest > 0.0f ? (0.96f + 0.34f * rest / 256.0f) * last + 8.0f : 0.0f) + 0.9f * (1.0f - even) * longest;
    }
    const int64_t segs = (int64_t)batch * kv_heads;
    const float margin = segs >= 32 && items >= 512 ? 1.11f + 0.02f * (float)(segs * max_len) / 524288.0f : 1.03f;
    return keys >= (float)q_len && whole > margin * shares;      // a segment holds at least the chunk
}

extern "C" int64_t trimkv_prefill_shares_workspace(int batch, int kv_heads, int group, int q_len) {
    if (batch <= 0 || kv_heads <= 0 || group < 1 || group > 8 || q_len < 64) return 0;
    int64_t tiles, rows;
    query_tiles(group, q_len, &tiles, &rows);
    return (int64_t)2 * PF2_GROUPS * rows * PF_PART_ROW + (tiles * batch * kv_heads + 1) * 4;
}

extern "C" int trimkv_prefill_attn_shares(const void* q, int64_t q_stride_b, int64_t q_stride_h, int64_t q_stride_t, void* out,
                                          const void* k_slab, const void* v_slab, const int32_t* seg_len, const int32_t* seg_start,
                                          int batch, int kv_heads, int group, int q_len, int cap, int head_dim, int dtype, float scale,
                                          int max_len, void* workspace, int64_t workspace_bytes, void* stream) {
    const char* fn = "trimkv_prefill_attn_shares";
    PrefillArgs a;
    if (int bad = prefill_args(fn, a, q, q_stride_b, q_stride_h, q_stride_t, out, k_slab, v_slab, seg_len, seg_start, batch, kv_heads,
                               group, q_len, cap, head_dim, dtype, scale, max_len)) return bad;
    if (q_len < 64) return fail(TRIMKV_ERR_SHAPE, "%s: chunks of 64 queries and more (got %d)", fn, q_len);
    int64_t tiles, rows;
    query_tiles(group, q_len, &tiles, &rows);
    const int64_t items = tiles * batch * kv_heads, key_tiles = ((int64_t)max_len + PF2_BN - 1) / PF2_BN;
    if (items > (1 << 24) || items * key_tiles > (1 << 30)) return fail(TRIMKV_ERR_SHAPE, "%s: %lld query tiles of %d keys are too many", fn, (long long)items, max_len);
    const int64_t need = trimkv_prefill_shares_workspace(batch, kv_heads, group, q_len);
    if (!workspace || workspace_bytes < need || (uintptr_t)workspace & 15)
        return fail(TRIMKV_ERR_CAPACITY, "%s: needs a 16-byte aligned workspace of %lld bytes (got %lld)", fn, (long long)need, (long long)workspace_bytes);
    a.part = (float*)workspace;
    a.part_ml = a.part + (int64_t)2 * PF2_GROUPS * rows * PF_D;
    a.plan = (int*)(a.part_ml + (int64_t)2 * PF2_GROUPS * rows * 2);
    a.query_tiles = (int)tiles; a.items = (int)items;
    hipStream_t st = (hipStream_t)stream;
    const int rc = dtype == TRIMKV_F16 ? launch_prefill_shares<true>(a, batch * kv_heads, st) : launch_prefill_shares<false>(a, batch * kv_heads, st);
    if (rc) return fail(rc, "%s: hipFuncSetAttribute failed (%d)", fn, rc);
    return launch_status(fn);
}

// Chunk attention where the chip is not full: little work, or keys in shares by sizes -- gfx950.  Included by attn_prefill.hip, whose
// arguments, tiles in LDS and checks these are.
//
// MFMA 32x32x16 register layout (lane l, half hl = l / 32):
//   A (32 x 16): row l % 32, k = 8 * hl + 0..7          B (16 x 32): column l % 32, k = 8 * hl + 0..7
//   C (32 x 32): column l % 32, register v holds row 8 * (v / 4) + 4 * hl + v % 4
// S^T = K . Q^T per 32-key block: after it a lane holds, for its query, keys 8c + 4hl + i (c, i in 0..3).
// The second product consumes 16 keys per MFMA; step st takes from lane half hl the keys of c = 2st and
// 2st + 1, i.e. registers v = 8st .. 8st + 7 in order: keys 16 st + 4 hl + 0..3 and 16 st + 8 + 4 hl + 0..3.
//
// All wavefronts are in step here, with exponentials between the products and one barrier per 64 keys.  Where matrix load takes the clock down the
// kernel of two parts is faster (attn_prefill.hip), but its wavefronts wait for one another twice per 32 keys: where the chip is
// not full, the clock is high and the time is the chain of one workgroup, and that costs 1 to 3 us a launch (fp16, which keeps row maxima, up to a
// fifth).  us here | in two parts, bf16: 64 query tiles of 2048 keys 42.9 | 46.4, 96 rows of 300 keys 12.8 | 14.6, 16 tiles of 4096 keys in shares 34.4 |
// 36.1, 8 of 512 17.6 | 19.5; the rule for whole tiles is at its launch.
#pragma once

namespace trimkv {
namespace few {

template <bool F16>
__device__ __forceinline__ pf_f32x16 mfma_32x32x16(pf_bf16x8 a, pf_bf16x8 b, pf_f32x16 c) {
    if constexpr (F16) return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(pf_f16x8, a), __builtin_bit_cast(pf_f16x8, b), c, 0, 0, 0);
    else return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}
constexpr int PF2_PD = 3;                           // LDS operand reads in flight ahead of the MFMA that consumes them

// One query tile against `count` tiles of keys from tile t_first on (PART; else against all of them).  Where that is not all that the
// query tile sees, unnormalised outputs with their exponent references and row sums (fp32) are left in `slot` for the merge kernel.
// V in LDS: the 32-byte pair p of row r sits at pair position p ^ (2 (r & 3)).
template <bool F16, bool PART>
__device__ __forceinline__ void attend_query_tile(const PrefillArgs& a, int seg, int tile, int t_first, int count, int64_t slot) {
    extern __shared__ __attribute__((aligned(16))) char pf2_lds[];
    PF_LDS3 char* const lds3 = (PF_LDS3 char*)pf2_lds;
    const uint32_t lds0 = (uint32_t)(uintptr_t)lds3;
    const int b = seg / a.kv_heads, h = seg - b * a.kv_heads;
    int n = a.seg_len ? a.seg_len[seg] : a.max_len;
    n = max(0, min(n, a.max_len));
    int tid = threadIdx.x;
    const int lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);   // wave-uniform by construction; saying so keeps what derives from it in scalar registers
    const int j = lane & 31, hl = lane >> 5;    // MFMA column (query) and lane half
    const int G = a.group, Q = a.q_len;
    const int BT = (PF2_WAVES * 32) / G;        // query times per workgroup; rows BT * G .. 255 are padding
    const int t_wg0 = tile * BT;
    const int r = w * 32 + j;
    const int g = r % G;
    const int t_q = t_wg0 + r / G;              // this lane's query time
    const int t_w_first = t_wg0 + (w * 32) / G;
    const int64_t row0 = a.seg_start ? (int64_t)a.seg_start[seg] : (int64_t)seg * a.cap;

    // The rows of Q are asked for in front of the first keys and turned into fragments behind them: one memory round trip for both.
    pf_u32x4 qraw[8];
    {
        const uint16_t* qrow = a.q + (int64_t)b * a.q_sb + (int64_t)(h * G + g) * a.q_sh + (int64_t)min(t_q, Q - 1) * a.q_st;
#pragma unroll
        for (int ks = 0; ks < 8; ++ks) qraw[ks] = *(const pf_u32x4*)(qrow + min(ks * 16 + hl * 8, a.hd - 8));
    }

    pf_f32x16 o[4];   // O^T: o[db][v] = d (db * 32 + 8 * (v / 4) + 4 * hl + v % 4) of query j
#pragma unroll
    for (int db = 0; db < 4; ++db)
#pragma unroll
        for (int v = 0; v < 16; ++v) o[db][v] = 0.0f;
    // Exponent reference (log2 units) and this lane's share of the row sum.  The score MFMAs start from -m_ref in their
    // accumulator (negm, all 16 registers alike: a lane is one query), so what they deliver is already s - m_ref.  The
    // reference starts at 0 and is moved onto the row maximum by the first block.  A query that sees no key at all
    // (segment shorter than the chunk) keeps reference 0: its masked scores give exp2(-huge) = 0, never exp2(0).
    float m_ref = 0.0f, l_run = 0.0f;
    pf_f32x16 negm;
#pragma unroll
    for (int v = 0; v < 16; ++v) negm[v] = 0.0f;

    const int t_last = min(Q - 1, t_wg0 + BT - 1);
    const int k_end = max(0, min(n, n - Q + t_last + 1));     // keys the query tile sees
    const int all_tiles = (k_end + PF2_BN - 1) / PF2_BN;
    const int vis_j = n - Q + t_q;                            // last key this lane's query sees
    const int vis_lo = n - Q + t_w_first;                     // ... the wavefront's first query
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
    const uint32_t st_vcol = min((uint32_t)((((st_pos >> 1) ^ (2 * (st_row & 3))) << 1) | (st_pos & 1)) * 16u, row_bytes - 16u);
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
    // Q fragments (B operand of S^T): 8 d of step ks at d = ks * 16 + hl * 8, multiplied by scale * log2(e) and rounded back
    // to 16 bits once, here: the score MFMAs then deliver exponents of two directly and the loop never multiplies a score.
    pf_bf16x8 qf[8];
#pragma unroll
    for (int ks = 0; ks < 8; ++ks) {
        pf_u32x4 sc;
#pragma unroll
        for (int x = 0; x < 4; ++x) {
            float lo, hi;
            if (F16) { lo = f16_bits_to_f32((uint16_t)(qraw[ks][x] & 0xffffu)); hi = f16_bits_to_f32((uint16_t)(qraw[ks][x] >> 16)); }
            else { lo = __uint_as_float(qraw[ks][x] << 16); hi = __uint_as_float(qraw[ks][x] & 0xffff0000u); }
            sc[x] = pack_kv<F16>(lo * a.scale_log2, hi * a.scale_log2);
        }
        if (ks * 16 + hl * 8 >= a.hd) sc = pf_u32x4{0u, 0u, 0u, 0u};   // padded features: whatever K holds there counts for nothing
        qf[ks] = __builtin_bit_cast(pf_bf16x8, sc);
    }

    // per-lane LDS read offsets; the buffer, the 32-key block and the step are immediates on top of them
    PF_LDS3 char* k_ptr[8];
    PF_LDS3 char* v_ptr[4];
#pragma unroll
    for (int ks = 0; ks < 8; ++ks) {
        k_ptr[ks] = lds3 + (j * 256 + (((2 * ks + hl) ^ (j & 15)) << 4));
        asm volatile("" : "+v"(k_ptr[ks]));          // a value in a register from here on, not an expression to recompute in the loop
    }
    {
        const int i = lane & 15, jhalf = (lane >> 4) & 1;
        const int kx = 4 * hl + (i >> 2);            // key (within its group of 8) this lane supplies to the transposing read
#pragma unroll
        for (int db = 0; db < 4; ++db) {
            v_ptr[db] = lds3 + (PF2_VBASE + kx * 256 + (((2 * db + jhalf) ^ (2 * (kx & 3))) << 5) + (i & 3) * 8);
            asm volatile("" : "+v"(v_ptr[db]));
        }
    }
    auto k_frag = [&](int imm, int ks) __attribute__((always_inline)) {
        return *(const PF_LDS3 pf_bf16x8*)(k_ptr[ks] + imm);
    };
    auto v_frag = [&](int imm, int st, int db) __attribute__((always_inline)) {
        PF_LDS3 char* p = v_ptr[db] + imm + st * 16 * 256;
        const pf_s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((PF_LDS3 pf_s16x4*)p);                // keys 16 st + 4 hl + 0..3
        const pf_s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((PF_LDS3 pf_s16x4*)(p + 8 * 256));    // ... + 8
        return __builtin_bit_cast(pf_bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
    };

    // Mask (diagonal blocks only), row maximum, and the lazy move of the exponent reference: O and l are
    // rescaled only when some row of the wavefront outgrows its reference by 2^PF2_LAZY.  FIRST: the wavefront's first
    // block puts the reference on the row maximum wherever it lies (O and l are still zero: nothing to rescale).
    // tmax: the maximum of s before masking, as the step computed it under its P.V MFMAs (ignored by FIRST).
    auto max16 = [&](const pf_f32x16& s) __attribute__((always_inline)) {
        float t = s[0];
#pragma unroll
        for (int v = 1; v < 16; ++v) t = __builtin_fmaxf(t, s[v]);
        return t;
    };
    auto prepare = [&](pf_f32x16& s, int blk, float tmax, auto first_c) __attribute__((always_inline)) {
        constexpr bool FIRST = decltype(first_c)::value;
        if (FIRST) tmax = max16(s);
        const int key0 = (blk + 2 * t_first) * 32;
        if (key0 + 31 > vis_lo) {   // wave-uniform: some query of the wavefront does not see the whole block
            // (the empty volatile statement keeps this a branch: as 48 speculated selects it would run for every block)
            asm volatile("" ::: );
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                const int key = key0 + 8 * (v >> 2) + 4 * hl + (v & 3);
                s[v] = key <= vis_j ? s[v] : PF_NEG;
            }
            tmax = max16(s);
        }
        if (FIRST || __builtin_amdgcn_ballot_w64(tmax > PF2_LAZY) != 0) {
            const float t2 = __builtin_fmaxf(tmax, __shfl_xor(tmax, 32, 64));   // both halves of a query agree on the reference
            // how far the reference moves: onto the maximum (first block; not at all for a row that sees nothing), else up only
            const float d = FIRST ? (t2 > 0.5f * PF_NEG ? t2 : 0.0f) : __builtin_fmaxf(t2, 0.0f);
            m_ref += d;
#pragma unroll
            for (int v = 0; v < 16; ++v) { s[v] -= d; negm[v] = -m_ref; }
            if (!FIRST) {
                const float alpha = __builtin_amdgcn_exp2f(-d);
                l_run *= alpha;
#pragma unroll
                for (int db = 0; db < 4; ++db)
#pragma unroll
                    for (int v = 0; v < 16; ++v) o[db][v] *= alpha;
            }
        }
    };
    // P = exp2(s - ref) as bf16 (two scores -> one dword) and the row sum of the rounded P
    auto p_pair = [&](const pf_f32x16& s, int x) __attribute__((always_inline)) {
        const float p0 = __builtin_amdgcn_exp2f(s[2 * x]);
        const float p1 = __builtin_amdgcn_exp2f(s[2 * x + 1]);
        const uint32_t pw = pack_kv<F16>(p0, p1);
        l_run = add_pair<F16>(pw, l_run);
        return pw;
    };
    // One pipeline step, in issue order (the fences keep the compiler from regrouping it): the 8 MFMAs of the next
    // block's scores, each followed by one eighth of this block's exponentials; then the 8 MFMAs of P.V, with the maximum
    // of the next block's scores computed in their shadow.  s_cur and s_nxt are two register blocks that swap roles from
    // step to step (no copy).  The 16 MFMA operands of a step (8 K fragments, then 8 V fragments) belong to one stream of
    // LDS reads that runs across steps: each is requested PD MFMAs before the one that consumes it, so the first PD K
    // fragments of a step were requested by the step before it (pre[], in and out).
    //   kimm, vimm: byte offsets of this step's K block and V block; nkimm: of the next step's K block
    //   HAS_NEXT = false: last block of the wavefront, no scores to compute.  FEEDS_NEXT = false: no step follows that wants K.
    //   SYNC: the iteration's barrier, between the two groups of MFMAs (the score MFMAs drain while the wavefront waits).
    // Returns the row maximum of s_nxt (this lane's 16 scores).
    auto step = [&](const pf_f32x16& s_cur, pf_f32x16& s_nxt, pf_bf16x8 (&pre)[PF2_PD], auto kimm_c, auto vimm_c, auto nkimm_c, auto has_next,
                    auto feeds_next, auto sync_c) __attribute__((always_inline)) -> float {
        constexpr bool HAS_NEXT = decltype(has_next)::value, FEEDS_NEXT = decltype(feeds_next)::value, SYNC = decltype(sync_c)::value;
        const int KIMM = kimm_c, VIMM = vimm_c, NKIMM = nkimm_c;   // integral constants in the main loop (instruction immediates), plain ints in the tail
        constexpr int PD = PF2_PD;
        pf_bf16x8 frag[16 + PD];
        uint32_t pw[8];
        auto request = [&](int m) __attribute__((always_inline)) {
            if (m < 8) {
                if (HAS_NEXT) frag[m] = k_frag(KIMM, m);
            } else if (m < 16) {
                frag[m] = v_frag(VIMM, (m - 8) >> 2, (m - 8) & 3);
            } else if (FEEDS_NEXT) {
                frag[m] = k_frag(NKIMM, m - 16);
            }
        };
#pragma unroll
        for (int m = 0; m < PD; ++m) frag[m] = pre[m];
#pragma unroll
        for (int ks = 0; ks < 8; ++ks) {
            request(ks + PD);
            pw[ks] = p_pair(s_cur, ks);
            if (HAS_NEXT) s_nxt = mfma_32x32x16<F16>(frag[ks], qf[ks], ks == 0 ? negm : s_nxt);
            __builtin_amdgcn_sched_barrier(0);
        }
        if (SYNC) {   // behind the barrier the next tile is visible: every thread has waited for its own four loads of it
            asm volatile("s_waitcnt vmcnt(4)" ::: "memory");   // (the four of the tile after it may still be in flight)
            __syncthreads();
            __builtin_amdgcn_sched_barrier(0);
        }
        pf_bf16x8 pfrag[2];
#pragma unroll
        for (int st = 0; st < 2; ++st) {
            const pf_u32x4 pq = {pw[4 * st], pw[4 * st + 1], pw[4 * st + 2], pw[4 * st + 3]};
            pfrag[st] = __builtin_bit_cast(pf_bf16x8, pq);
        }
        // the maximum of the next block's scores as a tree of three-input maxima, one or two per P.V MFMA from the third
        // on (the last score MFMA has landed by then); the empty volatile statements fix where each is computed: between
        // these two MFMAs, not after the last one
        float mt[7];
        auto max3 = [](float x, float y, float z) __attribute__((always_inline)) { return __builtin_fmaxf(__builtin_fmaxf(x, y), z); };
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            request(8 + i + PD);
            o[i & 3] = mfma_32x32x16<F16>(frag[8 + i], pfrag[i >> 2], o[i & 3]);
            if (HAS_NEXT) {
                if (i >= 2 && i <= 6) { mt[i - 2] = max3(s_nxt[3 * (i - 2)], s_nxt[3 * (i - 2) + 1], s_nxt[3 * (i - 2) + 2]); asm volatile("" : "+v"(mt[i - 2])); }
                if (i == 6) { mt[5] = max3(mt[0], mt[1], s_nxt[15]); asm volatile("" : "+v"(mt[5])); }
                if (i == 7) { mt[6] = max3(mt[2], mt[3], mt[4]); asm volatile("" : "+v"(mt[6])); }
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        if (FEEDS_NEXT) {
#pragma unroll
            for (int m = 0; m < PD; ++m) pre[m] = frag[16 + m];
        }
        float mx = HAS_NEXT ? __builtin_fmaxf(mt[5], mt[6]) : 0.0f;
        // both values are wanted here, at the end of the step: without this the compiler moves the maxima and the row-sum
        // additions behind the branch that follows, out of the shadow of the MFMAs
        asm volatile("" : "+v"(mx), "+v"(l_run));
        return mx;
    };

    // Pipeline over 32-key blocks: while the exponentials of block b run on the VALU, the MFMA unit computes the scores
    // of block b + 1 and then P.V of block b.  Every wavefront walks all blocks of the workgroup's tiles: the blocks that
    // lie wholly above a wavefront's diagonal (at most two of up to several hundred, the workgroup spans BT query times)
    // are masked like the diagonal ones and contribute zeros, which keeps the loop free of per-wavefront branches.
    if (ntiles > 0) {
        pf_f32x16 s_a, s_b;   // scores of the current and of the next block, roles swapping every step
        pf_bf16x8 pre[PF2_PD];
        asm volatile("s_waitcnt vmcnt(4)" ::: "memory");
        __syncthreads();
        {
            s_a = negm;
#pragma unroll
            for (int ks = 0; ks < 8; ++ks) s_a = mfma_32x32x16<F16>(k_frag(0, ks), qf[ks], s_a);
#pragma unroll
            for (int m = 0; m < PF2_PD; ++m) pre[m] = k_frag(PF2_TILE / 2, m);
        }
        prepare(s_a, 0, 0.0f, std::true_type{});
        // Iteration t (tile t in the buffer at off0, tile t + 1 at off1): blocks 2t and 2t + 1, and the scores of block 2t + 2.
        // Tile t + 2 is requested first, into the buffer tile t - 2 used (every wavefront left it before the barrier of
        // iteration t - 1).  The one barrier of an iteration sits inside its first step, between the score MFMAs and the
        // P.V MFMAs: behind it tile t + 1 is visible, in time for the K fragments that the end of that step requests.
        auto iteration = [&](int t, int b2, auto off0, auto off1) __attribute__((always_inline)) {
            constexpr std::integral_constant<int, PF2_TILE / 2> half{};
            request_tile(t + 2, b2);          // unconditional (rows clamped): the count of loads in flight stays fixed
            const float ma = step(s_a, s_b, pre, off0 + half, off0, off1, std::true_type{}, std::true_type{}, std::true_type{});
            prepare(s_b, 2 * t + 1, ma, std::false_type{});
            const float mb = step(s_b, s_a, pre, off1, off0 + half, off1 + half, std::true_type{}, std::true_type{}, std::false_type{});
            prepare(s_a, 2 * t + 2, mb, std::false_type{});
        };
        using I0 = std::integral_constant<int, 0>; using I1 = std::integral_constant<int, PF2_TILE>;
        using I2 = std::integral_constant<int, 2 * PF2_TILE>; using I3 = std::integral_constant<int, 3 * PF2_TILE>;
        int t = 0;
        for (; t + 4 < ntiles; t += 4) {      // four tiles per turn: buffer offsets are immediates of the LDS reads
            iteration(t, 2, I0{}, I1{});
            iteration(t + 1, 3, I1{}, I2{});
            iteration(t + 2, 0, I2{}, I3{});
            iteration(t + 3, 1, I3{}, I0{});
        }
        for (; t + 1 < ntiles; ++t)           // up to three more, offsets computed
            iteration(t, (t + 2) & 3, (t & 3) * PF2_TILE, ((t + 1) & 3) * PF2_TILE);
        {   // the last tile: its second block has no successor
            const int off = (t & 3) * PF2_TILE;
            const float ma = step(s_a, s_b, pre, off + PF2_TILE / 2, off, 0, std::true_type{}, std::false_type{}, std::false_type{});
            prepare(s_b, 2 * t + 1, ma, std::false_type{});
            step(s_b, s_a, pre, 0, off + PF2_TILE / 2, 0, std::false_type{}, std::false_type{}, std::false_type{});
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // the look-ahead tiles were requested too: nothing may land after the wavefront has gone
    }

    // the two halves of a query hold disjoint keys: add their sums, then normalise and store
    l_run += __shfl_xor(l_run, 32, 64);
    if (PART && all_tiles > ntiles) {
        if (hl == 0) *(float2*)(a.part_ml + (slot * (PF2_WAVES * 32) + r) * 2) = make_float2(m_ref, l_run);
        float4* po = (float4*)a.part + (slot * PF2_WAVES + w) * (16 * 64) + lane;   // in register order: 1 KB per store
#pragma unroll
        for (int db = 0; db < 4; ++db)
#pragma unroll
            for (int c = 0; c < 4; ++c)
                po[(db * 4 + c) * 64] = make_float4(o[db][4 * c], o[db][4 * c + 1], o[db][4 * c + 2], o[db][4 * c + 3]);
        return;
    }
    // A lane holds four features of a row at a time: stored from there, a row of 256 bytes would leave in 16 pieces.  The wavefront's
    // 32 rows take the way through LDS instead (8 KB of its own; the 16-byte piece c of row j at c ^ (j % 16)) and leave whole.
    const float inv = l_run > 0.0f ? 1.0f / l_run : 0.0f;
    PF_LDS3 char* const mine = lds3 + w * 8192;
    __syncthreads();                             // every wavefront has left the tiles
#pragma unroll
    for (int db = 0; db < 4; ++db)
#pragma unroll
        for (int c = 0; c < 4; ++c)
            *(PF_LDS3 pf_u32x2*)(mine + j * 256 + (((db * 4 + c) ^ (j & 15)) << 4) + hl * 8) =
                pf_u32x2{pack_kv<F16>(o[db][4 * c] * inv, o[db][4 * c + 1] * inv), pack_kv<F16>(o[db][4 * c + 2] * inv, o[db][4 * c + 3] * inv)};
    const int piece = lane & 15;
#pragma unroll
    for (int x = 0; x < 8; ++x) {
        const int row = 4 * x + (lane >> 4), rr = w * 32 + row, t = t_wg0 + rr / G;
        const pf_u32x4 v = *(const PF_LDS3 pf_u32x4*)(mine + row * 256 + ((piece ^ (row & 15)) << 4));
        if (rr < BT * G && t < Q && piece * 8 < a.hd)
            *(pf_u32x4*)(a.out + (((int64_t)b * Q + t) * (a.kv_heads * G) + (h * G + rr % G)) * a.hd + piece * 8) = v;
    }
}
// A workgroup per query tile; SPLIT: blockIdx.z takes split_tiles tiles of the keys, and the merge kernel puts shares together.
template <bool F16, bool SPLIT>
__global__ __launch_bounds__(PF2_THREADS) void prefill_few_kernel(PrefillArgs a) {
    int seg = blockIdx.y, tile = (int)gridDim.x - 1 - (int)blockIdx.x;
    if ((gridDim.y & 7) == 0) {
        const int lin = (int)blockIdx.y * (int)gridDim.x + (int)blockIdx.x;
        const int turn = lin >> 3;
        seg = (lin & 7) + 8 * (turn / (int)gridDim.x);
        tile = (int)gridDim.x - 1 - turn % (int)gridDim.x;
    }
    const int t_first = SPLIT ? (int)blockIdx.z * a.split_tiles : 0;
    if (SPLIT && t_first > 0 && t_first >= tiles_seen(a, seg, tile)) return;
    attend_query_tile<F16, SPLIT>(a, seg, tile, t_first, a.split_tiles, ((int64_t)blockIdx.z * gridDim.y + seg) * gridDim.x + tile);
}
// The shares of the keys put together: one wavefront per (query tile, 32 of its rows, 32 features), lanes as they wrote.
// A share that a row saw nothing of has sum 0 and a reference of no meaning: it is left out.
template <bool F16>
__global__ __launch_bounds__(256) void prefill_few_merge_kernel(PrefillArgs a) {
    const int seg = blockIdx.y, tile = (int)blockIdx.x >> 3, w = (int)blockIdx.x & 7, tiles = (int)gridDim.x >> 3;
    const int b = seg / a.kv_heads, h = seg - b * a.kv_heads;
    int n = a.seg_len ? a.seg_len[seg] : a.max_len;
    n = max(0, min(n, a.max_len));
    const int db = threadIdx.x >> 6, lane = threadIdx.x & 63, j = lane & 31, hl = lane >> 5;
    const int G = a.group, Q = a.q_len, BT = (PF2_WAVES * 32) / G;
    const int t_last = min(Q - 1, tile * BT + BT - 1);
    const int all_tiles = (max(0, min(n, n - Q + t_last + 1)) + PF2_BN - 1) / PF2_BN;
    const int shares = (all_tiles + a.split_tiles - 1) / a.split_tiles;
    if (shares <= 1) return;                  // its workgroup wrote the result
    const int r = w * 32 + j, g = r % G, t_q = tile * BT + r / G;
    if (r >= BT * G || t_q >= Q) return;
    const int64_t wg = (int64_t)seg * tiles + tile, per_share = (int64_t)gridDim.y * tiles;
    auto slot = [&](int z) -> int64_t { return wg + z * per_share; };
    const float2* ml = (const float2*)a.part_ml + r;
    const float4* po = (const float4*)a.part + w * (16 * 64) + db * (4 * 64) + lane;
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
        const int d = db * 32 + 8 * c + 4 * hl;
        if (d < a.hd) *(uint2*)(orow + d * 2) = make_uint2(pack_kv<F16>(o[c].x * inv, o[c].y * inv), pack_kv<F16>(o[c].z * inv, o[c].w * inv));
    }
}

}  // namespace few
}  // namespace trimkv

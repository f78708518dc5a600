// Sliding-window attention of one new token per sequence -- gfx950 (masks, ring and arithmetic: window.hip.h).
//
//   window_decode_kernel   walks the rows in use in storage order without any mask; rows split over workgroups (split-K), all
//                          query heads of a KV head share the rows; 64 / L rows per load instruction, L lanes with 8 features
//                          each per row
//   window_combine_kernel  the splits' shares
#include "window.hip.h"
#include <type_traits>

namespace trimkv {

// ---- decode --------------------------------------------------------------------------------------
template <int CTRL>
__device__ __forceinline__ float dpp_add(float v) {
    return v + __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, true));
}
// sum over aligned groups of L lanes, result in every lane
template <int L>
__device__ __forceinline__ float group_sum(float v) {
    v = dpp_add<0xB1>(v);                        // quad_perm 1,0,3,2
    v = dpp_add<0x4E>(v);                        // quad_perm 2,3,0,1
    if constexpr (L >= 8) v = dpp_add<0x141>(v); // row_half_mirror
    if constexpr (L >= 16) v = dpp_add<0x140>(v);// row_mirror
    if constexpr (L >= 32) v += __shfl_xor(v, 16, 64);
    if constexpr (L >= 64) v += __shfl_xor(v, 32, 64);
    return v;
}

struct Row8 { float f[8]; };
__device__ __forceinline__ hy_u32x4 raw8(const bf16_t* p) { return __builtin_nontemporal_load((const hy_u32x4*)p); }
__device__ __forceinline__ void widen(hy_u32x4 r, float (&f)[8]) {
#pragma unroll
    for (int x = 0; x < 4; ++x) { f[2 * x] = __uint_as_float(r[x] << 16); f[2 * x + 1] = __uint_as_float(r[x] & 0xffff0000u); }
}
struct Raw8f { float4 lo, hi; };
__device__ __forceinline__ Raw8f raw8(const float* p) { return {*(const float4*)p, *(const float4*)(p + 4)}; }
__device__ __forceinline__ void widen(Raw8f r, float (&f)[8]) {
    f[0] = r.lo.x; f[1] = r.lo.y; f[2] = r.lo.z; f[3] = r.lo.w; f[4] = r.hi.x; f[5] = r.hi.y; f[6] = r.hi.z; f[7] = r.hi.w;
}

// Rows of 16 lanes in bf16: a lane's sixteen products (16 / GQ rows and GQ heads) are added up over the lanes of a row so that lane c ends with the sum of
// product summed_at(c).  Its bits 0, 1, 2 and 3 pick the half that it keeps at each step (of bits 3, 1, 2 and 0 of the product's place).
__device__ __forceinline__ float sum_to_lanes(float (&v)[16], int c) {
    auto fold = [&](int half, bool upper, auto ctrl) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            if (i >= half) continue;
            const float stays = upper ? v[i + half] : v[i], goes = upper ? v[i] : v[i + half];
            v[i] = stays + __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(goes), decltype(ctrl)::value, 0xf, 0xf, true));
        }
    };
    fold(8, c & 4, std::integral_constant<int, 0x141>{});       // row_half_mirror: lane c ^ 7
    fold(4, c & 1, std::integral_constant<int, 0xB1>{});        // lane c ^ 1
    fold(2, c & 2, std::integral_constant<int, 0x4E>{});        // lane c ^ 2
    fold(1, c & 8, std::integral_constant<int, 0x128>{});       // row_ror:8: lane c ^ 8
    return v[0];
}
// place of (row u, head x): rows on the low lane bits, so that lanes c ^ 1, c ^ 2 and c ^ 7 have other rows of one head
template <int GQ> __device__ __forceinline__ constexpr int place_of(int u, int x) {
    const int c = u + x * (16 / GQ);                 // the lane that ends with it
    return (c & 4) << 1 | (c & 1) << 2 | (c & 2) | c >> 3;
}
template <int CTRL> __device__ __forceinline__ float dpp_max(float v) {
    return fmaxf(v, __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, true)));
}
__device__ __forceinline__ float dot8(hy_u32x4 a, hy_u32x4 b) {
    float d = 0.0f;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const uint32_t p = a[i], r = b[i];          // a bit cast of a vector's element itself takes the first one
        d = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(hy_bf16x2, p), __builtin_bit_cast(hy_bf16x2, r), d, false);
    }
    return d;
}

// Rows of 16 lanes in bf16, shared by two heads or more: with every product summed over a row's lanes by itself (four additions in each of them) and every
// exponential taken by all sixteen, vector instructions bounded it.  Here the sums of sixteen products take 15 additions together, a lane takes one exponential of a
// step, and factors that are 1 are not multiplied with; the rest is the stream of rows and sequences of unlike length, whose workgroups do not end together.  us, with
// the combination: 8 KV heads of 128, 64 sequences of 256 .. 4096 rows, 4 heads each 85 -> 73, of 4096 184 -> 175, of 64 .. 1024 35 -> 29, 128 of 256 .. 4096 151 -> 132; 8
// heads each, 32 of 256 .. 4096 80 -> 57; 2 heads each, 64 of 128 .. 2048 41.5 -> 39.  Rows of all sequences cut into equal shares for as many workgroups as are
// resident: 75 - 79, of 4096 165, of 4 .. 64 52 for 12: not taken.
template <typename T, int L, int GQ>
__global__ __launch_bounds__(256) void window_decode_kernel(WindowArgs a) {
    constexpr bool SHARED = std::is_same<T, bf16_t>::value && L == 16 && GQ >= 2;
    constexpr int R = 64 / L, U = SHARED ? 16 / GQ : GQ >= 8 ? 2 : 4, WAVES = 4;
    extern __shared__ float lds[];                  // [WAVES][GQ][L * 8 + 2]
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    const int per = a.H / a.G, passes = (per + GQ - 1) / GQ;
    // heads on the fast axis: workgroups go to the eight XCDs in turn, and with the splits there the XCDs of the later ones, which
    // short sequences do not have, would idle
    // The sequences begin five further on with every split: with them in one order the shares of a sequence, a multiple of `batch`
    // workgroups apart, meet on the same compute units (8 sequences of 256 .. 4096 rows 27.5 -> 20.8 us in one order, 25.5 -> 21.0 in
    // another, 16 of them 32.8 -> 30.0 and 30.1 -> 31.1).
    const int split = blockIdx.z, g = blockIdx.x / passes, h0 = (blockIdx.x % passes) * GQ, b = (int)((blockIdx.y + 5 * blockIdx.z) % gridDim.y);
    const int nh = min(GQ, per - h0);
    const int slot = a.slots[b], cap = a.keep + a.size;
    const int n = min(a.seen[2 * slot] + 1, cap);
    const int r0 = split * a.chunk, r1 = min(n, r0 + a.chunk);
    const int e = (lane % L) * 8, sub = lane / L;
    const bool kin = e < a.Dp, vin = e < a.Dvp;     // padded dims are multiples of 8
    const T* rk = (const T*)a.rk + ((int64_t)slot * a.G + g) * cap * a.Dp + (kin ? e : 0);
    const T* rv = (const T*)a.rv + ((int64_t)slot * a.G + g) * cap * a.Dvp + (vin ? e : 0);
    float m[GQ], l[GQ], acc[GQ][8];
#pragma unroll
    for (int x = 0; x < GQ; ++x) {
        m[x] = WA_NEG; l[x] = 0.0f;
#pragma unroll
        for (int y = 0; y < 8; ++y) acc[x][y] = 0.0f;
    }
    if constexpr (SHARED) {
        hy_u32x4 q[GQ];
#pragma unroll
        for (int x = 0; x < GQ; ++x) {
            q[x] = raw8((const T*)a.q + ((int64_t)b * a.H + g * per + h0 + min(x, nh - 1)) * a.Dp + (kin ? e : 0));
            q[x] = kin ? q[x] : hy_u32x4{0, 0, 0, 0};
        }
        if (r0 >= n) return;                        // a short sequence has fewer shares; the combination knows (q is on its way by now)
        const int c = lane & 15, mine = c % U;      // this lane's row of a step; its head is c / U
        float* const sh = lds + wv * 128 + sub * 16;            // a step's probabilities of this row of lanes, [U][GQ], and 64 further on its heads' factors
        float top = WA_NEG, sum = 0.0f;
        hy_u32x4 kn[U], vn[U];
        auto request = [&](int base) __attribute__((always_inline)) {       // rows that are not there are the last one again
#pragma unroll
            for (int u = 0; u < U; ++u) kn[u] = raw8(rk + (int64_t)min(base + u * R + sub, r1 - 1) * a.Dp);
#pragma unroll
            for (int u = 0; u < U; ++u) vn[u] = raw8(rv + (int64_t)min(base + u * R + sub, r1 - 1) * a.Dvp);
        };
        constexpr bool AHEAD = U <= 4;              // the next step's rows are requested before this one's are used, where registers allow it
        if (AHEAD) request(r0 + wv * R * U);
        for (int base = r0 + wv * R * U; base < r1; base += WAVES * R * U) {
            if (!AHEAD) request(base);
            hy_u32x4 kr[U], vr[U];
#pragma unroll
            for (int u = 0; u < U; ++u) { kr[u] = kn[u]; vr[u] = vn[u]; }
            if (AHEAD) request(base + WAVES * R * U);
            float d[16];
#pragma unroll
            for (int u = 0; u < U; ++u)
#pragma unroll
                for (int x = 0; x < GQ; ++x) d[place_of<GQ>(u, x)] = dot8(q[x], kr[u]);
            float s = sum_to_lanes(d, c) * a.scale_log2;
            s = base + mine * R + sub < r1 ? s : WA_NEG;
            float mn = dpp_max<0xB1>(s);
            if constexpr (U >= 4) mn = dpp_max<0x4E>(mn);
            if constexpr (U >= 8) mn = dpp_max<0x141>(mn);
            mn = fmaxf(top, mn);
            const float alpha = __builtin_amdgcn_exp2f(top - mn), p = s > 0.5f * WA_NEG ? __builtin_amdgcn_exp2f(s - mn) : 0.0f;
            top = mn;
            sum = sum * alpha + p;
            sh[mine * GQ + c / U] = p;
            const bool moved = __builtin_amdgcn_ballot_w64(!(alpha == 1.0f)) != 0;      // wavefront-uniform; seldom after the first rows
            if (moved && mine == 0) sh[64 + c / U] = alpha;
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");       // of this wavefront's own
            if (moved) {
#pragma unroll
                for (int x = 0; x < GQ; ++x) {
                    const float f = sh[64 + x];
#pragma unroll
                    for (int y = 0; y < 8; ++y) acc[x][y] *= f;
                }
            }
#pragma unroll
            for (int u = 0; u < U; ++u) {
                float vf[8], w[GQ];
                widen(vr[u], vf);
#pragma unroll
                for (int x = 0; x < GQ; ++x) w[x] = sh[u * GQ + x];
#pragma unroll
                for (int x = 0; x < GQ; ++x)
#pragma unroll
                    for (int y = 0; y < 8; ++y) acc[x][y] = fmaf(w[x], vf[y], acc[x][y]);
            }
            asm volatile("" ::: "memory");          // the next step's are written behind these reads
        }
        sum = dpp_add<0xB1>(sum);
        if constexpr (U >= 4) sum = dpp_add<0x4E>(sum);
        if constexpr (U >= 8) sum = dpp_add<0x141>(sum);
        if (mine == 0) { sh[c / U] = top; sh[64 + c / U] = sum; }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
        for (int x = 0; x < GQ; ++x) { m[x] = sh[x]; l[x] = sh[64 + x]; }
        __syncthreads();                            // the sums below take this room
    } else {
        float q[GQ][8];
#pragma unroll
        for (int x = 0; x < GQ; ++x) {
            widen(raw8((const T*)a.q + ((int64_t)b * a.H + g * per + h0 + min(x, nh - 1)) * a.Dp + (kin ? e : 0)), q[x]);
#pragma unroll
            for (int y = 0; y < 8; ++y) q[x][y] = kin ? q[x][y] * a.scale_log2 : 0.0f;
        }
        if (r0 >= n) return;
        using Raw = decltype(raw8((const T*)nullptr));
        for (int base = r0 + wv * R * U; base < r1; base += WAVES * R * U) {
            Raw kr[U], vr[U];
#pragma unroll
            for (int u = 0; u < U; ++u) kr[u] = raw8(rk + (int64_t)min(base + u * R + sub, r1 - 1) * a.Dp);
#pragma unroll
            for (int u = 0; u < U; ++u) vr[u] = raw8(rv + (int64_t)min(base + u * R + sub, r1 - 1) * a.Dvp);
            float s[U][GQ];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                float kf[8];
                widen(kr[u], kf);
                const bool in = base + u * R + sub < r1;
#pragma unroll
                for (int x = 0; x < GQ; ++x) {
                    float d = 0.0f;
#pragma unroll
                    for (int y = 0; y < 8; ++y) d = fmaf(q[x][y], kf[y], d);
                    d = group_sum<L>(d);
                    s[u][x] = in ? d : WA_NEG;
                }
            }
#pragma unroll
            for (int x = 0; x < GQ; ++x) {
                float mn = m[x];
#pragma unroll
                for (int u = 0; u < U; ++u) mn = fmaxf(mn, s[u][x]);
                const float alpha = __builtin_amdgcn_exp2f(m[x] - mn);
                m[x] = mn;
                float ps = 0.0f;
#pragma unroll
                for (int u = 0; u < U; ++u) { s[u][x] = s[u][x] > 0.5f * WA_NEG ? __builtin_amdgcn_exp2f(s[u][x] - mn) : 0.0f; ps += s[u][x]; }
                l[x] = l[x] * alpha + ps;
#pragma unroll
                for (int y = 0; y < 8; ++y) acc[x][y] *= alpha;
            }
#pragma unroll
            for (int u = 0; u < U; ++u) {
                float vf[8];
                widen(vr[u], vf);
#pragma unroll
                for (int x = 0; x < GQ; ++x)
#pragma unroll
                    for (int y = 0; y < 8; ++y) acc[x][y] = fmaf(s[u][x], vf[y], acc[x][y]);
            }
        }
    }
    // lanes that hold the same features of different rows meet, then the wavefronts
    constexpr int ROW = L * 8 + 2;
#pragma unroll
    for (int x = 0; x < GQ; ++x) {
#pragma unroll
        for (int d = L; d < 64; d <<= 1) {
            const float mo = __shfl_xor(m[x], d, 64), lo = __shfl_xor(l[x], d, 64), mn = fmaxf(m[x], mo);
            const float f0 = __builtin_amdgcn_exp2f(m[x] - mn), f1 = __builtin_amdgcn_exp2f(mo - mn);
            m[x] = mn;
            l[x] = l[x] * f0 + lo * f1;
#pragma unroll
            for (int y = 0; y < 8; ++y) acc[x][y] = acc[x][y] * f0 + __shfl_xor(acc[x][y], d, 64) * f1;
        }
        float* row = lds + (wv * GQ + x) * ROW;
        if (sub == 0) {
#pragma unroll
            for (int y = 0; y < 8; ++y) row[e + y] = acc[x][y];
            if (lane == 0) { row[L * 8] = m[x]; row[L * 8 + 1] = l[x]; }
        }
    }
    __syncthreads();
    for (int idx = tid; idx < nh * a.Dv; idx += 256) {
        const int x = idx / a.Dv, d = idx - x * a.Dv;
        float mm = WA_NEG;
#pragma unroll
        for (int w = 0; w < WAVES; ++w) mm = fmaxf(mm, lds[(w * GQ + x) * ROW + L * 8]);
        float num = 0.0f, den = 0.0f;
#pragma unroll
        for (int w = 0; w < WAVES; ++w) {
            const float* row = lds + (w * GQ + x) * ROW;
            const float f = __builtin_amdgcn_exp2f(row[L * 8] - mm);
            num += row[d] * f;
            den += row[L * 8 + 1] * f;
        }
        const int h = g * per + h0 + x;
        if (a.splits == 1) {
            st((T*)a.out + ((int64_t)b * a.H + h) * a.Dv + d, num / (den + window_sink(a, mm)) * window_gate<T>(a, b, h, d));
        } else {
            float* w = a.ws + (((int64_t)b * a.H + h) * a.splits + split) * (a.Dv + 2);
            w[d] = num;
            if (d == 0) { w[a.Dv] = mm; w[a.Dv + 1] = den; }
        }
    }
}

template <typename T>
__global__ __launch_bounds__(256) void window_combine_kernel(WindowArgs a) {
    __shared__ float f[256];                        // a split's share of the result
    __shared__ float part[4];
    const int64_t bh = blockIdx.x;
    const int64_t b = bh / a.H;
    const int h = (int)(bh - b * a.H), tid = threadIdx.x, row = a.Dv + 2;
    const float* w = a.ws + bh * a.splits * row;
    // everything is requested before the number of shares is known
    float m = w[min(tid, a.splits - 1) * row + a.Dv], l = w[min(tid, a.splits - 1) * row + a.Dv + 1];
    const int shares = min(a.splits, (min(a.seen[2 * a.slots[b]] + 1, a.keep + a.size) + a.chunk - 1) / a.chunk);
    m = tid < shares ? m : WA_NEG;
    l = tid < shares ? l : 0.0f;
    const float wm = wave_max_f(m);
    if ((tid & 63) == 0) part[tid >> 6] = wm;
    __syncthreads();
    const float mm = fmaxf(fmaxf(part[0], part[1]), fmaxf(part[2], part[3]));
    __syncthreads();
    const float e = __builtin_amdgcn_exp2f(m - mm);
    const float inv = 1.0f / (block_sum_f(l * e, part, 4) + window_sink(a, mm));
    f[tid] = e * inv;
    __syncthreads();
    for (int d = tid; d < a.Dv; d += 256) {
        float num = 0.0f;
#pragma unroll 8
        for (int s = 0; s < shares; ++s) num += w[s * row + d] * f[s];
        st((T*)a.out + bh * a.Dv + d, num * window_gate<T>(a, b, h, d));
    }
}

template <typename T, int L>
static void launch_window_decode(const WindowArgs& a, int batch, hipStream_t s) {
    const int per = a.H / a.G;
    auto go = [&](auto gq) {
        constexpr int GQ = decltype(gq)::value;
        const int passes = (per + GQ - 1) / GQ;
        hipLaunchKernelGGL((window_decode_kernel<T, L, GQ>), dim3(a.G * passes, batch, a.splits), dim3(256), 4 * GQ * (L * 8 + 2) * sizeof(float), s, a);
    };
    if (per == 1) go(std::integral_constant<int, 1>{});
    else if (per == 2) go(std::integral_constant<int, 2>{});
    else if (per <= 4 || L >= 64) go(std::integral_constant<int, 4>{});
    else go(std::integral_constant<int, 8>{});
}

}  // namespace trimkv

using namespace trimkv;

constexpr int SHARE_ROWS = 1024;

extern "C" int trimkv_window_decode_splits(int batch, int kv_heads, int capacity) {
    if (batch <= 0 || kv_heads <= 0 || capacity <= 0) return 1;
    // Enough workgroups to fill the chip, at least 128 rows for each and no more than 1024: a batch's sequences differ in length, and
    // the launch ends with the workgroup that has the most rows.  At most 1024, 820, 512 rows, us: 64 sequences of 256 .. 4096 rows x 8
    // heads of 128 71, 73, 71 (in another order 76, 76, 73), of 64 .. 1024 rows 29, 28, 29, of full windows of 4096 176, 173, 180;
    // 128 sequences of 256 .. 4096 134, 133, 132, of full windows 346, 353, 361: fewer rows than 1024 cost the fuller batches.
    // With enough pairs to fill the chip as they are (2048) others run while the longest ones finish, and splitting costs full
    // windows more than it gives unequal ones.  With the bound of 1024 rows -> without, us, before a row's lanes shared their sums, full windows | lengths from 256 rows
    // up (log-uniform): 2048 pairs of 4096 rows 705 -> 650 | 263 -> 288, 4096 of 4096 1434 -> 1281 | 520 -> 500, of 2048 720 -> 644 |
    // 335 -> 315; kept below: 512 of 16384 696 -> 659 | 216 -> 263, of 8192 351 -> 340 | 143 -> 154, 1024 of 4096 353 -> 342 | 155 -> 163.
    const int64_t pairs = (int64_t)batch * kv_heads;
    int64_t s = (2048 + pairs - 1) / pairs;
    const int most = (capacity + 127) / 128, least = (capacity + SHARE_ROWS - 1) / SHARE_ROWS;
    if (pairs < 2048 && s < least) s = least;
    s = s < 1 ? 1 : s > most ? most : s;
    return (int)(s > 256 ? 256 : s);
}

extern "C" int trimkv_window_decode(const void* q, const void* ring_k, const void* ring_v, const int32_t* slots, const int32_t* seen,
                                    const void* gate, int64_t gate_stride, void* out, int batch, int heads, int kv_heads, int dim, int vdim,
                                    int dim_stride, int vdim_stride, int keep_first, int window, float scale, int head_gate, int sink, int splits, float* workspace,
                                    int dtype, void* stream) {
    const char* fn = "trimkv_window_decode";
    WindowArgs a{};
    a.q = q; a.rk = ring_k; a.rv = ring_v; a.slots = slots; a.seen = seen; a.gate = gate; a.gate_stride = gate_stride; a.out = out;
    a.H = heads; a.G = kv_heads; a.D = dim; a.Dv = vdim; a.Dp = dim_stride; a.Dvp = vdim_stride; a.keep = keep_first; a.size = window;
    a.scale_log2 = scale * 1.4426950408889634f; a.splits = splits; a.ws = workspace; a.head_gate = head_gate; a.sink = sink;
    if (int rc = window_common(fn, a, batch, dtype)) return rc;
    if (splits < 1 || splits > 256 || (splits > 1 && !workspace)) return fail(TRIMKV_ERR_WORKSPACE, "%s: splits=%d needs a workspace", fn, splits);
    const int cap = keep_first + window;
    a.chunk = (cap + splits - 1) / splits;
    const int lanes = ((dim_stride > vdim_stride ? dim_stride : vdim_stride) + 7) / 8;
    hipStream_t s = (hipStream_t)stream;
    HY_BY_DTYPE(dtype, T,
        if (lanes <= 4) launch_window_decode<T, 4>(a, batch, s);
        else if (lanes <= 8) launch_window_decode<T, 8>(a, batch, s);
        else if (lanes <= 16) launch_window_decode<T, 16>(a, batch, s);
        else if (lanes <= 32) launch_window_decode<T, 32>(a, batch, s);
        else launch_window_decode<T, 64>(a, batch, s));
    int rc = launch_status(fn);
    if (rc || splits == 1) return rc;
    HY_BY_DTYPE(dtype, T, hipLaunchKernelGGL((window_combine_kernel<T>), dim3(batch * heads), dim3(256), 0, s, a));
    return launch_status(fn);
}

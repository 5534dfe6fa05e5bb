// mid_k_kernel.hip - the kernel of batches that mix rows: greedy rows, rows that sample from k <= 2048 candidates and rows
// with every token a candidate (top_k = 0), with every penalty, and verification windows with penalties.
//
// One workgroup of SK_LT threads per (row, segment), the segment's logits requested at once and kept in registers, as in
// the small-k kernel. A row's segments agree on one bound before any of them writes a candidate:
//   - the window's ids in the segment are a bitmap laid out by thread (and 16-bit counts, frequency / presence): each
//     wave moves its flagged logits to a list in LDS (a long window's to memory) and penalises them while the row's
//     segments meet, one entry per lane, so the rest of the segment needs no penalty arithmetic;
//   - each wave sorts its 64 lane maxima in registers and publishes them at 16 ranks (1, 2, 3, ... 64, weights adding up
//     to 64); the row's segments meet (an L2 counter), and every one takes the same bound from the row's published keys:
//     the largest T such that the ranks published at or above T add up to k. k distinct logits of the row then reach T,
//     whatever the other segments hold;
//   - the logits at or above T (about 1.05 k to 1.4 k per row) go to the row's list, one L2 atomic per wave for its
//     places; the last segment to finish (an L2 ticket) sorts the list and samples the row.
// The waiting is bounded and a row's segments are consecutive workgroups of one XCD, dispatched in order; a segment that
// gives up (or a list that overflows: thousands of equal logits at the bound) marks the row, and its last segment then
// selects the row's exact top k from the logits alone (mk_slow). Equal logits at the bound in larger numbers than the list
// takes are counted first (one meeting more), and only the row's first ones written.
// Bound: HBM, one read of the logits, then the chain behind a row's last logits.
// Measured against the fused kernel (running bounds, per-row merges of the segments' lists): 256 rows of 262144 logits
// with k from 1 to 2048 and every penalty 124 us -> 75; 24 rows of 100003 logits, k 200, frequency / presence 35 -> 17.9;
// 40 rows of a verification window over 262144 logits, k 50, repetition 26.5 -> 22.
// Rows with every token a candidate (ak_segment, ak_finish) stay in registers through all their passes; the fused kernel
// reads such a row again for each, and gave flat ones to one workgroup: 32 rows of 65536 N(0, 2) logits at temperature 1
// 51.5 us -> 24.2, 3 rows of 178740 698 -> 28.6, 64 rows of 262144 heavy-tailed logits with top-p 0.95 37.5 -> 37.1.
#include "exp_table.hpp"
#include "row_device.hpp"

#include <type_traits>

namespace fs {

constexpr int MK_K = 2048;                 // largest k
constexpr int MK_LCAP = MK_LIST;           // entries of a row's list
constexpr int MK_TOP = 2560;               // sorted candidates: k plus the rest of the bin that holds the k-th
constexpr int MK_BINS = 2048;              // bins of the merge's counting sort
constexpr int MK_H = 1024;                 // bins of the bound's histograms and of mk_slow's digits
constexpr int MK_PC = 512;                 // penalised logits of a segment kept in LDS
constexpr int MK_W = 4;                    // window ids per thread requested behind the logits
// published ranks of a wave's 64 sorted lane maxima, and what each adds to the rank before it
constexpr uint64_t MK_RANK_LO = 0x0A08060504030201ull, MK_RANK_HI = 0x403028201814100Cull;   // 1..6, 8, 10; 12..64
__device__ __forceinline__ uint32_t mk_rank(int j) {
    return (uint32_t)((j < 8 ? MK_RANK_LO >> (8 * j) : MK_RANK_HI >> (8 * (j - 8))) & 0xFFu);
}

constexpr int AK_BINS = 2048;              // every token a candidate: mass bins of a row
constexpr int AK_STAGE = 1024;             // logits of the searched bins that a segment stages, per list
constexpr int AK_LIST = MK_LCAP / 2;       // entries of a row's two lists of such logits
constexpr int AK_VALS = 64;                // distinct values of the searched bins in a chunk of ak_values
constexpr float AK_DEPTH = 32.0f;          // temperatures below the maximum that the bins reach
constexpr double AK_FX = 17592186044416.0; // 2^44: fixed-point mass scale of ak_slow (a mass is <= 1)

struct MkShared {
    // in turn: the window's 16-bit counts per logit of the segment (frequency / presence); the merge's sorted candidates
    // and its bins
    union {
        uint32_t cnt[SK_LT * 16 * 4 / 2];
        struct {
            uint64_t top[MK_TOP];
            uint32_t bins[MK_BINS + 1];
        } m;
        struct {
            uint64_t top[MK_K];            // (u.m.top's head)
            double e[MK_K];                // their masses, then probabilities
        } w;
        struct {
            uint64_t mass[AK_BINS];        // every token a candidate: fixed-point masses by bin, the segment's, then
            uint64_t cum[SK_LT];           //   the row's, and the mass up to and with each eight
        } a;
        struct {
            uint64_t l[2][AK_STAGE];       //   this segment's logits of the bins searched, ~id above the value
        } g;
        struct {
            uint32_t cnt[SK_LT * 8 * 4 / 2];   // ak_slow: a chunk's counts beside a digit's masses
            union {
                uint64_t mass[MK_H];
                uint64_t sub[2][MK_H];         // ak_values: masses within the crossing's bin, within the draw's
                struct {
                    uint32_t key[AK_VALS], cnt[AK_VALS];
                } val[2];                      //   a chunk's values of both, and how often each occurs
            };
        } z;
    } u;
    union {
        uint32_t hist[MK_H];               // the bound's histograms; mk_slow's digits
        uint32_t rk[SK_LT];                // partial ranks of a short list
        uint32_t srt[SK_NW][WAVE];         // the waves' sorted lane maxima
        double2 pow2[64];                  // every token a candidate: 2^(j/64) in two parts
    } h;
    union {
        uint32_t bmp[SK_LT * 2];           // one bit per logit of the window's ids: 64 bits per thread; mk_slow: by id
        float pv[MK_PC];                   // (the bits are read) the flagged logits, raw, then penalised
    } b;
    uint16_t prel[MK_PC];                  //   and their places in the segment
    uint32_t np;                           //   places given out
    uint64_t w64[SK_NW];
    double wf[SK_NW];
    uint32_t w32[SK_NW];
    uint32_t misc[6];
    double dmisc;
    uint64_t umisc[2];
    uint32_t gn[4];
#ifdef FS_TRACE
    uint64_t trace_t[16];
#endif
};

// ---- block reductions of SK_LT threads (each starts after and ends with a barrier)
__device__ __forceinline__ uint32_t mk_excl_u32(uint32_t v, MkShared& s, uint32_t& total) {
    const int w = threadIdx.x / WAVE;
    const uint32_t x = wave_incl_scan_u32(v);
    if (lane_id() == WAVE - 1) s.w32[w] = x;
    __syncthreads();
    uint32_t off = 0u, tot = 0u;
#pragma unroll
    for (int q = 0; q < SK_NW; ++q) {
        off += q < w ? s.w32[q] : 0u;
        tot += s.w32[q];
    }
    __syncthreads();
    total = tot;
    return off + x - v;
}
__device__ __forceinline__ double mk_excl_f64(double v, MkShared& s, double& total) {
    const int w = threadIdx.x / WAVE;
    const double x = wave_scan_f64(v);
    const double ex = dpp_f64<0x138, 0xF>(x);                  // wave_shr:1 (lane 0 reads 0)
    if (lane_id() == WAVE - 1) s.wf[w] = x;
    __syncthreads();
    double off = 0.0, tot = 0.0;
#pragma unroll
    for (int q = 0; q < SK_NW; ++q) {
        if (q < w) off += s.wf[q];
        tot += s.wf[q];
    }
    __syncthreads();
    total = tot;
    return off + ex;
}
template <class Op>
__device__ __forceinline__ uint64_t mk_reduce_u64(uint64_t v, MkShared& s, Op op) {
    v = wave_allreduce(v, op);
    if (lane_id() == 0) s.w64[threadIdx.x / WAVE] = v;
    __syncthreads();
    uint64_t m = s.w64[0];
#pragma unroll
    for (int w = 1; w < SK_NW; ++w) m = op(m, s.w64[w]);
    __syncthreads();
    return m;
}
__device__ __forceinline__ uint64_t mk_max_u64(uint64_t v, MkShared& s) {
    return mk_reduce_u64(v, s, [](uint64_t x, uint64_t y) { return y > x ? y : x; });
}
__device__ __forceinline__ uint64_t mk_min_u64(uint64_t v, MkShared& s) {
    return mk_reduce_u64(v, s, [](uint64_t x, uint64_t y) { return y < x ? y : x; });
}

// From s.h.hist: the bin b with count(bins > b) < kk <= count(bins >= b) and the count above it; false when the
// histogram holds fewer than kk. Whole workgroup, after a barrier; ends with one.
__device__ __forceinline__ bool mk_locate(MkShared& s, uint32_t kk, uint32_t& b, uint32_t& above) {
    static_assert(MK_H == 4 * SK_LT, "four bins per thread");
    const int tid = threadIdx.x;
    const uint4 c = *reinterpret_cast<const uint4*>(&s.h.hist[MK_H - 4 - 4 * tid]);   // descending: w, z, y, x
    const uint32_t mine = c.x + c.y + c.z + c.w;
    uint32_t tot;
    const uint32_t ex = mk_excl_u32(mine, s, tot);
    if (tot < kk) return false;                                // uniform
    if (ex < kk && ex + mine >= kk) {
        uint32_t a = ex, j = 0u;
        if (a + c.w < kk) { a += c.w; j = 1u;
            if (a + c.z < kk) { a += c.z; j = 2u;
                if (a + c.y < kk) { a += c.y; j = 3u; } } }
        s.misc[0] = (uint32_t)(MK_H - 1 - 4 * tid) - j;
        s.misc[1] = a;
    }
    __syncthreads();
    b = s.misc[0];
    above = s.misc[1];
    return true;
}

// The row's bound from its segments' published keys (nseg * SK_NW lists of 16): the largest 20-bit prefix T (sign,
// exponent, 11 mantissa bits) such that the weights of the keys at or above it add up to k, 1 when they do not. Two
// histograms of ten key bits each in LDS. sum: those weights' sum; need: what the keys of T's own prefix have to add.
// Whole workgroup; s.h.hist is zero on entry.
template <int NQ>
__device__ __forceinline__ uint32_t mk_bound(const uint32_t* qk, int nseg, int k, MkShared& s, uint32_t& sum,
                                             uint32_t& need) {
    const int tid = threadIdx.x;
    const int n4 = nseg * SK_NW * 4;                           // 16-byte quarters of the lists
    uint4 e[NQ];
#pragma unroll
    for (int r = 0; r < NQ; ++r) {
        const int i = r * SK_LT + tid;
        e[r] = i < n4 ? reinterpret_cast<const uint4*>(qk)[i] : make_uint4(0u, 0u, 0u, 0u);
    }
    // weights of quarter (tid & 3) of a list: 1 1 1 1 | 1 1 2 2 | 2 4 4 4 | 8 8 8 16
    const uint32_t pk = (tid & 3) == 0 ? 0x01010101u : (tid & 3) == 1 ? 0x02020101u : (tid & 3) == 2 ? 0x04040402u : 0x10080808u;
    auto add = [&](uint32_t key, uint32_t wgt, uint32_t hi, int level) {
        if (key == 0u) return;
        if (level == 0) atomicAdd(&s.h.hist[key >> 22], wgt);
        else if (key >> 22 == hi) atomicAdd(&s.h.hist[(key >> 12) & 1023u], wgt);
    };
    uint32_t hi = 0u, lo = 0u, above = 0u, above2 = 0u;
#pragma unroll
    for (int r = 0; r < NQ; ++r) {
        add(e[r].x, pk & 255u, 0u, 0);
        add(e[r].y, (pk >> 8) & 255u, 0u, 0);
        add(e[r].z, (pk >> 16) & 255u, 0u, 0);
        add(e[r].w, pk >> 24, 0u, 0);
    }
    __syncthreads();
    sum = need = 0u;
    if (!mk_locate(s, (uint32_t)k, hi, above)) return 1u;
    *reinterpret_cast<uint4*>(&s.h.hist[4 * tid]) = make_uint4(0u, 0u, 0u, 0u);   // (mk_locate's reads are over)
    __syncthreads();
#pragma unroll
    for (int r = 0; r < NQ; ++r) {
        add(e[r].x, pk & 255u, hi, 1);
        add(e[r].y, (pk >> 8) & 255u, hi, 1);
        add(e[r].z, (pk >> 16) & 255u, hi, 1);
        add(e[r].w, pk >> 24, hi, 1);
    }
    __syncthreads();
    (void)mk_locate(s, (uint32_t)k - above, lo, above2);
    sum = above + above2 + s.h.hist[lo];
    need = (uint32_t)k - above - above2;
    const uint32_t T = (hi << 22) | (lo << 12);
    return T ? T : 1u;
}

// T's other twelve bits: the largest key such that the weights of the keys at or above it add up to k.
__device__ __forceinline__ uint32_t mk_bound_exact(const uint32_t* qk, int nseg, uint32_t T, uint32_t need, MkShared& s) {
    const int tid = threadIdx.x;
    const uint32_t wgt = mk_rank(tid & 15) - ((tid & 15) ? mk_rank((tid & 15) - 1) : 0u);
#pragma unroll 1
    for (int sh = 2, bits = 10; sh >= 0; sh -= 2, bits = 2) {
        __syncthreads();
        *reinterpret_cast<uint4*>(&s.h.hist[4 * tid]) = make_uint4(0u, 0u, 0u, 0u);
        __syncthreads();
#pragma unroll 1
        for (int i = tid; i < nseg * SK_NW * 16; i += SK_LT) {
            const uint32_t key = qk[i];
            if (key >> (sh + bits) == T >> (sh + bits)) atomicAdd(&s.h.hist[(key >> sh) & ((1u << bits) - 1u)], wgt);
        }
        __syncthreads();
        uint32_t b = 0u, above = 0u;
        (void)mk_locate(s, need, b, above);
        T |= b << sh;
        need -= above;
    }
    return T;
}

// The row's window of history ids: na ids of the stream's history, then nb of the drafts fed before this row.
struct MkWin {
    const int32_t* pa;
    const int32_t* pb;
    int64_t na;
    int nb;
    __device__ __forceinline__ int at(int64_t i) const { return i < na ? pa[i] : pb[i - na]; }
    __device__ __forceinline__ int64_t n() const { return na + nb; }
};
struct MkPen {
    float rep, fq, pres, cap;
    bool rep_on, fp_on;
    // ferro's penalties on one raw logit with c occurrences in the window (sampler.cpp:11-18 and the extension)
    __device__ __forceinline__ float apply(float l, uint32_t c) const {
        if (rep_on) l = l > 0.0f ? __fdiv_rn(l, rep) : __fmul_rn(l, rep);
        if (fp_on) l = __fsub_rn(l, __fadd_rn(__fmul_rn((float)c, fq), pres));
        return l;
    }
};

// f(logit, place) for a chunk of n logits of a row that one workgroup selects alone: eight loads in flight per thread.
template <class F>
__device__ __forceinline__ void slow_each(const float* p, int n, F f) {
#pragma unroll 1
    for (int i0 = threadIdx.x; i0 < n; i0 += 8 * SK_LT) {
        float x[8];
#pragma unroll
        for (int q = 0; q < 8; ++q) x[q] = i0 + q * SK_LT < n ? p[i0 + q * SK_LT] : 0.0f;
#pragma unroll 1
        for (int q = 0; q < 8 && i0 + q * SK_LT < n; ++q) {
            float l = x[0];
#pragma unroll
            for (int t = 1; t < 8; ++t) l = q == t ? x[t] : l;
            f(l, i0 + q * SK_LT);
        }
    }
}

// The exact top k of a row, from its logits alone, by one workgroup: a radix select over the composites, ten bits at a
// time (it stops where a digit's bin is wholly inside), then the composites at or above the k-th to the row's list.
// The penalties are counted again chunk by chunk. Returns the list's length. For rows with thousands of equal logits at
// the bound, and rows whose segments gave up waiting.
template <bool CAP>
__device__ __forceinline__ uint32_t mk_slow(const float* rowp, int V, int k, bool pen, const MkWin& win, const MkPen& pn,
                                            uint64_t* list, MkShared& s) {
    constexpr int CH = SK_LT * 16 * 4;                         // logits per chunk
    const int tid = threadIdx.x;
    uint64_t prefix = 0ull, mask = 0ull;
    uint32_t need = (uint32_t)k;
    int sh = 54;
    bool gather = false;
    if (tid == 0) s.misc[2] = 0u;
#pragma unroll 1
    for (;;) {                                                 // a pass: one digit's counts, at last the gather
        const int sft = sh < 0 ? 0 : sh;
        const uint64_t dm = sh < 0 ? 0x3FFull >> -sh : 0x3FFull;
        __syncthreads();
        *reinterpret_cast<uint4*>(&s.h.hist[4 * tid]) = make_uint4(0u, 0u, 0u, 0u);
        __syncthreads();
#pragma unroll 1
        for (int lo = 0; lo < V; lo += CH) {
            const int n = V - lo < CH ? V - lo : CH;
            if (pen) {
                __syncthreads();
                for (int i = tid; i < CH / 32; i += SK_LT) s.b.bmp[i] = 0u;
                if (pn.fp_on)
                    for (int i = tid; i < CH / 2; i += SK_LT) s.u.cnt[i] = 0u;
                __syncthreads();
#pragma unroll 1
                for (int64_t i = tid; i < win.n(); i += SK_LT) {
                    const uint32_t rel = (uint32_t)win.at(i) - (uint32_t)lo;
                    if (rel < (uint32_t)n) {
                        atomicOr(&s.b.bmp[rel >> 5], 1u << (rel & 31u));
                        if (pn.fp_on) atomicAdd(&s.u.cnt[rel >> 1], 1u << ((rel & 1u) * 16u));
                    }
                }
                __syncthreads();
            }
            slow_each(rowp + lo, n, [&](float l, int i) {
                if (CAP && pn.cap > 0.0f) l = softcap_one(l, pn.cap);
                if (pen && ((s.b.bmp[i >> 5] >> (i & 31)) & 1u))
                    l = pn.apply(l, pn.fp_on ? (s.u.cnt[i >> 1] >> ((i & 1) * 16)) & 0xFFFFu : 0u);
                const uint32_t key = key_of(l);
                const uint64_t c = comp_of(key, (uint32_t)(lo + i));
                if (key == 0u) return;
                if (gather) {
                    if ((c & mask) >= prefix) {
                        const uint32_t pos = atomicAdd(&s.misc[2], 1u);
                        if (pos < (uint32_t)MK_LCAP) st_agent(&list[pos], (c << 32) | (uint64_t)__float_as_uint(l));
                    }
                } else if ((c & mask) == prefix) {
                    atomicAdd(&s.h.hist[(uint32_t)(c >> sft) & (uint32_t)dm], 1u);
                }
            });
        }
        __syncthreads();
        if (gather) break;
        uint32_t b, above;
        if (!mk_locate(s, need, b, above)) {                   // (the first digit only) fewer than k candidates: all
            prefix = mask = 0ull;
            gather = true;
            continue;
        }
        const uint32_t in = s.h.hist[b];
        need -= above;
        prefix |= (uint64_t)b << sft;
        mask |= dm << sft;
        gather = in == need || sh < 0;                         // the whole bin is inside
        sh -= 10;
    }
    vm_drain();
    __syncthreads();
    return s.misc[2];
}

// Of the composites in registers (0: none) exactly the k largest, 0 in the place of the others, packed; there are at
// least k. A radix select as mk_slow's, for lists that mk_sort does not take. Whole workgroup.
template <int EPT>
__device__ __forceinline__ void mk_trim(uint64_t (&e)[EPT], int k, MkShared& s) {
    const int tid = threadIdx.x;
    uint64_t prefix = 0ull, mask = 0ull;
    uint32_t need = (uint32_t)k;
#pragma unroll 1
    for (int sh = 54;; sh -= 10) {
        const int sft = sh < 0 ? 0 : sh;
        const uint64_t dm = sh < 0 ? 0x3FFull >> -sh : 0x3FFull;
        __syncthreads();
        *reinterpret_cast<uint4*>(&s.h.hist[4 * tid]) = make_uint4(0u, 0u, 0u, 0u);
        __syncthreads();
#pragma unroll
        for (int q = 0; q < EPT; ++q)
            if (e[q] != 0ull && (e[q] & mask) == prefix) atomicAdd(&s.h.hist[(uint32_t)(e[q] >> sft) & (uint32_t)dm], 1u);
        __syncthreads();
        uint32_t b = 0u, above = 0u;
        (void)mk_locate(s, need, b, above);
        need -= above;
        prefix |= (uint64_t)b << sft;
        mask |= dm << sft;
        if (s.h.hist[b] == need || sh < 0) break;              // the whole bin is inside
    }
    if (tid == 0) s.misc[2] = 0u;
    __syncthreads();
#pragma unroll
    for (int q = 0; q < EPT; ++q)
        if (e[q] != 0ull && (e[q] & mask) >= prefix) s.u.m.top[atomicAdd(&s.misc[2], 1u)] = e[q];
    __syncthreads();
#pragma unroll
    for (int q = 0; q < EPT; ++q) e[q] = q * SK_LT + tid < k ? s.u.m.top[q * SK_LT + tid] : 0ull;
    __syncthreads();
}

// Sorts the ranges of s.u.m.top on the work list (s.prel: start, length; s.misc[3] of them) in place, descending: a
// counting sort over the range's span, 1024 bins at a time, entries ranked within their bin; a bin of more than MK_HEAVY
// goes back on the list (equal logits: the bins then spread their ids). Whole workgroup, after a barrier; ends with one.
constexpr uint32_t MK_HEAVY = 64;
__device__ __forceinline__ void mk_spread(MkShared& s) {
    constexpr int RPT = MK_TOP / SK_LT;
    const int tid = threadIdx.x;
#pragma unroll 1
    for (uint32_t work = s.misc[3]; work != 0u; work = s.misc[3]) {
        const int lo = s.prel[2 * work - 2], n = s.prel[2 * work - 1];
        uint64_t* t = s.u.m.top + lo;
        uint64_t e[RPT], mn = ~0ull, mx = 0ull;
        uint32_t at[RPT];
#pragma unroll
        for (int q = 0; q < RPT; ++q) {
            const int i = q * SK_LT + tid;
            e[q] = i < n ? t[i] : 0ull;
            if (i < n) {
                mn = e[q] < mn ? e[q] : mn;
                mx = e[q] > mx ? e[q] : mx;
            }
        }
        *reinterpret_cast<uint4*>(&s.h.hist[4 * tid]) = make_uint4(0u, 0u, 0u, 0u);
        mn = mk_min_u64(mn, s);
        mx = mk_max_u64(mx, s);
        if (tid == 0) s.misc[3] = work - 1u;                   // (every thread has read it)
        const int bits = 64 - __clzll((long long)((mx - mn) | 1ull)), sh = bits > 10 ? bits - 10 : 0;
#pragma unroll
        for (int q = 0; q < RPT; ++q) {
            at[q] = 0u;
            if (q * SK_LT + tid < n) {
                const uint32_t b = (uint32_t)((mx - e[q]) >> sh);
                at[q] = (b << 16) | atomicAdd(&s.h.hist[b], 1u);
            }
        }
        __syncthreads();
        const uint4 c = *reinterpret_cast<const uint4*>(&s.h.hist[4 * tid]);
        uint32_t tot;
        const uint32_t o0 = mk_excl_u32(c.x + c.y + c.z + c.w, s, tot), o1 = o0 + c.x, o2 = o1 + c.y, o3 = o2 + c.z;
        *reinterpret_cast<uint4*>(&s.h.hist[4 * tid]) = make_uint4(o0, o1, o2, o3);
        auto again = [&](uint32_t o, uint32_t m) {
            if (m > MK_HEAVY) {
                const uint32_t w = atomicAdd(&s.misc[3], 1u);
                s.prel[2 * w] = (uint16_t)(lo + (int)o);
                s.prel[2 * w + 1] = (uint16_t)m;
            }
        };
        again(o0, c.x); again(o1, c.y); again(o2, c.z); again(o3, c.w);
        __syncthreads();
#pragma unroll
        for (int q = 0; q < RPT; ++q)
            if (q * SK_LT + tid < n) t[s.h.hist[at[q] >> 16] + (at[q] & 0xFFFFu)] = e[q];
        __syncthreads();
#pragma unroll
        for (int q = 0; q < RPT; ++q) {
            const int i = q * SK_LT + tid;
            at[q] = 0u;
            if (i < n) {
                e[q] = t[i];
                const uint32_t b = (uint32_t)((mx - e[q]) >> sh);
                const uint32_t b0 = s.h.hist[b], b1 = b < (uint32_t)MK_H - 1u ? s.h.hist[b + 1] : (uint32_t)n;
                uint32_t x = b0;
                if (b1 - b0 > MK_HEAVY) x = (uint32_t)i;
                else
                    for (uint32_t j = b0; j < b1; ++j) x += t[j] > e[q] ? 1u : 0u;
                at[q] = x;
            }
        }
        __syncthreads();
#pragma unroll
        for (int q = 0; q < RPT; ++q)
            if (q * SK_LT + tid < n) t[at[q]] = e[q];
        __syncthreads();
    }
}

// Sorts the row's list (n <= MK_LCAP composites in registers, 0: none) into s.u.m.top[0, min(n, k)), descending: a
// counting sort over the span of the composites, of which only the bins that hold the first k are placed; entries rank
// themselves within their bin, and bins of many entries (equal logits) are spread further first (ranked at once, rows of
// logits rounded to whole numbers took 120 us: 32 rows of 262144, k 200; now 31). Whole workgroup.
// In two parts (mk_sort_end does not depend on EPT: one copy of it for the kernel's instruction cache).
struct MkSorted {
    uint64_t cmx;                          // the largest composite; the bins' shift; entries placed, -1: none, as the bins
                                           // that hold the first k have more than MK_TOP (hundreds of ties at the k-th)
    int sh, m;
};
template <int EPT>
__device__ __forceinline__ MkSorted mk_sort(const uint64_t (&v)[EPT], int n, int k, MkShared& s) {
    const int tid = threadIdx.x;
    uint64_t cmn = ~0ull, cmx = 0ull;
#pragma unroll
    for (int q = 0; q < EPT; ++q) {
        if (q * SK_LT + tid < n) {
            cmn = v[q] < cmn ? v[q] : cmn;
            cmx = v[q] > cmx ? v[q] : cmx;
        }
    }
    for (int i = tid; i < MK_BINS; i += SK_LT) s.u.m.bins[i] = 0u;
    if (tid == 0) s.misc[3] = 0u;                              // bins to spread
    cmn = mk_min_u64(cmn, s);
    cmx = mk_max_u64(cmx, s);
    const uint64_t span = cmx - cmn;
    const int lz = span ? __clzll((long long)span) : 64;
    const int sh = 64 - lz > 11 ? 64 - lz - 11 : 0;
    static_assert(MK_BINS == 1 << 11, "span >> sh fits eleven bits");
    uint32_t place[EPT];                                    // bin << 16 | slot
#pragma unroll
    for (int q = 0; q < EPT; ++q) {
        place[q] = 0u;
        if (q * SK_LT + tid < n) {
            const uint32_t b = (uint32_t)((cmx - v[q]) >> sh);
            place[q] = (b << 16) | atomicAdd(&s.u.m.bins[b], 1u);
        }
    }
    __syncthreads();
    constexpr int BPT = MK_BINS / SK_LT;
    uint32_t c[BPT], sum = 0u;
#pragma unroll
    for (int j = 0; j < BPT; ++j) {
        c[j] = s.u.m.bins[BPT * tid + j];
        sum += c[j];
    }
    uint32_t tot;
    uint32_t off = mk_excl_u32(sum, s, tot);
#pragma unroll
    for (int j = 0; j < BPT; ++j) {
        s.u.m.bins[BPT * tid + j] = off;
        if (off < (uint32_t)k && off + c[j] >= (uint32_t)k) s.misc[4] = off + c[j];
        if (off < (uint32_t)k && c[j] > MK_HEAVY && off + c[j] <= (uint32_t)MK_TOP) {
            const uint32_t w = atomicAdd(&s.misc[3], 1u);
            s.prel[2 * w] = (uint16_t)off;
            s.prel[2 * w + 1] = (uint16_t)c[j];
        }
        off += c[j];
    }
    static_assert(2 * (MK_TOP / (int)MK_HEAVY) <= MK_PC, "the work list holds every heavy bin");
    if (tid == SK_LT - 1) s.u.m.bins[MK_BINS] = off;
    __syncthreads();
    const int m = n <= k ? n : (int)s.misc[4];
    if (m > MK_TOP) return {0ull, 0, -1};
#pragma unroll
    for (int q = 0; q < EPT; ++q) {
        if (q * SK_LT + tid < n) {
            const uint32_t pos = s.u.m.bins[place[q] >> 16] + (place[q] & 0xFFFFu);
            if (pos < (uint32_t)m) s.u.m.top[pos] = v[q];
        }
    }
    __syncthreads();
    return {cmx, sh, m};
}
__device__ __forceinline__ void mk_sort_end(const MkSorted& o, int k, MkShared& s) {
    constexpr int RPT = MK_TOP / SK_LT;
    const int tid = threadIdx.x, m = o.m;
    if (s.misc[3] != 0u) mk_spread(s);
    uint64_t e[RPT];
    uint32_t r[RPT];
#pragma unroll
    for (int q = 0; q < RPT; ++q) {
        const int i = q * SK_LT + tid;
        e[q] = 0ull;
        r[q] = 0xFFFFFFFFu;
        if (i < m) {
            e[q] = s.u.m.top[i];
            const uint32_t b = (uint32_t)((o.cmx - e[q]) >> o.sh);
            const uint32_t lo = s.u.m.bins[b], hi = s.u.m.bins[b + 1];
            uint32_t x = lo;
            if (hi - lo > MK_HEAVY) x = (uint32_t)i;           // (spread: in place already)
            else
                for (uint32_t j = lo; j < hi; ++j) x += s.u.m.top[j] > e[q] ? 1u : 0u;
            r[q] = x;
        }
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < RPT; ++q)
        if (r[q] < (uint32_t)k) s.u.m.top[r[q]] = e[q];
    __syncthreads();
}

// Softmax at temperature, min-p, top-p and the draw (sampler.cpp:37-49) over the k <= MK_K sorted candidates in
// s.u.w.top; the optional candidate outputs. Masses are taken strided, prefixes over ceil(k / SK_LT) neighbours per
// thread. Whole workgroup; the results are uniform.
__device__ __forceinline__ void mk_softmax(const SkArgs& a, const fs_row_params& p, int row, int k, double u, MkShared& s,
                                           int& tok, int& keep) {
    const int tid = threadIdx.x, per = (k + SK_LT - 1) / SK_LT, i0 = tid * per;
    const int i1 = i0 + per < k ? i0 + per : k;
    const uint64_t* top = s.u.w.top;
    double* E = s.u.w.e;
    const float mx = val_of(comp_key(top[0]));
    const double Td = (double)p.temperature;
    double run = 0.0, sum;
#pragma unroll 1
    for (int i = tid; i < k; i += SK_LT) {
        const float d = val_of(comp_key(top[i])) - mx;         // fp32 subtraction, as ferro
        const double m = exp((double)d / Td);
        E[i] = m;
        run += m;
    }
    (void)mk_excl_f64(run, s, sum);                            // (its barriers publish E)
    run = 0.0;
    uint64_t last = 0ull;                                      // min-p: 1 + the last index not below pr[0] * min_p
    const double thr = (1.0 / sum) * (double)p.min_p;
#pragma unroll 1
    for (int i = i0; i < i1; ++i) {
        const double pr = E[i] / sum;
        E[i] = pr;
        run += pr;
        if (!(pr < thr)) last = (uint64_t)(i + 1);
    }
    int keep_m = k;
    if (p.min_p > 0.0f) {
        last = mk_max_u64(last, s);
        keep_m = last > 1ull ? (int)last : 1;
    }
    double all;
    const double off = mk_excl_f64(run, s, all);
    keep = keep_m;
    if (p.top_p < 1.0f) {
        uint64_t first = ~0ull;
        run = 0.0;
#pragma unroll 1
        for (int i = i0; i < i1; ++i) {
            run += E[i];
            if (first == ~0ull && i < keep_m && run + off >= (double)p.top_p) first = (uint64_t)i;
        }
        first = mk_min_u64(first, s);
        if (first != ~0ull) keep = (int)first + 1 < keep_m ? (int)first + 1 : keep_m;
        if (keep < 1) keep = 1;
    }
    if (i0 < keep && keep <= i0 + per) {                       // tot: the kept prefix's sum
        run = 0.0;
        for (int i = i0; i < keep; ++i) run += E[i];
        s.dmisc = run + off;
    }
    __syncthreads();
    const double rr = u * s.dmisc + 0.0;
    uint64_t hit = ~0ull;
    run = 0.0;
#pragma unroll 1
    for (int i = i0; i < i1; ++i) {
        run += E[i];
        if (hit == ~0ull && i < keep && rr <= run + off) hit = (uint64_t)i;
    }
    hit = mk_min_u64(hit, s);
    tok = (int)comp_id(top[hit == ~0ull ? keep - 1 : (int)hit]);
    if (a.mode != MODE_VERIFY) {
        const int m = k < a.kcap ? k : a.kcap;
        for (int i = tid; i < m; i += SK_LT) {
            if (a.cand_ids) a.cand_ids[(int64_t)row * a.kcap + i] = (int32_t)comp_id(top[i]);
            if (a.cand_probs) a.cand_probs[(int64_t)row * a.kcap + i] = E[i];
        }
    }
}

// ---- every token a candidate (top_k = 0: k = V)
__device__ __forceinline__ double ak_mass(float x, float mx, double Td) { return exp((double)(x - mx) / Td); }

// A row's segments meet: arrive, then wait (bounded) for `target` arrivals. What the caller published is drained first.
// Whole workgroup; returns false when the row gave up.
__device__ __forceinline__ bool mk_meet(uint32_t* ctr, uint32_t target, uint32_t spins_max, MkShared& s) {
    vm_drain();
    __syncthreads();
    if (threadIdx.x == 0) {
        __hip_atomic_fetch_add(ctr, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        uint32_t ok = 1u, spins = 0u;
        for (;;) {
            const uint32_t c = __hip_atomic_fetch_add(ctr, 0x10000u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
            if ((c & 0xFFFFu) >= target && spins_max != 0u) break;
            if (++spins >= spins_max) { ok = 0u; break; }
            __builtin_amdgcn_s_sleep(1);
        }
        s.misc[5] = ok;
        if (!ok) __hip_atomic_fetch_or(ctr + 34, 2u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    }
    __syncthreads();
    return s.misc[5] != 0u;
}

// The bin that holds the target-th unit of the row's mass, and the mass before it: cum (LDS) holds the mass up to and
// with bins 8t .. 8t + 7, rm (LDS) the bins. Each wave finds it by itself, the same in all (no barrier); false when the row's
// mass does not reach the target.
__device__ __forceinline__ bool ak_locate(const uint64_t* cum, const uint64_t* rm, uint64_t target, int& bin,
                                          uint64_t& before) {
    const int lane = lane_id();
    if (target == 0ull) target = 1ull;
    const uint64_t m4 = __ballot(cum[4 * lane + 3] >= target);
    if (m4 == 0ull) return false;
    const int g4 = 4 * (__ffsll((unsigned long long)m4) - 1);  // four groups of eight bins
    const uint64_t m1 = __ballot(lane < 4 && cum[g4 + (lane & 3)] >= target);
    const int g = g4 + __ffsll((unsigned long long)m1) - 1;
    const uint64_t at = g > 0 ? cum[g - 1] : 0ull;
    uint64_t h = lane < 8 ? rm[8 * g + lane] : 0ull, inc = h;
#pragma unroll
    for (int o = 1; o < 8; o <<= 1) {
        const uint64_t y = __shfl_up(inc, o);
        if (lane >= o) inc += y;
    }
    const int j = __ffsll((unsigned long long)__ballot(lane < 8 && at + inc >= target)) - 1;
    bin = 8 * g + j;
    before = at + read_lane(inc, j) - read_lane(h, j);
    return true;
}

// The first of the n sorted candidates in s.u.w.top at which above + the masses so far reach the target, -1 when they do
// not; *cum: the sum there. COUNTED: each stands for as many equal ones as its low 16 bits say. Whole workgroup.
template <bool COUNTED>
__device__ __forceinline__ int ak_walk(int n, double above, double target, float mx, double Td, MkShared& s, double& cum) {
    const int tid = threadIdx.x, per = (n + SK_LT - 1) / SK_LT, i0 = tid * per, i1 = i0 + per < n ? i0 + per : n;
    double* E = s.u.w.e;
#pragma unroll 1
    for (int i = tid; i < n; i += SK_LT) {
        const uint64_t c = s.u.w.top[i];
        const double m = ak_mass(val_of(comp_key(c)), mx, Td);
        E[i] = COUNTED ? (double)((uint32_t)c & 0xFFFFu) * m : m;
    }
    __syncthreads();
    double run = 0.0, all;
#pragma unroll 1
    for (int i = i0; i < i1; ++i) run += E[i];
    const double off = mk_excl_f64(run, s, all) + above;
    uint64_t first = ~0ull;
    double at = 0.0;
    run = 0.0;
#pragma unroll 1
    for (int i = i0; i < i1; ++i) {
        run += E[i];
        if (first == ~0ull && run + off >= target) { first = (uint64_t)i; at = run + off; }
    }
    const uint64_t hit = mk_min_u64(first, s);
    if (first == hit && first != ~0ull) s.dmisc = at;
    __syncthreads();
    cum = s.dmisc;
    __syncthreads();
    return hit == ~0ull ? -1 : (int)hit;
}

// A row with every token a candidate from its logits alone, by one workgroup: extremes and the mass total in one pass,
// then for top-p's crossing and for the draw a radix select by mass over the composites, ten bits at a time. Exact, and
// slow (about 20 passes): rows whose mass no single bin narrows down (all logits equal), infinite maxima, give-ups.
template <bool CAP>
__device__ __forceinline__ void ak_slow(const float* rowp, int V, bool pen, const MkWin& win, const MkPen& pn,
                                        const fs_row_params& p, double u, MkShared& s, int& tok, int& keep) {
    constexpr int CH = SK_LT * 8 * 4;                          // logits per chunk
    const int tid = threadIdx.x;
    const double Td = (double)p.temperature;
    float mx = 0.0f;
    double S = 0.0, target = 0.0, cum = 0.0, top_cum = 0.0;
    uint64_t cmax = 0ull, cmin = ~0ull, nv = 0ull, prefix = 0ull, mask = 0ull, before = 0ull, xc = 0ull;
    int phase = 0, sh = 54;                                    // 0 extremes, 1 total, 2 top-p's select, 3 its count, 4 the draw's
    tok = 0;
    keep = 0;
#pragma unroll 1
    for (;;) {
        const int sft = sh < 0 ? 0 : sh;
        const uint64_t dm = sh < 0 ? 0x3FFull >> -sh : 0x3FFull;
        __syncthreads();
        for (int i = tid; i < MK_H; i += SK_LT) s.u.z.mass[i] = 0ull;
        __syncthreads();
        uint64_t mxc = 0ull, mnc = ~0ull, n_ = 0ull;
        double part = 0.0;
#pragma unroll 1
        for (int lo = 0; lo < V; lo += CH) {
            const int n = V - lo < CH ? V - lo : CH;
            if (pen) {
                __syncthreads();
                for (int i = tid; i < CH / 32; i += SK_LT) s.b.bmp[i] = 0u;
                if (pn.fp_on)
                    for (int i = tid; i < CH / 2; i += SK_LT) s.u.z.cnt[i] = 0u;
                __syncthreads();
#pragma unroll 1
                for (int64_t i = tid; i < win.n(); i += SK_LT) {
                    const uint32_t rel = (uint32_t)win.at(i) - (uint32_t)lo;
                    if (rel < (uint32_t)n) {
                        atomicOr(&s.b.bmp[rel >> 5], 1u << (rel & 31u));
                        if (pn.fp_on) atomicAdd(&s.u.z.cnt[rel >> 1], 1u << ((rel & 1u) * 16u));
                    }
                }
                __syncthreads();
            }
            slow_each(rowp + lo, n, [&](float l, int i) {
                if (CAP && pn.cap > 0.0f) l = softcap_one(l, pn.cap);
                if (pen && ((s.b.bmp[i >> 5] >> (i & 31)) & 1u))
                    l = pn.apply(l, pn.fp_on ? (s.u.z.cnt[i >> 1] >> ((i & 1) * 16)) & 0xFFFFu : 0u);
                const uint32_t key = key_of(l);
                if (key == 0u) return;
                const uint64_t c = comp_of(key, (uint32_t)(lo + i));
                if (phase == 0) {
                    mxc = c > mxc ? c : mxc;
                    mnc = c < mnc ? c : mnc;
                    ++n_;
                } else if (phase == 3) {
                    n_ += c >= xc ? 1ull : 0ull;
                } else {
                    const double m = ak_mass(l, mx, Td);
                    if (phase == 1) part += m;
                    else if ((c & mask) == prefix)
                        atomicAdd(reinterpret_cast<unsigned long long*>(&s.u.z.mass[(uint32_t)(c >> sft) & (uint32_t)dm]),
                                  (unsigned long long)(m * AK_FX + 0.5));
                }
            });
        }
        __syncthreads();
        if (phase == 0) {
            cmax = mk_max_u64(mxc, s);
            cmin = mk_min_u64(mnc, s);
            nv = mk_reduce_u64(n_, s, [](uint64_t x, uint64_t y) { return x + y; });
            if (nv == 0ull) return;                            // no number in the row: token 0, nothing kept
            mx = val_of(comp_key(cmax));
            keep = (int)nv;
            phase = 1;
            continue;
        }
        if (phase == 1) {
            (void)mk_excl_f64(part, s, S);
            if (S != S) {                                      // an infinite maximum: nothing is cut, and the draw falls
                tok = (int)comp_id(cmin);                      // through to the last candidate (sampler.cpp:43-49)
                return;
            }
            cum = S;
            phase = p.top_p < 1.0f ? 2 : 4;
            target = phase == 2 ? (double)p.top_p * S : u * S;
            continue;
        }
        if (phase == 3) {
            keep = (int)mk_reduce_u64(n_, s, [](uint64_t x, uint64_t y) { return x + y; });
            phase = 4;
            target = u * top_cum;
            prefix = mask = before = 0ull;
            sh = 54;
            continue;
        }
        // the digit's bin, from the top: thread t sums bins 1023 - 4t .. 1020 - 4t
        uint64_t h[4], mine = 0ull;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            h[j] = s.u.z.mass[MK_H - 1 - 4 * tid - j];
            mine += h[j];
        }
        uint64_t inc = mine;
#pragma unroll
        for (int o = 1; o < WAVE; o <<= 1) {
            const uint64_t y = __shfl_up(inc, o);
            if (lane_id() >= o) inc += y;
        }
        if (lane_id() == WAVE - 1) s.w64[tid / WAVE] = inc;
        __syncthreads();
        uint64_t ex = before + inc - mine;
#pragma unroll
        for (int w = 0; w < SK_NW; ++w) ex += w < tid / WAVE ? s.w64[w] : 0ull;
        uint64_t want = (uint64_t)(target * AK_FX);
        want = want ? want : 1ull;
        if (tid == 0) s.umisc[0] = ~0ull;
        __syncthreads();
        if (ex < want && ex + mine >= want) {
            uint64_t b = ex;
            int at = 0;
#pragma unroll
            for (int j = 0; j < 4; ++j)
                if (b + h[j] < want && at == j) { b += h[j]; at = j + 1; }
            s.umisc[0] = (uint64_t)(MK_H - 1 - 4 * tid - at);
            s.umisc[1] = b;
        }
        __syncthreads();
        const bool none = s.umisc[0] == ~0ull;                 // past the last candidate (the sums' rounding)
        if (!none) {
            prefix |= s.umisc[0] << sft;
            mask |= dm << sft;
            before = s.umisc[1];
            sh -= 10;
            if (sh > -10) continue;
        }
        const uint64_t c = none ? (phase == 2 || xc == 0ull ? cmin : xc) : prefix;
        if (phase == 2) {
            xc = c;
            top_cum = none ? cum : (double)before / AK_FX + ak_mass(val_of(comp_key(c)), mx, Td);
            phase = 3;
            continue;
        }
        tok = (int)comp_id(xc != 0ull && c < xc ? xc : c);
        return;
    }
}

// What a row's segments agree on: the maximum, the mass total S, the draw; top-p's crossing bin bc with the mass above it
// (cut), the bins d0 .. d1 that hold the draw; plain: nothing to search (no number, an infinite maximum, all logits equal).
struct AkRow {
    float mx;
    uint32_t nv;
    double S, u, above_c, above_d;
    int bc, d0, d1;
    bool cut, plain;
    float scale;                           // bins per unit below mx; 0 with plain: one value
    bool tail;                             // the bins end above the row's minimum
};
// One segment of such a row: extremes, meet, masses into the row's 2048 bins (linear in the logit from the row's maximum
// down to its minimum, or 32 temperatures below: about 500 logits in the fullest bin of a normal row of 262144 whatever
// its width), meet, and the logits of the bins that top-p's crossing and the draw fall in to the row's lists. The logits
// stay in registers throughout. Returns false when the row gave up.
template <int NL, bool CAP, class P, class E>
__device__ __forceinline__ bool ak_segment(float (&v)[NL][4], const MkArgs& mk, const fs_row_params& p, int row, int seg,
                                           int nseg, int seg_lo, uint32_t* ctr, uint64_t* list, P penalise, E pen_at,
                                           uint32_t nf, double u, AkRow& r, MkShared& s) {
    const int tid = threadIdx.x, lane = lane_id(), w = tid / WAVE;
    const double Td = (double)p.temperature, inv = 1.0 / Td;
    const float invf = 1.0f / p.temperature;
    r.u = u;
    const double2 pow2 = reinterpret_cast<const double2*>(exp_pow2)[lane];   // (it arrives behind the meeting)
    penalise();
    if (CAP && p.softcap > 0.0f) {
#pragma unroll
        for (int q = 0; q < NL; ++q) softcap_vals(v[q], p.softcap);
    }
    float hi = __builtin_nanf(""), lo = hi;                    // (fmaxf and fminf drop NaN)
    uint32_t n = NL * 4;                                       // the lane's numbers
    bool nans = false;
#pragma unroll
    for (int q = 0; q < NL; ++q) {
        hi = fmaxf(hi, fmaxf(fmaxf(v[q][0], v[q][1]), fmaxf(v[q][2], v[q][3])));
        lo = fminf(lo, fminf(fminf(v[q][0], v[q][1]), fminf(v[q][2], v[q][3])));
        nans |= __builtin_isunordered(v[q][0], v[q][1]) || __builtin_isunordered(v[q][2], v[q][3]);
    }
    if (__ballot(nans) != 0ull) {
        n = 0u;
#pragma unroll
        for (int q = 0; q < NL; ++q)
#pragma unroll
            for (int c = 0; c < 4; ++c) n += v[q][c] == v[q][c] ? 1u : 0u;
    }
    for (uint32_t i = (uint32_t)lane; i < nf; i += WAVE) {
        const float x = __uint_as_float((uint32_t)pen_at(i));
        hi = fmaxf(hi, x);
        lo = fminf(lo, x);
        n += x == x ? 1u : 0u;
    }
    auto add_u = [](uint32_t x, uint32_t y) { return x + y; };
    auto add_f = [](float x, float y) { return x + y; };
    auto add_d = [](double x, double y) { return x + y; };
    uint32_t kx = wave_max(key_of(hi)), kn = wave_min(lo == lo ? key_of(lo) : 0xFFFFFFFFu);
    // A minimum far down (masked tokens) would spread the bins over a range without logits: the wave's minimum is then that
    // of its logits less than AK_DEPTH temperatures below its maximum; the others are none of the row's bins' either. (32
    // rows of 262144 N(0, 2) logits at temperature 3, one of a hundred at -inf: 6640 us, thousands per bin; now 54. Not
    // for rows with tails, which spread over the bins anyway, where the second look cost 2 us of 36: the minimum is very
    // far down, or most lanes' maxima are near the wave's.)
    bool cut = false;
    const float low = val_of(kx) - AK_DEPTH * p.temperature;
    if (kx > 0x007FFFFFu && kn < kx && val_of(kn) < low &&
        (val_of(kn) < val_of(kx) - 32.0f * AK_DEPTH * p.temperature ||
         __popcll(__ballot(hi > val_of(kx) - 0.5f * AK_DEPTH * p.temperature)) >= 48)) {
        auto above = [&](float x) { return x >= low ? x : __builtin_nanf(""); };
        lo = __builtin_nanf("");
#pragma unroll
        for (int q = 0; q < NL; ++q)
            lo = fminf(lo, fminf(fminf(above(v[q][0]), above(v[q][1])), fminf(above(v[q][2]), above(v[q][3]))));
        for (uint32_t i = (uint32_t)lane; i < nf; i += WAVE) lo = fminf(lo, above(__uint_as_float((uint32_t)pen_at(i))));
        kn = wave_min(lo == lo ? key_of(lo) : 0xFFFFFFFFu);
        cut = true;
    }
    n = wave_allreduce(n, add_u);
    // two 128-byte lines per segment, one per meeting (a line is read by others only after the meeting it is written for)
    uint64_t* line = reinterpret_cast<uint64_t*>(mk.qk) + ((int64_t)row * nseg) * 32;
    // a bound of the wave's mass, relative to its maximum: its lane maxima's masses, times the most logits a lane has
    const float wm = kx > 0x007FFFFFu ? val_of(kx) : -__builtin_huge_valf();
    const float wb = wave_allreduce(hi > -__builtin_huge_valf() ? __expf((hi - wm) * invf) : 0.0f, add_f) *
                     (float)(NL * 4 + (nf + WAVE - 1) / WAVE);
    if (lane == 0) {
        s.w64[w] = ((uint64_t)kx << 32) | kn;
        s.w32[w] = n | (cut ? 0x80000000u : 0u);
        line[seg * 32 + 2 + w] = ((uint64_t)__float_as_uint(wm) << 32) | __float_as_uint(wb);
    }
    __syncthreads();
    if (tid == 0) {
#pragma unroll
        for (int q = 1; q < SK_NW; ++q) {
            const uint32_t a = (uint32_t)(s.w64[q] >> 32), b = (uint32_t)s.w64[q];
            kx = a > kx ? a : kx;
            kn = b < kn ? b : kn;
            n += s.w32[q] & 0x7FFFFFFFu;
            cut |= (s.w32[q] & 0x80000000u) != 0u;
        }
        line[seg * 32] = ((uint64_t)kx << 32) | kn;
        line[seg * 32 + 1] = n | ((uint64_t)cut << 32);
    }
    if (!mk_meet(ctr, (uint32_t)nseg, mk.spins, s)) return false;
    SK_MARK(2);
    if (tid < 64) s.h.pow2[tid] = pow2;                        // (the barrier before the masses publishes it)
    uint64_t we[SK_NW];
    {
        const uint64_t e = lane < nseg ? line[lane * 32] : 0xFFFFFFFFull;
#pragma unroll
        for (int q = 0; q < SK_NW; ++q) we[q] = lane < nseg ? line[lane * 32 + 2 + q] : 0xFF800000ull << 32;
        const uint64_t c = lane < nseg ? line[lane * 32 + 1] : 0ull;
        r.nv = wave_allreduce((uint32_t)c, add_u);
        cut = __ballot(c >> 32 != 0ull) != 0ull;
        kx = wave_max((uint32_t)(e >> 32));
        kn = wave_min((uint32_t)e);
    }
    const float mx = val_of(kx), mn = val_of(kn);
    r.mx = mx;
    // The bins' fixed-point scale, a power of two: the largest at which the row's mass fits 63 bits, by the segments' bounds
    // (one per cent for their roundings), and at most 2^52 (a mass is <= 1). A spiky row (bound < 2048) sums its masses to
    // 2^-53, as fp64 does; the flattest row the layout takes (262144 equal logits) to 2^-45.
    float bound = 0.0f;
#pragma unroll
    for (int q = 0; q < SK_NW; ++q) {
        const float x = __uint_as_float((uint32_t)(we[q] >> 32));
        if (x > -__builtin_huge_valf()) bound += __uint_as_float((uint32_t)we[q]) * __expf((x - mx) * invf);
    }
    bound = wave_allreduce(bound, add_f) * 1.01f;
    const int be = (int)((__float_as_uint(bound) >> 23) & 255u) - 126;          // bound < 2^be
    const int fxe = __builtin_amdgcn_readfirstlane(63 - be < 52 ? 63 - be : 52);
    const double fx = __builtin_ldexp(1.0, fxe), ifx = __builtin_ldexp(1.0, -fxe);
    // (cut: the lowest in the last bin, whatever its place's rounding; one value and masked tokens: all in the first bin)
    float depth = (mx - mn) * invf * (cut ? 1.0001f : 1.0f);
    const bool tail = cut || !(depth < AK_DEPTH);
    depth = depth < AK_DEPTH && !(cut && !(mn < mx)) ? depth : AK_DEPTH;
    const float scale = (float)AK_BINS / (depth * p.temperature);
    r.scale = cut || mn < mx || !(mx < __builtin_huge_valf()) || !(mx > -__builtin_huge_valf()) ? scale : 0.0f;
    r.tail = tail;
    r.plain = r.nv == 0u || !(mx < __builtin_huge_valf()) || !(mx > -__builtin_huge_valf()) || !(cut || mn < mx) ||
              !(scale > 0.0f) || !(scale < __builtin_huge_valf());
    if (r.plain) return true;                                  // uniform over the row
    for (int i = tid; i < AK_BINS / 2; i += SK_LT) reinterpret_cast<ulonglong2*>(s.u.a.mass)[i] = make_ulonglong2(0ull, 0ull);
    __syncthreads();
    // a logit's place below the maximum, in bins, and its bin (AK_BINS: none), the same function of its value in both
    // passes; it never falls as the logit falls (NaN: not a candidate)
    auto place_of = [&](float x) { return (mx - x) * scale; };
    auto bin_at = [&](float t) {
        const int b = (int)fminf(t, (float)AK_BINS);
        return t == t ? (tail ? b : (b < AK_BINS ? b : AK_BINS - 1)) : AK_BINS;
    };
    auto bin_of = [&](float x) { return bin_at(place_of(x)); };
    // Sixteen logits of the segment at a time, taken from the registers by a uniform index: the bodies below are not
    // repeated 64 times (unrolled, the kernel outgrew the instruction cache and its registers: 69 us on the nucleus rows)
    // (by masks: the compiler turns selects between array elements into an array in memory)
    auto pick16 = [&](float (&x)[4][4], int h) {
        uint32_t m[NL / 4];
#pragma unroll
        for (int g = 0; g < NL / 4; ++g) m[g] = (uint32_t)__builtin_amdgcn_readfirstlane(h == g ? -1 : 0);
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                uint32_t y = __float_as_uint(v[q][c]) & m[0];
#pragma unroll
                for (int g = 1; g < NL / 4; ++g) y |= __float_as_uint(v[4 * g + q][c]) & m[g];
                x[q][c] = __uint_as_float(y);
            }
    };
    // the groups of sixteen in which some lane of the wave has a logit at or above x
    auto groups_above = [&](float x) {
        uint32_t m = 0u;
#pragma unroll
        for (int h = 0; h < NL / 4; ++h) {
            float g = __builtin_nanf("");
#pragma unroll
            for (int q = 0; q < 4; ++q)
                g = fmaxf(g, fmaxf(fmaxf(v[4 * h + q][0], v[4 * h + q][1]), fmaxf(v[4 * h + q][2], v[4 * h + q][3])));
            m |= __ballot(g >= x) != 0ull ? 1u << h : 0u;
        }
        return (uint32_t)__builtin_amdgcn_readfirstlane((int)m);
    };
    // the value `bins` bins below the maximum, a little lower (the place's roundings are below 1e-6 of it)
    auto value_at = [&](float bins) { return mx - bins * 1.00001f / scale - fabsf(mx) * 1e-6f; };
    double part = 0.0;
    float rest = 0.0f;                                         // masses below e^-32 (see the fused kernel's large rows)
    const float faint = (float)AK_BINS * (104.0f / depth);     // from here on expf is 0
    auto add = [&](float x, int b) {
        if (b < AK_BINS) {
            const double d = (double)(x - mx);                 // fp32 subtraction, as ferro; then d / Td, correctly rounded
            double z = d * inv;
            z = __builtin_fma(__builtin_fma(-z, Td, d), inv, z);
            const double m = exp_table(z, s.h.pow2);
            part += m;
            const uint64_t f = (uint64_t)__double_as_longlong(__builtin_fma(m, fx, 0x1p52)) - 0x4330000000000000ull;
            atomicAdd(reinterpret_cast<unsigned long long*>(&s.u.a.mass[b]), (unsigned long long)f);
        } else if (x == x) {
            rest += __expf((x - mx) * invf);
        }
    };
#pragma unroll 1
    for (uint32_t todo = groups_above(value_at(faint)); todo != 0u; todo &= todo - 1u) {
        const int h = __ffs((int)todo) - 1;
        float x[4][4];
        pick16(x, h);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            float at[4];
#pragma unroll
            for (int c = 0; c < 4; ++c) at[c] = place_of(x[q][c]);
            const float first = fminf(fminf(at[0], at[1]), fminf(at[2], at[3]));
            if (__ballot(first < (tail ? (float)AK_BINS : __builtin_huge_valf())) != 0ull) {
#pragma unroll
                for (int c = 0; c < 4; ++c) add(x[q][c], bin_at(at[c]));
            } else if (__ballot(first < faint) != 0ull) {
#pragma unroll
                for (int c = 0; c < 4; ++c) rest += x[q][c] == x[q][c] ? __expf((x[q][c] - mx) * invf) : 0.0f;
            }
        }
    }
    for (uint32_t i = (uint32_t)lane; i < nf; i += WAVE) {
        const float x = __uint_as_float((uint32_t)pen_at(i));
        add(x, bin_of(x));
    }
    SK_MARK(3);
    double sum;
    (void)mk_excl_f64(part + (double)rest, s, sum);            // (its barriers complete the bins)
    uint64_t* rm = mk.mass + (int64_t)row * AK_BINS;
#pragma unroll
    for (int j = 0; j < AK_BINS / SK_LT; ++j) {
        const uint64_t h = s.u.a.mass[j * SK_LT + tid];
        if (h != 0ull) __hip_atomic_fetch_add(rm + j * SK_LT + tid, h, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    }
    if (tid == 0) line[seg * 32 + 16] = (uint64_t)__double_as_longlong(sum);
    if (!mk_meet(ctr, 2u * (uint32_t)nseg, mk.spins, s)) return false;
    SK_MARK(4);
    r.S = wave_allreduce(lane < nseg ? __longlong_as_double((long long)line[lane * 32 + 16]) : 0.0, add_d);
    {
        uint64_t mine = 0ull;
#pragma unroll
        for (int j = 0; j < 4; ++j) {                          // (the segment's own bins are spent)
            const ulonglong2 x = reinterpret_cast<const ulonglong2*>(rm)[4 * tid + j];
            reinterpret_cast<ulonglong2*>(s.u.a.mass)[4 * tid + j] = x;
            mine += x.x + x.y;
        }
        uint64_t inc = mine;
#pragma unroll
        for (int o = 1; o < WAVE; o <<= 1) {
            const uint64_t y = __shfl_up(inc, o);
            if (lane >= o) inc += y;
        }
        if (lane == WAVE - 1) s.w64[w] = inc;
        if (tid < 4) s.gn[tid] = 0u;
        __syncthreads();
#pragma unroll
        for (int q = 0; q < SK_NW; ++q) inc += q < w ? s.w64[q] : 0ull;
        const uint64_t *cum = s.u.a.cum, *row_mass = s.u.a.mass;
        s.u.a.cum[tid] = inc;
        __syncthreads();
        uint64_t before = 0ull;
        r.cut = p.top_p < 1.0f;
        r.bc = -1;
        bool ok = true;
        if (r.cut) {
            // top-p keeps through its crossing candidate (sampler.cpp:44), so the kept total lies in [tgt, tgt + the
            // largest mass of bin bc]: the draw's bin at both ends
            const double tgt = (double)p.top_p * r.S;
            ok = ak_locate(cum, row_mass, (uint64_t)(tgt * fx), r.bc, before);
            r.above_c = (double)before * ifx;
            const double most = exp_table(-(double)(ok ? r.bc : 0) * (double)depth * (1.0 / AK_BINS), s.h.pow2) * (1.0 + 1e-4);
            const double thi = tgt + most < r.S ? tgt + most : r.S;
            if (ok) ok = ak_locate(cum, row_mass, (uint64_t)(u * tgt * (1.0 - 1e-12) * fx), r.d0, before);
            r.above_d = (double)before * ifx;
            if (ok && !ak_locate(cum, row_mass, (uint64_t)(u * thi * (1.0 + 1e-12) * fx), r.d1, before)) r.d1 = r.bc;
            if (r.d1 > r.bc) r.d1 = r.bc;
        } else {
            ok = ak_locate(cum, row_mass, (uint64_t)(u * r.S * fx), r.d0, before);
            r.above_d = (double)before * ifx;
            r.d1 = r.d0;
        }
        r.plain = !ok;                                         // past the binned mass: the row is selected alone
        if (!ok) return true;
        __syncthreads();                                       // every wave has read the bins (the lists below take their place)
    }
    // the searched bins' logits, staged in LDS (the bins there are spent), then to the row's lists
    uint32_t above = 0u;
    auto stage = [&](float x, int b, uint32_t nid) {
        if (b == r.bc) {
            const uint32_t at = atomicAdd(&s.gn[0], 1u);
            if (at < (uint32_t)AK_STAGE) s.u.g.l[0][at] = ((uint64_t)nid << 32) | __float_as_uint(x);
        }
        if (b >= r.d0 && b <= r.d1) {
            const uint32_t at = atomicAdd(&s.gn[1], 1u);
            if (at < (uint32_t)AK_STAGE) s.u.g.l[1][at] = ((uint64_t)nid << 32) | __float_as_uint(x);
        }
    };
    const int deepest = r.bc > r.d1 ? r.bc : r.d1;
#pragma unroll 1
    for (uint32_t todo = groups_above(value_at((float)(deepest + 1))); todo != 0u; todo &= todo - 1u) {
        const int h = __ffs((int)todo) - 1;
        float x[4][4];
        pick16(x, h);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            bool any = false;
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                const int b = bin_of(x[q][c]);
                above += b < r.bc ? 1u : 0u;
                any |= b == r.bc || (b >= r.d0 && b <= r.d1);
            }
            if (__ballot(any) != 0ull) {
                const uint32_t own = ~(uint32_t)(seg_lo + ((4 * h + q) * SK_LT + tid) * 4);
#pragma unroll 1
                for (int c = 0; c < 4; ++c) {
                    const float y = c == 0 ? +x[q][0] : c == 1 ? +x[q][1] : c == 2 ? +x[q][2] : +x[q][3];
                    stage(y, bin_of(y), own - (uint32_t)c);
                }
            }
        }
    }
    for (uint32_t i = (uint32_t)lane; i < nf; i += WAVE) {
        const uint64_t e = pen_at(i);
        const float x = __uint_as_float((uint32_t)e);
        const int b = bin_of(x);
        above += b < r.bc ? 1u : 0u;
        stage(x, b, (uint32_t)(e >> 32) | 0x80000000u);
    }
    above = wave_allreduce(above, add_u);
    if (lane == 0 && above != 0u) atomicAdd(&s.gn[2], above);
    __syncthreads();
    const uint32_t n0 = s.gn[0], n1 = s.gn[1];
    if (tid == 0) {
        uint64_t at = 0ull;                                    // both lists' places in one round trip
        if ((n0 | n1) != 0u)
            at = __hip_atomic_fetch_add(reinterpret_cast<uint64_t*>(ctr + 38), ((uint64_t)n1 << 32) | n0, __ATOMIC_RELAXED,
                                        __HIP_MEMORY_SCOPE_WORKGROUP);
        s.misc[0] = (uint32_t)at;
        s.misc[1] = (uint32_t)(at >> 32);
        if (s.gn[2]) __hip_atomic_fetch_add(ctr + 37, s.gn[2], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        if (n0 > (uint32_t)AK_STAGE || n1 > (uint32_t)AK_STAGE)
            __hip_atomic_fetch_or(ctr + 34, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    }
    __syncthreads();
    const uint32_t b0 = s.misc[0], b1 = s.misc[1];
    for (uint32_t i = (uint32_t)tid; i < n0 && i < (uint32_t)AK_STAGE; i += SK_LT)
        if (b0 + i < (uint32_t)AK_LIST) list[b0 + i] = s.u.g.l[0][i];
    for (uint32_t i = (uint32_t)tid; i < n1 && i < (uint32_t)AK_STAGE; i += SK_LT)
        if (b1 + i < (uint32_t)AK_LIST) list[AK_LIST + b1 + i] = s.u.g.l[1][i];
    return true;
}

// The row's end, by its last segment: top-p's crossing and the draw located exactly in their bins' sorted logits. Returns
// false when a target lies outside its bin's exact masses (a rounding step at the edge). c0, c1: the lists' first WAVE
// entries; lists no longer than that (most are: a spiky row's bins hold a few logits) are sorted and summed in registers,
// by every wave for itself, without a barrier.
__device__ __forceinline__ bool ak_finish(const uint64_t* list, uint32_t n0, uint32_t n1, uint64_t c0, uint64_t c1,
                                          uint32_t above, const AkRow& r, const fs_row_params& p, MkShared& s, int& tok,
                                          int& keep) {
    const int tid = threadIdx.x, lane = lane_id();
    const double Td = (double)p.temperature;
    uint64_t xc = 0ull;
    double tot = r.S;
    keep = (int)r.nv;
    if (n0 <= (uint32_t)WAVE && n1 <= (uint32_t)WAVE) {
#pragma unroll 1
        for (int pass = r.cut ? 0 : 1; pass < 2; ++pass) {
            const uint32_t n = pass == 0 ? n0 : n1;
            const uint64_t c = pass == 0 ? c0 : c1;
            const uint64_t v =
                sort64<true>((uint32_t)lane < n ? ((uint64_t)key_of(__uint_as_float((uint32_t)c)) << 32) | (c >> 32) : 0ull);
            const double e = (uint32_t)lane < n ? ak_mass(val_of(comp_key(v)), r.mx, Td) : 0.0;
            const double cum = wave_scan_f64(e) + (pass == 0 ? r.above_c : r.above_d);
            const double target = pass == 0 ? (double)p.top_p * r.S : r.u * tot + 0.0;
            const uint64_t hit = __ballot((uint32_t)lane < n && cum >= target);
            if (hit == 0ull) return false;
            const int at = __ffsll((unsigned long long)hit) - 1;
            const uint64_t x = read_lane(v, at);
            if (pass == 0) {
                xc = x;
                tot = lane_f64(cum, at);
                keep = (int)above + at + 1;
            } else {
                tok = (int)comp_id(x < xc ? xc : x);
            }
        }
        return true;
    }
#pragma unroll 1
    for (int pass = r.cut ? 0 : 1; pass < 2; ++pass) {
        const int n = (int)(pass == 0 ? n0 : n1);
        if (n == 0) return false;
        constexpr int EPT = AK_LIST / SK_LT;
        auto entry = [&](int i) {
            const uint64_t c = i < n ? ld_agent(&list[pass * AK_LIST + i]) : 0ull;
            return c == 0ull ? 0ull : ((uint64_t)key_of(__uint_as_float((uint32_t)c)) << 32) | (c >> 32);
        };
        if (n <= SK_LT) {
            uint64_t* cand = s.u.m.top + MK_TOP - SK_LT;
            const uint64_t c = entry(tid);
            __syncthreads();                                   // (the first pass's lists are spent)
            cand[tid] = c;
            __syncthreads();
            sk_rank(cand, s.h.rk, n, [&](uint32_t rank, uint64_t e) { s.u.m.top[rank] = e; });
            __syncthreads();
        } else {
            uint64_t e[EPT];
#pragma unroll
            for (int q = 0; q < EPT; ++q) e[q] = entry(q * SK_LT + tid);
            __syncthreads();
            mk_sort_end(mk_sort(e, n, n, s), n, s);            // (n <= AK_LIST: they all fit)
        }
        double cum;
        const double target = pass == 0 ? (double)p.top_p * r.S : r.u * tot + 0.0;
        const int at = ak_walk<false>(n, pass == 0 ? r.above_c : r.above_d, target, r.mx, Td, s, cum);
        if (at < 0) return false;
        const uint64_t c = s.u.w.top[at];
        if (pass == 0) {
            xc = c;
            tot = cum;
            keep = (int)above + at + 1;
        } else {
            tok = (int)comp_id(c < xc ? xc : c);
        }
    }
    return true;
}

// The row's end where the searched bins hold more logits than a list takes (coarse logits: equal values share a bin; a row of
// one value; rows narrow in units of the bins, with a logit far from the others): by its last segment, from the row's
// logits. Chunk by chunk the bins' values and how often each occurs (a wave counts each value of its 64 logits at once);
// crossing and draw are located among the values, in the order of their chunks, and the draw's id in its chunk. More than
// AK_VALS values of a bin in a chunk: the bins' masses are summed again in 1024 parts of each, and the values are those of
// the parts that hold crossing and draw (32 rows of 262144 N(0, 0.05) logits and one at 10: 9510 us with ak_slow, 1460;
// 160 on the fused kernel, whose histogram is of keys). Returns false when a part holds too many, too, or a target lies
// outside. One workgroup, two passes (four with the parts): 32 rows of 262144 logits rounded to halves 10140 us with ak_slow,
// now 830 (2460 on the fused kernel).
template <bool CAP>
__device__ __forceinline__ bool ak_values(const float* rowp, int V, bool pen, const MkWin& win, const MkPen& pn, uint64_t* list,
                                          uint32_t above, const AkRow& r, const fs_row_params& p, MkShared& s, int& tok,
                                          int& keep) {
    constexpr int PT = 32, CH = SK_LT * PT;                    // logits of a thread, of a chunk
    const int tid = threadIdx.x, lane = lane_id();
    const double Td = (double)p.temperature;
    const bool one = r.plain;
    const int bc = one ? 0 : r.bc, d0 = one ? 0 : r.d0, d1 = one ? 0 : r.d1;
    const bool cut = p.top_p < 1.0f;
    const double S = one ? (double)r.nv : r.S;
    auto bin_of = [&](float x) {                               // as ak_segment's
        const float t = (r.mx - x) * r.scale;
        const int b = (int)fminf(t, (float)AK_BINS);
        return t == t ? (r.tail ? b : (b < AK_BINS ? b : AK_BINS - 1)) : AK_BINS;
    };
    // its part among those of the bins b0 .. b1 (never falls as the logit falls)
    auto part_of = [&](float x, int b0, int b1) {
        const float t = ((r.mx - x) * r.scale - (float)b0) * ((float)MK_H / (float)(b1 - b0 + 1));
        return (int)fminf(fmaxf(t, 0.0f), (float)(MK_H - 1));
    };
    bool fine = false;                                         // the parts c0 and e0 .. e1 only
    int c0 = 0, e0 = 0, e1 = 0;
    double above_c = one ? 0.0 : r.above_c, above_d = one ? 0.0 : r.above_d;
    auto in_crossing = [&](float x, int b) { return cut && b == bc && (!fine || part_of(x, bc, bc) == c0); };
    auto in_draw = [&](float x, int b) {
        if (b < d0 || b > d1) return false;
        const int q = fine ? part_of(x, d0, d1) : 0;
        return q >= e0 && q <= e1;
    };
    auto window = [&](int lo, int n) {                         // a chunk's window ids, with their counts
        for (int i = tid; i < CH / 32; i += SK_LT) s.b.bmp[i] = 0u;
        for (int i = tid; i < CH / 2; i += SK_LT) s.u.z.cnt[i] = 0u;
        __syncthreads();
#pragma unroll 1
        for (int64_t i = tid; i < win.n(); i += SK_LT) {
            const uint32_t rel = (uint32_t)win.at(i) - (uint32_t)lo;
            if (rel < (uint32_t)n) {
                atomicOr(&s.b.bmp[rel >> 5], 1u << (rel & 31u));
                atomicAdd(&s.u.z.cnt[rel >> 1], 1u << ((rel & 1u) * 16u));
            }
        }
        __syncthreads();
    };
    auto value = [&](float l, int i) {                         // i: in the chunk
        if (CAP && pn.cap > 0.0f) l = softcap_one(l, pn.cap);
        if (pen && ((s.b.bmp[i >> 5] >> (i & 31)) & 1u)) l = pn.apply(l, (s.u.z.cnt[i >> 1] >> ((i & 1) * 16)) & 0xFFFFu);
        return l;
    };
    auto put = [&](int l, uint32_t key, uint32_t n) {          // open addressing
        uint32_t h = (key * 0x9E3779B1u) >> 26;
        static_assert(AK_VALS == 1 << (32 - 26) && AK_VALS == WAVE, "the hash gives a place; a lane per place");
#pragma unroll 1
        for (int i = 0; i < AK_VALS; ++i, h = (h + 1u) & (AK_VALS - 1u)) {
            const uint32_t old = atomicCAS(&s.u.z.val[l].key[h], 0u, key);
            if (old == 0u || old == key) {
                atomicAdd(&s.u.z.val[l].cnt[h], n);
                return;
            }
        }
        s.gn[3] = 1u;
    };
    // f(final logit) for a chunk's logits, all lanes of a wave together (past the chunk: NaN), while go() holds
    auto each = [&](int lo, int n, auto go, auto f) {
#pragma unroll 1
        for (int q0 = 0; q0 < PT && go(); q0 += 8) {
            float x[8];
#pragma unroll
            for (int q = 0; q < 8; ++q) {
                const int i = (q0 + q) * SK_LT + tid;
                x[q] = i < n ? rowp[lo + i] : __builtin_nanf("");
            }
#pragma unroll 1
            for (int q = 0; q < 8; ++q) {
                float y = x[0];
#pragma unroll
                for (int t = 1; t < 8; ++t) y = q == t ? x[t] : y;
                f(value(y, (q0 + q) * SK_LT + tid));
            }
        }
    };
    // The part in which the masses, from the first on, reach the target (in units), and the units before it: wave 0 looks at
    // sixteen parts per lane. -1: they do not.
    auto locate = [&](const uint64_t* m, uint64_t target, uint64_t& before) {
        if (tid < WAVE) {
            uint64_t h = 0ull;
            for (int q = 0; q < MK_H / WAVE; ++q) h += m[lane * (MK_H / WAVE) + q];
            uint64_t inc = h;
#pragma unroll
            for (int o = 1; o < WAVE; o <<= 1) {
                const uint64_t y = __shfl_up(inc, o);
                if (lane >= o) inc += y;
            }
            if (target == 0ull) target = 1ull;
            const uint64_t hit = __ballot(inc >= target);
            if (hit == 0ull) {
                if (lane == 0) s.umisc[0] = ~0ull;
            } else if (lane == __ffsll((unsigned long long)hit) - 1) {
                uint64_t at = inc - h;
                int q = lane * (MK_H / WAVE);
                while (at + m[q] < target) at += m[q++];
                s.umisc[0] = (uint64_t)q;
                s.umisc[1] = at;
            }
        }
        __syncthreads();
        const int q = (int)s.umisc[0];
        before = s.umisc[1];
        __syncthreads();
        return q;
    };
#pragma unroll 1
    for (;;) {
        if (tid < 4) s.gn[tid] = 0u;                               // the lists' lengths; [3]: too many values
#pragma unroll 1
        for (int lo = 0, chunk = 0; lo < V && (chunk == 0 || s.gn[3] == 0u); lo += CH, ++chunk) {
            const int n = V - lo < CH ? V - lo : CH;
            __syncthreads();
            if (tid < 4 * AK_VALS) reinterpret_cast<uint32_t*>(s.u.z.val)[tid] = 0u;
            if (pen) window(lo, n);
            else __syncthreads();
            each(lo, n, [&]() { return s.gn[3] == 0u; }, [&](float y) {
                    const int b = bin_of(y);
                    const bool in_c = in_crossing(y, b), in_d = in_draw(y, b);
                    const uint32_t key = key_of(y);
#pragma unroll 1
                    for (uint64_t left = __ballot(in_c || in_d); left != 0ull;) {
                        const int first = __ffsll((unsigned long long)left) - 1;
                        const uint64_t eq = __ballot(key == read_lane(key, first)) & left;
                        if (lane == first) {
                            if (in_c) put(0, key, (uint32_t)__popcll(eq));
                            if (in_d) put(1, key, (uint32_t)__popcll(eq));
                        }
                        left &= ~eq;
                    }
            });
            __syncthreads();
            // entries: the value's key, the chunk (descending), the count. (Waves 0 and 1: a list each.)
            if (tid < 2 * WAVE) {
                const int l = tid / WAVE;
                const uint32_t key = s.u.z.val[l].key[lane];
                const uint64_t has = __ballot(key != 0u);
                const uint32_t at = s.gn[l] + (uint32_t)__popcll(has & ((1ull << lane) - 1ull));
                if (key != 0u && at < (uint32_t)AK_LIST)
                    st_agent(&list[l * AK_LIST + at],
                             ((uint64_t)key << 32) | ((uint32_t)(63 - chunk) << 16) | s.u.z.val[l].cnt[lane]);
                if (lane == 0) s.gn[l] += (uint32_t)__popcll(has);
            }
        }
        vm_drain();
        __syncthreads();
        if (s.gn[3] == 0u && s.gn[0] <= (uint32_t)AK_LIST && s.gn[1] <= (uint32_t)AK_LIST) break;
        if (fine || one) return false;
        // the masses again, in parts of the bins (in units that the row's mass is less than 2^63 of), and the crossing bin's
        // counts
        const int fxe = 62 - ilogb(S) < 52 ? 62 - ilogb(S) : 52;
        const double fx = __builtin_ldexp(1.0, fxe), ifx = __builtin_ldexp(1.0, -fxe);
        __syncthreads();
        for (int i = tid; i < 2 * MK_H; i += SK_LT) s.u.z.sub[i / MK_H][i % MK_H] = 0ull;
        *reinterpret_cast<uint4*>(&s.h.hist[4 * tid]) = make_uint4(0u, 0u, 0u, 0u);
#pragma unroll 1
        for (int lo = 0; lo < V; lo += CH) {
            const int n = V - lo < CH ? V - lo : CH;
            __syncthreads();
            if (pen) window(lo, n);
            each(lo, n, []() { return true; }, [&](float y) {
                const int b = bin_of(y);
                const bool in_c = cut && b == bc, in_d = b >= d0 && b <= d1;
                if (in_c || in_d) {
                    const unsigned long long m = (unsigned long long)(ak_mass(y, r.mx, Td) * fx + 0.5);
                    if (in_c) {
                        atomicAdd(reinterpret_cast<unsigned long long*>(&s.u.z.sub[0][part_of(y, bc, bc)]), m);
                        atomicAdd(&s.h.hist[part_of(y, bc, bc)], 1u);
                    }
                    if (in_d) atomicAdd(reinterpret_cast<unsigned long long*>(&s.u.z.sub[1][part_of(y, d0, d1)]), m);
                }
            });
        }
        __syncthreads();
        auto units = [&](double x) { return x > 0.0 ? (uint64_t)(x * fx) : 0ull; };
        uint64_t before = 0ull;
        double lo_t = r.u * S, hi_t = lo_t;                        // the draw, at both ends of the kept total
        if (cut) {
            const double tgt = (double)p.top_p * S;
            c0 = locate(s.u.z.sub[0], units(tgt - above_c), before);
            if (c0 < 0) return false;
            above_c += (double)before * ifx;
            uint32_t up = 0u;
            for (int i = tid; i < c0; i += SK_LT) up += s.h.hist[i];
            uint32_t ups;
            (void)mk_excl_u32(up, s, ups);
            above += ups;
            // (a logit of the part has at most the mass at the part's upper end)
            const double most = exp(-((double)bc + (double)c0 / MK_H) / ((double)r.scale * Td)) * (1.0 + 1e-4);
            lo_t = r.u * tgt;
            hi_t = r.u * (tgt + most < S ? tgt + most : S);
        }
        e1 = locate(s.u.z.sub[1], units(hi_t * (1.0 + 1e-12) - above_d), before);
        if (e1 < 0) e1 = MK_H - 1;
        e0 = locate(s.u.z.sub[1], units(lo_t * (1.0 - 1e-12) - above_d), before);
        if (e0 < 0) return false;
        above_d += (double)before * ifx;
        fine = true;
    }
    const uint32_t n0 = s.gn[0], n1 = s.gn[1];
    uint64_t xc = 0ull, c = 0ull;
    double tot = S;
    keep = (int)r.nv;
#pragma unroll 1
    for (int pass = cut ? 0 : 1; pass < 2; ++pass) {
        const int n = (int)(pass == 0 ? n0 : n1);
        if (n == 0) return false;
        uint64_t e[AK_LIST / SK_LT];
#pragma unroll
        for (int q = 0; q < AK_LIST / SK_LT; ++q)
            e[q] = q * SK_LT + tid < n ? ld_agent(&list[pass * AK_LIST + q * SK_LT + tid]) : 0ull;
        __syncthreads();                                       // (the first pass's entries are spent)
        mk_sort_end(mk_sort(e, n, n, s), n, s);
        double cum;
        const double target = pass == 0 ? (double)p.top_p * S : r.u * tot + 0.0;
        const int at = ak_walk<true>(n, pass == 0 ? above_c : above_d, target, r.mx, Td, s, cum);
        if (at < 0) return false;
        // the j-th of the entry's equal logits reaches the target; c becomes the entry's value and chunk above ~j
        c = s.u.w.top[at];
        const uint32_t cnt = (uint32_t)c & 0xFFFFu;
        const double m = ak_mass(val_of(comp_key(c)), r.mx, Td), from = cum - (double)cnt * m;
        const double want = ceil((target - from) / m);
        uint32_t j = want >= (double)cnt ? cnt : want > 1.0 ? (uint32_t)want : 1u;
        if (j > 1u && from + (double)(j - 1u) * m >= target) --j;
        c = (c & ~0xFFFFull) | (0xFFFFull - j);
        if (pass == 0) {
            uint64_t before = 0ull;
            for (int i = tid; i < at; i += SK_LT) before += s.u.w.top[i] & 0xFFFFull;
            before = mk_reduce_u64(before, s, [](uint64_t x, uint64_t y) { return x + y; });
            xc = c;
            tot = from + (double)j * m;
            keep = (int)above + (int)before + (int)j;
        }
    }
    if (c < xc) c = xc;
    // the id of its j-th logit
    const int lo = (63 - (int)((c >> 16) & 0xFFFFull)) * CH, n = V - lo < CH ? V - lo : CH;
    const uint32_t j = 0xFFFFu - ((uint32_t)c & 0xFFFFu);
    __syncthreads();
    if (pen) window(lo, n);
    uint32_t eq = 0u;                                          // a bit per logit of the thread, which are neighbours here
#pragma unroll 4
    for (int q = 0; q < PT; ++q) {
        const int i = tid * PT + q;
        const float y = value(i < n ? rowp[lo + i] : __builtin_nanf(""), i);
        eq |= (key_of(y) == comp_key(c) ? 1u : 0u) << q;
    }
    uint32_t all;
    uint32_t before = mk_excl_u32((uint32_t)__popc(eq), s, all);
    if (before < j && j <= before + (uint32_t)__popc(eq)) {
        while (++before < j) eq &= eq - 1u;
        s.misc[4] = (uint32_t)(lo + tid * PT + __ffs((int)eq) - 1);
    }
    __syncthreads();
    tok = (int)s.misc[4];
    return true;
}

struct MkKernargs {
    const float* logits;
    int64_t ld;
    int B, V, nseg, flags;
    const fs_row_params* params;
    const int64_t* hist_off;
    const int32_t* hist;
    MkArgs m;
};
constexpr size_t MK_ARGS_OFF = offsetof(MkKernargs, m);

// CAP: some row of the batch has a softcap. It never decreases, so the bound is taken over raw logits and the merge caps
// the list (an entry whose value is final already, a penalised one, has its id word's top bit cleared).
// ALL: some row samples with every token a candidate.
template <int NL, bool CAP, bool ALL>
__global__ __launch_bounds__(SK_LT, 4) void mid_k_kernel(const float* logits, int64_t ld, int B, int V, int nseg,
                                                         int flags, const fs_row_params* params,
                                                         const int64_t* hist_off, const int32_t* hist, MkArgs m_) {
    constexpr int SEG = SK_LT * NL * 4;
    __shared__ __align__(16) MkShared s;
    const int tid = threadIdx.x, lane = lane_id(), w = tid / WAVE;
    // a row's segments are consecutive workgroups of one index class mod XCDS: they share an XCD and its L2
    const int x = (int)(blockIdx.x % (unsigned)XCDS);
    const int j = (int)(blockIdx.x / (unsigned)XCDS);
    const int q_row = __builtin_amdgcn_readfirstlane(j / nseg);
    const int seg = j - q_row * nseg;
    const int row = x + XCDS * q_row;
    if (row >= B) return;
    SK_MARK(0);
    for (int i_ = 1; i_ < 13; ++i_) SK_TAG(i_, 0);
    SK_TAG(13, 3); SK_TAG(14, row); SK_TAG(15, seg);
    const int seg_lo = seg * SEG;
    const int n_in = V - seg_lo < SEG ? V - seg_lo : SEG;      // logits of this segment (>= 1)
    const float* rowp = logits + (int64_t)row * ld;
    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float*>(rowp + seg_lo), (short)0, ((n_in + 3) & ~3) * 4, 0x00020000);
    float v[NL][4];
    auto load = [&](int q) {
        const f32x4 t = raw_buffer_load_f32x4(rs, (q * SK_LT + tid) * 16, 0, 2);    // nontemporal: read once
        v[q][0] = t.x; v[q][1] = t.y; v[q][2] = t.z; v[q][3] = t.w;
    };
    // the first half, then the window's ids, then the rest: a wave's loads return in order, and so the bitmap is built
    // while the rest streams in (segments of 4096 logits are all requested at once: their ids come last anyway)
    constexpr int NL0 = NL > 4 ? NL / 2 : NL;
#pragma unroll
    for (int q = 0; q < NL0; ++q) load(q);
    __builtin_amdgcn_sched_barrier(0);
    // the other arguments through a pointer the compiler cannot trace (it would load some of them before the logits)
    const __attribute__((address_space(4))) char* kseg =
        (const __attribute__((address_space(4))) char*)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(kseg) : : "memory");
    const MkArgs& mk = *(const MkArgs*)(kseg + MK_ARGS_OFF);
    const SkArgs& a = mk.a;
    (void)m_;

    // the row's parameters (verification: its stream's) and its window; its first ids requested behind the logits
    int pidx = row, fed = 0;
    MkWin win = {hist, nullptr, 0, 0};
    if (flags & MK_VERIFY) {
        // the largest s with row_off[s] <= row: where it lies if every stream has as many rows, else by bisection
        int s0 = (int)((int64_t)row * a.n_streams / B), s1 = s0 + 1;
        if (ld_const(a.row_off + s0) > row || ld_const(a.row_off + s1) <= row) { s0 = 0; s1 = a.n_streams; }
        while (s1 - s0 > 1) {
            const int m = (s0 + s1) >> 1;
            if (ld_const(a.row_off + m) <= row) s0 = m; else s1 = m;
        }
        pidx = s0;
        const int64_t r0 = ld_const(a.row_off + s0);
        win.pb = a.rows + r0 + 1;
        fed = row - (int)r0;
    }
    fs_row_params p;
    {
        uint32_t pw[sizeof(fs_row_params) / 4];
        const uint32_t* src = reinterpret_cast<const uint32_t*>(params + pidx);
#pragma unroll
        for (int i = 0; i < (int)(sizeof(fs_row_params) / 4); ++i) pw[i] = ld_const(src + i);
        __builtin_memcpy(&p, pw, sizeof(p));
    }
    bool pen = false;
    MkPen pn;
    pn.rep = p.repetition_penalty; pn.fq = p.frequency_penalty; pn.pres = p.presence_penalty; pn.cap = p.softcap;
    pn.rep_on = pn.rep != 1.0f;
    pn.fp_on = pn.fq != 0.0f || pn.pres != 0.0f;
    int wid[MK_W];
#pragma unroll
    for (int r = 0; r < MK_W; ++r) wid[r] = -1;
    if (flags & SK_MAY_PEN) {
        int64_t h0 = 0, lenA = 0;
        if (hist_off && hist) {
            h0 = ld_const(hist_off + pidx);
            lenA = ld_const(hist_off + pidx + 1) - h0;
        }
        const int64_t len = lenA + fed;
        pen = (pn.rep_on || pn.fp_on) && p.repeat_last_n != 0 && len > 0;
        const int64_t b = window_begin(len, p);
        if (b >= len) pen = false;
        if (pen) {
            win.pa = hist + h0 + (b < lenA ? b : lenA);
            win.na = b < lenA ? lenA - b : 0;
            win.nb = fed - (b > lenA ? (int)(b - lenA) : 0);
            win.pb += fed - win.nb;
#pragma unroll
            for (int r = 0; r < MK_W; ++r)
                if (r * SK_LT + tid < win.na) wid[r] = win.pa[r * SK_LT + tid];
        }
    }
    const bool cp_on = (flags & SK_COPY) != 0;
    SkCopy cp = {};
    if (cp_on) cp = sk_cp_load(hist_off, hist, row, seg, nseg);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int q = NL0; q < NL; ++q) load(q);
    __builtin_amdgcn_sched_barrier(0);
    const bool greedy = p.temperature <= 0.0f || p.top_k == 1;
    const bool scan = greedy && !(CAP && pn.cap > 0.0f);       // (a capped greedy row goes the sampled rows' way, k = 1)
    const int k = greedy ? 1 : ((p.top_k > 0 && p.top_k < V) ? p.top_k : V);

    // the window's ids of this segment: a bit per logit, 64 bits per thread (its own logits), and counts
    uint32_t* ctr = mk.ctr + (int64_t)row * MK_CTR;            // [0] barrier; [32] ticket, [33] list length, [34] slow, [35] spill
    uint64_t* list = mk.list + (int64_t)row * MK_LCAP;
    uint64_t* spill = mk.spill + (int64_t)row * MK_SPILL;
    // this wave's flagged logits: nf of them, in LDS from place pb on, or in the row's spill list (far; over: it is full)
    uint32_t nf = 0u, pb = 0u;
    bool far = false, over = false;
    if (pen) {
        uint32_t m0 = 0u, m1 = 0u;
        bool ovf = false;
        for (int i = tid; i < SK_LT * 2; i += SK_LT) s.b.bmp[i] = 0u;
        if (tid == 0) s.np = 0u;
        if (pn.fp_on)
            for (int i = tid; i < SEG / 8; i += SK_LT) reinterpret_cast<uint4*>(s.u.cnt)[i] = make_uint4(0u, 0u, 0u, 0u);
        __syncthreads();
        auto set = [&](uint32_t rel) {
            const uint32_t g = rel >> 2;
            atomicOr(&s.b.bmp[(g % SK_LT) * 2 + g / (SK_LT * 8)], 1u << (4u * ((g / SK_LT) & 7u) + (rel & 3u)));
        };
        auto mark4 = [&](int i0, int i1, int i2, int i3) {     // (the counts' old values are in flight together)
            const uint32_t lo = (uint32_t)seg_lo;
            const uint32_t rel[4] = {(uint32_t)i0 - lo, (uint32_t)i1 - lo, (uint32_t)i2 - lo, (uint32_t)i3 - lo};
            const uint32_t m01 = rel[0] < rel[1] ? rel[0] : rel[1], m23 = rel[2] < rel[3] ? rel[2] : rel[3];
            if ((m01 < m23 ? m01 : m23) >= (uint32_t)n_in) return;   // (most hold no id of the segment)
            if (pn.fp_on) {
                uint32_t old[4];
#pragma unroll
                for (int c = 0; c < 4; ++c)
                    old[c] = rel[c] < (uint32_t)n_in ? atomicAdd(&s.u.cnt[rel[c] >> 1], 1u << ((rel[c] & 1u) * 16u)) : 0u;
#pragma unroll
                for (int c = 0; c < 4; ++c)
                    if (rel[c] < (uint32_t)n_in) {
                        const uint32_t had = (old[c] >> ((rel[c] & 1u) * 16u)) & 0xFFFFu;
                        ovf |= had == 0xFFFFu;
                        if (had == 0u) set(rel[c]);
                    }
            } else {
#pragma unroll
                for (int c = 0; c < 4; ++c)
                    if (rel[c] < (uint32_t)n_in) set(rel[c]);
            }
        };
#pragma unroll
        for (int r = 0; r < MK_W; ++r) asm volatile("" : "+v"(wid[r]));   // (no wait for the ids above this branch)
        static_assert(MK_W == 4, "one batch of prefetched ids");
        // batches of four ids per thread: the prefetched ones, the drafts and the ends of the rest, then the rest's 16-byte
        // blocks, four loads in flight
        const int32_t* hp = win.pa + MK_W * SK_LT;
        const int64_t n = win.na - MK_W * SK_LT;               // ids past the prefetched ones
        const int ab = (int)((0u - (unsigned)((uintptr_t)hp >> 2)) & 3u);
        const int64_t nv = n > ab ? (n - ab) >> 2 : 0;
        const int64_t rest = ab + 4 * nv;
        const int4* hv = reinterpret_cast<const int4*>(hp + ab);
        int4 w4[4];
        w4[0] = make_int4(wid[0], wid[1], wid[2], wid[3]);
        w4[1] = make_int4(tid < win.nb ? win.pb[tid] : -1, tid < ab && tid < n ? hp[tid] : -1,
                          rest + tid < n ? hp[rest + tid] : -1, SK_LT + tid < win.nb ? win.pb[SK_LT + tid] : -1);
        w4[2] = w4[3] = make_int4(-1, -1, -1, -1);
        int nr = win.nb > 0 || n > 0 ? 2 : 1;
        int64_t d0 = 2 * SK_LT;
#pragma unroll 1
        for (int64_t j0 = 0;;) {
#pragma unroll 1
            for (int r = 0; r < nr; ++r) {
                // (unary plus: selects of values, not of addresses, which would put the array in memory)
                const int i0 = r == 0 ? +w4[0].x : r == 1 ? +w4[1].x : r == 2 ? +w4[2].x : +w4[3].x;
                const int i1 = r == 0 ? +w4[0].y : r == 1 ? +w4[1].y : r == 2 ? +w4[2].y : +w4[3].y;
                const int i2 = r == 0 ? +w4[0].z : r == 1 ? +w4[1].z : r == 2 ? +w4[2].z : +w4[3].z;
                const int i3 = r == 0 ? +w4[0].w : r == 1 ? +w4[1].w : r == 2 ? +w4[2].w : +w4[3].w;
                mark4(i0, i1, i2, i3);
            }
            if (j0 < nv) {
                nr = 4;
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    w4[r] = j0 + r * SK_LT + tid < nv ? hv[j0 + r * SK_LT + tid] : make_int4(-1, -1, -1, -1);
                j0 += 4 * SK_LT;
            } else if (d0 < win.nb) {                          // (a stream of more than 512 rows)
                nr = 1;
                w4[0] = make_int4(d0 + tid < win.nb ? win.pb[d0 + tid] : -1, -1, -1, -1);
                d0 += SK_LT;
            } else {
                break;
            }
        }
        if (ovf) atomicOr(a.err, FS_DEVERR_COUNT_OVERFLOW);
        __syncthreads();
        m0 = s.b.bmp[2 * tid];
        m1 = NL > 8 ? s.b.bmp[2 * tid + 1] : 0u;
        // the flagged logits to the wave's list, and out of the registers (NaN: no comparison takes it)
        const uint32_t mine = (uint32_t)(__popc(m0) + __popc(m1));
        const uint32_t incl = wave_incl_scan_u32(mine);
        nf = (uint32_t)__builtin_amdgcn_readlane((int)incl, WAVE - 1);
        __syncthreads();                                       // every thread has read its bits
        if (nf != 0u) {
            if (lane == 0) pb = atomicAdd(&s.np, nf);
            pb = (uint32_t)__builtin_amdgcn_readfirstlane((int)pb);
            far = pb + nf > (uint32_t)MK_PC;
            if (far) {
                if (lane == 0) pb = __hip_atomic_fetch_add(ctr + 35, nf, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                pb = (uint32_t)__builtin_amdgcn_readfirstlane((int)pb);
                over = pb + nf > (uint32_t)MK_SPILL;
                if (over) nf = 0u;
            }
            uint32_t at = pb + incl - mine;
#pragma unroll
            for (int q = 0; q < NL; ++q) {
                const uint32_t nib = ((q < 8 ? m0 : m1) >> (4 * (q & 7))) & 15u;
                if (__ballot(nib != 0u) != 0ull) {
#pragma unroll
                    for (int c = 0; c < 4; ++c) {
                        if ((nib >> c) & 1u) {
                            const uint32_t rel = (uint32_t)((q * SK_LT + tid) * 4 + c);
                            if (!far) {
                                s.b.pv[at] = v[q][c];
                                s.prel[at] = (uint16_t)rel;
                            } else if (!over) {
                                spill[at] = ((uint64_t)rel << 32) | __float_as_uint(v[q][c]);
                            }
                            ++at;
                            v[q][c] = __builtin_nanf("");
                        }
                    }
                }
            }
        }
    }
    if (n_in < SEG) {                                          // past the row's end: NaN, no comparison takes it
#pragma unroll
        for (int q = 0; q < NL; ++q)
#pragma unroll
            for (int c = 0; c < 4; ++c)
                if ((q * SK_LT + tid) * 4 + c >= n_in) v[q][c] = __builtin_nanf("");
    }
    float lm = __builtin_nanf("");                             // the lane maximum (fmaxf drops NaN)
#pragma unroll
    for (int q = 0; q < NL; ++q) lm = fmaxf(lm, fmaxf(fmaxf(v[q][0], v[q][1]), fmaxf(v[q][2], v[q][3])));
    const bool capped = CAP && pn.cap > 0.0f;
    // the wave's flagged logits, penalised in place; afterwards entry i as ~id above the value (far: read past the L1)
    auto penalise = [&]() {
        if (far) vm_drain();
#pragma unroll 1
        for (uint32_t i = (uint32_t)lane; i < nf; i += WAVE) {
            const uint64_t e = far ? ld_agent(&spill[pb + i]) : 0ull;
            const uint32_t rel = far ? (uint32_t)(e >> 32) : s.prel[pb + i];
            float l = far ? __uint_as_float((uint32_t)e) : s.b.pv[pb + i];
            if (CAP && pn.cap > 0.0f) l = softcap_one(l, pn.cap);
            l = pn.apply(l, pn.fp_on ? (s.u.cnt[rel >> 1] >> ((rel & 1u) * 16u)) & 0xFFFFu : 0u);
            if (far) st_agent(&spill[pb + i], (e & 0xFFFFFFFF00000000ull) | __float_as_uint(l));
            else s.b.pv[pb + i] = l;
        }
        if (far) vm_drain();
    };
    auto pen_at = [&](uint32_t i) {
        const uint64_t e = far ? ld_agent(&spill[pb + i]) : 0ull;
        uint32_t nid = ~((uint32_t)seg_lo + (far ? (uint32_t)(e >> 32) : (uint32_t)s.prel[pb + i]));
        if (CAP && pn.cap > 0.0f) nid &= 0x7FFFFFFFu;          // (its value is capped already)
        return ((uint64_t)nid << 32) | (far ? (uint32_t)e : __float_as_uint(s.b.pv[pb + i]));
    };
    SK_MARK(1);
    const bool every = ALL && k > MK_K;                        // every token a candidate
    float tr = 0.0f, tc = 0.0f;                                // the bound: raw, capped
    float tb = 0.0f, tu = 0.0f;                                // a tied bound: its raw value, the first above its capped one
    bool go = true, tied = false;
    AkRow ak = {};
    SkDraw dr = {0.0, 0};
    if (ALL && every) {
        dr = sk_draw(a, row);
        go = ak_segment<NL, CAP>(v, mk, p, row, seg, nseg, seg_lo, ctr, list, penalise, pen_at, nf, dr.u, ak, s);
    } else if (!scan) {
        // the lane maxima, sorted in each wave, published at 16 ranks
        const uint32_t srt = sort64_desc_u32(key_of(lm));
        s.h.srt[w][lane] = srt;
        uint32_t* qk = mk.qk + (int64_t)row * nseg * (SK_NW * 16);
        if (lane < 16) qk[(seg * SK_NW + w) * 16 + lane] = s.h.srt[w][mk_rank(lane) - 1];
        SK_MARK(2);
        vm_drain();
        __syncthreads();
        if (tid == 0) __hip_atomic_fetch_add(ctr, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        penalise();                                            // (while the other segments arrive)
        if (tid == 0) {
            uint32_t ok = 1u, spins = 0u;
            for (;;) {                                         // (a poll that adds: it executes in the L2)
                const uint32_t c = __hip_atomic_fetch_add(ctr, 0x10000u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                if ((c & 0xFFFFu) >= (uint32_t)nseg && mk.spins != 0u) break;
                if (++spins >= mk.spins) { ok = 0u; break; }
                __builtin_amdgcn_s_sleep(1);
            }
            s.misc[5] = ok;
            if (!ok) __hip_atomic_fetch_or(ctr + 34, 2u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        }
        *reinterpret_cast<uint4*>(&s.h.hist[4 * tid]) = make_uint4(0u, 0u, 0u, 0u);   // (the ranks are read)
        __syncthreads();
        SK_MARK(3);
        go = s.misc[5] != 0u;
        if (go) {
            uint32_t sum, need;
            uint32_t T = mk_bound<NL == 16 ? 1 : 2>(qk, nseg, k, s, sum, need);
            // Lane maxima without ties add up to k and a few more. More than an eighth over it, and the bound is one value
            // of many logits (a masked vocabulary with fewer than k tokens allowed, coarse logits): where so many lanes
            // reach it that the row's list may overflow (half of them, or 2048), the segments count them and take the
            // first ones only. Below that the list takes them all, and is faster (32 rows of 262144 logits rounded to
            // halves, k 50: 21 us, 28 counted). The same for every segment of the row.
            const uint32_t lanes = (uint32_t)nseg * SK_LT, many = lanes < MK_LIST ? lanes / 2u : MK_LIST / 2u;
            tied = sum > (uint32_t)(k + k / 8 + 48) && sum > many;
            if (tied) T = mk_bound_exact(qk, nseg, T, need, s);
            SK_MARK(4);
            tc = T > 0x007FFFFFu ? val_of(T) : -__builtin_huge_valf();
            tr = tb = tc;
            if (CAP && pn.cap > 0.0f) {
                // tc: the capped bound; tr: a raw value that every logit whose capped value reaches tc reaches. Lane
                // l < 32 caps the value 2^l keys below the bound (lane 32 the bound): the first that falls below tc
                const uint32_t kb = T > 0x007FFFFFu ? T : 0x007FFFFFu, room = kb - 0x007FFFFFu;
                const uint32_t step = lane < 32 ? 1u << lane : 0u;
                const float c = softcap_one(val_of(room > step ? kb - step : 0x007FFFFFu + (lane < 32 ? 0u : room)), pn.cap);
                tc = room != 0u ? read_lane(c, 32) : tc;       // (no bound: every number, a penalised one below -cap too)
                const uint64_t below = __ballot(lane < 32 && c < tc);
                tr = -__builtin_huge_valf();
                if (below) {
                    const uint32_t st = 1u << (__ffsll((unsigned long long)below) - 1);
                    tr = room > st ? val_of(kb - st) : tr;
                }
                if (tied) {                                    // as tr, on the other side
                    const uint32_t up = 0xFF800000u - kb;      // (the key of inf is the highest)
                    const float h = softcap_one(val_of(kb + (up > step ? step : up)), pn.cap);
                    const uint64_t over_ = __ballot(lane < 32 && h > read_lane(c, 32));
                    tu = __builtin_nanf("");
                    if (over_) {
                        const uint32_t st = 1u << (__ffsll((unsigned long long)over_) - 1);
                        tu = val_of(kb + (up > st ? st : up));
                    }
                }
            }
        }
    }
    if (scan) {
        // the segment's first maximum (ferro's scan, sampler.cpp:19-23)
        uint64_t best = 0ull;
        if (lm == lm) {
            uint32_t first = 0u;
#pragma unroll
            for (int q = NL - 1; q >= 0; --q)
#pragma unroll
                for (int c = 3; c >= 0; --c)
                    first = v[q][c] == lm ? (uint32_t)(q * SK_LT * 4 + c) : first;
            best = comp_of(key_of(lm), (uint32_t)(seg_lo + tid * 4) + first);
        }
        penalise();
        for (uint32_t i = (uint32_t)lane; i < nf; i += WAVE) {    // and the penalised ones
            const uint64_t e = pen_at(i);
            const uint32_t key = key_of(__uint_as_float((uint32_t)e));
            const uint64_t c = ((uint64_t)key << 32) | (e >> 32);
            if (key != 0u && c > best) best = c;
        }
        best = mk_max_u64(best, s);
        if (tid == 0) list[seg] = best;
    } else if (!every) {
        uint64_t gm = 0ull;
        if (tied) {
            // Of the logits at the bound only the first can be among the row's top k: as many as the logits above it and
            // those at it in earlier segments leave of k. The segments count both and meet once more. (Every logit of a
            // tied row went to the list before, which overflowed: 32 rows of 262144 logits, 20 of them allowed, k 200:
            // 2920 us with one workgroup per row selecting it, 637 on the fused kernel, now 50.)
            // With a softcap, logits from tr up to tu have the bound's capped value: those not at the bound go to the list
            // uncounted.
            uint64_t eq = 0ull;
            uint32_t n_up = 0u;
#pragma unroll
            for (int q = 0; q < NL; ++q) {
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    gm |= (uint64_t)(v[q][c] >= tr ? 1u : 0u) << (4 * q + c);
                    eq |= (uint64_t)(v[q][c] == tb ? 1u : 0u) << (4 * q + c);
                    if (CAP) n_up += v[q][c] >= tu ? 1u : 0u;
                }
            }
            gm &= ~eq;
            if (!capped) n_up = (uint32_t)__popcll(gm);
            auto add = [](uint32_t x, uint32_t y) { return x + y; };
            const uint32_t g = wave_allreduce(n_up, add);
            if (lane == 0) s.w32[w] = g;
#pragma unroll 1
            for (int q = 0; q < NL; ++q) {                     // in the order of their ids: by q, then by wave
                const uint32_t t = wave_allreduce((uint32_t)__popc((uint32_t)(eq >> (4 * q)) & 15u), add);
                if (lane == 0) s.h.hist[q * SK_NW + w] = t;
            }
            __syncthreads();
            const uint32_t t = lane < NL * SK_NW ? s.h.hist[lane] : 0u;
            const uint32_t incl = wave_incl_scan_u32(t);
            if (tid == WAVE - 1) {
                ctr[64 + 2 * seg] = s.w32[0] + s.w32[1] + s.w32[2] + s.w32[3];
                ctr[65 + 2 * seg] = incl;
            }
            go = mk_meet(ctr, 2u * (uint32_t)nseg, mk.spins, s);
            const uint32_t above = wave_allreduce(lane < nseg ? ld_agent(ctr + 64 + 2 * lane) : 0u, add) +
                                   wave_allreduce(lane < seg ? ld_agent(ctr + 65 + 2 * lane) : 0u, add);
            const uint32_t left = above < (uint32_t)k ? (uint32_t)k - above : 0u;
#pragma unroll 1
            for (int q = 0; q < NL; ++q) {
                const uint32_t nib = (uint32_t)(eq >> (4 * q)) & 15u, n = (uint32_t)__popc(nib);
                uint32_t at = (uint32_t)__shfl((int)(incl - t), q * SK_NW + w) + wave_incl_scan_u32(n) - n;
                for (int c = 0; c < 4; ++c)
                    if ((nib >> c) & 1u) {
                        if (at < left) gm |= 1ull << (4 * q + c);
                        ++at;
                    }
            }
        }
        if (go) {
            // the logits at or above the bound to the row's list, the penalised ones against the capped bound
            uint32_t np = 0u;
            for (uint32_t i = (uint32_t)lane; i < nf; i += WAVE) np += __uint_as_float((uint32_t)pen_at(i)) >= tc ? 1u : 0u;
            if (!tied) {
#pragma unroll
                for (int q = 0; q < NL; ++q)                   // (most groups hold none)
                    if (__ballot(fmaxf(fmaxf(v[q][0], v[q][1]), fmaxf(v[q][2], v[q][3])) >= tr) != 0ull) {
#pragma unroll
                        for (int c = 0; c < 4; ++c) gm |= (uint64_t)(v[q][c] >= tr ? 1u : 0u) << (4 * q + c);
                    }
            }
            if (!tied && tr == -__builtin_huge_valf()) {
                // fewer than k lane maxima (NaN): of the logits at -inf only this wave's first k ids can be among the
                // row's top k
                uint64_t eq = 0ull;
#pragma unroll
                for (int q = 0; q < NL; ++q)
#pragma unroll
                    for (int c = 0; c < 4; ++c) eq |= (uint64_t)(v[q][c] == tr ? 1u : 0u) << (4 * q + c);
                gm &= ~eq;
                uint32_t seen = 0u;
#pragma unroll 1
                for (int q = 0; q < NL && seen < (uint32_t)k; ++q) {
                    uint32_t nib = (uint32_t)(eq >> (4 * q)) & 15u;
                    const uint32_t incl = wave_incl_scan_u32((uint32_t)__popc(nib));
                    uint32_t before = seen + incl - (uint32_t)__popc(nib);
                    for (int c = 0; c < 4; ++c)
                        if ((nib >> c) & 1u) {
                            if (before < (uint32_t)k) gm |= 1ull << (4 * q + c);
                            ++before;
                        }
                    seen += (uint32_t)__builtin_amdgcn_readlane((int)incl, WAVE - 1);
                }
            }
            const uint32_t n = (uint32_t)__popcll(gm) + np;
            const uint32_t incl = wave_incl_scan_u32(n);
            const uint32_t nw = (uint32_t)__builtin_amdgcn_readlane((int)incl, WAVE - 1);
            if (nw != 0u) {
                uint32_t base = 0u;
                if (lane == 0) base = __hip_atomic_fetch_add(ctr + 33, nw, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                base = (uint32_t)__builtin_amdgcn_readlane((int)base, 0);
                if (base + nw <= (uint32_t)MK_LCAP) {          // (else the list's length shows it)
                    uint64_t* at = list + (base + incl - n);
                    if (np != 0u)
                        for (uint32_t i = (uint32_t)lane; i < nf; i += WAVE) {
                            const uint64_t e = pen_at(i);
                            if (__uint_as_float((uint32_t)e) >= tc) *at++ = e;
                        }
#pragma unroll
                    for (int q = 0; q < NL; ++q) {
                        const uint32_t nib = (uint32_t)(gm >> (4 * q)) & 15u;
                        if (__ballot(nib != 0u) != 0ull) {
                            const uint32_t id0 = ~(uint32_t)(seg_lo + (q * SK_LT + tid) * 4);   // ~(x + c) = ~x - c
#pragma unroll
                            for (int c = 0; c < 4; ++c)
                                if ((nib >> c) & 1u) *at++ = ((uint64_t)(id0 - (uint32_t)c) << 32) | __float_as_uint(v[q][c]);
                        }
                    }
                }
            }
        }
    }
    if (over && lane == 0)                                     // too many penalised ids: the row is selected alone
        __hip_atomic_fetch_or(ctr + 34, 4u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    if (cp_on) sk_cp_store(a, cp, row, seg);
    SK_MARK(5);
    vm_drain();                                                // the candidates are in the L2
    __syncthreads();
    if (tid == 0)
        s.misc[0] = __hip_atomic_fetch_add(ctr + 32, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) ==
                    (uint32_t)nseg - 1u ? 1u : 0u;
    __syncthreads();
    SK_MARK(6);
    if (s.misc[0] == 0u) {
        SK_FLUSH();
        return;
    }
    SK_TAG(13, 4);
    // ---- the row's end, by its last segment. (The lists are read at agent scope: past this CU's L1.)
    if (!greedy && !(ALL && every)) dr = sk_draw(a, row);
    int tok = 0, keep = 1;
    // a greedy row's token (ferro keeps index 0 when its logit is NaN)
    auto greedy_end = [&](uint64_t top) {
        tok = (rowp[0] != rowp[0] || top == 0ull) ? 0 : (int)comp_id(top);
        if (lane == 0 && a.mode != MODE_VERIFY && a.kcap > 0) {
            if (a.cand_ids) a.cand_ids[(int64_t)row * a.kcap] = tok;
            if (a.cand_probs) a.cand_probs[(int64_t)row * a.kcap] = 1.0;
        }
    };
    const uint32_t slow = ld_agent(ctr + 34);                  // uniform
    uint32_t n0 = 0u, n1 = 0u, above = 0u;
    uint64_t c0 = 0ull, c1 = 0ull;
    if (ALL && every) {                                        // (one round trip with the flags)
        n0 = ld_agent(ctr + 38);
        n1 = ld_agent(ctr + 39);
        above = ld_agent(ctr + 37);
        c0 = ld_agent(&list[lane]);
        c1 = ld_agent(&list[AK_LIST + lane]);
    }
    if (scan && slow == 0u) {
        if (w != 0) return;
        greedy_end(wave_max(lane < nseg ? ld_agent(&list[lane]) : 0ull));
        if (lane == 0) {
            ctr[32] = 0u;
            ctr[35] = 0u;
        }
    } else if (ALL && every) {
        __syncthreads();
        if (tid == 0) {                                        // every segment has met and counted: left at 0
            ctr[0] = 0u;
            for (int i = 32; i < 40; ++i) ctr[i] = 0u;
            if (slow & 2u) atomicOr(a.err, FS_DEVERR_INTERNAL);
        }
        ulonglong2* rm = reinterpret_cast<ulonglong2*>(mk.mass + (int64_t)row * AK_BINS);
        for (int i = tid; i < AK_BINS / 2; i += SK_LT) rm[i] = make_ulonglong2(0ull, 0ull);
        const bool fits = n0 <= (uint32_t)AK_LIST && n1 <= (uint32_t)AK_LIST;
        bool done = false;
        if (slow == 0u && !ak.plain && fits) done = ak_finish(list, n0, n1, c0, c1, above, ak, p, s, tok, keep);
        else if ((slow & ~1u) == 0u && (!ak.plain || (ak.nv != 0u && ak.scale == 0.0f)))
            done = ak_values<CAP>(rowp, V, pen, win, pn, list, above, ak, p, s, tok, keep);
        if (!done) ak_slow<CAP>(rowp, V, pen, win, pn, p, dr.u, s, tok, keep);
        if (w != 0) return;
    } else {
        uint32_t C = ld_agent(ctr + 33);
        bool capped_list = capped;
        const bool again = slow != 0u || C > (uint32_t)MK_LCAP;   // uniform
        __syncthreads();
        if (tid == 0) {                                        // every segment has met and counted: left at 0
            ctr[0] = 0u;
            ctr[32] = 0u;
            ctr[33] = 0u;
            ctr[34] = 0u;
            ctr[35] = 0u;
            if (slow & 2u) atomicOr(a.err, FS_DEVERR_INTERNAL);
        }
        do {
            if (again) {
                C = mk_slow<CAP>(rowp, V, k, pen, win, pn, list, s);
                capped_list = false;
            }
            if (C == 0u) {                                     // every logit NaN: token 0, nothing kept
                keep = greedy ? 1 : 0;
                if (greedy && w == 0) greedy_end(0ull);
                break;
            }
            const int kk = (uint32_t)k < C ? k : (int)C;
            // the list's entries (~id above the logit's bits) as the composites ferro ranks; raw logits are capped here
            auto entry = [&](uint64_t c) {
                uint32_t nid = (uint32_t)(c >> 32);
                float l = __uint_as_float((uint32_t)c);
                if (CAP) {
                    if (capped_list && (nid & 0x80000000u)) l = softcap_one(l, pn.cap);
                    nid |= 0x80000000u;
                }
                return c == 0ull ? 0ull : ((uint64_t)key_of(l) << 32) | nid;
            };
            if (k <= WAVE && C <= (uint32_t)SK_LT) {
                uint64_t* cand = s.u.m.top;
                if ((uint32_t)tid < C) cand[tid] = entry(ld_agent(&list[tid]));
                if (tid < WAVE) cand[SK_LT + tid] = 0ull;
                __syncthreads();
                sk_rank(cand, s.h.rk, (int)C, [&](uint32_t r, uint64_t c) { if (r < (uint32_t)WAVE) cand[SK_LT + r] = c; });
                __syncthreads();
                if (w != 0) return;
                SK_MARK(7);
                if (greedy) {
                    greedy_end(read_lane(cand[SK_LT + lane], 0));
                    break;
                }
                Args fa = {};
                fa.mode = a.mode; fa.kcap = a.kcap; fa.cand_ids = a.cand_ids; fa.cand_probs = a.cand_probs;
                RowCtx rc = {};
                rc.row = row;
                rc.p = p;
                wave_softmax(fa, rc, lane < kk ? cand[SK_LT + lane] : 0ull, kk, dr.u, tok, keep);
                break;
            }
            // the list in registers, as many entries per thread as it needs
            auto sort_list = [&](auto ept) {
                constexpr int EPT = decltype(ept)::value;
                uint64_t e[EPT];
#pragma unroll
                for (int q = 0; q < EPT; ++q)
                    e[q] = (uint32_t)(q * SK_LT + tid) < C ? ld_agent(&list[q * SK_LT + tid]) : 0ull;
                if (CAP) {                                     // (a rolled loop: one copy of the cap)
#pragma unroll 1
                    for (int q = 0; q < EPT; ++q) {
                        uint64_t c = e[0];
#pragma unroll
                        for (int t = 1; t < EPT; ++t) c = q == t ? e[t] : c;
                        c = entry(c);
#pragma unroll
                        for (int t = 0; t < EPT; ++t) e[t] = q == t ? c : e[t];
                    }
                } else {
#pragma unroll
                    for (int q = 0; q < EPT; ++q) e[q] = entry(e[q]);
                }
                __syncthreads();
                MkSorted o = mk_sort(e, (int)C, k, s);
                if (EPT * SK_LT > MK_TOP && o.m < 0) {         // ties at the k-th
                    mk_trim(e, k, s);
                    o = mk_sort(e, k, k, s);
                }
                return o;
            };
            if (C <= (uint32_t)SK_LT) {
                uint64_t* cand = s.u.m.top + MK_TOP - SK_LT;
                if ((uint32_t)tid < C) cand[tid] = entry(ld_agent(&list[tid]));
                __syncthreads();
                sk_rank(cand, s.h.rk, (int)C, [&](uint32_t r, uint64_t c) { if (r < (uint32_t)k) s.u.m.top[r] = c; });
                __syncthreads();
            } else {
                const MkSorted o = C <= 4u * SK_LT ? sort_list(std::integral_constant<int, 4>{})
                                                   : sort_list(std::integral_constant<int, MK_LCAP / SK_LT>{});
                mk_sort_end(o, k, s);
            }
            SK_MARK(7);
            if (greedy) {
                if (w == 0) greedy_end(s.u.m.top[0]);
                break;
            }
            mk_softmax(a, p, row, kk, dr.u, s, tok, keep);
        } while (false);
        if (w != 0) return;
    }
    SK_TAG(9, k);
    sk_finish(a, row, pidx, !greedy, tok, keep, cp, dr.idx, &s.u.m.top[0]);
    SK_MARK(8);
    SK_FLUSH();
}

hipError_t launch_mid_k(int nl, bool capped, bool all, unsigned grid, int flags, const MkArgs& m, hipStream_t st) {
    auto go = [&](auto kern) {
        hipLaunchKernelGGL(kern, dim3(grid), dim3(SK_LT), 0, st, m.a.logits, m.a.ld, m.a.B, m.a.V, m.a.nseg, flags,
                           m.a.params, m.a.hist_off, m.a.hist, m);
    };
    auto by_nl = [&](auto cap, auto every) {
        constexpr bool C = decltype(cap)::value, A = decltype(every)::value;
        if (nl == 16) go(mid_k_kernel<16, C, A>);
        else if (nl == 8) go(mid_k_kernel<8, C, A>);
        else go(mid_k_kernel<4, C, A>);
    };
    const std::true_type yes;
    const std::false_type no;
    if (capped) {
        if (all) by_nl(yes, yes);
        else by_nl(yes, no);
    } else {
        if (all) by_nl(no, yes);
        else by_nl(no, no);
    }
    return hipGetLastError();
}

}  // namespace fs

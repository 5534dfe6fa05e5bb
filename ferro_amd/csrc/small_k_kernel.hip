// small_k_kernel.hip - the kernel of batches whose every row is greedy or samples from at most 64 candidates.
#include "row_device.hpp"

#include <type_traits>

namespace fs {

// ------------------------------------------------------------------------------------------------ small-k kernel
// A separate kernel for batches whose every row is greedy or samples from k <= SK_K candidates with at most a
// repetition penalty (no frequency / presence counts) - the serving batches of ferro's decode loop (server.cpp:603-606:
// top-k 40-64 on every row). The host picks it from a host copy of the parameters (fs_sample_batch_hp). It has its own
// register budget (it shares no code path with the fused kernel), which lets it stream a row differently:
//   - one workgroup of SK_LT threads per (row, segment): every load of the segment (NL float4 per thread) is issued at
//     once, so the whole batch is requested at the start. The memory system serves the requests roughly in dispatch
//     order, so a row's segments (consecutive workgroups) receive their data together, and rows finish one after
//     another: the merge of an early row overlaps the streaming of later rows;
//   - per group of four logits only a maximum and, later, one compare: the bound is the ceil(k / waves)-th largest
//     lane maximum of each wave, the smallest over the waves (each lane maximum is a distinct logit of the segment, so
//     at least k logits of the segment reach it). Groups whose maximum reaches it are written to LDS, expanded to the
//     candidates at or above it (about 1.5 k per segment on heavy-tailed rows), and sorted exactly into the segment's
//     top k by a bitonic network in registers (DPP and permlane moves: no LDS round trips);
//   - the last segment of a row to finish (an L2 ticket) merges the row's sorted lists by a tree of bitonic merges and
//     finishes the row in one wave (softmax at temperature, min-p, top-p, draw: the merge path's wave_softmax).
// A segment with more than SK_CAP candidates (ties at its bound) selects its exact top k by a radix select over the
// composites held in registers instead (slow, exact).
struct SkShared {
    float4 gval[SK_NW][SK_GCAP + 1];       // groups of four whose maximum reaches the bound (+ a dummy slot)
    int32_t gidx[SK_NW][SK_GCAP + 1];      //   and the segment offset of their first logit
    uint64_t cand[SK_CAP];                 // the segment's candidates (composites)
    uint64_t wl[SK_NW][SK_K];              // per-wave sorted lists (segment sort, row merge)
    uint32_t bmp[SK_LT * 16 * 4 / 32];     // repetition window ids in the segment (largest segment: NL = 16)
    uint32_t hist[16];                     // radix select digits (exact fallback)
    uint32_t wb[SK_NW];
    uint32_t wcnt[SK_NW];
    uint32_t tscan[SK_NW];
    uint32_t misc[4];
#ifdef FS_TRACE
    uint64_t trace_t[16];
#endif
};
static_assert(offsetof(SkShared, cand) % 16 == 0, "the rank loops read the candidates in 16-byte pairs");
// Phase timestamps of the small-k kernel (FS_TRACE builds only; thread 0, after the barrier that closes a phase):
// 0 start, 11 the segment's logits in and transformed, 12 lane maxima sorted, 2 bound, 3 groups handed over,
// 4 candidates expanded, 5 list ranked and published, 6 ticket taken; merging workgroup: 7 lists folded, 8 row
// finished (greedy rows set only 0, 5-8). Slots 9-10: candidates and groups of the segment; 13-15: role (3 segment,
// 4 segment + merge), row, segment. ferro_amd/trace_phases.py --route host reads them.

// The exact path, for segments whose candidates at the bound overflow SK_CAP (ties at the bound): the segment's
// logits are re-read from memory (the L2 holds them by then) in batches of SK_EB per thread, sixteen loads in flight,
// and transformed again (softcap, then the repetition penalty from the segment's bitmap; past n: NaN).
constexpr int SK_EB = 16;
template <bool CAP, class F>
__device__ __forceinline__ void sk_each(const float* segp, int n, int nseg_elems, float cap, bool pen, float rep,
                                        const uint32_t* bmp, F f) {
    const int tid = threadIdx.x;
#pragma unroll 1
    for (int i0 = 0; i0 < nseg_elems; i0 += SK_LT * SK_EB) {
        float x[SK_EB];
#pragma unroll
        for (int j = 0; j < SK_EB; ++j) {
            const int i = i0 + j * SK_LT + tid;
            x[j] = i < n ? segp[i] : 0.0f;
        }
        if (CAP && cap > 0.0f) softcap_vals(x, cap);
#pragma unroll
        for (int j = 0; j < SK_EB; ++j) {
            const int i = i0 + j * SK_LT + tid;
            float l = x[j];
            if (pen && i < n && ((bmp[i >> 5] >> (i & 31)) & 1u)) l = l > 0.0f ? __fdiv_rn(l, rep) : __fmul_rn(l, rep);
            f(i, i < n ? key_of(l) : 0u);
        }
    }
}
// The exact k-th largest composite of the segment (every composite is distinct: the id is part of it), by a radix
// select over 4-bit digits. Slow, and rare.
template <bool CAP>
__device__ __forceinline__ uint64_t sk_kth_exact(const float* segp, int seg_lo, int n, int nseg_elems, float cap,
                                                 bool pen, float rep, int k, SkShared& s) {
    const int tid = threadIdx.x;
    uint64_t prefix = 0ull;
    int need = k;
#pragma unroll 1
    for (int sh = 60; sh >= 0; sh -= 4) {
        if (tid < 16) s.hist[tid] = 0u;
        __syncthreads();
        const uint64_t hi_mask = sh + 4 >= 64 ? 0ull : (~0ull << (sh + 4));
        sk_each<CAP>(segp, n, nseg_elems, cap, pen, rep, s.bmp, [&](int i, uint32_t key) {
            const uint64_t cm = comp_of(key, (uint32_t)(seg_lo + i));
            if (key != 0u && (cm & hi_mask) == prefix) atomicAdd(&s.hist[(uint32_t)(cm >> sh) & 15u], 1u);
        });
        __syncthreads();
        if (tid == 0) {
            int d = 15;
            for (; d > 0; --d) {
                const int c = (int)s.hist[d];
                if (c >= need) break;
                need -= c;
            }
            s.misc[2] = (uint32_t)d;
            s.misc[3] = (uint32_t)need;
        }
        __syncthreads();
        prefix |= (uint64_t)s.misc[2] << sh;
        need = (int)s.misc[3];
        __syncthreads();
    }
    return prefix;
}

// The merge of a row with many lists (more than 4 * SK_NW: the tree of bitonic merges then takes several rounds of
// list reads). Thread t reads entries 4 (t % 4) .. + 3 of list t / 4: the first 16 of every list in one round trip. The
// q-th entries of the lists, q = ceil(2 k / nseg), bound the row's k-th: m = ceil(k / q) of them at or above a value
// make q m >= k entries that reach it. The entries at or above the m-th largest (about 1.5 k) are ranked at once.
// 8 rows of 64 lists, k 50, a whole call: 18.6 us with the tree, 14.8 with this.
// Returns false, with nothing placed, when a list may hold more than its first 16 entries above the bound or more than
// SK_LT entries reach it (the tree then runs). The row's sorted top goes to s.wl[0]. Whole workgroup.
constexpr int SK_HEAD = 16;
__device__ __forceinline__ bool sk_merge_many(const uint64_t* rl, int nseg, int k, SkShared& s) {
    const int tid = threadIdx.x, lane = lane_id(), w = tid / WAVE;
    const int L = tid >> 2, part = tid & 3;
    uint64_t e[4] = {0ull, 0ull, 0ull, 0ull};
    if (L < nseg) {
        const ulonglong2* p2 = reinterpret_cast<const ulonglong2*>(rl + (int64_t)L * SK_K + 4 * part);
        const ulonglong2 x = p2[0], y = p2[1];
        e[0] = x.x; e[1] = x.y; e[2] = y.x; e[3] = y.y;
    }
    const int q = (2 * k + nseg - 1) / nseg, m = (k + q - 1) / q;
    uint32_t* hq = reinterpret_cast<uint32_t*>(&s.wl[0][0]);       // [SK_MAX_SEGS] keys of the q-th entries
    if (part == (q - 1) >> 2) {
        const int j = (q - 1) & 3;
        hq[L] = comp_key(j == 0 ? e[0] : j == 1 ? e[1] : j == 2 ? e[2] : e[3]);
    }
    __syncthreads();
    uint32_t T = (uint32_t)__builtin_amdgcn_readlane((int)sort64_desc_u32(hq[lane]), m - 1);
    if (T == 0u) T = 1u;                                           // fewer than m lists reach q entries: every entry
    uint32_t n = 0u;
#pragma unroll
    for (int j = 0; j < 4; ++j) n += comp_key(e[j]) >= T ? 1u : 0u;
    const uint32_t incl = wave_incl_scan_u32(n);
    const bool more = part == 3 && n == 4u && k > SK_HEAD;         // the list may go on above the bound
    const uint64_t mo = __ballot(more);
    if (lane == WAVE - 1) s.tscan[w] = incl;
    if (lane == 0) s.wcnt[w] = mo != 0ull ? 1u : 0u;
    __syncthreads();
    uint32_t base = 0u, tot = 0u, ovf = 0u;
#pragma unroll
    for (int v = 0; v < SK_NW; ++v) {
        base += v < w ? s.tscan[v] : 0u;
        tot += s.tscan[v];
        ovf |= s.wcnt[v];
    }
    if (ovf != 0u || tot > (uint32_t)SK_LT) return false;          // uniform
    uint32_t pos = base + incl - n;
#pragma unroll
    for (int j = 0; j < 4; ++j)
        if (comp_key(e[j]) >= T) s.cand[pos++] = e[j];
    if (tid < SK_K) s.wl[0][tid] = 0ull;                           // (hq is spent)
    __syncthreads();
    sk_rank(s.cand, reinterpret_cast<uint32_t*>(&s.wl[1][0]), (int)tot, [&](uint32_t r, uint64_t c) { if (r < (uint32_t)SK_K) s.wl[0][r] = c; });
    return true;
}

// CAP: some row of the batch has a softcap (the cap's code is left out of batches without one).
struct Ids16 {
    int32_t v[16];
};

// small_k_kernel's argument list as a struct: the argument segment follows the same layout rules
struct SkKernargs {
    const float* logits;
    int64_t ld;
    int B, V, nseg, flags;
    const fs_row_params* params;
    const int64_t* hist_off;
    const int32_t* hist;
    SkArgs a;
};
constexpr size_t SK_ARGS_OFF = offsetof(SkKernargs, a);

// Dynamic LDS a launch requests beyond SkShared (unused): with it a CU holds 4 workgroups (≈35 KB each of its 160 KB),
// as the kernel's 96 VGPRs would otherwise allow 5. Measured on MI355X with this instantiation: a 272-row call of 1088
// workgroups 21.3 -> 20.6 us with the limit, the headline's 1024 workgroups unchanged. (All-greedy batches run the
// greedy-only instantiation without it.)
constexpr unsigned SK_PAD_LDS = 16384;

// MANY: more than 4 * SK_NW lists per row (sk_merge_many; left out of the others, which it cost 0.2 us of 8.4).
// GREEDY: every row of the batch is greedy (the selection code is left out: fewer registers, more workgroups per CU).
template <int NL, bool CAP, bool GREEDY, bool MANY>
__global__ __launch_bounds__(SK_LT, 4) void small_k_kernel(const float* logits, int64_t ld, int B, int V, int nseg,
                                                        int flags, const fs_row_params* params,
                                                        const int64_t* hist_off, const int32_t* hist, SkArgs a_) {
    // The leading arguments arrive in SGPRs at wave launch (kernel-argument preloading), so the logits are requested
    // before any scalar memory round trip. A call with a repetition window (SK_MAY_PEN, set by the host from its copy of
    // the parameters) then reads the row's window bounds and requests its ids behind the logits.
    constexpr int SEG = SK_LT * NL * 4;
    static_assert(NL <= 16, "the repetition bitmap covers NL <= 16");
    constexpr int SK_WL = NL <= 8 ? 8 : 2;                     // 16-byte loads of a long window in flight (registers)
    __shared__ __align__(16) SkShared s;
    const int tid = threadIdx.x, lane = lane_id(), w = tid / WAVE;
    // workgroup i: XCD slot i % XCDS takes rows x, x + XCDS, ...: a row's segments are consecutive workgroups of one
    // index class mod XCDS, so they share an XCD and its L2 (the ticket and the lists)
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
    const int n_in = V - seg_lo < SEG ? V - seg_lo : SEG;             // logits of this segment (>= 1)

    // every load of the segment at once; past the row's end (rounded up to four, inside ld) reads are zeros, masked
    const float* rowp = logits + (int64_t)row * ld;
    const int nrec = ((n_in + 3) & ~3) * 4;
    const __amdgpu_buffer_rsrc_t rs =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(rowp + seg_lo), (short)0, nrec, 0x00020000);
    float4 v[NL];
#pragma unroll
    for (int q = 0; q < NL; ++q) {
        const f32x4 t = raw_buffer_load_f32x4(rs, (q * SK_LT + tid) * 16, 0, 2);    // nontemporal: read once
        v[q] = make_float4(t.x, t.y, t.z, t.w);
    }
    __builtin_amdgcn_sched_barrier(0);

    // the repetition window [wb0, len) over the row's history (sampling rows only: verification windows reach this
    // kernel only without an active penalty); its first 512 ids are requested behind the logits, two per thread
    bool pen = false, cnt_on = false;
    float rep = 1.0f, fq = 0.0f, pres = 0.0f;
    int64_t h0 = 0, len = 0, wb0 = 0;
    int wid[2] = {-1, -1};
    if (flags & SK_MAY_PEN) {
        const fs_row_params* pr = params + row;
        rep = ld_const(&pr->repetition_penalty);
        fq = ld_const(&pr->frequency_penalty);
        pres = ld_const(&pr->presence_penalty);
        fs_row_params pw;
        pw.repeat_last_n = ld_const(&pr->repeat_last_n);
        pw.penalty_from = ld_const(&pr->penalty_from);
        h0 = ld_const(hist_off + row);
        len = ld_const(hist_off + row + 1) - h0;
        // frequency / presence penalties (greedy rows only, segments of 4096 logits: the host checks both) need
        // each window id's count in the segment
        cnt_on = NL == 4 && (fq != 0.0f || pres != 0.0f);
        pen = (rep != 1.0f || cnt_on) && pw.repeat_last_n != 0 && len > 0;
        wb0 = window_begin(len, pw);                           // unconditionally: all five loads in one round trip
        if (!pen || wb0 >= len) { pen = false; wb0 = len; }
#pragma unroll
        for (int r = 0; r < 2; ++r) {
            const int64_t i = wb0 + r * SK_LT + tid;
            wid[r] = (pen && i < len) ? hist[h0 + i] : -1;
        }
    }
    const bool cp_on = (flags & SK_COPY) != 0;                 // a decode step: this segment's share of the history
    SkCopy cp = {};
    if (cp_on) cp = sk_cp_load(hist_off, hist, row, seg, nseg);
    // The remaining arguments are read from here on, through a pointer the compiler cannot trace back to the argument
    // segment: otherwise it loads some of them early and, short of scalar registers, spills them to vector lanes,
    // which waits for those loads before the logits are requested.
    const __attribute__((address_space(4))) char* kseg =
        (const __attribute__((address_space(4))) char*)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(kseg) : : "memory");
    const SkArgs& a = *(const SkArgs*)(kseg + SK_ARGS_OFF);
    (void)a_;

    // verification: the row's stream (its parameters); sampling: the row's own
    int pidx = row;
    if (a.mode == MODE_VERIFY) {
        int s0 = 0, s1 = a.n_streams;                          // the largest s with row_off[s] <= row
        while (s1 - s0 > 1) {
            const int m = (s0 + s1) >> 1;
            if (ld_const(a.row_off + m) <= row) s0 = m; else s1 = m;
        }
        pidx = s0;
    }
    const fs_row_params* pp = params + pidx;
    const float temp = ld_const(&pp->temperature);
    const int top_k = ld_const(&pp->top_k);
    const float cap = CAP ? ld_const(&pp->softcap) : 0.0f;
    const bool greedy = GREEDY || temp <= 0.0f || top_k == 1;
    const int k = greedy ? 1 : ((top_k > 0 && top_k < V) ? top_k : V);

    // repetition penalty: an exact bitmap of the window's ids in this segment (each distinct id once: sampler.cpp:14-17).
    // rep >= 1 never raises a logit (l > 0: l / rep <= l; l <= 0: l * rep <= l), so the bound is taken over the raw
    // logits, the bitmap is filled while the bound is sorted (the ids arrive right behind the logits), and the penalty
    // is applied to the handed-over logits only; the bound then needs a check (below). rep < 1 raises the flagged
    // logits: they are penalised before the bound (the bitmap first).
    // greedy rows take the penalty before their maximum (no bound to protect), with its counts when cnt_on
    const bool pen_late = pen && rep >= 1.0f && !greedy;
    const bool pen_early = pen && !pen_late;
    cnt_on = cnt_on && pen;
    // The softcap never decreases (tanhf does not, over every float, and the divide and multiply around it round a
    // monotone result), so sampled rows without an early penalty find their bound over the raw logits and cap only the
    // handed-over ones: a tanhf for about 100 logits of a segment instead of all of them (64 rows of 262144 logits,
    // k 64: 68.4 us -> 28.3).
    const bool cap_late = CAP && cap > 0.0f && !greedy && !pen_early;
    // cnt_on: 16-bit counts of the window's ids per logit of the segment, in the group buffer (unused on this path)
    uint32_t* cnt = reinterpret_cast<uint32_t*>(&s.gval[0][0]);
    static_assert(sizeof(SkShared::gval) >= SK_LT * 4 * 4 / 2 * sizeof(uint32_t),
                  "a 4096-logit segment's 16-bit counts fit the group buffer");
    bool ovf = false;
    auto mark = [&](int id) {
        const uint32_t rel = (uint32_t)(id - seg_lo);
        if (id >= 0 && id < V && rel < (uint32_t)SEG) {
            const uint32_t bit = 1u << (rel & 31u);
            atomicOr(&s.bmp[rel >> 5], bit);
            if (cnt_on) {
                const uint32_t sh = (rel & 1u) * 16u;
                const uint32_t old = atomicAdd(&cnt[rel >> 1], 1u << sh);
                ovf |= ((old >> sh) & 0xFFFFu) == 0xFFFFu;
            }
        }
    };
    // four ids of a long window. Most segments hold few of them: one compare sorts those out. Its ids repeat, and a
    // wave's atomics on one word run one after another, so a bit that already reads set is left (a stale read only sets
    // it again); the four reads are in flight together.
    const uint32_t in_seg = (uint32_t)n_in;                    // ids of this segment, from seg_lo
    auto mark4 = [&](const int4& id) {
        const uint32_t rel[4] = {(uint32_t)(id.x - seg_lo), (uint32_t)(id.y - seg_lo), (uint32_t)(id.z - seg_lo),
                                 (uint32_t)(id.w - seg_lo)};
        const uint32_t m01 = rel[0] < rel[1] ? rel[0] : rel[1], m23 = rel[2] < rel[3] ? rel[2] : rel[3];
        if ((m01 < m23 ? m01 : m23) < in_seg) {
            if (cnt_on) {
                mark(id.x); mark(id.y); mark(id.z); mark(id.w);
            } else {
                uint32_t word[4];
#pragma unroll
                for (int c = 0; c < 4; ++c) word[c] = *(volatile uint32_t*)&s.bmp[rel[c] < in_seg ? rel[c] >> 5 : 0u];
#pragma unroll
                for (int c = 0; c < 4; ++c)
                    if (rel[c] < in_seg && ((word[c] >> (rel[c] & 31u)) & 1u) == 0u)
                        atomicOr(&s.bmp[rel[c] >> 5], 1u << (rel[c] & 31u));
            }
        }
    };
    auto mark_window = [&]() {
        // the ids arrive behind the logits: an empty asm keeps the compiler from hoisting their first use (and the
        // wait for every load it needs) above the branch that calls this
        int i0 = wid[0], i1 = wid[1];
        asm volatile("" : "+v"(i0), "+v"(i1));
        mark(i0);
        mark(i1);
        // the rest of a long window: 16 bytes per load from the first 16-byte block on, SK_WL loads in flight (with one
        // id per load and round trip, decode steps of 8 rows of 262144 logits with 4096 to 28672 ids each, the copy
        // included: 49 us; now 22)
        const int64_t i = wb0 + 2 * SK_LT;
        if (i < len) {
            const int32_t* hp = a.hist + h0;
            const int64_t ab = i + (int64_t)((0u - (unsigned)((uintptr_t)(hp + i) >> 2)) & 3u);
            if (i + tid < ab && i + tid < len) mark(hp[i + tid]);      // at most three ids before it
            const int4* hv = reinterpret_cast<const int4*>(hp + ab);
            const int64_t nv = ab < len ? (len - ab) >> 2 : 0;
            int64_t j0 = 0;
            for (; j0 + SK_WL * SK_LT <= nv; j0 += SK_WL * SK_LT) {
                int4 w4[SK_WL];
#pragma unroll
                for (int r = 0; r < SK_WL; ++r) w4[r] = hv[j0 + r * SK_LT + tid];
#pragma unroll
                for (int r = 0; r < SK_WL; ++r) mark4(w4[r]);
            }
            for (int64_t j = j0 + tid; j < nv; j += 2 * SK_LT) {       // the last ones, two in flight
                const int4 x = hv[j];
                const bool more = j + SK_LT < nv;
                const int4 y = more ? hv[j + SK_LT] : x;
                mark4(x);
                if (more) mark4(y);
            }
            const int64_t rest = ab + 4 * nv;
            if (rest + tid < len) mark(hp[rest + tid]);                // at most three ids after the last block
        }
    };
    if (pen) {
        for (int i = tid; i < SEG / 32; i += SK_LT) s.bmp[i] = 0u;
        if (cnt_on)
            for (int i = tid; i < SEG / 2; i += SK_LT) cnt[i] = 0u;
        __syncthreads();
    }
    uint64_t pm = 0ull;                        // rep < 1 or greedy: 4 bits per group of this thread
    if (pen_early) {
        mark_window();
        if (ovf) atomicOr(a.err, FS_DEVERR_COUNT_OVERFLOW);
        __syncthreads();
#pragma unroll
        for (int q = 0; q < NL; ++q) {
            const uint32_t rel = (uint32_t)(q * SK_LT + tid) * 4u;
            pm |= (uint64_t)((s.bmp[rel >> 5] >> (rel & 31u)) & 0xFu) << (4 * q);
        }
    }
    const bool wpen = __ballot(pm != 0ull) != 0ull;
    const bool tail = n_in < SEG;

    // the logits as ferro's sampler sees them (softcap; rep < 1: the penalty; past the row's end: NaN, never a
    // candidate) and the lane maximum (NaN-free: fmaxf drops NaN; NaN when every logit of the lane is NaN)
    float lm = __builtin_nanf("");
#pragma unroll
    for (int q = 0; q < NL; ++q) {
        float e[4] = {v[q].x, v[q].y, v[q].z, v[q].w};
        if (CAP && cap > 0.0f && !cap_late) softcap_vals(e, cap);   // a rolled loop: one copy of the cap per group
        if (wpen) {
            const uint32_t nib = (uint32_t)(pm >> (4 * q)) & 0xFu;
            if (__ballot(nib != 0u)) {
#pragma unroll
                for (int c = 0; c < 4; ++c)
                    if ((nib >> c) & 1u) {
                        float l = e[c] > 0.0f ? __fdiv_rn(e[c], rep) : __fmul_rn(e[c], rep);
                        if (cnt_on) {                      // l - (count * frequency + presence), as the fused kernel
                            const uint32_t rel = (uint32_t)(q * SK_LT + tid) * 4u + (uint32_t)c;
                            const float cc = (float)((cnt[rel >> 1] >> ((rel & 1u) * 16u)) & 0xFFFFu);
                            l = __fsub_rn(l, __fadd_rn(__fmul_rn(cc, fq), pres));
                        }
                        e[c] = l;
                    }
            }
        }
        if (tail) {
            const int e0 = (q * SK_LT + tid) * 4;
#pragma unroll
            for (int c = 0; c < 4; ++c)
                if (e0 + c >= n_in) e[c] = __builtin_nanf("");
        }
        v[q] = make_float4(e[0], e[1], e[2], e[3]);
        lm = fmaxf(lm, fmaxf(fmaxf(e[0], e[1]), fmaxf(e[2], e[3])));
    }
    // Greedy rows (their penalties already applied above): the segment's list is its first maximum alone (ferro's
    // scan, sampler.cpp:19-23, takes a larger logit only: the lowest index among equal maxima; NaN never), so the
    // bound, the candidates and their ranks are skipped: a lane's first index holding its maximum, then the largest
    // composite of the workgroup (value first, then the lower id). The rest of the list is zeros, which every merge
    // reads as empty.
    uint64_t* myl = a.lists + ((int64_t)row * a.nseg + seg) * SK_K;
    const bool gfast = greedy;
    if (gfast) {
        uint64_t best = 0ull;
        if (lm == lm) {                                        // NaN: every logit of the lane is NaN
            uint32_t first = 0u;
#pragma unroll
            for (int q = NL - 1; q >= 0; --q) {
                const uint32_t e0 = (uint32_t)(seg_lo + (q * SK_LT + tid) * 4);
                first = v[q].w == lm ? e0 + 3u : first;
                first = v[q].z == lm ? e0 + 2u : first;
                first = v[q].y == lm ? e0 + 1u : first;
                first = v[q].x == lm ? e0 : first;
            }
            best = comp_of(key_of(lm), first);
        }
        best = wave_max(best);
        if (lane == 0) s.wl[w][0] = best;
        __syncthreads();
        if (w == 0) {
            const uint64_t m = wave_max(lane < SK_NW ? s.wl[lane][0] : 0ull);
            myl[lane] = lane == 0 ? m : 0ull;
        }
    } else {
        // the bound: each wave sorts its lane maxima in registers (no scalar round trips per step); lane kq - 1 holds
        // its kq-th largest, and the smallest over the waves counts SK_NW kq >= k distinct logits (one lane more per
        // wave when the penalty comes later: the raw logits counted may be among the penalised ones)
        const uint32_t kq = (uint32_t)((k + SK_NW - 1) / SK_NW) + (pen_late ? 1u : 0u);
        SK_MARK(11);
        {
            const uint32_t srt = sort64_desc_u32(key_of(lm));
            if (lane == (int)kq - 1) s.wb[w] = srt;
        }
        if (pen_late) mark_window();                               // completed by the barrier below
        SK_MARK(12);
        __syncthreads();
        SK_MARK(2);
        uint32_t tau = s.wb[0];
#pragma unroll
        for (int q = 1; q < SK_NW; ++q) tau = s.wb[q] < tau ? s.wb[q] : tau;
        if (tau == 0u) tau = 1u;                                   // NaN (key 0) is never a candidate
        const float tf = tau > 0x007FFFFFu ? val_of(tau) : -__builtin_huge_valf();
        // cap_late: the candidates are the logits whose capped value reaches the capped bound tc; tr is a raw value that
        // every one of them reaches: lane j < 32 caps the value 2^j keys below the bound (lane 32 the bound itself), and the first that falls
        // below tc (the cap is flat where it saturates) ends the range.
        float tc = tf, tr = tf;
        if (cap_late) {
            const uint32_t kb = tau > 0x007FFFFFu ? tau : 0x007FFFFFu;          // (the key of -inf is the lowest)
            const uint32_t step = lane < 32 ? 1u << lane : 0u, room = kb - 0x007FFFFFu;
            const float c = softcap_one(val_of(room > step ? kb - step : 0x007FFFFFu + (lane < 32 ? 0u : room)), cap);
            // no bound (fewer than k numbers among the maxima counted, or one at -inf): every number is a candidate, a
            // penalised one below -cap too
            tc = room != 0u ? read_lane(c, 32) : tf;
            const uint64_t below = __ballot(lane < 32 && c < tc);
            tr = -__builtin_huge_valf();
            if (below) {
                const uint32_t st = 1u << (__ffsll((unsigned long long)below) - 1);
                tr = room > st ? val_of(kb - st) : tr;
            }
        }
        // groups whose maximum reaches the bound: this wave's region of the group buffer, in lane order
        uint32_t gmask = 0u;
#pragma unroll
        for (int q = 0; q < NL; ++q)                     // the group's raw maximum (recomputed: no register array)
            gmask |= (fmaxf(fmaxf(v[q].x, v[q].y), fmaxf(v[q].z, v[q].w)) >= tr ? 1u : 0u) << q;
        const uint32_t gn = (uint32_t)__popc(gmask);
        const uint32_t gincl = wave_incl_scan_u32(gn);
        const uint32_t wtot = (uint32_t)__builtin_amdgcn_readlane((int)gincl, WAVE - 1);
        uint32_t go = gincl - gn;
        // the groups any lane of the wave hands over (one scalar mask); per such group every lane writes, those without
        // it into the region's dummy slot, so no per-lane branch waits on a compare
        const uint32_t wmask = (uint32_t)__builtin_amdgcn_readfirstlane(
            (int)wave_allreduce(gmask, [](uint32_t x, uint32_t y) { return x | y; }));
#pragma unroll
        for (int q = 0; q < NL; ++q) {
            if ((wmask >> q) & 1u) {
                const bool mine = ((gmask >> q) & 1u) != 0u && go < (uint32_t)SK_GCAP;
                const uint32_t slot = mine ? go : (uint32_t)SK_GCAP;
                s.gval[w][slot] = v[q];
                s.gidx[w][slot] = (int32_t)((uint32_t)(q * SK_LT + tid) * 4u);
                go += (gmask >> q) & 1u;
            }
        }
        if (lane == 0) s.wcnt[w] = wtot;
        __syncthreads();
        SK_MARK(3);
        // expansion: thread t takes group t of the concatenated regions, its logits at or above the bound become
        // candidates
        uint32_t goff[SK_NW + 1];
        goff[0] = 0u;
        bool gover = false;
#pragma unroll
        for (int q = 0; q < SK_NW; ++q) {
            const uint32_t c = s.wcnt[q];
            gover |= c > (uint32_t)SK_GCAP;
            goff[q + 1] = goff[q] + (c < (uint32_t)SK_GCAP ? c : (uint32_t)SK_GCAP);
        }
        const uint32_t G = goff[SK_NW];
        uint64_t cm[4] = {0ull, 0ull, 0ull, 0ull};
        bool cp[4] = {false, false, false, false};
        uint32_t nc = 0u;
        if (!gover && (uint32_t)tid < G) {
            int r = 0;
            uint32_t gb = 0u;
#pragma unroll
            for (int q = 1; q < SK_NW; ++q) {
                const bool past = (uint32_t)tid >= goff[q];
                r += past ? 1 : 0;
                gb = past ? goff[q] : gb;
            }
            const uint32_t gi = (uint32_t)tid - gb;
            const float4 gv = s.gval[r][gi];
            const uint32_t gw = (uint32_t)s.gidx[r][gi];
            const int e0 = (int)gw;
            // rep >= 1: the group's penalised logits, from the bitmap (its 4 bits share a word: e0 % 4 == 0)
            float e[4] = {gv.x, gv.y, gv.z, gv.w};
            if (CAP && cap_late) {
#pragma unroll 1
                for (int c = 0; c < 4; c += 2) {
                    float e2[2] = {c ? e[2] : e[0], c ? e[3] : e[1]};
                    softcap_vals_unrolled(e2, cap);
                    if (c) { e[2] = e2[0]; e[3] = e2[1]; } else { e[0] = e2[0]; e[1] = e2[1]; }
                }
            }
            if (pen_late) {
                const uint32_t nib = (s.bmp[(uint32_t)e0 >> 5] >> ((uint32_t)e0 & 31u)) & 0xFu;
#pragma unroll
                for (int c = 0; c < 4; ++c)
                    if ((nib >> c) & 1u) e[c] = e[c] > 0.0f ? __fdiv_rn(e[c], rep) : __fmul_rn(e[c], rep);
            }
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                cp[c] = e[c] >= tc;
                cm[c] = comp_of(key_of(e[c]), (uint32_t)(seg_lo + e0 + c));
                nc += cp[c] ? 1u : 0u;
            }
        }
        if (G > (uint32_t)SK_LT) gover = true;                     // more groups than threads: the exact path
        // block exclusive scan of the candidate counts
        const uint32_t cincl = wave_incl_scan_u32(nc);
        if (lane == WAVE - 1) s.tscan[w] = cincl;
        __syncthreads();
        SK_MARK(4);
        uint32_t cbase = 0u, ntot = 0u;
#pragma unroll
        for (int q = 0; q < SK_NW; ++q) {
            const uint32_t t = s.tscan[q];
            cbase += q < w ? t : 0u;
            ntot += t;
        }
        // With the penalty applied after the bound, fewer than k logits may stay at or above it: the segment's top k
        // may then hold a logit below the bound, which was not handed over (never expected with the spare lane per
        // wave)
        const bool short_k = pen_late && ntot < (uint32_t)k && tf > -__builtin_huge_valf();
        const bool exact = gover || short_k || ntot > (uint32_t)SK_CAP;   // uniform
        if (!exact) {
            uint32_t pos = cbase + cincl - nc;
#pragma unroll
            for (int c = 0; c < 4; ++c)
                if (cp[c]) s.cand[pos++] = cm[c];
        }
        if (exact) {
            // ties at the bound: the exact k-th composite of the segment, then the (exactly k) composites at or above
            // it
            const float* segp = rowp + seg_lo;
            const uint64_t kth = sk_kth_exact<CAP>(segp, seg_lo, n_in, SEG, cap, pen, rep, k, s);
            if (tid == 0) s.misc[0] = 0u;
            __syncthreads();
            sk_each<CAP>(segp, n_in, SEG, cap, pen, rep, s.bmp, [&](int i, uint32_t key) {
                const uint64_t c64 = comp_of(key, (uint32_t)(seg_lo + i));
                if (key != 0u && c64 >= kth) {
                    const uint32_t p = atomicAdd(&s.misc[0], 1u);
                    if (p < (uint32_t)SK_K) s.cand[p] = c64;
                }
            });
            __syncthreads();
            ntot = s.misc[0] < (uint32_t)SK_K ? s.misc[0] : (uint32_t)SK_K;
        }
        __syncthreads();
        // the segment's top k, sorted by rank
        {
            const int n = (int)ntot;
            if (n <= SK_LT) {
                sk_rank(s.cand, reinterpret_cast<uint32_t*>(&s.wl[1][0]), n, [&](uint32_t r, uint64_t c) { if (r < (uint32_t)k) myl[r] = c; });   // the published list
            } else {                                               // 256 < n <= SK_CAP: two candidates per thread
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const int c = tid + h * SK_LT;
                    if (c < n) {
                        const uint64_t me = s.cand[c];
                        uint32_t r = 0u;
                        int jj = 0;
                        const ulonglong2* c2 = reinterpret_cast<const ulonglong2*>(s.cand);
                        for (; jj + 8 <= n; jj += 8) {
                            const ulonglong2 e0 = c2[jj >> 1], e1 = c2[(jj >> 1) + 1], e2 = c2[(jj >> 1) + 2],
                                             e3 = c2[(jj >> 1) + 3];
                            r += (e0.x > me ? 1u : 0u) + (e0.y > me ? 1u : 0u) + (e1.x > me ? 1u : 0u) +
                                 (e1.y > me ? 1u : 0u) + (e2.x > me ? 1u : 0u) + (e2.y > me ? 1u : 0u) +
                                 (e3.x > me ? 1u : 0u) + (e3.y > me ? 1u : 0u);
                        }
                        for (; jj < n; ++jj) r += s.cand[jj] > me ? 1u : 0u;
                        if (r < (uint32_t)k) myl[r] = me;
                    }
                }
            }
            if (tid >= (n < k ? n : k) && tid < SK_K) myl[tid] = 0ull;   // slots past the segment's top k
        }
        SK_TAG(9, ntot);
        SK_TAG(10, G);
    }
    if (cp_on) sk_cp_store(a, cp, row, seg);
    vm_drain();                                                // the list is in the L2
    __syncthreads();
    SK_MARK(5);
    if (tid == 0) {
        const uint32_t t = __hip_atomic_fetch_add(a.ticket + row, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        s.misc[1] = t == (uint32_t)a.nseg - 1u ? 1u : 0u;
    }
    __syncthreads();
    SK_MARK(6);
    if (s.misc[1] == 0u) {
        SK_FLUSH();
        return;
    }
    SK_TAG(13, 4);
    // a decode step's draw takes two dependent reads: requested before the lists, so that they overlap the merge
    SkDraw dr = {0.0, 0};
    if (!greedy && a.dmt) dr = sk_draw(a, row);
    // ---- the row's merge (the last of its segments): wave w folds lists w, w + SK_NW, ... (the first as stored,
    // the rest reversed: ascending), then wave 0 folds the waves' lists
    const uint64_t* rl = a.lists + (int64_t)row * a.nseg * SK_K;
    uint64_t acc = 0ull;
    if (greedy) {
        // k = 1: every list holds its segment's top composite first; wave 0 takes the largest of the nseg heads
        if (w != 0) return;
        SK_MARK(7);
        if (tid == 0) a.ticket[row] = 0u;                     // all segments have counted: reset for the next call
        acc = wave_max(lane < a.nseg ? rl[lane * SK_K] : 0ull);
    } else if (MANY && sk_merge_many(rl, a.nseg, k, s)) {
        __syncthreads();
        if (w != 0) return;
        SK_MARK(7);
        if (tid == 0) a.ticket[row] = 0u;                     // all segments have counted: reset for the next call
        acc = s.wl[0][lane];
    } else {
        for (int L0 = w; L0 < a.nseg; L0 += 4 * SK_NW) {
            // four lists per wave, requested together: lists 0 and 2 as stored (descending), 1 and 3 reversed
            uint64_t b[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int L = L0 + r * SK_NW;
                b[r] = L < a.nseg ? rl[L * SK_K + ((r & 1) ? WAVE - 1 - lane : lane)] : 0ull;
            }
            // two independent merges (their latencies overlap), then one
            const uint64_t m01 = merge_top64<true>(b[0], b[1]);
            const uint64_t m23 = merge_top64<false>(b[2], b[3]);
            if (L0 == w) acc = merge_top64<true>(m01, m23);
            else acc = merge_top64<true>(acc, merge_top64<false>(m01, m23));
        }
        // across the waves: waves 0 and 2 fold 1 and 3 (in parallel), then wave 0 folds wave 2's
        s.wl[w][lane] = acc;
        __syncthreads();
        if (w == 0 || w == 2) acc = merge_top64(acc, s.wl[w + 1][WAVE - 1 - lane]);
        if (w == 2) s.wl[2][lane] = acc;
        __syncthreads();
        if (w != 0) return;
        SK_MARK(7);
        if (tid == 0) a.ticket[row] = 0u;                     // all segments have counted: reset for the next call
        acc = merge_top64(acc, s.wl[2][WAVE - 1 - lane]);
    }
    // the row's candidates: lane i holds the i-th in ferro's order (value desc, id asc); NaN never is one
    const int kk = __popcll(__ballot(lane < k && acc != 0ull));
    Args fa = {};
    fa.mode = MODE_SAMPLE; fa.kcap = a.kcap; fa.cand_ids = a.cand_ids; fa.cand_probs = a.cand_probs;
    RowCtx rc = {};
    rc.row = row;
    rc.p.temperature = temp; rc.p.top_k = top_k;
    rc.p.top_p = ld_const(&pp->top_p); rc.p.min_p = ld_const(&pp->min_p);
    int tok = 0, keep = 1;
    if (greedy) {
        // ferro's scan (sampler.cpp:19-23) keeps index 0 when its logit is NaN; otherwise the first maximum
        float l0 = ld_const(rowp);
        if (CAP && cap > 0.0f) l0 = softcap_one(l0, cap);
        tok = (l0 != l0 || kk == 0) ? 0 : (int)comp_id(read_lane(acc, 0));
        if (lane == 0 && a.kcap > 0) {
            if (a.cand_ids) a.cand_ids[(int64_t)row * a.kcap] = tok;
            if (a.cand_probs) a.cand_probs[(int64_t)row * a.kcap] = 1.0;
        }
    } else if (kk == 0) {
        tok = 0; keep = 0;                                     // every logit NaN: token 0, nothing kept
    } else {
        if (!a.dmt) dr = sk_draw(a, row);
        wave_softmax(fa, rc, lane < kk ? acc : 0ull, kk, dr.u, tok, keep);
    }
    sk_finish(a, row, pidx, !greedy, tok, keep, cp, dr.idx, &s.cand[0]);
    SK_MARK(8);
    SK_FLUSH();
}

hipError_t launch_small_k(int nl, bool capped, bool all_greedy, unsigned grid, int flags, const SkArgs& k,
                          hipStream_t st) {
    const dim3 gd(grid), bd(SK_LT);
    // all-greedy batches: the greedy-only kernel, without the LDS pad (its registers allow more workgroups per CU)
    auto go = [&](auto kern, unsigned pad) {
        hipLaunchKernelGGL(kern, gd, bd, pad, st, k.logits, k.ld, k.B, k.V, k.nseg, flags, k.params, k.hist_off,
                           k.hist, k);
    };
    auto by_nl = [&](auto cap, auto greedy, auto many) {
        constexpr bool C = decltype(cap)::value, G = decltype(greedy)::value, M = decltype(many)::value;
        const unsigned pad = G ? 0u : SK_PAD_LDS;
        if (nl == 16) go(small_k_kernel<16, C, G, M>, pad);
        else if (nl == 8) go(small_k_kernel<8, C, G, M>, pad);
        else go(small_k_kernel<4, C, G, M>, pad);
    };
    const std::true_type yes;
    const std::false_type no;
    if (all_greedy) {
        if (capped) by_nl(yes, yes, no);
        else by_nl(no, yes, no);
    } else if (k.nseg > 4 * SK_NW) {
        if (capped) by_nl(yes, no, yes);
        else by_nl(no, no, yes);
    } else {
        if (capped) by_nl(yes, no, no);
        else by_nl(no, no, no);
    }
    return hipGetLastError();
}

}  // namespace fs

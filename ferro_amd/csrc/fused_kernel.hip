// fused_kernel.hip - the kernel that samples every batch (segment_kernel), and its merge alone (merge_kernel).
//
// One kernel per call on the caller's stream (two when a row is shorter than one 4096-logit tile).
//
// segment_kernel (one 512-thread workgroup per (row, segment) item, two per CU): a row of V fp32 logits is split
// into nseg segments of seg_tiles tiles (TILE = 4096 logits); the items are dealt to the 8 XCDs so that a row's
// segments share one XCD and its L2. A segment is streamed from HBM with PF tiles in flight (16-byte buffer
// loads, the only pass over the logits). Per tile:
//   - penalty pass on the fly (reference src/sampler.cpp:11-18, plus the frequency/presence extension):
//     repetition only - an exact bitmap of the window's ids in the segment; with counts - the window ids that fall
//     in the tile are counted in a 16-bit LDS table; each thread patches the few penalised logits it holds;
//   - greedy rows (temperature <= 0 or top_k == 1, sampler.cpp:19): each lane keeps its first maximum;
//   - top-k rows: every logit is compared with a running fp32 bound tf (a lower bound of the row's k-th key) in a
//     wave ballot; the few that pass are appended to an LDS buffer as 64-bit composites (key << 32 | ~id: integer
//     order = ferro's candidate order, value desc then id asc, sampler.cpp:30).
// The bound starts from tile 0's histogram and is raised from a per-row histogram of counted logits shared by the
// row's segments (L2 atomics): any k counted logits at or above a bin make its lower edge a valid bound. The
// buffer is compacted (entries below the bound dropped, else the exact k-th composite kept) when it could
// overflow. Each segment publishes its candidates at or above its final bound.
//
// The merge (a role of the same grid: one workgroup per row after the segments, on the row's XCD; a separate
// merge_kernel launch when rows are shorter than one tile): waits for the row's segment count in the L2, gathers
// the segments' lists, L = max of the segments' bounds bounds the
// row's k-th key from below, a histogram over [L, max] gives a tight T1, the ~k candidates >= T1 are sorted in
// LDS (ferro's cand_, sampler.cpp:25-35; rank sort or a counting sort), then the double-precision softmax at
// temperature, min-p, top-p and the draw r = u * tot (sampler.cpp:37-49), with scans in place of the sequential
// sums. Rows with k > 2048 are sampled here by whole-row passes. Verify windows (server.cpp:627-637): the last
// row of a stream to finish (agent-scope sc1 stores, a vmcnt drain and an agent-scope counter, no L2 write-back)
// computes the accepted prefix.
#include "sampler_device.hpp"
#include "sampler_launch.hpp"

namespace fs {

// ------------------------------------------------------------------------------------------------ kernel
struct Shared {
    uint64_t cand[CAP];                // candidate buffer / merge gather
    uint32_t scr[TILE / 2 + NBINS];    // per-tile 16-bit penalty counts, then histograms; or a 64-bit stage
    uint32_t off[MAX_SEGS + 1];        // merge: flat offsets of the segment lists
    int32_t ids[WIDS];                 // the penalty window's ids that fall in the current segment
    uint32_t wsum[NWAVES];
    uint32_t count;
    uint32_t tmax;                     // segment kernel: the largest key of tile 0
    uint32_t rc64[WAVE];               // segment kernel: tile-0 counts in the 64 coarse bins up to tmax's
    uint32_t nids;
    uint32_t nfast;                    // large-row segment: the cut's survivors written to the slot
    uint32_t wcnt[NWAVES];             // large-row segment: each wave's part of the cut's LDS list
    uint32_t tmx[2][NWAVES];           // large-row segment: the waves' tile maxima (keys), alternating tiles
    uint32_t misc_alone;               // merge role: the row is computed from its logits alone
#ifdef FS_TRACE
    uint64_t trace_t[16];              // this workgroup's phase timestamps (written to a.trace at its end)
#endif
    Red red;
    __device__ __forceinline__ uint32_t* cnt() { return scr; }
    __device__ __forceinline__ uint32_t* bins() { return scr + TILE / 2; }
    __device__ __forceinline__ uint64_t* stage() { return reinterpret_cast<uint64_t*>(scr); }   // KMAX entries
};

// Descending sort of m <= KMAX distinct composites a[0, m), in place (whole block; returns after a barrier). A
// counting sort: NB bins span [min, max] of the composites (bin 0 = the largest); each entry takes a slot in its
// bin with an LDS atomic (cnt) and is scattered to tmp[bin start + slot]; then each entry counts the larger entries
// of its own bin and lands at bin start + that count. Bins of a smooth tail hold a few entries each (equal keys
// spread over the id bits); when one holds more than BIN_SORT_MAX the bitonic network sorts instead (a must then
// hold the next power of two >= m entries). cnt and start hold NB counters each; tmp holds m entries.
constexpr int BIN_SORT_MAX = 48;
template <int NB>
__device__ __forceinline__ uint32_t bin_sort_desc(uint64_t* a, int m, uint64_t* tmp, uint32_t* cnt, uint32_t* start,
                                                  Red& red, uint32_t* wsum) {
    constexpr int EPT = KMAX / BLOCK;            // entries per thread
    constexpr int BPT = NB / BLOCK;              // bins per thread
    static_assert(BPT >= 1 && NB == BPT * BLOCK, "whole bins per thread");
    const int tid = threadIdx.x;
    uint64_t v[EPT];
    uint64_t cmn = ~0ull, cmx = 0ull;
#pragma unroll
    for (int q = 0; q < EPT; ++q) {
        const int i = q * BLOCK + tid;
        v[q] = i < m ? a[i] : 0ull;
        if (i < m) {
            cmn = v[q] < cmn ? v[q] : cmn;
            cmx = v[q] > cmx ? v[q] : cmx;
        }
    }
#pragma unroll
    for (int q = 0; q < BPT; ++q) cnt[q * BLOCK + tid] = 0u;
    cmn = block_min_u64(cmn, red);               // its barriers also order the zeroed counts
    cmx = block_max_u64(cmx, red);
    if (m <= 1) return 0u;
    int sh = 0;                                  // composites cmn..cmx map to bins NB-1..0
    while (((cmx - cmn) >> sh) >= (uint64_t)NB) ++sh;
    uint32_t bin[EPT], slot[EPT];
#pragma unroll
    for (int q = 0; q < EPT; ++q) {
        bin[q] = 0u;
        slot[q] = 0u;
        if (q * BLOCK + tid < m) {
            bin[q] = (uint32_t)(NB - 1) - (uint32_t)((v[q] - cmn) >> sh);
            slot[q] = atomicAdd(&cnt[bin[q]], 1u);
        }
    }
    __syncthreads();
    uint32_t c[BPT], sum = 0u, big = 0u;
#pragma unroll
    for (int j = 0; j < BPT; ++j) {
        c[j] = cnt[BPT * tid + j];
        sum += c[j];
        big = c[j] > big ? c[j] : big;
    }
    uint32_t tot;
    uint32_t off = block_excl_scan<uint32_t>(sum, wsum, &tot);
#pragma unroll
    for (int j = 0; j < BPT; ++j) {
        start[BPT * tid + j] = off;
        off += c[j];
    }
    big = block_max_u32(big, red);               // its barriers also publish the starts
    if (big > (uint32_t)BIN_SORT_MAX) {
        int np = 1;
        while (np < m) np <<= 1;
        for (int i = m + tid; i < np; i += BLOCK) a[i] = 0ull;
        __syncthreads();
        bitonic_desc(a, np);
        return big;
    }
#pragma unroll
    for (int q = 0; q < EPT; ++q)
        if (q * BLOCK + tid < m) tmp[start[bin[q]] + slot[q]] = v[q];
    __syncthreads();
#pragma unroll
    for (int q = 0; q < EPT; ++q) {
        if (q * BLOCK + tid < m) {
            const uint32_t b0 = start[bin[q]], n = cnt[bin[q]];
            uint32_t r = 0u, j = 0u;
            for (; j + 4u <= n; j += 4u) {              // four LDS reads in flight per step
                const uint64_t t0 = tmp[b0 + j], t1 = tmp[b0 + j + 1], t2 = tmp[b0 + j + 2], t3 = tmp[b0 + j + 3];
                r += (t0 > v[q] ? 1u : 0u) + (t1 > v[q] ? 1u : 0u) + (t2 > v[q] ? 1u : 0u) + (t3 > v[q] ? 1u : 0u);
            }
            for (; j < n; ++j) r += tmp[b0 + j] > v[q] ? 1u : 0u;
            a[b0 + r] = v[q];
        }
    }
    __syncthreads();
    return big;                                  // the largest bin (> BIN_SORT_MAX: the bitonic network sorted)
}
// The candidate buffer's first m <= KMAX entries, with the second KMAX entries as the scatter area.
__device__ __forceinline__ uint32_t bin_sort_desc(int m, Shared& s) {
    static_assert(TILE / 2 >= NBINS && 2 * KMAX <= CAP, "counts in cnt(), starts in bins(), scatter after the input");
    return bin_sort_desc<NBINS>(s.cand, m, s.cand + KMAX, s.cnt(), s.bins(), s.red, s.wsum);
}
static_assert((TILE / 2 + NBINS) / 2 >= KMAX, "the stage holds a compacted top k");

// Issue the loads of one tile (TPT logits per thread: float4 j at element lo + (j*BLOCK + t)*4) without waiting.
// Lanes past the row's end read a clamped in-bounds address and are zeroed. The float4 holding element V-1 may
// extend up to 12 bytes past it, inside the same 16-byte-aligned block (never into another page); masked too.
// The segment kernel only streams full tiles (a row's partial last tile is handled by the merge kernel).
__device__ __forceinline__ void load_tile(float (&x)[TPT], const float* rowp, int lo) {
    const float4* p = reinterpret_cast<const float4*>(rowp + lo) + threadIdx.x;
#pragma unroll
    for (int j = 0; j < NV; ++j) {
        const float4 t = p[j * BLOCK];
        x[4 * j + 0] = t.x; x[4 * j + 1] = t.y; x[4 * j + 2] = t.z; x[4 * j + 3] = t.w;
    }
}
// Tile t of a segment through its buffer resource: a tile past the segment's end reads zeros without a memory
// access, so the tile loop requests its next tiles unconditionally (straight-line loads keep the compiler's
// memory-counter waits exact: consuming a tile waits for that tile only).
template <int AUX = 0>
__device__ __forceinline__ void load_seg_tile(float (&x)[TPT], __amdgpu_buffer_rsrc_t rs, int t) {
#pragma unroll
    for (int j = 0; j < NV; ++j) {
        const f32x4 v = raw_buffer_load_f32x4(rs, (j * BLOCK + (int)threadIdx.x) * 16, t * TILE * 4, AUX);
        x[4 * j + 0] = v.x; x[4 * j + 1] = v.y; x[4 * j + 2] = v.z; x[4 * j + 3] = v.w;
    }
}
// element id of this thread's i-th logit of the tile starting at lo
__device__ __forceinline__ int elem_id(int lo, int i) { return lo + ((i >> 2) * BLOCK + (int)threadIdx.x) * 4 + (i & 3); }

// Penalty pass on one tile in registers (sampler.cpp:11-18; frequency/presence extension): the window's ids that
// fall in [lo, lo + TILE) are counted in a 16-bit LDS table, then each thread patches its counted logits.
// Entry: the table may still be read by the previous tile's patching, so the caller has passed a barrier.
__device__ __forceinline__ void apply_penalties(float (&x)[TPT], const Args& a, const RowCtx& rc, int lo, Shared& s) {
    const int tid = threadIdx.x;
    for (int i = tid; i < TILE / 8; i += BLOCK) reinterpret_cast<uint4*>(s.cnt())[i] = make_uint4(0u, 0u, 0u, 0u);
    __syncthreads();
    bool ovf = false;
    auto count_id = [&](int id) {
        const uint32_t rel = (uint32_t)(id - lo);
        if (rel < (uint32_t)TILE) {
            const uint32_t sh = (rel & 1u) * 16u;
            const uint32_t old = atomicAdd(&s.cnt()[rel >> 1], 1u << sh);
            ovf |= ((old >> sh) & 0xFFFFu) == 0xFFFFu;
        }
    };
    const int nids = (int)s.nids;
    if (nids <= WIDS)                                 // the segment's window ids, gathered in LDS
        for (int i = tid; i < nids; i += BLOCK) count_id(s.ids[i]);
    else                                              // a longer window: the whole window again, from memory
        for (int64_t i = rc.b + tid; i < rc.len; i += BLOCK) {
            const int id = hist_at(a, rc, i);
            if (id >= 0 && id < a.V) count_id(id);
        }
    if (ovf) atomicOr(a.err, FS_DEVERR_COUNT_OVERFLOW);
    __syncthreads();
    const float rp = rc.p.repetition_penalty, fq = rc.p.frequency_penalty, pr = rc.p.presence_penalty;
#pragma unroll
    for (int j = 0; j < NV; ++j) {
        const int local = (j * BLOCK + tid) * 4;
        const uint2 c2 = *reinterpret_cast<const uint2*>(&s.cnt()[local >> 1]);
        if ((c2.x | c2.y) != 0u) {
            const uint32_t cc[4] = {c2.x & 0xFFFFu, c2.x >> 16, c2.y & 0xFFFFu, c2.y >> 16};
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                if (cc[q] != 0u) {
                    float l = x[4 * j + q];
                    if (rc.rep_on) l = l > 0.0f ? __fdiv_rn(l, rp) : __fmul_rn(l, rp);
                    if (rc.fp_on) l = __fsub_rn(l, __fadd_rn(__fmul_rn((float)cc[q], fq), pr));
                    x[4 * j + q] = l;
                }
            }
        }
    }
}

// The segment's window ids s.ids[0, nids) (nids <= WIDS, gathered by gather_window) reordered by tile, a counting
// sort: the ids of the segment's tile t are s.ids[t > 0 ? s.off[t - 1] : 0, s.off[t]) (s.off holds the bucket ends;
// ntiles <= 2 * BLOCK). Ends with a barrier.
__device__ __forceinline__ void bucket_window(int seg_lo, int ntiles, Shared& s) {
    const int tid = threadIdx.x;
    const int n = (int)s.nids;
    constexpr int Q = WIDS / BLOCK;
    int id[Q], tl[Q];
#pragma unroll
    for (int q = 0; q < Q; ++q) {
        const int i = tid + q * BLOCK;
        id[q] = i < n ? s.ids[i] : 0;
        tl[q] = i < n ? (id[q] - seg_lo) / TILE : -1;
    }
    for (int t = tid; t < ntiles; t += BLOCK) s.off[t] = 0u;
    __syncthreads();
#pragma unroll
    for (int q = 0; q < Q; ++q)
        if (tl[q] >= 0) atomicAdd(&s.off[tl[q]], 1u);
    __syncthreads();
    const uint32_t c0 = 2 * tid < ntiles ? s.off[2 * tid] : 0u;
    const uint32_t c1 = 2 * tid + 1 < ntiles ? s.off[2 * tid + 1] : 0u;
    uint32_t tot;
    const uint32_t base = block_excl_scan<uint32_t>(c0 + c1, s.wsum, &tot);   // its barriers end the reads above
    if (2 * tid < ntiles) s.off[2 * tid] = base;                              // bucket starts
    if (2 * tid + 1 < ntiles) s.off[2 * tid + 1] = base + c0;
    __syncthreads();
#pragma unroll
    for (int q = 0; q < Q; ++q)
        if (tl[q] >= 0) s.ids[atomicAdd(&s.off[tl[q]], 1u)] = id[q];         // the starts advance to the ends
    __syncthreads();
}

// Penalty pass on one tile (the tt-th of the segment, starting at lo) in registers, wave by wave: the ids of the
// tile's bucket (bucket_window) that fall on this wave's logits are counted in the wave's own 16-bit table, then
// each lane patches its counted logits. Element lo + e belongs to wave (e % (4 * BLOCK)) / (4 * WAVE), at index
// (e / (4 * BLOCK)) * 4 * WAVE + e % (4 * WAVE) of its table (lane l's four logits of float4 j sit at
// j * 4 * WAVE + 4 * l). A wave's LDS accesses complete in order, so no barrier is needed; tiles holding no window
// id skip the pass. Same arithmetic as apply_penalties.
__device__ __forceinline__ void wave_penalties(float (&x)[TPT], const RowCtx& rc, int lo, int tt, Shared& s) {
    static_assert(NV * 4 * WAVE * NWAVES == TILE, "a tile is the waves' float4 columns");
    static_assert(WIDS < 0xFFFF, "16-bit counts");
    const int b0 = tt > 0 ? (int)s.off[tt - 1] : 0, b1 = (int)s.off[tt];
    if (b0 == b1) return;                                // uniform: no window id in this tile
    const int lane = lane_id();
    const uint32_t w = threadIdx.x / WAVE;
    uint32_t* tb = s.cnt() + w * (NV * 4 * WAVE / 2);    // NV * 4 * WAVE 16-bit counts (all waves: TILE / 2 words)
    // Every table access is a 32-bit access of tb, with compiler barriers between the clear, the counts and the
    // reads: the hardware keeps a wave's LDS accesses in order, but vector-typed accesses are not ordered by the
    // compiler against the 32-bit atomics (no barrier here does it).
#pragma unroll
    for (int j = 0; j < NV; ++j) {
        tb[2 * (j * WAVE + lane)] = 0u;
        tb[2 * (j * WAVE + lane) + 1] = 0u;
    }
    __asm__ volatile("" ::: "memory");
    // at most WIDS ids in the segment: a 16-bit count cannot overflow
    for (int i = b0 + lane; i < b1; i += WAVE) {
        const uint32_t e = (uint32_t)(s.ids[i] - lo);   // < TILE
        if ((e % (4u * BLOCK)) / (4u * WAVE) == w) {
            const uint32_t idx = (e / (4u * BLOCK)) * (4u * WAVE) + e % (4u * WAVE);
            atomicAdd(&tb[idx >> 1], 1u << ((idx & 1u) * 16u));
        }
    }
    __asm__ volatile("" ::: "memory");
    const float rp = rc.p.repetition_penalty, fq = rc.p.frequency_penalty, pr = rc.p.presence_penalty;
#pragma unroll
    for (int j = 0; j < NV; ++j) {
        const uint2 c2 = make_uint2(tb[2 * (j * WAVE + lane)], tb[2 * (j * WAVE + lane) + 1]);
        if ((c2.x | c2.y) != 0u) {
            const uint32_t cc[4] = {c2.x & 0xFFFFu, c2.x >> 16, c2.y & 0xFFFFu, c2.y >> 16};
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                if (cc[q] != 0u) {
                    float l = x[4 * j + q];
                    if (rc.rep_on) l = l > 0.0f ? __fdiv_rn(l, rp) : __fmul_rn(l, rp);
                    if (rc.fp_on) l = __fsub_rn(l, __fadd_rn(__fmul_rn((float)cc[q], fq), pr));
                    x[4 * j + q] = l;
                }
            }
        }
    }
}

// The penalty window's ids in [seg_lo, seg_hi) into s.ids (s.nids counts past WIDS). Called with the segment's
// first tiles in flight; ends with a barrier.
__device__ __forceinline__ void gather_window(const Args& a, const RowCtx& rc, int seg_lo, int seg_hi, Shared& s) {
    const int tid = threadIdx.x;
    if (tid == 0) s.nids = 0u;
    __syncthreads();
    auto take = [&](int id) {
        const bool in = id >= seg_lo && id < seg_hi;
        const uint64_t m = __ballot(in);
        if (m != 0ull) {
            uint32_t base = 0u;
            if (lane_id() == 0) base = atomicAdd(&s.nids, (uint32_t)__popcll(m));
            base = (uint32_t)__builtin_amdgcn_readlane((int)base, 0);
            const uint32_t pos = base + mbcnt(m);
            if (in && pos < (uint32_t)WIDS) s.ids[pos] = id;
        }
    };
    // the first GW * BLOCK ids requested together (one round trip), the rest round by round
    constexpr int GW = 4;
    int idq[GW];
#pragma unroll
    for (int q = 0; q < GW; ++q) {
        const int64_t i = rc.b + q * BLOCK + tid;
        idq[q] = i < rc.len ? hist_at(a, rc, i) : -1;
    }
#pragma unroll
    for (int q = 0; q < GW; ++q) take(idq[q]);
    for (int64_t i0 = rc.b + GW * BLOCK; i0 < rc.len; i0 += BLOCK) {
        const int64_t i = i0 + tid;
        take(i < rc.len ? hist_at(a, rc, i) : -1);
    }
    __syncthreads();
}

// Narrow [rlo, rhi] onto the kk-th largest value among the entries a visitor yields (32-bit values, entries
// outside [rlo, rhi] ignored; count(value > rhi) == *above < kk <= count(value >= rlo) on entry). On return
// rlo == rhi is that value, *above = count(value > it), *at = count(value >= it).
template <class Each>
__device__ __forceinline__ void narrow32(Each each, int kk, uint32_t& rlo, uint32_t& rhi, uint32_t* above, uint32_t* at, Shared& s) {
    const int tid = threadIdx.x;
    for (int level = 0; level < 4 && rlo != rhi; ++level) {
        const int sh = range_shift(rlo, rhi);
        for (int i = tid; i < NBINS; i += BLOCK) s.bins()[i] = 0u;
        __syncthreads();
        const uint32_t lo = rlo, hi = rhi;
        each([&](uint32_t v) { if (v >= lo && v <= hi) atomicAdd(&s.bins()[(v - lo) >> sh], 1u); });
        __syncthreads();
        uint32_t ab, atb;
        const int bsel = hist_locate(s.bins(), kk - (int)*above, &ab, &atb, s.wsum, s.red);
        const uint64_t nlo = (uint64_t)rlo + ((uint64_t)bsel << sh);
        const uint64_t nhi = (uint64_t)rlo + (((uint64_t)bsel + 1) << sh) - 1;
        rlo = (uint32_t)nlo;
        rhi = nhi < rhi ? (uint32_t)nhi : rhi;
        *above += ab;
        *at = *above + (atb - ab);
    }
}

// Keeps the entries >= X of the n in s.cand (at the front, through the stage) and returns their count; when more
// than KMAX would remain, changes nothing and returns -1. Whole block; returns after a barrier.
__device__ __forceinline__ int keep_from(int n, uint64_t X, Shared& s) {
    const int tid = threadIdx.x;
    uint32_t mine = 0u;
    for (int i = tid; i < n; i += BLOCK) mine += s.cand[i] >= X ? 1u : 0u;
    uint32_t tot;
    uint32_t pos = block_excl_scan<uint32_t>(mine, s.wsum, &tot);
    if (tot > (uint32_t)KMAX) return -1;
    uint64_t* st = s.stage();
    for (int i = tid; i < n; i += BLOCK) {
        const uint64_t c = s.cand[i];
        if (c >= X) st[pos++] = c;
    }
    __syncthreads();
    for (uint32_t i = tid; i < tot; i += BLOCK) s.cand[i] = st[i];
    if (tid == 0) s.count = tot;
    __syncthreads();
    return (int)tot;
}

// Exact k-th largest composite X among the n > k candidates in s.cand, then keep exactly the k entries >= X.
// Returns X. Keys first (histogram levels over [min, max]), then, if the k-th key is tied, the ids among the ties.
__device__ __forceinline__ uint64_t compact_exact(int n, int k, Shared& s) {
    const int tid = threadIdx.x;
    uint32_t kmn = 0xFFFFFFFFu, kmx = 0u;
    for (int i = tid; i < n; i += BLOCK) {
        const uint32_t kk = comp_key(s.cand[i]);
        kmn = kk < kmn ? kk : kmn;
        kmx = kk > kmx ? kk : kmx;
    }
    block_minmax_u32(kmn, kmx, s.red);
    uint32_t rlo = kmn, rhi = kmx, above = 0u, at = (uint32_t)n;
    narrow32([&](auto&& f) { for (int i = tid; i < n; i += BLOCK) f(comp_key(s.cand[i])); }, k, rlo, rhi, &above, &at,
             s);
    const uint32_t t = rlo;                                   // the k-th key
    const uint32_t need = (uint32_t)k - above;                // ties at t that belong to the top k
    uint64_t X = (uint64_t)t << 32;
    if (at - above != need) {
        // the need-th largest low word (the need-th smallest id) among the entries with key t
        uint32_t lmn = 0xFFFFFFFFu, lmx = 0u;
        for (int i = tid; i < n; i += BLOCK) {
            const uint64_t c = s.cand[i];
            if (comp_key(c) == t) {
                const uint32_t lw = (uint32_t)c;
                lmn = lw < lmn ? lw : lmn;
                lmx = lw > lmx ? lw : lmx;
            }
        }
        block_minmax_u32(lmn, lmx, s.red);
        uint32_t ab2 = 0u, at2 = 0u;
        narrow32(
            [&](auto&& f) {
                for (int i = tid; i < n; i += BLOCK) {
                    const uint64_t c = s.cand[i];
                    if (comp_key(c) == t) f((uint32_t)c);
                }
            },
            (int)need, lmn, lmx, &ab2, &at2, s);
        X |= lmn;
    }
    (void)keep_from(n, X, s);                                 // exactly k entries are >= X
    return X;
}

// The merge of one row: gathers the segments' candidates, selects and sorts the row's top k, then softmax / min-p / top-p / draw (sampler.cpp:25-49).
// ------------------------------------------------------------------------------------------------ large k
// Rows that sample with k > KMAX candidates (top_k = 0 or > 2048; ferro's k = n / top_k, sampler.cpp:26) are handled
// by one workgroup with several streaming passes over the row (it stays in L2 / MALL after the first):
//   1. the max / min composite and the count of ordered (non-NaN) logits;
//   2. the k-th composite Xk (key histograms, then ids among ties), unless every logit is a candidate;
//   3. S = sum of exp((double)(float)(v - mx) / T) over the candidates (sampler.cpp:37-41);
//   4. min-p: pr = e / S is monotone in the logit, so the kept keys are found by a binary search over keys;
//   5. top-p and the draw: the first candidate (candidate order) whose cumulative mass reaches a target, by a
//      descent over fp64 mass histograms of the keys, then the j-th smallest id among the ties at the final key.
// Sums run in a different order than ferro's sequential loop (probabilities agree to ~1e-15 relative).
constexpr int LPF = 2;                    // tiles in flight per large-row pass
constexpr int MB = 256;                   // mass histogram bins

// One pass over the whole row, LPF tiles in flight, penalties applied (the window ids are in s.ids): g(x, lo) per
// tile, called by every thread (g may use barriers). Element i of a thread is elem_id(lo, i) when < V. The tiles are
// read through a buffer resource over the row (rounded up to whole float4s, which stay inside the row's ld-strided
// allocation): loads past it return zeros without a memory access, so every tile's successor is requested
// unconditionally and the compiler's memory-counter waits stay exact (consuming a tile waits for that tile only).
template <class G>
__device__ __forceinline__ void row_tiles(const Args& a, const RowCtx& rc, Shared& s, G g) {
    const int V = a.V;
    const float* rowp = a.logits + (int64_t)rc.row * a.ld;
    const int ntile = (V + TILE - 1) / TILE;
    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(rowp), (short)0,
                                                                        ((V + 3) & ~3) * 4, 0x00020000);
    float buf[LPF][TPT];
#pragma unroll
    for (int p = 0; p < LPF; ++p) load_seg_tile(buf[p], rs, p);
    for (int t0 = 0; t0 < ntile; t0 += LPF) {
#pragma unroll
        for (int p = 0; p < LPF; ++p) {
            const int t = t0 + p;
            float x[TPT];
#pragma unroll
            for (int i = 0; i < TPT; ++i) x[i] = buf[p][i];
            load_seg_tile(buf[p], rs, t + LPF);
            if (t < ntile) {
                if (rc.capped) softcap_vals(x, rc.p.softcap);
                if (rc.pen) {
                    __syncthreads();                 // the previous tile's table reads are done
                    apply_penalties(x, a, rc, t * TILE, s);
                }
                g(x, t * TILE);
            }
        }
    }
    __syncthreads();
}

// Per ordered element (non-NaN, id < V): f(x, key, composite).
template <class F>
__device__ __forceinline__ void row_elems(const Args& a, const RowCtx& rc, Shared& s, F f) {
    const int V = a.V;
    row_tiles(a, rc, s, [&](const float (&x)[TPT], int lo) {
#pragma unroll
        for (int i = 0; i < TPT; ++i) {
            const int e = elem_id(lo, i);
            if (e < V && x[i] == x[i]) {
                const uint32_t kq = key_of(x[i]);
                f(x[i], kq, comp_of(kq, (uint32_t)e));
            }
        }
    });
}

__device__ __forceinline__ double mass_of(float x, float mx, double Td) {
    const float d = x - mx;                    // fp32 subtraction, as ferro
    return exp((double)d / Td);
}

// The kk-th largest composite among the ordered elements with composite in [lo_c, hi_c) (1 <= kk <= their count;
// keys of that set span [klo, khi]).
__device__ __forceinline__ uint64_t large_kth(const Args& a, const RowCtx& rc, Shared& s, int kk, uint64_t lo_c, uint64_t hi_c,
                              uint32_t klo, uint32_t khi) {
    uint32_t rlo = klo, rhi = khi, above = 0u, at = 0u;
    narrow32([&](auto&& f) {
                 row_elems(a, rc, s, [&](float, uint32_t kq, uint64_t c) { if (c >= lo_c && c < hi_c) f(kq); });
             },
             kk, rlo, rhi, &above, &at, s);
    const uint32_t t = rlo;
    const uint32_t need = (uint32_t)kk - above;
    uint32_t lmn = 0xFFFFFFFFu - (uint32_t)(a.V - 1), lmx = 0xFFFFFFFFu;
    uint32_t ab2 = 0u, at2 = 0u;
    narrow32([&](auto&& f) {
                 row_elems(a, rc, s, [&](float, uint32_t kq, uint64_t c) {
                     if (kq == t && c >= lo_c && c < hi_c) f((uint32_t)c);
                 });
             },
             (int)need, lmn, lmx, &ab2, &at2, s);
    return ((uint64_t)t << 32) | lmn;
}

// The j-th smallest id among the ordered elements with key t and composite >= lo_c (their largest id if fewer
// than j): one id-ordered pass. Returns its composite (0: none).
__device__ __forceinline__ uint64_t large_pick(const Args& a, const RowCtx& rc, Shared& s, uint32_t t, uint64_t lo_c, uint32_t j) {
    const int tid = threadIdx.x;
    const int V = a.V;
    uint32_t running = 0u;                     // flagged elements in earlier tiles (uniform)
    uint64_t found = 0ull, last = ~0ull;
    row_tiles(a, rc, s, [&](const float (&x)[TPT], int lo) {
        bool f[TPT];
        uint32_t c0 = 0u, c1 = 0u;
#pragma unroll
        for (int i = 0; i < TPT; ++i) {
            const int e = elem_id(lo, i);
            f[i] = e < V && x[i] == x[i] && key_of(x[i]) == t && comp_of(t, (uint32_t)e) >= lo_c;
            if (f[i]) {
                if (i < 4) ++c0; else ++c1;
                const uint64_t c = comp_of(t, (uint32_t)e);
                last = c < last ? c : last;
            }
        }
        uint32_t tot;                          // ids in a tile: float4 0 of every thread, then float4 1
        const uint32_t pre = block_excl_scan<uint32_t>(c0 | (c1 << 16), s.wsum, &tot);
        uint32_t r0 = running + (pre & 0xFFFFu);
        uint32_t r1 = running + (tot & 0xFFFFu) + (pre >> 16);
#pragma unroll
        for (int i = 0; i < TPT; ++i) {
            if (f[i]) {
                const uint32_t rank = i < 4 ? r0++ : r1++;
                if (rank + 1u == j) found = comp_of(t, (uint32_t)elem_id(lo, i));
            }
        }
        running += (tot & 0xFFFFu) + (tot >> 16);
    });
    found = block_max_u64(found, s.red);
    last = block_min_u64(last, s.red);
    (void)tid;
    return found != 0ull ? found : (last != ~0ull ? last : 0ull);
}

// The first candidate, in candidate order among the ordered elements with composite >= lo_c, at which the
// cumulative mass reaches target (0: the total stays below it). Keys of that set span [klo, khi].
__device__ __forceinline__ uint64_t large_mass_select(const Args& a, const RowCtx& rc, Shared& s, double target, uint64_t lo_c,
                                      uint32_t klo, uint32_t khi, float mx, double Td) {
    const int tid = threadIdx.x;
    const int w = tid / WAVE;
    double* hd = reinterpret_cast<double*>(s.cand);          // [NWAVES][MB] per-wave masses
    uint32_t* hc = s.bins();                                  // [MB] counts
    double above = 0.0;
    while (klo != khi) {
        int sh = 0;
        while (((khi - klo) >> sh) >= (uint32_t)MB) ++sh;
        for (int i = tid; i < NWAVES * MB; i += BLOCK) hd[i] = 0.0;
        for (int i = tid; i < MB; i += BLOCK) hc[i] = 0u;
        __syncthreads();
        const uint32_t lo = klo, hi = khi;
        row_elems(a, rc, s, [&](float x, uint32_t kq, uint64_t c) {
            if (c >= lo_c && kq >= lo && kq <= hi) {
                const uint32_t b = (kq - lo) >> sh;
                atomicAdd(&hd[w * MB + b], mass_of(x, mx, Td));
                atomicAdd(&hc[b], 1u);
            }
        });
        // thread t < MB owns bin MB-1-t: cumulative from the top in a fixed order
        double m = 0.0;
        uint32_t cnt = 0u;
        if (tid < MB) {
            const int b = MB - 1 - tid;
#pragma unroll
            for (int q = 0; q < NWAVES; ++q) m += hd[q * MB + b];
            cnt = hc[b];
        }
        double tot;
        const double ex = block_excl_scan<double>(m, s.red.f64, &tot);
        const int hit = (tid < MB && cnt != 0u && above + ex + m >= target) ? tid : 0x7fffffff;
        const int first = block_min_i32(hit, s.red);
        if (first == 0x7fffffff) return 0ull;
        if (tid == first) s.red.dmisc[1] = ex;
        __syncthreads();
        above += s.red.dmisc[1];
        __syncthreads();
        const uint32_t b = (uint32_t)(MB - 1 - first);
        const uint64_t nlo = (uint64_t)klo + ((uint64_t)b << sh);
        const uint64_t nhi = (uint64_t)klo + (((uint64_t)b + 1) << sh) - 1;
        klo = (uint32_t)nlo;
        khi = nhi < khi ? (uint32_t)nhi : khi;
    }
    const double et = mass_of(val_of(klo), mx, Td);
    double jd = et > 0.0 ? ceil((target - above) / et) : 1.0;
    if (!(jd >= 1.0)) jd = 1.0;
    const uint32_t j = jd > 4294967295.0 ? 0xFFFFFFFFu : (uint32_t)jd;
    return large_pick(a, rc, s, klo, lo_c, j);
}

// The exact multi-pass selection (narrowing histograms over the keys; about 15 passes over the row): the fallback
// of large_row when a coarse-bin step does not apply. Sets the token and the kept count.
__device__ __forceinline__ void large_row_exact(const Args& a, const RowCtx& rc, Shared& s, int& tok_out, int& keep_out) {
    const int tid = threadIdx.x;
    const int row = rc.row;
    const fs_row_params& p = rc.p;
    // 1. extremes and count of the ordered elements
    uint64_t cmax = 0ull, cmin = ~0ull;
    uint32_t nv = 0u;
    row_elems(a, rc, s, [&](float, uint32_t, uint64_t c) {
        cmax = c > cmax ? c : cmax;
        cmin = c < cmin ? c : cmin;
        ++nv;
    });
    cmax = block_max_u64(cmax, s.red);
    cmin = block_min_u64(cmin, s.red);
    uint32_t ntot;
    (void)block_excl_scan<uint32_t>(nv, s.wsum, &ntot);
    if (ntot == 0u) {                         // every logit NaN: no order to sample from
        tok_out = 0;
        keep_out = 0;
        return;
    }
    const uint32_t kmax = comp_key(cmax);
    const float mx = val_of(kmax);
    const double Td = (double)p.temperature;
    // 2. the candidates: composites >= Xk
    const int keff = (uint32_t)rc.k < ntot ? rc.k : (int)ntot;
    const uint64_t Xk = (uint32_t)keff == ntot ? cmin : large_kth(a, rc, s, keff, 1ull, ~0ull, comp_key(cmin), kmax);
    const uint32_t kk = comp_key(Xk);
    // 3. the softmax denominator
    double part = 0.0;
    row_elems(a, rc, s, [&](float x, uint32_t, uint64_t c) { if (c >= Xk) part += mass_of(x, mx, Td); });
    const double S = block_sum_f64(part, s.red);
    if (S != S) {                             // an infinite maximum: every mass NaN, nothing cut, the draw falls
        tok_out = (int)comp_id(Xk);           // through to the last candidate (sampler.cpp:43-49)
        keep_out = keff;
        return;
    }
    // 4. min-p: the smallest key whose pr reaches pr[0] * min_p (pr[0] = 1 / S)
    uint64_t Xkeep = Xk;
    if (p.min_p > 0.0f) {
        const double thr = (1.0 / S) * (double)p.min_p;
        auto ok = [&](uint32_t key) { return mass_of(val_of(key), mx, Td) / S >= thr; };
        uint64_t Xm;
        if (!ok(kmax)) {
            Xm = cmax;                                  // keep >= 1
        } else {
            uint32_t lo = kk, hi = kmax;
            while (lo < hi) {
                const uint32_t mid = lo + ((hi - lo) >> 1);
                if (ok(mid)) hi = mid; else lo = mid + 1u;
            }
            Xm = (uint64_t)lo << 32;
        }
        Xkeep = Xm > Xkeep ? Xm : Xkeep;
    }
    // 5. top-p: the crossing candidate is the last one kept (sampler.cpp:44)
    if (p.top_p < 1.0f) {
        const uint64_t Xc = large_mass_select(a, rc, s, (double)p.top_p * S, Xk, kk, kmax, mx, Td);
        if (Xc != 0ull) Xkeep = Xc > Xkeep ? Xc : Xkeep;
    }
    // tot over the kept prefix, its size and its last candidate
    double tpart = 0.0;
    uint32_t kc = 0u;
    uint64_t clast = ~0ull;
    row_elems(a, rc, s, [&](float x, uint32_t, uint64_t c) {
        if (c >= Xkeep) {
            tpart += mass_of(x, mx, Td);
            ++kc;
            clast = c < clast ? c : clast;
        }
    });
    const double tot = block_sum_f64(tpart, s.red);
    uint32_t keep;
    (void)block_excl_scan<uint32_t>(kc, s.wsum, &keep);
    clast = block_min_u64(clast, s.red);
    // 6. the draw r = u * tot (sampler.cpp:45-49), in mass units
    const double u = row_u(a, row);
    uint64_t pick = large_mass_select(a, rc, s, u * tot + 0.0, Xkeep, comp_key(Xkeep), kmax, mx, Td);
    if (pick == 0ull) pick = clast;
    tok_out = (int)comp_id(pick);
    keep_out = (int)keep;
    (void)tid;
}

// Optional outputs of a large row: the first min(k, kcap) candidates in candidate order, KMAX at a time.
__device__ __forceinline__ void large_outputs(const Args& a, const RowCtx& rc, Shared& s, int keff, uint64_t Xk, uint32_t kk,
                                              uint32_t kmax, float mx, double Td, double S) {
    const int tid = threadIdx.x;
    const int row = rc.row;
    if (a.mode != MODE_VERIFY && a.kcap > 0 && (a.cand_ids || a.cand_probs)) {
        const int mtot = keff < a.kcap ? keff : a.kcap;
        uint64_t hi_c = ~0ull;                          // this chunk: composites in [Xc, hi_c)
        for (int done = 0; done < mtot;) {
            const int m = mtot - done < KMAX ? mtot - done : KMAX;
            const uint32_t khi = hi_c == ~0ull ? kmax : comp_key(hi_c - 1ull);
            const uint64_t Xc = done + m == keff ? Xk : large_kth(a, rc, s, m, Xk, hi_c, kk, khi);
            if (tid == 0) s.count = 0u;
            __syncthreads();
            const int V = a.V;
            row_tiles(a, rc, s, [&](const float (&x)[TPT], int lo) {
#pragma unroll
                for (int i = 0; i < TPT; ++i) {
                    const int e = elem_id(lo, i);
                    const bool in = e < V && x[i] == x[i] && comp_of(key_of(x[i]), (uint32_t)e) >= Xc &&
                                    comp_of(key_of(x[i]), (uint32_t)e) < hi_c;
                    wave_append(in, in ? comp_of(key_of(x[i]), (uint32_t)e) : 0ull, s.cand, &s.count, CAP);
                }
            });
            bin_sort_desc(m, s);
            for (int i = tid; i < m; i += BLOCK) {
                const uint64_t c = s.cand[i];
                const int64_t o = (int64_t)row * a.kcap + done + i;
                if (a.cand_ids) a.cand_ids[o] = (int32_t)comp_id(c);
                if (a.cand_probs) a.cand_probs[o] = mass_of(val_of(comp_key(c)), mx, Td) / S;
            }
            __syncthreads();
            done += m;
            hi_c = Xc;
        }
    }
}


// ---- large k through coarse key bins: a few passes instead of ~15
// Pass 1: extremes and a count histogram over LB coarse bins (key >> LB_SHIFT). Xk (the k-th composite, k < the
// count) is narrowed inside its coarse bin. Pass 2: S (a deterministic fp64 block sum, as the exact path) and a
// fixed-point mass histogram over the same bins (integer sums: deterministic, within 2^-44 per element). The bins'
// masses stay in registers (thread t: descending positions PT*t ..). The top-p and draw targets each pick a coarse
// bin from them; one pass gathers that bin's candidates into LDS, a counting sort orders them and the exact fp64
// masses are walked in candidate order from the bin's fixed-point "above" mass. A target that does not fall inside
// its bin's exact masses (a rounding step at the bin edge), or a bin of more than KMAX candidates, takes the exact
// multi-pass selection instead.
constexpr int LB_SHIFT = 32 - 12;
constexpr int LPT = LB / BLOCK;             // coarse bins per thread
constexpr double FXS = 17592186044416.0;    // 2^44: fixed-point mass scale (an element's mass is <= 1)
static_assert(LB * 8 <= CAP * 8, "the fixed-point mass histogram fits the candidate buffer");

// Smallest descending position d (bin LB-1-d) at which the running total from the top reaches target, given each
// thread's LPT values at positions LPT*t + j; *above = the total of the positions before d. -1: never reached.
template <class T>
__device__ __forceinline__ int desc_locate(const T (&v)[LPT], T target, T* above, T* wsum, Shared& s) {
    const int tid = threadIdx.x;
    T sum = T(0);
#pragma unroll
    for (int j = 0; j < LPT; ++j) sum += v[j];
    T tot;
    T run = block_excl_scan<T>(sum, wsum, &tot);
    int hit = 0x7fffffff;
    T ab = T(0);
#pragma unroll
    for (int j = 0; j < LPT; ++j) {
        if (hit == 0x7fffffff && v[j] != T(0) && run + v[j] >= target) {
            hit = LPT * tid + j;
            ab = run;
        }
        run += v[j];
    }
    const int d = block_min_i32(hit, s.red);
    if (d == 0x7fffffff) return -1;
    if (hit == d) s.red.u64b[0] = (uint64_t)ab;
    __syncthreads();
    *above = (T)s.red.u64b[0];
    __syncthreads();
    return d;
}
// Gathers the candidates (composite >= lo_c) of coarse bin b into s.cand[0, n) and sorts them; returns n, or -1
// when more than KMAX (the caller falls back). Extra per-element work f(x, key, composite) for every candidate.
template <class F>
__device__ __forceinline__ int large_gather_bin(const Args& a, const RowCtx& rc, Shared& s, uint32_t b, uint64_t lo_c, F f) {
    const int V = a.V;
    if (threadIdx.x == 0) s.count = 0u;
    __syncthreads();
    row_tiles(a, rc, s, [&](const float (&x)[TPT], int lo) {
#pragma unroll
        for (int i = 0; i < TPT; ++i) {
            const int e = elem_id(lo, i);
            const bool ok = e < V && x[i] == x[i];
            const uint32_t kq = key_of(x[i]);
            const uint64_t c = comp_of(kq, (uint32_t)e);
            const bool cand = ok && c >= lo_c;
            if (cand) f(x[i], kq, c);
            const bool in = cand && (kq >> LB_SHIFT) == b;
            wave_append(in, c, s.cand, &s.count, KMAX);
        }
    });
    const int n = (int)s.count;                       // row_tiles ends with a barrier
    if (n > KMAX) return -1;
    bin_sort_desc(n, s);
    return n;
}

// The first of the n sorted entries s.cand[0, n) with composite >= lo_c at which above + the running exact mass
// reaches target: its index, and the running mass there in *cum. -1: above >= target (the crossing lies in a higher
// bin); -2: the bin's masses end below target.
__device__ __forceinline__ int large_walk(Shared& s, int n, uint64_t lo_c, double above, double target, float mx, double Td,
                                          double* cum) {
    const int i0 = (int)threadIdx.x * KPT;
    if (!(above < target)) return -1;
    double e[KPT], run = 0.0;
#pragma unroll
    for (int q = 0; q < KPT; ++q) {
        const int i = i0 + q;
        e[q] = (i < n && s.cand[i] >= lo_c) ? mass_of(val_of(comp_key(s.cand[i])), mx, Td) : 0.0;
        run += e[q];
    }
    double tot;
    const double off = block_excl_scan<double>(run, s.red.f64, &tot);
    double c = above + off;
    int hit = 0x7fffffff;
    double ch = 0.0;
#pragma unroll
    for (int q = 0; q < KPT; ++q) {
        c += e[q];
        if (hit == 0x7fffffff && i0 + q < n && e[q] > 0.0 && c >= target) { hit = i0 + q; ch = c; }
    }
    const int first = block_min_i32(hit, s.red);
    if (first == 0x7fffffff) return -2;
    if (hit == first) s.red.dmisc[2] = ch;
    __syncthreads();
    *cum = s.red.dmisc[2];
    __syncthreads();
    return first;
}

// What a large row's optional candidate outputs need (large_outputs), left by large_row or large_segment.
struct LargeOut {
    bool valid;
    int keff;
    uint64_t Xk;
    uint32_t kmax;
    double S;
};

// The whole large-k sample of one row: token and kept count; lo describes the candidates for the optional outputs.
__device__ __forceinline__ void large_row(const Args& a, const RowCtx& rc, Shared& s, int& tok_out, int& keep_out,
                                          LargeOut& lo) {
    lo.valid = false;
    const int tid = threadIdx.x;
    const int row = rc.row;
    const fs_row_params& p = rc.p;
    if (rc.pen) gather_window(a, rc, 0, a.V, s);
    // 1. extremes, count of the ordered elements, their coarse-bin counts (only needed to find the k-th when k < V:
    //    k >= V takes every ordered logit)
    uint32_t* hc = reinterpret_cast<uint32_t*>(s.cand);
    const bool need_kth = rc.k < a.V;
    for (int i = tid; i < LB; i += BLOCK) hc[i] = 0u;
    __syncthreads();
    uint64_t cmax = 0ull, cmin = ~0ull;
    uint32_t nv = 0u;
    row_elems(a, rc, s, [&](float, uint32_t kq, uint64_t c) {
        cmax = c > cmax ? c : cmax;
        cmin = c < cmin ? c : cmin;
        ++nv;
        if (need_kth) atomicAdd(&hc[kq >> LB_SHIFT], 1u);
    });
    cmax = block_max_u64(cmax, s.red);
    cmin = block_min_u64(cmin, s.red);
    uint32_t ntot;
    (void)block_excl_scan<uint32_t>(nv, s.wsum, &ntot);
    if (ntot == 0u) {                         // every logit NaN: no order to sample from
        tok_out = 0;
        keep_out = rc.greedy ? 1 : 0;
        return;
    }
    const uint32_t kmax = comp_key(cmax);
    const float mx = val_of(kmax);
    if (rc.greedy) {                          // ferro's scan (sampler.cpp:19-23): the first maximum above -inf,
        tok_out = mx > -__builtin_huge_valf() ? (int)comp_id(cmax) : 0;       // never moving off a NaN at index 0
        if (ld_const(a.logits + (int64_t)row * a.ld) != ld_const(a.logits + (int64_t)row * a.ld)) tok_out = 0;
        keep_out = 1;
        if (tid == 0 && a.mode != MODE_VERIFY && a.kcap > 0) {
            if (a.cand_ids) a.cand_ids[(int64_t)row * a.kcap] = tok_out;
            if (a.cand_probs) a.cand_probs[(int64_t)row * a.kcap] = 1.0;
        }
        return;
    }
    const double Td = (double)p.temperature;
    const int keff = (uint32_t)rc.k < ntot ? rc.k : (int)ntot;
    uint64_t Xk = cmin;
    if ((uint32_t)keff < ntot) {                          // the k-th composite, inside its coarse bin
        uint32_t cv[LPT];
#pragma unroll
        for (int j = 0; j < LPT; ++j) cv[j] = hc[LB - 1 - (LPT * tid + j)];
        uint32_t abk = 0u;
        const int dk = desc_locate<uint32_t>(cv, (uint32_t)keff, &abk, s.wsum, s);
        const uint32_t bk = (uint32_t)(LB - 1 - dk);
        const uint32_t blo = bk << LB_SHIFT, bhi = blo | ((1u << LB_SHIFT) - 1u);
        Xk = large_kth(a, rc, s, keff - (int)abk, 1ull, ~0ull, blo, bhi);
    }
    const uint32_t kk = comp_key(Xk);
    // 2. S and the fixed-point mass histogram of the candidates
    uint64_t* hm = reinterpret_cast<uint64_t*>(s.cand);
    for (int i = tid; i < LB; i += BLOCK) hm[i] = 0ull;
    __syncthreads();
    double part = 0.0;
    row_elems(a, rc, s, [&](float x, uint32_t kq, uint64_t c) {
        if (c >= Xk) {
            const double m = mass_of(x, mx, Td);
            part += m;
            atomicAdd(reinterpret_cast<unsigned long long*>(&hm[kq >> LB_SHIFT]), (unsigned long long)(m * FXS + 0.5));
        }
    });
    const double S = block_sum_f64(part, s.red);          // its barriers also complete the histogram
    if (S != S) {                                         // an infinite maximum: every mass NaN, nothing cut, the
        lo.valid = true; lo.keff = keff; lo.Xk = Xk; lo.kmax = kmax; lo.S = S;   // draw falls through to the last
        tok_out = (int)comp_id(Xk);                       // candidate (sampler.cpp:43-49)
        keep_out = keff;
        return;
    }
    uint64_t mv[LPT];
#pragma unroll
    for (int j = 0; j < LPT; ++j) mv[j] = hm[LB - 1 - (LPT * tid + j)];
    __syncthreads();                                      // the candidate buffer is reused below
    // 3. min-p: the smallest key whose pr reaches pr[0] * min_p (pr[0] = 1 / S)
    bool ok_fast = true;
    uint64_t Xm = 0ull;
    uint32_t km = 0xFFFFFFFFu;
    if (p.min_p > 0.0f) {
        const double thr = (1.0 / S) * (double)p.min_p;
        auto ok = [&](uint32_t key) { return mass_of(val_of(key), mx, Td) / S >= thr; };
        if (!ok(kmax)) {
            Xm = cmax;                                    // keep >= 1
        } else {
            uint32_t lo = kk, hi = kmax;
            while (lo < hi) {
                const uint32_t mid = lo + ((hi - lo) >> 1);
                if (ok(mid)) hi = mid; else lo = mid + 1u;
            }
            km = lo;
            Xm = (uint64_t)lo << 32;
        }
    }
    // 4. top-p's crossing bin, gathered with the min-p counts and masses
    uint64_t Xc = 0ull;
    uint32_t keep_c = 0u;
    double tot_c = 0.0;
    int nc = -1;                                          // top-p's bin, sorted in s.cand (-1: none)
    uint32_t bc = 0u;
    double above_c = 0.0;
    uint32_t cnt_m = 0u, ca_c = 0u;
    double sum_m = 0.0;
    uint64_t cl_m = ~0ull;
    const bool need_m = p.min_p > 0.0f && Xm != cmax;
    if (p.top_p < 1.0f || need_m) {
        const double tgt = (double)p.top_p * S;
        uint64_t abfx = 0ull;
        int dc = -1;
        if (p.top_p < 1.0f) {
            dc = desc_locate<uint64_t>(mv, (uint64_t)(tgt * FXS), &abfx, s.red.u64b, s);
            if (dc < 0) dc = LB - 1 - (int)(kk >> LB_SHIFT);     // the total rounds below the target: last bin
            bc = (uint32_t)(LB - 1 - dc);
            above_c = (double)abfx / FXS;
        }
        const uint32_t bsel = p.top_p < 1.0f ? bc : 0xFFFFFFFFu;
        uint32_t my_ca = 0u, my_cm = 0u;
        double my_sm = 0.0;
        uint64_t my_cl = ~0ull;
        nc = large_gather_bin(a, rc, s, bsel, Xk, [&](float x, uint32_t kq, uint64_t c) {
            if ((kq >> LB_SHIFT) > bsel && bsel != 0xFFFFFFFFu) ++my_ca;
            if (need_m && kq >= km) {
                ++my_cm;
                my_sm += mass_of(x, mx, Td);
                my_cl = c < my_cl ? c : my_cl;
            }
        });
        (void)block_excl_scan<uint32_t>(my_ca, s.wsum, &ca_c);
        if (need_m) {
            (void)block_excl_scan<uint32_t>(my_cm, s.wsum, &cnt_m);
            sum_m = block_sum_f64(my_sm, s.red);
            cl_m = block_min_u64(my_cl, s.red);
        }
        if (p.top_p < 1.0f) {
            if (nc < 0) {
                ok_fast = false;
            } else {
                double cum = 0.0;
                const int ic = large_walk(s, nc, Xk, above_c, tgt, mx, Td, &cum);
                if (ic < 0) {
                    ok_fast = false;
                } else {
                    Xc = s.cand[ic];
                    keep_c = ca_c + (uint32_t)ic + 1u;
                    tot_c = cum;
                }
            }
        }
    }
    lo.valid = true; lo.keff = keff; lo.Xk = Xk; lo.kmax = kmax; lo.S = S;
    if (!ok_fast) {
        large_row_exact(a, rc, s, tok_out, keep_out);
        return;
    }
    // the kept prefix: the largest of the three thresholds (sampler.cpp:43-44)
    uint64_t Xkeep = Xk, clast = Xk;
    uint32_t keep = (uint32_t)keff;
    double tot = S;
    if (p.min_p > 0.0f && Xm > Xkeep) {
        Xkeep = Xm;
        if (Xm == cmax) { keep = 1u; tot = 1.0; clast = cmax; }   // mass_of(mx) = exp(0)
        else { keep = cnt_m; tot = sum_m; clast = cl_m; }
    }
    if (p.top_p < 1.0f && Xc > Xkeep) {
        Xkeep = Xc;
        keep = keep_c;
        tot = tot_c;
        clast = Xc;
    }
    // 5. the draw r = u * tot (sampler.cpp:45-49), in mass units
    const double u = row_u(a, row);
    const double r = u * tot + 0.0;
    uint64_t abd = 0ull;
    int dd = desc_locate<uint64_t>(mv, (uint64_t)(r * FXS), &abd, s.red.u64b, s);
    uint64_t pick = 0ull;
    bool drawn = false;
    if (dd >= 0) {
        const uint32_t bd = (uint32_t)(LB - 1 - dd);
        int nd = -1;
        if (nc >= 0 && bd == bc && p.top_p < 1.0f) {
            nd = nc;                                          // the same bin is in LDS already
        } else {
            nd = large_gather_bin(a, rc, s, bd, Xkeep, [&](float, uint32_t, uint64_t) {});
        }
        if (nd >= 0) {
            double cum = 0.0;
            const int id = large_walk(s, nd, Xkeep, (double)abd / FXS, r, mx, Td, &cum);
            if (id >= 0) {
                pick = s.cand[id];
                drawn = true;
            } else if (id == -2 && comp_key(Xkeep) >> LB_SHIFT == bd) {
                drawn = true;                                 // past the last kept candidate: clast
            }
        }
    }
    if (!drawn) pick = large_mass_select(a, rc, s, r, Xkeep, comp_key(Xkeep), kmax, mx, Td);
    if (pick == 0ull) pick = clast;
    tok_out = (int)comp_id(pick);
    keep_out = (int)keep;
}

// Large rows sampled by their segments together (large_segment, below): the list slot's scalars and the row barrier.
// Slot layout: each phase's scalars in a 128-byte line of their own, then three gather regions of whole lines. A
// segment reads another segment's line only after the barrier that follows its writing, and never earlier in the
// call, so no line it reads can be stale in its L1.
constexpr int LLINE = 16;                      // composites per 128-byte line
constexpr int LSC = 5 * LLINE;                 // scalar lines at the head of a large-row segment's list slot
constexpr int LLR = ((CAP - LSC) / 3) / LLINE * LLINE;   // capacity of each of its three gather regions
enum LargeSlot : int {
    LS_MAX = 0, LS_MIN, LS_NV,                                   // P1: largest / smallest composite, ordered count
    LS_FN, LS_FC, LS_FT,                                         // P1, every token a candidate: the cut's list count,
                                                                 // its fp64 mass and the rest's (both relative to LS_MAX)
    LS_SHI = LLINE, LS_NBK,                                      // P2: fp64 mass of the candidates above bk; bin bk's count
    LS_NBC = 2 * LLINE, LS_CA, LS_CNTM, LS_SUMM, LS_CLM,         // P3: bin bc's count, candidates above bc, min-p's
    LS_NBD = 3 * LLINE,                                          // P4: bin bd's count
    LS_TOK = 4 * LLINE, LS_XK, LS_S, LS_KEFF, LS_STATUS          // segment 0: token | keep << 32, Xk, S, keff | kmax << 32, 1 = done
};
static_assert(LS_STATUS < LSC, "the scalars fit the slot head");
static_assert(LSC + 3 * LLR <= CAP, "three gather regions after the scalars");

// The row barrier counter: the row histogram's bin RBINS - 2, above every ordered key (bins <= 4088) like the
// completion counter. Low 15 bits: arrivals; bit 15: the row is abandoned.
__device__ __forceinline__ uint32_t* row_sync_ctr(const Args& a, int row) {
    return a.rhist + (int64_t)row * RBINS + (RBINS - 2);
}
constexpr uint32_t ROW_ABANDONED = 0x8000u;
__device__ __forceinline__ void row_abandon(const Args& a, int row) {
    if (threadIdx.x == 0) __hip_atomic_fetch_or(row_sync_ctr(a, row), ROW_ABANDONED, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
// ------------------------------------------------------------------------------------------------ one-wave finish
// For k <= 64 once the block has narrowed the row to c1 <= 128 candidates (composites, all distinct, containing the
// top k) and ranked them (block_ranks): wave 0 places them (lane i = candidate i in ferro's order) and runs the
// softmax / min-p / top-p / draw of sampler.cpp:37-49, the sums as DPP wave scans in candidate order. LDS accesses
// of one wave are ordered, so no further block barrier is needed: the other waves go straight to the epilogue.

// Ranks of the c1 <= 128 candidates in[0, c1) (whole block, one barrier): thread t compares candidate t % 128
// with a quarter of the list; rk[q*128 + e] is candidate e's count of larger entries in quarter q. Pads in[c1, 128)
// with 0 first. Returns after a barrier.
__device__ __forceinline__ void block_ranks(uint64_t* in, int c1, uint32_t* rk) {
    const int tid = threadIdx.x;
    if (tid >= c1 && tid < 2 * WAVE) in[tid] = 0ull;
    __syncthreads();
    const int e = tid & (2 * WAVE - 1), q = tid / (2 * WAVE);
    const uint64_t me = in[e];
    int r = 0;
#pragma unroll
    for (int j = 0; j < 2 * WAVE / 4; ++j) r += in[q * (2 * WAVE / 4) + j] > me ? 1 : 0;
    rk[q * 2 * WAVE + e] = (uint32_t)r;
    __syncthreads();
}
static_assert(BLOCK == 4 * 2 * WAVE, "block_ranks splits 128 candidates into four quarters");

__device__ __forceinline__ void wave_finish(const Args& a, const RowCtx& rc, const uint64_t* in, const uint32_t* rk,
                                            int k, double u, double* wbuf, int& tok_out, int& keep_out) {
    const int lane = lane_id();
    const int row = rc.row;
    // lane holds candidates lane and lane + 64 (0 = none) with their ranks from block_ranks
    const uint64_t m0 = in[lane], m1 = in[lane + WAVE];
    int r0 = 0, r1 = 0;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        r0 += (int)rk[q * 2 * WAVE + lane];
        r1 += (int)rk[q * 2 * WAVE + lane + WAVE];
    }
    uint64_t* sorted = reinterpret_cast<uint64_t*>(wbuf) + WAVE;     // [WAVE] after the [WAVE] doubles
    if (m0 != 0ull && r0 < k) sorted[r0] = m0;
    if (m1 != 0ull && r1 < k) sorted[r1] = m1;
    const uint64_t v = lane < k ? sorted[lane] : 0ull;               // candidate `lane` in ferro's order
    // softmax at temperature, min-p, top-p, draw (sampler.cpp:37-49)
    const fs_row_params& p = rc.p;
    const float mx = val_of(comp_key(sorted[0]));
    const double Td = (double)p.temperature;
    double e = 0.0;
    if (lane < k) {
        const float d = val_of(comp_key(v)) - mx;        // fp32 subtraction, as ferro
        e = exp((double)d / Td);
    }
    const double sum = lane_f64(wave_scan_f64(e), WAVE - 1);   // lanes >= k hold 0
    const double pr = e / sum;
    const double cum = wave_scan_f64(pr);                 // ferro's running c (sampler.cpp:44,47)
    int keep_m = k;
    if (p.min_p > 0.0f) {                                 // keep = 1 + the last index not below pr[0]*min_p (NaN masses stay)
        const double thr = lane_f64(pr, 0) * (double)p.min_p;
        const uint64_t mm = __ballot(lane < k && !(pr < thr));
        keep_m = mm ? 64 - __clzll((long long)mm) : 1;
    }
    int keep = keep_m;
    if (p.top_p < 1.0f) {
        const uint64_t mm = __ballot(lane < keep_m && cum >= (double)p.top_p);
        if (mm) {
            const int first = __ffsll((unsigned long long)mm) - 1;
            keep = first + 1 < keep_m ? first + 1 : keep_m;
        }
    }
    const double tot = lane_f64(cum, keep - 1);
    const double rr = u * tot + 0.0;
    const uint64_t hm = __ballot(lane < keep && rr <= cum);
    const int at = hm ? __ffsll((unsigned long long)hm) - 1 : keep - 1;
    tok_out = (int)comp_id(sorted[at]);
    keep_out = keep;
    if (a.mode != MODE_VERIFY) {
        const int m = k < a.kcap ? k : a.kcap;
        if (lane < m) {
            if (a.cand_ids) a.cand_ids[(int64_t)row * a.kcap + lane] = (int32_t)comp_id(v);
            if (a.cand_probs) a.cand_probs[(int64_t)row * a.kcap + lane] = pr;
        }
    }
}

// The segment lists of a row, loaded at the merge kernel's entry (before the row's parameters, whose latency they
// overlap): tps threads per list, each holding the list's meta and SPEC entries r_me, r_me + tps, ... (entries past
// the list's count are stale and masked once the counts are known).
struct Pre {
    int tps, c_me, r_me;
    bool act;
    uint32_t t0m, cnm;
    uint64_t v[SPEC];
    double u;                              // the row's draw (requested with the lists)
    float l0;                              // the row's first logit (a NaN there is ferro's greedy answer)
};

__device__ __forceinline__ void prefetch_lists(const Args& a, const RowCtx& rc, Pre& pre) {
    const int row = rc.row;
    const int nseg = rc.nseg;
    const int tid = threadIdx.x;
    pre.tps = nseg > 0 ? BLOCK / nseg : 0;    // >= 1: the host keeps nseg < BLOCK
    pre.c_me = nseg > 0 ? tid % nseg : 0;
    pre.r_me = nseg > 0 ? tid / nseg : 0;
    pre.act = nseg > 0 && pre.r_me < pre.tps;
    const int64_t slot = slot_of(rc, pre.c_me);
    const uint64_t* lst = a.cand + slot * CAP;
    pre.u = row_u(a, row);
    pre.l0 = ld_const(a.logits + (int64_t)row * a.ld);
    pre.t0m = 0u;
    pre.cnm = 0u;
    if (nseg > 0) {
        pre.t0m = a.meta[2 * slot];
        pre.cnm = a.meta[2 * slot + 1];
    }
#pragma unroll
    for (int q = 0; q < SPEC; ++q) pre.v[q] = nseg > 0 ? lst[pre.act ? pre.r_me + q * pre.tps : 0] : 0ull;
}

// The short merge: rows with no partial tail tile whose segment lists lie inside the prefetched windows.
//   - greedy rows: the largest of the segments' maxima (wave 0; lanes < nseg hold entry 0 of every list);
//   - k <= WAVE: the candidates at or above L (the largest of the lists' bounds; at least k of the row's logits reach
//     every bound) go into LDS (one LDS atomic per wave); when there are at most 2 * BLOCK / 4 of them the block ranks
//     them (P threads per candidate, each comparing with 1/P of the list), places the first k by rank, and wave 0
//     finishes the row.
// Returns false, after a barrier and with nothing written, when the row does not fit (the general merge then runs).
constexpr int FRANK = BLOCK / 2;          // largest candidate count the short merge ranks
__device__ __forceinline__ bool merge_fast(const Args& a, const RowCtx& rc, Shared& s, const Pre& pre, int& tok,
                                           int& keep) {
    const int tid = threadIdx.x;
    const int k = rc.k;
    if (rc.nseg > FAST_SEGS) return false;
    const uint32_t cmax = wave_max(pre.cnm);
    if (cmax > (uint32_t)(SPEC * pre.tps)) return false;        // uniform: every wave holds every list's meta
    if (rc.greedy) {
        if (tid < WAVE) {
            uint64_t best = (pre.act && pre.r_me == 0) ? pre.v[0] : 0ull;   // each segment's best (entry 0)
            best = wave_max(best);
            tok = best != 0ull ? (int)comp_id(best) : 0;      // nothing above -inf / NaN: ferro's scan stays at 0
            if (pre.l0 != pre.l0) tok = 0;                    // ferro's scan never moves off a NaN at index 0
            keep = 1;
            if (tid == 0 && a.mode != MODE_VERIFY) {
                if (a.cand_ids && a.kcap > 0) a.cand_ids[(int64_t)rc.row * a.kcap] = tok;
                if (a.cand_probs && a.kcap > 0) a.cand_probs[(int64_t)rc.row * a.kcap] = 1.0;
            }
        }
        return true;
    }
    if (k > WAVE) return false;
    const uint32_t L = wave_max(pre.t0m);
    // the candidates >= L into LDS: one atomic per wave for all of a thread's entries
    {
        uint64_t bal[SPEC];
        uint32_t tot = 0u;
#pragma unroll
        for (int q = 0; q < SPEC; ++q) {
            const uint64_t w = pre.v[q];
            const bool in = pre.act && (uint32_t)(pre.r_me + q * pre.tps) < pre.cnm && w != 0ull && comp_key(w) >= L;
            bal[q] = __ballot(in);
            tot += (uint32_t)__popcll(bal[q]);
        }
        if (tid == 0) s.count = 0u;
        __syncthreads();
        if (tot != 0u) {
            uint32_t base = 0u;
            if (lane_id() == 0) base = atomicAdd(&s.count, tot);
            base = (uint32_t)__builtin_amdgcn_readlane((int)base, 0);
#pragma unroll
            for (int q = 0; q < SPEC; ++q) {
                if ((bal[q] >> lane_id()) & 1ull) s.cand[base + mbcnt(bal[q])] = pre.v[q];
                base += (uint32_t)__popcll(bal[q]);
            }
        }
    }
    __syncthreads();
    FS_MARK(2);
    const int n = (int)s.count;
    if (n < k || n > FRANK) {                                    // uniform
        __syncthreads();
        return false;
    }
    // ranks: P threads per candidate (c = tid % per), part q compares candidate c with entries [q*span, (q+1)*span)
    const int P = n <= BLOCK / 4 ? 4 : 2;
    const int per = BLOCK / P;
    const int span = (n + P - 1) / P;
    const int c = tid % per, q = tid / per;
    uint32_t* rk = reinterpret_cast<uint32_t*>(s.cand + FRANK);            // [BLOCK]
    uint64_t* sorted = s.cand + FRANK + BLOCK / 2;                        // [WAVE]
    if (c < n) {
        const uint64_t me = s.cand[c];
        const int j0 = q * span, j1 = j0 + span < n ? j0 + span : n;
        uint32_t r = 0u;
        int j = j0;
        for (; j + 4 <= j1; j += 4) {                  // four LDS reads in flight per step
            const uint64_t e0 = s.cand[j], e1 = s.cand[j + 1], e2 = s.cand[j + 2], e3 = s.cand[j + 3];
            r += (e0 > me ? 1u : 0u) + (e1 > me ? 1u : 0u) + (e2 > me ? 1u : 0u) + (e3 > me ? 1u : 0u);
        }
        for (; j < j1; ++j) r += s.cand[j] > me ? 1u : 0u;
        rk[q * per + c] = r;
    }
    __syncthreads();
    if (tid < n) {
        uint32_t r = 0u;
        for (int qq = 0; qq < P; ++qq) r += rk[qq * per + tid];
        if (r < (uint32_t)k) sorted[r] = s.cand[tid];
    }
    __syncthreads();
    FS_MARK(3);
    if (tid < WAVE) wave_softmax(a, rc, tid < k ? sorted[tid] : 0ull, k, pre.u, tok, keep);
    return true;
}

// ------------------------------------------------------------------------------------------------ decode step
// fs_decode_step's two additions to a row's merge (server.cpp:603-606, then gen_token's hist.push_back,
// server.cpp:342): its stream's history copied to the new histories (while the merge waits for its segments) and
// the token appended after it; and the row's draw committed (its stream advanced) once every reader is done.
// Stream s = row s; the new histories start at 0 and each stream gains one id (fs_hist_append's layout).
__device__ __forceinline__ void decode_hist_copy(const Args& a, int row) {
    if (!a.out_hist_off) return;
    const int64_t h0 = a.hist_off ? a.hist_off[0] : 0, b = a.hist_off ? a.hist_off[row] : 0;
    const int64_t e = a.hist_off ? a.hist_off[row + 1] : 0;
    const int64_t nb = b - h0 + row;
    for (int64_t i = threadIdx.x; i < e - b; i += BLOCK)
        if (nb + i < a.out_cap) a.out_hist[nb + i] = a.hist[b + i];
    if (threadIdx.x == 0) {
        a.out_hist_off[row] = nb;
        if (row == a.B - 1) a.out_hist_off[a.B] = e - h0 + a.B;
        if (nb + (e - b) + 1 > a.out_cap) atomicOr(a.err, FS_DEVERR_HIST_APPEND);
    }
}
__device__ __forceinline__ void decode_commit(const Args& a, const RowCtx& rc, Shared& s, int tok) {
    const int row = rc.row, t = threadIdx.x;
    if (a.out_hist_off && t == 0) {
        const int64_t h0 = a.hist_off ? a.hist_off[0] : 0, b = a.hist_off ? a.hist_off[row] : 0;
        const int64_t e = a.hist_off ? a.hist_off[row + 1] : 0;
        const int64_t at = b - h0 + row + (e - b);
        if (at < a.out_cap) a.out_hist[at] = tok;
    }
    if (!a.dmt || !samples(rc.p)) return;                // uniform; greedy rows draw nothing (sampler.cpp:19-23)
    uint64_t* mt = a.dmt + (int64_t)row * MT_N;
    const int idx = a.didx[row];
    if (idx < MT_N) {
        if (t == 0) a.didx[row] = idx + 1;
        return;
    }
    // the state's twist (the draw was its first value), in LDS: entries k < N - M need old values only, the others
    // the new ones below N - M and their own old neighbour (entry N - 1: the new entry 0)
    uint64_t* w = s.cand;
    __syncthreads();
    if (t < MT_N) w[t] = mt[t];
    __syncthreads();
    uint64_t nv = 0ull;
    if (t < MT_N - MT_M) nv = mt_twist_one(w[t], w[t + 1], w[t + MT_M]);
    __syncthreads();
    if (t < MT_N - MT_M) w[t] = nv;
    __syncthreads();
    if (t >= MT_N - MT_M && t < MT_N) nv = mt_twist_one(w[t], w[(t + 1) % MT_N], w[t - (MT_N - MT_M)]);
    __syncthreads();
    if (t >= MT_N - MT_M && t < MT_N) w[t] = nv;
    __syncthreads();
    if (t < MT_N) mt[t] = w[t];
    if (t == 0) a.didx[row] = 1;
}

__device__ __forceinline__ void merge_row(const Args& a, const RowCtx& rc, Shared& s, const Pre& pre, bool alone = false) {
    const int tid = threadIdx.x;
    const int row = rc.row;
    const int V = a.V;
    const int nseg = rc.nseg;
    const int tail_lo = (V / TILE) * TILE;            // the segment kernel streamed [0, tail_lo)
    const int ntail = V - tail_lo;                    // < TILE logits left for this kernel
    int k = rc.k;
    (void)nseg;
    int tok = 0, keep = 1;

    bool fast = false;
    LargeOut lo;
    lo.valid = false;
    bool whole = rc.large || alone;                   // sampled as a whole row: by the segments together or here
    bool from_segs = false;
    bool cut_done = false;                            // sampled by large_cut: the histograms were never touched
    if (rc.large && !alone && nseg > 0) {
        // the row's segments sampled it together (large_segment): segment 0's slot holds the result unless the row
        // was abandoned (then it is sampled here alone, exactly)
        const uint64_t* s0 = a.cand + slot_of(rc, 0) * CAP;
        const uint32_t sc = *reinterpret_cast<volatile const uint32_t*>(row_sync_ctr(a, row));   // not read before
        if (!(sc & ROW_ABANDONED) && s0[LS_STATUS] != 0ull) {
            cut_done = s0[LS_STATUS] == 2ull;
            const uint64_t tk = s0[LS_TOK];
            tok = (int)(uint32_t)tk;
            keep = (int)(tk >> 32);
            const uint64_t kw = s0[LS_KEFF];
            lo.valid = keep > 0;
            lo.keff = (int)(uint32_t)kw;
            lo.Xk = s0[LS_XK];
            lo.kmax = (uint32_t)(kw >> 32);
            lo.S = __longlong_as_double((long long)s0[LS_S]);
            from_segs = true;
        }
    }
    if (whole) {
        if (!from_segs) large_row(a, rc, s, tok, keep, lo);          // from the logits alone
        if (lo.valid && a.mode != MODE_VERIFY && a.kcap > 0 && (a.cand_ids || a.cand_probs)) {
            if (rc.pen && from_segs) gather_window(a, rc, 0, a.V, s);   // the output passes apply the penalties
            large_outputs(a, rc, s, lo.keff, lo.Xk, comp_key(lo.Xk), lo.kmax, val_of(lo.kmax),
                          (double)rc.p.temperature, lo.S);
        }
    } else if (ntail == 0 && (fast = merge_fast(a, rc, s, pre, tok, keep))) {
        // the short merge wrote the row's outputs
    } else {
    // ---- the row's tail: loads first, then its penalty pass (the same arithmetic as the segment kernel)
    constexpr int TT = TILE / BLOCK;                  // tail logits per thread: element tail_lo + r*BLOCK + tid
    float tx[TT];
    const float* rowp = a.logits + (int64_t)row * a.ld;
#pragma unroll
    for (int r = 0; r < TT; ++r) {
        const int e = tail_lo + r * BLOCK + tid;
        tx[r] = e < V ? rowp[e] : 0.f;
    }
    if (ntail > 0 && rc.capped) softcap_vals(tx, rc.p.softcap);
    if (ntail > 0 && rc.pen) {
        for (int i = tid; i < TILE / 8; i += BLOCK) reinterpret_cast<uint4*>(s.cnt())[i] = make_uint4(0u, 0u, 0u, 0u);
        __syncthreads();
        bool ovf = false;
        for (int64_t i = rc.b + tid; i < rc.len; i += BLOCK) {
            const int id = hist_at(a, rc, i);
            const uint32_t rel = (uint32_t)(id - tail_lo);
            if (id >= 0 && id < V && rel < (uint32_t)TILE) {
                const uint32_t sh = (rel & 1u) * 16u;
                const uint32_t old = atomicAdd(&s.cnt()[rel >> 1], 1u << sh);
                ovf |= ((old >> sh) & 0xFFFFu) == 0xFFFFu;
            }
        }
        if (ovf) atomicOr(a.err, FS_DEVERR_COUNT_OVERFLOW);
        __syncthreads();
        const float rp = rc.p.repetition_penalty, fq = rc.p.frequency_penalty, pr = rc.p.presence_penalty;
#pragma unroll
        for (int r = 0; r < TT; ++r) {
            const int rel = r * BLOCK + tid;
            const uint32_t cc = (s.cnt()[rel >> 1] >> ((rel & 1) * 16)) & 0xFFFFu;
            if (cc != 0u && tail_lo + rel < V) {
                float l = tx[r];
                if (rc.rep_on) l = l > 0.0f ? __fdiv_rn(l, rp) : __fmul_rn(l, rp);
                if (rc.fp_on) l = __fsub_rn(l, __fadd_rn(__fmul_rn((float)cc, fq), pr));
                tx[r] = l;
            }
        }
        __syncthreads();
    }

    if (rc.greedy) {
        uint64_t best = (pre.act && pre.r_me == 0) ? pre.v[0] : 0ull;    // each segment's best (entry 0)
#pragma unroll
        for (int r = 0; r < TT; ++r) {                // > -inf, as the segment kernel's IEEE compare from -inf:
            const int e = tail_lo + r * BLOCK + tid;  // NaN and -inf are never taken
            if (e < V && tx[r] > -__builtin_huge_valf()) {
                const uint64_t c = comp_of(key_of(tx[r]), (uint32_t)e);
                best = c > best ? c : best;
            }
        }
        best = block_max_u64(best, s.red);
        tok = best != 0 ? (int)comp_id(best) : 0;      // nothing above -inf / NaN: ferro's scan stays at 0
        const float l0 = rowp[0];
        if (l0 != l0) tok = 0;                         // ferro's scan never moves off a NaN at index 0
        if (tid == 0 && a.mode != MODE_VERIFY) {
            if (a.cand_ids && a.kcap > 0) a.cand_ids[(int64_t)row * a.kcap] = tok;
            if (a.cand_probs && a.kcap > 0) a.cand_probs[(int64_t)row * a.kcap] = 1.0;
        }
    } else {
        // ---- fast path: no tail, every list inside its prefetched window, k <= 64. L (the largest list bound)
        // comes from a wave reduction over the lists' bounds; T1 from a histogram of the prefetched registers over
        // [L, max]; the <= 128 candidates reaching T1 are ranked and finished by wave 0. Any other shape (or more
        // than 128 candidates at T1) takes the general path below.
        bool fast_done = false;
        if (ntail == 0 && k <= WAVE && nseg <= FAST_SEGS) {
            // every wave holds every list's (bound, count) pair (lane l: list l % nseg): no barrier
            const uint32_t L = wave_max(pre.t0m);
            const uint32_t cmax = wave_max(pre.cnm);
            if (cmax <= (uint32_t)(SPEC * pre.tps)) {
                for (int i = tid; i < NBINS; i += BLOCK) s.bins()[i] = 0u;
                if (tid == 0) { s.count = 0u; s.nids = 0u; }
                __syncthreads();
                // every candidate >= L into the candidate buffer (<= SPEC * BLOCK of them), tracking the max key
                uint32_t kmax = L;
#pragma unroll
                for (int q = 0; q < SPEC; ++q) {
                    const uint64_t w = pre.v[q];
                    const bool in = pre.act && (uint32_t)(pre.r_me + q * pre.tps) < pre.cnm && w != 0 && comp_key(w) >= L;
                    if (in) kmax = comp_key(w) > kmax ? comp_key(w) : kmax;
                    wave_append(in, w, s.cand, &s.count, CAP);
                }
                kmax = block_max_u32(kmax, s.red);            // its barrier also completes the appends
                const uint32_t n = s.count;
                uint64_t* list = s.cand;
                uint32_t c1 = n;
                if (n > (uint32_t)(2 * WAVE)) {
                    // more than 128: T1 from a histogram of the list over [L, kmax], then the <= 128 >= T1
                    const int sh = range_shift(L, kmax);
                    for (uint32_t i = tid; i < n; i += BLOCK) atomicAdd(&s.bins()[(comp_key(s.cand[i]) - L) >> sh], 1u);
                    __syncthreads();
                    const uint32_t T1 = hist_threshold(s.bins(), L, sh, k, &c1, s.wsum, s.red);
                    if (c1 >= (uint32_t)k && c1 <= (uint32_t)(2 * WAVE)) {
                        list = s.cand + SPEC * BLOCK;         // past the full list
                        for (uint32_t i0 = 0; i0 < n; i0 += BLOCK) {
                            const uint32_t i = i0 + tid;
                            const uint64_t c = i < n ? s.cand[i] : 0ull;
                            wave_append(c != 0 && comp_key(c) >= T1, c, list, &s.nids, 2 * WAVE);
                        }
                        __syncthreads();
                    }
                }
                if (c1 >= (uint32_t)k && c1 <= (uint32_t)(2 * WAVE)) {
                    uint64_t* small_out = list + SMALL;
                    uint32_t* rk = reinterpret_cast<uint32_t*>(small_out + 2 * WAVE);   // past wave_finish's buffers
                    block_ranks(list, (int)c1, rk);
                    if (tid < WAVE) wave_finish(a, rc, list, rk, k, pre.u, reinterpret_cast<double*>(small_out), tok, keep);
                    fast_done = true;
                }
            }
        }
        if (!fast_done) {
        // ---- the tail's own top k becomes one more list, kept in LDS at the top of the candidate buffer
        // (tl[0, nt); ttkey bounds the k-th key if the tail holds at least k candidates); the gather below then
        // fills at most gcap entries
        uint64_t* tl = s.cand + (CAP - KMAX);
        const uint32_t gcap = ntail > 0 ? (uint32_t)(CAP - KMAX) : (uint32_t)CAP;
        int nt = 0;
        uint32_t ttkey = 0u;
        if (ntail > 0) {
            if (tid == 0) s.count = 0u;
            __syncthreads();
#pragma unroll
            for (int r = 0; r < TT; ++r) {
                const int e = tail_lo + r * BLOCK + tid;
                const bool in = e < V && tx[r] == tx[r];
                wave_append(in, in ? comp_of(key_of(tx[r]), (uint32_t)e) : 0ull, s.cand, &s.count, CAP);
            }
            __syncthreads();
            nt = (int)s.count;
            if (nt > k) {
                ttkey = comp_key(compact_exact(nt, k, s));
                nt = k;
            }
            for (int i = tid; i < nt; i += BLOCK) tl[i] = s.cand[i];   // nt <= KMAX: no overlap
            __syncthreads();
        }
        // The segment lists (prefetched at kernel entry) and the tail list: L = the largest of their k-th key
        // bounds bounds the row's k-th key from below.
        const int tps = pre.tps, c_me = pre.c_me, r_me = pre.r_me;
        const bool act = pre.act;
        const uint32_t cnm = pre.cnm;
        const uint64_t* lst = a.cand + slot_of(rc, c_me) * CAP;
        if (act && r_me == 0) s.off[c_me] = cnm;
        if (tid == 0) s.count = 0u;
        // one reduction: L (bit 63 set when a list is longer than its prefetched window, or the lists' total may
        // overflow LDS: then the flat offsets below are needed)
        const bool longl = act && r_me == 0 && cnm > (uint32_t)(SPEC * tps);
        const uint64_t red = block_max_u64(((uint64_t)(longl ? 1u : 0u) << 63) | (act ? pre.t0m : 0u), s.red);
        uint32_t L = (uint32_t)red;
        L = ttkey > L ? ttkey : L;
        const bool need_off = (red >> 63) != 0ull || (uint32_t)nseg * (uint32_t)(SPEC * tps) + (uint32_t)nt > (uint32_t)CAP;
        // flat offsets of the segment lists (used when the candidates >= L overflow LDS)
        uint32_t total = 0u;
        if (need_off) {
            const uint32_t mine = tid < nseg ? s.off[tid] : 0u;
            const uint32_t o = block_excl_scan<uint32_t>(mine, s.wsum, &total);
            if (tid < nseg) s.off[tid] = o;
            if (tid == 0) s.off[nseg] = total;
            __syncthreads();
        }
        auto fetch = [&](uint32_t f) -> uint64_t {          // flat index -> candidate (0 past the end)
            const uint32_t g = f < total ? f : total - 1u;  // branch-free: the load is always issued in bounds
            int c0 = 0, c1 = nseg;                           // largest c with off[c] <= g
            while (c1 - c0 > 1) {
                const int m = (c0 + c1) >> 1;
                if (s.off[m] <= g) c0 = m; else c1 = m;
            }
            const uint64_t w = a.cand[slot_of(rc, c0) * CAP + (g - s.off[c0])];
            return f < total ? w : 0ull;
        };
        // gather the candidates >= L into LDS (counted past CAP), tracking their max key
        uint32_t kmax = L;
        for (int i0 = 0; i0 < nt; i0 += BLOCK) {
            const int i = i0 + tid;
            const uint64_t w = i < nt ? tl[i] : 0ull;
            const bool in = w != 0 && comp_key(w) >= L;
            if (in) kmax = comp_key(w) > kmax ? comp_key(w) : kmax;
            wave_append(in, w, s.cand, &s.count, gcap);
        }
        {                                           // the prefetched entries: one LDS atomic per wave
            uint64_t bal[SPEC];
            uint32_t tot = 0u;
#pragma unroll
            for (int q = 0; q < SPEC; ++q) {
                const uint64_t w = pre.v[q];
                const bool in = act && (uint32_t)(r_me + q * tps) < cnm && w != 0 && comp_key(w) >= L;
                if (in) kmax = comp_key(w) > kmax ? comp_key(w) : kmax;
                bal[q] = __ballot(in);
                tot += (uint32_t)__popcll(bal[q]);
            }
            if (tot != 0u) {
                uint32_t base = 0u;
                if (lane_id() == 0) base = atomicAdd(&s.count, tot);
                base = (uint32_t)__builtin_amdgcn_readlane((int)base, 0);
#pragma unroll
                for (int q = 0; q < SPEC; ++q) {
                    if ((bal[q] >> lane_id()) & 1ull) {
                        const uint32_t pos = base + mbcnt(bal[q]);
                        if (pos < gcap) s.cand[pos] = pre.v[q];
                    }
                    base += (uint32_t)__popcll(bal[q]);
                }
            }
        }
        // long lists: the entries past the prefetched window, LL loads in flight per thread and round (a list of
        // k ~ 2048 entries then costs one or two L2 round trips instead of one per tps entries)
        constexpr int LL = 8;
        for (uint32_t i0 = (uint32_t)(r_me + SPEC * tps); act && i0 < cnm; i0 += (uint32_t)(LL * tps)) {
            uint64_t w[LL];
#pragma unroll
            for (int q = 0; q < LL; ++q) {
                const uint32_t i = i0 + (uint32_t)(q * tps);
                w[q] = i < cnm ? lst[i] : 0ull;
            }
#pragma unroll
            for (int q = 0; q < LL; ++q) {
                const bool in = w[q] != 0 && comp_key(w[q]) >= L;
                if (in) kmax = comp_key(w[q]) > kmax ? comp_key(w[q]) : kmax;
                wave_append(in, w[q], s.cand, &s.count, gcap);
            }
        }
        for (int i = tid; i < NBINS; i += BLOCK) s.bins()[i] = 0u;
        uint32_t kmin = L;
        block_minmax_u32(kmin, kmax, s.red);
        FS_MARK(5);                                 // general merge: candidates >= L gathered
        const uint32_t n = s.count;
        const bool in_lds = n <= gcap;
        // T1: tight threshold from a histogram of the candidates' keys over [L, kmax]
        const int sh = range_shift(L, kmax);
        if (in_lds) {
            for (uint32_t i = tid; i < n; i += BLOCK) atomicAdd(&s.bins()[(comp_key(s.cand[i]) - L) >> sh], 1u);
        } else {
            for (uint32_t f = tid; f < total; f += BLOCK) {
                const uint64_t c = fetch(f);
                if (c != 0 && comp_key(c) >= L) atomicAdd(&s.bins()[(comp_key(c) - L) >> sh], 1u);
            }
            for (int i = tid; i < nt; i += BLOCK) {
                const uint64_t c = tl[i];
                if (comp_key(c) >= L) atomicAdd(&s.bins()[(comp_key(c) - L) >> sh], 1u);
            }
        }
        __syncthreads();
        uint32_t c1;
        const uint32_t T1 = hist_threshold(s.bins(), L, sh, k, &c1, s.wsum, s.red);
        FS_MARK(6);                                 // T1 known
        FS_TAG(9, c1); FS_TAG(10, n); FS_TAG(11, in_lds ? 1 : 0);
        if (c1 < (uint32_t)k) {
            // Fewer than k candidates: with L = 0 (no bound above NaN's key) every number of the row is a candidate,
            // so the row holds fewer than k numbers and samples over them (NaN is never a candidate); with L > 0 the
            // bounds promised k, an invariant failure. Never read past the list.
            if (tid == 0 && L != 0u) atomicOr(a.err, FS_DEVERR_INTERNAL);
            k = (int)c1;
        }
        // the c1 >= k candidates with key >= T1 contain the top k: sort them
        uint64_t* top;
        bool wave_done = false;                   // wave 0 finished the row (k <= 64, c1 <= 128)
        uint64_t* small_in = reinterpret_cast<uint64_t*>(s.bins());
        uint64_t* small_out = small_in + SMALL;
        if (tid == 0) s.count = 0u;
        __syncthreads();
        if (c1 <= (uint32_t)SMALL) {
            if (in_lds) {
                for (uint32_t i0 = 0; i0 < n; i0 += BLOCK) {
                    const uint32_t i = i0 + tid;
                    const uint64_t c = i < n ? s.cand[i] : 0ull;
                    wave_append(c != 0 && comp_key(c) >= T1, c, small_in, &s.count, SMALL);
                }
            } else {
                for (uint32_t f0 = 0; f0 < total; f0 += BLOCK) {
                    const uint64_t c = fetch(f0 + tid);
                    wave_append(c != 0 && comp_key(c) >= T1, c, small_in, &s.count, SMALL);
                }
                for (int i0 = 0; i0 < nt; i0 += BLOCK) {
                    const uint64_t c = i0 + tid < nt ? tl[i0 + tid] : 0ull;
                    wave_append(c != 0 && comp_key(c) >= T1, c, small_in, &s.count, SMALL);
                }
            }
            __syncthreads();
            if (c1 <= (uint32_t)(2 * WAVE) && k <= WAVE && k > 0) {
                uint32_t* rk = reinterpret_cast<uint32_t*>(small_out + 2 * WAVE);   // past wave_finish's buffers
                block_ranks(small_in, (int)c1, rk);
                if (tid < WAVE) wave_finish(a, rc, small_in, rk, k, pre.u, reinterpret_cast<double*>(small_out), tok, keep);
                wave_done = true;
            } else if (c1 <= (uint32_t)(4 * WAVE)) {
                rank_sort(small_in, (int)c1, small_out, k);
            } else {
                // the gathered list is spent: its buffer takes the scatter; counts and starts in cnt()
                static_assert(2 * (NBINS / 2) <= TILE / 2, "two half-size bin arrays in cnt()");
                bin_sort_desc<NBINS / 2>(small_in, (int)c1, s.cand, s.cnt(), s.cnt() + NBINS / 2, s.red, s.wsum);
            }
            top = !wave_done && c1 > (uint32_t)(4 * WAVE) ? small_in : small_out;   // binned sort: in place
        } else {
            // more than SMALL candidates reach T1: reduce to exactly the k >= X in LDS, then sort those
            int m = (int)n;
            if (!in_lds) {
                uint64_t X = 0;                         // threshold for a gather of <= CAP entries
                if (c1 > gcap) {
                    X = radix_kth(
                        [&](auto&& f) {
                            for (uint32_t f0 = tid; f0 < total; f0 += BLOCK) {
                                const uint64_t c = fetch(f0);
                                f(c != 0 && comp_key(c) >= L ? c : 0ull);
                            }
                            for (int i = tid; i < nt; i += BLOCK) f(comp_key(tl[i]) >= L ? tl[i] : 0ull);
                        },
                        k, s.bins(), s.wsum, s.red);
                }
                if (tid == 0) s.count = 0u;
                __syncthreads();
                for (uint32_t f0 = 0; f0 < total; f0 += BLOCK) {
                    const uint64_t c = fetch(f0 + tid);
                    wave_append(c != 0 && comp_key(c) >= T1 && c >= X, c, s.cand, &s.count, gcap);
                }
                for (int i0 = 0; i0 < nt; i0 += BLOCK) {
                    const uint64_t c = i0 + tid < nt ? tl[i0 + tid] : 0ull;
                    wave_append(c != 0 && comp_key(c) >= T1 && c >= X, c, s.cand, &s.count, gcap);
                }
                __syncthreads();
                m = (int)s.count;
            }
            if (in_lds) {                               // the c1 >= k entries at or above T1 hold the top k
                const int mt = keep_from(m, (uint64_t)T1 << 32, s);
                if (mt >= 0) m = mt;
            }
            if (m > KMAX) {                             // else the counting sort orders all m; the first k are used
                compact_exact(m, k, s);
                m = k;
            }
            const uint32_t big = bin_sort_desc(m, s);
            FS_TAG(12, big);
            (void)big;
            top = s.cand;
            c1 = (uint32_t)m;
        }
        FS_MARK(7);                                 // the top candidates sorted
        if (!wave_done) {
            if (c1 < (uint32_t)k) {                       // c1 >= k after the clamp above; never read past the list
                if (tid == 0) atomicOr(a.err, FS_DEVERR_INTERNAL);
                k = (int)c1;
            }
            if (k == 0) {                                 // every logit NaN: token 0, nothing kept
                tok = 0;
                keep = 0;
            } else {

            // ---- softmax at temperature, min-p, top-p, draw (sampler.cpp:37-49), k <= KMAX
            const fs_row_params& p = rc.p;
            const int i0 = tid * KPT;
            const float mx = val_of(comp_key(top[0]));
            const double Td = (double)p.temperature;
            double e[KPT];
            double part = 0.0;
#pragma unroll
            for (int q = 0; q < KPT; ++q) {
                const int i = i0 + q;
                e[q] = 0.0;
                if (i < k) {
                    const float d = val_of(comp_key(top[i])) - mx;   // fp32 subtraction, as ferro
                    e[q] = exp((double)d / Td);
                    part += e[q];
                }
            }
            const double sum = block_sum_f64(part, s.red);
            FS_MARK(8);                                 // exp and their sum
            double pr[KPT];
#pragma unroll
            for (int q = 0; q < KPT; ++q) pr[q] = e[q] / sum;
            // min-p: keep = 1 + the last index not below pr[0]*min_p (NaN masses stay) (at least 1)
            int keep_m = k;
            if (p.min_p > 0.0f) {
                const double thr = (1.0 / sum) * (double)p.min_p;
                int last = -1;
#pragma unroll
                for (int q = 0; q < KPT; ++q)
                    if (i0 + q < k && !(pr[q] < thr)) last = i0 + q;
                last = block_max_i32(last, s.red);
                keep_m = last + 1 > 1 ? last + 1 : 1;
            }
            // inclusive prefix of pr in candidate order
            double c[KPT];
            double run = 0.0;
#pragma unroll
            for (int q = 0; q < KPT; ++q) { run += pr[q]; c[q] = run; }
            double tot_all;
            const double off = block_excl_scan<double>(run, s.red.f64, &tot_all);
#pragma unroll
            for (int q = 0; q < KPT; ++q) c[q] += off;
            keep = keep_m;
            if (p.top_p < 1.0f) {
                int first = 0x7fffffff;
#pragma unroll
                for (int q = 0; q < KPT; ++q)
                    if (i0 + q < keep_m && c[q] >= (double)p.top_p && first == 0x7fffffff) first = i0 + q;
                first = block_min_i32(first, s.red);
                if (first != 0x7fffffff) keep = first + 1 < keep_m ? first + 1 : keep_m;
                if (keep < 1) keep = 1;
            }
            // tot = sum of the kept prefix; r = u * tot; the first i with r <= c_i
#pragma unroll
            for (int q = 0; q < KPT; ++q)
                if (i0 + q == keep - 1) s.red.dmisc[0] = c[q];
            __syncthreads();
            const double tot = s.red.dmisc[0];
            const double u = pre.u;
            const double rr = u * tot + 0.0;
            int hit = 0x7fffffff;
#pragma unroll
            for (int q = 0; q < KPT; ++q)
                if (i0 + q < keep && rr <= c[q] && hit == 0x7fffffff) hit = i0 + q;
            hit = block_min_i32(hit, s.red);
            const int pos = hit == 0x7fffffff ? keep - 1 : hit;
            tok = (int)comp_id(top[pos]);
            if (a.mode != MODE_VERIFY) {
                const int m = k < a.kcap ? k : a.kcap;
                if (a.cand_ids)
                    for (int i = tid; i < m; i += BLOCK) a.cand_ids[(int64_t)row * a.kcap + i] = (int32_t)comp_id(top[i]);
                if (a.cand_probs) {
#pragma unroll
                    for (int q = 0; q < KPT; ++q)
                        if (i0 + q < m) a.cand_probs[(int64_t)row * a.kcap + i0 + q] = pr[q];
                }
            }
            }                                             // k > 0
        }
        }                                             // general path
    }
    }
    if (!rc.greedy && nseg > 0 && !alone) {           // the segments' row histogram is spent: leave it at 0
        uint4* rz = reinterpret_cast<uint4*>(a.rhist + (int64_t)row * RBINS);
        for (int i = cut_done ? RBINS / 4 - 1 + tid : tid; i < RBINS / 4; i += BLOCK)   // (large_cut: the counters)
            rz[i] = make_uint4(0u, 0u, 0u, 0u);
        if (rc.large && !cut_done) {                   // and a large row's mass histogram
            uint4* mz = reinterpret_cast<uint4*>(a.rmass + (int64_t)row * LB);
            for (int i = tid; i < LB / 2; i += BLOCK) mz[i] = make_uint4(0u, 0u, 0u, 0u);
        }
    }
    if (a.out_hist_off || a.dmt) decode_commit(a, rc, s, tok);   // uniform (a decode step)
    if (a.mode != MODE_VERIFY) {
        if (tid == 0) {
            a.tok[row] = tok;
            if (a.keep) a.keep[row] = keep;
        }
    } else if (tid < WAVE) {
        // verify: the last row of a stream to finish computes the accepted prefix (server.cpp:627-637), wave 0.
        // Streams of up to 32 rows: one 64-bit atomic per row (the count of rows done, and a bit for each row that
        // ends the walk), the last row's fetched value gives the prefix; longer ones: tokens at agent scope, a row
        // counter after the 64-bit words, and the walk.
        const int st = rc.pidx;
        const int64_t r0 = a.row_off[st];
        const int m = (int)(a.row_off[st + 1] - r0);
        if (m <= 32) {
            if (tid == 0) {
                a.tok[row] = tok;
                const int rr = row - (int)r0;
                const bool stop = (a.eos >= 0 && tok == a.eos) || rr + 1 >= m || tok != a.rows[row + 1];
                const uint64_t mine = stop ? (1ull << rr) : 0ull;
                uint64_t* cnt = reinterpret_cast<uint64_t*>(a.stream_cnt) + st;
                const uint64_t old = __hip_atomic_fetch_add(cnt, (1ull << 32) | mine, __ATOMIC_RELAXED,
                                                            __HIP_MEMORY_SCOPE_AGENT);
                if ((uint32_t)(old >> 32) == (uint32_t)m - 1u) {
                    __hip_atomic_store(cnt, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    a.accepted[st] = __ffs((int)((uint32_t)old | (uint32_t)mine));
                }
            }
        } else {
            uint32_t* cnt32 = a.stream_cnt + 2 * (int64_t)a.n_streams + st;
            uint32_t old = 0u;
            if (tid == 0) {
                st_agent(&a.tok[row], (int32_t)tok);
                vm_drain();
                old = __hip_atomic_fetch_add(cnt32, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
            if (read_lane(old, 0) == (uint32_t)m - 1u) {
                if (tid == 0) st_agent(cnt32, 0u);
                const int acc = accepted_prefix(a.tok, a.rows, r0, m, a.eos);
                if (tid == 0) a.accepted[st] = acc;
            }
        }
    }
    __syncthreads();                                   // LDS is reused by the caller's next chunk
}

// A wave's snapshot of its row's histogram: lane l holds the counts of bins b0 + 4 (63 - l) + j, j = 0..3, where
// b0 is the wave's current bound's bin rounded down to a multiple of 4: the 256 bins (32 binades) from the bound
// up, in lane order = descending bins; counts above the window are left out (fewer counts: the bound stays
// valid).
// The row histogram lives in the L2 of the XCD that runs the row's segments (the grid places them there): counts
// are L2 atomics and snapshots are group-scope loads, served by that L2 or by a line the CU's L1 still holds from
// an earlier snapshot (older counts). Every access is an increment of zeroed memory or a read, so a read returns
// at most the row's true counts - stale, or with a segment on another XCD missing - and every bound stays valid.
struct RowSnap {
    uint64_t w[2];
    uint32_t b0;
};
// Through a buffer resource over the row histogram. With 0 records the load returns zeros without a memory access,
// so the tile loop can request it unconditionally (straight-line loads keep the compiler's memory-counter waits
// exact).
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
__device__ u32x4 raw_buffer_load_u32x4(__amdgpu_buffer_rsrc_t rs, int voffset, int soffset, int aux)
    __asm("llvm.amdgcn.raw.ptr.buffer.load.v4i32");
__device__ uint32_t raw_buffer_load_u32(__amdgpu_buffer_rsrc_t rs, int voffset, int soffset, int aux)
    __asm("llvm.amdgcn.raw.ptr.buffer.load.i32");
constexpr int AUX_SC0 = 1;               // cache policy sc0: group scope (the CU's L1, else the XCD's L2)
__device__ __forceinline__ RowSnap row_snap(__amdgpu_buffer_rsrc_t rs, uint32_t tkey) {
    RowSnap r;
    r.b0 = (tkey >> RSHIFT) & ~3u;
    const uint32_t first = r.b0 + 4u * (uint32_t)(WAVE - 1 - lane_id());
    const uint32_t f = first <= (uint32_t)RBINS - 4u ? first : (uint32_t)RBINS - 4u;   // past the top: ignored
    const u32x4 v = raw_buffer_load_u32x4(rs, (int)(f * 4u), 0, AUX_SC0);
    r.w[0] = (uint64_t)v.x | ((uint64_t)v.y << 32);
    r.w[1] = (uint64_t)v.z | ((uint64_t)v.w << 32);
    return r;
}
// From a snapshot: the lower edge of the highest bin with at least k counted logits in it and the bins above. At
// least k logits of the row reach it, so it bounds the row's k-th key from below (0: the snapshot holds fewer than
// k). No barrier: each wave takes its own snapshot, and any snapshot gives a valid bound.
__device__ __forceinline__ uint32_t row_bound(const RowSnap& r, int k) {
    const int lane = lane_id();
    const uint32_t first = r.b0 + 4u * (uint32_t)(WAVE - 1 - lane);
    const bool valid = first <= (uint32_t)RBINS - 4u;
    const uint32_t c0 = valid ? (uint32_t)r.w[0] : 0u, c1 = valid ? (uint32_t)(r.w[0] >> 32) : 0u;
    const uint32_t c2 = valid ? (uint32_t)r.w[1] : 0u, c3 = valid ? (uint32_t)(r.w[1] >> 32) : 0u;
    const uint32_t mine = c0 + c1 + c2 + c3;
    const uint32_t cum = wave_incl_scan_u32(mine);
    const uint32_t ex = cum - mine;
    const bool hit = ex < (uint32_t)k && cum >= (uint32_t)k;
    const uint32_t a3 = ex + c3, a2 = a3 + c2, a1 = a2 + c1;
    const uint32_t bin = first + (a3 >= (uint32_t)k ? 3u : a2 >= (uint32_t)k ? 2u : a1 >= (uint32_t)k ? 1u : 0u);
    const uint64_t hb = __ballot(hit);
    if (hb == 0ull) return 0u;
    return (uint32_t)__builtin_amdgcn_readlane((int)bin, __ffsll((unsigned long long)hb) - 1) << RSHIFT;
}

// The first PF tiles of a segment, requested from the kernel arguments alone (before the row's parameters arrive).
struct SegStart {
    int seg_lo, ntiles;
    const float* rowp;
    __amdgpu_buffer_rsrc_t rs;   // [seg_lo, seg_lo + ntiles * TILE) of the row
};
// spec: the balanced layout may still move this workgroup, and its loads are then overwritten before use. They are
// marked volatile (aux bit 31) so that the compiler keeps them at kernel entry instead of sinking them past the layout.
template <bool SPEC = false>
__device__ __forceinline__ SegStart seg_start(const Args& a, int row, int seg, int st, float (&buf)[PF][TPT]) {
    SegStart g;
    g.seg_lo = seg * st * TILE;
    const int left = a.V / TILE - seg * st;                         // full tiles left in the row
    g.ntiles = left < st ? left : st;                               // >= 1
    g.rowp = a.logits + (int64_t)row * a.ld;
    g.rs = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(g.rowp + g.seg_lo), (short)0, g.ntiles * TILE * 4,
                                             0x00020000);
#pragma unroll
    for (int p = 0; p < PF; ++p) load_seg_tile<SPEC ? (int)0x80000000 : 0>(buf[p], g.rs, p);
    return g;
}

// One (row, segment) item: stream the segment's full tiles with PF tiles in flight, apply the penalties, and keep
// the running candidates.
//   - greedy rows: each lane's first maximum;
//   - top-k rows: every logit with key >= tkey, a lower bound of the row's k-th key (at least k logits of the row
//     reach it). tkey starts from tile 0 (the highest coarse bin with >= k of the tile's lane maxima at or above
//     it) and is raised from the row histogram (a.rhist): the segments add counts of real logits to their row's
//     coarse bins (tile 0's lane maxima, then the buffered logits of tiles 1-4), and every wave snapshots the
//     counts and takes the highest bin with >= k counted logits at or above it. Counts only grow, so any snapshot
//     gives a valid bound, and the bound combines the whole row's evidence instead of one segment's.
// The segment publishes its candidates with key >= the final tkey (plain stores; the merge kernel runs after this
// kernel). They include every logit of the row's top k that lies in this segment.
__device__ __forceinline__ void process_segment(const Args& a, const RowCtx& rc, int seg, Shared& s,
                                                float (&buf)[PF][TPT], const SegStart& g) {
    const int tid = threadIdx.x;
    const int seg_lo = g.seg_lo;
    const int ntiles = g.ntiles;

    // the window ids (their loads return after the first tiles': the bitmap below waits for those anyway)
    constexpr int WPF = 2;
    int wid[WPF];
#pragma unroll
    for (int q = 0; q < WPF; ++q) {
        const int64_t i = rc.b + q * BLOCK + tid;
        wid[q] = (rc.pen && i < rc.len) ? hist_at(a, rc, i) : -1;
    }
    // Tile 0 is staged in the candidate buffer's tail (tile 0's own appends, at most one tile, stay below it) and
    // tile PF requested in its registers as soon as tile 0 arrives: tile 0's bound computation (two barriers) and
    // appends then run with PF tiles in flight. (Staging it before the penalty set-up, so that tile PF is requested
    // earlier still, measured slower: +1.1 us on a B=64 x V=262144 top-k 64 batch, +1.5 us on a mixed B=256 one.)
    float4* const stage0 = reinterpret_cast<float4*>(s.cand + (CAP - TILE / 2));
    static_assert(TILE + TILE / 2 <= CAP, "tile 0's appends stay below its stage");
    auto stage_tile0 = [&]() {
#pragma unroll
        for (int j = 0; j < NV; ++j)
            stage0[j * BLOCK + tid] = make_float4(buf[0][4 * j], buf[0][4 * j + 1], buf[0][4 * j + 2], buf[0][4 * j + 3]);
        load_seg_tile(buf[0], g.rs, PF);
    };
    // Penalties. With a repetition penalty alone (sampler.cpp:11-18) only membership in the window matters: an
    // exact bitmap of the segment's window ids (bmp, in the merge's offset array, unused by this kernel) is built
    // once, and a thread's four consecutive logits share one bitmap word, so each tile costs two LDS reads and no
    // barrier. Frequency / presence penalties need counts: the segment's window ids bucketed by tile once, then
    // counted wave by wave (wave_penalties; segments of >= 4 tiles), else a per-tile count table (apply_penalties).
    const int seg_hi = seg_lo + ntiles * TILE;
    const bool fastpen = rc.pen && rc.rep_on && !rc.fp_on && seg_hi - seg_lo <= 32 * (MAX_SEGS + 1);
    const bool slowpen = rc.pen && !fastpen;
    uint32_t* bmp = s.off;
    const float rp = rc.p.repetition_penalty;
    if (slowpen) gather_window(a, rc, seg_lo, seg_hi, s);
    // counts (frequency / presence): the window's ids bucketed by tile once, then counted per wave (no barriers);
    // a window with more than WIDS ids in the segment keeps the per-tile table (apply_penalties)
    const bool wavepen = slowpen && s.nids <= (uint32_t)WIDS && ntiles >= 4 && ntiles <= 2 * BLOCK;
    const bool tablepen = slowpen && !wavepen;
    if (wavepen) bucket_window(seg_lo, ntiles, s);
    if (fastpen) {
        for (int i = tid; i <= MAX_SEGS; i += BLOCK) bmp[i] = 0u;
        __syncthreads();
        auto mark = [&](int id) {
            const uint32_t rel = (uint32_t)(id - seg_lo);
            if (id >= seg_lo && id < seg_hi) atomicOr(&bmp[rel >> 5], 1u << (rel & 31u));
        };
#pragma unroll
        for (int q = 0; q < WPF; ++q) mark(wid[q]);
        for (int64_t i = rc.b + WPF * BLOCK + tid; i < rc.len; i += BLOCK) mark(hist_at(a, rc, i));
        __syncthreads();
    }
    auto bitmap_pen = [&](float (&x)[TPT], int lo) {
#pragma unroll
        for (int j = 0; j < NV; ++j) {
            const uint32_t rel = (uint32_t)(lo - seg_lo) + (uint32_t)(j * BLOCK + tid) * 4u;
            const uint32_t nib = (bmp[rel >> 5] >> (rel & 31u)) & 0xFu;
            if (nib != 0u) {
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const float l = x[4 * j + q];
                    if ((nib >> q) & 1u) x[4 * j + q] = l > 0.0f ? __fdiv_rn(l, rp) : __fmul_rn(l, rp);
                }
            }
        }
    };

    const int k = rc.k;
    const bool topk = !rc.greedy;      // large rows never reach this function
    float bv = -__builtin_huge_valf(); // greedy: this lane's first maximum (IEEE >: NaN never taken, -0 == +0)
    int bs = -1;                       //         and its slot tile*TPT + i (-1: none)
    uint32_t tkey = 0u;                // top-k: candidates are the logits with key >= tkey
    float tf = -__builtin_huge_valf(); //         in fp32: x >= tf (NaN never passes)
    uint32_t* rh = a.rhist + (int64_t)rc.row * RBINS;
    const __amdgpu_buffer_rsrc_t rsr = __builtin_amdgcn_make_buffer_rsrc(rh, (short)0, RBINS * 4, 0x00020000);
    // Row bounds from the row histogram. Segments of >= 3 tiles: each wave snapshots it after tile 0 and takes the
    // bound before appending tile 1; segments of >= 5 tiles snapshot again at tile 3 and take at tile 4, within one
    // iteration of the tile loop (no load outstanding across its back edge).
    // Shorter segments: one block-wide read at tile 0 (thread t holds bin b0 + BLOCK-1-t), taken after the loop.
    uint32_t scnt = 0u, sb0 = 0u;
    uint32_t rc0 = 0u;                 // lowest coarse bin of the tile-0 counts
    bool spending = false;
    if (tid == 0) { s.count = 0u; s.tmax = 0u; }
    if (tid < WAVE) s.rc64[tid] = 0u;
    __syncthreads();

    auto raise_key = [&](uint32_t kq) {
        if (kq > tkey) {
            tkey = kq;
            tf = kq > 0x007FFFFFu ? val_of(kq) : -__builtin_huge_valf();   // keys below -inf's are NaN patterns
        }
    };
    auto row_read = [&](uint32_t b0) -> uint32_t {
        const uint32_t b = b0 + (uint32_t)(BLOCK - 1 - tid);
        return raw_buffer_load_u32(rsr, (int)(4u * (b < (uint32_t)RBINS ? b : (uint32_t)RBINS - 1u)), 0, AUX_SC0);
    };
    // the highest bin b (>= rb0) with at least k counted logits in bins [b, rb0 + BLOCK - 1]: a row-wide bound
    auto row_take = [&](uint32_t rb0, uint32_t rcnt) {
        const uint32_t c = rb0 + (uint32_t)(BLOCK - 1 - tid) < (uint32_t)RBINS ? rcnt : 0u;
        uint32_t tot;
        const uint32_t above = block_excl_scan<uint32_t>(c, s.wsum, &tot);   // thread order = descending bins
        const int hit = (c != 0u && above + c >= (uint32_t)k) ? tid : BLOCK;
        const int first = block_min_i32(hit, s.red);
        if (first < BLOCK) raise_key((rb0 + (uint32_t)(BLOCK - 1 - first)) << RSHIFT);
    };
    // Top-k buffer discipline: after tile 0 the buffer is checked (barrier) every R tiles, R sized so the expected
    // appends fill at most half the headroom, and rows with k > 64 also at every iteration's first tile, where their
    // new entries are counted into the row histogram (the other segments' bounds tighten sooner: fewer appends row
    // wide); an overflow (appends past CAP are dropped) is detected at the next check and the segment is streamed
    // again in safe mode (a check after every tile).
    auto greedy_update = [&](const float (&x)[TPT], int tt) {
        const int sb = tt * TPT;
#pragma unroll
        for (int i = 0; i < TPT; ++i)
            if (x[i] > bv) { bv = x[i]; bs = sb + i; }
    };
    // appends of one tile: one fp32 compare per logit folded into a wave ballot; composites, LDS slots and row
    // counts are formed only where some lane passed
    auto topk_append = [&](const float (&x)[TPT], int lo) {
        uint64_t bal[TPT];
        uint64_t any = 0ull;
#pragma unroll
        for (int i = 0; i < TPT; ++i) {
            bal[i] = __ballot(x[i] >= tf);
            any |= bal[i];
        }
        if (any == 0ull) return;                     // wave-uniform
        const int lane = lane_id();
        uint32_t tot = 0u;
#pragma unroll
        for (int i = 0; i < TPT; ++i) tot += (uint32_t)__popcll(bal[i]);
        uint32_t base = 0u;
        if (lane == 0) base = atomicAdd(&s.count, tot);
        base = (uint32_t)__builtin_amdgcn_readlane((int)base, 0);
#pragma unroll
        for (int i = 0; i < TPT; ++i) {
            if (bal[i] != 0ull) {
                if ((bal[i] >> lane) & 1ull) {
                    const uint32_t kq = key_of(x[i]);
                    const uint32_t pos = base + mbcnt(bal[i]);
                    if (pos < (uint32_t)CAP) s.cand[pos] = comp_of(kq, (uint32_t)elem_id(lo, i));
                }
                base += (uint32_t)__popcll(bal[i]);
            }
        }
    };
    int counted = 0;                   // buffer entries [0, counted) are in the row histogram or never will be
    // Adds the buffered logits [from, count) of tiles >= 1 with key >= tkey to the row histogram, at their coarse
    // bins from tkey's (higher ones at the 64th: fewer counts, bounds stay valid). Tile 0 is counted already. The
    // waves' tkeys can differ (each wave takes its own row bounds), so each wave histograms the entries it reads
    // relative to its own tkey in its own 64 bins (in bins(), free between checks) and adds them to the row at
    // that base; a wave's LDS accesses complete in order, so no barrier is needed.
    // Entry: nb = the buffer's count, read by every wave after a barrier that followed the last append and before
    // any wave appends again; the next check's barrier ends the bins' use.
    auto count_row = [&](int from, int nb) {
        const uint32_t rb = tkey >> RSHIFT;
        uint32_t* wb = s.bins() + (tid / WAVE) * WAVE;
        wb[lane_id()] = 0u;
        if (nb <= CAP) {
            for (int i = from + tid; i < nb; i += BLOCK) {
                const uint64_t c = s.cand[i];
                if (comp_id(c) >= (uint32_t)(seg_lo + TILE) && comp_key(c) >= tkey) {
                    const uint32_t d = (comp_key(c) >> RSHIFT) - rb;
                    atomicAdd(&wb[d < (uint32_t)WAVE ? d : (uint32_t)WAVE - 1u], 1u);
                }
            }
        }
        const uint32_t c = wb[lane_id()];
        if (c != 0u && rb + (uint32_t)lane_id() < (uint32_t)RBINS)
            __hip_atomic_fetch_add(rh + rb + lane_id(), c, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);   // an L2 atomic
        counted = nb;
    };
    // barrier + count; returns it (> CAP: overflowed). Compacts when the headroom gets short: for k <= 256, in safe
    // mode and at the end (the published list then holds at most max(k, CAP - TILE)), when another whole tile could
    // overflow; otherwise when less than 3 tiles' worth at the observed append rate (at least 341) is left - an
    // overflow past that is caught at the next check and the segment streamed again in safe mode. A compaction
    // first drops the entries below the row bound (the largest of the waves' tkeys: one pass); only if that leaves
    // the headroom short (or more than KMAX entries) it keeps exactly the segment's k largest.
    int lastn = 0;
    const bool dyncount = topk && k > WAVE;      // k > 64: the buffered entries are counted at checks
    // last: the segment's final check, after which nothing is appended (its count needs no second barrier)
    auto check = [&](int tiles, bool strict, bool last = false) -> int {
        __syncthreads();
        int n = (int)s.count;
        if (!last) __syncthreads();                    // every wave holds the same count before any appends again
        int rate = (n - lastn) / (tiles > 0 ? tiles : 1);
        rate = rate > 341 ? rate : 341;
        auto short_room = [&](int m) {
            return m > k && (strict || k <= 4 * WAVE ? m > CAP - TILE : CAP - m < 3 * rate);
        };
        if (n <= CAP && short_room(n)) {
            if (dyncount && !strict) count_row(counted, n);   // before the order changes (not in safe mode)
            raise_key(block_max_u32(tkey, s.red));          // its barriers also end count_row's use of bins()
            const int m = keep_from(n, (uint64_t)tkey << 32, s);
            if (m >= 0) {
                n = m;
                counted = m;
            }
            if (m < 0 || short_room(n)) {
                // the entries at or above the k-th largest key (a radix select over the key bytes: 4 passes of an
                // 8-bit LDS histogram); if ties at that key leave too little room, exactly the k largest composites
                int nn = n;
                auto each = [&](auto&& f) { for (int i = tid; i < nn; i += BLOCK) f(s.cand[i]); };
                uint64_t X = radix_kth(each, k, s.bins(), s.wsum, s.red, 32);
                const int m2 = keep_from(nn, X, s);
                if (m2 >= 0) nn = m2;
                if (m2 < 0 || short_room(nn)) {
                    X = radix_kth(each, k, s.bins(), s.wsum, s.red);
                    (void)keep_from(nn, X, s);   // exactly k (composites are distinct)
                    nn = k;
                }
                raise_key(comp_key(X));
                n = nn;
                counted = n;               // the survivors are left uncounted (fewer counts: bounds stay valid)
            }
        }
        lastn = n;
        return n;
    };
    static_assert(PF == 2, "the row read is issued and taken within one iteration of the tile loop");
    RowSnap snap1;                     // the row histogram after tile 0 (segments of >= 3 tiles)
    for (int pass = 0; pass < 2; ++pass) {
        const bool safe = pass == 1;
        // k <= 64: tile 0's candidates are appended at tile 1, after the first row bound (its penalised logits wait in
        // the candidate buffer's tail; each thread reads back its own). Rows with the per-tile count table, and rows
        // with larger k (whose tile-0 bound lets through half a tile or more), append at once.
        const bool defer0 = topk && !safe && ntiles >= 2 && !tablepen && k <= WAVE;
        bool overflow = false;
        int R = 1;
        // ---- tile 0 (peeled: the initial threshold is computed here), through its stage
        {
            float x[TPT];
            const int lo = seg_lo;
            {
                stage_tile0();
                if (!safe) { FS_MARK(1); }
#pragma unroll
                for (int j = 0; j < NV; ++j) {
                    const float4 v = stage0[j * BLOCK + tid];
                    x[4 * j] = v.x; x[4 * j + 1] = v.y; x[4 * j + 2] = v.z; x[4 * j + 3] = v.w;
                }
            }
            if (rc.capped) softcap_vals_unrolled(x, rc.p.softcap);
            if (tablepen) apply_penalties(x, a, rc, lo, s);
            if (wavepen) wave_penalties(x, rc, lo, 0, s);
            if (fastpen) bitmap_pen(x, lo);
            if (rc.greedy) {
                greedy_update(x, 0);
            } else {
                if (!safe) {
                    // T0 and the row counts from the tile's lane maxima (all 8 logits of a lane when k > 64): a
                    // histogram over the 64 coarse bins up to the tile's largest key (rc0 = its lowest), in LDS.
                    // Its bins go to the row histogram at once, and T0 = the lower edge of the highest bin with at
                    // least k counted logits at or above it. Logits below the 64 bins are not counted (fewer
                    // counts: every bound read from them stays valid).
                    uint32_t kq[TPT];
                    uint32_t m1 = 0u;
                    if (k > WAVE) {
#pragma unroll
                        for (int i = 0; i < TPT; ++i) {
                            kq[i] = key_of(x[i]);
                            m1 = kq[i] > m1 ? kq[i] : m1;
                        }
                    } else {                             // the lane's largest logit (fmaxf passes over NaN)
                        float fm = x[0];
#pragma unroll
                        for (int i = 1; i < TPT; ++i) fm = fmaxf(fm, x[i]);
                        m1 = key_of(fm);
                    }
                    const uint32_t wm = wave_max(m1);
                    if (lane_id() == 0) atomicMax(&s.tmax, wm);
                    __syncthreads();
                    const uint32_t topb = s.tmax >> RSHIFT;
                    rc0 = topb >= (uint32_t)(WAVE - 1) ? topb - (uint32_t)(WAVE - 1) : 0u;
                    if (k > WAVE) {
#pragma unroll
                        for (int i = 0; i < TPT; ++i) {
                            const uint32_t d = (kq[i] >> RSHIFT) - rc0;
                            if (d < (uint32_t)WAVE) atomicAdd(&s.rc64[d], 1u);
                        }
                    } else {
                        const uint32_t d = (m1 >> RSHIFT) - rc0;
                        if (d < (uint32_t)WAVE) atomicAdd(&s.rc64[d], 1u);
                    }
                    __syncthreads();
                    const uint32_t cb = s.rc64[WAVE - 1 - lane_id()];   // lane order = descending bins
                    const uint64_t hb = __ballot(wave_incl_scan_u32(cb) >= (uint32_t)k);
                    if (hb != 0ull)
                        raise_key((rc0 + (uint32_t)(WAVE - 1) - (uint32_t)(__ffsll((unsigned long long)hb) - 1)) << RSHIFT);
                    if (tid < WAVE) {
                        const uint32_t c = s.rc64[tid];
                        if (c != 0u) __hip_atomic_fetch_add(rh + rc0 + tid, c, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                    }
                }
                if (defer0) {                            // the penalised tile waits in its stage for tile 1
#pragma unroll
                    for (int j = 0; j < NV; ++j)
                        stage0[j * BLOCK + tid] = make_float4(x[4 * j], x[4 * j + 1], x[4 * j + 2], x[4 * j + 3]);
                } else {
                    topk_append(x, lo);
                }
            }
            if (topk) {
                lastn = 0;
                // with tile 0's appends deferred the buffer is still empty: no check (two barriers) is needed
                const int n = defer0 ? 0 : check(1, safe);
                overflow = n > CAP;
                if (!safe && ntiles >= 3) snap1 = row_snap(rsr, tkey);
                const int per_tile = n > 32 ? n : 32;
                R = safe ? 1 : (CAP - n) / (2 * per_tile);
                if (R < 1) R = 1;
                if (!safe && ntiles < 3) {               // short segments: read once, taken at the end
                    sb0 = tkey >> RSHIFT;
                    scnt = row_read(sb0);
                    spending = true;
                }
            } else if (tablepen) {
                __syncthreads();                         // penalty-table reads of this tile are done
            }
            if (!safe) { FS_MARK(2); FS_MARKW(5); }
        }
        // ---- tiles 1.. (PF in flight; tile t is in buf[t % 2]). Iterations start at odd tiles, so the order in
        // which the two buffers were requested is the same on entry and around the back edge.
        int since = 0;
        // k > 64: a snapshot requested at every iteration's first tile (after its check and row count, before its
        // successor's loads), read at the next iteration's first tile: waiting for that tile covers it. Other rows
        // request it from an empty resource (no memory access).
        const bool dynrow = topk && !safe && k > WAVE;
        const __amdgpu_buffer_rsrc_t rsh = __builtin_amdgcn_make_buffer_rsrc(rh, (short)0, dynrow ? RBINS * 4 : 0,
                                                                             0x00020000);
        RowSnap snapd;
        bool dpend = false;
        for (int t0 = 1; t0 < ntiles && !overflow; t0 += PF) {
            const bool take1 = topk && !safe && t0 == 1 && ntiles >= 3;   // bound before tile 1
            const bool snap = topk && !safe && (t0 == 3 || t0 == 5) && t0 + 1 < ntiles;   // snapshot at 3/5, bound at 4/6
            const bool count2 = topk && !safe && t0 == 3 && ntiles >= 7 && k <= WAVE;   // tiles 1-4 at tile 4
            RowSnap snap2;
#pragma unroll
            for (int p = 0; p < PF; ++p) {
                const int tt = t0 + p;
                float (&x)[TPT] = buf[(p + 1) & 1];
                const bool live = tt < ntiles && !overflow;
                if (live) {
                    const int lo = seg_lo + tt * TILE;
                    if (rc.capped) softcap_vals_unrolled(x, rc.p.softcap);
                    if (tablepen) apply_penalties(x, a, rc, lo, s);
                    if (wavepen) wave_penalties(x, rc, lo, tt, s);
                    if (fastpen) bitmap_pen(x, lo);
                    if (p == 0 && take1) raise_key(row_bound(snap1, k));
                    if (p == 0 && dpend) raise_key(row_bound(snapd, k));
                    if (p == 1 && snap) raise_key(row_bound(snap2, k));
                    if (rc.greedy) {
                        greedy_update(x, tt);
                    } else {
                        if (p == 0 && defer0 && t0 == 1) {
                            float x0[TPT];
#pragma unroll
                            for (int j = 0; j < NV; ++j) {
                                const float4 v = stage0[j * BLOCK + tid];
                                x0[4 * j] = v.x; x0[4 * j + 1] = v.y; x0[4 * j + 2] = v.z; x0[4 * j + 3] = v.w;
                            }
                            topk_append(x0, seg_lo);
                        }
                        topk_append(x, lo);
                    }
                }
                // past the end: zeros, no memory access. The first tile of an iteration requests its successor
                // after the check and the row snapshot: the snapshot is then taken at the next tile with that
                // tile's successor still in flight (waits on the memory counter complete in request order).
                if (p == 1) load_seg_tile(x, g.rs, tt + PF);
                if (live) {
                    if (topk) {
                        bool checked = false;
                        if (++since >= R || tablepen || (dynrow && p == 0)) {
                            overflow = check(since, safe) > CAP;   // uniform: every thread read the same count
                            since = 0;
                            checked = true;
                        }
                        if (p == 0 && checked && dynrow && !overflow && t0 + PF < ntiles) count_row(counted, lastn);
                        if (p == 0) dpend = dynrow && !overflow && t0 + PF < ntiles;
                        if (p == 0 && snap) snap2 = row_snap(rsr, tkey);
                        if (p == 1 && count2 && !overflow) {
                            // second count: the buffered logits of tiles 1-4
                            __syncthreads();
                            const int nb = (int)s.count;
                            __syncthreads();
                            count_row(0, nb);
                        }
                    } else if (tablepen) {
                        __syncthreads();                 // penalty-table reads of this tile are done
                    }
                }
                if (p == 0) {
                    snapd = row_snap(rsh, tkey);
                    load_seg_tile(x, g.rs, tt + PF);
                }
                if (!safe && tt < 8) FS_MARKW(5 + tt);
            }
        }

        if (!topk) break;
        if (!overflow) overflow = check(since, true, true) > CAP;
        if (!overflow) break;
        // overflow: the buffer lost candidates. tkey is still a valid bound; stream the segment again in safe mode
        // (its logits are already counted in the row histogram).
        __syncthreads();
        if (tid == 0) s.count = 0u;
        spending = false;
#pragma unroll
        for (int p = 0; p < PF; ++p) load_seg_tile(buf[p], g.rs, p);
        __syncthreads();
    }
    if (topk && spending) row_take(sb0, scnt);
    FS_MARK(3);

    // ---- publish this segment's candidates (read by the merge kernel after this kernel completes)
    const int64_t slot = slot_of(rc, seg);
    uint64_t* gout = a.cand + (int64_t)slot * CAP;
    if (rc.greedy) {
        uint64_t best = 0ull;
        if (bs >= 0) best = comp_of(key_of(bv), (uint32_t)elem_id(seg_lo + (bs / TPT) * TILE, bs % TPT));
        best = block_max_u64(best, s.red);
        if (tid == 0) {
            gout[0] = best;
            a.meta[2 * slot] = comp_key(best);
            a.meta[2 * slot + 1] = 1u;
        }
    } else {
        // the buffered candidates with key >= tkey, in buffer order (thread t: entries t, t + BLOCK, ...)
        const int n = (int)s.count;              // <= CAP: no overflow past the checks above
        uint32_t mine = 0u;
        for (int i = tid; i < n; i += BLOCK)
            if (comp_key(s.cand[i]) >= tkey) ++mine;
        uint32_t tot;
        uint32_t pos = block_excl_scan<uint32_t>(mine, s.wsum, &tot);
        for (int i = tid; i < n; i += BLOCK) {
            const uint64_t c = s.cand[i];
            if (comp_key(c) >= tkey) gout[pos++] = c;
        }
        if (tid == 0) {
            a.meta[2 * slot] = tkey;              // at least k of the row's logits reach it
            a.meta[2 * slot + 1] = tot;
        }

    }
    __syncthreads();                               // LDS is reused by the next item
}

// ------------------------------------------------------------------------------------------------ large k, split
// Rows sampled with k > KMAX (top_k = 0 included: ferro's k = n, sampler.cpp:26) are sampled by the row's segment
// workgroups together: the passes of large_row (the one-workgroup version, kept as the fallback) each run over
// every segment at once, and the segments meet at row barriers between them. After each barrier every segment reads
// the others' published partial results and computes the same row-wide decision (the same inputs in the same
// order), so no workgroup waits for a coordinator:
//   P1 extremes, ordered count and (k < V) coarse-bin counts (added to the row histogram) -> the k-th's coarse bin bk;
//   P2 the masses exp((v - mx) / T) of the candidates above bk (fp64 partial sums, fixed-point mass histogram added
//      to the row's in the workspace) and bin bk's elements gathered -> the exact k-th Xk, S and the mass histogram;
//   P3 top-p's crossing bin bc gathered, with min-p's counts and masses -> the kept prefix and its total;
//   P4 the draw's bin bd gathered, unless it is bc (already sorted in LDS) -> the token.
// Segment 0 publishes the token and what the merge needs for the optional candidate outputs. A bin too large for
// one sort, a target outside its bin's exact masses, or a barrier that waits too long abandons the row (a flag on
// the barrier counter); the merging workgroup then samples it alone with large_row (exact).
// Arrive and wait until `target` arrivals (every segment of the row at this barrier). This workgroup's stores and
// atomics complete first (vmcnt(0)). No cache maintenance follows: what the others published lies in lines that no
// workgroup of the row reads before this barrier (their own lines per phase, see the slot layout), so this CU's L1
// holds no copy of them and the loads are served by the XCD's L2. (An agent-scope invalidate, buffer_inv sc1, cost
// about 10 us per barrier here.) The poll is an atomic that is not idempotent (it executes in the L2). Bounded: past
// a.merge_spins polls the row is abandoned. Returns false when the row is abandoned.
__device__ __forceinline__ bool row_sync(const Args& a, int row, uint32_t target, Shared& s) {
    vm_drain();
    __syncthreads();
    if (threadIdx.x == 0) {
        uint32_t* c = row_sync_ctr(a, row);
        __hip_atomic_fetch_add(c, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        uint32_t ok = 1u, spins = 0u;
        for (;;) {
            const uint32_t v = __hip_atomic_fetch_add(c, 0x10000u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
            if (v & ROW_ABANDONED) { ok = 0u; break; }
            if ((v & 0x7FFFu) >= target && a.merge_spins != 0u) break;
            if (++spins >= a.merge_spins) {
                __hip_atomic_fetch_or(c, ROW_ABANDONED, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                ok = 0u;
                break;
            }
            __builtin_amdgcn_s_sleep(1);
        }
        s.red.misc[4] = ok;
    }
    __syncthreads();
    const bool ok = s.red.misc[4] != 0u;
    __syncthreads();                                     // misc[4] is reused by the next barrier
    return ok;
}

// One pass over a large-row segment's tiles [lo0, hi) (the last segment also takes the row's partial tile), two
// tiles in flight, softcap and penalties applied: f(x, key, composite) per ordered element. Ends with a barrier.
// bmp: a repetition penalty alone, from a bitmap of the window's ids over the segment (bit i = id lo0 + i; a
// thread's four consecutive logits share a word), else the per-tile count table (s.ids holds the window's ids).
// g(x): a per-tile hook, called on each tile's (softcapped, penalised) logits before f sees them.
template <class F, class G>
__device__ __forceinline__ void seg_elems_g(const Args& a, const RowCtx& rc, Shared& s, int lo0, int hi, bool bmp, F f, G g) {
    const float* rowp = a.logits + (int64_t)rc.row * a.ld;
    const int nt = (hi - lo0 + TILE - 1) / TILE;
    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(rowp + lo0), (short)0,
                                                                        ((hi - lo0 + 3) & ~3) * 4, 0x00020000);
    float buf[LPF][TPT];
#pragma unroll
    for (int p = 0; p < LPF; ++p) load_seg_tile(buf[p], rs, p);
    for (int t0 = 0; t0 < nt; t0 += LPF) {
#pragma unroll
        for (int p = 0; p < LPF; ++p) {
            const int t = t0 + p;
            float x[TPT];
#pragma unroll
            for (int i = 0; i < TPT; ++i) x[i] = buf[p][i];
            load_seg_tile(buf[p], rs, t + LPF);
            if (t < nt) {
                const int lo = lo0 + t * TILE;
                if (rc.capped) softcap_vals(x, rc.p.softcap);
                if (rc.pen && bmp) {
                    const uint32_t* bm = reinterpret_cast<const uint32_t*>(s.ids);
                    const float rp = rc.p.repetition_penalty;
#pragma unroll
                    for (int j = 0; j < NV; ++j) {
                        const uint32_t rel = (uint32_t)(lo - lo0) + (uint32_t)(j * BLOCK + (int)threadIdx.x) * 4u;
                        const uint32_t nib = (bm[rel >> 5] >> (rel & 31u)) & 0xFu;
                        if (nib != 0u) {
#pragma unroll
                            for (int q = 0; q < 4; ++q) {
                                const float l = x[4 * j + q];
                                if ((nib >> q) & 1u) x[4 * j + q] = l > 0.0f ? __fdiv_rn(l, rp) : __fmul_rn(l, rp);
                            }
                        }
                    }
                } else if (rc.pen) {
                    __syncthreads();                     // the previous tile's table reads are done
                    apply_penalties(x, a, rc, lo, s);
                }
                g(x, lo);
#pragma unroll
                for (int i = 0; i < TPT; ++i) {
                    const int e = elem_id(lo, i);
                    const bool ok = e < hi && x[i] == x[i];
                    const uint32_t kq = key_of(x[i]);
                    f(ok, x[i], kq, comp_of(kq, (uint32_t)e));
                }
            }
        }
    }
    __syncthreads();
}

template <class F>
__device__ __forceinline__ void seg_elems(const Args& a, const RowCtx& rc, Shared& s, int lo0, int hi, bool bmp, F f) {
    seg_elems_g(a, rc, s, lo0, hi, bmp, f, [](const float (&)[TPT], int) {});
}

// The gathered lists of one region of every segment of the row, concatenated into s.cand[0, n) and sorted in
// candidate order (descending composites). Returns n, or -1 when a list overflowed or they exceed KMAX together.
// Called after a row barrier (the lists are in the L2; this workgroup's L1 is invalidated).
__device__ __forceinline__ int load_lists(const Args& a, const RowCtx& rc, int region, int cnt_slot, Shared& s) {
    const int tid = threadIdx.x, nseg = rc.nseg;
    uint32_t mine = 0u;
    bool over = false;
    for (int j = tid; j < nseg; j += BLOCK) {
        const uint64_t c = a.cand[slot_of(rc, j) * CAP + cnt_slot];
        over |= c > (uint64_t)LLR;
    }
    // offsets: thread j < nseg holds list j's count (nseg < BLOCK, kept so by the host)
    if (tid < nseg) {
        const uint64_t c = a.cand[slot_of(rc, tid) * CAP + cnt_slot];
        mine = c > (uint64_t)LLR ? 0u : (uint32_t)c;
    }
    uint32_t tot;
    const uint32_t off = block_excl_scan<uint32_t>(mine, s.wsum, &tot);
    const bool any_over = block_max_u32(over ? 1u : 0u, s.red) != 0u;
    if (any_over || tot > (uint32_t)KMAX) return -1;    // uniform
    if (tid < nseg) s.off[tid] = off;
    if (tid == 0) s.off[nseg] = tot;
    __syncthreads();
    for (uint32_t f = tid; f < tot; f += BLOCK) {        // flat index -> (list, position)
        int c0 = 0, c1 = nseg;
        while (c1 - c0 > 1) {
            const int m = (c0 + c1) >> 1;
            if (s.off[m] <= f) c0 = m; else c1 = m;
        }
        s.cand[f] = a.cand[slot_of(rc, c0) * CAP + LSC + region * LLR + (f - s.off[c0])];
    }
    __syncthreads();
    bin_sort_desc((int)tot, s);
    return (int)tot;
}

// A row-wide sum over the segments' published scalar (fp64 bits at cnt_slot), in a fixed order (deterministic).
__device__ __forceinline__ double sum_slots_f64(const Args& a, const RowCtx& rc, int sl, Shared& s) {
    double v = 0.0;
    for (int j = threadIdx.x; j < rc.nseg; j += BLOCK) v += __longlong_as_double((long long)a.cand[slot_of(rc, j) * CAP + sl]);
    return block_sum_f64(v, s.red);
}
__device__ __forceinline__ uint64_t sum_slots_u64(const Args& a, const RowCtx& rc, int sl, Shared& s) {
    uint64_t v = 0ull;
    for (int j = threadIdx.x; j < rc.nseg; j += BLOCK) v += a.cand[slot_of(rc, j) * CAP + sl];
    uint64_t tot;
    (void)block_excl_scan<uint64_t>(v, s.red.u64b, &tot);
    return tot;
}

// Rows where every token is a candidate (k >= V) sampled from the logits within CUT_C * T of the row's maximum,
// when the rest provably holds neither top-p's crossing, min-p's boundary nor the draw: after the first row barrier
// every segment decides the same way from the published scalars (same inputs, same order); segment 0 then gathers the
// lists (at most KMAX logits), sorts them, and runs sampler.cpp:37-49 over them in double precision, the rest's mass
// (every element below e^-CUT_C of the maximum) added to S. Returns true when the row is done (or given to the merge:
// a target that still lands in the rest abandons the row to the exact path); false: the segments go on with the
// passes of the general large-row path.
constexpr float CUT_C = 16.0f;
constexpr double CFXS = 1125899906842624.0;      // 2^50: fixed-point scale of the lists' masses (each <= 1, <= CAP)

template <bool DESC>
__device__ __forceinline__ uint64_t sort64(uint64_t v);

// large_cut's finish when the lists hold at most 64 logits and the row has at most 64 segments: one wave, the
// logits in lanes (sampler.cpp:28-49 as in the block version below, with wave scans in candidate order).
// Returns false when a target lands in the rest (the caller abandons the row).
__device__ __forceinline__ bool wave_cut_finish(const Args& a, const RowCtx& rc, uint64_t* my, float mx, float cut,
                                                double Td, double st, uint32_t ntot, int keff, uint32_t kmax,
                                                uint64_t cmin, double u, bool min_in, uint32_t cnt) {
    const int lane = lane_id(), nseg = rc.nseg;
    const fs_row_params& p = rc.p;
    // the lists' offsets (lane j: list j's count cnt), then lane f takes flat entry f
    const uint32_t inc = wave_incl_scan_u32(cnt);
    const uint32_t off = inc - cnt;
    const uint32_t tot = (uint32_t)__builtin_amdgcn_readlane((int)inc, 63);
    int j = 0;
    for (int q = 1; q < nseg; ++q)
        if ((uint32_t)lane >= (uint32_t)__builtin_amdgcn_readlane((int)off, q)) j = q;
    const uint32_t my_off = (uint32_t)__builtin_amdgcn_ds_bpermute(j << 2, (int)off);
    uint64_t c = 0ull;
    if ((uint32_t)lane < tot) c = a.cand[slot_of(rc, j) * CAP + LSC + ((uint32_t)lane - my_off)];
    const float x = val_of(comp_key(c));
    const bool in = (uint32_t)lane < tot && x >= mx - cut;
    const uint64_t dm = ((uint32_t)lane < tot && !in) ? (uint64_t)(mass_of(x, mx, Td) * CFXS + 0.5) : 0ull;
    const uint64_t dfx = wave_allreduce(dm, [](uint64_t p_, uint64_t q_) { return p_ + q_; });
    const uint64_t v = sort64<true>(in ? c : 0ull);      // ferro's order; lanes >= n hold 0
    const int n = __popcll(__ballot(in));
    const double rest = st + (double)dfx / CFXS;
    double e = 0.0;
    if (lane < n) e = mass_of(val_of(comp_key(v)), mx, Td);
    const double S = lane_f64(wave_scan_f64(e), WAVE - 1) + rest;
    const double pr = e / S;
    const double cum = wave_scan_f64(pr);
    int keep_m = n;
    bool m_beyond = (uint32_t)n < ntot;
    if (p.min_p > 0.0f) {
        const double thr = (1.0 / S) * (double)p.min_p;
        const uint64_t mm = __ballot(lane < n && !(pr < thr));
        keep_m = mm ? 64 - __clzll((long long)mm) : 1;
        m_beyond = keep_m == n && (uint32_t)n < ntot && !min_in;
    }
    int keep = keep_m;
    bool beyond = m_beyond;
    if (p.top_p < 1.0f) {
        const uint64_t mm = __ballot(lane < keep_m && cum >= (double)p.top_p);
        if (mm) {
            const int first = __ffsll((unsigned long long)mm) - 1;
            keep = first + 1 < keep_m ? first + 1 : keep_m;
            beyond = false;
        } else if (m_beyond) {
            return false;                                // top-p's crossing lies in the rest
        }
    } else if (m_beyond && p.min_p > 0.0f) {
        return false;                                    // min-p's boundary lies in the rest
    }
    const double totk = beyond ? lane_f64(cum, n - 1) + rest / S : lane_f64(cum, keep - 1);
    const double rr = u * totk + 0.0;
    const int lim = beyond ? n : keep;
    const uint64_t hm = __ballot(lane < lim && rr <= cum);
    int at;
    if (hm) at = __ffsll((unsigned long long)hm) - 1;
    else if (beyond) return false;                       // the draw lies in the rest
    else at = keep - 1;
    const uint64_t pick = read_lane(v, at);
    if (lane == 0) {
        const uint32_t kp = beyond ? ntot : (uint32_t)keep;
        my[LS_TOK] = (uint64_t)comp_id(pick) | ((uint64_t)kp << 32);
        my[LS_XK] = cmin;
        my[LS_S] = (uint64_t)__double_as_longlong(S);
        my[LS_KEFF] = (uint64_t)(uint32_t)keff | ((uint64_t)kmax << 32);
        my[LS_STATUS] = 2ull;
    }
    return true;
}

// The cut's decision from the row's published sums: sc / st the listed logits' / the rest's mass relative to the
// row's maximum, nft the lists' total. True when the rest provably holds neither top-p's crossing, min-p's boundary
// nor the draw (estimates within 1e-5; the exact walk still checks).
__device__ __forceinline__ bool cut_decide(const fs_row_params& p, double sc, double st, uint64_t nft, bool ovf,
                                           double u, bool& min_in) {
    const double S_est = sc + st;
    const double e_c = exp(-(double)CUT_C);
    const double sc_lo = sc - (double)nft * e_c;          // the row's cut moves at most e^-CUT_C per listed logit
    const double mrg = 1.0 + 1e-5;
    min_in = p.min_p > 0.0f && (double)p.min_p >= e_c * 1.01;   // min-p keeps only listed logits
    bool within = min_in;
    if (p.top_p < 1.0f) within = within || (double)p.top_p * S_est * mrg < sc_lo;
    if (!(p.top_p < 1.0f) && !(p.min_p > 0.0f)) within = u * S_est * mrg < sc_lo;
    return !ovf && nft >= 1u && nft <= (uint64_t)KMAX && within;
}

// large_cut's finish by the whole block (the lists hold more than 64 logits, or the row more than 64 segments).
__device__ __forceinline__ void cut_finish_block(const Args& a, const RowCtx& rc, Shared& s, uint64_t* my, float mx,
                                                 uint32_t kmax, uint64_t cmin, uint32_t ntot, int keff, double st,
                                                 double u, bool min_in) {
    const int tid = threadIdx.x, nseg = rc.nseg, row = rc.row;
    const fs_row_params& p = rc.p;
    const double Td = (double)p.temperature;
    const float cut = CUT_C * p.temperature;
    // ---- segment 0: the lists above mx - cut, sorted (sampler.cpp:28-35)
    uint32_t mine = 0u;
    if (tid < nseg) mine = (uint32_t)a.cand[slot_of(rc, tid) * CAP + LS_FN];
    uint32_t tot;
    const uint32_t off = block_excl_scan<uint32_t>(mine, s.wsum, &tot);
    if (tid < nseg) s.off[tid] = off;
    if (tid == 0) { s.off[nseg] = tot; s.count = 0u; }
    __syncthreads();
    uint64_t drop = 0ull;                                // fixed point: the lists' order is not fixed
    for (uint32_t b0 = 0u; b0 < tot; b0 += BLOCK) {
        const uint32_t f = b0 + (uint32_t)tid;
        uint64_t c = 0ull;
        if (f < tot) {
            int c0 = 0, c1 = nseg;
            while (c1 - c0 > 1) {
                const int m = (c0 + c1) >> 1;
                if (s.off[m] <= f) c0 = m; else c1 = m;
            }
            c = a.cand[slot_of(rc, c0) * CAP + LSC + (f - s.off[c0])];
        }
        const float x = val_of(comp_key(c));
        const bool in = f < tot && x >= mx - cut;
        if (f < tot && !in) drop += (uint64_t)(mass_of(x, mx, Td) * CFXS + 0.5);
        wave_append(in, c, s.cand, &s.count, (uint32_t)CAP);
    }
    uint64_t dfx;
    (void)block_excl_scan<uint64_t>(drop, s.red.u64b, &dfx);   // its barriers also complete the appends
    const int n = (int)s.count;
    FS_MARK(7);                                          // lists gathered
    __syncthreads();
    bin_sort_desc(n, s);
    FS_MARK(2);                                          // sorted
    // ---- softmax over the list plus the rest's mass, min-p, top-p, draw (sampler.cpp:37-49)
    const int i0 = tid * KPT;
    double e[KPT];
    double part = 0.0;
#pragma unroll
    for (int q = 0; q < KPT; ++q) {
        e[q] = i0 + q < n ? mass_of(val_of(comp_key(s.cand[i0 + q])), mx, Td) : 0.0;
        part += e[q];
    }
    const double rest = st + (double)dfx / CFXS;
    const double S = block_sum_f64(part, s.red) + rest;
    FS_MARK(3);                                          // S
    double pr[KPT];
#pragma unroll
    for (int q = 0; q < KPT; ++q) pr[q] = e[q] / S;
    int keep_m = n;
    bool m_beyond = (uint32_t)n < ntot;                  // every listed logit kept so far and the rest after them
    if (p.min_p > 0.0f) {
        const double thr = (1.0 / S) * (double)p.min_p;
        int last = -1;
#pragma unroll
        for (int q = 0; q < KPT; ++q)
            if (i0 + q < n && !(pr[q] < thr)) last = i0 + q;
        last = block_max_i32(last, s.red);
        keep_m = last + 1 > 1 ? last + 1 : 1;
        m_beyond = keep_m == n && (uint32_t)n < ntot && !min_in;
    }
    double c[KPT];
    double run = 0.0;
#pragma unroll
    for (int q = 0; q < KPT; ++q) { run += pr[q]; c[q] = run; }
    double tot_all;
    const double coff = block_excl_scan<double>(run, s.red.f64, &tot_all);
#pragma unroll
    for (int q = 0; q < KPT; ++q) c[q] += coff;
    int keep = keep_m;
    bool beyond = m_beyond;
    bool fail = false;
    if (p.top_p < 1.0f) {
        int first = 0x7fffffff;
#pragma unroll
        for (int q = 0; q < KPT; ++q)
            if (i0 + q < keep_m && c[q] >= (double)p.top_p && first == 0x7fffffff) first = i0 + q;
        first = block_min_i32(first, s.red);
        if (first != 0x7fffffff) {
            keep = first + 1 < keep_m ? first + 1 : keep_m;
            beyond = false;
        } else if (m_beyond) {
            fail = true;                                 // top-p's crossing lies in the rest
        }
    } else if (m_beyond && p.min_p > 0.0f) {
        fail = true;                                     // min-p's boundary lies in the rest
    }
    // tot = the kept prefix's sum; r = u * tot; the first i with r <= c_i
    double totk = 0.0;
    if (!beyond) {
#pragma unroll
        for (int q = 0; q < KPT; ++q)
            if (i0 + q == keep - 1) s.red.dmisc[0] = c[q];
        __syncthreads();
        totk = s.red.dmisc[0];
    } else {
        totk = tot_all + rest / S;
    }
    const double rr = u * totk + 0.0;
    const int lim = beyond ? n : keep;
    int hit = 0x7fffffff;
#pragma unroll
    for (int q = 0; q < KPT; ++q)
        if (i0 + q < lim && rr <= c[q] && hit == 0x7fffffff) hit = i0 + q;
    hit = block_min_i32(hit, s.red);
    if (hit == 0x7fffffff) {
        if (beyond) fail = true;                         // the draw lies in the rest
        else hit = keep - 1;
    }
    FS_MARK(8);                                          // walked
    if (fail) {
        row_abandon(a, row);
        return;
    }
    if (tid == 0) {
        const uint32_t kp = beyond ? ntot : (uint32_t)keep;
        my[LS_TOK] = (uint64_t)comp_id(s.cand[hit]) | ((uint64_t)kp << 32);
        my[LS_XK] = cmin;
        my[LS_S] = (uint64_t)__double_as_longlong(S);
        my[LS_KEFF] = (uint64_t)(uint32_t)keff | ((uint64_t)kmax << 32);
        my[LS_STATUS] = 2ull;
    }
}

__device__ __forceinline__ bool large_cut(const Args& a, const RowCtx& rc, Shared& s, int seg, uint64_t* my, float mx,
                                          uint32_t kmax, uint64_t cmin, uint32_t ntot, int keff) {
    const int tid = threadIdx.x, nseg = rc.nseg, row = rc.row;
    const fs_row_params& p = rc.p;
    if (!(mx > -__builtin_huge_valf() && mx < __builtin_huge_valf())) return false;   // uniform
    const double Td = (double)p.temperature;
    // row-wide: the lists' total, their masses and the rest's, relative to mx
    uint32_t nf = 0u, ovf = 0u;
    double sc = 0.0, st = 0.0;
    for (int j = tid; j < nseg; j += BLOCK) {
        const uint64_t* sl = a.cand + slot_of(rc, j) * CAP;
        const uint64_t n = sl[LS_FN];
        if (n > (uint64_t)LLR) ovf = 1u; else nf += (uint32_t)n;
        if (sl[LS_NV] != 0ull) {
            const double F = exp(((double)val_of(comp_key(sl[LS_MAX])) - (double)mx) / Td);
            sc += F * __longlong_as_double((long long)sl[LS_FC]);
            st += F * __longlong_as_double((long long)sl[LS_FT]);
        }
    }
    uint32_t nft;
    (void)block_excl_scan<uint32_t>(nf, s.wsum, &nft);
    ovf = block_max_u32(ovf, s.red);
    sc = block_sum_f64(sc, s.red);
    st = block_sum_f64(st, s.red);
    const double u = row_u(a, row);
    bool min_in;
    if (!cut_decide(p, sc, st, nft, ovf != 0u, u, min_in)) return false;   // uniform
    if (seg != 0) return true;
    cut_finish_block(a, rc, s, my, mx, kmax, cmin, ntot, keff, st, u, min_in);
    return true;
}

// A crowded coarse bin (more candidates than the gather regions hold, e.g. the middle of a flat row): the element
// at which the cumulative mass in ferro's order, from the row's top, reaches `target` inside bin b, through one
// level of finer bins (the next FSB key bits). above_b is the mass of the candidates above bin b. All segments run
// it together (uniform arguments, row barriers from nsync on):
//   1. the row's fine histogram is cleared (rmass: fixed-point masses, rhist: counts; neither is read any more)
//   2. each segment streams its tiles: masses and counts of its candidates in bin b by fine bin, added to the row's
//   3. every segment locates the fine bin of the target (the same sums, the same decision) and gathers it
//   4. the gathered lists, sorted, are walked in exact fp64 masses (large_walk)
// Returns false (the row is then abandoned) when the fine bin still overflows or the walk leaves it; otherwise the
// element, the cumulative mass through it and the number of candidates in bin b before it.
constexpr int FSB = 11;                                    // fine bins: 2048 (row histogram bins below its counters)
constexpr int FBN = 1 << FSB;
constexpr int FSH = LB_SHIFT - FSB;
static_assert(FBN <= RBINS - 2 && FBN <= LB && FSH >= 0, "fine bins fit the row histograms");
__device__ __forceinline__ bool refine_bin(const Args& a, const RowCtx& rc, Shared& s, int seg_i, uint64_t* my, int lo0, int hi,
                                        bool bmpen, uint32_t b, uint64_t Xlo, double above_b, double target, float mx,
                                        double Td, uint32_t& nsync, uint64_t& pick, double& cum, uint32_t& before) {
    const int tid = threadIdx.x, row = rc.row, nseg = rc.nseg;
    uint64_t* rm = a.rmass + (int64_t)row * LB;
    uint32_t* rh = a.rhist + (int64_t)row * RBINS;
    // 1. clear this segment's slice of the row's fine histogram
    const int per = (FBN + nseg - 1) / nseg;
    for (int i = seg_i * per + tid; i < (seg_i + 1) * per && i < FBN; i += BLOCK) { rm[i] = 0ull; rh[i] = 0u; }
    ++nsync;
    if (!row_sync(a, row, nsync * (uint32_t)nseg, s)) return false;
    // 2. this segment's candidates in bin b, by fine bin (LDS: masses in s.cand[0, FBN), counts after them)
    uint64_t* fm = s.cand;
    uint32_t* fc = reinterpret_cast<uint32_t*>(s.cand + FBN);
    for (int i = tid; i < FBN; i += BLOCK) { fm[i] = 0ull; fc[i] = 0u; }
    __syncthreads();
    seg_elems(a, rc, s, lo0, hi, bmpen, [&](bool ok, float x, uint32_t kq, uint64_t c) {
        if (ok && c >= Xlo && (kq >> LB_SHIFT) == b) {
            const uint32_t f = (kq >> FSH) & (uint32_t)(FBN - 1);
            atomicAdd(reinterpret_cast<unsigned long long*>(&fm[f]), (unsigned long long)(mass_of(x, mx, Td) * FXS + 0.5));
            atomicAdd(&fc[f], 1u);
        }
    });
    for (int i = tid; i < FBN; i += BLOCK) {
        if (fm[i] != 0ull) __hip_atomic_fetch_add(rm + i, fm[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        if (fc[i] != 0u) __hip_atomic_fetch_add(rh + i, fc[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    }
    ++nsync;
    if (!row_sync(a, row, nsync * (uint32_t)nseg, s)) return false;
    l1_invalidate();                                     // lines this call read before may be stale in the L1
    // 3. the fine bin holding the target (thread t: fine bins FBN-1-t*FPT .. descending), then its candidates
    constexpr int FPT = FBN / BLOCK;
    uint64_t v[LPT] = {};
    uint32_t cnt_v[FPT];
#pragma unroll
    for (int j = 0; j < FPT; ++j) {
        const int f = FBN - 1 - (FPT * tid + j);
        v[j] = __hip_atomic_load(rm + f, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        cnt_v[j] = __hip_atomic_load(rh + f, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    }
    const double rest = target - above_b;
    uint64_t abf = 0ull;
    const uint64_t tfx = rest > 0.0 ? (uint64_t)(rest * FXS) : 0ull;
    // desc_locate over the FBN fine bins (LPT slots per thread, the first FPT used)
    int d;
    {
        uint64_t sum = 0ull;
#pragma unroll
        for (int j = 0; j < FPT; ++j) sum += v[j];
        uint64_t tot;
        uint64_t run = block_excl_scan<uint64_t>(sum, s.red.u64b, &tot);
        int hit = 0x7fffffff;
        uint64_t ab = 0ull;
#pragma unroll
        for (int j = 0; j < FPT; ++j) {
            if (hit == 0x7fffffff && v[j] != 0ull && run + v[j] >= tfx) { hit = FPT * tid + j; ab = run; }
            run += v[j];
        }
        d = block_min_i32(hit, s.red);
        if (d == 0x7fffffff) d = -1;
        if (d >= 0 && hit == d) s.red.u64b[0] = ab;
        __syncthreads();
        abf = d >= 0 ? s.red.u64b[0] : 0ull;
        __syncthreads();
    }
    if (d < 0) return false;                             // uniform
    const uint32_t fb = (uint32_t)(FBN - 1 - d);
    uint32_t cab = 0u;                                   // candidates in the fine bins above fb
#pragma unroll
    for (int j = 0; j < FPT; ++j) cab += (FPT * tid + j) < d ? cnt_v[j] : 0u;
    uint32_t cabt;
    (void)block_excl_scan<uint32_t>(cab, s.wsum, &cabt);
    if (tid == 0) s.count = 0u;
    __syncthreads();
    uint64_t* regC = my + LSC + 2 * LLR;
    seg_elems(a, rc, s, lo0, hi, bmpen, [&](bool ok, float, uint32_t kq, uint64_t c) {
        const bool in = ok && c >= Xlo && (kq >> LB_SHIFT) == b && ((kq >> FSH) & (uint32_t)(FBN - 1)) == fb;
        wave_append(in, c, regC, &s.count, (uint32_t)LLR);
    });
    if (tid == 0) my[LS_NBD] = s.count;
    ++nsync;
    if (!row_sync(a, row, nsync * (uint32_t)nseg, s)) return false;
    l1_invalidate();                                     // lines this call read before may be stale in the L1
    // 4. the walk inside the fine bin
    const int n = load_lists(a, rc, 2, LS_NBD, s);
    if (n < 0) return false;
    const int ic = large_walk(s, n, Xlo, above_b + (double)abf / FXS, target, mx, Td, &cum);
    if (ic < 0) return false;
    pick = s.cand[ic];
    before = cabt + (uint32_t)ic;
    return true;
}

// This segment's part of a large row (see above).
__device__ __forceinline__ void large_segment(const Args& a, const RowCtx& rc, int seg, Shared& s, const SegStart& g) {
    const int tid = threadIdx.x;
    const int row = rc.row, nseg = rc.nseg;
    const fs_row_params& p = rc.p;
    const int lo0 = g.seg_lo;
    const int hi = seg == nseg - 1 ? a.V : lo0 + g.ntiles * TILE;      // the last segment takes the partial tile
    uint64_t* my = a.cand + slot_of(rc, seg) * CAP;
    if (ld_agent(a.dirty) != 0) return;                 // a dirty context: the merge samples the row alone
    if (seg == 0 && tid == 0) my[LS_STATUS] = 0ull;
    // Penalties: a repetition penalty alone as an exact bitmap of the window's ids over this segment (in s.ids, built
    // once for every pass), frequency / presence with the per-tile count table over the gathered window.
    const bool bmpen = rc.pen && rc.rep_on && !rc.fp_on && ((hi - lo0 + TILE - 1) / TILE) * TILE <= 32 * WIDS;
    if (bmpen) {
        uint32_t* bm = reinterpret_cast<uint32_t*>(s.ids);
        for (int i = tid; i < WIDS; i += BLOCK) bm[i] = 0u;
        __syncthreads();
        for (int64_t i = rc.b + tid; i < rc.len; i += BLOCK) {
            const int id = hist_at(a, rc, i);
            if (id >= lo0 && id < hi) atomicOr(&bm[(uint32_t)(id - lo0) >> 5], 1u << ((uint32_t)(id - lo0) & 31u));
        }
        __syncthreads();
    } else if (rc.pen) {
        gather_window(a, rc, lo0, hi, s);
    }
    // ---- P1: extremes, ordered count, coarse-bin counts of the k-th's search (k < V)
    const bool need_kth = rc.k < a.V;
    uint32_t* hc = reinterpret_cast<uint32_t*>(s.cand);  // [LB]
    if (need_kth) {
        for (int i = tid; i < LB; i += BLOCK) hc[i] = 0u;
        __syncthreads();
    }
    uint64_t cmax = 0ull, cmin = ~0ull;
    uint32_t nv = 0u;
    // Every token a candidate (k >= V): the logits within cut = CUT_C * T of the workgroup's running maximum (over its
    // tiles so far, the current one included) go to an LDS list; the others (masses below e^-CUT_C of the row's, since
    // the running maximum never exceeds the row's) are summed in single precision relative to that maximum, rescaled
    // when it rises. Both depend only on the data (a barrier per tile), so the sums are deterministic.
    const bool fastc = !need_kth;
    const float cut = CUT_C * p.temperature;
    const float inv_tl2 = 1.4426950408889634f / p.temperature;   // log2(e) / T: the rest's masses as powers of 2
    float ref = -__builtin_huge_valf();
    float tacc = 0.0f;
    constexpr uint32_t WREG = CAP / NWAVES;              // each wave's own part of the LDS list: no atomics
    uint64_t* const wl = s.cand + (tid / WAVE) * WREG;
    uint32_t wcnt = 0u;                                  // wave-uniform
    // (fastc: the extremes tracked as floats with their first / last index, as the composite order ranks ties)
    float bmax = -__builtin_huge_valf(), bmin = __builtin_huge_valf();
    int bmax_id = -1, bmin_id = -1;
    if (!fastc) {
        seg_elems(a, rc, s, lo0, hi, bmpen, [&](bool ok, float, uint32_t kq, uint64_t c) {
            if (ok) {
                cmax = c > cmax ? c : cmax;
                cmin = c < cmin ? c : cmin;
                ++nv;
                if (need_kth) atomicAdd(&hc[kq >> LB_SHIFT], 1u);
            }
        });
    } else {
        seg_elems_g(a, rc, s, lo0, hi, bmpen, [](bool, float, uint32_t, uint64_t) {}, [&](const float (&x)[TPT], int lo) {
            const bool full = lo + TILE <= hi;
            bool valid[TPT];
            float tm = -__builtin_huge_valf();
#pragma unroll
            for (int i = 0; i < TPT; ++i) {
                valid[i] = (full || elem_id(lo, i) < hi) && x[i] == x[i];
                tm = valid[i] && x[i] > tm ? x[i] : tm;
                nv += valid[i] ? 1u : 0u;
                if (valid[i] && x[i] <= bmin) { bmin = x[i]; bmin_id = elem_id(lo, i); }
                if (valid[i] && (x[i] > bmax || bmax_id < 0)) { bmax = x[i]; bmax_id = elem_id(lo, i); }
            }
            // the running maximum of the workgroup's tiles so far (this one included), behind a barrier
            uint32_t mk = wave_max(key_of(tm));
            uint32_t* tmw = s.tmx[((lo - lo0) / TILE) & 1];
            if (lane_id() == 0) tmw[tid / WAVE] = mk;
            __syncthreads();
#pragma unroll
            for (int w = 0; w < NWAVES; ++w) mk = tmw[w] > mk ? tmw[w] : mk;
            const float nr = mk > key_of(-__builtin_huge_valf()) ? val_of(mk) : -__builtin_huge_valf();
            if (nr > ref) {
                if (tacc != 0.0f) tacc *= __builtin_amdgcn_exp2f((ref - nr) * inv_tl2);
                ref = nr;
            }
            const float thr = ref - cut;
            uint32_t cm = 0u;
#pragma unroll
            for (int i = 0; i < TPT; ++i) {
                const bool cand = valid[i] && x[i] >= thr;
                cm |= cand ? 1u << i : 0u;
                const float t = __builtin_amdgcn_exp2f((x[i] - ref) * inv_tl2);
                tacc += (valid[i] && !cand) ? t : 0.0f;
            }
            if (__ballot(cm != 0u) != 0ull) {
#pragma unroll
                for (int i = 0; i < TPT; ++i) {
                    const bool cand = (cm >> i) & 1u;
                    const uint64_t m = __ballot(cand);
                    if (m != 0ull) {
                        const uint32_t pos = wcnt + mbcnt(m);
                        if (cand && pos < WREG) wl[pos] = comp_of(key_of(x[i]), (uint32_t)elem_id(lo, i));
                        wcnt += (uint32_t)__popcll(m);
                    }
                }
            }
        });
    }
    if (fastc) {
        cmax = bmax_id >= 0 ? comp_of(key_of(bmax), (uint32_t)bmax_id) : 0ull;
        cmin = bmin_id >= 0 ? comp_of(key_of(bmin), (uint32_t)bmin_id) : ~0ull;
    }
    FS_MARK(1);                                          // P1 streamed
    if (fastc && lane_id() == 0) s.wcnt[tid / WAVE] = wcnt;
    cmax = block_max_u64(cmax, s.red);
    cmin = block_min_u64(cmin, s.red);
    uint32_t nseg_v;
    (void)block_excl_scan<uint32_t>(nv, s.wsum, &nseg_v);
    if (fastc) {
        // the list cut again at this segment's maximum; its survivors to gather region 0 of the slot, their exact
        // masses and the rest's summed relative to that maximum
        // (the list's order depends on the waves' timing: its masses are summed in fixed point, order-free)
        uint32_t n0 = 0u, wofs[NWAVES];                   // (the reductions above end with barriers)
        bool wovf = false;
#pragma unroll
        for (int w = 0; w < NWAVES; ++w) {
            wofs[w] = n0;
            wovf |= s.wcnt[w] > WREG;
            n0 += s.wcnt[w];
        }
        const float smax = nseg_v > 0u ? val_of(comp_key(cmax)) : -__builtin_huge_valf();
        const double Td = (double)p.temperature;
        double tsum = 0.0;
        if (tacc != 0.0f) tsum = (double)tacc * exp((double)(ref - smax) / Td);
        uint64_t cfx = 0ull, tfx = 0ull;
        if (tid == 0) s.nfast = 0u;
        __syncthreads();
        if (!wovf && smax > -__builtin_huge_valf() && smax < __builtin_huge_valf()) {
            for (uint32_t b0 = 0u; b0 < n0; b0 += BLOCK) {
                const uint32_t i = b0 + (uint32_t)tid;
                int w = 0;
#pragma unroll
                for (int v = 1; v < NWAVES; ++v) w = i >= wofs[v] ? v : w;
                const uint64_t c = i < n0 ? s.cand[w * WREG + (i - wofs[w])] : 0ull;
                const float x = val_of(comp_key(c));
                const bool keep = i < n0 && x >= smax - cut;
                if (i < n0) {
                    const uint64_t m = (uint64_t)(mass_of(x, smax, Td) * CFXS + 0.5);
                    if (keep) cfx += m; else tfx += m;
                }
                wave_append(keep, c, my + LSC, &s.nfast, (uint32_t)LLR);
            }
        }
        uint64_t t_;
        (void)block_excl_scan<uint64_t>(cfx, s.red.u64b, &t_);
        const double csum = (double)t_ / CFXS;
        (void)block_excl_scan<uint64_t>(tfx, s.red.u64b, &t_);
        tsum = block_sum_f64(tsum, s.red) + (double)t_ / CFXS;
        if (tid == 0) {
            const bool ok = !wovf && s.nfast <= (uint32_t)LLR;
            my[LS_FN] = ok ? s.nfast : 0xFFFFFFFFull;
            my[LS_FC] = (uint64_t)__double_as_longlong(csum);
            my[LS_FT] = (uint64_t)__double_as_longlong(tsum);
        }
    }
    uint32_t* rh = a.rhist + (int64_t)row * RBINS;
    if (need_kth)
        for (int i = tid; i < LB; i += BLOCK)
            if (hc[i] != 0u) __hip_atomic_fetch_add(rh + i, hc[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    if (tid == 0) { my[LS_MAX] = cmax; my[LS_MIN] = cmin; my[LS_NV] = nseg_v; }
    if (!row_sync(a, row, (uint32_t)nseg, s)) return;
    FS_MARK(5);                                          // past the first barrier
    if (fastc && nseg <= WAVE) {
        // wave 0 reads every segment's published line once: the row's extremes and count, and the cut's decision
        // (large_cut below, in wave reductions); segment 0's wave 0 then samples a short list at once
        if (tid < WAVE) {
            const int lane = tid;
            uint64_t smx = 0ull, smn = ~0ull, snv = 0ull, sfn = 0ull;
            double sfc = 0.0, sft = 0.0;
            if (lane < nseg) {
                const uint64_t* sl = a.cand + slot_of(rc, lane) * CAP;
                smx = sl[LS_MAX]; smn = sl[LS_MIN]; snv = sl[LS_NV]; sfn = sl[LS_FN];
                sfc = __longlong_as_double((long long)sl[LS_FC]);
                sft = __longlong_as_double((long long)sl[LS_FT]);
            }
            auto add_u = [](uint64_t x_, uint64_t y_) { return x_ + y_; };
            auto add_d = [](double x_, double y_) { return x_ + y_; };
            const uint64_t rmx = wave_max(smx), rmn = wave_min(smn), rnv = wave_allreduce(snv, add_u);
            const float mxf = val_of(comp_key(rmx));
            const bool fin = rnv != 0ull && mxf > -__builtin_huge_valf() && mxf < __builtin_huge_valf();
            const double Td = (double)p.temperature;
            const double F = fin && lane < nseg && snv != 0ull
                                 ? exp(((double)val_of(comp_key(smx)) - (double)mxf) / Td) : 0.0;
            const double sc = wave_allreduce(F * sfc, add_d), st = wave_allreduce(F * sft, add_d);
            const bool ovf = wave_max(sfn > (uint64_t)LLR ? 1u : 0u) != 0u;
            const uint64_t nft = wave_allreduce(sfn > (uint64_t)LLR ? 0ull : sfn, add_u);
            const double u = row_u(a, row);
            bool min_in = false;
            const bool fast = fin && cut_decide(p, sc, st, nft, ovf, u, min_in);
            bool done = false;
            if (fast && seg == 0 && nft <= (uint64_t)WAVE) {
                FS_MARK(6);
                if (!wave_cut_finish(a, rc, my, mxf, CUT_C * p.temperature, Td, st, (uint32_t)rnv, (int)rnv,
                                     comp_key(rmx), rmn, u, min_in, (uint32_t)sfn))
                    row_abandon(a, row);
                FS_MARK(8);
                done = true;
            }
            if (lane == 0) {
                s.red.u64[0] = rmx; s.red.u64b[0] = rmn; s.red.misc[0] = (uint32_t)rnv;
                s.red.misc[1] = (fast ? 1u : 0u) | (done ? 2u : 0u) | (min_in ? 4u : 0u);
                s.red.dmisc[0] = st; s.red.dmisc[1] = u;
            }
        }
        __syncthreads();
        cmax = s.red.u64[0]; cmin = s.red.u64b[0]; nv = s.red.misc[0];
        const uint32_t fl = s.red.misc[1];
        const double st = s.red.dmisc[0], u = s.red.dmisc[1];
        __syncthreads();                                 // Red is reused below
        if (fl & 1u) {
            if (seg == 0 && !(fl & 2u))
                cut_finish_block(a, rc, s, my, val_of(comp_key(cmax)), comp_key(cmax), cmin, nv, (int)nv, st, u,
                                 (fl & 4u) != 0u);
            return;
        }
    } else {
    // row-wide: extremes, count; the k-th's coarse bin from the row histogram
        uint64_t mx_ = 0ull, mn_ = ~0ull, nv_ = 0ull;
        for (int j = tid; j < nseg; j += BLOCK) {
            const uint64_t* sl = a.cand + slot_of(rc, j) * CAP;
            mx_ = sl[LS_MAX] > mx_ ? sl[LS_MAX] : mx_;
            mn_ = sl[LS_MIN] < mn_ ? sl[LS_MIN] : mn_;
            nv_ += sl[LS_NV];
        }
        cmax = block_max_u64(mx_, s.red);
        cmin = block_min_u64(mn_, s.red);
        uint64_t t_;
        (void)block_excl_scan<uint64_t>(nv_, s.red.u64b, &t_);
        nv = (uint32_t)t_;
    }
    const uint32_t ntot = nv;
    if (ntot == 0u) {                                    // every logit NaN: no order to sample from
        if (seg == 0 && tid == 0) { my[LS_TOK] = 0ull; my[LS_STATUS] = 1ull; }
        return;
    }
    const uint32_t kmax = comp_key(cmax);
    const float mx = val_of(kmax);
    const double Td = (double)p.temperature;
    const int keff = (uint32_t)rc.k < ntot ? rc.k : (int)ntot;
    if (fastc && nseg > WAVE && large_cut(a, rc, s, seg, my, mx, kmax, cmin, ntot, keff)) return;
    uint32_t bk = 0xFFFFFFFFu, abk = 0u;                 // the k-th's coarse bin (none: every element a candidate)
    if ((uint32_t)keff < ntot) {
        uint32_t cv[LPT];
#pragma unroll
        for (int j = 0; j < LPT; ++j) {
            const int b = LB - 1 - (LPT * tid + j);
            cv[j] = b <= (int)(0xFF800000u >> LB_SHIFT) ? rh[b] : 0u;   // the counters above the keys are not counts
        }
        const int dk = desc_locate<uint32_t>(cv, (uint32_t)keff, &abk, s.wsum, s);
        if (dk < 0) { row_abandon(a, row); return; }    // uniform (the counts disagree with ntot: never expected)
        bk = (uint32_t)(LB - 1 - dk);
    }
    // ---- P2: candidate masses above bk, bin bk gathered
    FS_MARK(6);                                          // P2 starts
    uint64_t* hm = reinterpret_cast<uint64_t*>(s.cand);  // [LB] fixed-point masses
    for (int i = tid; i < LB; i += BLOCK) hm[i] = 0ull;
    if (tid == 0) s.count = 0u;
    __syncthreads();
    // An element whose mass exp((v - mx) / T) is below e^-32 (1.3e-14) adds 0 to the fixed-point histogram (2^-44
    // units) and at most 262144 * 1.3e-14 to S (>= 1) altogether: it takes a single-precision exp (relative error
    // ~1e-7 of a negligible term) instead of the fp64 one, so S stays within ~1e-14 relative of the exact sum.
    double part = 0.0;
    float part_tiny = 0.0f;
    const float inv_tf = 1.0f / p.temperature;
    uint64_t* regA = my + LSC;
    seg_elems(a, rc, s, lo0, hi, bmpen, [&](bool ok, float x, uint32_t kq, uint64_t c) {
        const uint32_t b = kq >> LB_SHIFT;
        if (ok && (bk == 0xFFFFFFFFu || b > bk)) {
            const float d = x - mx;                      // fp32 subtraction, as ferro
            const float zf = d * inv_tf;
            if (!(zf < -32.0f)) {                    // (NaN, from inf - inf, stays on the exact path)
                const double m = exp((double)d / Td);
                part += m;
                atomicAdd(reinterpret_cast<unsigned long long*>(&hm[b]), (unsigned long long)(m * FXS + 0.5));
            } else {
                part_tiny += __expf(zf);
            }
        }
        wave_append(ok && b == bk, c, regA, &s.count, (uint32_t)LLR);
    });
    part += (double)part_tiny;
    FS_MARK(2);                                          // P2 streamed
    const double shi = block_sum_f64(part, s.red);      // its barriers also complete the LDS histogram
    uint64_t* rm = a.rmass + (int64_t)row * LB;
    for (int i = tid; i < LB; i += BLOCK)
        if (hm[i] != 0ull) __hip_atomic_fetch_add(rm + i, hm[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    if (tid == 0) {
        my[LS_SHI] = (uint64_t)__double_as_longlong(shi);
        my[LS_NBK] = s.count;
    }
    if (!row_sync(a, row, 2u * (uint32_t)nseg, s)) return;
    FS_MARK(7);                                          // past the second barrier
    double S = sum_slots_f64(a, rc, LS_SHI, s);
    uint64_t Xk = cmin;
    uint64_t fx_bk = 0ull;                               // fixed-point mass of bin bk's candidates
    if (bk != 0xFFFFFFFFu) {
        const int n = load_lists(a, rc, 0, LS_NBK, s);
        const int need = keff - (int)abk;                // >= 1: the k-th lies in bin bk
        if (n < need || need < 1) { row_abandon(a, row); return; }   // uniform
        Xk = s.cand[need - 1];
        double sb = 0.0;
        uint64_t fb = 0ull;
        for (int i = tid; i < need; i += BLOCK) {
            const double m = mass_of(val_of(comp_key(s.cand[i])), mx, Td);
            sb += m;
            fb += (uint64_t)(m * FXS + 0.5);
        }
        S += block_sum_f64(sb, s.red);
        uint64_t t_;
        (void)block_excl_scan<uint64_t>(fb, s.red.u64b, &t_);
        fx_bk = t_;
    }
    FS_MARK(3);                                          // past the second barrier: S and Xk known
    if (S != S) {                                        // an infinite maximum: every mass NaN, nothing cut, the
        if (seg == 0 && tid == 0) {                      // draw falls through to the last candidate (sampler.cpp:43-49)
            my[LS_TOK] = (uint64_t)comp_id(Xk) | ((uint64_t)(uint32_t)keff << 32);
            my[LS_XK] = Xk;
            my[LS_S] = (uint64_t)__double_as_longlong(S);
            my[LS_KEFF] = (uint64_t)keff | ((uint64_t)kmax << 32);
            my[LS_STATUS] = 1ull;
        }
        return;
    }
    const uint32_t kk = comp_key(Xk);
    uint64_t mv[LPT];                                    // the candidates' mass histogram, descending positions
#pragma unroll
    for (int j = 0; j < LPT; ++j) {
        const int b = LB - 1 - (LPT * tid + j);
        mv[j] = rm[b] + ((uint32_t)b == bk ? fx_bk : 0ull);
    }
    // min-p: the smallest key whose pr reaches pr[0] * min_p (pr[0] = 1 / S): a search over keys, no pass
    uint64_t Xm = 0ull;
    uint32_t km = 0xFFFFFFFFu;
    if (p.min_p > 0.0f) {
        const double thr = (1.0 / S) * (double)p.min_p;
        auto okm = [&](uint32_t key) { return mass_of(val_of(key), mx, Td) / S >= thr; };
        if (!okm(kmax)) {
            Xm = cmax;
        } else {
            uint32_t lo = kk, h = kmax;
            while (lo < h) {
                const uint32_t mid = lo + ((h - lo) >> 1);
                if (okm(mid)) h = mid; else lo = mid + 1u;
            }
            km = lo;
            Xm = (uint64_t)lo << 32;
        }
    }
    const bool need_m = p.min_p > 0.0f && Xm != cmax;
    // ---- P3: top-p's crossing bin gathered, with min-p's counts and masses
    uint64_t Xc = 0ull;
    uint32_t keep_c = 0u, cnt_m = 0u;
    double tot_c = 0.0, sum_m = 0.0;
    uint64_t cl_m = ~0ull;
    int nc = -1;
    uint32_t bc = 0xFFFFFFFFu;
    uint32_t bd_pred = 0xFFFFFFFFu;                      // the draw's bin, when P3 can gather it too
    bool refined_c = false;                              // top-p's crossing bin was refined (gather region 2 in use)
    uint32_t nsync = 2u;
    if (p.top_p < 1.0f || need_m) {
        const double tgt = (double)p.top_p * S;
        double above_c = 0.0;
        if (p.top_p < 1.0f) {
            uint64_t abfx = 0ull;
            int dc = desc_locate<uint64_t>(mv, (uint64_t)(tgt * FXS), &abfx, s.red.u64b, s);
            if (dc < 0) dc = LB - 1 - (int)(kk >> LB_SHIFT);   // the total rounds below the target: the last bin
            bc = (uint32_t)(LB - 1 - dc);
            above_c = (double)abfx / FXS;
            if (p.min_p <= 0.0f) {
                // Without min-p the kept total lies in [tgt, min(S, tgt + the largest mass in bin bc)] (top-p keeps
                // through the crossing candidate, sampler.cpp:44). When the draw u * tot falls in one coarse bin over
                // that whole range, this pass gathers that bin too and no draw pass is needed.
                const uint32_t top_key = ((bc << LB_SHIFT) | ((1u << LB_SHIFT) - 1u)) < kmax
                                             ? ((bc << LB_SHIFT) | ((1u << LB_SHIFT) - 1u)) : kmax;
                const double mhi = mass_of(val_of(top_key), mx, Td);
                const double thi = tgt + mhi < S ? tgt + mhi : S;
                const double u0 = row_u(a, rc.row);
                uint64_t ab_;
                const int d0 = desc_locate<uint64_t>(mv, (uint64_t)(u0 * tgt * (1.0 - 1e-12) * FXS), &ab_, s.red.u64b, s);
                const int d1 = desc_locate<uint64_t>(mv, (uint64_t)(u0 * thi * (1.0 + 1e-12) * FXS), &ab_, s.red.u64b, s);
                if (d0 >= 0 && d0 == d1 && (uint32_t)(LB - 1 - d0) != bc) bd_pred = (uint32_t)(LB - 1 - d0);
            }
        }
        uint32_t my_ca = 0u, my_cm = 0u;
        double my_sm = 0.0;
        uint64_t my_cl = ~0ull;
        if (tid == 0) { s.count = 0u; s.tmax = 0u; }
        __syncthreads();
        uint64_t* regB = my + LSC + LLR;
        uint64_t* regC = my + LSC + 2 * LLR;
        seg_elems(a, rc, s, lo0, hi, bmpen, [&](bool ok, float x, uint32_t kq, uint64_t c) {
            const bool cand = ok && c >= Xk;
            if (cand && bc != 0xFFFFFFFFu && (kq >> LB_SHIFT) > bc) ++my_ca;
            if (cand && need_m && kq >= km) {
                ++my_cm;
                my_sm += mass_of(x, mx, Td);
                my_cl = c < my_cl ? c : my_cl;
            }
            wave_append(cand && (kq >> LB_SHIFT) == bc, c, regB, &s.count, (uint32_t)LLR);
            wave_append(cand && (kq >> LB_SHIFT) == bd_pred, c, regC, &s.tmax, (uint32_t)LLR);
        });
        uint32_t ca_t, cm_t;
        (void)block_excl_scan<uint32_t>(my_ca, s.wsum, &ca_t);
        (void)block_excl_scan<uint32_t>(my_cm, s.wsum, &cm_t);
        const double sm_t = block_sum_f64(my_sm, s.red);
        const uint64_t cl_t = block_min_u64(my_cl, s.red);
        if (tid == 0) {
            my[LS_NBC] = s.count;
            my[LS_CA] = ca_t;
            my[LS_CNTM] = cm_t;
            my[LS_SUMM] = (uint64_t)__double_as_longlong(sm_t);
            my[LS_CLM] = cl_t;
            my[LS_NBD] = s.tmax;
        }
        FS_MARK(8);                                      // P3 streamed
        nsync = 3u;
        if (!row_sync(a, row, 3u * (uint32_t)nseg, s)) return;
        FS_MARK(9);                                      // past the third barrier
        const uint32_t ca_c = (uint32_t)sum_slots_u64(a, rc, LS_CA, s);
        if (need_m) {
            cnt_m = (uint32_t)sum_slots_u64(a, rc, LS_CNTM, s);
            sum_m = sum_slots_f64(a, rc, LS_SUMM, s);
            uint64_t c_ = ~0ull;
            for (int j = tid; j < nseg; j += BLOCK) {
                const uint64_t v = a.cand[slot_of(rc, j) * CAP + LS_CLM];
                c_ = v < c_ ? v : c_;
            }
            cl_m = block_min_u64(c_, s.red);
        }
        if (p.top_p < 1.0f) {
            nc = load_lists(a, rc, 1, LS_NBC, s);
            if (nc < 0) {
                // a crowded crossing bin: one level of finer bins (its gather region is spent, and the draw's
                // pre-gathered bin is overwritten)
                uint64_t pk = 0ull;
                double cm = 0.0;
                uint32_t bf = 0u;
                if (!refine_bin(a, rc, s, seg, my, lo0, hi, bmpen, bc, Xk, above_c, tgt, mx, Td, nsync, pk, cm, bf)) {
                    row_abandon(a, row);
                    return;
                }
                Xc = pk;
                keep_c = ca_c + bf + 1u;
                tot_c = cm;
                bd_pred = 0xFFFFFFFFu;
                refined_c = true;
            } else {
                double cum = 0.0;
                const int ic = large_walk(s, nc, Xk, above_c, tgt, mx, Td, &cum);
                if (ic < 0) { row_abandon(a, row); return; }   // outside the bin's exact masses: the exact path
                Xc = s.cand[ic];
                keep_c = ca_c + (uint32_t)ic + 1u;
                tot_c = cum;
            }
        }
    }
    // the kept prefix: the largest of the three thresholds (sampler.cpp:43-44)
    uint64_t Xkeep = Xk, clast = Xk;
    uint32_t keep = (uint32_t)keff;
    double tot = S;
    if (p.min_p > 0.0f && Xm > Xkeep) {
        Xkeep = Xm;
        if (Xm == cmax) { keep = 1u; tot = 1.0; clast = cmax; }
        else { keep = cnt_m; tot = sum_m; clast = cl_m; }
    }
    if (p.top_p < 1.0f && Xc > Xkeep) {
        Xkeep = Xc;
        keep = keep_c;
        tot = tot_c;
        clast = Xc;
    }
    // ---- P4: the draw r = u * tot (sampler.cpp:45-49) in its coarse bin
    const double u = row_u(a, rc.row);
    const double r = u * tot + 0.0;
    if (!(r > 0.0)) {                                    // r = 0: ferro's first candidate (r <= pr[0], sampler.cpp:48)
        if (seg == 0 && tid == 0) {
            my[LS_TOK] = (uint64_t)comp_id(cmax) | ((uint64_t)keep << 32);
            my[LS_XK] = Xk;
            my[LS_S] = (uint64_t)__double_as_longlong(S);
            my[LS_KEFF] = (uint64_t)keff | ((uint64_t)kmax << 32);
            my[LS_STATUS] = 1ull;
        }
        return;
    }
    uint64_t abd = 0ull;
    const int dd = desc_locate<uint64_t>(mv, (uint64_t)(r * FXS), &abd, s.red.u64b, s);
    if (dd < 0) { row_abandon(a, row); return; }
    const uint32_t bd = (uint32_t)(LB - 1 - dd);
    int nd;
    if (nc >= 0 && bd == bc) {
        nd = nc;                                         // the same bin is sorted in LDS already
    } else if (bd == bd_pred) {
        nd = load_lists(a, rc, 2, LS_NBD, s);           // gathered by P3
    } else {
        // after a refinement of top-p's bin the other segments may still read gather region 2: region 1 instead
        // (its lists were never read), read through an invalidated L1 (its counts were)
        const int rg = refined_c ? 1 : 2;
        const int rs = refined_c ? LS_NBC : LS_NBD;
        if (tid == 0) s.count = 0u;
        __syncthreads();
        uint64_t* regC = my + LSC + rg * LLR;
        seg_elems(a, rc, s, lo0, hi, bmpen, [&](bool ok, float, uint32_t kq, uint64_t c) {
            wave_append(ok && c >= Xkeep && (kq >> LB_SHIFT) == bd, c, regC, &s.count, (uint32_t)LLR);
        });
        if (tid == 0) my[rs] = s.count;
        FS_MARK(10);                                     // P4 streamed
        ++nsync;
        if (!row_sync(a, row, nsync * (uint32_t)nseg, s)) return;
        FS_MARK(11);                                     // past the last barrier
        if (refined_c) l1_invalidate();
        nd = load_lists(a, rc, rg, rs, s);
    }
    uint64_t pick = 0ull;
    if (nd < 0) {                                        // a crowded draw bin: one level of finer bins
        double cm = 0.0;
        uint32_t bf = 0u;
        if (!refine_bin(a, rc, s, seg, my, lo0, hi, bmpen, bd, Xkeep, (double)abd / FXS, r, mx, Td, nsync, pick, cm,
                        bf)) {
            row_abandon(a, row);
            return;
        }
    } else {
        double cum = 0.0;
        const int id = large_walk(s, nd, Xkeep, (double)abd / FXS, r, mx, Td, &cum);
        if (id >= 0) {
            pick = s.cand[id];
        } else if (!(id == -2 && comp_key(Xkeep) >> LB_SHIFT == bd)) {
            row_abandon(a, row);                         // a rounding step at the bin edge: the exact path
            return;
        }
    }
    if (pick == 0ull) pick = clast;                      // past the last kept candidate
    if (seg == 0 && tid == 0) {
        my[LS_TOK] = (uint64_t)comp_id(pick) | ((uint64_t)keep << 32);
        my[LS_XK] = Xk;
        my[LS_S] = (uint64_t)__double_as_longlong(S);
        my[LS_KEFF] = (uint64_t)keff | ((uint64_t)kmax << 32);
        my[LS_STATUS] = 1ull;
    }
}

// ------------------------------------------------------------------------------------------------ row layout
// By default every row has nseg segments of seg_tiles tiles. With a.balance, each XCD splits its W workgroups among
// its R rows (x, x + XCDS, ...) by the rows' cost per tile, so that rows with a large k, which cost up to three
// times a greedy row per tile, get more segments and a mixed batch's rows finish together. Every workgroup of the
// XCD computes the same split from the same parameters with integer arithmetic. Costs (per tile, relative to a
// greedy row = 100; measured on MI355X on uniform B=256 x V=262144 batches): k = 64 119, k = 256 158, k = 2048
// 292, whole-row sampling (k > 2048) about 400; frequency/presence penalties x1.25, a repetition penalty x1.05.
// What the cost needs of a row's parameters: two 16-byte buffer loads (temperature, top_k, top_p, min_p; repetition,
// frequency, presence, repeat_last_n). A segment workgroup requests them before its first tiles, behind a scheduling
// barrier, so that waiting for them (vector loads complete in order) does not wait for the tiles.
struct CostIn {
    float t, rep, fq, pr;
    int tk;
};
__device__ __forceinline__ CostIn cost_in(const Args& a, int row) {
    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(const_cast<fs_row_params*>(a.params), (short)0,
                                                                        a.B * (int)sizeof(fs_row_params), 0x00020000);
    const u32x4 lo = raw_buffer_load_u32x4(rs, row * (int)sizeof(fs_row_params), 0, 0);
    const u32x4 hi = raw_buffer_load_u32x4(rs, row * (int)sizeof(fs_row_params) + 16, 0, 0);
    CostIn c;
    c.t = __uint_as_float(lo.x); c.tk = (int)lo.y;
    c.rep = __uint_as_float(hi.x); c.fq = __uint_as_float(hi.y); c.pr = __uint_as_float(hi.z);
    return c;
}
__device__ __forceinline__ uint32_t row_cost(const Args& a, const CostIn& in) {
    const float t = in.t, rep = in.rep, fq = in.fq, pr = in.pr;
    const int tk = in.tk;
    if (t <= 0.0f || tk == 1) return 100u;
    const int k = (tk > 0 && tk < a.V) ? tk : a.V;
    float c;
    if (k > KMAX) {
        c = 400.0f;
    } else {
        const float l = __log2f((float)k);
        c = k <= 64 ? 100.0f + 3.0f * l : (k <= 256 ? 119.0f + 19.5f * (l - 6.0f) : 158.0f + 44.7f * (l - 8.0f));
    }
    if (fq != 0.0f || pr != 0.0f) c *= 1.25f;
    else if (rep != 1.0f) c *= 1.05f;
    return (uint32_t)c;
}
// Lane r < R: row x + XCDS * r gets n segments (at most its tiles), its first workgroup being base among the XCD's W.
// in: lane r's row parameters (cost_in of row x + XCDS * r, or of row x past R).
__device__ __forceinline__ CostIn xcd_cost_in(const Args& a, int x) {
    const int R = (a.B - x + XCDS - 1) / XCDS;
    return cost_in(a, x + XCDS * (lane_id() < R ? lane_id() : 0));
}
__device__ __forceinline__ void xcd_layout(const Args& a, int x, const CostIn& in, uint32_t& n, uint32_t& base) {
    const int lane = lane_id();
    const int R = (a.B - x + XCDS - 1) / XCDS;          // rows on this XCD (1 <= R <= WAVE: the host checks B)
    const uint32_t W = (uint32_t)(a.nseg * ((a.B + XCDS - 1) / XCDS));
    const uint32_t tiles_row = (uint32_t)(a.V / TILE);
    const uint32_t w = lane < R ? row_cost(a, in) : 0u;  // lane r: row x + XCDS r's cost
    const uint32_t tot = (uint32_t)__builtin_amdgcn_readlane((int)wave_incl_scan_u32(w), WAVE - 1);
    const uint32_t spare = W - (uint32_t)R;
    const uint32_t num = spare * w;
    const uint32_t tq = tot > 0u ? tot : 1u;            // >= 100 per row
    const uint32_t f = num / tq, rem = num % tq;
    n = lane < R ? 1u + f : 0u;
    const uint32_t left = W - (uint32_t)__builtin_amdgcn_readlane((int)wave_incl_scan_u32(n), WAVE - 1);
    uint32_t rank = 0u;                                  // the largest remainders get the leftover workgroups
    for (int s2 = 0; s2 < R; ++s2) {
        const uint32_t r2 = (uint32_t)__builtin_amdgcn_readlane((int)rem, s2);
        rank += (r2 > rem || (r2 == rem && s2 < lane)) ? 1u : 0u;
    }
    if (lane < R && rank < left) n += 1u;
    const uint32_t cap = tiles_row < (uint32_t)(BLOCK - 1) ? tiles_row : (uint32_t)(BLOCK - 1);
    if (n > cap) n = cap;                                // workgroups past a row's tiles stay idle
    base = wave_incl_scan_u32(n) - n;
}
// The layout of row x + XCDS * q into rc (merging workgroups): its lane q of xcd_layout.
__device__ __forceinline__ void row_layout(const Args& a, RowCtx& rc) {
    if (!a.balance || rc.nseg == 0) return;
    uint32_t n, base;
    xcd_layout(a, rc.lx, xcd_cost_in(a, rc.lx), n, base);
    const int q = rc.row / XCDS;
    const uint32_t nq = (uint32_t)__builtin_amdgcn_readlane((int)n, q);
    const uint32_t st = ((uint32_t)(a.V / TILE) + nq - 1u) / nq;
    rc.st = (int)st;
    rc.nseg = (int)(((uint32_t)(a.V / TILE) + st - 1u) / st);
    rc.lbase = __builtin_amdgcn_readlane((int)base, q);
}

// The row's completion counter: the row histogram's last bin, which no ordered key reaches (keys of non-NaN values
// are at most +inf's, bin 4088). Segments add 1 (an L2 atomic); the merge role polls it.
__device__ __forceinline__ uint32_t* row_counter(const Args& a, int row) {
    return a.rhist + (int64_t)row * RBINS + (RBINS - 1);
}
static_assert(((0xFF800000u >> RSHIFT) < (uint32_t)(RBINS - 1)), "the counter bin lies above every ordered key");

// Merge role of the segment grid: one workgroup per row, placed after the segments on the row's XCD (slot x of
// the last XCDS * ceil(B / XCDS) workgroups merges rows x, x + XCDS, ...). Workgroups are dispatched in index
// order, so the row's segments are running or done when it starts: it waits for their count (an atomic that
// is not idempotent, so it executes in the L2 and is never folded into an L1-served load), invalidates its L1
// and reads the lists from the L2. The wait is bounded (a.merge_spins polls): past it FS_DEVERR_INTERNAL is
// raised, the context is marked dirty and the row is computed from its logits alone (exact, one workgroup); a
// dirty context computes every row that way until fs_device_error clears the workspace.
__device__ __forceinline__ void merge_role(const Args& a, int mi, Shared& s) {
    const int row = mi % XCDS + XCDS * (mi / XCDS);
    if (row >= a.B) return;
    FS_TAG(13, 2); FS_TAG(14, row); FS_TAG(15, 0);
    RowCtx rc = row_ctx(a, row);                     // the row's inputs are read while the segments run
    row_layout(a, rc);
    decode_hist_copy(a, row);                        // a decode step: while the segments run
    uint32_t* ctr = row_counter(a, row);
    if (threadIdx.x == 0) {
        // A context left dirty by an earlier give-up: its row histograms and counters may hold a late segment's
        // additions, so no segment output is trusted and the row is computed from its logits alone. Otherwise a
        // bounded wait for the row's segments; past it the context is marked dirty (a segment that finishes later
        // still adds to this row's counter and histogram) and this row, too, is computed alone.
        uint32_t alone = ld_agent(a.dirty) != 0 ? 1u : 0u;
        uint32_t spins = 0u;
        while (!alone && (a.merge_spins == 0u ||
                          (__hip_atomic_fetch_add(ctr, 0x10000u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) &
                           0xFFFFu) < (uint32_t)rc.nseg)) {
            if (++spins >= a.merge_spins) {
                atomicOr(a.err, FS_DEVERR_INTERNAL);
                __hip_atomic_store(a.dirty, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                // err[2..3]: the address of a host-mapped flag that the next call reads on the host (or 0)
                int32_t* hf = (int32_t*)ld_agent(reinterpret_cast<const uint64_t*>(a.err + 2));
                if (hf) __hip_atomic_store(hf, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
                alone = 1u;
                break;
            }
            __builtin_amdgcn_s_sleep(1);
        }
        s.misc_alone = alone;
    }
    FS_MARK(1);
    __syncthreads();
    const bool alone = s.misc_alone != 0u;
    Pre pre = {};
    if (!alone) {
        l1_invalidate();
        prefetch_lists(a, rc, pre);
        if (threadIdx.x == 0) *ctr = 0u;             // the bin is left at 0 with the rest of the row histogram
    }
    merge_row(a, rc, s, pre, alone);                 // one call site: the merge code is inlined once
}

// Segment kernel: one (row, segment) item per workgroup (rows sampled with k > KMAX only count themselves done),
// then the merge role.
// The fields a workgroup needs first come as separate leading parameters: gfx950 preloads those into SGPRs at
// wave launch (build flag -amdgpu-kernarg-preload-count), so the first tile loads wait for no argument load.
__global__ __launch_bounds__(BLOCK, 4) void segment_kernel(const float* logits, int64_t ld, int B, int V, int nseg,
                                                           int seg_tiles, const fs_row_params* params,
                                                           const int64_t* hist_off, Args a) {
    static_assert(KMAX + TILE <= CAP, "a compacted buffer plus one tile must fit the candidate buffer");
    __shared__ __align__(16) Shared s;
    a.logits = logits; a.ld = ld; a.B = B; a.V = V; a.nseg = nseg; a.seg_tiles = seg_tiles; a.params = params;
    a.hist_off = hist_off;
    // One (row, segment) item per workgroup. Workgroup i runs on XCD i % XCDS (round-robin dispatch): slot
    // x = i % XCDS takes the rows x, x + XCDS, ..., all segments of a row in consecutive rounds, so a row's segments
    // share one XCD and its L2 (the row histogram). Slots past the last row return at once.
    const unsigned seg_grid = (unsigned)(XCDS * a.nseg * ((a.B + XCDS - 1) / XCDS));
    FS_MARK(0);
    for (int i_ = 1; i_ < 13; ++i_) FS_TAG(i_, 0);
    FS_TAG(13, 0);
    if (blockIdx.x >= seg_grid) {
        merge_role(a, (int)(blockIdx.x - seg_grid), s);
        FS_MARK(4);
        FS_FLUSH();
        return;
    }
    const int x = (int)(blockIdx.x % (unsigned)XCDS);
    const int j = (int)(blockIdx.x / (unsigned)XCDS);
    int q = __builtin_amdgcn_readfirstlane(j / a.nseg);          // uniform: lets the compiler use scalar loads
    int seg = j - q * a.nseg;
    int row = x + XCDS * q;
    if (row >= a.B && !a.balance) return;
    float buf[PF][TPT];
    // the layout's parameter loads come first, then the default layout's tiles, then the row's parameters; a balanced
    // layout that moves this workgroup requests its own tiles and parameters
    CostIn cin = {};
    if (a.balance) cin = xcd_cost_in(a, x);
    __builtin_amdgcn_sched_barrier(0);
    SegStart g = a.balance ? seg_start<true>(a, row < a.B ? row : a.B - 1, seg, a.seg_tiles, buf)
                           : seg_start<false>(a, row < a.B ? row : a.B - 1, seg, a.seg_tiles, buf);
    RowCtx rc = row_ctx(a, row < a.B ? row : a.B - 1);
    int st = a.seg_tiles, nsr = a.nseg, lbase = q * a.nseg;
    if (a.balance) {
        uint32_t n, base;
        xcd_layout(a, x, cin, n, base);
        const uint64_t mine = __ballot((uint32_t)j >= base && (uint32_t)j < base + n);
        if (mine == 0ull) return;                        // past the XCD's rows (or a capped row's tiles): idle
        const int r = __ffsll((unsigned long long)mine) - 1;
        const uint32_t nr = (uint32_t)__builtin_amdgcn_readlane((int)n, r);
        lbase = __builtin_amdgcn_readlane((int)base, r);
        st = (int)(((uint32_t)(a.V / TILE) + nr - 1u) / nr);
        nsr = (a.V / TILE + st - 1) / st;
        const int nseg_r = __builtin_amdgcn_readfirstlane(j - lbase);
        if (nseg_r >= nsr) return;                       // the row's tiles are covered by its first nsr workgroups
        if (r != q || nseg_r != seg || st != a.seg_tiles) {
            const bool moved_row = r != q || row >= a.B;
            q = r;
            seg = nseg_r;
            row = x + XCDS * q;
            g = seg_start(a, row, seg, st, buf);
            if (moved_row) rc = row_ctx(a, row);
        }
    }
    FS_TAG(13, 1); FS_TAG(14, row); FS_TAG(15, seg);
    rc.st = st;
    rc.nseg = nsr;
    rc.lbase = lbase;
    if (!rc.large) process_segment(a, rc, seg, s, buf, g);
    else large_segment(a, rc, seg, s, g);           // the row's segments sample it together
    vm_drain();                                      // the list and meta stores are in the L2
    __syncthreads();
    if (threadIdx.x == 0) __hip_atomic_fetch_add(row_counter(a, row), 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    FS_MARK(4);
    FS_FLUSH();
}

// Merge kernel: one workgroup per row, for rows shorter than one tile (no segments; the segment lists are requested
// first, so their latency overlaps the row's parameter loads), or, with `alone`, every row sampled from its logits by
// one workgroup (a device whose XCD layout the segment grid's hand-off cannot rely on).
__global__ __launch_bounds__(BLOCK) void merge_kernel(int nseg, uint64_t* cand, uint32_t* meta, uint32_t* rhist,
                                                      const fs_row_params* params, int alone, Args a) {
    static_assert(2 * SMALL * 8 <= NBINS * 4, "rank-sort buffers alias the histogram");
    __shared__ __align__(16) Shared s;
    a.nseg = nseg; a.cand = cand; a.meta = meta; a.rhist = rhist; a.params = params;
    const int row = __builtin_amdgcn_readfirstlane((int)blockIdx.x);
    Pre pre = {};
    const RowCtx rc = row_ctx(a, row);
    if (!alone) prefetch_lists(a, rc, pre);
    decode_hist_copy(a, row);
    merge_row(a, rc, s, pre, alone != 0);
}

// fs_softcap_batch: the sampler's fused final-logit cap as a standalone elementwise pass.

hipError_t launch_segments(const Args& a, unsigned grid, hipStream_t st) {
    hipLaunchKernelGGL(segment_kernel, dim3(grid), dim3(BLOCK), 0, st, a.logits, a.ld, a.B, a.V, a.nseg, a.seg_tiles,
                       a.params, a.hist_off, a);
    return hipGetLastError();
}

hipError_t launch_merges(const Args& a, unsigned rows, int nseg, int alone, hipStream_t st) {
    hipLaunchKernelGGL(merge_kernel, dim3(rows), dim3(BLOCK), 0, st, nseg, a.cand, a.meta, a.rhist, a.params, alone, a);
    return hipGetLastError();
}

}  // namespace fs

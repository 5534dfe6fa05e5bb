// row_device.hpp - what the kernels that give a row one workgroup per segment share: the decode step's history copy and
// draw, and a row's end (outputs, a verification window's accepted prefix).
#ifndef FERRO_ROW_DEVICE_HPP
#define FERRO_ROW_DEVICE_HPP

#include "sampler_device.hpp"
#include "sampler_launch.hpp"

namespace fs {

// fs_decode_step_hp on the small-k kernel (the fused kernel's decode_hist_copy / row_u / decode_commit for this
// kernel): each segment's workgroup copies its share of the stream's history to the new histories; the draw is read
// from the stream without advancing it; after the token, wave 0 of the merging workgroup appends it and advances the
// stream (greedy rows draw nothing).
// The share of segment seg: ids [seg * n, (seg + 1) * n) of the row's history, n = its length over the row's segments,
// rounded up. The first SK_CP ids per thread are requested with the window's (cp_load) and stored once the logits are
// spent (cp_store), so the copy costs no round trip of its own. (Before, the merging workgroup copied the row's whole
// history, one id per thread and round trip: a decode step of 32 rows with 175 to 1225 ids each 13.1 us -> 12.5, the
// draw's early reads included.)
constexpr int SK_CP = 2;
struct SkCopy {
    int64_t b, e, nb;                      // this segment's ids [b, e) of the histories; the row's new offset
    int64_t h0, len;                       // the row's first id, its history's length
    int id[SK_CP];
};
__device__ __forceinline__ SkCopy sk_cp_load(const int64_t* hist_off, const int32_t* hist, int row, int seg, int nseg) {
    SkCopy c;
    const int64_t base = hist_off ? ld_const(hist_off) : 0;
    c.h0 = hist_off ? ld_const(hist_off + row) : 0;
    const int64_t e = hist_off ? ld_const(hist_off + row + 1) : 0;
    c.len = e - c.h0;
    const int64_t n = (c.len + nseg - 1) / nseg;
    c.b = c.h0 + n * seg < e ? c.h0 + n * seg : e;
    c.e = c.b + n < e ? c.b + n : e;
    c.nb = c.h0 - base + row;
#pragma unroll
    for (int r = 0; r < SK_CP; ++r) {
        const int64_t i = c.b + r * SK_LT + (int)threadIdx.x;
        c.id[r] = i < c.e ? hist[i] : 0;
    }
    return c;
}
__device__ __forceinline__ void sk_cp_store(const SkArgs& a, const SkCopy& c, int row, int seg) {
    const int64_t d = c.nb - c.h0;                          // new position minus old
#pragma unroll
    for (int r = 0; r < SK_CP; ++r) {
        const int64_t i = c.b + r * SK_LT + (int)threadIdx.x;
        if (i < c.e && i + d < a.out_cap) a.out_hist[i + d] = c.id[r];
    }
    constexpr int U = 8;                                   // a longer share: eight loads in flight
    for (int64_t i0 = c.b + SK_CP * SK_LT + (int)threadIdx.x; i0 < c.e; i0 += U * SK_LT) {
        int v[U];
#pragma unroll
        for (int r = 0; r < U; ++r) v[r] = i0 + r * SK_LT < c.e ? a.hist[i0 + r * SK_LT] : 0;
#pragma unroll
        for (int r = 0; r < U; ++r) {
            const int64_t i = i0 + r * SK_LT;
            if (i < c.e && i + d < a.out_cap) a.out_hist[i + d] = v[r];
        }
    }
    if (seg == 0 && threadIdx.x == 0) {
        const int64_t end = c.nb + c.len + 1;
        a.out_hist_off[row] = c.nb;
        if (row == a.B - 1) a.out_hist_off[a.B] = end;
        if (end > a.out_cap) atomicOr(a.err, FS_DEVERR_HIST_APPEND);
    }
}
struct SkDraw {
    double u;
    int idx;                               // a decode step: the stream's next index, before this draw
};
__device__ __forceinline__ SkDraw sk_draw(const SkArgs& a, int row) {
    SkDraw d;
    d.idx = 0;
    if (a.dmt) {
        const uint64_t* mt = a.dmt + (int64_t)row * MT_N;
        d.idx = a.didx[row];
        const uint64_t y = d.idx < MT_N ? mt[d.idx] : mt_twist_one(mt[0], mt[1], mt[MT_M]);
        d.u = mt_canonical(mt_temper(y));
    } else {
        d.u = a.u ? ld_const(a.u + row) : 0.0;              // (a scalar load: no wait before it is used)
    }
    return d;
}
// Wave 0 alone: w is LDS scratch of MT_N entries. The twist in three passes, each reading every value it needs
// before it writes: entries below N - M from old values only (all computed, then written); the rest in ascending
// chunks of one wave (each reads its own and the next old entry and a new one below N - M; entry N - 1 the new
// entry 0), so no entry is overwritten before it is read.
__device__ __forceinline__ void sk_decode_commit(const SkArgs& a, int row, bool sampled, int tok, const SkCopy& c,
                                                 int idx, uint64_t* w) {
    const int lane = lane_id();
    if (a.out_hist_off && lane == 0 && c.nb + c.len < a.out_cap) a.out_hist[c.nb + c.len] = tok;
    if (!a.dmt || !sampled) return;
    uint64_t* mt = a.dmt + (int64_t)row * MT_N;
    if (idx < MT_N) {
        if (lane == 0) a.didx[row] = idx + 1;
        return;
    }
    auto wave_sync = []() {
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        __builtin_amdgcn_wave_barrier();
    };
    for (int t = lane; t < MT_N; t += WAVE) w[t] = mt[t];
    wave_sync();
    constexpr int LO = MT_N - MT_M, NLO = (LO + WAVE - 1) / WAVE;
    uint64_t nv[NLO];
#pragma unroll
    for (int c = 0; c < NLO; ++c) {
        const int t = c * WAVE + lane;
        nv[c] = t < LO ? mt_twist_one(w[t], w[t + 1], w[t + MT_M]) : 0ull;
    }
    wave_sync();
#pragma unroll
    for (int c = 0; c < NLO; ++c) {
        const int t = c * WAVE + lane;
        if (t < LO) w[t] = nv[c];
    }
    wave_sync();
    for (int t0 = LO; t0 < MT_N; t0 += WAVE) {
        const int t = t0 + lane;
        uint64_t v = 0ull;
        if (t < MT_N) v = mt_twist_one(w[t], w[(t + 1) % MT_N], w[t - LO]);
        wave_sync();
        if (t < MT_N) w[t] = v;
        wave_sync();
    }
    for (int t = lane; t < MT_N; t += WAVE) mt[t] = w[t];
    if (lane == 0) a.didx[row] = 1;
}

#ifdef FS_TRACE
#define SK_MARK(i) do { if (threadIdx.x == 0) s.trace_t[(i)] = __builtin_amdgcn_s_memrealtime(); } while (0)
#define SK_TAG(i, v) do { if (threadIdx.x == 0) s.trace_t[(i)] = (uint64_t)(v); } while (0)
#define SK_FLUSH() do { if (threadIdx.x == 0 && a.trace) \
    for (int i_ = 0; i_ < TRACE_W; ++i_) a.trace[(int64_t)blockIdx.x * TRACE_W + i_] = s.trace_t[i_]; } while (0)
#else
#define SK_MARK(i) do {} while (0)
#define SK_TAG(i, v) do {} while (0)
#define SK_FLUSH() do {} while (0)
#endif

// Ranks of the n <= SK_LT composites cand[0, n) (16-byte aligned LDS), all distinct: P threads per candidate each count the larger entries
// in 1/P of the list (LDS reads of one address per wave: broadcasts), the partial counts are summed and place(rank,
// composite) runs once per candidate. Whole workgroup; rk: LDS scratch of SK_LT words.
template <class F>
__device__ __forceinline__ void sk_rank(const uint64_t* cand, uint32_t* rk, int n, F place) {
    const int tid = threadIdx.x;
    // rk: [P][per] partial ranks
    const int P = n <= SK_LT / 4 ? 4 : (n <= SK_LT / 2 ? 2 : 1);
    const int per = SK_LT / P;
    const int c = tid % per, qq = tid / per;
    const int span = (((n + P - 1) / P) + 1) & ~1;                 // even: every part starts on a 16-byte pair
    if (c < n) {
        const uint64_t me = cand[c];
        const int j0 = qq * span, j1 = j0 + span < n ? j0 + span : n;
        uint32_t r = 0u;
        int jj = j0;
        const ulonglong2* c2 = reinterpret_cast<const ulonglong2*>(cand);
        for (; jj + 8 <= j1; jj += 8) {                            // eight entries per step: four 16-byte LDS reads
            const ulonglong2 e0 = c2[jj >> 1], e1 = c2[(jj >> 1) + 1], e2 = c2[(jj >> 1) + 2], e3 = c2[(jj >> 1) + 3];
            r += (e0.x > me ? 1u : 0u) + (e0.y > me ? 1u : 0u) + (e1.x > me ? 1u : 0u) + (e1.y > me ? 1u : 0u) +
                 (e2.x > me ? 1u : 0u) + (e2.y > me ? 1u : 0u) + (e3.x > me ? 1u : 0u) + (e3.y > me ? 1u : 0u);
        }
        for (; jj < j1; ++jj) r += cand[jj] > me ? 1u : 0u;
        rk[qq * per + c] = r;
    }
    __syncthreads();
    if (tid < n) {
        uint32_t r = 0u;
        for (int p2 = 0; p2 < P; ++p2) r += rk[p2 * per + tid];
        place(r, cand[tid]);
    }
}

// The row's end, in the merging workgroup's wave 0: its token and kept count, a decode step's append and draw, or the
// verification window's exchange. w: LDS scratch of MT_N entries.
__device__ __forceinline__ void sk_finish(const SkArgs& a, int row, int pidx, bool sampled, int tok, int keep,
                                          const SkCopy& cp, int idx, uint64_t* w) {
    const int lane = lane_id();
    if (a.mode != MODE_VERIFY) {
        if (lane == 0) {
            a.tok[row] = tok;
            if (a.keep) a.keep[row] = keep;
        }
        if (a.out_hist_off || a.dmt) sk_decode_commit(a, row, sampled, tok, cp, idx, w);
    } else {
        // the last row of a stream to finish computes its accepted prefix (server.cpp:627-637): the stream's rows
        // run on several XCDs, so the exchange is agent-scope.
        const int64_t r0 = ld_const(a.row_off + pidx);
        const int m = (int)(ld_const(a.row_off + pidx + 1) - r0);
        if (m <= 32) {
            // Streams of up to 32 rows: one 64-bit atomic per row carries everything - the count of rows done in its
            // high word, in its low word a bit for each row that ends the walk (an eos token, the last row, or a
            // token other than the next row's draft). The last row's fetched value holds every other row's bit, so
            // its accepted prefix is the lowest set bit + 1, with no token exchanged and no wait for stores.
            if (lane == 0) {
                a.tok[row] = tok;
                const int rr = row - (int)r0;
                const bool stop = (a.eos >= 0 && tok == a.eos) || rr + 1 >= m || tok != ld_const(a.rows + row + 1);
                const uint64_t mine = stop ? (1ull << rr) : 0ull;
                uint64_t* cnt = reinterpret_cast<uint64_t*>(a.stream_cnt) + pidx;
                const uint64_t old = __hip_atomic_fetch_add(cnt, (1ull << 32) | mine, __ATOMIC_RELAXED,
                                                            __HIP_MEMORY_SCOPE_AGENT);
                if ((uint32_t)(old >> 32) == (uint32_t)m - 1u) {
                    __hip_atomic_store(cnt, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    a.accepted[pidx] = __ffs((int)((uint32_t)old | (uint32_t)mine));
                }
            }
            return;
        }
        // longer streams: the token at agent scope, a row counter (after the 64-bit words), the last row walks
        uint32_t* cnt32 = a.stream_cnt + 2 * (int64_t)a.n_streams + pidx;
        uint32_t old = 0u;
        if (lane == 0) {
            st_agent(&a.tok[row], (int32_t)tok);
            vm_drain();
            old = __hip_atomic_fetch_add(cnt32, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        if (read_lane(old, 0) == (uint32_t)m - 1u) {
            if (lane == 0) st_agent(cnt32, 0u);
            const int acc = accepted_prefix(a.tok, a.rows, r0, m, a.eos);
            if (lane == 0) a.accepted[pidx] = acc;
        }
    }
}

}  // namespace fs

#endif  // FERRO_ROW_DEVICE_HPP

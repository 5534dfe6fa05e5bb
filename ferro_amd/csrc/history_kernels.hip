// history_kernels.hip - prompt-lookup drafting and the history append on device CSR histories.
#include "sampler_device.hpp"
#include "sampler_launch.hpp"

namespace fs {

constexpr int LD_BLOCK = 256;             // threads of the append kernel

// History append (the per-stream hist.push_back of each consumed token, server.cpp:342, as the decode loop at
// server.cpp:603-606 and the verify window at server.cpp:627-637 feed them), on CSR histories and out of place: stream
// s keeps its old ids and gains tok[row_off[s] + i], i < n_s, where n_s is count[s] (NULL: 1) clamped to its rows
// [0, row_off[s+1] - row_off[s]]. The new offsets are old (rebased to 0) + the exclusive prefix of the n_s.
__device__ __forceinline__ int64_t app_n(const int64_t* row_off, const int32_t* count, int s, bool* bad) {
    const int64_t r0 = row_off ? row_off[s] : (int64_t)s;
    const int64_t nr = row_off ? row_off[s + 1] - r0 : 1;
    int64_t n = count ? (int64_t)count[s] : 1;
    if (n < 0 || n > nr) {
        *bad = true;
        n = n < 0 ? 0 : nr;
    }
    return n;
}

// One workgroup: the new offsets, streams in chunks of BLOCK (carry in int64).
__global__ __launch_bounds__(BLOCK) void hist_offsets_kernel(int S, const int64_t* hist_off, const int64_t* row_off,
                                                             const int32_t* count, int64_t* out_off, int64_t out_cap,
                                                             int32_t* err) {
    __shared__ uint32_t wsum[NWAVES];
    const int tid = threadIdx.x;
    const int64_t h0 = hist_off[0];
    int64_t carry = 0;
    bool bad = false;
    for (int c0 = 0; c0 < S; c0 += BLOCK) {
        const int s = c0 + tid;
        const uint32_t n = s < S ? (uint32_t)app_n(row_off, count, s, &bad) : 0u;
        uint32_t tot;
        const uint32_t ex = block_excl_scan<uint32_t>(n, wsum, &tot);
        if (s < S) out_off[s] = hist_off[s] - h0 + carry + ex;
        carry += tot;
        __syncthreads();                                 // wsum is reused by the next chunk
    }
    if (tid == 0) {
        const int64_t end = hist_off[S] - h0 + carry;
        out_off[S] = end;
        if (end > out_cap) atomicOr(err, FS_DEVERR_HIST_APPEND);
    }
    if (bad) atomicOr(err, FS_DEVERR_HIST_APPEND);
}

// One workgroup per stream: its old ids, then its appended tokens (positions >= out_cap are not written).
__global__ __launch_bounds__(LD_BLOCK) void hist_append_kernel(const int32_t* hist, const int64_t* hist_off,
                                                               const int32_t* tok, const int64_t* row_off,
                                                               const int32_t* count, const int64_t* out_off,
                                                               int32_t* out, int64_t out_cap) {
    const int s = (int)blockIdx.x;
    bool bad = false;
    const int64_t n = app_n(row_off, count, s, &bad);
    const int64_t a = hist_off[s], L = hist_off[s + 1] - a;
    const int64_t o = out_off[s];
    const int64_t r0 = row_off ? row_off[s] : (int64_t)s;
    for (int64_t i = threadIdx.x; i < L + n; i += LD_BLOCK) {
        const int64_t d = o + i;
        if (d < out_cap) out[d] = i < L ? hist[a + i] : tok[r0 + (i - L)];
    }
}

// ------------------------------------------------------------------------------------------------ prompt lookup
// Prompt-lookup drafting (server.cpp:552-564), one workgroup per stream. The reference tries n = min(4, L-1) down to
// min_n and, for each n, takes the most recent p with h[p, p+n) == the history's last n tokens and a non-eos token
// after the match (a match whose continuation is empty is skipped); the tokens after it, up to kmax and stopping
// before eos, are the draft. Seen from the continuation e = p + n, a match of n tokens ends at e - 1 whatever n is, so
// one pass finds every n at once: m(e), how many of the tokens before e equal the history's last ones (at most
// min(4, L-1)), and the draft starts at the e that is largest by (m(e), e) among those with m(e) >= min_n.
// Bound: one read of the history (32 KB for 8192 ids), so latency. The history is taken in tiles of LU_TILE ids from
// its end (LU_PER loads in flight per thread, staged in LDS, where each thread reads four ids and the four before them
// at once); a tile that holds a match of full length ends the search, older ones cannot beat it. The draft is copied by
// one wave, eos found with a ballot. 64 streams of 8192 ids on average: 38-43 us with one pass per
// match length, an id per load and round trip and a serial copy; now 5.3 us.
constexpr int LU_BLOCK = 1024;
constexpr int LU_PER = 16;
constexpr int LU_TILE = LU_BLOCK * LU_PER;
constexpr int LU_N = 4;                   // longest match tried; ids of a block

__global__ __launch_bounds__(LU_BLOCK) void lookup_draft_kernel(const int32_t* hist, const int64_t* hist_off,
                                                                const int32_t* kmax_arr, const int32_t* min_n_arr,
                                                                int eos, int32_t* draft, int draft_ld,
                                                                int32_t* ndraft) {
    __shared__ __align__(16) int32_t ids[LU_N + LU_TILE];              // ids[i]: id c0 - LU_N + i of the history
    __shared__ uint64_t wbest[LU_BLOCK / WAVE];
    const int st = (int)blockIdx.x;
    const int tid = threadIdx.x, lane = lane_id();
    const int64_t h0 = hist_off[st];
    const int64_t L = hist_off[st + 1] - h0;
    const int32_t* h = hist + h0;
    int kmax = kmax_arr ? kmax_arr[st] : draft_ld;
    kmax = kmax < draft_ld ? kmax : draft_ld;
    const int64_t want_n = min_n_arr ? min_n_arr[st] : 2;
    const int64_t lo_n = want_n > 0 ? want_n : 0;        // (an empty match is the shortest there is)
    const int64_t nmax = L - 1 < LU_N ? L - 1 : LU_N;
    uint64_t best = 0ull;                                // (1 + m) << 56 | e
    if (nmax >= lo_n && kmax > 0) {
        int32_t t[LU_N];                                 // the history's last ids, the last one first
#pragma unroll
        for (int q = 0; q < LU_N; ++q) t[q] = q < nmax ? h[L - 1 - q] : 0;
        for (int64_t c1 = L; c1 > 0; c1 -= LU_TILE) {    // tile: continuations e in [c0, c1)
            const int64_t c0 = c1 > LU_TILE ? c1 - LU_TILE : 0;
            const int n = (int)(c1 - c0);
            int32_t v[LU_PER];
#pragma unroll
            for (int j = 0; j < LU_PER; ++j) v[j] = j * LU_BLOCK + tid < n ? h[c0 + j * LU_BLOCK + tid] : 0;
            if (tid < LU_N) ids[tid] = c0 - LU_N + tid >= 0 ? h[c0 - LU_N + tid] : 0;
#pragma unroll
            for (int j = 0; j < LU_PER; ++j) ids[LU_N + j * LU_BLOCK + tid] = v[j];
            __syncthreads();
            int bm = -1, bi = 0;                         // this thread's longest match, the most recent of those
            const int start = c0 < LU_N ? (int)c0 : LU_N;   // ids before the tile (no match reaches past the history's first)
#pragma unroll
            for (int j = 0; j < LU_PER / LU_N; ++j) {
                const int i0 = (j * LU_BLOCK + tid) * LU_N;
                if (i0 < n) {
                    const int4 p = *reinterpret_cast<const int4*>(&ids[i0]);
                    const int4 c = *reinterpret_cast<const int4*>(&ids[i0 + LU_N]);
                    const int32_t w[2 * LU_N] = {p.x, p.y, p.z, p.w, c.x, c.y, c.z, c.w};
#pragma unroll
                    for (int r = 0; r < LU_N; ++r) {
                        int m = w[r] == t[3] ? 4 : 3;
                        m = w[r + 1] == t[2] ? m : 2;
                        m = w[r + 2] == t[1] ? m : 1;
                        m = w[r + 3] == t[0] ? m : 0;
                        m = m < (int)nmax ? m : (int)nmax;
                        m = m < start + i0 + r ? m : start + i0 + r;
                        if (i0 + r < n && w[r + LU_N] != eos && m >= bm) { bm = m; bi = i0 + r; }
                    }
                }
            }
            if (bm >= lo_n) {
                const uint64_t key = ((uint64_t)(1 + bm) << 56) | (uint64_t)(c0 + bi);
                best = key > best ? key : best;
            }
            best = wave_max(best);
            if (lane == 0) wbest[tid / WAVE] = best;
            __syncthreads();
            best = wave_max(wbest[lane & (LU_BLOCK / WAVE - 1)]);
            if ((int64_t)(best >> 56) == 1 + nmax) break;
        }                                                // (every wave has read wbest before the next tile's barrier)
    }
    if (tid >= WAVE) return;
    int d = 0;
    if (best != 0ull) {
        const int64_t e = (int64_t)(best & ((1ull << 56) - 1ull));
        const int64_t most = L - e < kmax ? L - e : kmax;
        for (; d < most; d += WAVE) {
            const bool in = d + lane < most;
            const int32_t id = in ? h[e + d + lane] : eos;
            const uint64_t stop = __ballot(!in || id == eos);
            const int n = stop ? __ffsll((unsigned long long)stop) - 1 : WAVE;
            if (lane < n) draft[(int64_t)st * draft_ld + d + lane] = id;
            if (n < WAVE) { d += n; break; }
        }
    }
    if (lane == 0) ndraft[st] = d;
}

hipError_t launch_lookup_draft(int n_streams, const int32_t* hist, const int64_t* hist_off, const int32_t* kmax,
                               const int32_t* min_n, int eos, int32_t* draft, int draft_ld, int32_t* ndraft,
                               hipStream_t st) {
    hipLaunchKernelGGL(lookup_draft_kernel, dim3((unsigned)n_streams), dim3(LU_BLOCK), 0, st, hist, hist_off, kmax,
                       min_n, eos, draft, draft_ld, ndraft);
    return hipGetLastError();
}

hipError_t launch_hist_append(int S, const int32_t* hist, const int64_t* hist_off, const int32_t* tok,
                              const int64_t* row_off, const int32_t* count, int32_t* out, int64_t* out_off,
                              int64_t out_cap, int32_t* err, hipStream_t st) {
    hipLaunchKernelGGL(hist_offsets_kernel, dim3(1), dim3(BLOCK), 0, st, S, hist_off, row_off, count, out_off, out_cap,
                       err);
    if (S == 0) return hipGetLastError();
    hipLaunchKernelGGL(hist_append_kernel, dim3((unsigned)S), dim3(LD_BLOCK), 0, st, hist, hist_off, tok, row_off,
                       count, out_off, out, out_cap);
    return hipGetLastError();
}

}  // namespace fs

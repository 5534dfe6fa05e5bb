// history_kernels.hip - prompt-lookup drafting and the history append on device CSR histories.
#include "sampler_device.hpp"
#include "sampler_launch.hpp"

namespace fs {

// ------------------------------------------------------------------------------------------------ prompt lookup
// Prompt-lookup drafting (server.cpp:552-564), one workgroup per stream: for n = min(4, L-1) down to min_n, every
// thread tests its positions p for h[p, p+n) == the history's last n tokens with a non-eos token after the match
// (the reference skips a match whose continuation is empty); the largest such p (the most recent occurrence) wins,
// and the tokens after it, up to kmax and stopping before eos, are the draft.
constexpr int LD_BLOCK = 256;

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

__global__ __launch_bounds__(LD_BLOCK) void lookup_draft_kernel(const int32_t* hist, const int64_t* hist_off,
                                                                const int32_t* kmax_arr, const int32_t* min_n_arr,
                                                                int eos, int32_t* draft, int draft_ld,
                                                                int32_t* ndraft) {
    __shared__ int64_t wbest[LD_BLOCK / WAVE];
    const int st = (int)blockIdx.x;
    const int tid = threadIdx.x;
    const int64_t h0 = hist_off[st];
    const int64_t L = hist_off[st + 1] - h0;
    const int32_t* h = hist + h0;
    int kmax = kmax_arr ? kmax_arr[st] : draft_ld;
    kmax = kmax < draft_ld ? kmax : draft_ld;
    const int min_n = min_n_arr ? min_n_arr[st] : 2;
    int d = 0;
    for (int64_t n = (L - 1 < 4 ? L - 1 : 4); n >= min_n && kmax > 0; --n) {
        int32_t t[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) t[q] = q < n ? h[L - n + q] : 0;
        int64_t best = -1;
        for (int64_t p = tid; p <= L - n - 1; p += LD_BLOCK) {
            bool eq = true;
#pragma unroll
            for (int q = 0; q < 4; ++q) eq = eq && (q >= n || h[p + q] == t[q]);
            if (eq && h[p + n] != eos) best = p;               // p grows: the last hit is this thread's largest
        }
        best = wave_max(best);
        if (lane_id() == 0) wbest[tid / WAVE] = best;
        __syncthreads();
#pragma unroll
        for (int w = 0; w < LD_BLOCK / WAVE; ++w) best = wbest[w] > best ? wbest[w] : best;
        __syncthreads();
        if (best >= 0) {
            if (tid == 0)
                for (int64_t k = best + n; k < L && d < kmax; ++k) {
                    if (h[k] == eos) break;
                    draft[(int64_t)st * draft_ld + d++] = h[k];
                }
            break;
        }
    }
    if (tid == 0) ndraft[st] = d;
}
hipError_t launch_lookup_draft(int n_streams, const int32_t* hist, const int64_t* hist_off, const int32_t* kmax,
                               const int32_t* min_n, int eos, int32_t* draft, int draft_ld, int32_t* ndraft,
                               hipStream_t st) {
    hipLaunchKernelGGL(lookup_draft_kernel, dim3((unsigned)n_streams), dim3(LD_BLOCK), 0, st, hist, hist_off, kmax,
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

// sampler_launch.hpp - the launchers that the host side (sampler_kernels.hip) calls in the other kernel files.
#ifndef FERRO_SAMPLER_LAUNCH_HPP
#define FERRO_SAMPLER_LAUNCH_HPP

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/ferro_sampler.h"

namespace fs {

struct Args;
// The fused kernel's grid (segments, then merges), and its merge alone (alone != 0: each row from its logits).
hipError_t launch_segments(const Args& a, unsigned grid, hipStream_t st);
hipError_t launch_merges(const Args& a, unsigned rows, int nseg, int alone, hipStream_t st);

constexpr int SK_LT = 256;                 // threads per segment workgroup
constexpr int SK_NW = SK_LT / 64;
constexpr int SK_K = 64;                   // largest k (one candidate per lane of the finishing wave)
constexpr int SK_GCAP = 128;               // groups of four a wave can hand to the expansion
constexpr int SK_CAP = 512;                // candidates a segment ranks in LDS
constexpr int SK_MAX_SEGS = 64;            // segments per row

struct SkArgs {
    const float* logits;
    int64_t ld;
    int B, V, nseg;
    const int32_t* hist;
    const int64_t* hist_off;
    const fs_row_params* params;
    const double* u;
    int32_t* tok;
    int kcap;
    int32_t* cand_ids;
    double* cand_probs;
    int32_t* keep;
    uint64_t* lists;                       // [B * nseg][SK_K]: each segment's top k, sorted, 0-padded
    uint32_t* ticket;                      // [B]: segments finished (left at 0)
    int32_t* err;
    uint64_t* trace;                       // FS_TRACE builds: per-workgroup phase timestamps (NULL: none)
    // verification windows (mode MODE_VERIFY; the host sends only windows without an active penalty here)
    int mode;
    const int32_t* rows;                   // token fed at each row
    const int64_t* row_off;                // stream -> rows
    int n_streams, eos;
    int32_t* accepted;
    uint32_t* stream_cnt;                  // [3 n_streams]: 64-bit counts + stop bits, 32-bit counts (left at 0)
    // a decode step (fs_decode_step_hp; NULL otherwise): draw streams and the histories with the tokens appended
    uint64_t* dmt;
    int32_t* didx;
    int32_t* out_hist;
    int64_t* out_hist_off;
    int64_t out_cap;
};

// flags of a launch: some row has an active penalty window; a decode step (the histories are copied); a verification
// window (mid-k kernel)
constexpr int SK_MAY_PEN = 1, SK_COPY = 2, MK_VERIFY = 4;
// nl: float4 loads per thread (4, 8 or 16); the grid and k's layout come from the small-k plan.
hipError_t launch_small_k(int nl, bool capped, bool all_greedy, unsigned grid, int flags, const SkArgs& k,
                          hipStream_t st);

// The mid-k kernel: the small-k kernel's arguments (lists and ticket unused) and its own workspace.
constexpr int MK_LIST = 4096;              // entries of a row's candidate list
constexpr int MK_SPILL = 16384;            // entries of a row's list of penalised logits past those its segments keep in LDS
constexpr int MK_CTR = 128;                // words of a row's counters; from 64 on two per segment
// Segments per row, which wait for each other. A process has four hardware queues unless it asks for more, and each can
// hold one row whose segments are not all dispatched: 4 * 31 workgroups waiting leave room on an XCD (32 CUs of four
// workgroups), so calls of several contexts on several streams always go on. With 64 segments three calls could fill an
// XCD and wait out their limit. It is faster, too: 16 rows of 262144 logits, k 100: 18.1 us with 64 segments, 14.3 with 32.
constexpr int MK_MAX_SEGS = 32;
static_assert(64 + 2 * MK_MAX_SEGS <= MK_CTR, "");
struct MkArgs {
    SkArgs a;
    uint32_t* ctr;                         // [B][MK_CTR], left at 0
    uint32_t* qk;                          // [B][nseg][SK_NW][16] published lane maxima
    uint64_t* list;                        // [B][MK_LIST]
    uint64_t* spill;                       // [B][MK_SPILL]
    uint64_t* mass;                        // [B][2048] mass bins of rows with every token a candidate, left at 0
    uint32_t spins;                        // bounded wait for a row's segments (polls)
};
// all: some row samples with every token a candidate
hipError_t launch_mid_k(int nl, bool capped, bool all, unsigned grid, int flags, const MkArgs& m, hipStream_t st);

hipError_t launch_lookup_draft(int n_streams, const int32_t* hist, const int64_t* hist_off, const int32_t* kmax,
                               const int32_t* min_n, int eos, int32_t* draft, int draft_ld, int32_t* ndraft,
                               hipStream_t st);
hipError_t launch_hist_append(int S, const int32_t* hist, const int64_t* hist_off, const int32_t* tok,
                              const int64_t* row_off, const int32_t* count, int32_t* out, int64_t* out_off,
                              int64_t out_cap, int32_t* err, hipStream_t st);

}  // namespace fs

#endif  // FERRO_SAMPLER_LAUNCH_HPP

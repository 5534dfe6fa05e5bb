// sampler_device.hpp - what the kernels of the sampler share: the argument and row structs, order-preserving keys,
// wave and block primitives, the softcap, the one-wave softmax and the register sorts.
#ifndef FERRO_SAMPLER_DEVICE_HPP
#define FERRO_SAMPLER_DEVICE_HPP

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>
#include <cstring>
#include <mutex>
#include <new>
#include <random>
#include <vector>

#include "../../include/ferro_sampler.h"

#if !defined(__gfx950__) && defined(__HIP_DEVICE_COMPILE__)
#error "ferro sampler kernels are written for gfx950 only"
#endif

namespace fs {

constexpr int BLOCK = 512;                // threads per workgroup: 8 wave64s, two workgroups per CU
constexpr int WAVE = 64;
constexpr int NWAVES = BLOCK / WAVE;
constexpr int TPT = 8;                    // logits per thread per tile
constexpr int NV = TPT / 4;               // float4 loads per thread per tile
constexpr int TILE = BLOCK * TPT;         // 4096 logits per tile
constexpr int PF = 2;                     // tiles in flight per workgroup
constexpr int KMAX = 2048;                // largest k on the fused select path
constexpr int KPT = KMAX / BLOCK;         // candidates per thread in the softmax / draw phase
constexpr int CAP = KMAX + TILE;          // candidate buffer (LDS), per-segment list in the workspace, merge gather
constexpr int HBITS = 11;
constexpr int NBINS = 1 << HBITS;         // threshold histograms
constexpr int SMALL = 512;                // rank-sort capacity of the merge
constexpr int MAX_SEGS = 1024;            // segments per row
constexpr int SPEC = 2;                   // merge gather: loads in flight per thread per round
constexpr int FAST_SEGS = 64;             // merge fast path: a wave reads every list's bound and count
static_assert(SPEC * BLOCK + SMALL + 2 * WAVE + 4 * 2 * WAVE / 2 <= CAP, "merge fast path: list, ranks and finish buffers fit");
constexpr int RBITS = 12;                 // row histogram: bins of the top key bits, shared by a row's segments
constexpr int RBINS = 1 << RBITS;
constexpr int RSHIFT = 32 - RBITS;
constexpr int XCDS = 8;                   // MI355X: 8 XCDs, workgroups dealt round-robin by index
constexpr int WIDS = 2048;                // penalty-window ids of one segment kept in LDS (longer: rescanned per tile)

constexpr int LB = 4096;                    // coarse key bins of the large-k path
constexpr uint32_t MERGE_SPINS = 1u << 20;   // bounded wait of the merge role (far above any segment's time)

enum Mode : int { MODE_SAMPLE = 0, MODE_ARGMAX = 1, MODE_VERIFY = 2 };

struct Args {
    const float* logits;
    int64_t ld;
    int B;            // rows
    int V;
    const int32_t* hist;
    const int64_t* hist_off;
    const fs_row_params* params;   // NULL: no penalties (argmax mode only)
    const double* u;
    int32_t* tok;
    int kcap;
    int32_t* cand_ids;
    double* cand_probs;
    int32_t* keep;
    const int32_t* rows;           // verify: tokens fed per row
    const int64_t* row_off;        // verify: stream -> rows
    int n_streams;
    int eos;
    int32_t* accepted;
    int mode;
    int nseg;                      // segments per row (the default layout)
    int balance;                   // nonzero: each XCD splits its workgroups among its rows by the rows' cost
    int seg_tiles;                 // tiles per segment
    uint64_t* cand;                // [B*nseg][CAP]
    uint32_t* meta;                // [B*nseg][2]: lower bound of the k-th key, count
    uint32_t* rhist;               // [B][RBINS] row histograms of the segments' candidates, left at 0
    uint64_t* rmass;               // [B][4096] fixed-point mass histograms of large rows' candidates, left at 0
    uint32_t* stream_cnt;          // [n_streams] verify completion counters, left at 0
    int32_t* err;                  // device error bits
    int32_t* dirty;                // nonzero: a merge gave up waiting; the row histograms and counters may be stale
    uint32_t merge_spins;          // bounded wait of the merge role (polls); 0: give up without waiting
    uint64_t* trace;               // FS_TRACE builds: per-workgroup phase timestamps (NULL: none)
    // one-launch decode step (fs_decode_step): the draws come from device streams (row r = stream r) instead of u,
    // and each row's token is appended to its stream's history, out of place
    uint64_t* dmt;                 // [B][312] mt19937_64 states (NULL: draws from u)
    int32_t* didx;                 // [B] their next indices
    int32_t* out_hist;             // the histories with the tokens appended (NULL: no append)
    int64_t* out_hist_off;         // [B + 1]
    int64_t out_cap;               // ids out_hist holds
};

constexpr int MT_N = 312, MT_M = 156;
constexpr uint64_t MT_A = 0xB5026F5AA96619E9ull, MT_UPPER = 0xFFFFFFFF80000000ull, MT_LOWER = 0x7FFFFFFFull;

__device__ __forceinline__ uint64_t mt_temper(uint64_t y) {
    y ^= (y >> 29) & 0x5555555555555555ull;
    y ^= (y << 17) & 0x71D67FFFEDA60000ull;
    y ^= (y << 37) & 0xFFF7EEE000000000ull;
    y ^= y >> 43;
    return y;
}
__device__ __forceinline__ uint64_t mt_twist_one(uint64_t cur, uint64_t next, uint64_t far) {
    const uint64_t x = (cur & MT_UPPER) | (next & MT_LOWER);
    return far ^ (x >> 1) ^ ((x & 1ull) ? MT_A : 0ull);
}
__device__ void mt_twist(uint64_t* mt) {
    for (int k = 0; k < MT_N; ++k) mt[k] = mt_twist_one(mt[k], mt[(k + 1) % MT_N], mt[(k + MT_M) % MT_N]);
}
__device__ __forceinline__ double mt_canonical(uint64_t x) {
    const double r = __ull2double_rn(x) * 0x1p-64;
    return r < 1.0 ? r : 0x1.fffffffffffffp-1;
}
__device__ __forceinline__ bool samples(const fs_row_params& p) { return p.temperature > 0.0f && p.top_k != 1; }

// The draw of row `row` (sampler.cpp:45-46): u from the caller, or, in a decode step, the next value of the row's
// device stream, read without advancing it (the row's merge commits it after every reader is done).
__device__ __forceinline__ double row_u(const Args& a, int row) {
    if (a.dmt) {
        const uint64_t* mt = a.dmt + (int64_t)row * MT_N;
        const int idx = a.didx[row];
        const uint64_t y = idx < MT_N ? mt[idx] : mt_twist_one(mt[0], mt[1], mt[MT_M]);
        return mt_canonical(mt_temper(y));
    }
    return a.u ? a.u[row] : 0.0;
}

// Phase timestamps (FS_TRACE builds only; the product library compiles these to nothing): thread 0 of a workgroup
// keeps the constant 100 MHz clock (s_memrealtime) of phase i in LDS (no memory store, so no wait on the memory
// counter in the middle of the kernel) and writes them to trace[blockIdx * TRACE_W + i] at its end; slots 13-15 hold
// the role (1 segment, 2 merge), the row and the segment.
[[maybe_unused]] constexpr int TRACE_W = 16;
#ifdef FS_TRACE
#define FS_MARK(i)                                                                                        \
    do {                                                                                                  \
        if (threadIdx.x == 0) s.trace_t[(i)] = __builtin_amdgcn_s_memrealtime();                          \
    } while (0)
#define FS_TAG(i, v)                                                                                      \
    do {                                                                                                  \
        if (threadIdx.x == 0) s.trace_t[(i)] = (uint64_t)(v);                                            \
    } while (0)
// the latest of the workgroup's waves to reach phase i (lane 0 of each wave)
#define FS_MARKW(i)                                                                                       \
    do {                                                                                                  \
        if (lane_id() == 0) atomicMax((unsigned long long*)&s.trace_t[(i)],                               \
                                      (unsigned long long)__builtin_amdgcn_s_memrealtime());              \
    } while (0)
#define FS_FLUSH()                                                                                        \
    do {                                                                                                  \
        if (threadIdx.x == 0 && a.trace)                                                                  \
            for (int i_ = 0; i_ < TRACE_W; ++i_) a.trace[(int64_t)blockIdx.x * TRACE_W + i_] = s.trace_t[i_]; \
    } while (0)
#else
#define FS_MARK(i) do {} while (0)
#define FS_TAG(i, v) do {} while (0)
#define FS_MARKW(i) do {} while (0)
#define FS_FLUSH() do {} while (0)
#endif

// ------------------------------------------------------------------------------------------------ keys
// Order-preserving map fp32 -> u32: larger float -> larger key; -0 and +0 share a key (sampler.cpp:30 compares
// with == and >, under which they are equal); NaN maps below every number.
__device__ __forceinline__ uint32_t key_of(float x) {
    uint32_t u = __float_as_uint(x);
    if (x != x) return 0u;
    if (u == 0x80000000u) u = 0u;
    return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}
__device__ __forceinline__ float val_of(uint32_t k) {
    const uint32_t u = (k & 0x80000000u) ? (k & 0x7fffffffu) : ~k;
    return __uint_as_float(u);
}
// Composite: ordered like ferro's candidate order (value desc, id asc) when compared as integers, descending.
__device__ __forceinline__ uint64_t comp_of(uint32_t key, uint32_t id) {
    return ((uint64_t)key << 32) | (uint64_t)(0xFFFFFFFFu - id);
}
__device__ __forceinline__ uint32_t comp_id(uint64_t c) { return 0xFFFFFFFFu - (uint32_t)c; }
__device__ __forceinline__ uint32_t comp_key(uint64_t c) { return (uint32_t)(c >> 32); }

// ------------------------------------------------------------------------------------------------ hand-off I/O
// Agent-scope relaxed accesses compile to sc1 loads/stores: coherent across the XCDs' L2s without a write-back.
__device__ __forceinline__ void st_agent(uint64_t* p, uint64_t v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void st_agent(uint32_t* p, uint32_t v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void st_agent(int32_t* p, int32_t v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ uint64_t ld_agent(const uint64_t* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ uint32_t ld_agent(const uint32_t* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ int32_t ld_agent(const int32_t* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// Wait until this wave's vector memory operations (the sc1 stores above) have completed.
__device__ __forceinline__ void vm_drain() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }
// Invalidate the CU's L1 (vector cache): later loads are served by the XCD's L2, which holds what other workgroups
// of this XCD stored or added (stores write through the L1; atomics execute in the L2).
__device__ __forceinline__ void l1_invalidate() { asm volatile("buffer_inv sc0" ::: "memory"); }

// ------------------------------------------------------------------------------------------------ wave/block
__device__ __forceinline__ int lane_id() { return __lane_id(); }
__device__ __forceinline__ uint32_t mbcnt(uint64_t m) {
    return __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
}

// Cross-lane moves for whole waves (every call site runs with all 64 lanes active). DPP moves and lane reads stay
// in the VALU; the LDS permute path (__shfl*) costs an LDS round trip per step.
template <int CTRL, int ROWMASK = 0xF>
__device__ __forceinline__ uint32_t dpp32(uint32_t v) {        // lanes without a source read 0
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, ROWMASK, 0xF, false);
}
template <int CTRL, class T>
__device__ __forceinline__ T dpp_move(T v) {
    static_assert(sizeof(T) == 4 || sizeof(T) == 8, "32- or 64-bit lanes");
    if constexpr (sizeof(T) == 4) {
        return __builtin_bit_cast(T, dpp32<CTRL>(__builtin_bit_cast(uint32_t, v)));
    } else {
        const uint64_t u = __builtin_bit_cast(uint64_t, v);
        const uint64_t lo = dpp32<CTRL>((uint32_t)u), hi = dpp32<CTRL>((uint32_t)(u >> 32));
        return __builtin_bit_cast(T, (hi << 32) | lo);
    }
}
template <class T>
__device__ __forceinline__ T read_lane(T v, int lane) {
    if constexpr (sizeof(T) == 4) {
        return __builtin_bit_cast(T, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), lane));
    } else {
        const uint64_t u = __builtin_bit_cast(uint64_t, v);
        const uint64_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)u, lane);
        const uint64_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(u >> 32), lane);
        return __builtin_bit_cast(T, (hi << 32) | lo);
    }
}
// op over the wave, result uniform: butterflies within each row of 16 lanes (quad swaps, half-row and row
// mirrors), then the four rows' lane 0
template <class T, class Op>
__device__ __forceinline__ T wave_allreduce(T v, Op op) {
    v = op(v, dpp_move<0xB1>(v));     // quad_perm [1,0,3,2]
    v = op(v, dpp_move<0x4E>(v));     // quad_perm [2,3,0,1]
    v = op(v, dpp_move<0x141>(v));    // row_half_mirror
    v = op(v, dpp_move<0x140>(v));    // row_mirror
    return op(op(read_lane(v, 0), read_lane(v, 16)), op(read_lane(v, 32), read_lane(v, 48)));
}
template <class T>
__device__ __forceinline__ T wave_max(T v) {
    return wave_allreduce(v, [](T x, T y) { return y > x ? y : x; });
}
template <class T>
__device__ __forceinline__ T wave_min(T v) {
    return wave_allreduce(v, [](T x, T y) { return y < x ? y : x; });
}
// The verification rule (server.cpp:627-637) over a stream's m >= 1 tokens, read by the whole wave at once (agent
// scope: the stream's rows ran on several XCDs): 1 + the leading rows whose token equals the next row's draft, the
// walk ending after an eos token. Uniform over the wave.
__device__ __forceinline__ int accepted_prefix(const int32_t* tok, const int32_t* rows, int64_t r0, int m, int eos) {
    for (int c0 = 0; c0 < m; c0 += WAVE) {
        const int r = c0 + lane_id();
        bool stop = false;
        if (r < m) {
            const int t = ld_agent(&tok[r0 + r]);
            stop = (eos >= 0 && t == eos) || r + 1 >= m || t != rows[r0 + r + 1];
        }
        const uint64_t b = __ballot(stop);
        if (b) return c0 + __ffsll((unsigned long long)b);    // 1-based: the row that ends the walk, plus one
    }
    return m;
}
// inclusive sum over lanes 0..lane (32-bit integers): row shifts 1, 2, 4, 8, then row broadcasts 15 and 31
__device__ __forceinline__ uint32_t wave_incl_scan_u32(uint32_t x) {
    x += dpp32<0x111>(x);
    x += dpp32<0x112>(x);
    x += dpp32<0x114>(x);
    x += dpp32<0x118>(x);
    x += dpp32<0x142, 0xA>(x);
    x += dpp32<0x143, 0xC>(x);
    return x;
}
__device__ __forceinline__ double wave_sum_f64(double v) {
#pragma unroll
    for (int o = WAVE / 2; o > 0; o >>= 1) v += __shfl_xor(v, o);
    return v;
}

// Small shared scratch for block-wide reductions and broadcasts.
struct Red {
    uint64_t u64[NWAVES];
    uint64_t u64b[NWAVES];
    double f64[NWAVES];
    int i32[NWAVES];
    uint32_t u32[NWAVES];
    uint32_t misc[8];
    double dmisc[4];
};

__device__ __forceinline__ uint64_t block_max_u64(uint64_t v, Red& r) {
    v = wave_max(v);
    if (lane_id() == 0) r.u64[threadIdx.x / WAVE] = v;
    __syncthreads();
    uint64_t m = r.u64[0];
#pragma unroll
    for (int w = 1; w < NWAVES; ++w) m = r.u64[w] > m ? r.u64[w] : m;
    __syncthreads();
    return m;
}
__device__ __forceinline__ uint64_t block_min_u64(uint64_t v, Red& r) {
    v = wave_min(v);
    if (lane_id() == 0) r.u64[threadIdx.x / WAVE] = v;
    __syncthreads();
    uint64_t m = r.u64[0];
#pragma unroll
    for (int w = 1; w < NWAVES; ++w) m = r.u64[w] < m ? r.u64[w] : m;
    __syncthreads();
    return m;
}
__device__ __forceinline__ uint32_t block_max_u32(uint32_t v, Red& r) {
    v = wave_max(v);
    if (lane_id() == 0) r.u32[threadIdx.x / WAVE] = v;
    __syncthreads();
    uint32_t m = r.u32[0];
#pragma unroll
    for (int w = 1; w < NWAVES; ++w) m = r.u32[w] > m ? r.u32[w] : m;
    __syncthreads();
    return m;
}
// max and min in one round
__device__ __forceinline__ void block_minmax_u32(uint32_t& mn, uint32_t& mx, Red& r) {
    uint32_t a = wave_max(mx), b = wave_min(mn);
    if (lane_id() == 0) { r.u32[threadIdx.x / WAVE] = a; r.i32[threadIdx.x / WAVE] = (int)b; }
    __syncthreads();
    a = r.u32[0];
    b = (uint32_t)r.i32[0];
#pragma unroll
    for (int w = 1; w < NWAVES; ++w) {
        a = r.u32[w] > a ? r.u32[w] : a;
        b = (uint32_t)r.i32[w] < b ? (uint32_t)r.i32[w] : b;
    }
    __syncthreads();
    mx = a;
    mn = b;
}
__device__ __forceinline__ int block_min_i32(int v, Red& r) {
    v = wave_min(v);
    if (lane_id() == 0) r.i32[threadIdx.x / WAVE] = v;
    __syncthreads();
    int m = r.i32[0];
#pragma unroll
    for (int w = 1; w < NWAVES; ++w) m = r.i32[w] < m ? r.i32[w] : m;
    __syncthreads();
    return m;
}
__device__ __forceinline__ int block_max_i32(int v, Red& r) {
    v = wave_max(v);
    if (lane_id() == 0) r.i32[threadIdx.x / WAVE] = v;
    __syncthreads();
    int m = r.i32[0];
#pragma unroll
    for (int w = 1; w < NWAVES; ++w) m = r.i32[w] > m ? r.i32[w] : m;
    __syncthreads();
    return m;
}
// Deterministic double sum: fixed butterfly in each wave, waves added in order.
__device__ __forceinline__ double block_sum_f64(double v, Red& r) {
    v = wave_sum_f64(v);
    if (lane_id() == 0) r.f64[threadIdx.x / WAVE] = v;
    __syncthreads();
    double s = r.f64[0];
#pragma unroll
    for (int w = 1; w < NWAVES; ++w) s += r.f64[w];
    __syncthreads();
    return s;
}
// DPP moves of a double (two 32-bit halves); lanes without a source read 0 (bound_ctrl off, old = 0).
template <int CTRL, int ROWMASK>
__device__ __forceinline__ double dpp_f64(double v) {
    const uint64_t u = (uint64_t)__double_as_longlong(v);
    const int lo = __builtin_amdgcn_update_dpp(0, (int)(uint32_t)u, CTRL, ROWMASK, 0xF, false);
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(uint32_t)(u >> 32), CTRL, ROWMASK, 0xF, false);
    return __longlong_as_double((long long)(((uint64_t)(uint32_t)hi << 32) | (uint64_t)(uint32_t)lo));
}
// Inclusive wave scan: row_shr 1, 2, 4, 8 inside each 16-lane row, then row_bcast 15 / 31 across rows.
__device__ __forceinline__ double wave_scan_f64(double v) {
    v += dpp_f64<0x111, 0xF>(v);
    v += dpp_f64<0x112, 0xF>(v);
    v += dpp_f64<0x114, 0xF>(v);
    v += dpp_f64<0x118, 0xF>(v);
    v += dpp_f64<0x142, 0xA>(v);
    v += dpp_f64<0x143, 0xC>(v);
    return v;
}
// Exclusive prefix over threads (thread order), deterministic; *total = the sum over the block.
template <class T>
__device__ __forceinline__ T block_excl_scan(T v, T* wsum /*NWAVES*/, T* total) {
    const int lane = lane_id(), w = threadIdx.x / WAVE;
    T x, ex;
    if constexpr (sizeof(T) == 4 && T(-1) > T(0)) {            // 32-bit unsigned: DPP scan (exact in any order)
        x = wave_incl_scan_u32(v);
        ex = x - v;
    } else if constexpr (sizeof(T) == 8 && T(0.5) > T(0)) {    // double: DPP scan, then wave_shr:1 (lane 0 reads 0)
        x = wave_scan_f64(v);
        ex = dpp_f64<0x138, 0xF>(x);
    } else {                                                   // the fixed shuffle order of the sums
        x = v;
#pragma unroll
        for (int o = 1; o < WAVE; o <<= 1) {
            const T y = __shfl_up(x, o);
            if (lane >= o) x += y;
        }
        ex = __shfl_up(x, 1);
        if (lane == 0) ex = T(0);
    }
    if (lane == WAVE - 1) wsum[w] = x;
    __syncthreads();
    T off = T(0), tot = T(0);
#pragma unroll
    for (int q = 0; q < NWAVES; ++q) {
        if (q < w) off += wsum[q];
        tot += wsum[q];
    }
    __syncthreads();
    *total = tot;
    return off + ex;
}

// Append `pred` lanes' values to an LDS list (one LDS atomic per wave); entries past cap are counted, not stored.
__device__ __forceinline__ void wave_append(bool pred, uint64_t v, uint64_t* list, uint32_t* count, uint32_t cap) {
    const uint64_t m = __ballot(pred);
    if (m == 0) return;
    uint32_t base = 0;
    const int leader = __ffsll((unsigned long long)m) - 1;
    if (lane_id() == leader) base = atomicAdd(count, (uint32_t)__popcll(m));
    base = (uint32_t)__builtin_amdgcn_readlane((int)base, leader);   // a scalar read, no LDS round trip
    if (pred) {
        const uint32_t pos = base + mbcnt(m);
        if (pos < cap) list[pos] = v;
    }
}

// wave_append for a register element: the 64-bit composite is formed only when some lane of the wave appends.
__device__ __forceinline__ void wave_append_kv(bool pred, uint32_t key, uint32_t id, uint64_t* list, uint32_t* count,
                                               uint32_t cap) {
    const uint64_t m = __ballot(pred);
    if (m == 0) return;
    uint32_t base = 0;
    const int leader = __ffsll((unsigned long long)m) - 1;
    if (lane_id() == leader) base = atomicAdd(count, (uint32_t)__popcll(m));
    base = (uint32_t)__builtin_amdgcn_readlane((int)base, leader);   // a scalar read, no LDS round trip
    if (pred) {
        const uint32_t pos = base + mbcnt(m);
        if (pos < cap) list[pos] = comp_of(key, id);
    }
}

// Histogram helpers over keys in [base, base + (NBINS << shift)): bin = (key - base) >> shift.
__device__ __forceinline__ int range_shift(uint32_t lo, uint32_t hi) {
    const uint32_t span = hi - lo;                       // keys lo..hi map to bins 0..span>>shift < NBINS
    int s = 0;
    while ((span >> s) >= (uint32_t)NBINS) ++s;
    return s;
}
// From a filled histogram, the bin b holding the kk-th largest entry: count(bins > b) < kk <= count(bins >= b).
// *above = count(bins > b), *atb = count(bins >= b). Requires 1 <= kk <= total.
__device__ __forceinline__ int hist_locate(const uint32_t* bins, int kk, uint32_t* above_out, uint32_t* atb_out, uint32_t* wsum,
                           Red& r) {
    constexpr int BPT = NBINS / BLOCK;
    const int tid = threadIdx.x;
    uint32_t mine = 0;
#pragma unroll
    for (int i = 0; i < BPT; ++i) mine += bins[NBINS - 1 - (tid * BPT + i)];
    uint32_t tot;
    const uint32_t above = block_excl_scan<uint32_t>(mine, wsum, &tot);
    if (above < (uint32_t)kk && above + mine >= (uint32_t)kk) {
        uint32_t c = above;
        for (int i = 0; i < BPT; ++i) {
            const int bin = NBINS - 1 - (tid * BPT + i);
            const uint32_t nb = bins[bin];
            if (c + nb >= (uint32_t)kk) { r.misc[4] = (uint32_t)bin; r.misc[5] = c; r.misc[6] = c + nb; break; }
            c += nb;
        }
    }
    __syncthreads();
    const int b = (int)r.misc[4];
    *above_out = r.misc[5];
    *atb_out = r.misc[6];
    __syncthreads();
    return b;
}

// From a filled histogram: the largest bin b such that count(bins >= b) >= k. Returns T = base + (b << shift) and
// *cnt = count(bins >= b); T = 0 and *cnt = total when the histogram holds fewer than k entries.
__device__ __forceinline__ uint32_t hist_threshold(const uint32_t* bins, uint32_t base, int shift, int k, uint32_t* cnt,
                                   uint32_t* wsum, Red& r) {
    constexpr int BPT = NBINS / BLOCK;
    const int tid = threadIdx.x;
    uint32_t mine = 0;
#pragma unroll
    for (int i = 0; i < BPT; ++i) mine += bins[NBINS - 1 - (tid * BPT + i)];
    uint32_t tot;
    const uint32_t above = block_excl_scan<uint32_t>(mine, wsum, &tot);
    if (tid == 0) { r.misc[4] = 0u; r.misc[5] = tot; }
    __syncthreads();
    if (tot >= (uint32_t)k && above < (uint32_t)k && above + mine >= (uint32_t)k) {
        uint32_t c = above;
        for (int i = 0; i < BPT; ++i) {
            const int bin = NBINS - 1 - (tid * BPT + i);
            c += bins[bin];
            if (c >= (uint32_t)k) { r.misc[4] = base + ((uint32_t)bin << shift); r.misc[5] = c; break; }
        }
    }
    __syncthreads();
    *cnt = r.misc[5];
    const uint32_t T = r.misc[4];
    __syncthreads();
    return T;
}

// Exact k-th largest composite among the candidates a visitor yields (all distinct, 0 = absent; 1 <= k <= count).
// Radix select from the top byte: 8 passes of a 256-bin LDS histogram. each(f) calls f(c) for every candidate the
// calling thread holds. With last_shift = 32 it stops after the key bytes: the result is the k-th largest key (low
// word 0), which at least k candidates reach.
template <class Each>
__device__ __forceinline__ uint64_t radix_kth(Each each, int k, uint32_t* hist256, uint32_t* wsum, Red& r,
                                              int last_shift = 0) {
    uint64_t prefix = 0, mask = 0;
    int kk = k;
    const int tid = threadIdx.x;
    for (int shift = 56; shift >= last_shift; shift -= 8) {
        if (tid < 256) hist256[tid] = 0;
        __syncthreads();
        each([&](uint64_t c) {
            if (c != 0 && (c & mask) == prefix) atomicAdd(&hist256[(c >> shift) & 255], 1u);
        });
        __syncthreads();
        const uint32_t cnt = tid < 256 ? hist256[255 - tid] : 0u;   // thread t owns bin 255 - t: scan from the top
        uint32_t tot;
        const uint32_t above = block_excl_scan<uint32_t>(cnt, wsum, &tot);
        if (tid < 256 && above < (uint32_t)kk && above + cnt >= (uint32_t)kk) {
            r.misc[0] = 255 - tid;
            r.misc[1] = above;
        }
        __syncthreads();
        const uint64_t d = r.misc[0];
        kk -= (int)r.misc[1];
        prefix |= d << shift;
        mask |= (uint64_t)255 << shift;
        __syncthreads();
    }
    return prefix;
}

// Descending bitonic sort of n (a power of two, n <= 4 * BLOCK) composites in LDS, whole block. The stages of the
// network are taken two at a time: for a pair of strides 2^p1, 2^p2 thread t loads the four entries whose indices
// are t with zero bits inserted at p1 and p2, plus 0/1 in those bits, applies both stages in registers and stores
// them back. While both bits are below 8 the four entries lie in the 256-entry block of the thread's wave
// (index bits 8.. = wave id), and a wave's LDS accesses complete in order, so such rounds need no barrier; a
// barrier is placed only on each side of a round that crosses blocks.
__device__ __forceinline__ void bitonic_desc(uint64_t* a, int n) {
    static_assert(4 * BLOCK >= KMAX && 4 * WAVE == 256, "four entries per thread; a wave spans 256 entries");
    const int tid = threadIdx.x;
    if (n < 4) {
        if (n == 2 && tid == 0) {
            const uint64_t x = a[0], y = a[1];
            if (x < y) { a[0] = y; a[1] = x; }
        }
        __syncthreads();
        return;
    }
    int lg = 0;
    while ((1 << lg) < n) ++lg;
    const bool act = tid < (n >> 2);
    int m = 1, p = 0;                               // next stage: merge size 2^m, stride 2^p
    bool prev_cross = false;
    while (m <= lg) {
        // this round: the stage (m, p), the next one, and a third while its stride is one of the two
        int sm[3], sp[3], ns = 0;
        int b0 = p, b1 = -1;
        while (m <= lg && ns < 3) {
            if (p != b0 && p != b1) {
                if (b1 >= 0) break;
                b1 = p;
            }
            sm[ns] = m; sp[ns] = p; ++ns;
            if (p == 0) { ++m; p = m - 1; } else { --p; }
        }
        if (b1 < 0) b1 = b0 == 0 ? 1 : 0;           // a lone last stage: any second bit
        const int hi = b0 > b1 ? b0 : b1, lo = b0 > b1 ? b1 : b0;
        const bool cross = hi >= 8;
        if (cross || prev_cross) __syncthreads();
        prev_cross = cross;
        if (act) {
            const int t = tid;
            const int base = (t & ((1 << lo) - 1)) | (((t >> lo) & ((1 << (hi - lo - 1)) - 1)) << (lo + 1)) |
                             ((t >> (hi - 1)) << (hi + 1));
            const int ix[4] = {base, base + (1 << lo), base + (1 << hi), base + (1 << hi) + (1 << lo)};
            uint64_t e[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) e[j] = a[ix[j]];
            auto cx = [](uint64_t& x, uint64_t& y, bool desc) {
                const uint64_t lo_v = x < y ? x : y, hi_v = x < y ? y : x;
                x = desc ? hi_v : lo_v;
                y = desc ? lo_v : hi_v;
            };
#pragma unroll
            for (int q = 0; q < 3; ++q) {
                if (q >= ns) break;
                const int sh = sm[q];
                if (sp[q] == hi) {                      // partners two registers apart
                    cx(e[0], e[2], ((ix[0] >> sh) & 1) == 0);
                    cx(e[1], e[3], ((ix[1] >> sh) & 1) == 0);
                } else {
                    cx(e[0], e[1], ((ix[0] >> sh) & 1) == 0);
                    cx(e[2], e[3], ((ix[2] >> sh) & 1) == 0);
                }
            }
#pragma unroll
            for (int j = 0; j < 4; ++j) a[ix[j]] = e[j];
        }
    }
    __syncthreads();
}

// Rank sort of n <= SMALL distinct composites: out[rank] = in[i] for ranks < k.
__device__ __forceinline__ void rank_sort(const uint64_t* in, int n, uint64_t* out, int k) {
    for (int i = threadIdx.x; i < n; i += BLOCK) {
        const uint64_t c = in[i];
        int rank = 0;
        for (int m = 0; m < n; ++m) rank += in[m] > c ? 1 : 0;
        if (rank < k) out[rank] = c;
    }
    __syncthreads();
}

__device__ __forceinline__ int64_t window_begin(int64_t len, const fs_row_params& p) {
    int64_t b = (p.repeat_last_n > 0 && (int64_t)p.repeat_last_n < len) ? len - (int64_t)p.repeat_last_n : 0;
    if (p.penalty_from > 0 && (int64_t)p.penalty_from > b) b = p.penalty_from;
    return b;
}

// Per-row view of the arguments: params, greedy/k, and the two history segments (a verify row sees its stream's
// base history followed by the drafts fed before it).
struct RowCtx {
    int row, pidx;
    fs_row_params p;
    bool greedy, large, pen, rep_on, fp_on, capped;
    int k;
    int64_t hA0, lenA, lenB, b, len;     // window [b, len) over the concatenated history
    const int32_t* segB;
    // the row's segments: nseg of st tiles each (the last may be shorter); segment s publishes in list slot
    // lx + XCDS * (lbase + s) (the index of the segment workgroup that streams it)
    int nseg, st, lbase, lx;
};
__device__ __forceinline__ int64_t slot_of(const RowCtx& rc, int seg) {
    return (int64_t)rc.lx + (int64_t)XCDS * (int64_t)(rc.lbase + seg);
}

// Inputs that no kernel writes (params, history offsets, verify row offsets) are read through the constant address
// space, so uniform indices become scalar loads (lgkmcnt) and never wait behind the vector loads in flight.
template <class T>
__device__ __forceinline__ T ld_const(const T* p) {
#if defined(__HIP_DEVICE_COMPILE__)
    return *(const __attribute__((address_space(4))) T*)(p);
#else
    return *p;                                  // the host pass never runs device code
#endif
}

__device__ __forceinline__ RowCtx row_ctx(const Args& a, int row) {
    RowCtx rc;
    rc.row = row;
    rc.pidx = row;
    rc.nseg = a.nseg;
    rc.st = a.seg_tiles;
    rc.lx = row % XCDS;
    rc.lbase = (row / XCDS) * a.nseg;
    rc.hA0 = 0; rc.lenA = 0; rc.lenB = 0;
    rc.segB = nullptr;
    if (a.mode == MODE_VERIFY) {
        int s0 = 0, s1 = a.n_streams;           // largest s with row_off[s] <= row
        while (s1 - s0 > 1) {
            const int m = (s0 + s1) >> 1;
            if (ld_const(a.row_off + m) <= row) s0 = m; else s1 = m;
        }
        rc.pidx = s0;
        const int64_t r0 = ld_const(a.row_off + s0);
        rc.segB = a.rows + r0 + 1;
        rc.lenB = row - r0;
    }
    if (a.hist_off && a.hist) {
        rc.hA0 = ld_const(a.hist_off + rc.pidx);
        rc.lenA = ld_const(a.hist_off + rc.pidx + 1) - rc.hA0;
    }
    if (a.params) {                           // dword by dword: scalar loads (a struct copy becomes vector loads)
        static_assert(sizeof(fs_row_params) % 4 == 0, "fs_row_params is a sequence of dwords");
        uint32_t w[sizeof(fs_row_params) / 4];
        const uint32_t* src = reinterpret_cast<const uint32_t*>(a.params + rc.pidx);
#pragma unroll
        for (int i = 0; i < (int)(sizeof(fs_row_params) / 4); ++i) w[i] = ld_const(src + i);
        __builtin_memcpy(&rc.p, w, sizeof(fs_row_params));
    } else {
        rc.p.temperature = 0.f; rc.p.top_k = 1; rc.p.top_p = 1.f; rc.p.min_p = 0.f; rc.p.repetition_penalty = 1.f;
        rc.p.frequency_penalty = 0.f; rc.p.presence_penalty = 0.f; rc.p.repeat_last_n = 0; rc.p.penalty_from = 0;
        rc.p.softcap = 0.f;
    }
    const int V = a.V;
    rc.greedy = a.mode == MODE_ARGMAX || rc.p.temperature <= 0.0f || rc.p.top_k == 1;
    rc.k = rc.greedy ? 1 : ((rc.p.top_k > 0 && rc.p.top_k < V) ? rc.p.top_k : V);
    rc.large = rc.k > KMAX;                 // not on the segment path: sampled by large_row in the merge kernel
    rc.capped = rc.p.softcap > 0.0f;
    rc.rep_on = rc.p.repetition_penalty != 1.0f;
    rc.fp_on = rc.p.frequency_penalty != 0.0f || rc.p.presence_penalty != 0.0f;
    rc.len = rc.lenA + rc.lenB;
    rc.pen = (rc.rep_on || rc.fp_on) && rc.p.repeat_last_n != 0 && rc.len > 0;
    rc.b = rc.pen ? window_begin(rc.len, rc.p) : rc.len;
    if (rc.b >= rc.len) rc.pen = false;
    return rc;
}

__device__ __forceinline__ int hist_at(const Args& a, const RowCtx& rc, int64_t i) {
    return i < rc.lenA ? a.hist[rc.hA0 + i] : rc.segB[i - rc.lenA];
}

typedef float f32x4 __attribute__((ext_vector_type(4)));
__device__ f32x4 raw_buffer_load_f32x4(__amdgpu_buffer_rsrc_t rs, int voffset, int soffset, int aux)
    __asm("llvm.amdgcn.raw.ptr.buffer.load.v4f32");
// tanhf as the host C library computes it where ferro runs (glibc's float tanh, which follows Sun's fdlibm
// s_tanh.c / s_expm1.c in single precision): tanh(x) = -e/(e+2) with e = expm1(-2|x|) for |x| < 1,
// 1 - 2/(expm1(2|x|)+2) for 1 <= |x| < 22, +-1 beyond; expm1 reduces x = k ln2 + r (ln2 split into a 24-bit-exact
// hi part and a lo part), approximates expm1(r) by fdlibm's rational scheme (the degree-5 polynomial in r^2/2 with
// fdlibm's Q1..Q5 rounded to float) and rescales by 2^k. Every operation is a separately rounded IEEE fp32 add,
// multiply or divide (no contraction), so the result is bit-identical to the host's: the GPU test checks all 2^32
// inputs against the C library.
__device__ __forceinline__ float f_of(uint32_t u) { return __uint_as_float(u); }
// Straight-line form (every case computed, the result selected): no branches, so the eight-wide unrolled reads
// that call it stay one basic block each. Selecting between separately computed IEEE results changes none of them.
__device__ __forceinline__ float host_tanhf(float x) {
    const float ln2_hi = f_of(0x3f317180u), ln2_lo = f_of(0x3717f7d1u), invln2 = f_of(0x3fb8aa3bu);
    const float Q1 = f_of(0xbd088889u), Q2 = f_of(0x3ad00d01u), Q3 = f_of(0xb8a670cdu), Q4 = f_of(0x36867e54u),
                Q5 = f_of(0xb457edbbu);
    const uint32_t jx = __float_as_uint(x), ix = jx & 0x7fffffffu;
    const bool neg = (jx >> 31) != 0u;
    const float ax = __uint_as_float(ix);
    const bool big = ix >= 0x3f800000u;                     // |x| >= 1: tanh = 1 - 2/(expm1(2|x|)+2)
    const float y = big ? __fmul_rn(2.0f, ax) : __fmul_rn(-2.0f, ax);   // expm1's argument, in (-2, 44) for |x| < 22
    const uint32_t hy = __float_as_uint(y) & 0x7fffffffu;
    const bool yneg = !big;
    // expm1(y): y = k ln2 + r (|y| > ln2 / 2; k = +-1 below 1.5 ln2)
    const bool red = hy > 0x3eb17218u;
    const bool near = hy < 0x3F851592u;
    const float hiA = yneg ? __fadd_rn(y, ln2_hi) : __fsub_rn(y, ln2_hi);
    const float loA = yneg ? -ln2_lo : ln2_lo;
    const int kB = (int)__fadd_rn(__fmul_rn(invln2, y), yneg ? -0.5f : 0.5f);   // truncation toward zero
    const float tB = (float)kB;
    const float hiB = __fsub_rn(y, __fmul_rn(tB, ln2_hi));   // tB * ln2_hi is exact
    const float loB = __fmul_rn(tB, ln2_lo);
    const int k = red ? (near ? (yneg ? -1 : 1) : kB) : 0;
    const float hi = near ? hiA : hiB, lo = near ? loA : loB;
    const float xr = red ? __fsub_rn(hi, lo) : y;
    const float c = red ? __fsub_rn(__fsub_rn(hi, xr), lo) : 0.0f;
    const float hfx = __fmul_rn(0.5f, xr);
    const float hxs = __fmul_rn(xr, hfx);
    const float r1 = __fadd_rn(1.0f, __fmul_rn(hxs, __fadd_rn(Q1, __fmul_rn(hxs, __fadd_rn(Q2, __fmul_rn(hxs,
                     __fadd_rn(Q3, __fmul_rn(hxs, __fadd_rn(Q4, __fmul_rn(hxs, Q5))))))))));
    const float t = __fsub_rn(3.0f, __fmul_rn(r1, hfx));
    const float e = __fmul_rn(hxs, __fdiv_rn(__fsub_rn(r1, t), __fsub_rn(6.0f, __fmul_rn(xr, t))));
    const float R0 = __fsub_rn(xr, __fsub_rn(__fmul_rn(xr, e), hxs));                       // k = 0
    const float e2 = __fsub_rn(__fsub_rn(__fmul_rn(xr, __fsub_rn(e, c)), c), hxs);
    const float Rm1 = __fsub_rn(__fmul_rn(0.5f, __fsub_rn(xr, e2)), 0.5f);                 // k = -1
    const float R1 = xr < -0.25f ? __fmul_rn(-2.0f, __fsub_rn(e2, __fadd_rn(xr, 0.5f)))    // k = 1
                                 : __fadd_rn(1.0f, __fmul_rn(2.0f, __fsub_rn(xr, e2)));
    const int kc = k < -126 ? -126 : (k > 127 ? 127 : k);
    const float twopk = f_of(0x3f800000u + ((uint32_t)kc << 23));
    const float RL = __fsub_rn(__fmul_rn(__fsub_rn(1.0f, __fsub_rn(e2, xr)), twopk), 1.0f);  // k <= -2 or k > 56
    const int ks = k < 0 ? 0 : (k > 31 ? 31 : k);
    const float RS = __fmul_rn(__fsub_rn(f_of(0x3f800000u - (0x1000000u >> ks)), __fsub_rn(e2, xr)), twopk);   // 1 - 2^-k
    const int kt = k < 0 ? 0 : (k > 126 ? 126 : k);
    const float RB = __fmul_rn(__fadd_rn(__fsub_rn(xr, __fadd_rn(e2, f_of((uint32_t)(0x7f - kt) << 23))), 1.0f), twopk);
    float em = k == 0 ? R0 : k == -1 ? Rm1 : k == 1 ? R1 : (k <= -2 || k > 56) ? RL : k < 23 ? RS : RB;
    const float huge = 1.0e+30f;
    if (hy < 0x33000000u) em = __fsub_rn(y, __fsub_rn(__fadd_rn(huge, y), __fadd_rn(huge, y)));   // |y| < 2^-25
    // tanh from expm1
    float z = big ? __fsub_rn(1.0f, __fdiv_rn(2.0f, __fadd_rn(em, 2.0f))) : __fdiv_rn(-em, __fadd_rn(em, 2.0f));
    if (ix >= 0x41b00000u) z = __fsub_rn(1.0f, 1.0e-30f);      // |x| >= 22: +-1 (inexact)
    float r = neg ? -z : z;
    if (ix < 0x24000000u) r = __fmul_rn(x, __fadd_rn(1.0f, x));  // |x| < 2^-55
    if (ix >= 0x7f800000u)                                       // +-inf, NaN
        r = neg ? __fsub_rn(__fdiv_rn(1.0f, x), 1.0f) : __fadd_rn(__fdiv_rn(1.0f, x), 1.0f);
    return r;
}
// The model's final-logit softcap, moved into the read: l = cap * tanhf(l / cap) (model_gemma4_gpu.cpp:282-283:
// fp32 divide, the host C library's tanhf, fp32 multiply), before the penalties as in ferro, where the model caps
// the row first. Bit-identical to the host loop.
__device__ __forceinline__ float softcap_one(float l, float cap) { return __fmul_rn(cap, host_tanhf(__fdiv_rn(l, cap))); }
// Unrolled, for the streaming loop of the segment path (its three call sites): a rolled loop there changes the
// allocation of the tile registers and slows every row, capped or not.
template <int N>
__device__ __forceinline__ void softcap_vals_unrolled(float (&x)[N], float cap) {
#pragma unroll
    for (int i = 0; i < N; ++i) x[i] = softcap_one(x[i], cap);
}
// A rolled loop: one copy of the cap per call site (there are dozens, all unrolled eight-wide otherwise), for capped
// rows only; the element is picked and put back by index.
template <int N>
__device__ __forceinline__ void softcap_vals(float (&x)[N], float cap) {
#pragma unroll 1
    for (int i = 0; i < N; ++i) {
        float v = x[0];
#pragma unroll
        for (int j = 1; j < N; ++j) v = i == j ? x[j] : v;
        v = softcap_one(v, cap);
#pragma unroll
        for (int j = 0; j < N; ++j) x[j] = i == j ? v : x[j];
    }
}
__device__ __forceinline__ double lane_f64(double v, int lane) {   // lane: wave-uniform
    const uint64_t u = (uint64_t)__double_as_longlong(v);
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)u, lane);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(u >> 32), lane);
    return __longlong_as_double((long long)(((uint64_t)hi << 32) | lo));
}

// Softmax at temperature, min-p, top-p and the draw (sampler.cpp:37-49) over k <= WAVE candidates held by one wave:
// lane i holds candidate i in ferro's order (0 past k). Sums are DPP wave scans in candidate order. Writes the
// optional candidate outputs; returns the token and the kept count.
__device__ __forceinline__ void wave_softmax(const Args& a, const RowCtx& rc, uint64_t v, int k, double u, int& tok_out,
                                             int& keep_out) {
    const int lane = lane_id();
    const int row = rc.row;
    const fs_row_params& p = rc.p;
    const float mx = val_of(comp_key(read_lane(v, 0)));
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
    tok_out = (int)comp_id(read_lane(v, at));
    keep_out = keep;
    if (a.mode != MODE_VERIFY) {
        const int m = k < a.kcap ? k : a.kcap;
        if (lane < m) {
            if (a.cand_ids) a.cand_ids[(int64_t)row * a.kcap + lane] = (int32_t)comp_id(v);
            if (a.cand_probs) a.cand_probs[(int64_t)row * a.kcap + lane] = pr;
        }
    }
}

// lane ^ D over the wave, in the VALU: DPP for D < 16 (both shifts in full exec, then an arithmetic select: a branch
// would run each DPP move on half the lanes), permlane swaps for 16 and 32 (gfx950)
template <int D>
__device__ __forceinline__ uint32_t xor_lane32(uint32_t v) {
    if constexpr (D == 1) {
        return dpp32<0xB1>(v);                                  // quad_perm [1,0,3,2]
    } else if constexpr (D == 2) {
        return dpp32<0x4E>(v);                                  // quad_perm [2,3,0,1]
    } else if constexpr (D == 4 || D == 8) {
        const uint32_t up = dpp32<0x100 + D>(v), dn = dpp32<0x110 + D>(v);   // row_shl: lane + D; row_shr: lane - D
        const uint32_t m = 0u - (((uint32_t)lane_id() / D) & 1u);
        return up ^ ((up ^ dn) & m);
    } else if constexpr (D == 16) {
        const auto r = __builtin_amdgcn_permlane16_swap(v, v, false, false);
        return (lane_id() & 16) ? r[0] : r[1];
    } else {
        static_assert(D == 32, "xor distances 1..32");
        const auto r = __builtin_amdgcn_permlane32_swap(v, v, false, false);
        return (lane_id() & 32) ? r[0] : r[1];
    }
}
template <int D>
__device__ __forceinline__ uint64_t xor_lane64(uint64_t v) {
    return ((uint64_t)xor_lane32<D>((uint32_t)(v >> 32)) << 32) | (uint64_t)xor_lane32<D>((uint32_t)v);
}
// Bitonic compare-exchange at distance D: the lane keeps the larger of its pair iff (its bit D is clear) == up.
template <int D>
__device__ __forceinline__ uint64_t bcx(uint64_t v, bool up) {
    const uint64_t o = xor_lane64<D>(v);
    const bool keep_max = ((lane_id() & D) == 0) == up;
    return keep_max ? (v > o ? v : o) : (v < o ? v : o);
}
// 32-bit compare-exchange and descending sort of the wave's 64 values (lane 0 the largest), VALU only.
template <int D>
__device__ __forceinline__ uint32_t bcx32(uint32_t v, bool up) {
    const uint32_t o = xor_lane32<D>(v);
    const bool keep_max = ((lane_id() & D) == 0) == up;
    const uint32_t hi = v > o ? v : o, lo = v > o ? o : v;
    return keep_max ? hi : lo;
}
__device__ __forceinline__ uint32_t sort64_desc_u32(uint32_t v) {
    const int lane = lane_id();
    { const bool up = (lane & 2) == 0; v = bcx32<1>(v, up); }
    { const bool up = (lane & 4) == 0; v = bcx32<2>(v, up); v = bcx32<1>(v, up); }
    { const bool up = (lane & 8) == 0; v = bcx32<4>(v, up); v = bcx32<2>(v, up); v = bcx32<1>(v, up); }
    { const bool up = (lane & 16) == 0;
      v = bcx32<8>(v, up); v = bcx32<4>(v, up); v = bcx32<2>(v, up); v = bcx32<1>(v, up); }
    { const bool up = (lane & 32) == 0;
      v = bcx32<16>(v, up); v = bcx32<8>(v, up); v = bcx32<4>(v, up); v = bcx32<2>(v, up); v = bcx32<1>(v, up); }
    v = bcx32<32>(v, true); v = bcx32<16>(v, true); v = bcx32<8>(v, true); v = bcx32<4>(v, true);
    v = bcx32<2>(v, true);
    return bcx32<1>(v, true);
}

// The wave's 64 values sorted, descending (lane 0 the largest) or ascending.
template <bool DESC>
__device__ __forceinline__ uint64_t sort64(uint64_t v) {
    const int lane = lane_id();
    { const bool up = ((lane & 2) == 0) == DESC; v = bcx<1>(v, up); }
    { const bool up = ((lane & 4) == 0) == DESC; v = bcx<2>(v, up); v = bcx<1>(v, up); }
    { const bool up = ((lane & 8) == 0) == DESC; v = bcx<4>(v, up); v = bcx<2>(v, up); v = bcx<1>(v, up); }
    { const bool up = ((lane & 16) == 0) == DESC;
      v = bcx<8>(v, up); v = bcx<4>(v, up); v = bcx<2>(v, up); v = bcx<1>(v, up); }
    { const bool up = ((lane & 32) == 0) == DESC;
      v = bcx<16>(v, up); v = bcx<8>(v, up); v = bcx<4>(v, up); v = bcx<2>(v, up); v = bcx<1>(v, up); }
    v = bcx<32>(v, DESC); v = bcx<16>(v, DESC); v = bcx<8>(v, DESC); v = bcx<4>(v, DESC); v = bcx<2>(v, DESC);
    return bcx<1>(v, DESC);
}
// The top 64 of a (sorted descending) and b (sorted ascending), sorted descending (DESC) or ascending: the lane-wise
// maximum is a bitonic sequence holding them, then a bitonic merge.
template <bool DESC = true>
__device__ __forceinline__ uint64_t merge_top64(uint64_t a_desc, uint64_t b_asc) {
    uint64_t v = a_desc > b_asc ? a_desc : b_asc;
    v = bcx<32>(v, DESC); v = bcx<16>(v, DESC); v = bcx<8>(v, DESC); v = bcx<4>(v, DESC); v = bcx<2>(v, DESC);
    return bcx<1>(v, DESC);
}

}  // namespace fs

#endif  // FERRO_SAMPLER_DEVICE_HPP

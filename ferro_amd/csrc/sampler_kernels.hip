// sampler_kernels.hip - the C ABI of include/ferro_sampler.h: contexts, plans, the kernel choice and the launches; and the
// small kernels around sampling (softcap, penalties in place, draw streams).
#include "sampler_device.hpp"
#include "sampler_launch.hpp"

namespace fs {

__global__ __launch_bounds__(256) void softcap_kernel(const float* in, float* out, int64_t n, float cap) {
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256)
        out[i] = softcap_one(in[i], cap);
}

// In-place penalty pass (fs_penalize_batch): ferro's sample() leaves its host row penalised (sampler.cpp:11-18),
// and a caller that reads the row back afterwards (lm_cli.cpp:353) sees those values. One workgroup per
// (row, 8192-id chunk): the window's ids that fall in the chunk are counted in a 16-bit LDS table, then every
// counted logit is rewritten once with the same arithmetic as the sampling kernels.
constexpr int PEN_BLOCK = 256;
constexpr int PEN_CHUNK = 8192;

__global__ __launch_bounds__(PEN_BLOCK) void penalize_kernel(float* logits, int64_t ld, int V, const int32_t* hist,
                                                            const int64_t* hist_off, const fs_row_params* params,
                                                            int nchunk, int32_t* err) {
    __shared__ uint32_t cnt[PEN_CHUNK / 2];
    const int tid = threadIdx.x;
    const int row = (int)blockIdx.x / nchunk;
    const int lo = ((int)blockIdx.x - row * nchunk) * PEN_CHUNK;
    const fs_row_params p = ld_const(params + row);
    const bool rep_on = p.repetition_penalty != 1.0f;
    const bool fp_on = p.frequency_penalty != 0.0f || p.presence_penalty != 0.0f;
    if (!(rep_on || fp_on) || p.repeat_last_n == 0 || !hist || !hist_off) return;
    const int64_t h0 = ld_const(hist_off + row);
    const int64_t len = ld_const(hist_off + row + 1) - h0;
    const int64_t b = window_begin(len, p);
    if (b >= len) return;
    for (int i = tid; i < PEN_CHUNK / 2; i += PEN_BLOCK) cnt[i] = 0u;
    __syncthreads();
    bool ovf = false;
    for (int64_t i = b + tid; i < len; i += PEN_BLOCK) {
        const int id = hist[h0 + i];
        const uint32_t rel = (uint32_t)(id - lo);
        if (id >= 0 && id < V && rel < (uint32_t)PEN_CHUNK) {
            const uint32_t sh = (rel & 1u) * 16u;
            const uint32_t old = atomicAdd(&cnt[rel >> 1], 1u << sh);
            ovf |= ((old >> sh) & 0xFFFFu) == 0xFFFFu;
        }
    }
    if (ovf) atomicOr(err, FS_DEVERR_COUNT_OVERFLOW);
    __syncthreads();
    float* rowp = logits + (int64_t)row * ld + lo;
    for (int i = tid; i < PEN_CHUNK / 2; i += PEN_BLOCK) {
        const uint32_t c2 = cnt[i];
        if (c2 == 0u) continue;
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            const uint32_t c = (c2 >> (16 * q)) & 0xFFFFu;
            if (c != 0u) {                                  // a counted id is < V
                float l = rowp[2 * i + q];
                if (rep_on) l = l > 0.0f ? __fdiv_rn(l, p.repetition_penalty) : __fmul_rn(l, p.repetition_penalty);
                if (fp_on) l = __fsub_rn(l, __fadd_rn(__fmul_rn((float)c, p.frequency_penalty), p.presence_penalty));
                rowp[2 * i + q] = l;
            }
        }
    }
}

// ------------------------------------------------------------------------------------------------ draw streams
// std::mt19937_64 (the standard's parameters: n = 312, m = 156, r = 31, a = 0xB5026F5AA96619E9, tempering
// u = 29 / d = 0x5555555555555555, s = 17 / b = 0x71D67FFFEDA60000, t = 37 / c = 0xFFF7EEE000000000, l = 43) per
// stream, and libstdc++'s generate_canonical<double, 53> of one 64-bit output: (double)x / 2^64, kept below 1.
// This is ferro::Sampler's draw (sampler.h:25,32; sampler.cpp:45-46) moved next to the sampler.

// One thread per stream. Stream s owns rows row_off[s] .. row_off[s+1]-1 (row_off NULL: row s alone); each row
// whose stream samples takes one draw, in row order; greedy streams take none and get u = 0. peek != 0 leaves the
// state unchanged (the draws are computed from it: at most MT_M draws past a twist).
__global__ __launch_bounds__(64) void drng_draw_kernel(uint64_t* mts, int32_t* idxs, int n_streams,
                                                       const int64_t* row_off, const fs_row_params* params,
                                                       double* u, int peek, int32_t* err) {
    const int sidx = (int)(blockIdx.x * blockDim.x + threadIdx.x);
    if (sidx >= n_streams) return;
    uint64_t* mt = mts + (int64_t)sidx * MT_N;
    int idx = idxs[sidx];
    const int64_t r0 = row_off ? row_off[sidx] : sidx;
    const int64_t r1 = row_off ? row_off[sidx + 1] : sidx + 1;
    const bool smp = samples(params[sidx]);
    for (int64_t r = r0; r < r1; ++r) {
        if (!smp) { u[r] = 0.0; continue; }
        uint64_t y;
        if (!peek) {
            if (idx >= MT_N) { mt_twist(mt); idx = 0; }
            y = mt[idx++];
        } else {
            if (idx < MT_N) {
                y = mt[idx++];
            } else {
                const int k = idx - MT_N;                    // the k-th value of the next twist, from the old state
                if (k >= MT_M) { atomicOr(err, FS_DEVERR_INTERNAL); u[r] = 0.0; continue; }
                y = mt_twist_one(mt[k], mt[k + 1], mt[k + MT_M]);
                ++idx;
            }
        }
        u[r] = mt_canonical(mt_temper(y));
    }
    if (!peek) idxs[sidx] = idx;
}

// Advance stream s by counts[s] draws, or, for a stream that does not sample, by none.
__global__ __launch_bounds__(64) void drng_skip_kernel(uint64_t* mts, int32_t* idxs, int n_streams,
                                                       const int32_t* counts, const fs_row_params* params) {
    const int sidx = (int)(blockIdx.x * blockDim.x + threadIdx.x);
    if (sidx >= n_streams || !samples(params[sidx])) return;
    uint64_t* mt = mts + (int64_t)sidx * MT_N;
    int idx = idxs[sidx];
    for (int32_t c = counts[sidx]; c > 0;) {
        if (idx >= MT_N) { mt_twist(mt); idx = 0; }
        const int take = MT_N - idx < c ? MT_N - idx : c;
        idx += take;
        c -= take;
    }
    idxs[sidx] = idx;
}

}  // namespace fs

// ================================================================================================ host side
struct fs_context {
    std::mutex mu;
    int device = -1;
    int cus = 0;               // compute units of the device
    int xccs = 0;              // XCDs of the device (hipDeviceAttributeNumberOfXccs)
    bool seg_layout = true;    // the segment grid's hand-off holds on this device (XCDS % xccs == 0)
    int32_t* hflag = nullptr;  // host-mapped: a merge of an earlier call gave up (set by the kernel, read here)
    int32_t* hflag_dev = nullptr;
    bool captured = false;     // a call was recorded into a graph: workspaces are retired, never freed, on growth
    std::vector<void*> retired;
    uint64_t* sk_lists = nullptr;   // small-k kernel: [slots][SK_K] sorted segment lists
    size_t sk_slots = 0;
    uint32_t* sk_ticket = nullptr;  // small-k kernel: [rows] segment tickets, left at 0
    size_t sk_rows = 0;
    uint32_t* mk_ctr = nullptr;     // mid-k kernel: [mk_ctr_rows][MK_CTR] counters, left at 0
    uint64_t* mk_list = nullptr;    //   [mk_list_rows][MK_LIST] candidate lists
    uint64_t* mk_spill = nullptr;   //   [mk_spill_rows][MK_SPILL] penalised logits (batches with penalties)
    uint64_t* mk_mass = nullptr;    //   [mk_mass_rows][2048] mass bins, left at 0 (batches with every token a candidate)
    uint32_t* mk_qk = nullptr;      //   [mk_segs][SK_NW][16] published lane maxima
    size_t mk_ctr_rows = 0, mk_list_rows = 0, mk_spill_rows = 0, mk_mass_rows = 0, mk_segs = 0;
    int mk_wait = 0;                //   calls that still go without trying again after an allocation failed
    uint64_t* cand = nullptr;
    size_t cand_slots = 0;     // chunk slots of CAP entries
    uint32_t* meta = nullptr;
    uint32_t* rhist = nullptr;  // [row_cap][RBINS]
    uint64_t* rmass = nullptr;  // [row_cap][LB]
    size_t row_cap = 0;
    uint32_t* stream_cnt = nullptr;
    size_t stream_cap = 0;
    int32_t* err = nullptr;        // [0]: error bits; [1]: dirty (a merge gave up; see fs_device_error); [2..3]: hflag_dev
    uint32_t merge_spins = fs::MERGE_SPINS;
    int static_dev = -1;       // device whose static workspace fs_sample_batch_static used with this context
    uint64_t* trace = nullptr; // FS_TRACE builds: phase timestamps, trace_cap entries (fs_trace_set)
    int64_t trace_cap = 0;
    fs_row_params* greedy = nullptr;      // fs_argmax_batch without parameters: [greedy_cap] greedy records
    size_t greedy_cap = 0;
    std::vector<fs_row_params> h_greedy;  //   and their host copy (the small-k kernel's greedy path)
};

namespace fs {
__global__ __launch_bounds__(256) void zero_words_kernel(uint32_t* p, int64_t n) {
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) p[i] = 0u;
}
// n parameter records of a greedy row without penalties (fs_argmax_batch without parameters)
__global__ __launch_bounds__(256) void greedy_params_kernel(fs_row_params* p, int64_t n) {
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) {
        fs_row_params r;
        r.temperature = 0.0f; r.top_k = 1; r.top_p = 1.0f; r.min_p = 0.0f; r.repetition_penalty = 1.0f;
        r.frequency_penalty = 0.0f; r.presence_penalty = 0.0f; r.repeat_last_n = 0; r.penalty_from = 0;
        r.softcap = 0.0f;
        p[i] = r;
    }
}
}  // namespace fs

namespace {

// Zero n words on st with a fill kernel (no hipMemsetAsync: the call may be recorded into a graph).
void clear_words(hipStream_t st, void* p, int64_t n) {
    if (!p || n <= 0) return;
    const int64_t blocks = std::min<int64_t>(1024, (n + 255) / 256);
    hipLaunchKernelGGL(fs::zero_words_kernel, dim3((unsigned)blocks), dim3(256), 0, st, (uint32_t*)p, n);
}

// A workspace buffer that is replaced: freed, or, once a call of the context has been recorded into a HIP graph
// (whose replays keep using the old addresses), kept until fs_destroy.
void release(fs_context* c, void* p) {
    if (!p) return;
    if (c->captured) c->retired.push_back(p);
    else (void)hipFree(p);
}

int grow(fs_context* c, size_t slots, size_t rows, size_t streams) {
    if (slots > c->cand_slots) {
        release(c, c->cand);
        release(c, c->meta);
        c->cand = nullptr; c->meta = nullptr; c->cand_slots = 0;
        if (hipMalloc(&c->cand, slots * fs::CAP * sizeof(uint64_t)) != hipSuccess) return FS_E_NOMEM;
        if (hipMalloc(&c->meta, slots * 2 * sizeof(uint32_t)) != hipSuccess) return FS_E_NOMEM;
        c->cand_slots = slots;
    }
    if (rows > c->row_cap) {
        release(c, c->rhist);
        release(c, c->rmass);
        c->rhist = nullptr; c->rmass = nullptr; c->row_cap = 0;
        if (hipMalloc(&c->rhist, rows * fs::RBINS * sizeof(uint32_t)) != hipSuccess) return FS_E_NOMEM;
        if (hipMemset(c->rhist, 0, rows * fs::RBINS * sizeof(uint32_t)) != hipSuccess) return FS_E_HIP;
        if (hipMalloc(&c->rmass, rows * fs::LB * sizeof(uint64_t)) != hipSuccess) return FS_E_NOMEM;
        if (hipMemset(c->rmass, 0, rows * fs::LB * sizeof(uint64_t)) != hipSuccess) return FS_E_HIP;
        c->row_cap = rows;
    }
    if (streams > c->stream_cap) {
        release(c, c->stream_cnt);
        c->stream_cnt = nullptr; c->stream_cap = 0;
        if (hipMalloc(&c->stream_cnt, streams * sizeof(uint32_t)) != hipSuccess) return FS_E_NOMEM;
        if (hipMemset(c->stream_cnt, 0, streams * sizeof(uint32_t)) != hipSuccess) return FS_E_HIP;
        c->stream_cap = streams;
    }
    if (!c->hflag) {
        if (hipHostMalloc((void**)&c->hflag, sizeof(int32_t), hipHostMallocMapped) != hipSuccess) return FS_E_NOMEM;
        *(volatile int32_t*)c->hflag = 0;
        if (hipHostGetDevicePointer((void**)&c->hflag_dev, c->hflag, 0) != hipSuccess) return FS_E_HIP;
    }
    if (!c->err) {
        // error bits, dirty flag, then the device address of the host-mapped give-up flag (read by a give-up only)
        int32_t h[4] = {0, 0, 0, 0};
        const uint64_t fa = (uint64_t)(uintptr_t)c->hflag_dev;
        memcpy(h + 2, &fa, sizeof(fa));
        if (hipMalloc(&c->err, sizeof(h)) != hipSuccess) return FS_E_NOMEM;
        if (hipMemcpy(c->err, h, sizeof(h), hipMemcpyHostToDevice) != hipSuccess) return FS_E_HIP;
    }
    return FS_OK;
}

// Segments: at most two per CU over the whole batch (all resident at once: a second round of a few workgroups
// would double the time), at least one per row; a segment streams >= 1 full tile of 4096 logits. The merge
// handles each row's partial last tile (all of a row shorter than one tile). Sets a.nseg / a.seg_tiles and the
// workspace the call needs (items = (row, segment) slots).
// max_slots > 0 caps the workspace slots (XCDS * nseg * ceil(rows / XCDS)) by taking fewer segments per row; one
// segment per row always fits rows <= max_slots.
int plan(int cus, fs::Args& a, int64_t rows, int64_t& items, int64_t& seg_grid, int64_t max_slots = 0,
         int per_cu = 2) {
    const int64_t tiles_row = a.V / fs::TILE;
    const int64_t per_slot = (rows + fs::XCDS - 1) / fs::XCDS;
    a.nseg = 0;
    a.seg_tiles = 1;
    if (tiles_row > 0) {
        int64_t want = ((int64_t)per_cu * (int64_t)cus) / rows;
        if (want < 1) want = 1;
        if (want > tiles_row) want = tiles_row;
        if (want > fs::BLOCK - 1) want = fs::BLOCK - 1;   // the merge gives each list (segments + tail) a thread
        for (;;) {
            a.seg_tiles = (int)((tiles_row + want - 1) / want);
            a.nseg = (int)((tiles_row + a.seg_tiles - 1) / a.seg_tiles);
            if (max_slots <= 0 || want <= 1 || (int64_t)fs::XCDS * a.nseg * per_slot <= max_slots) break;
            --want;
        }
    }
    if (a.nseg > fs::MAX_SEGS) return FS_E_INVALID;
    items = rows * a.nseg;
    if (items > 0x7fffffff) return FS_E_INVALID;
    // one workgroup per (row, segment), the rows dealt to XCDS slots (segment_kernel); each segment workgroup's
    // list slot is its index, so the workspace holds seg_grid slots
    seg_grid = items > 0 ? (int64_t)fs::XCDS * a.nseg * ((rows + fs::XCDS - 1) / fs::XCDS) : 0;
    if (seg_grid > 0x7fffffff) return FS_E_INVALID;
    items = seg_grid;
    // balanced layouts (sampling, >= 2 segments per row, >= 2 rows on some XCD, <= WAVE rows per XCD)
    // Balanced layouts: sampling, >= 2 segments per row, 16 to WAVE rows per XCD. Computing the layout delays every
    // workgroup by about 2 us, which pays on large mixed batches (B=256 x V=262144 with k from 1 to 2048: -20 us)
    // but not on small ones.
    a.balance = (a.mode == fs::MODE_SAMPLE && a.nseg >= 2 && (rows + fs::XCDS - 1) / fs::XCDS >= 16 &&
                 (rows + fs::XCDS - 1) / fs::XCDS <= fs::WAVE) ? 1 : 0;
    return FS_OK;
}

// Launches the sampling grid on a bound workspace (a.cand / meta / rhist / stream_cnt / err / dirty).
int launch_planned(const fs::Args& a, int64_t rows, int64_t seg_grid, hipStream_t st) {
    if (seg_grid > 0) {                            // the segments, then one merging workgroup per row (same grid)
        const int64_t grid = seg_grid + (int64_t)fs::XCDS * ((rows + fs::XCDS - 1) / fs::XCDS);
        if (grid > 0x7fffffff) return FS_E_INVALID;
        return fs::launch_segments(a, (unsigned)grid, st) == hipSuccess ? FS_OK : FS_E_HIP;
    }
    return fs::launch_merges(a, (unsigned)rows, a.nseg, 0, st) == hipSuccess ? FS_OK : FS_E_HIP;
}

// Every row sampled alone by one workgroup from its logits (a device whose XCD layout the segment grid's hand-off
// does not fit).
int launch_alone(fs::Args a, int64_t rows, hipStream_t st) {
    a.nseg = 0;
    a.balance = 0;
    return fs::launch_merges(a, (unsigned)rows, 0, 1, st) == hipSuccess ? FS_OK : FS_E_HIP;
}

// The segment grid places a row's segments and its merging workgroup on workgroups of one index class mod XCDS, so
// that they share an XCD (and its L2) under round-robin dispatch over the device's XCDs: that holds when the XCD
// count divides XCDS (8, 4, 2 or 1: every MI355X partition mode). On other devices every row is sampled alone.
bool layout_fits(int xccs) { return xccs >= 1 && fs::XCDS % xccs == 0; }

int device_of(fs_context* ctx) {
    if (ctx->device < 0) {
        int dev = -1;
        if (hipGetDevice(&dev) != hipSuccess) return FS_E_HIP;
        if (hipDeviceGetAttribute(&ctx->cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
            return FS_E_HIP;
        int x = 0;
        if (hipDeviceGetAttribute(&x, hipDeviceAttributeNumberOfXccs, dev) != hipSuccess) return FS_E_HIP;
        ctx->xccs = x;
        ctx->seg_layout = layout_fits(x);
        ctx->device = dev;
    }
    return FS_OK;
}

// Whether an earlier call's merge gave up waiting for its segments (the kernel sets the host-mapped flag). The
// caller then enqueues, ahead of its own launch, fill kernels that clear what the late segments may have left (they
// have finished once the stream reaches the fills), so the call runs normally instead of computing every row alone;
// it returns FS_W_RECOVERED. The error bits stay for fs_device_error.
bool gave_up(int32_t* flag) {
    if (!flag || *(volatile int32_t*)flag == 0) return false;
    *(volatile int32_t*)flag = 0;
    return true;
}

bool capturing(hipStream_t st) {
    hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
    return hipStreamIsCapturing(st, &cs) == hipSuccess && cs != hipStreamCaptureStatusNone;
}

// ---- small-k kernel (fs_sample_batch_hp)
// Whether every row of the batch fits the small-k kernel: greedy, or k = min(top_k or V, V) <= SK_K, with no
// frequency / presence penalty (h: the host copy of the parameters).
// A batch whose rows cost very differently: rows sampled with 64 < k <= KMAX beside greedy or k <= 64 rows, none on
// the whole-row path (k > KMAX), 16 to 64 rows per XCD (the balanced layout). The host copy of the parameters shows
// the mix, and such batches take about four segments per CU instead of two, which gives the balanced layout finer
// shares to apportion. It is reached by batches the mid-k kernel does not take (more than 262144 logits, or too few for
// their largest k). k spread evenly over 1 to 2048 by its logarithm, with two segments per CU and with four: 384 rows of
// 262208 logits 224 us and 167, of 50000 106 and 88; but 256 rows of 262208 116 and 131, of 32000 89 and 96 (the rule dates
// from 256 rows of 262144, which the mid-k kernel now has). Uniform batches lose with more segments (more lists to merge, a
// second round of workgroups).
bool mixed_merges(const fs_row_params* h, int64_t B, int32_t V) {
    const int64_t per_x = (B + fs::XCDS - 1) / fs::XCDS;
    if (per_x < 16 || per_x > fs::WAVE) return false;
    bool heavy = false, light = false;
    for (int64_t b = 0; b < B; ++b) {
        const fs_row_params& p = h[b];
        const bool greedy = !(p.temperature > 0.0f && p.top_k != 1);
        const int64_t k = greedy ? 1 : ((p.top_k > 0 && p.top_k < V) ? p.top_k : V);
        if (k > fs::KMAX) return false;
        if (k > 64) heavy = true;
        else light = true;
    }
    return heavy && light;
}

bool small_k_batch(const fs_row_params* h, int64_t B, int32_t V) {
    for (int64_t b = 0; b < B; ++b) {
        const fs_row_params& p = h[b];
        const bool greedy = p.temperature <= 0.0f || p.top_k == 1;
        if (!greedy && (p.frequency_penalty != 0.0f || p.presence_penalty != 0.0f)) return false;
        const int64_t k = (p.top_k > 0 && p.top_k < V) ? p.top_k : V;
        if (!greedy && k > fs::SK_K) return false;
    }
    return true;
}

// Logits per thread (NL float4 loads) and segments per row: the largest segments that still give every CU four
// workgroups, else the smallest (most workgroups) whose row fits SK_MAX_SEGS lists; 0 when none does.
int small_k_plan(int cus, int64_t B, int32_t V, int& nl, int& nseg) {
    nl = 0;
    nseg = 0;
    const int nls[3] = {16, 8, 4};
    for (int i = 0; i < 3; ++i) {
        const int64_t seg = (int64_t)fs::SK_LT * nls[i] * 4;
        const int64_t n = ((int64_t)V + seg - 1) / seg;
        if (n > fs::SK_MAX_SEGS) break;
        nl = nls[i];
        nseg = (int)n;
        if (B * n >= 4 * (int64_t)cus) break;
    }
    return nl > 0 ? FS_OK : FS_E_INVALID;
}

int grow_small(fs_context* c, size_t slots, size_t rows) {
    if (slots > c->sk_slots) {
        release(c, c->sk_lists);
        c->sk_lists = nullptr; c->sk_slots = 0;
        if (hipMalloc(&c->sk_lists, slots * fs::SK_K * sizeof(uint64_t)) != hipSuccess) return FS_E_NOMEM;
        c->sk_slots = slots;
    }
    if (rows > c->sk_rows) {
        release(c, c->sk_ticket);
        c->sk_ticket = nullptr; c->sk_rows = 0;
        if (hipMalloc(&c->sk_ticket, rows * sizeof(uint32_t)) != hipSuccess) return FS_E_NOMEM;
        if (hipMemset(c->sk_ticket, 0, rows * sizeof(uint32_t)) != hipSuccess) return FS_E_HIP;
        c->sk_rows = rows;
    }
    return FS_OK;
}

// Verification windows fit the small-k kernel when every stream does and none has an active penalty (a row's
// history would then include the drafts fed before it).
bool small_k_windows(const fs_row_params* h, int64_t S, int32_t V) {
    if (!small_k_batch(h, S, V)) return false;
    for (int64_t s = 0; s < S; ++s)
        if ((h[s].repetition_penalty != 1.0f || h[s].frequency_penalty != 0.0f || h[s].presence_penalty != 0.0f) &&
            h[s].repeat_last_n != 0)
            return false;
    return true;
}

// B greedy parameter records without penalties on the device (filled by a kernel on st, no memset: the call may be
// captured) and on the host. The caller holds ctx->mu.
int greedy_params(fs_context* ctx, int64_t B, hipStream_t st) {
    if ((size_t)B <= ctx->greedy_cap) return FS_OK;
    const size_t cap = std::max<size_t>((size_t)B, 2 * ctx->greedy_cap);
    release(ctx, ctx->greedy);
    ctx->greedy = nullptr;
    ctx->greedy_cap = 0;
    if (hipMalloc(&ctx->greedy, cap * sizeof(fs_row_params)) != hipSuccess) return FS_E_NOMEM;
    const int64_t blocks = std::min<int64_t>(1024, ((int64_t)cap + 255) / 256);
    hipLaunchKernelGGL(fs::greedy_params_kernel, dim3((unsigned)blocks), dim3(256), 0, st, ctx->greedy, (int64_t)cap);
    if (hipGetLastError() != hipSuccess) return FS_E_HIP;
    fs_row_params r = {};
    r.temperature = 0.0f; r.top_k = 1; r.top_p = 1.0f; r.repetition_penalty = 1.0f;
    ctx->h_greedy.assign(cap, r);
    ctx->greedy_cap = cap;
    return FS_OK;
}

// The small-k kernel's plan for n host parameter records (B rows, or n_streams windows with `verify`): false when
// the batch does not fit it (the fused kernel runs). nl / nseg: its segments; all_greedy: the greedy-only form;
// capped: some row has a softcap; may_pen: some row has an active penalty window.
struct SmallKChoice {
    int nl = 0, nseg = 0;
    bool all_greedy = true, capped = false, may_pen = false;
};
bool small_k_choice(int cus, const fs_row_params* h, int64_t n, int64_t B, int32_t V, bool verify, SmallKChoice& c) {
    if (verify ? !small_k_windows(h, n, V) : !small_k_batch(h, n, V)) return false;
    if (small_k_plan(cus, B, V, c.nl, c.nseg) != FS_OK) return false;
    if ((int64_t)fs::XCDS * c.nseg * ((B + fs::XCDS - 1) / fs::XCDS) > 0x7fffffff) return false;
    bool counts = false;
    for (int64_t b = 0; b < n; ++b) {
        const fs_row_params& p = h[b];
        const bool fp = p.frequency_penalty != 0.0f || p.presence_penalty != 0.0f;
        c.all_greedy = c.all_greedy && !(p.temperature > 0.0f && p.top_k != 1);
        c.capped |= p.softcap > 0.0f;
        c.may_pen |= (p.repetition_penalty != 1.0f || fp) && p.repeat_last_n != 0;
        counts |= fp && p.repeat_last_n != 0;
    }
    return !(counts && c.nl != 4);               // count tables fit segments of 4096 logits only: the fused kernel
}

fs::SkArgs row_args(const fs_context* ctx, const fs::Args& a, int nseg) {
    fs::SkArgs k = {};
    k.logits = a.logits; k.ld = a.ld; k.B = a.B; k.V = a.V; k.nseg = nseg;
    k.hist = a.hist; k.hist_off = a.hist_off; k.params = a.params; k.u = a.u; k.tok = a.tok; k.kcap = a.kcap;
    k.cand_ids = a.cand_ids; k.cand_probs = a.cand_probs; k.keep = a.keep;
    k.err = ctx->err;
    k.mode = a.mode; k.rows = a.rows; k.row_off = a.row_off; k.n_streams = a.n_streams; k.eos = a.eos;
    k.accepted = a.accepted; k.stream_cnt = ctx->stream_cnt;
    k.dmt = a.dmt; k.didx = a.didx; k.out_hist = a.out_hist; k.out_hist_off = a.out_hist_off; k.out_cap = a.out_cap;
    return k;
}

// Launches the small-k kernel when the batch fits it; *used = false (nothing launched) otherwise. a.mode selects
// sampling (h_params: B records) or verification windows (h_params: n_streams records).
// h_params NULL: every row greedy without penalties (fs_argmax_batch without parameters): the context's greedy
// records stand for the parameters, on the device and the host.
int launch_small(fs_context* ctx, const fs::Args& a_in, const fs_row_params* h_params, hipStream_t st, bool& used) {
    used = false;
    std::lock_guard<std::mutex> g(ctx->mu);
    int rc = device_of(ctx);
    if (rc != FS_OK) return rc;
    fs::Args a = a_in;
    if (!h_params) {
        rc = greedy_params(ctx, a.B, st);
        if (rc != FS_OK) return rc;
        h_params = ctx->h_greedy.data();
        a.params = ctx->greedy;
    }
    const bool verify = a.mode == fs::MODE_VERIFY;
    if (!ctx->seg_layout) return FS_OK;
    SmallKChoice ch;
    if (!small_k_choice(ctx->cus, h_params, verify ? (int64_t)a.n_streams : (int64_t)a.B, a.B, a.V, verify, ch))
        return FS_OK;
    const int nl = ch.nl, nseg = ch.nseg;
    const int64_t per_x = ((int64_t)a.B + fs::XCDS - 1) / fs::XCDS;
    const int64_t grid = (int64_t)fs::XCDS * nseg * per_x;
    // the error word and the verify stream counters: a 64-bit word per stream, then the 32-bit counters of streams
    // longer than 32 rows
    rc = grow(ctx, 0, 0, verify ? 3 * (size_t)a.n_streams : 0);
    if (rc != FS_OK) return rc;
    rc = grow_small(ctx, (size_t)a.B * nseg, (size_t)a.B);
    if (rc != FS_OK) return rc;
    if (capturing(st)) ctx->captured = true;
    fs::SkArgs k = row_args(ctx, a, nseg);
    k.lists = ctx->sk_lists; k.ticket = ctx->sk_ticket;
    k.trace = nullptr;
#ifdef FS_TRACE
    if (ctx->trace && grid * fs::TRACE_W <= ctx->trace_cap) k.trace = ctx->trace;
#endif
    const bool capped = ch.capped, all_greedy = ch.all_greedy;
    bool may_pen = ch.may_pen;
    // a verification window reaches this kernel only without an active penalty (small_k_windows)
    may_pen = may_pen && !verify && a.hist && a.hist_off;
    const int flags = (may_pen ? fs::SK_MAY_PEN : 0) | (a.out_hist_off ? fs::SK_COPY : 0);
    if (fs::launch_small_k(nl, capped, all_greedy, (unsigned)grid, flags, k, st) != hipSuccess) return FS_E_HIP;
    used = true;
    return FS_OK;
}

// ---- mid-k kernel (fs_sample_batch_hp, fs_verify_hp, fs_decode_step_hp)
// Every row greedy or sampling from k <= 2048 candidates or from every token, with any penalty. The row's bound comes from its lanes'
// maxima (one per 4 * nl logits): twice as many as the largest k keep the candidates at about 1.4 k, and a row's
// segments publish at most 64 lists of 16 per 4 * nl loads, which the bound's search reads in one round.
struct MidKChoice {
    int nl = 0, nseg = 0;
    bool capped = false, may_pen = false, all = false;
};
bool mid_k_choice(int cus, const fs_row_params* h, int64_t n, int64_t rows, int32_t V, bool outputs, MidKChoice& c) {
    int64_t kmax = 1;
    for (int64_t b = 0; b < n; ++b) {
        const fs_row_params& p = h[b];
        const bool greedy = !(p.temperature > 0.0f && p.top_k != 1);
        const int64_t k = greedy ? 1 : ((p.top_k > 0 && p.top_k < V) ? p.top_k : V);
        if (k == V && k > fs::KMAX) {
            // every token a candidate: no candidate outputs and no min-p (its count and sum over the kept logits)
            // (taken whatever the rows hold, which the host cannot see. Rows whose mass is a few logits take about as long as
            // on the fused kernel with its short list: heavy-tailed logits at temperature 0.3, 1 row of 65536 19.1 us here
            // and 18.4 there, 16 rows 19.2 and 19.1, 64 of 262144 33.5 and 36.4. Rows with a body gain: 16 rows of 65536
            // N(0, 2) logits 24.0 and 28.3 at temperature 0.2, 27.5 and 62.4 at 1)
            if (outputs || p.min_p > 0.0f) return false;
            c.all = true;
        } else {
            kmax = std::max(kmax, k);
        }
        c.capped |= p.softcap > 0.0f;
        c.may_pen |= (p.repetition_penalty != 1.0f || p.frequency_penalty != 0.0f || p.presence_penalty != 0.0f) &&
                     p.repeat_last_n != 0;
    }
    if (kmax > fs::KMAX) return false;
    // the smallest segments whose workgroups are all resident at once (four per CU), else the largest: a second round of
    // a few workgroups delays its rows by a whole one (40 rows of 262144 logits, 1280 workgroups of 8192 logits: 30.8 us
    // against 24 with 640 of 16384)
    c.nl = 0;
    for (const int nl : {4, 8, 16}) {
        const int64_t seg = (int64_t)fs::SK_LT * nl * 4, n = ((int64_t)V + seg - 1) / seg;
        if (n * nl > 256 || n > fs::MK_MAX_SEGS) continue;
        c.nl = nl;
        c.nseg = (int)n;
        if (rows * n <= 4 * (int64_t)cus) break;
    }
    if (c.nl == 0 || (int64_t)V < 8 * c.nl * kmax) return false;
    return (int64_t)fs::XCDS * c.nseg * ((rows + fs::XCDS - 1) / fs::XCDS) <= 0x7fffffff;
}

// One buffer of the mid-k kernel's workspace: at least n elements of `per` words each, half as many again when it grows.
// FS_E_NOMEM leaves the old one as it was.
template <class T>
int grow_buffer(fs_context* c, T*& p, size_t& cap, size_t n, size_t per, bool zero) {
    if (n <= cap) return FS_OK;
    T* q = nullptr;
    size_t m = std::max(n, cap + cap / 2);
    if (hipMalloc(&q, m * per * sizeof(T)) != hipSuccess) {
        m = n;
        if (hipMalloc(&q, m * per * sizeof(T)) != hipSuccess) {
            (void)hipGetLastError();
            return FS_E_NOMEM;
        }
    }
    if (zero && hipMemset(q, 0, m * per * sizeof(T)) != hipSuccess) {
        (void)hipFree(q);
        return FS_E_HIP;
    }
    release(c, p);
    p = q;
    cap = m;
    return FS_OK;
}

// Whether a call needs more than the context holds.
bool mid_grows(const fs_context* c, const MidKChoice& ch, size_t rows) {
    return rows * ch.nseg > c->mk_segs || rows > c->mk_ctr_rows || rows > c->mk_list_rows ||
           (ch.may_pen && rows > c->mk_spill_rows) || (ch.all && rows > c->mk_mass_rows);
}

// About 33 KB per row, 128 KB more with penalties and 16 KB with every token a candidate. After a failed allocation the
// next 64 calls that would have to grow don't try.
int grow_mid(fs_context* c, const MidKChoice& ch, size_t rows) {
    if (!mid_grows(c, ch, rows)) return FS_OK;
    if (c->mk_wait > 0) {
        --c->mk_wait;
        return FS_E_NOMEM;
    }
    int rc = grow_buffer(c, c->mk_qk, c->mk_segs, rows * ch.nseg, fs::SK_NW * 16, false);
    if (rc == FS_OK) rc = grow_buffer(c, c->mk_ctr, c->mk_ctr_rows, rows, fs::MK_CTR, true);
    if (rc == FS_OK) rc = grow_buffer(c, c->mk_list, c->mk_list_rows, rows, fs::MK_LIST, false);
    if (rc == FS_OK && ch.may_pen) rc = grow_buffer(c, c->mk_spill, c->mk_spill_rows, rows, fs::MK_SPILL, false);
    if (rc == FS_OK && ch.all) rc = grow_buffer(c, c->mk_mass, c->mk_mass_rows, rows, 2048, true);
    if (rc == FS_E_NOMEM) c->mk_wait = 64;
    return rc;
}

// The fused kernel's layout for a call (a.nseg, a.seg_tiles, a.balance, its grid) and the workspace it needs.
int grow_fused(fs_context* ctx, fs::Args& a, int64_t rows, int64_t streams, int per_cu, int64_t* grid) {
    int64_t items = 0;
    const int rc = plan(ctx->cus, a, rows, items, *grid, 0, per_cu);
    if (rc != FS_OK) return rc;
    // verify: a 64-bit word per stream, then the 32-bit counters of streams longer than 32 rows
    return grow(ctx, (size_t)(items > 0 ? items : 1), (size_t)rows, (size_t)(streams > 0 ? 3 * streams : 1));
}

// Launches the mid-k kernel when the batch fits it; *used = false (nothing launched) otherwise. Under capture a
// workspace that would have to grow leaves the batch to the fused kernel (no allocation in a capture that worked
// without one), and so does one that the device has no room for.
// per_cu: as launch's; the fused kernel's workspace grows as launch would grow it, so that a context warmed up with any
// parameters of a shape allocates nothing when a call of that shape with others is recorded.
int launch_mid(fs_context* ctx, const fs::Args& a, const fs_row_params* h_params, hipStream_t st, bool& used, int per_cu = 2) {
    used = false;
    std::lock_guard<std::mutex> g(ctx->mu);
    int rc = device_of(ctx);
    if (rc != FS_OK) return rc;
    if (!ctx->seg_layout) return FS_OK;
    const bool verify = a.mode == fs::MODE_VERIFY;
    MidKChoice ch;
    if (!mid_k_choice(ctx->cus, h_params, verify ? (int64_t)a.n_streams : (int64_t)a.B, a.B, a.V,
                      a.cand_ids || a.cand_probs, ch))
        return FS_OK;
    const size_t streams = verify ? 3 * (size_t)a.n_streams : 0;
    const bool cap = capturing(st);
    if (cap && (mid_grows(ctx, ch, (size_t)a.B) || streams > ctx->stream_cap || !ctx->err)) return FS_OK;
    if (!cap) {
        fs::Args fused = a;
        int64_t fused_grid = 0;
        rc = grow_fused(ctx, fused, a.B, verify ? a.n_streams : 0, per_cu, &fused_grid);
    }
    if (rc == FS_E_NOMEM || rc == FS_E_INVALID) {   // (this kernel does not need it)
        (void)hipGetLastError();
        rc = grow(ctx, 0, 0, streams);
    }
    if (rc != FS_OK) return rc;
    rc = grow_mid(ctx, ch, (size_t)a.B);
    if (rc == FS_E_NOMEM) return FS_OK;
    if (rc != FS_OK) return rc;
    if (cap) ctx->captured = true;
    fs::MkArgs m = {};
    m.a = row_args(ctx, a, ch.nseg);
    m.ctr = ctx->mk_ctr; m.qk = ctx->mk_qk; m.list = ctx->mk_list; m.spill = ctx->mk_spill;
    m.mass = ctx->mk_mass; m.spins = ctx->merge_spins;
    const int64_t grid = (int64_t)fs::XCDS * ch.nseg * (((int64_t)a.B + fs::XCDS - 1) / fs::XCDS);
#ifdef FS_TRACE
    if (ctx->trace && grid * fs::TRACE_W <= ctx->trace_cap) m.a.trace = ctx->trace;
#endif
    const int flags = (ch.may_pen ? fs::SK_MAY_PEN : 0) | (a.out_hist_off ? fs::SK_COPY : 0) |
                      (verify ? fs::MK_VERIFY : 0);
    if (fs::launch_mid_k(ch.nl, ch.capped, ch.all, (unsigned)grid, flags, m, st) != hipSuccess) return FS_E_HIP;
    used = true;
    return FS_OK;
}

int launch(fs_context* ctx, fs::Args a, int64_t rows, int64_t streams, hipStream_t st, int per_cu = 2) {
    std::lock_guard<std::mutex> g(ctx->mu);
    int rc = device_of(ctx);
    if (rc != FS_OK) return rc;
    int64_t seg_grid = 0;
    rc = grow_fused(ctx, a, rows, streams, per_cu, &seg_grid);
    if (rc != FS_OK) return rc;
    if (capturing(st)) ctx->captured = true;
    a.cand = ctx->cand; a.meta = ctx->meta; a.rhist = ctx->rhist; a.rmass = ctx->rmass;
    a.stream_cnt = ctx->stream_cnt; a.err = ctx->err; a.dirty = ctx->err + 1; a.merge_spins = ctx->merge_spins;
    a.trace = nullptr;
    int done = FS_OK;
    if (gave_up(ctx->hflag)) {
        clear_words(st, ctx->rhist, (int64_t)(ctx->row_cap * fs::RBINS));
        clear_words(st, ctx->rmass, (int64_t)(ctx->row_cap * fs::LB * 2));
        clear_words(st, ctx->stream_cnt, (int64_t)ctx->stream_cap);
        clear_words(st, ctx->err + 1, 1);
        if (hipGetLastError() != hipSuccess) return FS_E_HIP;
        done = FS_W_RECOVERED;
    }
    if (!ctx->seg_layout) {
        rc = launch_alone(a, rows, st);
        return rc != FS_OK ? rc : done;
    }
#ifdef FS_TRACE
    {
        const int64_t grid = seg_grid > 0 ? seg_grid + (int64_t)fs::XCDS * ((rows + fs::XCDS - 1) / fs::XCDS) : rows;
        if (ctx->trace && grid * fs::TRACE_W <= ctx->trace_cap) a.trace = ctx->trace;   // else: untraced
    }
#endif
    rc = launch_planned(a, rows, seg_grid, st);
    return rc != FS_OK ? rc : done;
}

}  // namespace

// ------------------------------------------------------------------------------------------------ static workspace
// fs_sample_batch_static's workspace: one file-scope device array per GPU, held until the process ends, so the
// call allocates nothing. Layout (bytes): error word and dirty flag | meta [ST_SLOTS][2] | row histograms
// [ST_ROWS][RBINS] | large rows' mass histograms [ST_ROWS][LB] | candidate lists [ST_SLOTS][CAP]. The row and mass
// histograms (counters included) must be zero when a call starts; the kernels leave them so, and the first call on a
// device clears them with a fill kernel (no hipMemsetAsync: the call may be recorded into a graph).
constexpr int64_t ST_ROWS = 512;                                  // rows per call
constexpr int64_t ST_SLOTS = 512;                                 // (row, segment) slots per call
constexpr size_t ST_ERR_OFF = 0;                                  // int32 [2]: error bits, dirty
constexpr size_t ST_META_OFF = 256;
constexpr size_t ST_RHIST_OFF = ST_META_OFF + ((ST_SLOTS * 2 * sizeof(uint32_t) + 255) / 256) * 256;
constexpr size_t ST_RMASS_OFF = ST_RHIST_OFF + (size_t)ST_ROWS * fs::RBINS * sizeof(uint32_t);
constexpr size_t ST_CAND_OFF = ST_RMASS_OFF + (size_t)ST_ROWS * fs::LB * sizeof(uint64_t);
constexpr size_t ST_BYTES = ST_CAND_OFF + (size_t)ST_SLOTS * fs::CAP * sizeof(uint64_t);   // 50,336,000 B

static __device__ __align__(256) unsigned char scratch[ST_BYTES];


namespace {

constexpr int ST_MAX_DEVICES = 64;
std::mutex g_static_mu;
unsigned char* g_static_ptr[ST_MAX_DEVICES] = {};   // the device address of `scratch` on each device
int32_t* g_static_flag[ST_MAX_DEVICES] = {};        // host-mapped give-up flag of each device's static workspace

__global__ void store_u64_kernel(uint64_t* p, uint64_t v) { *p = v; }

// The static workspace of the current device: its address from hipGetSymbolAddress (the array's name is not a
// device address in host code), once per device; the first call also zeroes the error words and row histograms
// on `st`, ahead of its own launch.
int static_workspace(int dev, hipStream_t st, unsigned char** out) {
    if (dev < 0 || dev >= ST_MAX_DEVICES) return FS_E_INVALID;
    std::lock_guard<std::mutex> g(g_static_mu);
    if (!g_static_ptr[dev]) {
        void* ptr = nullptr;
        if (hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)) != hipSuccess || !ptr) return FS_E_HIP;
        unsigned char* base = (unsigned char*)ptr;
        int32_t* flag = nullptr;
        int32_t* flag_dev = nullptr;
        if (hipHostMalloc((void**)&flag, sizeof(int32_t), hipHostMallocMapped) != hipSuccess) return FS_E_NOMEM;
        *(volatile int32_t*)flag = 0;
        if (hipHostGetDevicePointer((void**)&flag_dev, flag, 0) != hipSuccess) return FS_E_HIP;
        hipLaunchKernelGGL(fs::zero_words_kernel, dim3(1), dim3(256), 0, st, (uint32_t*)(base + ST_ERR_OFF),
                           (int64_t)(ST_META_OFF / 4));
        // error word 2..3: the give-up flag's device address (a kernel store: the call may be under graph capture)
        hipLaunchKernelGGL(store_u64_kernel, dim3(1), dim3(1), 0, st, (uint64_t*)(base + ST_ERR_OFF + 8),
                           (uint64_t)(uintptr_t)flag_dev);
        g_static_flag[dev] = flag;
        hipLaunchKernelGGL(fs::zero_words_kernel, dim3(1024), dim3(256), 0, st, (uint32_t*)(base + ST_RHIST_OFF),
                           (int64_t)((ST_CAND_OFF - ST_RHIST_OFF) / 4));   // row and mass histograms
        if (hipGetLastError() != hipSuccess) return FS_E_HIP;
        g_static_ptr[dev] = base;
    }
    *out = g_static_ptr[dev];
    return FS_OK;
}

}  // namespace

namespace {

bool aligned16(const void* p) { return ((uintptr_t)p & 15u) == 0; }

int check_rows(const float* d_logits, int64_t ld, int32_t B, int32_t V) {
    if (!d_logits || B < 0 || V < 1 || V > FS_MAX_VOCAB || ld < V || (ld & 3) != 0 || !aligned16(d_logits))
        return FS_E_INVALID;
    return FS_OK;
}

}  // namespace

extern "C" {

int fs_create(fs_context** out) {
    if (!out) return FS_E_INVALID;
    *out = new (std::nothrow) fs_context();
    return *out ? FS_OK : FS_E_NOMEM;
}

int fs_destroy(fs_context* c) {
    if (!c) return FS_E_INVALID;
    (void)hipFree(c->sk_lists);
    (void)hipFree(c->sk_ticket);
    (void)hipFree(c->mk_ctr);
    (void)hipFree(c->mk_list);
    (void)hipFree(c->mk_spill);
    (void)hipFree(c->mk_mass);
    (void)hipFree(c->mk_qk);
    (void)hipFree(c->cand);
    (void)hipFree(c->meta);
    (void)hipFree(c->rhist);
    (void)hipFree(c->rmass);
    (void)hipFree(c->stream_cnt);
    (void)hipFree(c->err);
    (void)hipFree(c->greedy);
    for (void* p : c->retired) (void)hipFree(p);
    if (c->hflag) (void)hipHostFree(c->hflag);
    delete c;
    return FS_OK;
}

int fs_sample_batch(fs_context* ctx, const float* d_logits, int64_t ld, int32_t B, int32_t V, const int32_t* d_hist,
                    const int64_t* d_hist_off, const fs_row_params* d_params, const double* d_u, int32_t* d_tok,
                    int32_t kcap, int32_t* d_cand_ids, double* d_cand_probs, int32_t* d_keep, void* stream) {
    if (!ctx || !d_params || !d_tok || kcap < 0 || ((d_cand_ids || d_cand_probs) && kcap == 0)) return FS_E_INVALID;
    int rc = check_rows(d_logits, ld, B, V);
    if (rc != FS_OK) return rc;
    if (B == 0) return FS_OK;
    fs::Args a = {};
    a.logits = d_logits; a.ld = ld; a.B = B; a.V = V; a.hist = d_hist; a.hist_off = d_hist_off; a.params = d_params;
    a.u = d_u; a.tok = d_tok; a.kcap = kcap; a.cand_ids = d_cand_ids; a.cand_probs = d_cand_probs; a.keep = d_keep;
    a.mode = fs::MODE_SAMPLE; a.eos = -1;
    return launch(ctx, a, B, 0, (hipStream_t)stream);
}

int fs_sample_batch_hp(fs_context* ctx, const float* d_logits, int64_t ld, int32_t B, int32_t V,
                       const int32_t* d_hist, const int64_t* d_hist_off, const fs_row_params* d_params,
                       const fs_row_params* h_params, const double* d_u, int32_t* d_tok, int32_t kcap,
                       int32_t* d_cand_ids, double* d_cand_probs, int32_t* d_keep, void* stream) {
    if (!ctx || !d_params || !d_tok || kcap < 0 || ((d_cand_ids || d_cand_probs) && kcap == 0)) return FS_E_INVALID;
    int rc = check_rows(d_logits, ld, B, V);
    if (rc != FS_OK) return rc;
    if (B == 0) return FS_OK;
    fs::Args a = {};
    a.logits = d_logits; a.ld = ld; a.B = B; a.V = V; a.hist = d_hist; a.hist_off = d_hist_off; a.params = d_params;
    a.u = d_u; a.tok = d_tok; a.kcap = kcap; a.cand_ids = d_cand_ids; a.cand_probs = d_cand_probs; a.keep = d_keep;
    a.mode = fs::MODE_SAMPLE; a.eos = -1;
    if (h_params) {
        bool used = false;
        rc = launch_small(ctx, a, h_params, (hipStream_t)stream, used);
        if (rc != FS_OK || used) return rc;
        const int per_cu = mixed_merges(h_params, B, V) ? 4 : 2;
        rc = launch_mid(ctx, a, h_params, (hipStream_t)stream, used, per_cu);
        if (rc != FS_OK || used) return rc;
        return launch(ctx, a, B, 0, (hipStream_t)stream, per_cu);
    }
    return launch(ctx, a, B, 0, (hipStream_t)stream);
}

int fs_verify_hp(fs_context* ctx, const float* d_logits, int64_t ld, int32_t n_streams, int32_t total_rows, int32_t V,
                 const int32_t* d_rows, const int64_t* d_row_off, const int32_t* d_hist, const int64_t* d_hist_off,
                 const fs_row_params* d_params, const fs_row_params* h_params, const double* d_u, int32_t eos_id,
                 int32_t* d_tok, int32_t* d_accepted, void* stream) {
    if (!ctx || !d_rows || !d_row_off || !d_params || !d_tok || !d_accepted || n_streams < 0 || total_rows < 0)
        return FS_E_INVALID;
    int rc = check_rows(d_logits, ld, total_rows, V);
    if (rc != FS_OK) return rc;
    if (total_rows == 0 || n_streams == 0) return FS_OK;
    fs::Args a = {};
    a.logits = d_logits; a.ld = ld; a.B = total_rows; a.V = V; a.hist = d_hist; a.hist_off = d_hist_off;
    a.params = d_params; a.u = d_u; a.tok = d_tok; a.rows = d_rows; a.row_off = d_row_off; a.n_streams = n_streams;
    a.eos = eos_id; a.accepted = d_accepted; a.mode = fs::MODE_VERIFY;
    if (h_params) {
        bool used = false;
        rc = launch_small(ctx, a, h_params, (hipStream_t)stream, used);
        if (rc != FS_OK || used) return rc;
        rc = launch_mid(ctx, a, h_params, (hipStream_t)stream, used);
        if (rc != FS_OK || used) return rc;
    }
    return launch(ctx, a, total_rows, n_streams, (hipStream_t)stream);
}

int fs_small_k_plan(int32_t cus, int32_t B, int32_t V, int32_t* nl, int32_t* nseg) {
    if (cus < 1 || B < 1 || V < 1 || V > FS_MAX_VOCAB || !nl || !nseg) return FS_E_INVALID;
    int l = 0, n = 0;
    const int rc = small_k_plan(cus, B, V, l, n);
    *nl = l;
    *nseg = n;
    return rc == FS_OK ? FS_OK : FS_E_LIMIT;
}

int fs_route_plan(int32_t cus, const fs_row_params* h_params, int32_t n, int32_t total_rows, int32_t V,
                  int32_t verify, int32_t* kernel, int32_t* nl, int32_t* nseg, int32_t* per_cu) {
    if (cus < 1 || !h_params || n < 1 || total_rows < 1 || V < 1 || V > FS_MAX_VOCAB || !kernel || !nl || !nseg ||
        !per_cu)
        return FS_E_INVALID;
    if (!verify && total_rows != n) return FS_E_INVALID;
    SmallKChoice ch;
    *nl = 0;
    if (small_k_choice(cus, h_params, n, total_rows, V, verify != 0, ch)) {
        *kernel = ch.all_greedy ? 2 : 1;
        *nl = ch.nl;
        *nseg = ch.nseg;
        *per_cu = 0;
        return FS_OK;
    }
    fs::Args a = {};
    a.V = V;
    a.mode = verify ? fs::MODE_VERIFY : fs::MODE_SAMPLE;
    *per_cu = (!verify && mixed_merges(h_params, n, V)) ? 4 : 2;
    int64_t items = 0, seg_grid = 0;
    const int rc = plan(cus, a, total_rows, items, seg_grid, 0, *per_cu);
    if (rc != FS_OK) return rc;
    *kernel = 0;
    *nseg = a.nseg;
    return FS_OK;
}

int fs_mid_k_plan(int32_t cus, const fs_row_params* h_params, int32_t n, int32_t total_rows, int32_t V, int32_t* nl,
                  int32_t* nseg) {
    if (cus < 1 || !h_params || n < 1 || total_rows < 1 || V < 1 || V > FS_MAX_VOCAB || !nl || !nseg) return FS_E_INVALID;
    MidKChoice c;
    const bool fits = mid_k_choice(cus, h_params, n, total_rows, V, false, c);
    *nl = fits ? c.nl : 0;
    *nseg = fits ? c.nseg : 0;
    return fits ? FS_OK : FS_E_LIMIT;
}

int fs_sample_batch_static(fs_context* ctx, const float* d_logits, int64_t ld, int32_t B, int32_t V,
                           const int32_t* d_hist, const int64_t* d_hist_off, const fs_row_params* d_params,
                           const double* d_u, int32_t* d_tok, int32_t kcap, int32_t* d_cand_ids, double* d_cand_probs,
                           int32_t* d_keep, void* stream) {
    if (!ctx || !d_params || !d_tok || kcap < 0 || ((d_cand_ids || d_cand_probs) && kcap == 0)) return FS_E_INVALID;
    int rc = check_rows(d_logits, ld, B, V);
    if (rc != FS_OK) return rc;
    if (B == 0) return FS_OK;
    if (B > ST_ROWS) return FS_E_LIMIT;
    fs::Args a = {};
    a.logits = d_logits; a.ld = ld; a.B = B; a.V = V; a.hist = d_hist; a.hist_off = d_hist_off; a.params = d_params;
    a.u = d_u; a.tok = d_tok; a.kcap = kcap; a.cand_ids = d_cand_ids; a.cand_probs = d_cand_probs; a.keep = d_keep;
    a.mode = fs::MODE_SAMPLE; a.eos = -1;
    const hipStream_t st = (hipStream_t)stream;
    std::lock_guard<std::mutex> g(ctx->mu);
    rc = device_of(ctx);
    if (rc != FS_OK) return rc;
    int dev = -1;
    if (hipGetDevice(&dev) != hipSuccess) return FS_E_HIP;
    if (ctx->static_dev >= 0 && ctx->static_dev != dev) return FS_E_INVALID;   // a context stays on one device
    int64_t items = 0, seg_grid = 0;
    rc = plan(ctx->cus, a, B, items, seg_grid, ST_SLOTS);        // fewer segments per row where the slots run out
    if (rc != FS_OK) return rc;
    if (items > ST_SLOTS) return FS_E_LIMIT;
    unsigned char* base = nullptr;
    rc = static_workspace(dev, st, &base);
    if (rc != FS_OK) return rc;
    ctx->static_dev = dev;
    a.err = (int32_t*)(base + ST_ERR_OFF); a.dirty = a.err + 1;
    a.meta = (uint32_t*)(base + ST_META_OFF);
    a.rhist = (uint32_t*)(base + ST_RHIST_OFF);
    a.rmass = (uint64_t*)(base + ST_RMASS_OFF);
    a.cand = (uint64_t*)(base + ST_CAND_OFF);
    a.stream_cnt = nullptr;                          // sampling mode has no verify streams
    a.merge_spins = ctx->merge_spins;
    int done = FS_OK;
    int32_t* sflag = nullptr;
    {
        std::lock_guard<std::mutex> gs(g_static_mu);
        sflag = g_static_flag[dev];
    }
    if (gave_up(sflag)) {                            // an earlier call on the device gave up: clear what it left
        clear_words(st, base + ST_RHIST_OFF, (int64_t)((ST_CAND_OFF - ST_RHIST_OFF) / 4));
        clear_words(st, a.dirty, 1);
        if (hipGetLastError() != hipSuccess) return FS_E_HIP;
        done = FS_W_RECOVERED;
    }
    rc = ctx->seg_layout ? launch_planned(a, B, seg_grid, st) : launch_alone(a, B, st);
    return rc != FS_OK ? rc : done;
}

int fs_argmax_batch(fs_context* ctx, const float* d_logits, int64_t ld, int32_t B, int32_t V, const int32_t* d_hist,
                    const int64_t* d_hist_off, const fs_row_params* d_params, int32_t* d_tok, void* stream) {
    if (!ctx || !d_tok) return FS_E_INVALID;
    int rc = check_rows(d_logits, ld, B, V);
    if (rc != FS_OK) return rc;
    if (B == 0) return FS_OK;
    fs::Args a = {};
    a.logits = d_logits; a.ld = ld; a.B = B; a.V = V; a.hist = d_hist; a.hist_off = d_params ? d_hist_off : nullptr;
    a.params = d_params; a.tok = d_tok; a.mode = fs::MODE_ARGMAX; a.eos = -1;
    if (!d_params) {
        // no penalties: every row greedy, so the small-k kernel's greedy path takes the batch (its parameters are
        // greedy records the context keeps on the device and the host)
        fs::Args g = a;
        g.mode = fs::MODE_SAMPLE;
        g.hist = nullptr;
        bool used = false;
        rc = launch_small(ctx, g, nullptr, (hipStream_t)stream, used);
        if (rc != FS_OK || used) return rc;
    }
    return launch(ctx, a, B, 0, (hipStream_t)stream);
}

int fs_verify(fs_context* ctx, const float* d_logits, int64_t ld, int32_t n_streams, int32_t total_rows, int32_t V,
              const int32_t* d_rows, const int64_t* d_row_off, const int32_t* d_hist, const int64_t* d_hist_off,
              const fs_row_params* d_params, const double* d_u, int32_t eos_id, int32_t* d_tok, int32_t* d_accepted,
              void* stream) {
    if (!ctx || !d_rows || !d_row_off || !d_params || !d_tok || !d_accepted || n_streams < 0 || total_rows < 0)
        return FS_E_INVALID;
    int rc = check_rows(d_logits, ld, total_rows, V);
    if (rc != FS_OK) return rc;
    if (total_rows == 0 || n_streams == 0) return FS_OK;
    fs::Args a = {};
    a.logits = d_logits; a.ld = ld; a.B = total_rows; a.V = V; a.hist = d_hist; a.hist_off = d_hist_off;
    a.params = d_params; a.u = d_u; a.tok = d_tok; a.rows = d_rows; a.row_off = d_row_off; a.n_streams = n_streams;
    a.eos = eos_id; a.accepted = d_accepted; a.mode = fs::MODE_VERIFY;
    return launch(ctx, a, total_rows, n_streams, (hipStream_t)stream);
}

int fs_penalize_batch(fs_context* ctx, float* d_logits, int64_t ld, int32_t B, int32_t V, const int32_t* d_hist,
                      const int64_t* d_hist_off, const fs_row_params* d_params, void* stream) {
    if (!ctx || !d_params) return FS_E_INVALID;
    int rc = check_rows(d_logits, ld, B, V);
    if (rc != FS_OK) return rc;
    if (B == 0 || !d_hist || !d_hist_off) return FS_OK;
    const int64_t nchunk = ((int64_t)V + fs::PEN_CHUNK - 1) / fs::PEN_CHUNK;
    if ((int64_t)B * nchunk > 0x7fffffff) return FS_E_INVALID;
    {
        std::lock_guard<std::mutex> g(ctx->mu);
        rc = grow(ctx, 0, 0, 0);
        if (rc != FS_OK) return rc;
    }
    hipLaunchKernelGGL(fs::penalize_kernel, dim3((unsigned)(B * nchunk)), dim3(fs::PEN_BLOCK), 0, (hipStream_t)stream,
                       d_logits, ld, V, d_hist, d_hist_off, d_params, (int)nchunk, ctx->err);
    return hipGetLastError() == hipSuccess ? FS_OK : FS_E_HIP;
}

int fs_softcap_batch(const float* d_in, float* d_out, int64_t n, float cap, void* stream) {
    if (n < 0 || (n > 0 && (!d_in || !d_out)) || !(cap > 0.0f)) return FS_E_INVALID;
    if (n == 0) return FS_OK;
    int64_t blocks = (n + 255) / 256;
    if (blocks > 65536) blocks = 65536;
    hipLaunchKernelGGL(fs::softcap_kernel, dim3((unsigned)blocks), dim3(256), 0, (hipStream_t)stream, d_in, d_out, n,
                       cap);
    return hipGetLastError() == hipSuccess ? FS_OK : FS_E_HIP;
}

int fs_lookup_draft(fs_context* ctx, int32_t n_streams, const int32_t* d_hist, const int64_t* d_hist_off,
                    const int32_t* d_kmax, const int32_t* d_min_n, int32_t eos_id, int32_t* d_draft, int32_t draft_ld,
                    int32_t* d_ndraft, void* stream) {
    if (!ctx || n_streams < 0 || !d_hist_off || !d_draft || !d_ndraft || draft_ld < 1) return FS_E_INVALID;
    if (n_streams == 0) return FS_OK;
    return fs::launch_lookup_draft(n_streams, d_hist, d_hist_off, d_kmax, d_min_n, eos_id, d_draft, draft_ld, d_ndraft,
                                   (hipStream_t)stream) == hipSuccess ? FS_OK : FS_E_HIP;
}

int fs_hist_append(fs_context* ctx, int32_t n_streams, const int32_t* d_hist, const int64_t* d_hist_off,
                   const int32_t* d_tok, const int64_t* d_row_off, const int32_t* d_count, int32_t* d_out_hist,
                   int64_t out_cap, int64_t* d_out_hist_off, void* stream) {
    if (!ctx || n_streams < 0 || !d_hist_off || !d_out_hist_off || out_cap < 0) return FS_E_INVALID;
    if (n_streams > 0 && (!d_tok || !d_hist)) return FS_E_INVALID;
    if (out_cap > 0 && !d_out_hist) return FS_E_INVALID;
    if (d_out_hist_off == d_hist_off || (d_out_hist && d_out_hist == d_hist)) return FS_E_INVALID;   // out of place
    {
        std::lock_guard<std::mutex> g(ctx->mu);
        const int rc = grow(ctx, 1, 1, 1);               // the device error word
        if (rc != FS_OK) return rc;
    }
    return fs::launch_hist_append(n_streams, d_hist, d_hist_off, d_tok, d_row_off, d_count, d_out_hist, d_out_hist_off,
                                  out_cap, ctx->err, (hipStream_t)stream) == hipSuccess ? FS_OK : FS_E_HIP;
}

int fs_device_error(fs_context* ctx, void* stream, int32_t* bits) {
    if (!ctx || !bits) return FS_E_INVALID;
    *bits = 0;
    std::lock_guard<std::mutex> g(ctx->mu);
    if (!ctx->err && ctx->static_dev < 0) return FS_OK;
    if (hipStreamSynchronize((hipStream_t)stream) != hipSuccess) return FS_E_HIP;
    if (ctx->err) {
        int32_t h[2] = {0, 0};
        if (hipMemcpy(h, ctx->err, sizeof(h), hipMemcpyDeviceToHost) != hipSuccess) return FS_E_HIP;
        *bits |= h[0];
        if (h[1] != 0) {
            // a merge gave up: the segments it did not wait for have finished by now (the stream is idle), so the
            // row histograms and counters are cleared and the context leaves its compute-alone mode
            if (ctx->rhist && hipMemset(ctx->rhist, 0, ctx->row_cap * fs::RBINS * sizeof(uint32_t)) != hipSuccess)
                return FS_E_HIP;
            if (ctx->rmass && hipMemset(ctx->rmass, 0, ctx->row_cap * fs::LB * sizeof(uint64_t)) != hipSuccess)
                return FS_E_HIP;
            if (ctx->stream_cnt && hipMemset(ctx->stream_cnt, 0, ctx->stream_cap * sizeof(uint32_t)) != hipSuccess)
                return FS_E_HIP;
        }
        if (hipMemset(ctx->err, 0, sizeof(h)) != hipSuccess) return FS_E_HIP;
    }
    if (ctx->static_dev >= 0) {
        // the device's static workspace (fs_sample_batch_static), shared by every context on the device
        unsigned char* base = nullptr;
        {
            std::lock_guard<std::mutex> gs(g_static_mu);
            base = g_static_ptr[ctx->static_dev];
        }
        if (base) {
            int32_t h[2] = {0, 0};
            if (hipMemcpy(h, base + ST_ERR_OFF, sizeof(h), hipMemcpyDeviceToHost) != hipSuccess) return FS_E_HIP;
            *bits |= h[0];
            if (h[1] != 0 && hipMemset(base + ST_RHIST_OFF, 0, ST_CAND_OFF - ST_RHIST_OFF) != hipSuccess)
                return FS_E_HIP;
            if (hipMemset(base + ST_ERR_OFF, 0, sizeof(h)) != hipSuccess) return FS_E_HIP;
        }
    }
    return FS_OK;
}

int fs_plan_layout(int32_t cus, int32_t xccs, int32_t B, int32_t V, int32_t static_ws, int32_t* nseg,
                   int32_t* seg_tiles, int64_t* slots) {
    if (cus < 1 || xccs < 0 || B < 1 || V < 1 || V > FS_MAX_VOCAB || !nseg || !seg_tiles || !slots) return FS_E_INVALID;
    if (static_ws && B > ST_ROWS) return FS_E_LIMIT;
    *nseg = 0; *seg_tiles = 0; *slots = 0;
    if (!layout_fits(xccs)) return FS_OK;                 // every row sampled alone by one workgroup
    fs::Args a = {};
    a.B = B; a.V = V; a.mode = fs::MODE_SAMPLE;
    int64_t items = 0, seg_grid = 0;
    const int rc = plan(cus, a, B, items, seg_grid, static_ws ? ST_SLOTS : 0);
    if (rc != FS_OK) return rc;
    if (static_ws && items > ST_SLOTS) return FS_E_LIMIT;
    *nseg = a.nseg; *seg_tiles = a.seg_tiles; *slots = items;
    return FS_OK;
}

int fs_error_word(fs_context* ctx, const int32_t** d_bits) {
    if (!ctx || !d_bits) return FS_E_INVALID;
    std::lock_guard<std::mutex> g(ctx->mu);
    const int rc = grow(ctx, 0, 0, 0);
    if (rc != FS_OK) return rc;
    *d_bits = ctx->err;
    return FS_OK;
}

int fs_set_wait_limit(fs_context* ctx, uint32_t polls) {
    if (!ctx) return FS_E_INVALID;
    std::lock_guard<std::mutex> g(ctx->mu);
    ctx->merge_spins = polls == FS_WAIT_GIVE_UP ? 0u : (polls ? polls : fs::MERGE_SPINS);
    return FS_OK;
}

// Per-stream draw source of ferro::Sampler (sampler.h:25,32 and the draw at sampler.cpp:45-46): the same libstdc++
// engine and canonical mapping, so u * tot equals uniform_real_distribution<double>(0, tot)(rng) bit for bit.
struct fs_rng {
    std::mt19937_64 eng;
};

int fs_rng_create(uint64_t seed, fs_rng** out) {
    if (!out) return FS_E_INVALID;
    *out = new (std::nothrow) fs_rng();
    if (!*out) return FS_E_NOMEM;
    (*out)->eng.seed(seed ? seed : (uint64_t)std::random_device{}());
    return FS_OK;
}

int fs_rng_destroy(fs_rng* r) {
    if (!r) return FS_E_INVALID;
    delete r;
    return FS_OK;
}

int fs_rng_next_u(fs_rng* r, double* u, int32_t n) {
    if (!r || !u || n < 0) return FS_E_INVALID;
    for (int32_t i = 0; i < n; ++i) u[i] = std::generate_canonical<double, 53>(r->eng);
    return FS_OK;
}

int fs_rng_copy(const fs_rng* src, fs_rng* dst) {
    if (!src || !dst) return FS_E_INVALID;
    dst->eng = src->eng;
    return FS_OK;
}

// Device draw streams (see fs::drng_draw_kernel): the engines' states live in device memory; seeding follows the
// standard's seed sequence for mt19937_64 (x0 = seed, x_i = 6364136223846793005 * (x_{i-1} ^ (x_{i-1} >> 62)) + i),
// so stream s reproduces std::mt19937_64(seed_s) and ferro::Sampler's draws.
struct fs_drng {
    int device = -1;
    int n = 0;
    uint64_t* mt = nullptr;     // [n][312]
    int32_t* idx = nullptr;     // [n]
    int32_t* err = nullptr;
};

// fs_decode_step: fs_sample_batch with the draws taken from the device streams r (row s = stream s) and each row's
// token appended to its stream's history out of place, in the sampling grid itself (one launch).
int fs_decode_step_hp(fs_context* ctx, fs_drng* r, const float* d_logits, int64_t ld, int32_t B, int32_t V,
                      const int32_t* d_hist, const int64_t* d_hist_off, const fs_row_params* d_params,
                      const fs_row_params* h_params, int32_t* d_tok, int32_t* d_keep, int32_t* d_out_hist,
                      int64_t* d_out_hist_off, int64_t out_cap, void* stream) {
    if (!ctx || !r || !d_params || !d_tok || !d_out_hist_off || out_cap < 0 || (out_cap > 0 && !d_out_hist) ||
        (d_hist == nullptr) != (d_hist_off == nullptr) || B > r->n)
        return FS_E_INVALID;
    int rc = check_rows(d_logits, ld, B, V);
    if (rc != FS_OK) return rc;
    int dev = -1;
    if (hipGetDevice(&dev) != hipSuccess) return FS_E_HIP;
    if (dev != r->device) return FS_E_INVALID;
    if (B == 0) return FS_OK;
    fs::Args a = {};
    a.logits = d_logits; a.ld = ld; a.B = B; a.V = V; a.hist = d_hist; a.hist_off = d_hist_off; a.params = d_params;
    a.u = nullptr; a.tok = d_tok; a.kcap = 0; a.keep = d_keep;
    a.mode = fs::MODE_SAMPLE; a.eos = -1;
    a.dmt = r->mt; a.didx = r->idx; a.out_hist = d_out_hist; a.out_hist_off = d_out_hist_off; a.out_cap = out_cap;
    if (h_params) {
        bool used = false;
        rc = launch_small(ctx, a, h_params, (hipStream_t)stream, used);
        if (rc != FS_OK || used) return rc;
        rc = launch_mid(ctx, a, h_params, (hipStream_t)stream, used);
        if (rc != FS_OK || used) return rc;
    }
    return launch(ctx, a, B, 0, (hipStream_t)stream);
}

int fs_decode_step(fs_context* ctx, fs_drng* r, const float* d_logits, int64_t ld, int32_t B, int32_t V,
                   const int32_t* d_hist, const int64_t* d_hist_off, const fs_row_params* d_params, int32_t* d_tok,
                   int32_t* d_keep, int32_t* d_out_hist, int64_t* d_out_hist_off, int64_t out_cap, void* stream) {
    return fs_decode_step_hp(ctx, r, d_logits, ld, B, V, d_hist, d_hist_off, d_params, nullptr, d_tok, d_keep,
                             d_out_hist, d_out_hist_off, out_cap, stream);
}

int fs_drng_create(int32_t n_streams, const uint64_t* seeds, void* stream, fs_drng** out) {
    if (!out || n_streams < 1 || !seeds) return FS_E_INVALID;
    *out = nullptr;
    fs_drng* r = new (std::nothrow) fs_drng();
    if (!r) return FS_E_NOMEM;
    std::vector<uint64_t> mt((size_t)n_streams * fs::MT_N);
    std::vector<int32_t> idx((size_t)n_streams, fs::MT_N);
    std::random_device rd;
    for (int32_t s = 0; s < n_streams; ++s) {
        uint64_t* x = mt.data() + (size_t)s * fs::MT_N;
        x[0] = seeds[s] ? seeds[s] : (uint64_t)rd();                     // seed 0 = random, as ferro
        for (int i = 1; i < fs::MT_N; ++i) x[i] = 6364136223846793005ull * (x[i - 1] ^ (x[i - 1] >> 62)) + (uint64_t)i;
    }
    r->n = n_streams;
    int rc = FS_OK;
    if (hipGetDevice(&r->device) != hipSuccess) rc = FS_E_HIP;
    if (rc == FS_OK && (hipMalloc(&r->mt, mt.size() * sizeof(uint64_t)) != hipSuccess ||
                        hipMalloc(&r->idx, idx.size() * sizeof(int32_t)) != hipSuccess ||
                        hipMalloc(&r->err, sizeof(int32_t)) != hipSuccess))
        rc = FS_E_NOMEM;
    hipStream_t st = (hipStream_t)stream;
    if (rc == FS_OK && (hipMemcpyAsync(r->mt, mt.data(), mt.size() * sizeof(uint64_t), hipMemcpyHostToDevice, st) != hipSuccess ||
                        hipMemcpyAsync(r->idx, idx.data(), idx.size() * sizeof(int32_t), hipMemcpyHostToDevice, st) != hipSuccess ||
                        hipMemsetAsync(r->err, 0, sizeof(int32_t), st) != hipSuccess ||
                        hipStreamSynchronize(st) != hipSuccess))
        rc = FS_E_HIP;
    if (rc != FS_OK) { fs_drng_destroy(r); return rc; }
    *out = r;
    return FS_OK;
}

int fs_drng_destroy(fs_drng* r) {
    if (!r) return FS_E_INVALID;
    (void)hipFree(r->mt);
    (void)hipFree(r->idx);
    (void)hipFree(r->err);
    delete r;
    return FS_OK;
}

int fs_drng_draw(fs_drng* r, const int64_t* d_row_off, const fs_row_params* d_params, double* d_u, int32_t peek,
                 void* stream) {
    if (!r || !d_params || !d_u) return FS_E_INVALID;
    hipLaunchKernelGGL(fs::drng_draw_kernel, dim3((unsigned)((r->n + 63) / 64)), dim3(64), 0, (hipStream_t)stream,
                       r->mt, r->idx, r->n, d_row_off, d_params, d_u, peek ? 1 : 0, r->err);
    return hipGetLastError() == hipSuccess ? FS_OK : FS_E_HIP;
}

int fs_drng_skip(fs_drng* r, const int32_t* d_counts, const fs_row_params* d_params, void* stream) {
    if (!r || !d_counts || !d_params) return FS_E_INVALID;
    hipLaunchKernelGGL(fs::drng_skip_kernel, dim3((unsigned)((r->n + 63) / 64)), dim3(64), 0, (hipStream_t)stream,
                       r->mt, r->idx, r->n, d_counts, d_params);
    return hipGetLastError() == hipSuccess ? FS_OK : FS_E_HIP;
}

int fs_drng_error(fs_drng* r, void* stream, int32_t* bits) {
    if (!r || !bits) return FS_E_INVALID;
    if (hipStreamSynchronize((hipStream_t)stream) != hipSuccess) return FS_E_HIP;
    if (hipMemcpy(bits, r->err, sizeof(int32_t), hipMemcpyDeviceToHost) != hipSuccess) return FS_E_HIP;
    if (hipMemset(r->err, 0, sizeof(int32_t)) != hipSuccess) return FS_E_HIP;
    return FS_OK;
}

#ifdef FS_TRACE
// Trace builds only (not in the product library): phase timestamps of the next sampling grids into d_buf (cap
// entries, TRACE_W per workgroup); a grid larger than the buffer runs untraced.
int fs_trace_set(fs_context* ctx, uint64_t* d_buf, int64_t cap) {
    if (!ctx || cap < 0) return FS_E_INVALID;
    std::lock_guard<std::mutex> g(ctx->mu);
    ctx->trace = d_buf;
    ctx->trace_cap = d_buf ? cap : 0;
    return FS_OK;
}
#endif

const char* fs_strerror(int code) {
    switch (code) {
        case FS_OK: return "ok";
        case FS_E_INVALID: return "invalid argument";
        case FS_E_HIP: return "HIP runtime error";
        case FS_E_NOMEM: return "device allocation failed";
        case FS_E_DEVICE: return "device-side error";
        case FS_E_LIMIT: return "batch exceeds the static workspace of fs_sample_batch_static";
        case FS_W_RECOVERED: return "ok; an earlier call's merge gave up waiting and this call cleared its workspace";
        default: return "unknown error";
    }
}

}  // extern "C"

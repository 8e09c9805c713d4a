// batch.hip -- many requests of uneven length, window size and overlap in one
// launch sequence: one launch per window-size class present over that class's
// tile queue (tiles of G frames of one request), either one workgroup per tile
// or a persistent grid pulling tiles from a device-side counter.  The launch
// form, the workgroup shape (G) and the radix plan of each class are measured
// by the autotuner.
//
// The requests' records are built on the host in pinned memory; a small kernel
// ahead of the launches copies them to the descriptor block and writes the tile
// -> request table there.  (With an upload of records and table by a copy in
// the stream, the GPU stood idle 35-50 us between two batches: 9 before the
// copy, 9 for 200 KB, 17-33 after it.)  The launches are made one by one: replaying
// them from a captured graph with a node for each of the ten window sizes took
// longer for both mixes measured, 58 against 35 us a batch of 24 requests of three
// sizes, 280 against 257-274 us one of 256 requests of ten.
//
// Requests of windows >= 2^16 (one kernel or two passes) and requests of the matrix-core
// form run after the tile-queue launches, one request at a time, on the same
// stream.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <chrono>
#include <cstring>
#include <map>
#include <string>
#include <utility>
#include <vector>

#include "batch.hpp"
#include "capture.hpp"
#include "multipass.hpp"
#include "side_stream.hpp"

namespace ostft {

namespace {

constexpr int LOG_M_MIN = 5, LOG_M_MAX = 14, NCLS = LOG_M_MAX - LOG_M_MIN + 1;
constexpr size_t ALIGN = 256;
// Batches of so many window sizes and tiles, and so many tiles a request, use two
// streams: the last tiles of one class leave the GPU to the other stream's.
// One / two streams, requests of ten to sixty million samples in all, power.
//   Sizes (calls from C, in a row; each waited for), 60 requests, 31000 tiles, 50%:
//   two 264 / 265 and 274 / 293 us, three 284 / 278 and 293 / 304, four 298 / 290
//   and 307 / 313, five 293 / 282 and 303 / 305; 256 requests, 33000 tiles, 60%: five
//   310 / 295 and 326 / 325, six 326 / 309 and 357 / 340, eight 343 / 307 and 374 / 339.
//   Tiles a request: while the host, at 0.9 us a request from Python, is the slower
//   side, the fork and join cost it 60-100 us.  Six sizes, 60%, 400 requests of 91
//   tiles 393 / 475, 111 459 / 486, 131 528 / 514, 182 698 / 679; 1024 of 90 927 / 1075,
//   110 1099 / 1118, 130 1278 / 1261.
//   Tiles: the same for few requests, 64 of 101 tiles 106 / 131; 256 of 111 301 / 327,
//   of 132 364 / 343 (from C two streams win from 5000 tiles on).
constexpr int SIDE_SIZES = 5;
constexpr uint64_t SIDE_TILES = 32768, SIDE_TILES_PER_REQUEST = 128;
// captured batches keep so many blocks, and so many bytes of them, with the
// context; beyond that a captured batch is a launch per request, which keeps nothing
constexpr size_t HELD_BATCHES = 256, HELD_BYTES = (size_t)64 << 20;

size_t align_up(size_t x) { return (x + ALIGN - 1) & ~(ALIGN - 1); }

// A request as the host writes it.
struct BatchUpload {
    BatchJob job;
    uint64_t tiles_at;  // its first entry of the block's tile table
    uint32_t ntiles;
    uint32_t index;     // its place in its class
};
static_assert(sizeof(BatchJob) % 8 == 0 && sizeof(BatchUpload) % 8 == 0, "copied by 8-byte words");

// One descriptor block (claim counters, BatchJob records, tile table), the
// pinned records it is filled from, and the event after the last launch that
// reads it (both are reused only after it).  A captured batch's block and
// records are its own: every replay reads them.
struct Slot {
    char* d = nullptr;
    size_t d_cap = 0;
    BatchUpload* h = nullptr;
    size_t h_cap = 0;  // records
    hipEvent_t done = nullptr;
    bool used = false;
};

}  // namespace

struct BatchState {
    Slot slot[2];
    int next = 0;
    std::vector<Slot> held;  // of captured batches
    size_t held_bytes = 0;
    bool use_graphs = true;  // batch_config's; off: a batch of any number of sizes may be captured
    int cu_count = 0;
    int persistent[NCLS] = {};  // 1: persistent grid claiming tiles; 0: one workgroup per tile
    int per_cu[NCLS] = {};      // persistent workgroups per CU; 0: the occupancy limit
    int shape[NCLS] = {};       // workgroup shape (engine variant / 4); persistent needs 0
    int plan_override[NCLS];    // >= 0: radix plan for this class instead of the context's (autotuning)
    int variant[NCLS] = {};     // engine variant of each class in the current batch
    SideStreams sides;
    BatchClassInfo info[NCLS][FUSED_VARIANTS] = {};
    bool info_ok[NCLS][FUSED_VARIANTS] = {};

    BatchState()
    {
        for (int& p : plan_override)
            p = -1;
    }
};

namespace {

int state(ostft_ctx* ctx, BatchState** out)
{
    BatchState*& b = ctx_batch(ctx);
    if (!b) {
        BatchState* s = new BatchState();
        hipDeviceProp_t prop;
        hipError_t e = hipGetDeviceProperties(&prop, ctx_device(ctx));
        for (int i = 0; e == hipSuccess && i < 2; ++i)
            e = hipEventCreateWithFlags(&s->slot[i].done, hipEventDisableTiming);
        if (e != hipSuccess) {
            for (auto& sl : s->slot)
                if (sl.done)
                    (void)hipEventDestroy(sl.done);
            delete s;
            return ctx_hip_fail(ctx, e, "batch state");
        }
        s->cu_count = prop.multiProcessorCount;
        b = s;
    }
    *out = b;
    return OSTFT_OK;
}

int class_info(ostft_ctx* ctx, BatchState* st, int c, int v)
{
    if (!st->info_ok[c][v]) {
        const hipError_t e = batch_class_info(c + LOG_M_MIN, v, &st->info[c][v]);
        if (e != hipSuccess)
            return ctx_hip_fail(ctx, e, "batch kernel occupancy");
        if (st->info[c][v].max_blocks_per_cu < 1)
            return ctx_fail(ctx, OSTFT_ERR_HIP, "batch kernel does not fit on a CU");
        st->info_ok[c][v] = true;
    }
    return OSTFT_OK;
}

// Engine variant of class c: its workgroup shape with radix plan `plan`, or
// the default shape where that pair is not built.
int class_variant(const BatchState* st, int c, int plan)
{
    const int v = st->shape[c] * 4 + plan;
    return fused_variant_ok(c + LOG_M_MIN, v) ? v : plan;
}

// Grid of class c for a batch with `ntiles` tiles of it.
uint32_t class_grid(const BatchState* st, int c, uint64_t ntiles)
{
    if (!st->persistent[c])
        return (uint32_t)std::max<uint64_t>(ntiles, 1);
    const int mx = st->info[c][st->variant[c]].max_blocks_per_cu;
    const int pc = st->per_cu[c] > 0 ? std::min(st->per_cu[c], mx) : mx;
    return (uint32_t)pc * (uint32_t)st->cu_count;
}

// Workgroup (j, y) of `parts` per request: part y of request j's entries of the
// tile table, and its record.
constexpr int FILL_THREADS = 256;
__global__ void __launch_bounds__(FILL_THREADS)
    stft_batch_table_kernel(const BatchUpload* __restrict__ up, BatchJob* __restrict__ jobs,
                            uint32_t* __restrict__ tiles, uint32_t* __restrict__ counters)
{
    const uint32_t j = blockIdx.x, tid = threadIdx.x;
    const BatchUpload* u = up + j;
    const uint64_t at = u->tiles_at;
    const uint32_t n = u->ntiles, index = u->index;
    if (blockIdx.y == 0 && tid < sizeof(BatchJob) / 8)
        reinterpret_cast<uint64_t*>(jobs + j)[tid] = reinterpret_cast<const uint64_t*>(&u->job)[tid];
    if (j == 0 && blockIdx.y == 0 && tid < NCLS)
        counters[tid] = 0;
    for (uint64_t i = blockIdx.y * FILL_THREADS + tid; i < n; i += (uint64_t)gridDim.y * FILL_THREADS)
        tiles[at + i] = index;
}

hipError_t ensure_block(Slot& sl, size_t d_bytes)
{
    if (sl.d_cap >= d_bytes)
        return hipSuccess;
    if (sl.d)
        (void)hipFree(sl.d);
    sl.d_cap = 0;
    const hipError_t e = hipMalloc(&sl.d, d_bytes);
    if (e == hipSuccess)
        sl.d_cap = d_bytes;
    else
        sl.d = nullptr;
    return e;
}

hipError_t ensure_records(Slot& sl, size_t records)
{
    if (sl.h_cap >= records)
        return hipSuccess;
    if (sl.h)
        (void)hipHostFree(sl.h);
    sl.h_cap = 0;
    const hipError_t e = hipHostMalloc(&sl.h, records * sizeof(BatchUpload), hipHostMallocDefault);
    if (e == hipSuccess)
        sl.h_cap = records;
    else
        sl.h = nullptr;
    return e;
}

void free_slot(Slot& sl)
{
    if (sl.d)
        (void)hipFree(sl.d);
    if (sl.h)
        (void)hipHostFree(sl.h);
    if (sl.done)
        (void)hipEventDestroy(sl.done);
    sl = Slot{};
}

// The next of the two blocks that batches take in turn, once the GPU is done with it.
int next_slot(ostft_ctx* ctx, BatchState* st, size_t d_bytes, size_t records, Slot** out)
{
    Slot& sl = st->slot[st->next];
    st->next ^= 1;
    if (sl.used) {
        const hipError_t e = hipEventSynchronize(sl.done);
        if (e != hipSuccess)
            return ctx_hip_fail(ctx, e, "batch slot wait");
    }
    hipError_t e = hipSuccess;
    if (sl.d_cap < d_bytes)
        e = ensure_block(sl, std::max<size_t>(align_up(d_bytes + d_bytes / 2), 64 * 1024));
    if (e == hipSuccess && sl.h_cap < records)
        e = ensure_records(sl, std::max<size_t>(records + records / 2, 256));
    if (e != hipSuccess)
        return ctx_hip_fail(ctx, e, "batch descriptor block");
    *out = &sl;
    return OSTFT_OK;
}

// A captured batch's own block; null beyond the bound or without memory for it.
Slot* held_slot(BatchState* st, size_t d_bytes, size_t records)
{
    const size_t bytes = d_bytes + records * sizeof(BatchUpload);
    if (st->held.size() >= HELD_BATCHES || st->held_bytes + bytes > HELD_BYTES)
        return nullptr;
    const AllocateInCapture allow(true);
    Slot sl;
    hipError_t e = ensure_block(sl, d_bytes);
    if (e == hipSuccess)
        e = ensure_records(sl, records);
    if (e != hipSuccess) {
        (void)hipGetLastError();
        free_slot(sl);
        return nullptr;
    }
    st->held_bytes += bytes;
    st->held.push_back(sl);
    return &st->held.back();
}

}  // namespace

int run_batch(ostft_ctx* ctx, const ostft_job* jobs, uint32_t njobs, hipStream_t s)
{
    BatchState* st = nullptr;
    int rc = state(ctx, &st);
    if (rc != OSTFT_OK)
        return rc;
    // 1. validate every request first: a bad request fails the whole call
    //    before anything is launched
    std::vector<FusedArgs> args(njobs);
    std::vector<int> lm(njobs, 0);
    for (uint32_t i = 0; i < njobs; ++i) {
        const ostft_job& j = jobs[i];
        rc = ctx_prepare(ctx, &j.params, j.in, j.full_size, j.out, j.out_cap, &args[i], &lm[i]);
        if (rc != OSTFT_OK)
            return ctx_fail(ctx, rc, "job " + std::to_string(i) + ": " + ostft_last_error(ctx));
    }
    // 2. group by class; tiles per request
    std::vector<uint32_t> members[NCLS];
    uint64_t ntiles[NCLS] = {};
    std::vector<uint32_t> large, mfma;
    uint32_t mask = 0;
    int plan[NCLS];  // radix plan of each class: the context's, read once per class per batch
    for (int c = 0; c < NCLS; ++c)
        plan[c] = -1;
    for (uint32_t i = 0; i < njobs; ++i) {
        if (args[i].frames == 0)
            continue;
        if (!fused_supported(lm[i])) {
            large.push_back(i);
            continue;
        }
        if (jobs[i].params.flags & (OSTFT_FLAG_MFMA_FP16 | OSTFT_FLAG_MFMA_BF16)) {
            // the matrix-core form has no tile-queue kernel: such a request
            // runs on its own launch after the queues, with the one-request
            // kernel (the same result as ostft_run_device)
            mfma.push_back(i);
            continue;
        }
        const int c = lm[i] - LOG_M_MIN;
        if (plan[c] < 0) {
            plan[c] = st->plan_override[c] >= 0 ? st->plan_override[c] : args[i].plan;
            if (!fused_plan_ok(lm[i], plan[c]))
                plan[c] = 0;
            st->variant[c] = class_variant(st, c, plan[c]);
            if (!fused_variant_ok(lm[i], st->variant[c]))
                return ctx_fail(ctx, OSTFT_ERR_INVALID_ARG, "batch variant not built");
            rc = class_info(ctx, st, c, st->variant[c]);
            if (rc != OSTFT_OK)
                return rc;
        }
        // every request of a class runs the class's plan, in tiles of the
        // variant's workgroup
        args[i].plan = plan[c];
        args[i].tile_frames = (int32_t)fused_tile_frames(
            (uint64_t)st->info[c][st->variant[c]].frames_per_tile, 2ull << lm[i], args[i].hop);
        const uint64_t G = (uint64_t)args[i].tile_frames;
        members[c].push_back(i);
        ntiles[c] += (args[i].frames + G - 1) / G;
        mask |= 1u << c;
    }
    for (int c = 0; c < NCLS; ++c)
        if (ntiles[c] >= 0x7fffffffull - 2ull * (uint64_t)st->cu_count * 64u)  // grid limit; claims overrun by <= 2/workgroup
            return ctx_fail(ctx, OSTFT_ERR_TOO_LARGE, "more than 2^31 tiles of one window size in a batch");
    const Capture capture = mask ? capture_of(s) : Capture{};
    if (capture.on && st->use_graphs && __builtin_popcount(mask) >= 3)
        return ctx_fail(ctx, OSTFT_ERR_UNSUPPORTED, "a batch of three or more window sizes cannot be captured");
    // 3. descriptor block: claim counters, requests class by class, tile tables
    //    class by class
    size_t nreq = 0;
    uint64_t total = 0, most = 0;
    size_t first_job[NCLS] = {};
    uint64_t first_tile[NCLS] = {};
    for (int c = 0; c < NCLS; ++c) {
        first_job[c] = nreq;
        first_tile[c] = total;
        nreq += members[c].size();
        total += ntiles[c];
    }
    const size_t jobs_off = align_up(sizeof(uint32_t) * NCLS);
    const size_t tiles_off = align_up(jobs_off + sizeof(BatchJob) * nreq);
    const size_t d_bytes = tiles_off + sizeof(uint32_t) * total;
    Slot* slot = nullptr;
    std::vector<uint32_t> single;  // requests with a launch each, their arguments in it
    if (capture.on) {
        slot = held_slot(st, d_bytes, nreq);
        for (int c = 0; !slot && c < NCLS; ++c)
            single.insert(single.end(), members[c].begin(), members[c].end());
        mask = slot ? mask : 0;
    } else if (mask && (rc = next_slot(ctx, st, d_bytes, nreq, &slot)) != OSTFT_OK) {
        return rc;
    }
    if (mask) {
        Slot& sl = *slot;
        // 4. the requests' records
        for (int c = 0; c < NCLS; ++c) {
            uint64_t t = 0;
            for (size_t k = 0; k < members[c].size(); ++k) {
                BatchUpload& u = sl.h[first_job[c] + k];
                u.job.a = args[members[c][k]];
                u.job.tile_begin = t;
                const uint64_t nt = (u.job.a.frames + u.job.a.tile_frames - 1) / u.job.a.tile_frames;
                u.tiles_at = first_tile[c] + t;
                u.ntiles = (uint32_t)nt;
                u.index = (uint32_t)k;
                t += nt;
                most = std::max(most, nt);
            }
        }
        // 5. the descriptor block, then the launches
        uint32_t* const counters = reinterpret_cast<uint32_t*>(sl.d);
        BatchJob* const bj = reinterpret_cast<BatchJob*>(sl.d + jobs_off);
        uint32_t* const tj = reinterpret_cast<uint32_t*>(sl.d + tiles_off);
        const uint32_t parts = (uint32_t)std::min<uint64_t>(1 + most / (16 * FILL_THREADS), 256);
        hipLaunchKernelGGL(stft_batch_table_kernel, dim3((uint32_t)nreq, parts), dim3(FILL_THREADS), 0, s, sl.h, bj,
                           tj, counters);
        hipError_t e = hipGetLastError();
        // A large batch runs its classes on two streams in turn.  256 mixed requests
        // (47762 tiles of six classes): 470 -> 441 us (454 with each class on the
        // stream with fewer tiles so far)
        const bool two = total >= SIDE_TILES && total >= SIDE_TILES_PER_REQUEST * nreq &&
                         __builtin_popcount(mask) >= SIDE_SIZES;
        SideStream* const other = two ? &st->sides.of(capture) : nullptr;
        if (e == hipSuccess && other)
            e = other->fork(s);
        const bool forked = e == hipSuccess && other;
        int turn = 0;
        for (int c = 0; e == hipSuccess && c < NCLS; ++c) {
            if (!(mask >> c & 1u))
                continue;
            const bool side = other && (turn++ & 1);
            BatchClassArgs a;
            a.jobs = bj + first_job[c];
            a.tile_job = tj + first_tile[c];
            a.counter = counters + c;
            a.ntiles = (uint32_t)ntiles[c];
            e = launch_batch(c + LOG_M_MIN, st->variant[c], a, class_grid(st, c, ntiles[c]), st->persistent[c] != 0,
                             side ? other->stream : s);
        }
        if (forked) {  // also after a failed launch: what follows on s comes after the side stream's work
            const hipError_t j = other->join(s);
            e = e == hipSuccess ? j : e;
        }
        if (!capture.on) {  // also after a failed launch: what was queued may still read this slot
            const hipError_t r = hipEventRecord(sl.done, s);
            sl.used = sl.used || r == hipSuccess;
            e = e == hipSuccess ? r : e;
        }
        if (e != hipSuccess)
            return ctx_hip_fail(ctx, e, "batch launch");
    }
    for (uint32_t i : single) {
        FusedArgs& a = args[i];
        a.tile_frames = (int32_t)fused_tile_frames((uint64_t)fused_variant_frames(lm[i], a.plan), 2ull << lm[i], a.hop);
        const hipError_t e = launch_fused(lm[i], XF_FP32, a, 1, s);
        if (e != hipSuccess)
            return ctx_hip_fail(ctx, e, "batch launch");
    }
    for (uint32_t i : mfma) {
        const int xf = (jobs[i].params.flags & OSTFT_FLAG_MFMA_FP16) ? XF_MFMA_FP16 : XF_MFMA_BF16;
        const hipError_t e = launch_fused(lm[i], xf, args[i], 1, s);
        if (e != hipSuccess)
            return ctx_hip_fail(ctx, e, "batch MFMA launch");
    }
    for (uint32_t i : large) {
        rc = wide_supported(lm[i]) ? run_wide(ctx, lm[i], args[i], s) : run_multipass(ctx, lm[i], args[i], s);
        if (rc != OSTFT_OK)
            return rc;
    }
    return OSTFT_OK;
}

namespace {

constexpr float AUTOTUNE_MARGIN = 0.02f;

int class_of(ostft_ctx* ctx, int exp, int* c)
{
    *c = exp - 1 - LOG_M_MIN;
    if (*c < 0 || *c >= NCLS)
        return ctx_fail(ctx, OSTFT_ERR_UNSUPPORTED, "the batch kernels cover window exponents 6..15");
    return OSTFT_OK;
}

}  // namespace

int batch_config(ostft_ctx* ctx, int exp, int blocks_per_cu, int use_graphs, int* current)
{
    BatchState* st = nullptr;
    int rc = state(ctx, &st);
    if (rc != OSTFT_OK)
        return rc;
    if (use_graphs >= 0)
        st->use_graphs = use_graphs != 0;
    if (exp == 0)
        return OSTFT_OK;
    int c = 0;
    rc = class_of(ctx, exp, &c);
    if (rc != OSTFT_OK)
        return rc;
    if (blocks_per_cu > 0) {
        const int v = ctx_radix_plan(ctx, c + LOG_M_MIN);  // shape 0
        rc = class_info(ctx, st, c, v);
        if (rc != OSTFT_OK)
            return rc;
        st->shape[c] = 0;
        st->persistent[c] = 1;
        st->per_cu[c] = std::min(blocks_per_cu, st->info[c][v].max_blocks_per_cu);
    } else if (blocks_per_cu < 0) {
        st->persistent[c] = 0;
    }
    if (current) {
        int pc = 0;
        if (st->persistent[c]) {
            const int v = ctx_radix_plan(ctx, c + LOG_M_MIN);
            rc = class_info(ctx, st, c, v);
            if (rc != OSTFT_OK)
                return rc;
            const int mx = st->info[c][v].max_blocks_per_cu;
            pc = st->per_cu[c] > 0 ? std::min(st->per_cu[c], mx) : mx;
        }
        *current = pc;
    }
    return OSTFT_OK;
}

int engine_variant(ostft_ctx* ctx, int exp, int shape, int plan, int* cur_shape, int* cur_plan)
{
    BatchState* st = nullptr;
    int rc = state(ctx, &st);
    if (rc != OSTFT_OK)
        return rc;
    int c = 0;
    rc = class_of(ctx, exp, &c);
    if (rc != OSTFT_OK)
        return rc;
    const int log_m = c + LOG_M_MIN;
    if (plan >= 0 && !fused_plan_ok(log_m, plan))
        return ctx_fail(ctx, OSTFT_ERR_UNSUPPORTED, "radix plan " + std::to_string(plan) +
                                                        " is not built for window exponent " + std::to_string(exp));
    const int new_shape = shape >= 0 ? shape : st->shape[c];
    const int new_plan = plan >= 0 ? plan : ctx_radix_plan(ctx, log_m);
    if (new_shape < 0 || new_shape > 2 || !fused_variant_ok(log_m, new_shape * 4 + new_plan))
        return ctx_fail(ctx, OSTFT_ERR_UNSUPPORTED,
                        "workgroup shape " + std::to_string(new_shape) + " with radix plan " + std::to_string(new_plan) +
                            " is not built for window exponent " + std::to_string(exp));
    if (plan >= 0)
        ctx_set_radix_plan(ctx, log_m, plan);
    st->shape[c] = new_shape;
    if (new_shape != 0)
        st->persistent[c] = 0;  // the persistent kernel has shape 0 only
    if (cur_shape)
        *cur_shape = st->shape[c];
    if (cur_plan)
        *cur_plan = ctx_radix_plan(ctx, log_m);
    return OSTFT_OK;
}

// Times one class over a synthetic ragged batch (`samples` samples in 32
// requests with the window, overlap, output layout and flags of `like`, or
// without it overlap 0.5, Hann, DC removal, compat power) under every built
// variant (radix plan x workgroup shape) in the dispatch form, and for
// shape 0 in the persistent form at each workgroups-per-CU setting.  The
// default (variant 0, one workgroup per tile) is timed first and stays unless
// a candidate beats it by more than AUTOTUNE_MARGIN, in the sweep and again
// when the two are timed alternately: most candidates land within a percent
// or two of each other, where one timing's noise would otherwise decide.  Which variant wins depends on the requests: the N/2+1
// layouts write half the bytes of the N-value ones per frame, so the same
// candidates rank differently under them.
int autotune_batch(ostft_ctx* ctx, int exp, uint64_t samples, const ostft_params* like, int* best_blocks_per_cu,
                   int* best_shape, int* best_plan, double* best_ms)
{
    BatchState* st = nullptr;
    int rc = state(ctx, &st);
    if (rc != OSTFT_OK)
        return rc;
    int c = 0;
    rc = class_of(ctx, exp, &c);
    if (rc != OSTFT_OK)
        return rc;
    const int log_m = c + LOG_M_MIN;
    // candidates: (variant, workgroups per CU); 0 per CU = one workgroup per tile
    std::vector<std::pair<int, int>> cand;
    for (int v = 0; v < FUSED_VARIANTS; ++v) {
        if (!fused_variant_ok(log_m, v))
            continue;
        rc = class_info(ctx, st, c, v);
        if (rc != OSTFT_OK)
            return rc;
        cand.push_back({v, 0});
        if (v < 4) {  // shape 0: the persistent form too
            const int mx = st->info[c][v].max_blocks_per_cu;
            for (int k = 1; k < mx; k *= 2)
                cand.push_back({v, k});
            cand.push_back({v, mx});
        }
    }
    const uint64_t N = 1ull << exp;
    if (samples < N)
        samples = N;
    // 32 requests of 1/2 .. 3/2 x samples/32 each (ragged, not window
    // multiples): few enough that the host's preparation of a batch stays
    // shorter than the GPU's work on the previous one
    std::vector<uint64_t> lens;
    const uint64_t per = std::max<uint64_t>(samples / 32, N);
    for (int i = 0; i < 32; ++i)
        lens.push_back(per / 2 + (per * (uint64_t)(i % 8)) / 8 + (uint64_t)(i * 37) % N);
    ostft_params p;
    if (like) {
        p = *like;
        p.exp = exp;
        if (p.flags & (OSTFT_FLAG_MFMA_FP16 | OSTFT_FLAG_MFMA_BF16))
            return ctx_fail(ctx, OSTFT_ERR_INVALID_ARG,
                            "autotune: matrix-core requests do not run the batch kernels");
    } else {
        std::memset(&p, 0, sizeof(p));
        p.exp = exp;
        p.overlap = 0.5f;
        p.window = OSTFT_WIN_HANNING;
        p.output = OSTFT_OUT_COMPAT_POWER;
        p.flags = OSTFT_FLAG_REMOVE_DC;
    }
    std::vector<ostft_job> jobs(lens.size());
    uint64_t in_off = 0, out_off = 0;
    for (size_t i = 0; i < lens.size(); ++i) {
        ostft_geometry g;
        rc = ostft_get_geometry(&p, lens[i], &g);
        if (rc != OSTFT_OK)
            return ctx_fail(ctx, rc, "autotune geometry");
        jobs[i].full_size = lens[i];
        jobs[i].out_cap = g.out_floats;
        jobs[i].params = p;
        jobs[i].in = reinterpret_cast<const float*>(in_off);  // offsets until the buffers exist
        jobs[i].out = reinterpret_cast<float*>(out_off);
        in_off += lens[i];
        out_off += (g.out_floats + 3) & ~3ull;
    }
    float* din = nullptr;
    float* dout = nullptr;
    hipEvent_t e0 = nullptr, e1 = nullptr;
    hipStream_t s = nullptr;
    hipError_t e = hipMalloc(&din, sizeof(float) * in_off);
    if (e == hipSuccess)
        e = hipMalloc(&dout, sizeof(float) * out_off);
    if (e == hipSuccess)
        e = hipEventCreate(&e0);
    if (e == hipSuccess)
        e = hipEventCreate(&e1);
    if (e == hipSuccess)
        e = hipStreamCreateWithFlags(&s, hipStreamNonBlocking);
    if (e == hipSuccess)
        e = hipMemsetD32Async(reinterpret_cast<hipDeviceptr_t>(din), 0x3e800000u /* 0.25f */, in_off, s);
    if (e == hipSuccess)
        e = hipStreamSynchronize(s);
    if (e == hipSuccess) {
        for (auto& j : jobs) {
            j.in = din + reinterpret_cast<uint64_t>(j.in);
            j.out = dout + reinterpret_cast<uint64_t>(j.out);
        }
        const int saved_pc = st->per_cu[c], saved_ps = st->persistent[c], saved_shape = st->shape[c];
        // the GPU time of one batch under candidate (variant, per CU): min
        // over `rounds` - 1 timed rounds after a warming one
        auto timed = [&](const std::pair<int, int>& cd, int rounds) {
            const int v = cd.first, k = cd.second;
            st->shape[c] = v >> 2;
            st->plan_override[c] = v & 3;
            st->persistent[c] = k > 0;
            st->per_cu[c] = k;
            // run; e0; run; e1: the second batch is prepared while the first
            // runs, so e0 -> e1 is the GPU's time for one batch
            float tmin = 1e30f;
            for (int r = 0; r < rounds && rc == OSTFT_OK && e == hipSuccess; ++r) {
                rc = run_batch(ctx, jobs.data(), (uint32_t)jobs.size(), s);
                if (rc == OSTFT_OK)
                    e = hipEventRecord(e0, s);
                if (rc == OSTFT_OK && e == hipSuccess)
                    rc = run_batch(ctx, jobs.data(), (uint32_t)jobs.size(), s);
                if (rc == OSTFT_OK && e == hipSuccess)
                    e = hipEventRecord(e1, s);
                if (rc == OSTFT_OK && e == hipSuccess)
                    e = hipEventSynchronize(e1);
                float ms = 0.0f;
                if (rc == OSTFT_OK && e == hipSuccess)
                    e = hipEventElapsedTime(&ms, e0, e1);
                if (r > 0)  // the first round warms caches and tables
                    tmin = std::min(tmin, ms);
            }
            return tmin;
        };
        std::pair<int, int> best{0, 0};
        float best_t = 1e30f;
        for (const auto& cd : cand) {
            const float tmin = timed(cd, 5);
            if (rc != OSTFT_OK || e != hipSuccess)
                break;
            // the first candidate is the default; later ones must win clearly
            if (best_t == 1e30f || tmin < best_t * (1.0f - AUTOTUNE_MARGIN)) {
                best_t = tmin;
                best = cd;
            }
        }
        // a winner other than the default is timed against the default
        // again, alternately, and kept only if it still wins by the margin:
        // one lucky timing in the sweep does not decide
        if (rc == OSTFT_OK && e == hipSuccess && best != cand.front()) {
            float td = 1e30f, tb = 1e30f;
            for (int r = 0; r < 3 && rc == OSTFT_OK && e == hipSuccess; ++r) {
                td = std::min(td, timed(cand.front(), 3));
                tb = std::min(tb, timed(best, 3));
            }
            if (rc == OSTFT_OK && e == hipSuccess && !(tb < td * (1.0f - AUTOTUNE_MARGIN))) {
                best = cand.front();
                best_t = td;
            } else {
                best_t = tb;
            }
        }
        st->plan_override[c] = -1;
        st->per_cu[c] = saved_pc;
        st->persistent[c] = saved_ps;
        st->shape[c] = saved_shape;
        if (rc == OSTFT_OK && e == hipSuccess) {
            st->shape[c] = best.first >> 2;
            st->persistent[c] = best.second > 0;
            st->per_cu[c] = best.second;
            ctx_set_radix_plan(ctx, log_m, best.first & 3);
            if (best_blocks_per_cu)
                *best_blocks_per_cu = best.second;
            if (best_shape)
                *best_shape = best.first >> 2;
            if (best_plan)
                *best_plan = best.first & 3;
            if (best_ms)
                *best_ms = best_t;
        }
    }
    if (s) {
        (void)hipStreamSynchronize(s);
        (void)hipStreamDestroy(s);
    }
    if (e0)
        (void)hipEventDestroy(e0);
    if (e1)
        (void)hipEventDestroy(e1);
    if (din)
        (void)hipFree(din);
    if (dout)
        (void)hipFree(dout);
    if (e != hipSuccess)
        return ctx_hip_fail(ctx, e, "autotune");
    return rc;
}

void batch_release(ostft_ctx* ctx)
{
    BatchState*& b = ctx_batch(ctx);
    if (!b)
        return;
    for (auto& sl : b->slot) {
        if (sl.used)
            (void)hipEventSynchronize(sl.done);
        free_slot(sl);
    }
    for (auto& sl : b->held)
        free_slot(sl);
    b->sides.destroy();
    delete b;
    b = nullptr;
}

}  // namespace ostft

// multipass.hpp -- large-window path (complex transform sizes 2^16 .. 2^19, and
// short requests of 2^15).
#pragma once

#include <mutex>
#include <vector>

#include "capture.hpp"
#include "engine.hpp"
#include "side_stream.hpp"

struct ostft_ctx;

namespace ostft {

// The complex buffer between the two passes, owned by a context, grown on
// demand up to one chunk of frames.  Calls on different streams take turns:
// each call's launches wait for the previous call's (an event recorded on
// its stream) when the stream changes.  Captured calls have buffers of their own,
// together up to the budget; beyond that a graph uses this one.  What a graph
// uses is not freed before the context goes.
struct Scratch {
    struct Held {
        unsigned long long capture;  // the calls of this capture on this stream
        hipStream_t stream;
        float2* a;
        uint64_t cap;
    };
    float2* a = nullptr;
    uint64_t cap = 0;                      // complex elements
    bool in_graph = false;                 // a graph uses `a`
    std::vector<Held> held;
    uint64_t held_bytes = 0;
    uint64_t budget = (uint64_t)1 << 30;  // bytes it may take
    hipEvent_t done = nullptr;             // recorded after the last call's launches
    SideStreams sides;                     // every other chunk of a long request runs on one of these
    hipStream_t last = nullptr;            // the stream of that call
    bool used = false;
    hipError_t ensure(uint64_t n);
    float2* hold(const Capture& c, hipStream_t s, uint64_t n);  // a captured call's buffer, or null
    hipError_t acquire(hipStream_t s);  // order stream s after the previous user
    hipError_t handoff(hipStream_t s);  // record the end of this call's launches
    void release();                     // frees the buffer (after the last user's launches)
    void destroy();                     // everything (no graph uses it any more)
};

// accessors into the context (defined in capi.hip)
// W_m^j, j < count; with `noalloc` only a table already resident (else null
// and OSTFT_ERR_NOT_PREPARED in *rc)
float2* ctx_twiddles(ostft_ctx* ctx, int64_t m, int64_t count, int* rc, bool noalloc = false);
double2* ctx_twiddles64(ostft_ctx* ctx, int64_t m, int64_t count, int* rc, bool noalloc = false);
bool ctx_has_twiddles(ostft_ctx* ctx, int64_t m, int64_t count);  // that table is resident
Scratch& ctx_scratch(ostft_ctx* ctx);
std::mutex& ctx_scratch_mutex(ostft_ctx* ctx);  // held while a call queues its scratch launches

// Runs the two passes (the split epilogue inside the last).  Returns an OSTFT_*
// status; with `noalloc`, OSTFT_ERR_NOT_PREPARED (and no message) where the
// scratch that is there does not hold the request, or s is being captured.
int run_multipass(ostft_ctx* ctx, int log_m, const FusedArgs& a, hipStream_t s, bool noalloc = false);
// Window 2^16: the two passes for a few frames, else the one kernel (bitwise the same).
int run_wide(ostft_ctx* ctx, int log_m, const FusedArgs& a, hipStream_t s);
// The same without allocations: the passes where scratch and tables are there.
int run_wide_noalloc(ostft_ctx* ctx, int log_m, const FusedArgs& a, hipStream_t s);
// The same through the fixed per-device scratch array (no allocation, no
// event; the tables must be resident).  Calls that overlap on one GPU race.
int run_multipass_static(ostft_ctx* ctx, int device, int log_m, const FusedArgs& a, hipStream_t s);
// Looks up the fixed scratch of the current device, `device` (once per device).
hipError_t multipass_static_scratch_init(int device);

// Frames whose scratch fits `budget` bytes, at least one: the most that are
// between the two passes at any time.
uint64_t multipass_chunk_frames(uint64_t budget, int log_m);

bool multipass_supported(int log_m);  // complex sizes 2^15 .. 2^19

}  // namespace ostft

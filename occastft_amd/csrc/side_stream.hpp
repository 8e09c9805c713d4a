// side_stream.hpp -- a second stream for launches that may run beside the
// caller's: it forks from the caller's stream and joins it again, so that to
// the caller everything is ordered on the stream it gave.
#pragma once

#include <hip/hip_runtime.h>

#include <memory>
#include <vector>

#include "capture.hpp"

namespace ostft {

struct SideStream {
    hipStream_t stream = nullptr;
    hipEvent_t forked = nullptr, joined = nullptr;

    // `stream` follows what s holds so far
    hipError_t fork(hipStream_t s)
    {
        hipError_t e = hipSuccess;
        if (!forked)
            e = hipEventCreateWithFlags(&forked, hipEventDisableTiming);
        if (e == hipSuccess && !joined)
            e = hipEventCreateWithFlags(&joined, hipEventDisableTiming);
        if (e == hipSuccess && !stream)
            e = hipStreamCreateWithFlags(&stream, hipStreamNonBlocking);
        if (e == hipSuccess)
            e = hipEventRecord(forked, s);
        return e == hipSuccess ? hipStreamWaitEvent(stream, forked, 0) : e;
    }
    // s follows what `stream` holds so far
    hipError_t join(hipStream_t s)
    {
        const hipError_t e = hipEventRecord(joined, stream);
        return e == hipSuccess ? hipStreamWaitEvent(s, joined, 0) : e;
    }
    void destroy()
    {
        for (hipEvent_t* e : {&forked, &joined}) {
            if (*e)
                (void)hipEventDestroy(*e);
            *e = nullptr;
        }
        if (stream)
            (void)hipStreamDestroy(stream);
        stream = nullptr;
    }
};

// The side streams of one kind of launches (under its lock).  A stream forked
// from a capturing one belongs to that capture until it ends, and another call
// could not fork it: ordinary calls have a side stream of their own, and each
// capture under way has one, which a later capture takes over.
class SideStreams {
    struct Captured {
        SideStream side;
        unsigned long long id;
    };
    SideStream own;
    std::vector<std::unique_ptr<Captured>> captured;

public:
    SideStream& of(const Capture& c)
    {
        if (!c.on)
            return own;
        for (auto& k : captured)
            if (k->id == c.id)
                return k->side;
        for (auto& k : captured)
            if (!k->side.stream || !capture_of(k->side.stream).on) {
                k->id = c.id;
                return k->side;
            }
        captured.emplace_back(new Captured{SideStream{}, c.id});
        return captured.back()->side;
    }
    void destroy()
    {
        own.destroy();
        for (auto& k : captured)
            k->side.destroy();
        captured.clear();
    }
};

}  // namespace ostft

// capture.hpp -- calls on a stream that is being captured into a graph.
//
// The graph replays the launches with the addresses they had, at times the
// context does not see.  So a captured call shares no buffer and no event with
// other calls: what its launches need stays allocated with the context.
#pragma once

#include <hip/hip_runtime.h>

namespace ostft {

// The capture that a stream belongs to.
struct Capture {
    bool on = false;
    unsigned long long id = 0;
};
inline Capture capture_of(hipStream_t s)
{
    Capture c;
    hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
    // refused for the null stream while another stream is captured: not in that capture
    if (hipStreamGetCaptureInfo(s, &status, &c.id) != hipSuccess)
        (void)hipGetLastError();  // launches read the last error
    else
        c.on = status != hipStreamCaptureStatusNone;
    return c;
}

// Lets the calling thread allocate while a capture is under way.
class AllocateInCapture {
    hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
    bool on;

public:
    explicit AllocateInCapture(bool capturing) : on(capturing)
    {
        on = on && hipThreadExchangeStreamCaptureMode(&mode) == hipSuccess;
    }
    ~AllocateInCapture()
    {
        if (on)
            (void)hipThreadExchangeStreamCaptureMode(&mode);
    }
    AllocateInCapture(const AllocateInCapture&) = delete;
    AllocateInCapture& operator=(const AllocateInCapture&) = delete;
};

}  // namespace ostft

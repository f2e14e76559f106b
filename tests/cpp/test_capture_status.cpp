// stream_capturing() (cuflash-attn_amd/csrc/workspace.cpp) against a capture query with a chosen
// outcome. No GPU call is made.
#include <hip/hip_runtime.h>

#include <cstdio>

namespace {
hipError_t g_result = hipSuccess;
hipStreamCaptureStatus g_status = hipStreamCaptureStatusNone;
hipError_t query(hipStream_t, hipStreamCaptureStatus* status) {
    if (g_result == hipSuccess) *status = g_status;
    return g_result;
}
}  // namespace

#define hipStreamIsCapturing query
#include "../../cuflash-attn_amd/csrc/workspace.cpp"

int main() {
    struct Case {
        hipError_t result;
        hipStreamCaptureStatus status;
        bool capturing;
    };
    const Case cases[] = {
        {hipSuccess, hipStreamCaptureStatusNone, false},
        {hipSuccess, hipStreamCaptureStatusActive, true},
        {hipSuccess, hipStreamCaptureStatusInvalidated, true},
        {hipErrorStreamCaptureImplicit, hipStreamCaptureStatusNone, true},
        {hipErrorInvalidHandle, hipStreamCaptureStatusNone, true},
    };
    int bad = 0;
    for (const Case& c : cases) {
        g_result = c.result;
        g_status = c.status;
        const bool got = cuflash::detail::stream_capturing(nullptr);
        if (got != c.capturing) {
            std::printf("result %d, status %d: %d\n", c.result, c.status, got);
            ++bad;
        }
    }
    return bad;
}

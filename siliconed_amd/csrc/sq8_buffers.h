// sq8_buffers.h — a context's growable device buffers (the staged activation, repacked codes, partial sums).
//
// A buffer grows by replacement. One that a stream capture has used is written and read by every replay of that graph, so
// growing sets it aside instead of freeing it; what is set aside is freed with the context.
#pragma once

#include <hip/hip_runtime.h>

#include <new>

namespace sq8 {

struct Buffer {
    void *at;
    size_t bytes;
    bool in_graph;  // used under stream capture: a graph may hold its address
};

struct SetAside {
    void *at;
    SetAside *next;
};

// Whether `stream` is being captured into a graph (a query that fails, as on the null stream beside another stream's
// capture, counts as one).
inline bool capturing(hipStream_t stream) {
    hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(stream, &status) != hipSuccess) {
        (void)hipGetLastError();
        return true;
    }
    return status != hipStreamCaptureStatusNone;
}

// Grows `b` to `bytes` at least, after the stream has finished with the old memory (under capture the runtime refuses
// that wait), and marks it where the call that asks is being captured.
inline hipError_t reserve(Buffer &b, size_t bytes, hipStream_t stream, SetAside *&aside) {
    if (b.bytes < bytes) {
        if (b.at) {
            const hipError_t e = hipStreamSynchronize(stream);
            if (e != hipSuccess) return e;
            if (b.in_graph) {
                SetAside *kept = new (std::nothrow) SetAside{b.at, aside};
                if (!kept) return hipErrorOutOfMemory;
                aside = kept;
            } else {
                (void)hipFree(b.at);
            }
            b = Buffer{nullptr, 0, false};
        }
        const hipError_t e = hipMalloc(&b.at, bytes);
        if (e != hipSuccess) {
            b.at = nullptr;
            return e;
        }
        b.bytes = bytes;
    }
    if (capturing(stream)) b.in_graph = true;
    return hipSuccess;
}

inline void release(Buffer &b) {
    if (b.at) (void)hipFree(b.at);
    b = Buffer{nullptr, 0, false};
}

inline void release(SetAside *&aside) {
    while (aside) {
        SetAside *next = aside->next;
        (void)hipFree(aside->at);
        delete aside;
        aside = next;
    }
}

}  // namespace sq8

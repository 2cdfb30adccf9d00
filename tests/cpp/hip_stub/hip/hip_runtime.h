// Stand-ins for the few HIP calls of rllm_amd/csrc/workspace.h, so that its
// bookkeeping is tested on the CPU (test_workspace.cpp): device memory is host
// memory, a stream is a number, and `stub_capturing` is the stream being captured.
#pragma once

#include <cstdint>
#include <cstdlib>
#include <cstring>

typedef struct stub_stream* hipStream_t;
typedef int hipError_t;
enum : int { hipSuccess = 0 };
enum hipStreamCaptureStatus { hipStreamCaptureStatusNone = 0, hipStreamCaptureStatusActive = 1 };

inline uintptr_t stub_capturing = 0;

inline hipError_t hipGetDevice(int* dev) { *dev = 0; return hipSuccess; }
inline hipError_t hipStreamIsCapturing(hipStream_t s, hipStreamCaptureStatus* c) {
    *c = stub_capturing && reinterpret_cast<uintptr_t>(s) == stub_capturing ? hipStreamCaptureStatusActive
                                                                              : hipStreamCaptureStatusNone;
    return hipSuccess;
}
inline hipError_t hipMalloc(void** p, size_t n) { *p = std::malloc(n); return *p ? hipSuccess : 2; }
inline hipError_t hipMemsetAsync(void* p, int v, size_t n, hipStream_t) { std::memset(p, v, n); return hipSuccess; }

// What the library asks of the HIP runtime, answered without a GPU: an executable's own definitions come before those of the
// runtime it is linked with.  hipLaunchKernel is the including test's.
#pragma once
#include <hip/hip_runtime.h>

static alignas(256) unsigned char g_scratch[256];  // where the library's own scratch "is"
static bool g_capturing = false;

extern "C" {
hipError_t hipGetDevice(int* device) { *device = 0; return hipSuccess; }
hipError_t hipDeviceGetAttribute(int* value, hipDeviceAttribute_t, int) { *value = 256; return hipSuccess; }
hipError_t hipFuncSetAttribute(const void*, hipFuncAttribute, int) { return hipSuccess; }
hipError_t hipGetLastError(void) { return hipSuccess; }
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus* status) { *status = g_capturing ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone; return hipSuccess; }
hipError_t hipGetSymbolAddress(void** address, const void*) { *address = g_scratch; return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
}

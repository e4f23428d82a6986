// The runtime calls that a plan makes, on a machine without a GPU: memory is the host's, an address is "memory of" the device and
// kind that the test says, and uploads are noted by their form.
#include <hip/hip_runtime_api.h>

#include <cstdlib>
#include <cstring>

static int g_current, g_memory_device, g_memory_type, g_stream_device, g_kernels, g_copies;
static char g_scratch[256];

extern "C" {
void stand_in_set(int current, int memory_device, int memory_type, int stream_device) {
    g_current = current; g_memory_device = memory_device; g_memory_type = memory_type; g_stream_device = stream_device;
    g_kernels = g_copies = 0;
}
int stand_in_kernels() { return g_kernels; }
int stand_in_copies() { return g_copies; }

hipError_t hipGetDevice(int* d) { *d = g_current; return hipSuccess; }
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int) { *v = 256; return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipHostMalloc(void** p, size_t n, unsigned) { *p = malloc(n); return hipSuccess; }
hipError_t hipHostFree(void* p) { free(p); return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { *e = (hipEvent_t)1; return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipGetSymbolAddress(void** p, const void*) { *p = g_scratch; return hipSuccess; }
hipError_t hipStreamGetDevice(hipStream_t, hipDevice_t* d) { *d = g_stream_device; return hipSuccess; }
hipError_t hipPointerGetAttributes(hipPointerAttribute_t* a, const void*) {
    if (g_memory_type < 0) return hipErrorInvalidValue;
    memset(a, 0, sizeof(*a));
    a->type = (hipMemoryType)g_memory_type;
    a->device = g_memory_device;
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void* to, const void* from, size_t n, hipMemcpyKind, hipStream_t) {
    memcpy(to, from, n);
    ++g_copies;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void*, dim3, dim3, void**, size_t, hipStream_t) { ++g_kernels; return hipSuccess; }
}

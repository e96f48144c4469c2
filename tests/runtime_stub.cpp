// A HIP runtime without a GPU, for tests of what the library's host code asks of the real one: launches are counted and not run,
// device memory is host memory, of which there may be none (stub_no_memory) or so much (stub_memory_most), and addresses within [stub_device_first,
// stub_device_end) are reported as device memory.  Loaded before libsthip.so with its symbols global.
#include <hip/hip_runtime_api.h>

#include <cstdlib>
#include <cstring>
#include <map>

extern "C" {
int stub_no_memory = 0, stub_device = 0, stub_stream_device = 0;
unsigned long long stub_launches = 0, stub_frees = 0, stub_memory_used = 0, stub_memory_most = ~0ull;
const char *stub_device_first = nullptr, *stub_device_end = nullptr;
const void *stub_first_source = nullptr;  // of the runtime's copies

hipError_t hipGetDeviceCount(int *count) { *count = 1; return hipSuccess; }
hipError_t hipGetDevice(int *device) { *device = stub_device; return hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600 *props, int)
{
    std::memset(props, 0, sizeof *props);
    std::strcpy(props->gcnArchName, "gfx950");
    props->multiProcessorCount = 256;
    return hipSuccess;
}
hipError_t hipGetSymbolAddress(void **address, const void *symbol) { *address = const_cast<void *>(symbol); return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
static std::map<void *, size_t> &allocations() { static auto *all = new std::map<void *, size_t>; return *all; }
hipError_t hipMalloc(void **ptr, size_t bytes)
{
    if (stub_no_memory || stub_memory_used + bytes > stub_memory_most) return hipErrorOutOfMemory;
    *ptr = std::aligned_alloc(4096, (bytes + 4095) / 4096 * 4096);
    if (*ptr) stub_memory_used += allocations()[*ptr] = bytes;
    return *ptr ? hipSuccess : hipErrorOutOfMemory;
}
hipError_t hipFree(void *ptr)
{
    ++stub_frees;
    stub_memory_used -= allocations()[ptr];
    allocations().erase(ptr);
    std::free(ptr);
    return hipSuccess;
}
hipError_t hipHostMalloc(void **ptr, size_t bytes, unsigned)
{
    *ptr = std::aligned_alloc(4096, (bytes + 4095) / 4096 * 4096);
    return hipSuccess;
}
hipError_t hipHostFree(void *ptr) { std::free(ptr); return hipSuccess; }
hipError_t hipStreamCreate(hipStream_t *stream) { *stream = reinterpret_cast<hipStream_t>(std::malloc(1)); return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t stream) { std::free(stream); return hipSuccess; }
hipError_t hipStreamGetDevice(hipStream_t, hipDevice_t *device) { *device = stub_stream_device; return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus *status) { *status = hipStreamCaptureStatusNone; return hipSuccess; }
hipError_t hipThreadExchangeStreamCaptureMode(hipStreamCaptureMode *) { return hipSuccess; }
hipError_t hipFuncSetAttribute(const void *, hipFuncAttribute, int) { return hipSuccess; }
static dim3 pushed_grid, pushed_block;
unsigned stub_grid = 0;            // of the last launch: workgroups along x
unsigned long long stub_lds = 0;   // and its dynamic LDS
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t lds, hipStream_t)
{
    stub_grid = grid.x;
    stub_lds = lds;
    pushed_grid = grid;
    pushed_block = block;
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *grid, dim3 *block, size_t *lds, hipStream_t *stream)
{
    *grid = pushed_grid;
    *block = pushed_block;
    *lds = 0;
    *stream = nullptr;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void *, dim3, dim3, void **, size_t, hipStream_t)
{
    ++stub_launches;
    return hipSuccess;
}
static bool passes_device_end(const void *ptr, size_t bytes)
{
    const char *const at = static_cast<const char *>(ptr);
    return at >= stub_device_first && at < stub_device_end && bytes > static_cast<size_t>(stub_device_end - at);
}
hipError_t hipMemcpyAsync(void *dst, const void *src, size_t bytes, hipMemcpyKind, hipStream_t)
{
    if (passes_device_end(src, bytes) || passes_device_end(dst, bytes)) return hipErrorInvalidValue;
    if (stub_first_source == nullptr) stub_first_source = src;
    return hipSuccess;
}
hipError_t hipPointerGetAttributes(hipPointerAttribute_t *attributes, const void *ptr)
{
    const char *const at = static_cast<const char *>(ptr);
    if (at < stub_device_first || at >= stub_device_end) return hipErrorInvalidValue;
    std::memset(attributes, 0, sizeof *attributes);
    attributes->type = hipMemoryTypeDevice;
    return hipSuccess;
}
hipError_t hipMemGetAddressRange(hipDeviceptr_t *base, size_t *size, hipDeviceptr_t)  // (of what is device memory, asked before)
{
    *base = const_cast<char *>(stub_device_first);
    *size = static_cast<size_t>(stub_device_end - stub_device_first);
    return hipSuccess;
}
hipError_t hipMemsetAsync(void *, int, size_t, hipStream_t) { return hipSuccess; }
}

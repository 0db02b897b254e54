// The HIP calls of libtsac_hip.so made on the host alone, so that the library's memory
// management and launch shapes can be tested without a GPU: device memory is address
// space that is never touched, kernels are counted with their grids and not run, and
// copies to the host fill in one value. Loaded with global symbols before the library.
#include <hip/hip_runtime_api.h>

#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <string>

namespace
{
std::mutex mutex;
uintptr_t next_address = uintptr_t(1) << 44;
std::map<uintptr_t, size_t> device; // allocations
size_t device_total = size_t(288) << 30, device_used = 0, largest = ~size_t(0);
std::map<std::string, long> counts;
bool pinned_fails = false;
unsigned fill = 0x4000; // 16-bit value that copies to the host leave
thread_local hipError_t last_error = hipSuccess;
struct Launch
{
    dim3 grid, block;
    size_t shared;
    hipStream_t stream;
};
thread_local Launch pending;
std::map<const void*, std::string> names;
std::string launched; // "name x y z threads" lines

hipError_t failed(hipError_t e)
{
    return last_error = e;
}

hipError_t allocate(void** p, size_t bytes)
{
    const std::lock_guard<std::mutex> lock(mutex);
    if (bytes > largest || device_used + bytes > device_total)
    {
        return failed(hipErrorOutOfMemory);
    }
    *p = reinterpret_cast<void*>(next_address);
    device[next_address] = bytes;
    next_address += (bytes + 4095) / 4096 * 4096 + 4096;
    device_used += bytes;
    return hipSuccess;
}

hipError_t release(void* p)
{
    const std::lock_guard<std::mutex> lock(mutex);
    if (!p)
    {
        return hipSuccess;
    }
    const auto found = device.find(reinterpret_cast<uintptr_t>(p));
    if (found == device.end())
    {
        return failed(hipErrorInvalidValue);
    }
    device_used -= found->second;
    device.erase(found);
    return hipSuccess;
}

void count(const char* name)
{
    const std::lock_guard<std::mutex> lock(mutex);
    ++counts[name];
}

hipError_t copy(void* to, size_t bytes, hipMemcpyKind kind)
{
    if (kind == hipMemcpyDeviceToHost)
    {
        // A call's error words are at most 12 bytes, and none is set.
        for (size_t i = 0; i < bytes / 2; ++i)
        {
            static_cast<uint16_t*>(to)[i] = bytes <= 12 ? 0 : uint16_t(fill);
        }
    }
    return hipSuccess;
}
} // namespace

extern "C"
{
// ---- what tests set and read
void host_hip_total(size_t bytes)
{
    device_total = bytes;
}
void host_hip_largest(size_t bytes) // of one allocation
{
    largest = bytes;
}
size_t host_hip_used()
{
    return device_used;
}
long host_hip_count(const char* name)
{
    return counts[name];
}
void host_hip_pinned_fails(int on)
{
    pinned_fails = on;
}
const char* host_hip_launches() // since the last call
{
    static std::string text;
    text.swap(launched);
    launched.clear();
    return text.c_str();
}

// ---- HIP
hipError_t hipMalloc(void** p, size_t bytes)
{
    count("hipMalloc");
    return allocate(p, bytes);
}
hipError_t hipFree(void* p)
{
    count("hipFree");
    return release(p);
}
hipError_t hipMallocAsync(void** p, size_t bytes, hipStream_t)
{
    count("hipMallocAsync");
    return allocate(p, bytes);
}
hipError_t hipFreeAsync(void* p, hipStream_t)
{
    count("hipFreeAsync");
    return release(p);
}
hipError_t hipHostMalloc(void** p, size_t bytes, unsigned)
{
    count("hipHostMalloc");
    if (pinned_fails)
    {
        return failed(hipErrorOutOfMemory);
    }
    *p = std::calloc(bytes ? bytes : 1, 1);
    return hipSuccess;
}
hipError_t hipHostFree(void* p)
{
    std::free(p);
    return hipSuccess;
}
hipError_t hipHostGetDevicePointer(void** d, void* h, unsigned)
{
    *d = h;
    return hipSuccess;
}
hipError_t hipMemGetInfo(size_t* free, size_t* total)
{
    *free = device_total > device_used ? device_total - device_used : 0;
    *total = device_total;
    return hipSuccess;
}
hipError_t hipMemcpy(void* to, const void*, size_t bytes, hipMemcpyKind kind)
{
    return copy(to, bytes, kind);
}
hipError_t hipMemcpyAsync(void* to, const void*, size_t bytes, hipMemcpyKind kind, hipStream_t)
{
    return copy(to, bytes, kind);
}
hipError_t hipMemsetAsync(void*, int, size_t, hipStream_t)
{
    return hipSuccess;
}
hipError_t hipGetLastError()
{
    const hipError_t e = last_error;
    last_error = hipSuccess;
    return e;
}
const char* hipGetErrorString(hipError_t e)
{
    return e == hipErrorOutOfMemory ? "out of memory" : e == hipErrorInvalidConfiguration ? "invalid configuration" : "error";
}
hipError_t hipGetDevice(int* d)
{
    *d = 0;
    return hipSuccess;
}
hipError_t hipSetDevice(int)
{
    return hipSuccess;
}
hipError_t hipDeviceGetAttribute(int* value, hipDeviceAttribute_t, int)
{
    *value = 256; // compute units
    return hipSuccess;
}
hipError_t hipFuncSetAttribute(const void*, hipFuncAttribute, int)
{
    return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned)
{
    *s = reinterpret_cast<hipStream_t>(8);
    return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t)
{
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t)
{
    return hipSuccess;
}
hipError_t hipThreadExchangeStreamCaptureMode(hipStreamCaptureMode*)
{
    return hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t* e)
{
    *e = reinterpret_cast<hipEvent_t>(8);
    return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t)
{
    return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t, hipStream_t)
{
    return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t)
{
    return hipSuccess;
}
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t)
{
    *ms = 1.0f;
    return hipSuccess;
}

// ---- launches
void** __hipRegisterFatBinary(const void*)
{
    static void* handle;
    return &handle;
}
void __hipUnregisterFatBinary(void**)
{
}
void __hipRegisterFunction(void**, const void* function, char*, const char* name, unsigned, void*, void*, dim3*, dim3*,
                           int*)
{
    names[function] = name;
}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int)
{
}
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t shared, hipStream_t stream)
{
    pending = {grid, block, shared, stream};
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* grid, dim3* block, size_t* shared, hipStream_t* stream)
{
    *grid = pending.grid;
    *block = pending.block;
    *shared = pending.shared;
    *stream = pending.stream;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void* function, dim3 grid, dim3 block, void**, size_t, hipStream_t)
{
    count("hipLaunchKernel");
    // The limits of a grid: 2^32 work-items along each axis, 65,535 workgroups along y and z.
    const uint64_t limit = uint64_t(1) << 32;
    if (!grid.x || !grid.y || !grid.z || uint64_t(grid.x) * block.x >= limit || grid.y > 65535 || grid.z > 65535)
    {
        return failed(hipErrorInvalidConfiguration);
    }
    const std::lock_guard<std::mutex> lock(mutex);
    launched += names[function] + " " + std::to_string(grid.x) + " " + std::to_string(grid.y) + " " +
                std::to_string(grid.z) + " " + std::to_string(block.x) + "\n";
    return hipSuccess;
}
}

// The part of the HIP runtime's interface that host_transfer.hpp uses, on host
// memory: "device" arrays are ordinary ones that a test declares, copies happen
// at once, and every call is counted.
#pragma once

#include <atomic>
#include <cstddef>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>

enum hipError_t { hipSuccess = 0, hipErrorInvalidValue = 1, hipErrorOutOfMemory = 2 };
enum hipMemcpyKind { hipMemcpyHostToHost, hipMemcpyHostToDevice, hipMemcpyDeviceToHost, hipMemcpyDeviceToDevice, hipMemcpyDefault };
enum hipMemoryType { hipMemoryTypeUnregistered, hipMemoryTypeHost, hipMemoryTypeDevice, hipMemoryTypeManaged, hipMemoryTypeUnified };
enum { hipEventDisableTiming = 2, hipHostMallocCoherent = 0x40000000 };
typedef struct fake_stream* hipStream_t;
typedef struct fake_event* hipEvent_t;
typedef void* hipDeviceptr_t;

struct hipPointerAttribute_t
{
    hipMemoryType type;
    int device;
    void* devicePointer;
    void* hostPointer;
};

namespace fake
{
struct Range
{
    std::size_t bytes;
    hipMemoryType type;
    int device;
};
inline std::map<char*, Range> ranges;  // what the runtime knows of; set up before a transfer starts
inline std::atomic<int> copies, blocking_copies, events, pinned, threads_set, queries;
inline bool no_pinned = false;
inline unsigned pinned_flags = 0;
inline std::ptrdiff_t mapped = 0;  // distance of an array's address on the device

inline void reset() { copies = blocking_copies = events = pinned = threads_set = queries = 0; }
inline const Range* range_of(const void* p, char** base = nullptr)
{
    char* const c = static_cast<char*>(const_cast<void*>(p));
    auto it = ranges.upper_bound(c);
    if (it == ranges.begin()) return nullptr;
    --it;
    if (c >= it->first + it->second.bytes) return nullptr;
    if (base) *base = it->first;
    return &it->second;
}
}  // namespace fake

inline hipError_t hipSetDevice(int) { ++fake::threads_set; return hipSuccess; }
inline hipError_t hipGetLastError() { return hipSuccess; }
inline hipError_t hipHostMalloc(void** p, std::size_t n, unsigned flags)
{
    fake::pinned_flags = flags;
    if (fake::no_pinned) return hipErrorOutOfMemory;
    ++fake::pinned;
    *p = std::malloc(n);
    return hipSuccess;
}
inline hipError_t hipHostFree(void* p) { std::free(p); return hipSuccess; }
inline hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { *e = reinterpret_cast<hipEvent_t>(1); return hipSuccess; }
inline hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
inline hipError_t hipEventRecord(hipEvent_t, hipStream_t) { ++fake::events; return hipSuccess; }
inline hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
inline hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
inline hipError_t hipMemcpyAsync(void* d, const void* s, std::size_t n, hipMemcpyKind, hipStream_t)
{
    ++fake::copies;
    std::memcpy(d, s, n);
    return hipSuccess;
}
inline hipError_t hipMemcpy(void* d, const void* s, std::size_t n, hipMemcpyKind)
{
    ++fake::blocking_copies;
    std::memcpy(d, s, n);
    return hipSuccess;
}
inline hipError_t hipPointerGetAttributes(hipPointerAttribute_t* at, const void* p)
{
    ++fake::queries;
    const fake::Range* r = fake::range_of(p);
    if (!r) return hipErrorInvalidValue;
    char* const c = static_cast<char*>(const_cast<void*>(p));
    *at = hipPointerAttribute_t{r->type, r->device, c + fake::mapped, r->type == hipMemoryTypeDevice ? nullptr : c};
    return hipSuccess;
}
inline hipError_t hipMemGetAddressRange(hipDeviceptr_t* base, std::size_t* n, hipDeviceptr_t p)
{
    char* b = nullptr;
    const fake::Range* r = fake::range_of(static_cast<char*>(p) - fake::mapped, &b);
    if (!r) return hipErrorInvalidValue;
    *base = b + fake::mapped;
    *n = r->bytes;
    return hipSuccess;
}

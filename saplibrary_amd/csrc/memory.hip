// Allocation of the library's device buffers, and the kernels' LDS limits.
#include "sap_internal.hpp"

#include <atomic>
#include <cstdlib>
#include <map>
#include <mutex>
#include <utility>

namespace sap_amd {

namespace {

std::atomic<size_t> g_held{0};   // bytes of all buffers

// a number of bytes in the environment, 0 when unset
size_t env_bytes(const char* name)
{
    const char* e = std::getenv(name);
    return e ? (size_t)std::strtoull(e, nullptr, 10) : 0;
}

}  // namespace

void* device_alloc(size_t bytes)
{
    const size_t limit = env_bytes("SAP_AMD_DEVICE_LIMIT");
    void* p = nullptr;
    const hipError_t e = hipMalloc(&p, limit && g_held + bytes > limit ? (size_t)1 << 48 : bytes);
    if (e == hipErrorOutOfMemory) {
        (void)hipGetLastError();
        throw Error(SAP_ERR_OOM, "device buffer of " + std::to_string(bytes) + " bytes beside " +
                                     std::to_string(g_held) + " held: " + hipGetErrorString(e));
    }
    SAP_HIP_CHECK(e);
    g_held += bytes;
    return p;
}

void device_free(void* p, size_t bytes)
{
    (void)hipFree(p);
    g_held -= bytes;
}

void set_lds_limit(const void* kernel, size_t lds)
{
    static std::mutex mu;
    static std::map<std::pair<const void*, int>, size_t> done;
    int dev = 0;
    SAP_HIP_CHECK(hipGetDevice(&dev));
    std::lock_guard<std::mutex> lock(mu);
    size_t& have = done[{kernel, dev}];
    if (lds <= have) return;
    SAP_HIP_CHECK(hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    have = lds;
}

size_t device_free_bytes()
{
    if (const size_t set = env_bytes("SAP_AMD_DEVICE_FREE")) return set;
    size_t free = 0, total = 0;
    SAP_HIP_CHECK(hipMemGetInfo(&free, &total));
    return free;
}

}  // namespace sap_amd

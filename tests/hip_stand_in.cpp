// A HIP runtime without a GPU, for tests of the library's host code: memory is
// host memory, copies are done at once, launches are counted and their plan
// pointers checked, nothing is computed.  Load it with RTLD_GLOBAL before the
// library.  Time is the number of launches, a millisecond each.
#include <hip/hip_runtime_api.h>
#include <sys/mman.h>

#include <cstdint>
#include <cstring>
#include <map>
#include <mutex>
#include <string>
#include <vector>

namespace {
std::mutex mu;
std::map<uintptr_t, size_t> blocks;              // live device memory
std::map<const void *, std::string> kernels;     // by host stub
size_t live = 0, peak = 0, capacity = size_t(288) << 30;
int64_t launches = 0, bad_launches = 0;
int fail_malloc = 0;                             // 1: the next one fails
bool fail_host = false;                          // all pinned allocations fail
hipError_t last = hipSuccess;
struct Call {
    dim3 grid, block;
    size_t shmem;
    hipStream_t stream;
};
thread_local std::vector<Call> calls;

struct Event {
    int64_t at;
};

hipError_t fail(hipError_t e) { return last = e; }

bool is_device(const void *p)
{
    auto it = blocks.upper_bound((uintptr_t)p);
    if (it == blocks.begin())
        return false;
    --it;
    return (uintptr_t)p < it->first + it->second;
}

// Arguments of a kernel that have to point into device memory.
std::vector<int> pointers_of(const std::string &name)
{
    if (name.find("k_tile_adjoint") != std::string::npos)
        return {0, 1, 2, 3, 4, 6};
    if (name.find("k_tile") != std::string::npos)
        return {0, 1, 2, 3};
    if (name.find("k_batch_forward") != std::string::npos)
        return {0, 1, 3, 4, 5, 6};
    if (name.find("k_batch_reverse") != std::string::npos)
        return {0, 1, 3, 4, 5, 6, 7};
    return {};
}
}  // namespace

extern "C" {

// ------------------------------------------------------ what tests look at --
void stand_in_capacity(uint64_t bytes) { capacity = bytes; }
void stand_in_fail_malloc(int nth) { fail_malloc = nth; }
void stand_in_fail_host(int on) { fail_host = on != 0; }
int64_t stand_in_launches(void) { return launches; }
int64_t stand_in_bad_launches(void) { return bad_launches; }
uint64_t stand_in_peak(void) { return peak; }
uint64_t stand_in_reset_peak(void) { return peak = live; }

// ----------------------------------------------------------------- runtime --
void **__hipRegisterFatBinary(const void *)
{
    static void *module = nullptr;
    return &module;
}
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *host, char *, const char *name, unsigned, void *, void *, void *, void *,
                           int *)
{
    kernels[host] = name;
}
void __hipRegisterVar(void **, void *, char *, const char *, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t shmem, hipStream_t s)
{
    calls.push_back({grid, block, shmem, s});
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *grid, dim3 *block, size_t *shmem, hipStream_t *s)
{
    const Call c = calls.back();
    calls.pop_back();
    *grid = c.grid;
    *block = c.block;
    *shmem = c.shmem;
    *s = c.stream;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void *f, dim3 grid, dim3 block, void **args, size_t, hipStream_t)
{
    std::lock_guard<std::mutex> lk(mu);
    launches++;
    bool ok = grid.x > 0 && block.x > 0 && block.x <= 1024;
    for (int i : pointers_of(kernels[f]))
        ok = ok && is_device(*(void **)args[i]);
    bad_launches += !ok;
    return hipSuccess;
}

hipError_t hipMalloc(void **p, size_t bytes)
{
    std::lock_guard<std::mutex> lk(mu);
    *p = nullptr;
    if ((fail_malloc > 0 && --fail_malloc == 0) || live + bytes > capacity)
        return fail(hipErrorOutOfMemory);
    void *m = mmap(nullptr, bytes, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
    if (m == MAP_FAILED)
        return fail(hipErrorOutOfMemory);
    blocks[(uintptr_t)m] = bytes;
    live += bytes;
    peak = live > peak ? live : peak;
    *p = m;
    return hipSuccess;
}
hipError_t hipFree(void *p)
{
    std::lock_guard<std::mutex> lk(mu);
    auto it = blocks.find((uintptr_t)p);
    if (!p)
        return hipSuccess;
    if (it == blocks.end())
        return fail(hipErrorInvalidValue);
    live -= it->second;
    munmap(p, it->second);
    blocks.erase(it);
    return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t bytes, unsigned)
{
    std::lock_guard<std::mutex> lk(mu);
    *p = nullptr;
    if (fail_host)
        return fail(hipErrorOutOfMemory);
    *p = ::operator new(bytes);
    return hipSuccess;
}
hipError_t hipHostFree(void *p)
{
    ::operator delete(p);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void *dst, const void *src, size_t bytes, hipMemcpyKind, hipStream_t)
{
    std::memcpy(dst, src, bytes);
    return hipSuccess;
}
hipError_t hipMemGetInfo(size_t *free_bytes, size_t *total)
{
    std::lock_guard<std::mutex> lk(mu);
    *free_bytes = capacity > live ? capacity - live : 0;
    *total = capacity;
    return hipSuccess;
}

hipError_t hipGetDeviceCount(int *count)
{
    *count = 1;
    return hipSuccess;
}
hipError_t hipGetDevice(int *device)
{
    *device = 0;
    return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600 *p, int)
{
    std::memset(p, 0, sizeof(*p));
    std::strcpy(p->gcnArchName, "gfx950");
    p->multiProcessorCount = 256;
    p->totalGlobalMem = capacity;
    return hipSuccess;
}
hipError_t hipDeviceCanAccessPeer(int *ok, int, int)
{
    *ok = 0;
    return hipSuccess;
}
const char *hipGetErrorString(hipError_t e) { return e == hipSuccess ? "no error" : "an error of the stand-in"; }
hipError_t hipGetLastError(void)
{
    const hipError_t e = last;
    last = hipSuccess;
    return e;
}
hipError_t hipGetSymbolAddress(void **, const void *) { return fail(hipErrorInvalidSymbol); }

hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned)
{
    *s = (hipStream_t) new char;
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return fail(hipErrorNotSupported); }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t *) { return fail(hipErrorNotSupported); }
hipError_t hipGraphInstantiate(hipGraphExec_t *, hipGraph_t, hipGraphNode_t *, char *, size_t)
{
    return fail(hipErrorNotSupported);
}
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return fail(hipErrorNotSupported); }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }

hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned)
{
    *e = (hipEvent_t) new Event{0};
    return hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t *e) { return hipEventCreateWithFlags(e, 0); }
hipError_t hipEventDestroy(hipEvent_t e)
{
    delete (Event *)e;
    return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t)
{
    ((Event *)e)->at = launches;
    return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t a, hipEvent_t b)
{
    *ms = (float)(((Event *)b)->at - ((Event *)a)->at);
    return hipSuccess;
}

// states take plain allocations
hipError_t hipMemGetAllocationGranularity(size_t *, const hipMemAllocationProp *, hipMemAllocationGranularity_flags)
{
    return fail(hipErrorNotSupported);
}
hipError_t hipMemCreate(hipMemGenericAllocationHandle_t *, size_t, const hipMemAllocationProp *, unsigned long long)
{
    return fail(hipErrorNotSupported);
}
hipError_t hipMemRelease(hipMemGenericAllocationHandle_t) { return hipSuccess; }
hipError_t hipMemAddressReserve(void **, size_t, size_t, void *, unsigned long long) { return fail(hipErrorNotSupported); }
hipError_t hipMemAddressFree(void *, size_t) { return hipSuccess; }
hipError_t hipMemMap(void *, size_t, size_t, hipMemGenericAllocationHandle_t, unsigned long long)
{
    return fail(hipErrorNotSupported);
}
hipError_t hipMemUnmap(void *, size_t) { return hipSuccess; }
hipError_t hipMemSetAccess(void *, size_t, const hipMemAccessDesc *, size_t) { return fail(hipErrorNotSupported); }

}  // extern "C"

// A HIP runtime without a device, for CPU tests of the library's host side:
// preloaded before libvoxelcore.so it takes the place of the runtime's entry
// points that the library uses.  Device memory is reserved address space that
// nothing touches, kernels do not run, and copies to the host give zeros or the
// values a test queued.  It records what the host side asked for: the work-items
// of every launch, the waits, and what is allocated.
#include <sys/mman.h>

#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <cstdio>
#include <cstring>
#include <deque>
#include <map>
#include <mutex>
#include <string>

#include <hip/hip_runtime_api.h>

namespace
{
struct Call
{
    dim3 grid, block;
    size_t shared;
    hipStream_t stream;
};
thread_local std::deque<Call> t_calls;

std::mutex g_mu;
std::map<const void*, std::string> g_names; // kernels by host function
std::map<void*, size_t> g_mem[2];           // allocated: device, pinned host
std::map<hipStream_t, std::string> g_open;  // last kernel not waited for
std::deque<uint32_t> g_reads;               // next 4-byte copies to the host
std::string g_biggest, g_racing;
unsigned long long g_items = 0, g_launches = 0, g_free_bytes = 0, g_allocs = 0, g_frees = 0;
size_t g_limit = ~size_t(0); // device bytes that can be allocated
uintptr_t g_handle = 0x1000;

// a hipFree that waits until the test lets it go on, as one waits for a busy device
std::condition_variable g_cv;
bool g_hold = false;
std::atomic<int> g_held{0};

hipError_t reserve(int host, void** p, size_t bytes)
{
    std::lock_guard<std::mutex> lock(g_mu);
    size_t used = 0;
    for (const auto& m : g_mem[0])
        used += m.second;
    if (host == 0 && (bytes > g_limit || used > g_limit - bytes))
        return hipErrorOutOfMemory;
    const size_t n = (bytes + 4095) & ~size_t(4095);
    void* q = mmap(nullptr, n ? n : 4096, PROT_READ | PROT_WRITE,
                   MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
    if (q == MAP_FAILED)
        return hipErrorOutOfMemory;
    g_mem[host][q] = bytes;
    ++g_allocs;
    *p = q;
    return hipSuccess;
}
hipError_t give_back(int host, void* p)
{
    if (!p)
        return hipSuccess;
    std::unique_lock<std::mutex> lock(g_mu);
    if (host == 0 && g_hold)
    {
        ++g_held;
        g_cv.wait(lock, [] { return !g_hold; });
        --g_held;
    }
    auto it = g_mem[host].find(p);
    if (it == g_mem[host].end())
        return hipErrorInvalidValue;
    munmap(p, ((it->second + 4095) & ~size_t(4095)) ? (it->second + 4095) & ~size_t(4095) : 4096);
    g_free_bytes += it->second;
    ++g_frees;
    g_mem[host].erase(it);
    return hipSuccess;
}
void to_host(void* dst, size_t bytes)
{
    if (bytes == 4)
    {
        std::lock_guard<std::mutex> lock(g_mu);
        uint32_t v = 0;
        if (!g_reads.empty())
        {
            v = g_reads.front();
            g_reads.pop_front();
        }
        std::memcpy(dst, &v, 4);
    }
    else if (bytes <= 65536)
        std::memset(dst, 0, bytes);
}
// an operation of the null stream, which does not wait for the library's
// non-blocking streams
void null_stream(const char* what)
{
    std::lock_guard<std::mutex> lock(g_mu);
    for (const auto& o : g_open)
        if (!o.second.empty() && g_racing.empty())
            g_racing = std::string(what) + " beside " + o.second;
}
template <typename T> hipError_t handle(T* out)
{
    std::lock_guard<std::mutex> lock(g_mu);
    *out = reinterpret_cast<T>(g_handle += 16);
    return hipSuccess;
}
} // namespace

extern "C" {
// ---- what a test asks
void fake_reset()
{
    std::lock_guard<std::mutex> lock(g_mu);
    g_items = g_launches = g_free_bytes = g_allocs = g_frees = 0;
    g_biggest.clear();
    g_racing.clear();
    g_reads.clear();
    g_limit = ~size_t(0);
}
unsigned long long fake_items() { return g_items; }       // of the largest launch
const char* fake_biggest() { return g_biggest.c_str(); }  // its kernel
const char* fake_racing() { return g_racing.c_str(); }    // first unordered null-stream access
unsigned long long fake_launches() { return g_launches; }
unsigned long long fake_allocs() { return g_allocs; }
unsigned long long fake_frees() { return g_frees; }
int fake_unwaited() // streams with a kernel that was not waited for
{
    std::lock_guard<std::mutex> lock(g_mu);
    int n = 0;
    for (const auto& o : g_open)
        n += !o.second.empty();
    return n;
}
size_t fake_used(int host)
{
    std::lock_guard<std::mutex> lock(g_mu);
    size_t n = 0;
    for (const auto& m : g_mem[host])
        n += m.second;
    return n;
}
void fake_limit(size_t bytes) { g_limit = bytes; }
void fake_read(uint32_t v) { g_reads.push_back(v); }
void fake_hold(int on)
{
    {
        std::lock_guard<std::mutex> lock(g_mu);
        g_hold = on != 0;
    }
    g_cv.notify_all();
}
int fake_held() { return g_held; }

// ---- the runtime
void** __hipRegisterFatBinary(const void*)
{
    static void* h = nullptr;
    return &h;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* f, char*, const char* name, unsigned, void*, void*,
                           void*, void*, int*)
{
    std::lock_guard<std::mutex> lock(g_mu);
    g_names[f] = name;
}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t s, hipStream_t st)
{
    t_calls.push_back(Call{g, b, s, st});
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t* s, hipStream_t* st)
{
    const Call c = t_calls.back();
    t_calls.pop_back();
    *g = c.grid;
    *b = c.block;
    *s = c.shared;
    *st = c.stream;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void* f, dim3 g, dim3 b, void**, size_t, hipStream_t st)
{
    std::lock_guard<std::mutex> lock(g_mu);
    // the limit holds for each axis
    const unsigned long long n =
        std::max({(unsigned long long)g.x * b.x, (unsigned long long)g.y * b.y,
                  (unsigned long long)g.z * b.z});
    if (n > g_items)
    {
        g_items = n;
        g_biggest = g_names[f];
    }
    ++g_launches;
    g_open[st] = g_names[f];
    return hipSuccess;
}
hipError_t hipGetDeviceCount(int* n)
{
    *n = 1;
    return hipSuccess;
}
hipError_t hipGetDevice(int* d)
{
    *d = 0;
    return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
int hipGetStreamDeviceId(hipStream_t) { return 0; }
#undef hipGetDeviceProperties
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600* p, int)
{
    std::memset(p, 0, sizeof(*p));
    p->multiProcessorCount = 256;
    return hipSuccess;
}
const char* hipGetErrorString(hipError_t e) { return e == hipSuccess ? "ok" : "fake error"; }
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipGetSymbolAddress(void** p, const void*)
{
    static char array[64 << 20]; // never touched
    *p = array;
    return hipSuccess;
}
hipError_t hipMalloc(void** p, size_t n) { return reserve(0, p, n); }
hipError_t hipFree(void* p) { return give_back(0, p); }
hipError_t hipHostMalloc(void** p, size_t n, unsigned) { return reserve(1, p, n); }
hipError_t hipHostFree(void* p) { return give_back(1, p); }
hipError_t hipMemcpy(void* dst, const void*, size_t n, hipMemcpyKind k)
{
    null_stream("hipMemcpy");
    if (k == hipMemcpyDeviceToHost)
        to_host(dst, n);
    return hipSuccess;
}
hipError_t hipMemset(void*, int, size_t)
{
    null_stream("hipMemset");
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void* dst, const void*, size_t n, hipMemcpyKind k, hipStream_t)
{
    if (k == hipMemcpyDeviceToHost)
        to_host(dst, n);
    return hipSuccess;
}
hipError_t hipMemsetAsync(void*, int, size_t, hipStream_t) { return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { return handle(s); }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t s)
{
    std::lock_guard<std::mutex> lock(g_mu);
    g_open.erase(s);
    return hipSuccess;
}
hipError_t hipDeviceSynchronize()
{
    std::lock_guard<std::mutex> lock(g_mu);
    g_open.clear();
    return hipSuccess;
}
hipError_t hipStreamQuery(hipStream_t) { return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t* g) { return handle(g); }
hipError_t hipGraphInstantiate(hipGraphExec_t* x, hipGraph_t, hipGraphNode_t*, char*, size_t)
{
    return handle(x);
}
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipSuccess; }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) { return handle(e); }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return handle(e); }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t)
{
    *ms = 1.0f;
    return hipSuccess;
}
}

// A stand-in for the HIP runtime on the CPU: device memory is host memory (mapped, zero, not
// touched until used), copies happen at once, and kernels are recorded instead of run.  The
// library's host code linked against it can be made to see failed allocations and launches, an
// expired sweep, or a lack of host memory, and its launches, events and streams can be read back.
#include <hip/hip_runtime_api.h>
#include <sys/mman.h>
#include <unistd.h>

#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <new>
#include <string>

namespace {
struct State {
    std::mutex m;
    std::map<void*, size_t> mem;
    std::map<const void*, std::string> kernels;
    std::string log;
    long next_id = 1;
    int fail_malloc = -1;  // how many allocations still succeed (-1: all)
    int fail_launch = -1;
    hipError_t last = hipSuccess;
    int expire = 0;      // 1: sweeps raise their error flag; 2: and the norms come out NaN
    int graphs = 0;      // iterations can be captured
    bool capturing = false;
    int* captured = nullptr;  // the error flag of the captured sweeps
    int views = 0;       // repacked boxes so far: a read-back's box holds its number
    int slow_value = 0;  // copies to the host that start with this value are late
    dim3 grid, block;
    size_t shmem = 0;
    hipStream_t stream = nullptr;
};
State& st()
{
    static State* s = new State;
    return *s;
}
std::atomic<long> g_new_left{-1};  // operator new calls of the library that still succeed (-1: all)
thread_local int t_inside = 0;     // in the stand-in itself, whose own allocations do not count
struct Inside {
    std::unique_lock<std::mutex> g;
    Inside() : g((t_inside++, st().m)) {}
    ~Inside() { t_inside--; }
};

void note(const char* what, const std::string& a, const void* b)
{
    char t[64];
    std::snprintf(t, sizeof(t), " %p\n", b);
    st().log += what;
    st().log += " " + a + t;
}
std::string ptr(const void* p)
{
    char t[32];
    std::snprintf(t, sizeof(t), "%p", p);
    return t;
}
template <typename T>
T handle()
{
    Inside g;
    return (T)(st().next_id++ * 16);
}
hipError_t alloc(void** p, size_t n)
{
    Inside g;
    if (st().fail_malloc == 0) return st().last = hipErrorOutOfMemory;
    if (st().fail_malloc > 0) st().fail_malloc--;
    void* q = mmap(nullptr, n + 4096, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
    if (q == MAP_FAILED) return hipErrorOutOfMemory;
    st().mem[q] = n + 4096;
    *p = q;
    return hipSuccess;
}
hipError_t release(void* p)
{
    Inside g;
    auto q = st().mem.find(p);
    if (q == st().mem.end()) return p ? hipErrorInvalidValue : hipSuccess;
    munmap(q->first, q->second);
    st().mem.erase(q);
    return hipSuccess;
}
}  // namespace

// (bound inside this library only)
void* operator new(size_t n)
{
    long left = t_inside ? -1 : g_new_left.load();
    while (left > 0 && !g_new_left.compare_exchange_weak(left, left - 1)) {
    }
    if (left == 0) throw std::bad_alloc();
    if (void* p = std::malloc(n ? n : 1)) return p;
    throw std::bad_alloc();
}
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, size_t) noexcept { std::free(p); }

extern "C" {
// ---- controls
void stub_reset()
{
    State& s = st();
    Inside g;
    s.log.clear();
    s.fail_malloc = s.fail_launch = -1;
    s.expire = s.graphs = s.views = s.slow_value = 0;
    s.last = hipSuccess;
    g_new_left = -1;
}
void stub_fail_malloc(int after) { st().fail_malloc = after; }
void stub_fail_launch(int after) { st().fail_launch = after; }
void stub_fail_new(long after) { g_new_left = after; }
long stub_new_left() { return g_new_left; }
void stub_expire(int on) { st().expire = on; }
void stub_graphs(int on) { st().graphs = on; }
void stub_slow_value(int v) { st().slow_value = v; }
size_t stub_mapped()
{
    Inside g;
    return st().mem.size();
}
const char* stub_log() { return st().log.c_str(); }

// ---- the runtime
void** __hipRegisterFatBinary(const void*)
{
    static void* h = nullptr;
    return &h;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned, void*, void*, void*, void*, int*)
{
    Inside g;
    st().kernels[host] = name;
}
void __hipRegisterVar(void**, void*, char*, const char*, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t shmem, hipStream_t stream)
{
    State& s = st();
    s.grid = grid;
    s.block = block;
    s.shmem = shmem;
    s.stream = stream;
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* grid, dim3* block, size_t* shmem, hipStream_t* stream)
{
    State& s = st();
    *grid = s.grid;
    *block = s.block;
    *shmem = s.shmem;
    *stream = s.stream;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void* f, dim3, dim3, void** args, size_t, hipStream_t stream)
{
    State& s = st();
    Inside g;
    const std::string& name = s.kernels[f];
    note("launch", name, stream);
    if (s.fail_launch == 0) return s.last = hipErrorLaunchFailure;
    if (s.fail_launch > 0) s.fail_launch--;
    const bool wave = name.find("k_lusgs_wave") != std::string::npos;
    if (wave && s.capturing) s.captured = *(int**)args[6];
    if (s.capturing) return hipSuccess;
    if (wave && s.expire) **(int**)args[6] = 1;
    if (s.expire == 2 && name.find("k_norm_final") != std::string::npos) std::memset(*(void**)args[3], 0xff, 8);
    if (name.find("6k_viewILb0") != std::string::npos) {
        struct Box {
            double *field, *stage;
            long tot;
            int ncomp, n0, n1, cells;
        };
        const Box* b = (const Box*)args[0];
        s.views++;
        for (long q = 0; q < (long)b->cells * b->ncomp; q++) b->stage[q] = s.views;
    }
    return hipSuccess;
}
hipError_t hipGetLastError()
{
    const hipError_t e = st().last;
    st().last = hipSuccess;
    return e;
}
const char* hipGetErrorString(hipError_t) { return "stand-in error"; }
hipError_t hipGetDevice(int* d)
{
    *d = 0;
    return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipMalloc(void** p, size_t n) { return alloc(p, n); }
hipError_t hipFree(void* p) { return release(p); }
hipError_t hipHostMalloc(void** p, size_t n, unsigned) { return alloc(p, n); }
hipError_t hipHostFree(void* p) { return release(p); }
hipError_t hipGetSymbolAddress(void**, const void*) { return hipErrorInvalidSymbol; }
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind kind, hipStream_t)
{
    if (kind == hipMemcpyDeviceToHost && n >= 8 && st().slow_value && *(const double*)s == st().slow_value) usleep(20000);
    std::memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipMemsetAsync(void* p, int v, size_t n, hipStream_t)
{
    if (v == 0 && ((size_t)p & 4095) == 0 && n >= 4096) {  // (zero pages, not touched)
        const size_t whole = n / 4096 * 4096;
        madvise(p, whole, MADV_DONTNEED);
        std::memset((char*)p + whole, 0, n - whole);
    } else {
        std::memset(p, v, n);
    }
    return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned)
{
    *s = handle<hipStream_t>();
    Inside g;
    note("stream", "new", *s);
    return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned)
{
    Inside g;
    note("wait", ptr(e), s);
    return hipSuccess;
}
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode)
{
    st().capturing = st().graphs;
    return st().graphs ? hipSuccess : hipErrorNotSupported;
}
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t* g)
{
    st().capturing = false;
    *g = handle<hipGraph_t>();
    return hipSuccess;
}
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
hipError_t hipGraphInstantiate(hipGraphExec_t* x, hipGraph_t, hipGraphNode_t*, char*, size_t)
{
    *x = handle<hipGraphExec_t>();
    return hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t s)
{
    Inside g;
    note("launch", "graph", s);
    if (st().expire && st().captured) *st().captured = 1;
    return hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t* e)
{
    *e = handle<hipEvent_t>();
    return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s)
{
    Inside g;
    note("record", ptr(e), s);
    return hipSuccess;
}
hipError_t hipEventQuery(hipEvent_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t)
{
    *ms = 1.f;
    return hipSuccess;
}
}

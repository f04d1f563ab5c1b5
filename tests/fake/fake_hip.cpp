// A HIP runtime without a GPU, for tests of the library's host code: device
// memory is host memory, copies are made at once, and kernel launches only
// write a line to a log.  Loaded (RTLD_GLOBAL) before libp9idg.so, its symbols
// are the ones the library's calls bind to.
#include <hip/hip_runtime_api.h>

#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <string>
#include <vector>

namespace {

struct Fake {
    std::mutex m;
    std::map<const void*, std::string> kernels;  // host function -> name
    std::string log;
    std::map<void*, int> device_of;  // streams and events
    int devices = 2, device = 0;
    std::map<void*, size_t> blocks;
    size_t in_use = 0;
    // allocations of at least fail_from and at most fail_to bytes are refused
    size_t fail_from = ~(size_t)0, fail_to = 0;
    bool fail_pinned = false;
    // what analyse_kernel answers for every chunk, and how many of the next
    // deconvolver launches find their workgroups not all resident
    int nodes = 0, stalls = 0;
    hipError_t last = hipSuccess;
    dim3 grid, block;
    size_t shmem = 0;
    hipStream_t stream = nullptr;
};
Fake& fake() {
    static Fake* f = new Fake;  // used by other libraries' constructors
    return *f;
}
void note(const std::string& line) { fake().log += line + "\n"; }
std::string shape(dim3 g, dim3 b) {
    return std::to_string((size_t)g.x * g.y * g.z) + " x " + std::to_string((size_t)b.x * b.y * b.z);
}
template <typename T>
T handle(int device) {
    void* p = std::malloc(1);
    fake().device_of[p] = device;
    return reinterpret_cast<T>(p);
}
hipError_t launch(const char* how, const void* f, dim3 g, dim3 b, void** args, hipStream_t st) {
    Fake& k = fake();
    if (k.device_of[st] != k.device) return k.last = hipErrorInvalidHandle;
    const std::string name = k.kernels.count(f) ? k.kernels[f] : "?";
    note(how + name + " " + shape(g, b));
    // a launch has fewer than 2^32 threads in each dimension
    if ((size_t)g.x * b.x > 0xFFFFFFFFull) return k.last = hipErrorInvalidConfiguration;
    if (name.find("analyse_kernel") != std::string::npos) {
        int32_t* out = *static_cast<int32_t**>(args[4]);
        for (unsigned i = 0; i < g.x; i++) out[i] = k.nodes;
    }
    if (name.find("descent_kernel") != std::string::npos) {
        // the descent's argument block ends with the pointer to its results:
        // done, converged, updates, stalled
        int32_t* st = *reinterpret_cast<int32_t**>(static_cast<char*>(args[0]) + 96);
        std::memset(st, 0, 16);
        if (k.stalls > 0) {
            k.stalls--;
            st[3] = 1;
        } else {
            st[0] = 1;
            st[2] = 1;
        }
    }
    return hipSuccess;
}

}  // namespace

extern "C" {

// --- the tests' side
const char* fake_log() { return fake().log.c_str(); }
void fake_clear() { fake().log.clear(); }
void fake_fail_allocations(size_t from, size_t to) {
    fake().fail_from = from;
    fake().fail_to = to;
}
void fake_fail_pinned(int on) { fake().fail_pinned = on != 0; }
void fake_nodes(int n) { fake().nodes = n; }
void fake_stalls(int n) { fake().stalls = n; }
size_t fake_in_use() { return fake().in_use; }

// --- registration
void** __hipRegisterFatBinary(const void*) { return reinterpret_cast<void**>(std::malloc(sizeof(void*))); }
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned, void*, void*, void*, void*, int*) {
    fake().kernels[host] = name;
}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t shmem, hipStream_t st) {
    fake().grid = g;
    fake().block = b;
    fake().shmem = shmem;
    fake().stream = st;
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t* shmem, hipStream_t* st) {
    *g = fake().grid;
    *b = fake().block;
    *shmem = fake().shmem;
    *st = fake().stream;
    return hipSuccess;
}

// --- devices
hipError_t hipGetDeviceCount(int* n) {
    *n = fake().devices;
    return hipSuccess;
}
hipError_t hipGetDevice(int* d) {
    *d = fake().device;
    return hipSuccess;
}
hipError_t hipSetDevice(int d) {
    fake().device = d;
    return hipSuccess;
}
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t a, int) {
    *v = a == hipDeviceAttributeMultiprocessorCount ? 256 : 64;
    return hipSuccess;
}
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int* n, const void*, int, size_t) {
    *n = 2;
    return hipSuccess;
}
const char* hipGetErrorName(hipError_t) { return "hipError"; }
const char* hipGetErrorString(hipError_t) { return "fake error"; }
hipError_t hipGetLastError() {
    const hipError_t e = fake().last;
    fake().last = hipSuccess;
    return e;
}

// --- memory
hipError_t hipMalloc(void** p, size_t n) {
    Fake& f = fake();
    if (n >= f.fail_from && n <= f.fail_to) {
        note("refused " + std::to_string(n));
        return f.last = hipErrorOutOfMemory;
    }
    *p = std::calloc(n, 1);
    f.blocks[*p] = n;
    f.in_use += n;
    note("malloc " + std::to_string(n));
    return hipSuccess;
}
hipError_t hipFree(void* p) {
    Fake& f = fake();
    if (p) f.in_use -= f.blocks[p];
    f.blocks.erase(p);
    std::free(p);
    return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
    if (fake().fail_pinned) return hipErrorOutOfMemory;
    *p = std::calloc(n, 1);
    return hipSuccess;
}
hipError_t hipHostFree(void* p) {
    std::free(p);
    return hipSuccess;
}
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) {
    std::memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) {
    std::memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t) {
    std::memset(d, v, n);
    return hipSuccess;
}
hipError_t hipGetSymbolAddress(void**, const void*) { return hipErrorInvalidValue; }

// --- streams, events, graphs
hipError_t hipStreamCreate(hipStream_t* s) {
    *s = handle<hipStream_t>(fake().device);
    return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { return hipStreamCreate(s); }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) {
    note("begin capture");
    return hipSuccess;
}
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t* g) {
    note("end capture");
    *g = handle<hipGraph_t>(0);
    return hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t* e) {
    *e = handle<hipEvent_t>(fake().device);
    return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) {
    *ms = 1.f;
    return hipSuccess;
}
// an event can only be recorded on a stream of its own device
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
    Fake& f = fake();
    return f.device_of[e] == f.device_of[s] ? hipSuccess : hipErrorInvalidHandle;
}
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipGraphInstantiate(hipGraphExec_t* x, hipGraph_t, hipGraphNode_t*, char*, size_t) {
    *x = handle<hipGraphExec_t>(0);
    return hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipSuccess; }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }

// --- launches
hipError_t hipLaunchKernel(const void* f, dim3 g, dim3 b, void** args, size_t, hipStream_t st) { return launch("", f, g, b, args, st); }
hipError_t hipLaunchCooperativeKernel(const void* f, dim3 g, dim3 b, void** args, unsigned, hipStream_t st) {
    return launch("cooperative ", f, g, b, args, st);
}

// --- hipFFT
int hipfftPlan2d(void** p, int, int, int) {
    *p = nullptr;
    return 0;
}
int hipfftSetStream(void*, hipStream_t) { return 0; }
int hipfftDestroy(void*) { return 0; }
int hipfftExecC2C(void*, void*, void*, int) {
    note("hipfftExecC2C");
    return 0;
}
int hipfftExecZ2Z(void*, void*, void*, int) {
    note("hipfftExecZ2Z");
    return 0;
}

}  // extern "C"

// The HIP runtime calls of the library, answered on the host (test infrastructure): device memory is
// host memory, copies run at once, kernels do not run. It lets the CPU tests drive the library's own
// staging, launches and error exits and look at what they would have given the GPU:
// - every kernel launch is handed to a callback with its name and arguments;
// - every operation is pending from its enqueue until a call waits for it (streams, events and
//   stream waits are followed with one counter per stream), so a test can ask what a call left
//   in flight;
// - a named call can be made to fail;
// - a capture in global mode by another part of the program can be under way: calls that wait or allocate are
//   then refused, and end that capture, unless their thread has relaxed its mode.
// One thread at a time.
#include <hip/hip_runtime_api.h>

#include <algorithm>
#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <map>
#include <string>
#include <utility>
#include <vector>

struct ihipStream_t {
    size_t id;
};
struct ihipEvent_t {
    std::vector<uint64_t> snap;  // per stream: the operations it stands for
};

namespace {

// Made on first use: the code objects register themselves while the library is being loaded.
std::map<uintptr_t, size_t>& blocks() {  // device and pinned allocations
    static std::map<uintptr_t, size_t> m;
    return m;
}
std::map<const void*, std::string>& kernels() {  // host stub -> device name
    static std::map<const void*, std::string> m;
    return m;
}
std::map<const void*, void*>& vars() {  // host shadow -> block
    static std::map<const void*, void*> m;
    return m;
}
std::map<std::string, int> g_fail;  // call -> calls until it fails once
hipError_t g_last = hipSuccess;      // set by failed launches only
void (*g_on_launch)(const char*, void**) = nullptr;

bool g_capture = false, g_capture_ended = false;
hipStreamCaptureMode g_mode = hipStreamCaptureModeGlobal;  // the calling thread's
// Whether a call that a capture forbids is refused now.
bool forbidden() {
    if (!g_capture || g_mode == hipStreamCaptureModeRelaxed) return false;
    return g_capture_ended = true;
}

// Streams by id: operations issued, those known complete, and what each stream has waited for.
std::vector<uint64_t> g_issued, g_done;
std::vector<std::vector<uint64_t>> g_front;
struct HostRange {
    size_t stream;
    uint64_t seq;
    const char* lo;
    size_t bytes;
};
std::vector<HostRange> g_host;  // host memory that asynchronous copies read or write

uint64_t& slot(std::vector<uint64_t>& v, size_t i) {
    if (v.size() <= i) v.resize(i + 1, 0);
    return v[i];
}
void merge(std::vector<uint64_t>& into, const std::vector<uint64_t>& from) {
    for (size_t i = 0; i < from.size(); i++) slot(into, i) = std::max(slot(into, i), from[i]);
}
std::vector<uint64_t>& front(size_t stream) {
    if (g_front.size() <= stream) g_front.resize(stream + 1);
    slot(g_front[stream], stream) = slot(g_issued, stream);
    return g_front[stream];
}
size_t id_of(hipStream_t s) { return s ? s->id : 0; }
uint64_t issue(hipStream_t s) { return ++slot(g_issued, id_of(s)); }
void complete_all() { merge(g_done, g_issued); }

// Whether this call of `name` is the one told to fail.
bool failing(const std::string& name) {
    auto it = g_fail.find(name);
    if (it == g_fail.end() || --it->second > 0) return false;
    g_fail.erase(it);
    return true;
}
hipError_t get_block(void** p, size_t n) {
    *p = std::calloc(n ? n : 1, 1);
    if (!*p) return hipErrorOutOfMemory;
    blocks()[reinterpret_cast<uintptr_t>(*p)] = n;
    return hipSuccess;
}
void drop_block(void* p) {
    complete_all();  // a free waits for the device
    blocks().erase(reinterpret_cast<uintptr_t>(p));
    std::free(p);
}
hipError_t run_kernel(const void* f, void** args, hipStream_t s) {
    const std::string& name = kernels()[f];
    for (auto& kv : g_fail)
        if (kv.first.rfind("kernel:", 0) == 0 && name.find(kv.first.substr(7)) != std::string::npos) {
            if (failing(std::string(kv.first))) return g_last = hipErrorLaunchFailure;
            break;
        }
    issue(s);
    if (g_on_launch) g_on_launch(name.c_str(), args);
    return hipSuccess;
}

struct CallConfig {
    dim3 grid, block;
    size_t lds;
    hipStream_t stream;
} g_call;

}  // namespace

extern "C" {

// ---- what the tests ask

// Operations enqueued and not yet waited for.
uint64_t host_hip_pending(void) {
    uint64_t n = 0;
    for (size_t i = 0; i < g_issued.size(); i++) n += g_issued[i] - slot(g_done, i);
    return n;
}
// Pending copies that read or write host bytes [p, p + n).
uint64_t host_hip_pending_copies(const char* p, size_t n) {
    uint64_t k = 0;
    for (const HostRange& r : g_host)
        if (r.seq > slot(g_done, r.stream) && r.lo < p + n && p < r.lo + r.bytes) k++;
    return k;
}
// The allocation that holds p: its first byte and size, or 0.
int host_hip_block(const void* p, void** base, size_t* bytes) {
    auto it = blocks().upper_bound(reinterpret_cast<uintptr_t>(p));
    if (it == blocks().begin()) return 0;
    --it;
    if (reinterpret_cast<uintptr_t>(p) - it->first >= it->second) return 0;
    *base = reinterpret_cast<void*>(it->first);
    *bytes = it->second;
    return 1;
}
// The n-th call of `name` from now fails once ("kernel:<part of a kernel's name>" for a launch).
void host_hip_fail(const char* name, int n) { g_fail[name] = n; }
// Begins (1) or ends (0) a capture elsewhere in the program; returns whether one that ran was undisturbed.
int host_hip_capture(int on) {
    const bool whole = !g_capture_ended;
    g_capture = on;
    g_capture_ended = false;
    return whole && g_mode == hipStreamCaptureModeGlobal;
}
void host_hip_on_launch(void (*f)(const char*, void**)) { g_on_launch = f; }

// ---- the calls of the library

hipError_t hipGetDeviceCount(int* n) { return *n = 1, hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDevice(int* d) { return *d = 0, hipSuccess; }
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int) { return *v = 256, hipSuccess; }
hipError_t hipGetDeviceProperties(hipDeviceProp_t* p, int) {
    *p = hipDeviceProp_t{};
    std::strcpy(p->name, "host");
    std::strcpy(p->gcnArchName, "gfx950");
    return hipSuccess;
}
hipError_t hipFuncSetAttribute(const void*, hipFuncAttribute, int) { return hipSuccess; }
const char* hipGetErrorString(hipError_t e) {
    return e == hipSuccess ? "success" : e == hipErrorInvalidValue ? "invalid argument" : "failed by the test";
}
hipError_t hipGetLastError(void) {
    const hipError_t e = g_last;
    g_last = hipSuccess;
    return e;
}

hipError_t hipMalloc(void** p, size_t n) {
    if (forbidden()) return hipErrorStreamCaptureUnsupported;
    return failing("hipMalloc") ? hipErrorOutOfMemory : get_block(p, n);
}
hipError_t hipFree(void* p) { return p ? drop_block(p) : void(), hipSuccess; }
hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
    return failing("hipHostMalloc") ? hipErrorOutOfMemory : get_block(p, n);
}
hipError_t hipHostFree(void* p) { return hipFree(p); }
hipError_t hipGetSymbolAddress(void** p, const void* var) { return *p = vars()[var], *p ? hipSuccess : hipErrorInvalidSymbol; }

hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) {
    if (failing("hipMemcpy")) return hipErrorInvalidValue;
    if (n) std::memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind kind, hipStream_t st) {
    if (failing("hipMemcpyAsync")) return hipErrorInvalidValue;
    if (n) std::memcpy(d, s, n);
    const uint64_t seq = issue(st);
    if (kind != hipMemcpyDeviceToDevice)
        g_host.push_back({id_of(st), seq, static_cast<const char*>(kind == hipMemcpyHostToDevice ? s : d), n});
    return hipSuccess;
}
hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t st) {
    std::memset(d, v, n);
    issue(st);
    return hipSuccess;
}

hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) {
    static size_t next = 1;
    *s = new ihipStream_t{next++};
    return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t s) { return delete s, hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t s) {
    if (forbidden()) return hipErrorStreamCaptureUnsupported;
    if (failing("hipStreamSynchronize")) return hipErrorUnknown;
    merge(g_done, front(id_of(s)));
    return hipSuccess;
}
hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned) { return merge(front(id_of(s)), e->snap), hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return *e = new ihipEvent_t, hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) { return *e = new ihipEvent_t, hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t e) { return delete e, hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
    if (failing("hipEventRecord")) return hipErrorUnknown;
    e->snap = front(id_of(s));
    return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t e) {
    if (forbidden()) return hipErrorStreamCaptureUnsupported;
    if (failing("hipEventSynchronize")) return hipErrorUnknown;
    return merge(g_done, e->snap), hipSuccess;
}
hipError_t hipEventQuery(hipEvent_t e) {
    if (forbidden()) return hipErrorStreamCaptureUnsupported;
    for (size_t i = 0; i < e->snap.size(); i++)
        if (e->snap[i] > slot(g_done, i)) return hipErrorNotReady;
    return hipSuccess;
}
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) { return *ms = 1.0f, hipSuccess; }

hipError_t hipThreadExchangeStreamCaptureMode(hipStreamCaptureMode* m) { return std::swap(*m, g_mode), hipSuccess; }
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t* g) { return *g = nullptr, hipSuccess; }
hipError_t hipGraphInstantiate(hipGraphExec_t* x, hipGraph_t, hipGraphNode_t*, char*, size_t) {
    *x = reinterpret_cast<hipGraphExec_t>(&g_call);
    return hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t s) { return issue(s), hipSuccess; }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }

hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t lds, hipStream_t s) {
    g_call = {grid, block, lds, s};
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* grid, dim3* block, size_t* lds, hipStream_t* s) {
    *grid = g_call.grid;
    *block = g_call.block;
    *lds = g_call.lds;
    *s = g_call.stream;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void* f, dim3, dim3, void** args, size_t, hipStream_t s) { return run_kernel(f, args, s); }
hipError_t hipExtLaunchKernel(const void* f, dim3, dim3, void** args, size_t, hipStream_t s, hipEvent_t a, hipEvent_t b, int) {
    const hipError_t e = run_kernel(f, args, s);
    for (hipEvent_t ev : {a, b})
        if (ev) ev->snap = front(id_of(s));
    return e;
}

void** __hipRegisterFatBinary(const void*) {
    static void* handle = nullptr;
    return &handle;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned, void*, void*, void*, void*, int*) {
    kernels()[host] = name;
}
void __hipRegisterVar(void**, void* host, char*, char*, int, size_t bytes, int, int) { (void)get_block(&vars()[host], bytes); }

}  // extern "C"

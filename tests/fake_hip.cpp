/* A HIP runtime without a GPU, for tests of the library's host code on the CPU: loaded ahead of libsmq_gfx950.so with
 * RTLD_GLOBAL, it takes the place of the runtime's functions. Device addresses are numbers without memory behind them,
 * kernels are only recorded (fake_log: name, grid, stream), and the score workspaces of the attention kernels
 * are followed:
 *  - every access is ordered against the last one of each other stream by what the host did (stream order, events,
 *    waits, synchronizations), or fake_errors says "race";
 *  - an access to freed memory, a replay of a destroyed graph and a forbidden call inside a capture are errors too.
 * Freed graph handles are used again at once, as an allocator may. */
#define __HIP_PLATFORM_AMD__ 1
#include <hip/hip_runtime_api.h>

#include <cstdint>
#include <cstring>
#include <map>
#include <string>
#include <thread>
#include <vector>

namespace {

typedef std::map<void *, uint64_t> Clock; /* stream -> launches known to be complete or before */
struct Stream {
    bool capturing = false;
    std::thread::id by;
    bool invalid = false;
};
struct Node {
    std::string name;
    uint32_t grid, block;
    void *ws;
};
struct Graph {
    std::vector<Node> nodes;
    bool dead = false;
};

std::map<const void *, std::string> names;
std::map<void *, Stream> streams;
std::map<void *, Clock> seen; /* per stream: what its next launch comes after */
Clock host;
std::map<void *, uint64_t> launches;
std::map<void *, Clock> events;
std::map<uintptr_t, size_t> memory;
std::map<void *, Clock> touched; /* workspace -> stream -> launch number of the last access */
std::map<void *, std::vector<Node>> recording;
std::map<void *, Graph> execs;
std::vector<void *> free_execs;
std::string log_text, error_text;
uintptr_t next_address = 0x100000000000ull, next_handle = 0x1000;
size_t fail_size = 0;
uint64_t allocations = 0, frees = 0;
void (*on_exec_destroy)() = nullptr, (*on_is_capturing)() = nullptr; /* called once: what another thread may do there */
hipError_t last = hipSuccess;
struct Config {
    dim3 grid, block;
    size_t lds;
    hipStream_t s;
};
thread_local std::vector<Config> configs;

hipError_t ret(hipError_t e) {
    if (e != hipSuccess) last = e;
    return e;
}
void error(const std::string &s) { error_text += s + "\n"; }
void merge(Clock &a, const Clock &b) {
    for (auto &x : b)
        if (a[x.first] < x.second) a[x.first] = x.second;
}
void once(void (*&hook)()) {
    void (*f)() = hook;
    hook = nullptr;
    if (f) f();
}
bool forbidden() { /* inside a capture of this thread */
    for (auto &s : streams)
        if (s.second.capturing && s.second.by == std::this_thread::get_id()) {
            s.second.invalid = true;
            error("a call that a capture does not allow");
            return true;
        }
    return false;
}
bool live(void *p) {
    auto it = memory.upper_bound((uintptr_t)p);
    if (it == memory.begin()) return false;
    --it;
    return (uintptr_t)p < it->first + it->second;
}
/* the workspace argument of the kernels that have one */
void *workspace(const std::string &n, void **args) {
    auto has = [&](const char *k) { return n.find(k) != std::string::npos; };
    if (has("k_attend_scores_hd")) return *(void **)args[6];
    if (has("k_attend_scores")) return *(void **)args[8];
    if (has("k_attend_values")) return *(void **)args[8];
    if (has("k_ap_")) return *(void **)((char *)args[0] + 56); /* PreArgs::ws */
    return nullptr;
}
void run(const Node &n, void *s) {
    char line[400];
    snprintf(line, sizeof(line), "%s grid %u block %u stream %p ws %p\n", n.name.c_str(), n.grid, n.block, s, n.ws);
    log_text += line;
    merge(seen[s], host);
    const uint64_t me = ++launches[s];
    seen[s][s] = me;
    if (!n.ws) return;
    if (!live(n.ws)) error("a kernel uses freed memory: " + n.name);
    for (auto &t : touched[n.ws])
        if (t.first != s && seen[s][t.first] < t.second) error("race: " + n.name);
    touched[n.ws][s] = me;
}

}  // namespace

extern "C" {

const char *fake_log() { return log_text.c_str(); }
const char *fake_errors() { return error_text.c_str(); }
void fake_clear() { log_text.clear(), error_text.clear(); }
void fake_fail_size(size_t n) { fail_size = n; }
uint64_t fake_allocations() { return allocations; }
uint64_t fake_frees() { return frees; }
void fake_on_exec_destroy(void (*f)()) { on_exec_destroy = f; }
void fake_on_is_capturing(void (*f)()) { on_is_capturing = f; }

void **__hipRegisterFatBinary(const void *) {
    static void *h[1];
    return h;
}
void __hipRegisterFunction(void **, const void *host_fn, char *, const char *name, unsigned, void *, void *, void *, void *,
                           int *) {
    names[host_fn] = name;
}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
void __hipUnregisterFatBinary(void **) {}
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t lds, hipStream_t s) {
    configs.push_back({g, b, lds, s});
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *lds, hipStream_t *s) {
    *g = configs.back().grid, *b = configs.back().block, *lds = configs.back().lds, *s = configs.back().s;
    configs.pop_back();
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void *f, dim3 g, dim3 b, void **args, size_t, hipStream_t s) {
    if (!g.x || !g.y || !g.z) return ret(hipErrorInvalidConfiguration);
    const Node n = {names[f], g.x, b.x, workspace(names[f], args)};
    if (streams[s].capturing) recording[s].push_back(n);
    else run(n, s);
    return hipSuccess;
}

hipError_t hipGetDeviceCount(int *n) { return *n = 1, hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDevice(int *d) { return *d = 0, hipSuccess; }
hipError_t hipGetDeviceProperties(hipDeviceProp_t *p, int) {
    memset(p, 0, sizeof(*p));
    strcpy(p->gcnArchName, "gfx950:sramecc+:xnack-");
    return hipSuccess;
}
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t a, int) {
    *v = a == hipDeviceAttributeMultiprocessorCount ? 256 : 1;
    return hipSuccess;
}
const char *hipGetErrorString(hipError_t e) { return e == hipErrorOutOfMemory ? "out of memory" : "fake error"; }
hipError_t hipGetLastError() {
    const hipError_t e = last;
    last = hipSuccess;
    return e;
}
hipError_t hipFuncSetAttribute(const void *, hipFuncAttribute, int) { return hipSuccess; }
hipError_t hipFuncGetAttributes(hipFuncAttributes *a, const void *) { return memset(a, 0, sizeof(*a)), hipSuccess; }
hipError_t hipGetSymbolAddress(void **p, const void *) { return *p = (void *)0x10000, hipSuccess; }
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int *n, const void *, int, size_t) { return *n = 4, hipSuccess; }

hipError_t hipMalloc(void **p, size_t n) {
    if (forbidden()) return ret(hipErrorStreamCaptureUnsupported);
    if (fail_size && n == fail_size) return ret(hipErrorOutOfMemory);
    ++allocations;
    *p = (void *)next_address;
    memory[next_address] = n;
    next_address += (n + 0xffff) & ~(uintptr_t)0xffff;
    return hipSuccess;
}
hipError_t hipFree(void *p) {
    if (!p) return hipSuccess;
    if (forbidden()) return ret(hipErrorStreamCaptureUnsupported);
    ++frees;
    if (!memory.erase((uintptr_t)p)) error("a free of no allocation");
    for (auto &s : seen) merge(host, s.second); /* waits for the device */
    return hipSuccess;
}
hipError_t hipMemGetAddressRange(hipDeviceptr_t *base, size_t *n, hipDeviceptr_t p) {
    if (!live(p)) return ret(hipErrorNotFound);
    auto it = --memory.upper_bound((uintptr_t)p);
    *base = (hipDeviceptr_t)it->first, *n = it->second;
    return hipSuccess;
}
hipError_t hipMemset(void *, int, size_t) { return hipSuccess; }
hipError_t hipMemsetAsync(void *, int, size_t, hipStream_t) { return hipSuccess; }
hipError_t hipMemcpy(void *d, const void *, size_t n, hipMemcpyKind k) {
    if (k == hipMemcpyDeviceToHost) memset(d, 0, n);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind k, hipStream_t) { return hipMemcpy(d, s, n, k); }

hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) {
    *s = (hipStream_t)(next_handle += 0x10);
    streams[*s] = Stream();
    return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t s) { return streams.erase(s), hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t s) {
    if (streams[s].capturing) return ret(hipErrorStreamCaptureUnsupported);
    merge(host, seen[s]);
    return hipSuccess;
}
hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned) { return merge(seen[s], events[e]), hipSuccess; }
hipError_t hipEventCreate(hipEvent_t *e) {
    *e = (hipEvent_t)(next_handle += 0x10);
    return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
    if (streams[s].capturing) {
        error("an event recorded into a capture");
        return ret(hipErrorStreamCaptureUnsupported);
    }
    merge(seen[s], host);
    events[e] = seen[s];
    return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t e) { return merge(host, events[e]), hipSuccess; }
hipError_t hipEventQuery(hipEvent_t e) { /* complete once the host has waited for what it covers */
    for (auto &x : events[e])
        if (host[x.first] < x.second) return hipErrorNotReady;
    return hipSuccess;
}
hipError_t hipEventElapsedTime(float *t, hipEvent_t, hipEvent_t) { return *t = 1.0f, hipSuccess; }

hipError_t hipStreamBeginCapture(hipStream_t s, hipStreamCaptureMode) {
    if (streams[s].capturing) return ret(hipErrorIllegalState);
    streams[s].capturing = true;
    streams[s].by = std::this_thread::get_id();
    streams[s].invalid = false;
    recording[s].clear();
    return hipSuccess;
}
hipError_t hipStreamIsCapturing(hipStream_t s, hipStreamCaptureStatus *c) {
    *c = !streams[s].capturing ? hipStreamCaptureStatusNone
                               : streams[s].invalid ? hipStreamCaptureStatusInvalidated : hipStreamCaptureStatusActive;
    once(on_is_capturing);
    return hipSuccess;
}
hipError_t hipStreamEndCapture(hipStream_t s, hipGraph_t *g) {
    Stream &t = streams[s];
    if (!t.capturing) return ret(hipErrorIllegalState);
    if (t.by != std::this_thread::get_id()) return ret(hipErrorStreamCaptureWrongThread);
    t.capturing = false;
    if (t.invalid) return ret(hipErrorStreamCaptureInvalidated);
    *g = (hipGraph_t) new Graph{recording[s], false};
    return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t *e, hipGraph_t g, hipGraphNode_t *, char *, size_t) {
    void *h = (void *)(next_handle += 0x10);
    if (!free_execs.empty()) {
        h = free_execs.back();
        free_execs.pop_back();
    }
    execs[h] = *(Graph *)g;
    *e = (hipGraphExec_t)h;
    return hipSuccess;
}
hipError_t hipGraphDestroy(hipGraph_t g) { return delete (Graph *)g, hipSuccess; }
hipError_t hipGraphLaunch(hipGraphExec_t e, hipStream_t s) {
    if (!execs.count(e) || execs[e].dead) return error("a destroyed graph is replayed"), ret(hipErrorInvalidValue);
    for (auto &n : execs[e].nodes) run(n, s);
    return hipSuccess;
}
hipError_t hipGraphExecDestroy(hipGraphExec_t e) {
    if (!execs.count(e)) return ret(hipErrorInvalidValue);
    execs[e].dead = true;
    free_execs.push_back(e);
    once(on_exec_destroy);
    return hipSuccess;
}

}  // extern "C"

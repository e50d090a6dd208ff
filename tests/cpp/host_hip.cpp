// host_hip.cpp — the HIP runtime calls of libsli.so on host memory, for CPU tests of the engine's host side: which device
// is current at an allocation or a launch, what a failed allocation leaves, what is still to be read of a caller's
// memory when a call returns, what is launched and what is replayed. Kernels do nothing. Copies wait in their stream until it is
// synchronised, as the runtime may leave them. Loaded with RTLD_GLOBAL before libsli.so, whose references then find these.
#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <map>
#include <set>
#include <string>
#include <vector>

namespace {
constexpr int kOk = 0, kInvalid = 1, kOom = 2;
enum { kH2D = 1, kD2H = 2 };
struct Stream {
    int device;
    bool capturing = false;
    std::vector<std::function<void()>> todo;
    int host_reads = 0;  // queued copies out of host memory
};
thread_local int current = 0;
thread_local int last_error = kOk;
struct Dim3 {
    uint32_t x, y, z;
};
thread_local struct {
    Dim3 g, b;
    size_t sh;
    void* s;
} config;
int wrong_device = 0, launches = 0, graph_launches = 0, mallocs = 0, memsets = 0, fail_at = -1;
bool xcds = false;
std::string fail_launch;
size_t room = (size_t)-1, used = 0, free_bytes = (size_t)1 << 36;
std::map<int, int> mallocs_on, attributes_on;
std::map<void*, size_t> live;
std::set<Stream*> streams;
std::map<const void*, std::string> kernels;
std::set<std::string> launched;
std::string names;

int done(int e) {
    if (e != kOk) last_error = e;
    return e;
}
void drain(Stream* s) {
    for (auto& f : s->todo) f();
    s->todo.clear();
    s->host_reads = 0;
}
int queue(void* stream, bool reads_host, std::function<void()> f) {
    Stream* s = (Stream*)stream;
    if (!s) {
        f();
        return kOk;
    }
    if (s->capturing) return kOk;
    s->todo.push_back(std::move(f));
    s->host_reads += reads_host;
    return kOk;
}
}  // namespace

extern "C" {
// ---- what the tests read and set
int hh_wrong_device() { return wrong_device; }
int hh_launches() { return launches; }
int hh_graph_launches() { return graph_launches; }
int hh_mallocs() { return mallocs; }
int hh_mallocs_on(int d) { return mallocs_on[d]; }
int hh_attributes_on(int d) { return attributes_on[d]; }
int hh_live() { return (int)live.size(); }
void hh_fail_at(int k) { fail_at = k < 0 ? -1 : mallocs + k; }  // the k-th allocation from now (0: the next) fails
void hh_free(size_t n) { free_bytes = n ? n : (size_t)1 << 36; }  // what hipMemGetInfo tells (0: 64 GiB)
void hh_room(size_t n) { room = n ? used + n : (size_t)-1; }    // bytes left to allocate (0: no limit)
int hh_memsets() { return memsets; }                           // of streams
void hh_xcds(int on) { xcds = on; }                            // workgroups go to eight XCDs in turn (what xcd_kernel counts)
void hh_fail_launch(const char* name) { fail_launch = name; }  // the next launch of such a kernel fails
const char* hh_launched() {  // the kernels launched or recorded since the last call, one name a line
    names.clear();
    for (auto& n : launched) names += n + "\n";
    launched.clear();
    return names.c_str();
}
const char* hh_kernels() {  // those that the loaded libraries hold
    names.clear();
    for (auto& k : kernels) names += k.second + "\n";
    return names.c_str();
}
int hh_pending_host_reads() {
    int n = 0;
    for (Stream* s : streams) n += s->host_reads;
    return n;
}

// ---- the runtime
int hipGetDevice(int* d) { return *d = current, kOk; }
int hipSetDevice(int d) { return d < 0 || d >= 8 ? done(kInvalid) : (current = d, kOk); }
int hipGetDeviceCount(int* n) { return *n = 8, kOk; }
int hipDeviceGetAttribute(int* v, int, int) { return *v = 256, kOk; }
const char* hipGetErrorString(int e) { return e == kOom ? "out of memory" : "error"; }
int hipGetLastError() {
    const int e = last_error;
    last_error = kOk;
    return e;
}
int hipMalloc(void** p, size_t n) {
    const int i = mallocs++;
    *p = nullptr;
    if (i == fail_at || used + n > room) return done(kOom);
    ++mallocs_on[current];
    live[*p = calloc(1, n ? n : 1)] = n;
    used += n;
    return kOk;
}
int hipExtMallocWithFlags(void** p, size_t n, unsigned) { return hipMalloc(p, n); }
int hipFree(void* p) {
    if (!p) return kOk;
    for (Stream* s : streams) drain(s);
    const auto it = live.find(p);
    if (it == live.end()) return done(kInvalid);
    used -= it->second;
    live.erase(it);
    free(p);
    return kOk;
}
int hipMemGetInfo(size_t* f, size_t* t) { return *f = free_bytes, *t = (size_t)1 << 36, kOk; }
int hipMemcpy(void* d, const void* s, size_t n, int) { return memcpy(d, s, n), kOk; }
int hipMemset(void* d, int v, size_t n) { return memset(d, v, n), kOk; }
int hipMemcpyAsync(void* d, const void* s, size_t n, int kind, void* st) {
    return queue(st, kind == kH2D, [=] { memcpy(d, s, n); });
}
int hipMemcpy2DAsync(void* d, size_t dp, const void* s, size_t sp, size_t w, size_t h, int kind, void* st) {
    return queue(st, kind == kH2D, [=] {
        for (size_t i = 0; i < h; ++i) memcpy((char*)d + i * dp, (const char*)s + i * sp, w);
    });
}
int hipMemsetAsync(void* d, int v, size_t n, void* st) {
    ++memsets;
    return queue(st, false, [=] { memset(d, v, n); });
}
int hipStreamCreateWithFlags(void** s, unsigned) {
    Stream* n = new Stream{current};
    streams.insert(n);
    return *s = n, kOk;
}
int hipStreamDestroy(void* s) {
    drain((Stream*)s);
    streams.erase((Stream*)s);
    delete (Stream*)s;
    return kOk;
}
int hipStreamSynchronize(void* s) {
    if (s) drain((Stream*)s);
    return kOk;
}
int hipStreamQuery(void* s) { return hipStreamSynchronize(s); }
int hipStreamBeginCapture(void* s, int) { return ((Stream*)s)->capturing = true, kOk; }
int hipStreamEndCapture(void* s, void** g) {
    ((Stream*)s)->capturing = false;
    return *g = malloc(1), kOk;
}
int hipGraphInstantiate(void** e, void*, void**, char*, size_t) { return *e = malloc(1), kOk; }
int hipGraphDestroy(void* g) { return free(g), kOk; }
int hipGraphExecDestroy(void* e) { return free(e), kOk; }
int hipGraphLaunch(void*, void*) { return ++graph_launches, kOk; }
int hipFuncSetAttribute(const void*, int, int) { return ++attributes_on[current], kOk; }
int hipLaunchKernel(const void* f, Dim3 grid, Dim3, void** args, size_t, void* st) {
    if (!fail_launch.empty() && kernels[f].find(fail_launch) != std::string::npos) return fail_launch.clear(), done(kInvalid);
    if (xcds && kernels[f].find("xcd_kernel") != std::string::npos)
        for (int i = 0; i < 8; ++i) (*(uint32_t**)args[0])[i] = grid.x / 8;
    Stream* s = (Stream*)st;
    if (s && s->device != current) ++wrong_device;
    if (!s || !s->capturing) ++launches;
    launched.insert(kernels[f]);
    return kOk;
}
int __hipPushCallConfiguration(Dim3 g, Dim3 b, size_t sh, void* s) { return config = {g, b, sh, s}, kOk; }
int __hipPopCallConfiguration(Dim3* g, Dim3* b, size_t* sh, void** s) {
    return *g = config.g, *b = config.b, *sh = config.sh, *s = config.s, kOk;
}
void** __hipRegisterFatBinary(const void*) { return (void**)malloc(8); }
void __hipRegisterFunction(void**, const void* f, char*, const char* name, unsigned, void*, void*, void*, void*, int*) {
    kernels[f] = name;
}
void __hipUnregisterFatBinary(void** m) { free(m); }
int hipEventCreate(void** e) { return *e = malloc(1), kOk; }
int hipEventDestroy(void* e) { return free(e), kOk; }
int hipEventRecord(void*, void*) { return kOk; }
int hipEventSynchronize(void*) {
    for (Stream* s : streams) drain(s);
    return kOk;
}
int hipEventQuery(void* e) { return hipEventSynchronize(e); }
int hipEventElapsedTime(float* ms, void*, void*) { return *ms = 1.0f, kOk; }
}

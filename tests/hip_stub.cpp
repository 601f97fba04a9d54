// A host stand-in for the HIP runtime calls libaem.so makes: device memory is
// host memory, kernels do nothing but are counted by name, and a chosen call of
// a chosen function fails, as when memory runs out.  It lets the CPU tests take
// libaem's error paths and see which kernels a deck's steps launch.  Loaded with
// RTLD_GLOBAL before libaem.so, whose references then bind to these definitions.
#include <cstddef>
#include <cstdlib>
#include <cstring>
#include <map>
#include <string>

namespace {
constexpr int kOutOfMemory = 2, kCaptureUnsupported = 900, kIllegalState = 401;
std::string fail_name;
long fail_left = 0;      // > 0: the fail_left-th call of fail_name from now fails
int last_error = 0;
long live_graphs = 0, live_allocs = 0;
std::map<const void*, std::string> kernels;
std::map<std::string, long> calls;   // kernel launches by mangled name, runtime calls by name

struct Stream {
    bool capturing = false;
};
struct Event {};

int error(int e) {
    last_error = e;
    return e;
}
int enter(const char* name) {
    ++calls[name];
    if (fail_left > 0 && fail_name == name && --fail_left == 0) return error(kOutOfMemory);
    return 0;
}
// host and device meet here: not allowed while the stream is captured
int meet(const char* name, void* s) {
    if (int e = enter(name)) return e;
    if (s && static_cast<Stream*>(s)->capturing) return error(kCaptureUnsupported);
    return 0;
}
}  // namespace

extern "C" {

void stub_fail(const char* name, long nth) {
    fail_name = name;
    fail_left = nth;
}
long stub_pending() { return fail_left; }
long stub_graphs() { return live_graphs; }
long stub_allocs() { return live_allocs; }
// calls of a runtime function, or launches of the kernels whose mangled name
// holds `name` (with its length before it, as "9k_e_slabs")
long stub_calls(const char* name) {
    long n = 0;
    for (const auto& c : calls)
        if (c.first == name || (name[0] <= '9' && c.first.find(name) != std::string::npos)) n += c.second;
    return n;
}
void stub_forget() { calls.clear(); }

int hipMalloc(void** p, size_t n) {
    if (int e = enter("hipMalloc")) return e;
    *p = std::calloc(n, 1);
    ++live_allocs;
    return 0;
}
int hipFree(void* p) {
    if (p) --live_allocs;
    std::free(p);
    return 0;
}
int hipHostMalloc(void** p, size_t n, unsigned) {
    *p = std::calloc(n, 1);
    return 0;
}
int hipHostFree(void* p) {
    std::free(p);
    return 0;
}
int hipMemcpy(void* d, const void* s, size_t n, int) {
    if (int e = enter("hipMemcpy")) return e;
    std::memcpy(d, s, n);
    return 0;
}
int hipMemcpyAsync(void* d, const void* s, size_t n, int, void* st) {
    if (int e = meet("hipMemcpyAsync", st)) return e;
    std::memcpy(d, s, n);
    return 0;
}
int hipMemsetAsync(void* d, int v, size_t n, void* st) {
    if (int e = meet("hipMemsetAsync", st)) return e;
    std::memset(d, v, n);
    return 0;
}
int hipStreamCreateWithFlags(void** s, unsigned) {
    if (int e = enter("hipStreamCreateWithFlags")) return e;
    *s = new Stream;
    return 0;
}
int hipStreamDestroy(void* s) {
    delete static_cast<Stream*>(s);
    return 0;
}
int hipStreamSynchronize(void* s) { return meet("hipStreamSynchronize", s); }
int hipStreamWaitEvent(void*, void*, unsigned) { return enter("hipStreamWaitEvent"); }
int hipStreamBeginCapture(void* s, int) {
    if (int e = enter("hipStreamBeginCapture")) return e;
    if (static_cast<Stream*>(s)->capturing) return error(kIllegalState);
    static_cast<Stream*>(s)->capturing = true;
    return 0;
}
int hipStreamEndCapture(void* s, void** g) {
    if (!static_cast<Stream*>(s)->capturing) return error(kIllegalState);
    static_cast<Stream*>(s)->capturing = false;
    *g = nullptr;
    if (int e = enter("hipStreamEndCapture")) return e;
    *g = new int(0);
    ++live_graphs;
    return 0;
}
int hipGraphDestroy(void* g) {
    delete static_cast<int*>(g);
    --live_graphs;
    return 0;
}
int hipGraphInstantiate(void** x, void*, void*, char*, size_t) {
    if (int e = enter("hipGraphInstantiate")) return e;
    *x = new int(0);
    ++live_graphs;
    return 0;
}
int hipGraphExecDestroy(void* x) {
    delete static_cast<int*>(x);
    --live_graphs;
    return 0;
}
int hipGraphLaunch(void*, void*) { return enter("hipGraphLaunch"); }
int hipEventCreate(void** e) {
    *e = new Event;
    return 0;
}
int hipEventCreateWithFlags(void** e, unsigned) { return hipEventCreate(e); }
int hipEventDestroy(void* e) {
    delete static_cast<Event*>(e);
    return 0;
}
int hipEventRecord(void*, void*) { return enter("hipEventRecord"); }
int hipEventSynchronize(void*) { return enter("hipEventSynchronize"); }
int hipEventElapsedTime(float* ms, void*, void*) {
    *ms = 1.0f;
    return 0;
}
int hipGetDevice(int* d) {
    *d = 0;
    return 0;
}
int hipSetDevice(int) { return 0; }
const char* hipGetErrorString(int) { return "planted failure"; }
int hipGetLastError() {       // the last failure of any call, until it is read
    const int e = last_error;
    last_error = 0;
    return e;
}
int hipGetSymbolAddress(void** p, const void*) {
    static char* buf = static_cast<char*>(std::calloc(1 << 20, 1));
    *p = buf;
    return 0;
}
int hipLaunchKernel(const void* f, ...) {
    ++calls[kernels[f]];
    return 0;
}
int __hipPushCallConfiguration(...) { return 0; }
int __hipPopCallConfiguration(...) { return 0; }
void** __hipRegisterFatBinary(const void*) {
    static void* h = nullptr;
    return &h;
}
void __hipRegisterFunction(void**, const void* f, char*, const char* name, ...) { kernels[f] = name; }
void __hipRegisterVar(...) {}
void __hipUnregisterFatBinary(void**) {}

}  // extern "C"

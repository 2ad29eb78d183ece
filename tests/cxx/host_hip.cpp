// The HIP runtime calls that libddfmm.so makes, on host memory: kernels do nothing, streams
// count the work issued and known to be done.  Loaded before libddfmm.so (same soname as the
// runtime), it shows on the CPU what a context allocates, frees and waits for:
//   host_hip_live / host_hip_peak   bytes allocated now / at most since host_hip_reset
//   host_hip_fail(n)                the n-th fallible call from now fails (0: none)
//   host_hip_calls                  fallible calls since host_hip_reset
//   host_hip_early                  graphs destroyed before the host knew their last launch done
//   host_hip_reads                  copies to the host while some stream was not known to be done
//   host_hip_version(v)             the runtime version reported
//   host_hip_free_bytes(n)          the free device memory reported
// g++ -shared -fPIC -Wl,-soname,libamdhip64.so.7 -Wl,--version-script=host_hip.map
#include <cstddef>
#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <map>
#include <utility>

namespace {
struct Stream {
    int64_t issued = 0, done = 0;
};
struct Event {
    Stream* s = nullptr;
    int64_t at = 0;
};
struct Exec {
    Stream* s = nullptr;
    int64_t at = 0;
};
std::map<void*, size_t> blocks;
std::map<Stream*, int> streams;
int64_t live = 0, peak = 0, calls = 0, fail_in = 0, early = 0, reads = 0, free_bytes = int64_t(1) << 40;
int last = 0, version = 70200000;
Stream null_stream;

constexpr int OOM = 2;
int err() {
    ++calls;
    if (fail_in > 0 && --fail_in == 0) return last = OOM;
    return 0;
}
Stream* of(void* s) { return s ? (Stream*)s : &null_stream; }
void idle() {
    null_stream.done = null_stream.issued;
    for (auto& s : streams) s.first->done = s.first->issued;
}
}  // namespace

extern "C" {
int64_t host_hip_live() { return live; }
int64_t host_hip_peak() { return peak; }
int64_t host_hip_calls() { return calls; }
int64_t host_hip_early() { return early; }
int64_t host_hip_reads() { return reads; }
void host_hip_fail(int64_t n) { fail_in = n; }
void host_hip_version(int v) { version = v; }
void host_hip_free_bytes(int64_t n) { free_bytes = n; }
void host_hip_reset() {
    peak = live;
    calls = early = reads = fail_in = 0;
    last = 0;
}

int hipRuntimeGetVersion(int* v) { *v = version; return 0; }
int hipMemGetInfo(size_t* f, size_t* t) { *f = free_bytes; *t = free_bytes; return 0; }
int hipSetDevice(int) { return 0; }
int hipGetDevice(int* d) { *d = 0; return 0; }
const char* hipGetErrorString(int e) { return e ? "out of memory" : "no error"; }
int hipGetLastError() { int e = last; last = 0; return e; }

int hipMalloc(void** p, size_t n) {
    if (int e = err()) return e;
    *p = std::malloc(n ? n : 1);
    blocks[*p] = n;
    live += n;
    if (live > peak) peak = live;
    return 0;
}
int hipFree(void* p) {
    if (!p) return 0;
    auto it = blocks.find(p);
    if (it == blocks.end()) std::abort();
    idle();
    live -= it->second;
    blocks.erase(it);
    std::free(p);
    return 0;
}
int hipMemcpy(void* d, const void* s, size_t n, int kind) {
    if (int e = err()) return e;
    if (kind == 2)
        for (auto& x : streams) reads += x.first->done < x.first->issued;
    std::memcpy(d, s, n);
    return 0;
}
int hipMemcpyAsync(void* d, const void* s, size_t n, int, void* st) {
    if (int e = err()) return e;
    std::memcpy(d, s, n);
    ++of(st)->issued;
    return 0;
}
int hipMemset(void* d, int v, size_t n) {
    if (int e = err()) return e;
    std::memset(d, v, n);
    return 0;
}
int hipMemsetAsync(void* d, int v, size_t n, void* st) {
    ++of(st)->issued;
    return hipMemset(d, v, n);
}

int hipStreamCreateWithFlags(void** s, unsigned) {
    auto* x = new Stream();
    streams[x] = 1;
    *s = x;
    return 0;
}
int hipStreamCreate(void** s) { return hipStreamCreateWithFlags(s, 0); }
int hipStreamDestroy(void* s) {
    streams.erase((Stream*)s);
    delete (Stream*)s;
    return 0;
}
int hipStreamSynchronize(void* s) {
    if (int e = err()) return e;
    of(s)->done = of(s)->issued;
    return 0;
}
int hipDeviceSynchronize() { idle(); return 0; }
int hipStreamWaitEvent(void* s, void*, unsigned) { ++of(s)->issued; return 0; }
int hipEventCreateWithFlags(void** e, unsigned) { *e = new Event(); return 0; }
int hipEventCreate(void** e) { return hipEventCreateWithFlags(e, 0); }
int hipEventDestroy(void* e) { delete (Event*)e; return 0; }
int hipEventRecord(void* e, void* s) {
    auto* x = (Event*)e;
    x->s = of(s);
    x->at = ++of(s)->issued;
    return 0;
}
int hipEventSynchronize(void* e) {
    auto* x = (Event*)e;
    if (x->s && x->s->done < x->at) x->s->done = x->at;
    return 0;
}
int hipEventElapsedTime(float* ms, void*, void*) { *ms = 1; return 0; }

int hipStreamBeginCapture(void*, int) { return 0; }
int hipStreamEndCapture(void*, void** g) { *g = std::malloc(1); return 0; }
int hipGraphDestroy(void* g) { std::free(g); return 0; }
int hipGraphInstantiate(void** x, void*, void*, char*, size_t) { *x = new Exec(); return 0; }
int hipGraphLaunch(void* x, void* s) {
    auto* e = (Exec*)x;
    e->s = of(s);
    e->at = ++of(s)->issued;
    return 0;
}
int hipGraphExecDestroy(void* x) {
    auto* e = (Exec*)x;
    if (e->s && e->s->done < e->at) ++early;
    delete e;
    return 0;
}

int hipLaunchKernel(const void*, ...) { return err(); }
int hipGetSymbolAddress(void** p, const void*) {
    static char scratch[32 << 20];
    *p = scratch;
    return 0;
}
struct Dim {
    uint32_t x, y, z;
};
int __hipPushCallConfiguration(Dim, Dim, size_t, void*) { return 0; }
int __hipPopCallConfiguration(Dim* g, Dim* b, size_t* shared, void** s) {
    *g = *b = Dim{1, 1, 1};
    *shared = 0;
    *s = nullptr;
    return 0;
}
void** __hipRegisterFatBinary(const void*) { static void* h; return &h; }
void __hipRegisterFunction(void**, const void*, char*, const char*, unsigned, void*, void*, Dim*, Dim*, int*) {}
void __hipRegisterVar(void**, void*, char*, const char*, int, size_t, int, int) {}
void __hipUnregisterFatBinary(void**) {}
}

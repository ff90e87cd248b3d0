// A stand-in for the HIP runtime, for tests of the library's host code on a
// machine without a GPU: memory is host memory, kernels are reported to a
// callback (by name, with their grid) instead of run (but for the readback's copy,
// which the host waits for), streams and events only have a lifetime.  Every handle and pointer handed in is checked against the
// live ones; a wrong one ends the process with a message.  Deleted objects are
// overwritten and never handed out again, so that a late use shows.
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <set>
#include <string>
#include <vector>

#include <malloc.h>

#include <new>

#include <hip/hip_runtime_api.h>

namespace {
thread_local int t_in_stub = 0;   // the stand-in's own allocations never fail
thread_local long t_fail_in = -1;  // the library's that many from now does, once
struct InStub {
    InStub() { ++t_in_stub; }
    ~InStub() { --t_in_stub; }
};
}  // namespace

#ifndef STUB_PLAIN_DELETE  // (with a sanitizer, which does the rest better)
static void *allocate(size_t n) noexcept
{
    if (!t_in_stub && t_fail_in >= 0 && t_fail_in-- == 0) return nullptr;
    return malloc(n ? n : 1);
}
void *operator new(size_t n)
{
    if (void *p = allocate(n)) return p;
    throw std::bad_alloc();
}
void *operator new(size_t n, const std::nothrow_t &) noexcept { return allocate(n); }
void operator delete(void *p) noexcept
{
    // rising words: no two pointers left in it are equal, and none is an address
    if (p)
        for (size_t i = 0, n = malloc_usable_size(p) / 8; i < n; ++i)
            static_cast<volatile uint64_t *>(p)[i] = 0xA5A5A5A5A5A50000ull + 64 * i;
}
void operator delete(void *p, size_t) noexcept { operator delete(p); }
#endif

namespace {

using Callback = void (*)(const char *name, uint32_t grid, uint32_t block);

struct Launch {
    std::string name;
    uint32_t grid, block;
};
struct Stream {
    bool capturing = false;
    std::vector<Launch> graph;
};
struct Event {
    bool recorded = false;
    Stream *captured_on = nullptr;  // recorded into that stream's capture
};
using Graph = std::vector<Launch>;

std::recursive_mutex g_mutex;
std::map<char *, size_t> g_device, g_pinned;
size_t g_used = 0, g_limit = SIZE_MAX, g_mallocs = 0;
bool g_lose_copies = false;
std::set<void *> g_streams, g_events, g_graphs, g_execs;
std::map<Stream *, Stream *> g_joined;  // side stream -> the capturing one it was forked from
// (filled by the library's static constructors, which may run before this file's)
std::map<const void *, std::string> &names()
{
    static auto *m = new std::map<const void *, std::string>;
    return *m;
}

Callback g_callback = nullptr;
thread_local hipError_t t_last = hipSuccess;
thread_local struct { dim3 grid, block; size_t shared; hipStream_t stream; } t_config;

[[noreturn]] void wrong(const char *what, const void *p)
{
    fprintf(stderr, "hip stub: %s %p is not live\n", what, p);
    abort();
}

hipError_t ret(hipError_t e)
{
    if (e != hipSuccess) t_last = e;
    return e;
}

template <typename T>
T *live(std::set<void *> &s, void *p, const char *what)
{
    std::lock_guard<std::recursive_mutex> l(g_mutex);
    if (!s.count(p)) wrong(what, p);
    return static_cast<T *>(p);
}

template <typename T>
T *made(std::set<void *> &s, T *p)
{
    std::lock_guard<std::recursive_mutex> l(g_mutex);
    s.insert(p);
    return p;
}

// The bytes from p to the end of the live allocation it lies in; 0: in none.
size_t room(const std::map<char *, size_t> &m, const void *p)
{
    auto it = m.upper_bound(static_cast<char *>(const_cast<void *>(p)));
    if (it == m.begin()) return 0;
    --it;
    const char *end = it->first + it->second;
    return static_cast<const char *>(p) < end ? (size_t)(end - static_cast<const char *>(p)) : 0;
}

// As the runtime does: a range past the end of its allocation is refused.
hipError_t copy(void *d, const void *s, size_t n, hipMemcpyKind kind)
{
    std::lock_guard<std::recursive_mutex> l(g_mutex);
    const size_t rd = room(g_device, d), rs = room(g_device, s), hd = room(g_pinned, d), hs = room(g_pinned, s);
    if ((kind == hipMemcpyHostToDevice || kind == hipMemcpyDeviceToDevice) && !rd) wrong("copy to", d);
    if ((kind == hipMemcpyDeviceToHost || kind == hipMemcpyDeviceToDevice) && !rs) wrong("copy from", s);
    for (size_t r : { rd, rs, hd, hs })
        if (r && r < n) return ret(hipErrorInvalidValue);
    memcpy(d, s, n);
    return hipSuccess;
}

Stream *capture_of(Stream *s)
{
    if (!s) return nullptr;
    if (s->capturing) return s;
    auto it = g_joined.find(s);
    return it == g_joined.end() ? nullptr : it->second;
}

}  // namespace

extern "C" {

// ------------------------------------------------------------- test control
void stub_callback(Callback c) { g_callback = c; }
void stub_fail_new(long n) { t_fail_in = n; }  // negative: none
long stub_fail_left() { return t_fail_in; }
void stub_limit(size_t bytes) { g_limit = bytes; }
void stub_lose_copies(int lose) { g_lose_copies = lose != 0; }  // readbacks raise no flags
size_t stub_used() { return g_used; }
size_t stub_pinned()
{
    size_t n = 0;
    for (auto &p : g_pinned) n += p.second;
    return n;
}
size_t stub_mallocs() { return g_mallocs; }
// The k-th live pinned allocation of this size (address order); null past the last.
void *stub_pinned_of(size_t bytes, size_t k)
{
    for (auto &p : g_pinned)
        if (p.second == bytes && k-- == 0) return p.first;
    return nullptr;
}

// ------------------------------------------------------------------- memory
hipError_t hipMalloc(void **p, size_t n)
{
    InStub in_stub;
    std::lock_guard<std::recursive_mutex> l(g_mutex);
    ++g_mallocs;
    if (g_used + n > g_limit) return *p = nullptr, ret(hipErrorOutOfMemory);
    *p = calloc(1, n ? n : 1);
    if (!*p) return ret(hipErrorOutOfMemory);
    g_device[(char *)*p] = n;
    g_used += n;
    return hipSuccess;
}
hipError_t hipFree(void *p)
{
    InStub in_stub;
    std::lock_guard<std::recursive_mutex> l(g_mutex);
    if (!p) return hipSuccess;
    auto it = g_device.find((char *)p);
    if (it == g_device.end()) wrong("device memory", p);
    g_used -= it->second;
    g_device.erase(it);
    free(p);
    return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t n, unsigned)
{
    InStub in_stub;
    std::lock_guard<std::recursive_mutex> l(g_mutex);
    *p = calloc(1, n ? n : 1);
    g_pinned[(char *)*p] = n;
    return hipSuccess;
}
hipError_t hipHostFree(void *p)
{
    InStub in_stub;
    std::lock_guard<std::recursive_mutex> l(g_mutex);
    if (!p) return hipSuccess;
    if (!g_pinned.erase((char *)p)) wrong("pinned memory", p);
    free(p);
    return hipSuccess;
}
hipError_t hipHostGetDevicePointer(void **d, void *h, unsigned) { InStub in_stub; return *d = h, hipSuccess; }
hipError_t hipPointerGetAttributes(hipPointerAttribute_t *a, const void *p)
{
    InStub in_stub;
    std::lock_guard<std::recursive_mutex> l(g_mutex);
    memset(a, 0, sizeof *a);
    a->type = hipMemoryTypeUnregistered;
    for (auto &q : g_pinned)
        if ((char *)p >= q.first && (char *)p < q.first + q.second) a->type = hipMemoryTypeHost;
    return hipSuccess;
}
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind k) { InStub in_stub; return copy(d, s, n, k); }
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind k, hipStream_t st)
{
    InStub in_stub;
    if (st) live<Stream>(g_streams, st, "stream");
    return copy(d, s, n, k);
}
hipError_t hipMemcpy2D(void *d, size_t dp, const void *s, size_t sp, size_t w, size_t h, hipMemcpyKind k)
{
    InStub in_stub;
    hipError_t e = hipSuccess;
    for (size_t y = 0; y < h && e == hipSuccess; ++y) e = copy((char *)d + y * dp, (const char *)s + y * sp, w, k);
    return e;
}
hipError_t hipMemset(void *d, int v, size_t n)
{
    InStub in_stub;
    std::lock_guard<std::recursive_mutex> l(g_mutex);
    if (room(g_device, d) < n) wrong("set of", d);
    return memset(d, v, n), hipSuccess;
}
hipError_t hipGetSymbolAddress(void **p, const void *)
{
    InStub in_stub;
    static char *mem = nullptr;
    std::lock_guard<std::recursive_mutex> l(g_mutex);
    if (!mem) {
        mem = (char *)calloc(1, 64u << 20);
        g_device[mem] = 64u << 20;
    }
    return *p = mem, hipSuccess;
}

// ------------------------------------------------------------------- device
hipError_t hipGetDeviceCount(int *n) { InStub in_stub; return *n = 1, hipSuccess; }
hipError_t hipGetDevice(int *d) { InStub in_stub; return *d = 0, hipSuccess; }
hipError_t hipSetDevice(int) { InStub in_stub; return hipSuccess; }
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t, int) { InStub in_stub; return *v = 256, hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600 *p, int)
{
    InStub in_stub;
    memset(p, 0, sizeof *p);
    p->multiProcessorCount = 256;
    return hipSuccess;
}
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int *n, const void *, int, size_t) { InStub in_stub; return *n = 4, hipSuccess; }
const char *hipGetErrorString(hipError_t) { return "hip stub error"; }
hipError_t hipGetLastError()
{
    InStub in_stub;
    const hipError_t e = t_last;
    t_last = hipSuccess;
    return e;
}

// ---------------------------------------------------------- streams, events
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) { InStub in_stub; return *s = (hipStream_t)made(g_streams, new Stream), hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t s)
{
    InStub in_stub;
    Stream *p = live<Stream>(g_streams, s, "stream");
    std::lock_guard<std::recursive_mutex> l(g_mutex);
    g_streams.erase(p);
    delete p;
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t s)
{
    InStub in_stub;
    if (s) live<Stream>(g_streams, s, "stream");
    return hipSuccess;
}
hipError_t hipStreamQuery(hipStream_t s) { InStub in_stub; return hipStreamSynchronize(s); }
hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned)
{
    InStub in_stub;
    Stream *p = live<Stream>(g_streams, s, "stream");
    Event *v = live<Event>(g_events, e, "event");
    std::lock_guard<std::recursive_mutex> l(g_mutex);
    if (v->captured_on && p != v->captured_on) g_joined[p] = v->captured_on;
    return hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t *e) { InStub in_stub; return *e = (hipEvent_t)made(g_events, new Event), hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { InStub in_stub; return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t e)
{
    InStub in_stub;
    Event *v = live<Event>(g_events, e, "event");
    std::lock_guard<std::recursive_mutex> l(g_mutex);
    g_events.erase(v);
    delete v;
    return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s)
{
    InStub in_stub;
    Event *v = live<Event>(g_events, e, "event");
    Stream *p = s ? live<Stream>(g_streams, s, "stream") : nullptr;
    std::lock_guard<std::recursive_mutex> l(g_mutex);
    v->recorded = true;
    v->captured_on = capture_of(p);
    return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t e) { InStub in_stub; return live<Event>(g_events, e, "event"), hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) { InStub in_stub; return *ms = 1.f, hipSuccess; }

// ------------------------------------------------------------------- graphs
hipError_t hipStreamBeginCapture(hipStream_t s, hipStreamCaptureMode)
{
    InStub in_stub;
    Stream *p = live<Stream>(g_streams, s, "stream");
    p->capturing = true;
    p->graph.clear();
    return hipSuccess;
}
hipError_t hipStreamEndCapture(hipStream_t s, hipGraph_t *g)
{
    InStub in_stub;
    Stream *p = live<Stream>(g_streams, s, "stream");
    std::lock_guard<std::recursive_mutex> l(g_mutex);
    p->capturing = false;
    for (auto it = g_joined.begin(); it != g_joined.end();) it = it->second == p ? g_joined.erase(it) : std::next(it);
    *g = (hipGraph_t)made(g_graphs, new Graph(p->graph));
    return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t *e, hipGraph_t g, hipGraphNode_t *, char *, size_t)
{
    InStub in_stub;
    *e = (hipGraphExec_t)made(g_execs, new Graph(*live<Graph>(g_graphs, g, "graph")));
    return hipSuccess;
}
hipError_t hipGraphDestroy(hipGraph_t g)
{
    InStub in_stub;
    Graph *p = live<Graph>(g_graphs, g, "graph");
    std::lock_guard<std::recursive_mutex> l(g_mutex);
    g_graphs.erase(p);
    delete p;
    return hipSuccess;
}
hipError_t hipGraphExecDestroy(hipGraphExec_t e)
{
    InStub in_stub;
    Graph *p = live<Graph>(g_execs, e, "graph instance");
    std::lock_guard<std::recursive_mutex> l(g_mutex);
    g_execs.erase(p);
    delete p;
    return hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t e, hipStream_t s)
{
    InStub in_stub;
    live<Stream>(g_streams, s, "stream");
    for (const Launch &l : *live<Graph>(g_execs, e, "graph instance"))
        if (g_callback) g_callback(l.name.c_str(), l.grid, l.block);
    return hipSuccess;
}

// ----------------------------------------------------------------- launches
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t sh, hipStream_t s)
{
    InStub in_stub;
    t_config = { g, b, sh, s };
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *sh, hipStream_t *s)
{
    InStub in_stub;
    *g = t_config.grid, *b = t_config.block, *sh = t_config.shared, *s = t_config.stream;
    return hipSuccess;
}
// k_read_out(src, dst, words, count, flags, epoch): the copy, and a flag per 256 KB.
static void read_out(void **args)
{
    const char *src = *static_cast<const char **>(args[0]);
    char *dst = *static_cast<char **>(args[1]);
    const size_t bytes = 4 * (size_t)*static_cast<uint32_t *>(args[2]);
    uint32_t *flags = *static_cast<uint32_t **>(args[4]);
    if (room(g_device, src) < bytes) wrong("readback from", src);
    if (room(g_pinned, dst) < bytes) wrong("readback to", dst);
    memcpy(dst, src, bytes);
    if (g_lose_copies) return;
    for (size_t c = 0; c * (256u << 10) < bytes; ++c) flags[c] = *static_cast<uint32_t *>(args[5]);
}
hipError_t hipLaunchKernel(const void *f, dim3 g, dim3 b, void **args, size_t, hipStream_t s)
{
    InStub in_stub;
    Stream *p = s ? live<Stream>(g_streams, s, "stream") : nullptr;
    const Launch l{ names().at(f), g.x, b.x };
    if (!g.x || !b.x) return ret(hipErrorInvalidConfiguration);
    std::unique_lock<std::recursive_mutex> lock(g_mutex);
    if (l.name.find("k_read_out") != std::string::npos) read_out(args);
    if (Stream *c = capture_of(p)) c->graph.push_back(l);
    else if (lock.unlock(); g_callback) g_callback(l.name.c_str(), l.grid, l.block);
    return hipSuccess;
}
void **__hipRegisterFatBinary(const void *) { static void *m[1]; return m; }
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *f, char *, const char *name, unsigned, void *, void *, void *, void *, int *)
{
    InStub in_stub;
    names()[f] = name;
}
void __hipRegisterVar(void **, void *, char *, const char *, int, size_t, int, int) {}

}  // extern "C"

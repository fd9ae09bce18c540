// A stand-in for the HIP runtime that runs nothing: device memory is host memory, copies happen at once,
// kernels not at all, and every call that orders or allocates is written to a log.  Loaded before
// libpfh.so into a process of its own, it shows the host code's calls without a GPU.
#include <cstdarg>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <string>

namespace {
std::string g_log;
std::map<const void *, std::string> g_names;   // host function -> kernel
std::map<const void *, size_t> g_vars, g_blocks;
std::map<const void *, void *> g_var_mem;
size_t g_held = 0, g_limit = ~(size_t)0;
int g_attr_error = 0, g_last = 0, g_device = 0;
uintptr_t g_handles = 0x1000;
struct Dim3 {
    uint32_t x, y, z;
};
struct {
    Dim3 grid, block;
    size_t shmem;
    void *stream;
} g_call;

void say(const char *f, ...) {
    char line[512];
    va_list ap;
    va_start(ap, f);
    vsnprintf(line, sizeof line, f, ap);
    va_end(ap);
    g_log += line;
    g_log += '\n';
}
int done(int e) {
    if (e) g_last = e;
    return e;
}
std::string name_of(const void *f) { return g_names.count(f) ? g_names[f] : "?"; }
}  // namespace

extern "C" {
const char *rec_log() { return g_log.c_str(); }
void rec_clear() { g_log.clear(); }
void rec_limit(size_t bytes) { g_limit = bytes; }
size_t rec_held() { return g_held; }
void rec_attr_error(int e) { g_attr_error = e; }

void **__hipRegisterFatBinary(const void *) {
    static void *h;
    return &h;
}
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *host, char *, const char *name, unsigned, void *, void *, void *, void *, int *) {
    g_names[host] = name;
}
void __hipRegisterVar(void **, void *var, char *, char *, int, size_t size, int, int) { g_vars[var] = size; }
int __hipPushCallConfiguration(Dim3 grid, Dim3 block, size_t shmem, void *stream) {
    g_call = {grid, block, shmem, stream};
    return 0;
}
int __hipPopCallConfiguration(Dim3 *grid, Dim3 *block, size_t *shmem, void **stream) {
    *grid = g_call.grid, *block = g_call.block, *shmem = g_call.shmem, *stream = g_call.stream;
    return 0;
}
int hipLaunchKernel(const void *f, Dim3, Dim3, void **, size_t shmem, void *stream) {
    say("hipLaunchKernel %s %zu %p", name_of(f).c_str(), shmem, stream);
    return 0;
}
int hipFuncSetAttribute(const void *f, int attr, int value) {
    say("hipFuncSetAttribute %s %d %d", name_of(f).c_str(), attr, value);
    return done(g_attr_error);
}
int hipGetDeviceCount(int *n) {
    *n = 2;
    return 0;
}
int hipSetDevice(int d) {
    g_device = d;
    say("hipSetDevice %d", d);
    return 0;
}
int hipGetDevice(int *d) {
    *d = g_device;
    return 0;
}
const char *hipGetErrorString(int) { return "recorded error"; }
int hipGetLastError() {
    const int e = g_last;
    g_last = 0;
    return e;
}
int hipGetSymbolAddress(void **p, const void *var) {
    if (!g_var_mem.count(var)) g_var_mem[var] = calloc(g_vars[var], 1);
    *p = g_var_mem[var];
    return 0;
}

int hipMalloc(void **p, size_t n) {
    if (g_held + n > g_limit) {
        say("hipMalloc none %zu", n);
        return done(2);
    }
    *p = calloc(n, 1);
    g_blocks[*p] = n;
    g_held += n;
    say("hipMalloc %p %zu", *p, n);
    return 0;
}
int hipFree(void *p) {
    say("hipFree %p", p);
    if (p) g_held -= g_blocks[p], g_blocks.erase(p);
    free(p);
    return 0;
}
int hipHostMalloc(void **p, size_t n, unsigned flags) {
    *p = calloc(n, 1);
    say("hipHostMalloc %p %zu %x", *p, n, flags);
    return 0;
}
int hipHostFree(void *p) {
    free(p);
    return 0;
}
int hipMemcpy(void *d, const void *s, size_t n, int kind) {
    say("hipMemcpy %p %p %zu %d", d, s, n, kind);
    memcpy(d, s, n);
    return 0;
}
int hipMemcpy2D(void *d, size_t dp, const void *s, size_t sp, size_t w, size_t h, int kind) {
    say("hipMemcpy2D %p %p %zu %zu %d", d, s, w, h, kind);
    for (size_t r = 0; r < h; r++) memcpy((char *)d + r * dp, (const char *)s + r * sp, w);
    return 0;
}
int hipMemcpyAsync(void *d, const void *s, size_t n, int kind, void *stream) {
    say("hipMemcpyAsync %p %p %zu %d %p", d, s, n, kind, stream);
    memcpy(d, s, n);
    return 0;
}

int hipStreamCreateWithFlags(void **s, unsigned flags) {
    *s = (void *)(g_handles += 16);
    say("hipStreamCreateWithFlags %p %x", *s, flags);
    return 0;
}
int hipStreamDestroy(void *) { return 0; }
int hipStreamSynchronize(void *s) {
    say("hipStreamSynchronize %p", s);
    return 0;
}
int hipStreamWaitEvent(void *s, void *e, unsigned) {
    say("hipStreamWaitEvent %p %p", s, e);
    return 0;
}
int hipDeviceSynchronize() {
    say("hipDeviceSynchronize");
    return 0;
}
int hipEventCreateWithFlags(void **e, unsigned flags) {
    *e = (void *)(g_handles += 16);
    say("hipEventCreate %p %x", *e, flags);
    return 0;
}
int hipEventCreate(void **e) { return hipEventCreateWithFlags(e, 0); }
int hipEventDestroy(void *) { return 0; }
int hipEventRecord(void *e, void *s) {
    say("hipEventRecord %p %p", e, s);
    return 0;
}
int hipEventRecordWithFlags(void *e, void *s, unsigned) { return hipEventRecord(e, s); }
int hipEventSynchronize(void *e) {
    say("hipEventSynchronize %p", e);
    return 0;
}
int hipEventQuery(void *) { return 0; }
int hipEventElapsedTime(float *ms, void *, void *) {
    *ms = 0.0f;
    return 0;
}

int hipStreamBeginCapture(void *, int) { return 0; }
int hipStreamEndCapture(void *, void **g) {
    *g = (void *)(g_handles += 16);
    return 0;
}
int hipGraphInstantiate(void **x, void *, void *, char *, size_t) {
    *x = (void *)(g_handles += 16);
    say("hipGraphInstantiate %p", *x);
    return 0;
}
int hipGraphDestroy(void *) { return 0; }
int hipGraphExecDestroy(void *) { return 0; }
int hipGraphLaunch(void *x, void *s) {
    say("hipGraphLaunch %p %p", x, s);
    return 0;
}
}

// A HIP runtime without a GPU, for tests of what the library's host code enqueues, when it
// waits, and what it does when an allocation fails.  "Device" memory is host memory that
// copies really fill; kernels are recorded and never run.  Loaded with global symbols before
// libifs.so, whose calls then come here.
#include <stdint.h>
#include <stdlib.h>
#include <string.h>

#include <map>
#include <string>
#include <vector>

namespace {
struct Dim3 {
    uint32_t x, y, z;
};
constexpr int kOk = 0, kInvalid = 1, kNoMemory = 2, kCapture = 900;
std::string text;                       // one line per call
std::map<char *, size_t> live;          // allocations
std::map<const void *, std::string> kernels;
std::map<void *, int> capturing;        // stream -> 1 capturing, 2 capture broken
int last_error = kOk;
long alloc_count = 0, fail_alloc = -1;  // fail_alloc: allocations still granted, -1 all
size_t free_bytes = (size_t)64 << 30;
size_t stream_count = 0;
struct Watch {
    std::string kernel;
    int arg;
    size_t offset;
};
std::vector<Watch> watched;
struct {
    Dim3 grid, block;
    size_t shm;
    void *stream;
} config;

int fail(int e) {
    last_error = e;
    return e;
}
int any_capture() {
    for (auto &c : capturing)
        if (c.second) {
            c.second = 2;
            return 1;
        }
    return 0;
}
void say(const std::string &s) { text += s + "\n"; }
std::string name_of(void *s) { return std::to_string((uintptr_t)s); }
}  // namespace

extern "C" {
const char *fake_log() { return text.c_str(); }
void fake_clear() { text.clear(); }
void fake_fail_after(long n) { fail_alloc = n; }
long fake_allocs() { return alloc_count; }
long long fake_live_bytes() {
    long long b = 0;
    for (auto &a : live) b += (long long)a.second;
    return b;
}
void fake_set_free(size_t b) { free_bytes = b; }
// From now on every launch of a kernel whose name holds `kernel` also reports how many bytes lie
// behind the pointer at `offset` bytes into its argument `arg` (-1: freed, or never allocated).
void fake_watch(const char *kernel, int arg, size_t offset) { watched.push_back({kernel, arg, offset}); }

int hipMalloc(void **p, size_t n) {
    *p = nullptr;
    if (any_capture()) return fail(kCapture);
    ++alloc_count;
    if (fail_alloc == 0) {
        say("malloc " + std::to_string(n) + " failed");
        return fail(kNoMemory);
    }
    if (fail_alloc > 0) --fail_alloc;
    *p = calloc(1, n);
    if (!*p) return fail(kNoMemory);
    live[(char *)*p] = n;
    say("malloc " + std::to_string(n));
    return kOk;
}
int hipFree(void *p) {
    if (!p) return kOk;
    if (!live.erase((char *)p)) return fail(kInvalid);
    free(p);
    say("free");
    return kOk;
}
int hipMemcpy(void *d, const void *s, size_t n, int) {
    say("copy " + std::to_string(n));
    if (any_capture()) return fail(kCapture);
    memcpy(d, s, n);
    return kOk;
}
int hipMemcpyAsync(void *d, const void *s, size_t n, int, void *st) {
    say("copy_async " + name_of(st) + " " + std::to_string(n));
    if (!capturing[st]) memcpy(d, s, n);
    return kOk;
}
int hipMemset(void *d, int v, size_t n) {
    memset(d, v, n);
    return kOk;
}
int hipMemsetAsync(void *d, int v, size_t n, void *st) {
    say("memset " + name_of(st));
    memset(d, v, n);
    return kOk;
}
int hipMemGetInfo(size_t *f, size_t *t) {
    *f = *t = free_bytes;
    return kOk;
}
int hipGetDeviceCount(int *n) {
    *n = 1;
    return kOk;
}
int hipGetDevice(int *d) {
    *d = 0;
    return kOk;
}
int hipGetDevicePropertiesR0600(void *p, int) {
    memset(p, 0, 1024);
    return kOk;
}
int hipGetStreamDeviceId(void *) { return 0; }
int hipGetSymbolAddress(void **p, const void *) {
    static void *scratch = calloc(1, (size_t)64 << 20);
    *p = scratch;
    return kOk;
}
int hipGetLastError() {
    const int e = last_error;
    last_error = kOk;
    return e;
}
int hipPeekAtLastError() { return last_error; }

int hipStreamCreate(void **s) {
    *s = (void *)(++stream_count * 16);
    return kOk;
}
int hipStreamCreateWithFlags(void **s, unsigned) { return hipStreamCreate(s); }
int hipStreamDestroy(void *) { return kOk; }
int hipStreamSynchronize(void *s) {
    say("sync " + name_of(s));
    if (capturing[s]) {
        capturing[s] = 2;
        return fail(kCapture);
    }
    return kOk;
}
int hipStreamIsCapturing(void *s, int *st) {
    *st = capturing[s] ? 1 : 0;
    return kOk;
}
int hipStreamBeginCapture(void *s, int) {
    say("capture " + name_of(s));
    capturing[s] = 1;
    return kOk;
}
int hipStreamEndCapture(void *s, void **g) {
    const int was = capturing[s];
    if (was == 1) capturing[s] = 0;  // a broken capture leaves the stream unusable, as the GPU's runtime does
    *g = was == 1 ? (void *)16 : nullptr;
    say(was == 1 ? "captured" : "capture broken");
    return was == 1 ? kOk : fail(kCapture);
}
int hipGraphInstantiate(void **e, void *, void *, char *, size_t) {
    *e = (void *)16;
    return kOk;
}
int hipGraphLaunch(void *, void *s) {
    say("graph " + name_of(s));
    return kOk;
}
int hipGraphDestroy(void *) { return kOk; }
int hipGraphExecDestroy(void *) { return kOk; }

int hipEventCreate(void **e) {
    *e = (void *)16;
    return kOk;
}
int hipEventDestroy(void *) { return kOk; }
int hipEventRecord(void *, void *) { return kOk; }
int hipEventSynchronize(void *) { return kOk; }
int hipEventElapsedTime(float *ms, void *, void *) {
    *ms = 1.0f;
    return kOk;
}

void **__hipRegisterFatBinary(const void *) {
    static void *h = nullptr;
    return &h;
}
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *host, char *, const char *name, unsigned, void *, void *, void *,
                           void *, int *) {
    kernels[host] = name;
}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
int __hipPushCallConfiguration(Dim3 grid, Dim3 block, size_t shm, void *stream) {
    config = {grid, block, shm, stream};
    return kOk;
}
int __hipPopCallConfiguration(Dim3 *grid, Dim3 *block, size_t *shm, void **stream) {
    *grid = config.grid;
    *block = config.block;
    *shm = config.shm;
    *stream = config.stream;
    return kOk;
}
// Recorded as "launch <kernel> <stream> <dynamic LDS>", or "refused" beyond the limits of a launch.
int hipLaunchKernel(const void *f, Dim3 grid, Dim3 block, void **args, size_t shm, void *stream) {
    const std::string k = kernels.count(f) ? kernels[f] : "?";
    const bool ok = grid.x && grid.y && grid.z && grid.y <= 65535 && grid.z <= 65535 &&
                    block.x * block.y * block.z <= 1024 && shm <= 65536;
    if (capturing[stream] == 2) return fail(kCapture);
    say((ok ? "launch " : "refused ") + k + " " + name_of(stream) + " " + std::to_string(shm));
    for (auto &w : watched) {
        if (k.find(w.kernel) == std::string::npos) continue;
        char *p = *(char **)((char *)args[w.arg] + w.offset);
        auto a = live.upper_bound(p);
        long long left = -1;
        if (a != live.begin() && p < (--a)->first + a->second) left = (long long)(a->first + a->second - p);
        say("arg " + w.kernel + " " + std::to_string(w.arg) + " " + std::to_string(w.offset) + " " +
            std::to_string(left));
    }
    return ok ? kOk : fail(kInvalid);
}
}

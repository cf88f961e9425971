// A HIP runtime without a device, for tests of host logic (allocation, dispatch,
// error paths): preloaded before libamdhip64 it gives the library one gfx950
// device whose memory is host address space, counts and limits what is
// allocated, runs no kernel and records which kernels are launched.
#include <sys/mman.h>

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <string>

#include <hip/hip_runtime_api.h>

namespace {
struct State {
    std::map<void *, size_t> blocks;
    std::map<const void *, std::string> kernels;
    size_t used = 0, limit = ~(size_t)0;
    long mallocs = 0, frees = 0;
    bool copies = true, refuse = false;
    hipError_t last = hipSuccess;
    std::string launches;
    dim3 grid, block;
    size_t shared = 0;
    hipStream_t stream = nullptr;
};
State &S() {
    static State *s = new State;
    return *s;
}
}  // namespace

extern "C" {
// ------------------------------------------------------------ for the test
size_t fake_used() { return S().used; }
long fake_mallocs() { return S().mallocs; }
long fake_frees() { return S().frees; }
void fake_limit(size_t bytes) { S().limit = bytes; }
void fake_copies(int on) { S().copies = on != 0; }
// mangled names of every kernel in the library, a line each
const char *fake_kernels() {
    static std::string all;
    all.clear();
    for (auto &k : S().kernels) all += k.second + "\n";
    return all.c_str();
}
void fake_refuse(int on) { S().refuse = on != 0; }  // launches fail
// "mangled kernel name, grid x y z" lines since the last call
const char *fake_launches() {
    static std::string last;
    last.swap(S().launches);
    S().launches.clear();
    return last.c_str();
}

// -------------------------------------------------------------- the runtime
hipError_t hipGetDeviceCount(int *n) { return *n = 1, hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_t *p, int) {
    memset(p, 0, sizeof *p);
    strcpy(p->name, "fake");
    strcpy(p->gcnArchName, "gfx950");
    p->multiProcessorCount = 256;
    return hipSuccess;
}
hipError_t hipGetLastError() {
    const hipError_t e = S().last;
    S().last = hipSuccess;
    return e;
}
const char *hipGetErrorString(hipError_t e) { return e == hipSuccess ? "success" : "error"; }
hipError_t hipMalloc(void **p, size_t n) {
    State &s = S();
    *p = nullptr;
    if (n >> 46 || s.used > s.limit || n > s.limit - s.used) return hipErrorOutOfMemory;
    void *q = mmap(nullptr, n + 4096, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
    if (q == MAP_FAILED) return hipErrorOutOfMemory;
    s.blocks[q] = n;
    s.used += n;
    s.mallocs++;
    *p = q;
    return hipSuccess;
}
hipError_t hipFree(void *p) {
    if (!p) return hipSuccess;
    State &s = S();
    auto it = s.blocks.find(p);
    if (it == s.blocks.end()) {
        fprintf(stderr, "hipFree of an unknown block\n");
        abort();
    }
    s.used -= it->second;
    s.frees++;
    munmap(p, it->second + 4096);
    s.blocks.erase(it);
    return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t n, unsigned) { return *p = calloc(1, n), *p ? hipSuccess : hipErrorOutOfMemory; }
hipError_t hipHostFree(void *p) { return free(p), hipSuccess; }
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind) {
    if (S().copies) memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind k, hipStream_t) { return hipMemcpy(d, s, n, k); }
hipError_t hipMemcpy2DAsync(void *d, size_t dp, const void *s, size_t sp, size_t w, size_t h, hipMemcpyKind, hipStream_t) {
    for (size_t i = 0; i < h && S().copies; i++) memcpy((char *)d + i * dp, (const char *)s + i * sp, w);
    return hipSuccess;
}
hipError_t hipMemsetAsync(void *d, int v, size_t n, hipStream_t) {
    if (S().copies) memset(d, v, n);
    return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) { return *s = reinterpret_cast<hipStream_t>(16), hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipFuncSetAttribute(const void *, hipFuncAttribute, int) { return hipSuccess; }
hipError_t hipGetSymbolAddress(void **p, const void *) {
    static char symbol[4096];
    return *p = symbol, hipSuccess;
}

hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t sh, hipStream_t st) {
    State &s = S();
    s.grid = g, s.block = b, s.shared = sh, s.stream = st;
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *sh, hipStream_t *st) {
    State &s = S();
    *g = s.grid, *b = s.block, *sh = s.shared, *st = s.stream;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void *f, dim3 g, dim3 b, void **, size_t, hipStream_t) {
    if (S().refuse || !g.x || !g.y || !g.z || (size_t)g.x * b.x >> 32 || g.y > 65535 || g.z > 65535)
        return S().last = hipErrorInvalidValue;
    char line[64];
    snprintf(line, sizeof line, " %u %u %u\n", g.x, g.y, g.z);
    S().launches += S().kernels[f] + line;
    return hipSuccess;
}
void **__hipRegisterFatBinary(const void *) {
    static void *handle;
    return &handle;
}
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *host, char *, const char *name, unsigned, void *, void *, dim3 *, dim3 *, int *) {
    S().kernels[host] = name;
}
void __hipRegisterVar(void **, void *, char *, const char *, int, size_t, int, int) {}
}

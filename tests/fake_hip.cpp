/* A HIP runtime that launches nothing: it stands in for libamdhip64 when the
 * backend is loaded without a GPU, hands out lazily backed host memory as
 * device memory, and keeps a list of the launches it is asked for.  Loaded
 * with RTLD_GLOBAL before the backend, its symbols are the ones bound.  Used
 * by launches.py. */
#include <hip/hip_runtime_api.h>

#include <cxxabi.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>
#include <sys/mman.h>

#include <map>
#include <string>
#include <vector>

struct launch {
    std::string kernel;
    dim3 grid, block;
    size_t lds, lds_limit;
    uint64_t words[10]; /* the start of a skinny GEMM's argument struct */
};

static std::map<const void *, std::string> names;
static std::map<const void *, size_t> lds_limits;
static std::map<void *, size_t> blocks;
static std::map<const void *, void *> symbols;
static std::vector<launch> log_;
static dim3 push_grid, push_block;
static size_t push_lds, largest = ~(size_t)0, syncs;
static hipStream_t push_stream;

extern "C" {

/* device allocations above this many bytes fail from here on */
void fake_largest_block(size_t bytes) { largest = bytes; }
size_t fake_syncs() { return syncs; }

size_t fake_launches() { return log_.size(); }
void fake_clear() { log_.clear(); }
size_t fake_launch(size_t i, char *kernel, size_t size, uint64_t *out) {
    const launch &l = log_[i];
    snprintf(kernel, size, "%s", l.kernel.c_str());
    const uint64_t v[8] = {l.grid.x, l.grid.y, l.grid.z, l.block.x,
                           l.lds, l.lds_limit, 0, 0};
    memcpy(out, v, sizeof(v));
    memcpy(out + 8, l.words, sizeof(l.words));
    return l.grid.x;
}

void **__hipRegisterFatBinary(const void *) {
    static void *handle;
    return &handle;
}
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *host, char *,
                           const char *device, unsigned, void *, void *,
                           void *, void *, int *) {
    int status = 0;
    char *plain = abi::__cxa_demangle(device, nullptr, nullptr, &status);
    std::string name = plain ? plain : device;
    free(plain);
    if (name.rfind("void ", 0) == 0) name = name.substr(5);
    names[host] = name.substr(0, name.find('('));
}
void __hipRegisterVar(void **, void *var, char *, const char *, int,
                      size_t size, int, int) {
    symbols[var] = nullptr;
    (void)size;
}
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t lds,
                                      hipStream_t stream) {
    push_grid = grid; push_block = block;
    push_lds = lds; push_stream = stream;
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *grid, dim3 *block, size_t *lds,
                                     hipStream_t *stream) {
    *grid = push_grid; *block = push_block;
    *lds = push_lds; *stream = push_stream;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void *f, dim3 grid, dim3 block, void **args,
                           size_t lds, hipStream_t) {
    launch l = {names[f], grid, block, lds,
                lds_limits.count(f) ? lds_limits[f] : 64u * 1024, {}};
    if (l.kernel.find("hk_gemm_skinny") != std::string::npos)
        memcpy(l.words, args[0], sizeof(l.words));
    log_.push_back(l);
    return hipSuccess;
}
hipError_t hipFuncSetAttribute(const void *f, hipFuncAttribute, int value) {
    lds_limits[f] = (size_t)value;
    return hipSuccess;
}

static hipError_t give(void **p, size_t bytes) {
    *p = nullptr;
    void *m = mmap(nullptr, bytes, PROT_READ | PROT_WRITE,
                   MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
    if (m == MAP_FAILED) return hipErrorOutOfMemory;
    blocks[m] = bytes;
    *p = m;
    return hipSuccess;
}
hipError_t hipMalloc(void **p, size_t bytes) {
    return bytes > largest ? hipErrorOutOfMemory : give(p, bytes);
}
hipError_t hipFree(void *p) {
    auto it = blocks.find(p);
    if (it != blocks.end()) {
        munmap(p, it->second);
        blocks.erase(it);
    }
    return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t bytes, unsigned) {
    return give(p, bytes);
}
hipError_t hipHostFree(void *p) { return hipFree(p); }
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind) {
    memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind,
                          hipStream_t) {
    memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipMemGetInfo(size_t *available, size_t *total) {
    *available = *total = (size_t)288 << 30;
    return hipSuccess;
}
hipError_t hipGetSymbolAddress(void **p, const void *symbol) {
    void *&m = symbols[symbol];
    if (!m) (void)give(&m, (size_t)64 << 20);
    *p = m;
    return hipSuccess;
}

hipError_t hipGetDeviceCount(int *count) { *count = 1; return hipSuccess; }
hipError_t hipGetDevice(int *device) { *device = 0; return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600 *p, int) {
    memset(p, 0, sizeof(*p));
    p->multiProcessorCount = 256;
    return hipSuccess;
}
hipError_t hipGetLastError() { return hipSuccess; }
const char *hipGetErrorString(hipError_t e) {
    return e == hipSuccess ? "no error" : "out of memory";
}

hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) {
    static char stream;
    *s = (hipStream_t)&stream;
    return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { syncs++; return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) {
    return hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t *e) {
    static char event;
    *e = (hipEvent_t)&event;
    return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) {
    return hipEventCreate(e);
}
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) {
    *ms = 0.0f;
    return hipSuccess;
}

} /* extern "C" */

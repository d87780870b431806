/* A stand-in for the HIP runtime (CPU only): device memory is host memory,
 * kernels are not run, and the kernels launched and the allocations made are
 * logged.  Loaded globally before libhelio_hip.so, its symbols come first, so
 * a test sees which launches the host code chooses for a call, and what it
 * does when an allocation fails. */
#define _GNU_SOURCE
#include <stddef.h>
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>
#include <sys/mman.h>

typedef struct {
    uint32_t x, y, z;
} dim3_t;

enum { kMaxKernels = 512, kLog = 1 << 20, kHead = 4096 };
static struct {
    const void* host;
    char name[256];
} kernels[kMaxKernels];
static int num_kernels;
static char log_[kLog];
static size_t log_len, alloc_limit = (size_t)-1, largest;
static int last_error; /* of the last call that failed, until it is read */

static void note(const char* what, const char* arg, uint32_t n) {
    int k = snprintf(log_ + log_len, kLog - log_len, "%s %s %u\n", what, arg, n);
    if (k > 0 && log_len + (size_t)k < kLog) log_len += (size_t)k;
}

/* ---- for the test */
const char* stub_log(void) { return log_; }
void stub_reset(size_t limit) { /* allocations of more than limit bytes fail from here on */
    log_len = 0;
    log_[0] = 0;
    alloc_limit = limit;
    largest = 0;
}
size_t stub_largest(void) { return largest; }

/* ---- the runtime */
void** __hipRegisterFatBinary(const void* data) {
    static void* handle;
    (void)data;
    return &handle;
}
void __hipUnregisterFatBinary(void** m) { (void)m; }
void __hipRegisterFunction(void** m, const void* host, char* dev, const char* name, unsigned limit, void* a, void* b,
                           void* c, void* d, int* e) {
    (void)m, (void)dev, (void)limit, (void)a, (void)b, (void)c, (void)d, (void)e;
    if (num_kernels == kMaxKernels) abort();
    kernels[num_kernels].host = host;
    snprintf(kernels[num_kernels++].name, sizeof kernels[0].name, "%s", name);
}
void __hipRegisterVar(void** m, void* var, char* host, char* dev, int ext, size_t size, int constant, int global) {
    (void)m, (void)var, (void)host, (void)dev, (void)ext, (void)size, (void)constant, (void)global;
}
static struct {
    dim3_t grid, block;
    size_t shared;
    void* stream;
} conf;
int __hipPushCallConfiguration(dim3_t grid, dim3_t block, size_t shared, void* stream) {
    conf.grid = grid, conf.block = block, conf.shared = shared, conf.stream = stream;
    return 0;
}
int __hipPopCallConfiguration(dim3_t* grid, dim3_t* block, size_t* shared, void** stream) {
    *grid = conf.grid, *block = conf.block, *shared = conf.shared, *stream = conf.stream;
    return 0;
}
int hipLaunchKernel(const void* f, dim3_t grid, dim3_t block, void** args, size_t shared, void* stream) {
    (void)block, (void)args, (void)shared, (void)stream;
    for (int i = 0; i < num_kernels; ++i)
        if (kernels[i].host == f) {
            note("launch", kernels[i].name, grid.x);
            return 0;
        }
    abort();
}
int hipMalloc(void** p, size_t n) {
    if (n > largest) largest = n;
    if (n > alloc_limit) {
        *p = NULL;
        note("refused", "alloc", (uint32_t)(n >> 20));
        return last_error = 2; /* hipErrorOutOfMemory */
    }
    uint8_t* q = mmap(NULL, n + kHead, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
    if (q == MAP_FAILED) return 2;
    *(size_t*)q = n + kHead;
    *p = q + kHead;
    return 0;
}
int hipFree(void* p) {
    if (p) munmap((uint8_t*)p - kHead, *(size_t*)((uint8_t*)p - kHead));
    return 0;
}
int hipMemcpy(void* d, const void* s, size_t n, int kind) {
    (void)kind;
    memcpy(d, s, n);
    return 0;
}
int hipMemcpyAsync(void* d, const void* s, size_t n, int kind, void* st) {
    (void)st;
    return hipMemcpy(d, s, n, kind);
}
int hipMemset(void* d, int v, size_t n) {
    if (v) memset(d, v, n); /* fresh mappings are zero already */
    return 0;
}
int hipMemsetAsync(void* d, int v, size_t n, void* st) {
    (void)st;
    return hipMemset(d, v, n);
}
int hipGetSymbolAddress(void** p, const void* sym) {
    static uint8_t room[1 << 16];
    (void)sym;
    *p = room;
    return 0;
}
int hipOccupancyMaxActiveBlocksPerMultiprocessor(int* n, const void* f, int block, size_t dyn) {
    (void)f, (void)block, (void)dyn;
    *n = 1 << 12; /* persistent launches: a block per item */
    return 0;
}
int hipDeviceGetAttribute(int* v, int attr, int dev) {
    (void)attr, (void)dev;
    *v = 256;
    return 0;
}
int hipGetDeviceCount(int* n) {
    *n = 1;
    return 0;
}
int hipGetDevice(int* d) {
    *d = 0;
    return 0;
}
int hipSetDevice(int d) {
    (void)d;
    return 0;
}
int hipGetLastError(void) {
    int e = last_error;
    last_error = 0;
    return e;
}
const char* hipGetErrorString(int e) {
    (void)e;
    return "stand-in";
}
int hipStreamSynchronize(void* s) {
    (void)s;
    return 0;
}
int hipStreamCreateWithFlags(void** s, unsigned f) {
    static int one;
    (void)f;
    *s = &one;
    return 0;
}
int hipStreamDestroy(void* s) {
    (void)s;
    return 0;
}

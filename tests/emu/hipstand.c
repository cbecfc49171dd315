/*
 * TEST INFRASTRUCTURE ONLY: a stand-in for the host side of the HIP runtime,
 * for tests of what the engine allocates and launches on a machine without a
 * GPU.  Loaded with its symbols global before the engine library, it takes
 * that library's HIP calls: device memory is addresses counted against a
 * budget, copies do nothing, and a launch only records the kernel's name,
 * grid, block and LDS bytes.
 */
#include <stdint.h>
#include <stdlib.h>
#include <string.h>

typedef struct { uint32_t x, y, z; } Dim3;

enum { kOutOfMemory = 2, kMaxAllocs = 4096, kMaxKernels = 256, kMaxLaunches = 4096 };

static size_t budget = SIZE_MAX, used;
static uintptr_t next_address = (uintptr_t)1 << 40;
static struct { uintptr_t p; size_t bytes; } allocs[kMaxAllocs];
static int n_allocs, last_error, cus = 256;
static struct { const void* fn; const char* name; } kernels[kMaxKernels];
static int n_kernels;
static struct { const char* name; uint32_t grid, block; size_t lds; } launches[kMaxLaunches];
static int n_launches;
static struct { Dim3 grid, block; size_t lds; void* stream; } config;
static void* fat_binary;

/* ---- the test's side ---- */
void hipstand_budget(size_t bytes) { budget = bytes; }
size_t hipstand_used(void) { return used; }
void hipstand_cus(int n) { cus = n; }
void hipstand_clear(void) { n_launches = 0; }
int hipstand_launches(void) { return n_launches; }
const char* hipstand_launch(int i, uint32_t* grid, uint32_t* block, size_t* lds) {
    *grid = launches[i].grid;
    *block = launches[i].block;
    *lds = launches[i].lds;
    return launches[i].name;
}

#ifdef HIPSTAND_OTHER_BUILD
unsigned long long b3i_build_id(void) { return 1; }
#endif

/* ---- memory ---- */
int hipMalloc(void** p, size_t bytes) {
    *p = NULL;
    if (bytes > budget - (used < budget ? used : budget) || n_allocs == kMaxAllocs) return last_error = kOutOfMemory;
    allocs[n_allocs].p = next_address;
    allocs[n_allocs++].bytes = bytes;
    used += bytes;
    *p = (void*)next_address;
    next_address += (bytes + 4095) / 4096 * 4096;
    return 0;
}
int hipFree(void* p) {
    for (int i = 0; i < n_allocs; i++)
        if (allocs[i].p == (uintptr_t)p) {
            used -= allocs[i].bytes;
            allocs[i] = allocs[--n_allocs];
            return 0;
        }
    return last_error = 1;
}
int hipMemcpy(void* d, const void* s, size_t n, int k) { (void)d; (void)s; (void)n; (void)k; return 0; }
int hipMemcpyAsync(void* d, const void* s, size_t n, int k, void* st) { (void)st; return hipMemcpy(d, s, n, k); }
int hipMemset(void* d, int v, size_t n) { (void)d; (void)v; (void)n; return 0; }

/* ---- device ---- */
int hipGetDevice(int* d) { *d = 0; return 0; }
int hipDeviceGetAttribute(int* v, int a, int d) { (void)a; (void)d; *v = cus; return 0; }
int hipFuncSetAttribute(const void* f, int a, int v) { (void)f; (void)a; (void)v; return 0; }
int hipDeviceSynchronize(void) { return 0; }
int hipStreamSynchronize(void* s) { (void)s; return 0; }
int hipGetLastError(void) {
    int e = last_error;
    last_error = 0;
    return e;
}

/* ---- launches ---- */
void** __hipRegisterFatBinary(const void* data) { (void)data; return &fat_binary; }
void __hipUnregisterFatBinary(void** modules) { (void)modules; }
void __hipRegisterFunction(void** modules, const void* fn, char* device_fn, const char* name, unsigned threads,
        void* tid, void* bid, void* block, void* grid, int* wsize) {
    (void)modules; (void)device_fn; (void)threads; (void)tid; (void)bid; (void)block; (void)grid; (void)wsize;
    if (n_kernels < kMaxKernels) {
        kernels[n_kernels].fn = fn;
        kernels[n_kernels++].name = name;
    }
}
void __hipRegisterVar(void** modules, void* var, char* host, char* dev, int ext, size_t size, int constant, int global) {
    (void)modules; (void)var; (void)host; (void)dev; (void)ext; (void)size; (void)constant; (void)global;
}
int __hipPushCallConfiguration(Dim3 grid, Dim3 block, size_t lds, void* stream) {
    config.grid = grid;
    config.block = block;
    config.lds = lds;
    config.stream = stream;
    return 0;
}
int __hipPopCallConfiguration(Dim3* grid, Dim3* block, size_t* lds, void** stream) {
    *grid = config.grid;
    *block = config.block;
    *lds = config.lds;
    *stream = config.stream;
    return 0;
}
int hipLaunchKernel(const void* fn, Dim3 grid, Dim3 block, void** args, size_t lds, void* stream) {
    (void)args; (void)stream;
    const char* name = "?";
    for (int i = 0; i < n_kernels; i++)
        if (kernels[i].fn == fn) name = kernels[i].name;
    if (n_launches < kMaxLaunches) {
        launches[n_launches].name = name;
        launches[n_launches].grid = grid.x;
        launches[n_launches].block = block.x;
        launches[n_launches++].lds = lds;
    }
    return 0;
}

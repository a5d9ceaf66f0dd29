/* The HIP calls that libhoefem.so makes, without a GPU: memory is host memory, kernels do nothing. Loaded
 * before the library by tests of host code that needs no kernel's results. Counts pinned allocations. */
#include <stddef.h>
#include <stdlib.h>
#include <string.h>

static int pinned_now, pinned_total;
int stub_pinned_now(void) { return pinned_now; }
int stub_pinned_total(void) { return pinned_total; }

int hipMalloc(void** p, size_t n) { *p = malloc(n ? n : 1); return 0; }
int hipFree(void* p) { free(p); return 0; }
int hipHostMalloc(void** p, size_t n, unsigned f) { (void)f; *p = calloc(1, n ? n : 1); ++pinned_now; ++pinned_total; return 0; }
int hipHostFree(void* p) { free(p); --pinned_now; return 0; }
int hipMemcpy(void* d, const void* s, size_t n, int k) { (void)k; memcpy(d, s, n); return 0; }
int hipMemcpyAsync(void* d, const void* s, size_t n, int k, void* st) { (void)k; (void)st; memcpy(d, s, n); return 0; }
int hipMemset(void* d, int v, size_t n) { memset(d, v, n); return 0; }
int hipMemsetAsync(void* d, int v, size_t n, void* st) { (void)st; memset(d, v, n); return 0; }
int hipDeviceGetAttribute(int* v, int a, int d) { (void)a; (void)d; *v = 256; return 0; }
int hipGetDevice(int* d) { *d = 0; return 0; }
int hipGetLastError(void) { return 0; }
const char* hipGetErrorString(int e) { (void)e; return "stub"; }
int hipFuncSetAttribute(const void* f, int a, int v) { (void)f; (void)a; (void)v; return 0; }
int hipLaunchKernel(const void* f, ...) { (void)f; return 0; }
int hipExtLaunchKernel(const void* f, ...) { (void)f; return 0; }
int hipStreamSynchronize(void* s) { (void)s; return 0; }
int hipDeviceSynchronize(void) { return 0; }
int __hipPushCallConfiguration(void) { return 0; }
int __hipPopCallConfiguration(void* g, void* b, size_t* l, void** s) { (void)g; (void)b; *l = 0; *s = 0; return 0; }
void** __hipRegisterFatBinary(const void* d) { static void* h; (void)d; return &h; }
void __hipRegisterFunction(void) {}
void __hipRegisterVar(void) {}
void __hipUnregisterFatBinary(void** h) { (void)h; }

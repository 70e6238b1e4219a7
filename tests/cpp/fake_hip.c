/* A HIP runtime of host memory for tests of error paths on the CPU: preloaded,
 * it takes the calls that libibpm_gpu.so makes.  Kernels do nothing.  A call
 * named to fake_fail fails once, after `skip` calls that succeed, and leaves
 * its error behind for hipGetLastError, as the runtime does. */
#include <stdlib.h>
#include <string.h>

typedef int Err;
enum { OK = 0, OUT_OF_MEMORY = 2, INVALID = 1 };

static const char* fail_name = "";
static int fail_skip = 0;
static Err last = OK;
static int pending = 0;   /* launches and copies since the last synchronisation */

void fake_fail(const char* name, int skip) { fail_name = strdup(name); fail_skip = skip; }
int fake_failed(void) { return !*fail_name; }
int fake_pending(void) { return pending; }
static int uploads = 0;
int fake_uploads(void) { const int n = uploads; uploads = 0; return n; }   /* host to device copies since the last call */

static Err fails(const char* name, Err e) {
    if (strcmp(name, fail_name) || fail_skip-- > 0) return OK;
    fail_name = "";
    return last = e;
}
#define MAY_FAIL(e) do { Err r_ = fails(__func__, e); if (r_) return r_; } while (0)

Err hipGetDeviceCount(int* n) { *n = 1; return OK; }
Err hipGetDevice(int* d) { *d = 0; return OK; }
Err hipSetDevice(int d) { (void)d; return OK; }
Err hipGetLastError(void) { Err e = last; last = OK; return e; }
const char* hipGetErrorString(Err e) { return e == OK ? "no error" : e == OUT_OF_MEMORY ? "out of memory" : "invalid"; }
Err hipStreamCreate(void** s) { *s = malloc(8); return OK; }
Err hipStreamDestroy(void* s) { free(s); return OK; }
Err hipStreamSynchronize(void* s) { (void)s; pending = 0; return OK; }
Err hipMalloc(void** p, size_t n) { MAY_FAIL(OUT_OF_MEMORY); *p = malloc(n); return OK; }
Err hipFree(void* p) { free(p); return OK; }
Err hipHostMalloc(void** p, size_t n, unsigned f) { (void)f; MAY_FAIL(OUT_OF_MEMORY); *p = malloc(n); return OK; }
Err hipHostFree(void* p) { free(p); return OK; }
Err hipMemset(void* p, int v, size_t n) { memset(p, v, n); return OK; }
Err hipMemsetAsync(void* p, int v, size_t n, void* s) { (void)s; memset(p, v, n); ++pending; return OK; }
Err hipMemcpy(void* d, const void* h, size_t n, int k) { (void)k; memmove(d, h, n); return OK; }
Err hipMemcpyAsync(void* d, const void* h, size_t n, int k, void* s) {
    (void)s;
    MAY_FAIL(INVALID);
    uploads += k == 1;
    memmove(d, h, n);
    ++pending;
    return OK;
}
Err hipGetSymbolAddress(void** p, const void* sym) { (void)sym; *p = malloc(1 << 25); return OK; }
typedef struct { unsigned x, y, z; } Dim;
Err __hipPushCallConfiguration(Dim g, Dim b, size_t l, void* s) { (void)g; (void)b; (void)l; (void)s; return OK; }
Err __hipPopCallConfiguration(Dim* g, Dim* b, size_t* l, void** s) {
    memset(g, 0, sizeof *g); memset(b, 0, sizeof *b); *l = 0; *s = 0;
    return OK;
}
Err hipLaunchKernel(const void* f, Dim g, Dim b, void** a, size_t l, void* s) {
    (void)f; (void)g; (void)b; (void)a; (void)l; (void)s;
    ++pending;
    return OK;
}

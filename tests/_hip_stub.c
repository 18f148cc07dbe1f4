/* A HIP runtime without a device, for failure handling on the CPU: device and
 * page-locked memory are host memory, kernels do nothing, and the copies and
 * fills of a stream run when the stream is waited for.  One chosen call fails.
 * stub_pending() counts what is still queued, stub_torn() the transfers from
 * the host whose source changed between queueing and running. */
#include <stddef.h>
#include <stdint.h>
#include <stdlib.h>
#include <string.h>

enum { OK = 0, OUT_OF_MEMORY = 2, UNKNOWN = 999, HOST_TO_DEVICE = 1 };
typedef struct { unsigned x, y, z; } dim;

static struct op { void* dst; const void* src; size_t n; int fill; void* seen; } queue[4096];
static int n_queue, torn, countdown = -1, last_error;

void stub_fail_after(int calls) { countdown = calls; last_error = OK; }
int stub_pending(void) { return n_queue; }
int stub_torn(void) { return torn; }

static int result(int code)
{
    if (countdown < 0 || countdown-- > 0) return OK;
    last_error = code;
    return code;
}
static void run_queue(void)
{
    for (int i = 0; i < n_queue; ++i) {
        struct op* o = &queue[i];
        if (o->seen) {
            torn += memcmp(o->seen, o->src, o->n) != 0;
            free(o->seen);
        }
        if (o->src) memcpy(o->dst, o->src, o->n);
        else memset(o->dst, o->fill, o->n);
    }
    n_queue = 0;
}
static void push(struct op o)
{
    if (n_queue == 4096) abort();
    queue[n_queue++] = o;
}

int hipMalloc(void** p, size_t n)
{
    const int e = result(OUT_OF_MEMORY);
    if (e == OK) *p = calloc(1, n);
    return e;
}
int hipHostMalloc(void** p, size_t n, unsigned flags)
{
    (void)flags;
    return hipMalloc(p, n);
}
int hipFree(void* p) { run_queue(); free(p); return OK; } /* waits for the device, as HIP does */
int hipHostFree(void* p) { return hipFree(p); }
int hipMemcpy(void* d, const void* s, size_t n, int kind)
{
    const int e = result(UNKNOWN);
    (void)kind;
    if (e == OK) memcpy(d, s, n);
    return e;
}
int hipMemcpyAsync(void* d, const void* s, size_t n, int kind, void* stream)
{
    const int e = result(UNKNOWN);
    (void)stream;
    if (e != OK || n == 0) return e;
    void* seen = NULL;
    if (kind == HOST_TO_DEVICE) {
        seen = malloc(n);
        memcpy(seen, s, n);
    }
    push((struct op){d, s, n, 0, seen});
    return OK;
}
int hipMemset(void* d, int v, size_t n)
{
    const int e = result(UNKNOWN);
    if (e == OK) memset(d, v, n);
    return e;
}
int hipMemsetAsync(void* d, int v, size_t n, void* stream)
{
    const int e = result(UNKNOWN);
    (void)stream;
    if (e == OK) push((struct op){d, NULL, n, v, NULL});
    return e;
}
int hipStreamSynchronize(void* stream) { (void)stream; run_queue(); return OK; }
int hipEventSynchronize(void* event) { (void)event; run_queue(); return OK; }
int hipLaunchKernel(const void* f, dim g, dim b, void** args, size_t lds, void* stream)
{
    (void)f; (void)g; (void)b; (void)args; (void)lds; (void)stream;
    return result(UNKNOWN);
}
int hipGetLastError(void) { const int e = last_error; last_error = OK; return e; }
const char* hipGetErrorString(int e) { return e == OUT_OF_MEMORY ? "out of memory" : "error"; }

int hipGetDeviceCount(int* n) { *n = 1; return OK; }
int hipGetDevice(int* d) { *d = 0; return OK; }
int hipDeviceGetAttribute(int* v, int a, int d) { (void)a; (void)d; *v = 256; return OK; }
int hipGetDevicePropertiesR0600(void* p, int d) { (void)p; (void)d; return UNKNOWN; }
int hipStreamCreateWithFlags(void** s, unsigned f) { (void)f; *s = s; return OK; }
int hipStreamDestroy(void* s) { (void)s; return OK; }
int hipEventCreate(void** e) { *e = e; return OK; }
int hipEventCreateWithFlags(void** e, unsigned f) { (void)f; *e = e; return OK; }
int hipEventDestroy(void* e) { (void)e; return OK; }
int hipEventRecord(void* e, void* s) { (void)e; (void)s; return OK; }
int hipEventElapsedTime(float* ms, void* a, void* b) { (void)a; (void)b; *ms = 0.0f; return OK; }
int hipGetSymbolAddress(void** p, const void* symbol)
{
    static char array[1 << 23];
    (void)symbol;
    *p = array;
    return OK;
}
int hipStreamBeginCapture(void* s, int mode) { (void)s; (void)mode; return UNKNOWN; }
int hipStreamEndCapture(void* s, void** g) { (void)s; (void)g; return UNKNOWN; }
int hipGraphInstantiate(void** x, void* g, void* n, char* log, size_t len)
{
    (void)x; (void)g; (void)n; (void)log; (void)len;
    return UNKNOWN;
}
int hipGraphLaunch(void* x, void* s) { (void)x; (void)s; return UNKNOWN; }
int hipGraphDestroy(void* g) { (void)g; return OK; }
int hipGraphExecDestroy(void* x) { (void)x; return OK; }
int __hipPushCallConfiguration(dim g, dim b, size_t lds, void* s) { (void)g; (void)b; (void)lds; (void)s; return OK; }
int __hipPopCallConfiguration(dim* g, dim* b, size_t* lds, void** s)
{
    *g = *b = (dim){1, 1, 1};
    *lds = 0;
    *s = NULL;
    return OK;
}
void** __hipRegisterFatBinary(const void* data) { (void)data; static void* handle; return &handle; }
void __hipUnregisterFatBinary(void** h) { (void)h; }
void __hipRegisterFunction(void) {}
void __hipRegisterVar(void) {}

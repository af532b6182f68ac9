/*
 * hip_fake.c -- a HIP runtime on host memory, preloaded over the library's own, so that the host
 * side of the device layer (csrc/ .hip files) runs without a GPU: allocations are host memory, copies are
 * memcpy, kernels do nothing. Device allocations are counted and can be made to fail.
 */
#include <stddef.h>
#include <stdint.h>
#include <stdlib.h>
#include <string.h>

enum { OK = 0, ERR_VALUE = 1, ERR_OOM = 2 };

static struct block {
    void *p;
    size_t bytes;
} blocks[4096];
static size_t held, limit = (size_t)-1, copied;
static uint32_t fill;  /* every word of the next device allocation */
static int pending;   /* copies queued since the last wait */
static int early;     /* plans freed under them */
static int mallocs, live, captures, copies, fail_in = -1, fail_host_in = -1;

/* what the tests read and set */
int fake_mallocs(void) { return mallocs; }
int fake_live(void) { return live; }
int fake_early_frees(void) { return early; }
int fake_captures(void) { return captures; }
int fake_copies(void) { return copies; }
size_t fake_held(void) { return held; }
size_t fake_copied(void) { size_t c = copied; copied = 0; return c; }   /* since the last call */
void fake_fill(uint32_t word) { fill = word; }
void fake_limit(size_t bytes) { limit = bytes; }
/* after n more device allocations, or pinned ones, every one fails (-1: none does) */
void fake_fail_in(int n) { fail_in = n; }
void fake_fail_host_in(int n) { fail_host_in = n; }

int hipMalloc(void **p, size_t bytes)
{
    mallocs++;
    *p = NULL;
    if (fail_in == 0 || held + bytes > limit)
        return ERR_OOM;
    if (fail_in > 0)
        fail_in--;
    for (int i = 0; i < 4096; i++)
        if (!blocks[i].p) {
            *p = blocks[i].p = calloc(1, bytes ? bytes : 1);
            if (!*p)
                return ERR_OOM;
            for (size_t w = 0; fill && w < bytes / 4; w++)
                ((uint32_t *)*p)[w] = fill;
            fill = 0;
            blocks[i].bytes = bytes;
            held += bytes;
            live++;
            return OK;
        }
    return ERR_OOM;
}

int hipFree(void *p)
{
    if (!p)
        return OK;
    for (int i = 0; i < 4096; i++)
        if (blocks[i].p == p) {
            held -= blocks[i].bytes;
            live--;
            blocks[i].p = NULL;
            free(p);
            return OK;
        }
    abort();   /* not allocated, or freed before */
}

int hipHostMalloc(void **p, size_t bytes, unsigned flags)
{
    (void)flags;
    *p = NULL;
    if (fail_host_in == 0)
        return ERR_OOM;
    if (fail_host_in > 0)
        fail_host_in--;
    *p = calloc(1, bytes ? bytes : 1);
    return *p ? OK : ERR_OOM;
}

int hipHostFree(void *p)
{
    free(p);
    return OK;
}

static int copy(void *d, const void *s, size_t n)
{
    copies++;
    copied += n;
    memcpy(d, s, n);
    return OK;
}
int hipMemcpy(void *d, const void *s, size_t n, int k) { (void)k; return copy(d, s, n); }
int hipMemcpyAsync(void *d, const void *s, size_t n, int k, void *st)
{
    (void)k; (void)st;
    pending++;
    return copy(d, s, n);
}
int hipMemset(void *d, int v, size_t n) { memset(d, v, n); return OK; }
int hipMemsetAsync(void *d, int v, size_t n, void *st) { (void)st; memset(d, v, n); return OK; }
int hipPointerGetAttributes(void *at, const void *p) { (void)at; (void)p; return ERR_VALUE; }

int hipGetDeviceCount(int *n) { *n = 1; return OK; }
int hipGetDevice(int *d) { *d = 0; return OK; }
int hipSetDevice(int d) { (void)d; return OK; }
int hipDeviceGetAttribute(int *v, int a, int d) { (void)a; (void)d; *v = 256; return OK; }
int hipGetLastError(void) { return OK; }
const char *hipGetErrorString(int e) { return e == ERR_OOM ? "out of memory" : "error"; }
int hipGetSymbolAddress(void **p, const void *s)
{
    static char scratch[64];
    (void)s;
    *p = scratch;
    return OK;
}
int hipOccupancyMaxActiveBlocksPerMultiprocessor(int *n, const void *f, int b, size_t l)
{
    (void)f; (void)b; (void)l;
    *n = 4;
    return OK;
}

static int handle(void **h) { *h = malloc(1); return *h ? OK : ERR_OOM; }
int hipStreamCreateWithFlags(void **s, unsigned f) { (void)f; return handle(s); }
int hipStreamDestroy(void *s) { free(s); return OK; }
int hipStreamSynchronize(void *s) { (void)s; pending = 0; return OK; }
int hipEventCreate(void **e) { return handle(e); }
int hipEventCreateWithFlags(void **e, unsigned f) { (void)f; return handle(e); }
int hipEventDestroy(void *e) { free(e); return OK; }
int hipEventRecord(void *e, void *s) { (void)e; (void)s; return OK; }
int hipEventSynchronize(void *e) { (void)e; return OK; }
int hipEventQuery(void *e) { (void)e; return OK; }
int hipEventElapsedTime(float *ms, void *a, void *b) { (void)a; (void)b; *ms = 1.0f; return OK; }

int hipStreamBeginCapture(void *s, int m) { (void)s; (void)m; captures++; return OK; }
int hipStreamEndCapture(void *s, void **g) { (void)s; return handle(g); }
int hipGraphInstantiate(void **x, void *g, void **n, char *b, size_t z)
{
    (void)g; (void)n; (void)b; (void)z;
    return handle(x);
}
int hipGraphLaunch(void *x, void *s) { (void)x; (void)s; return OK; }
int hipGraphDestroy(void *g) { free(g); return OK; }
int hipGraphExecDestroy(void *x) { free(x); return OK; }

struct dim3 { uint32_t x, y, z; };
int __hipPushCallConfiguration(struct dim3 g, struct dim3 b, size_t l, void *s)
{
    (void)g; (void)b; (void)l; (void)s;
    return OK;
}
int __hipPopCallConfiguration(struct dim3 *g, struct dim3 *b, size_t *l, void **s)
{
    *g = *b = (struct dim3){1, 1, 1};
    *l = 0;
    *s = NULL;
    return OK;
}
int hipLaunchKernel(const void *f, struct dim3 g, struct dim3 b, void **a, size_t l, void *s)
{
    (void)f; (void)g; (void)b; (void)a; (void)l; (void)s;
    return OK;
}
void **__hipRegisterFatBinary(const void *d)
{
    static void *h;
    (void)d;
    return &h;
}
void __hipUnregisterFatBinary(void **h) { (void)h; }
void __hipRegisterFunction(void) {}
void __hipRegisterVar(void) {}

/* in front of the library's own: counts the plans freed while a copy may still read them */
static void (*own_plan_free)(void *);
void fake_plan_free_is(void (*own)(void *)) { own_plan_free = own; }
void ag_plan_free(void *plan)
{
    early += pending != 0;
    own_plan_free(plan);
}

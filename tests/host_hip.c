/* A stand-in, in host memory, for the HIP calls libcharm3d.so makes, so that
 * the host side of its entry points (argument checks, allocations and their
 * failures, stream order) can be tested where there is no GPU.  Device memory
 * is malloc'ed, kernels do nothing, fills and host-to-device copies stay queued
 * on their stream until it is synchronised (hipMalloc's limit and the queue are
 * read and set by the hh_ functions). */
#include <pthread.h>
#include <stdint.h>
#include <stdlib.h>
#include <string.h>

enum { OK = 0, INVALID = 1, NOMEM = 2, UNKNOWN = 999 };
enum { MAX_BLOCKS = 4096, MAX_OPS = 4096 };

static pthread_mutex_t mu = PTHREAD_MUTEX_INITIALIZER;
static struct { void *p; size_t bytes; } blk[MAX_BLOCKS];
static struct { void *st, *dst, *src; int value; size_t bytes; } op[MAX_OPS];
static int n_op, streams, launches;
static size_t live, limit = (size_t) 4 << 30;

/* stream NULL: every stream */
static void flush(void *st)
{
    int i, k = 0;
    for (i = 0; i < n_op; i++) {
        if (st && op[i].st != st) { op[k++] = op[i]; continue; }
        if (op[i].src) { memcpy(op[i].dst, op[i].src, op[i].bytes); free(op[i].src); }
        else memset(op[i].dst, op[i].value, op[i].bytes);
    }
    n_op = k;
}

static int push(void *dst, const void *src, int value, size_t bytes, void *st)
{
    if (!dst || n_op == MAX_OPS) return INVALID;
    op[n_op].st = st; op[n_op].dst = dst; op[n_op].value = value; op[n_op].bytes = bytes;
    op[n_op].src = NULL;
    if (src) { op[n_op].src = malloc(bytes + 1); memcpy(op[n_op].src, src, bytes); }
    n_op++;
    return OK;
}

void   hh_limit(size_t bytes) { limit = bytes; }
size_t hh_live(void) { return live; }
int    hh_queued(void) { return n_op; }
int    hh_streams(void) { return streams; }
int    hh_launches(void) { return launches; }

int hipMalloc(void **p, size_t bytes)
{
    int i, rc = NOMEM;
    pthread_mutex_lock(&mu);
    *p = NULL;
    for (i = 0; i < MAX_BLOCKS && blk[i].p; i++) { }
    if (i < MAX_BLOCKS && bytes <= limit && live <= limit - bytes && (*p = malloc(bytes))) {
        blk[i].p = *p; blk[i].bytes = bytes;
        live += bytes;
        rc = OK;
    }
    pthread_mutex_unlock(&mu);
    return rc;
}

int hipFree(void *p)
{
    int i;
    if (!p) return OK;
    pthread_mutex_lock(&mu);
    flush(NULL);
    for (i = 0; i < MAX_BLOCKS && blk[i].p != p; i++) { }
    if (i < MAX_BLOCKS) { live -= blk[i].bytes; blk[i].p = NULL; free(p); }
    pthread_mutex_unlock(&mu);
    return i < MAX_BLOCKS ? OK : INVALID;
}

int hipHostMalloc(void **p, size_t bytes, unsigned flags) { (void) flags; *p = malloc(bytes); return *p ? OK : NOMEM; }
int hipHostFree(void *p) { free(p); return OK; }
int hipHostGetDevicePointer(void **d, void *h, unsigned flags) { (void) flags; *d = h; return OK; }

int hipMemcpyAsync(void *dst, const void *src, size_t bytes, int kind, void *st)
{
    int rc = OK;
    if (!dst || !src) return INVALID;
    pthread_mutex_lock(&mu);
    if (kind == 1) rc = push(dst, src, 0, bytes, st);
    else { flush(st); memcpy(dst, src, bytes); }
    pthread_mutex_unlock(&mu);
    return rc;
}

int hipMemcpy(void *dst, const void *src, size_t bytes, int kind)
{
    (void) kind;
    if (!dst || !src) return INVALID;
    pthread_mutex_lock(&mu);
    flush(NULL);
    memcpy(dst, src, bytes);
    pthread_mutex_unlock(&mu);
    return OK;
}

int hipMemsetAsync(void *dst, int value, size_t bytes, void *st)
{
    int rc;
    pthread_mutex_lock(&mu);
    rc = push(dst, NULL, value, bytes, st);
    pthread_mutex_unlock(&mu);
    return rc;
}

int hipStreamCreate(void **st) { *st = malloc(1); __sync_fetch_and_add(&streams, 1); return OK; }
int hipStreamDestroy(void *st) { free(st); __sync_fetch_and_sub(&streams, 1); return OK; }
int hipStreamWaitEvent(void *st, void *ev, unsigned flags) { (void) st; (void) ev; (void) flags; return OK; }

int hipStreamSynchronize(void *st)
{
    pthread_mutex_lock(&mu);
    flush(st);
    pthread_mutex_unlock(&mu);
    return OK;
}

int hipEventCreate(void **ev) { *ev = malloc(1); return OK; }
int hipEventCreateWithFlags(void **ev, unsigned flags) { (void) flags; *ev = malloc(1); return OK; }
int hipEventDestroy(void *ev) { free(ev); return OK; }
int hipEventRecord(void *ev, void *st) { (void) ev; (void) st; return OK; }
int hipEventSynchronize(void *ev) { (void) ev; pthread_mutex_lock(&mu); flush(NULL); pthread_mutex_unlock(&mu); return OK; }
int hipEventElapsedTime(float *ms, void *a, void *b) { (void) a; (void) b; *ms = 0; return OK; }

int hipGetDeviceCount(int *n) { *n = 1; return OK; }
int hipGetDevice(int *d) { *d = 0; return OK; }
int hipSetDevice(int d) { return d ? INVALID : OK; }
int hipGetLastError(void) { return OK; }
const char *hipGetErrorString(int e) { return e == NOMEM ? "out of memory" : (e ? "invalid value" : "no error"); }
int hipDeviceGetAttribute(int *v, int attr, int dev) { (void) attr; (void) dev; *v = 160 * 1024; return OK; }
int hipGetDevicePropertiesR0600(void *p, int dev) { (void) p; (void) dev; return UNKNOWN; }
int hipFuncGetAttributes(void *a, const void *f) { (void) a; (void) f; return UNKNOWN; }
int hipFuncSetAttribute(const void *f, int attr, int v) { (void) f; (void) attr; (void) v; return OK; }
int hipGetSymbolAddress(void **p, const void *s) { (void) p; (void) s; return UNKNOWN; }

typedef struct { uint32_t x, y, z; } dim;
int hipLaunchKernel(const void *f, dim g, dim b, void **args, size_t lds, void *st)
{
    (void) f; (void) g; (void) b; (void) args; (void) lds; (void) st;
    __sync_fetch_and_add(&launches, 1);
    return OK;
}
int __hipPushCallConfiguration(dim g, dim b, size_t lds, void *st) { (void) g; (void) b; (void) lds; (void) st; return OK; }
int __hipPopCallConfiguration(dim *g, dim *b, size_t *lds, void **st)
{
    g->x = g->y = g->z = b->x = b->y = b->z = 1;
    *lds = 0;
    *st = NULL;
    return OK;
}
void **__hipRegisterFatBinary(const void *d) { static void *h; (void) d; return &h; }
void __hipUnregisterFatBinary(void **h) { (void) h; }
void __hipRegisterFunction(void **h, const void *f, char *n, const char *d, unsigned l, void *t, void *b, dim *bd, dim *gd, int *w)
{
    (void) h; (void) f; (void) n; (void) d; (void) l; (void) t; (void) b; (void) bd; (void) gd; (void) w;
}
void __hipRegisterVar(void **h, void *v, char *n, const char *d, int e, size_t s, int c, int g)
{
    (void) h; (void) v; (void) n; (void) d; (void) e; (void) s; (void) c; (void) g;
}

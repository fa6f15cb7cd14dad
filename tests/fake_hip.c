/*
 * A HIP runtime without a GPU, for tests of the library's host code: device
 * memory is host memory with a capacity, copies are made at once, a kernel is
 * a line in the log and a step of the clock, and the select kernels post the
 * frontier sizes of a prepared BFS.  Loaded globally ahead of libalbba.so, so
 * that the library's calls come here.
 */
#include <hip/hip_runtime_api.h>

#include <stdlib.h>
#include <string.h>
#include <sys/mman.h>
#include <unistd.h>

#include "../albba_amd/csrc/albd.h"

#define API __attribute__((visibility("default")))
#define DEVICES 2

/* ---- what a test sets and reads ---- */
#define MAX_LEVELS 64
API long long fake_capacity = 1ll << 40; /* bytes of one device */
API long long fake_live_bytes[DEVICES], fake_live_blocks[DEVICES];
API long long fake_pinned_max = 1ll << 40; /* larger pinned blocks fail */
API int fake_malloc_us;                  /* what an allocation takes */
API int fake_wrong_device;               /* launches on a stream of another than the current device */
API int fake_levels, fake_level;
API long long fake_frontier[MAX_LEVELS + 1], fake_edges[MAX_LEVELS + 1];
API char fake_log[1 << 22];              /* kernel names, one a line */
API long long fake_build_max[MAX_LEVELS * 64]; /* of the push finalizes, in turn */
API int fake_finalizes;
static size_t log_len;

API void fake_log_reset(void)
{
    fake_log[0] = 0;
    log_len = 0;
}

/* ---- kernels ---- */
static struct {
    const void *host;
    const char *name;
} kernels[4096];
static int nkernels;
static int current;
static double now; /* ms */

API void **__hipRegisterFatBinary(const void *data)
{
    static void *handle[1];
    (void)data;
    return handle;
}
API void __hipUnregisterFatBinary(void **m) { (void)m; }
API void __hipRegisterVar(void **m, void *var, char *hv, char *dv, int e, size_t s, int c, int g)
{
    (void)m; (void)var; (void)hv; (void)dv; (void)e; (void)s; (void)c; (void)g;
}
API void __hipRegisterFunction(void **m, const void *host, char *dev, const char *name, unsigned l, void *t, void *b,
                               void *bd, void *gd, int *w)
{
    (void)m; (void)dev; (void)l; (void)t; (void)b; (void)bd; (void)gd; (void)w;
    if (nkernels < 4096) {
        kernels[nkernels].host = host;
        kernels[nkernels++].name = name;
    }
}
static struct {
    dim3 grid, block;
    size_t shmem;
    hipStream_t stream;
} call;
API hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t s, hipStream_t st)
{
    call.grid = g;
    call.block = b;
    call.shmem = s;
    call.stream = st;
    return hipSuccess;
}
API hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *s, hipStream_t *st)
{
    *g = call.grid;
    *b = call.block;
    *s = call.shmem;
    *st = call.stream;
    return hipSuccess;
}

/* the counters that the select kernel of level `fake_level` leaves */
static void select_level(void **args)
{
    const albd_state *st = (const albd_state *)args[1];
    const albd_select_args *sel = (const albd_select_args *)args[2];
    if (sel->first) fake_level = 0;
    const int l = fake_level < fake_levels ? fake_level : fake_levels;
    albd_counters *c = st->ctr;
    c->frontier = l < fake_levels ? (unsigned long long)fake_frontier[l] : 0;
    c->frontier_edges = l < fake_levels ? (unsigned long long)fake_edges[l] : 0;
    c->heur_choice = 0; /* a push */
    c->sel_choice = sel->forced >= 0 ? sel->forced : 0;
    ++fake_level;
}

API hipError_t hipLaunchKernel(const void *f, dim3 grid, dim3 block, void **args, size_t shmem, hipStream_t s)
{
    (void)grid; (void)block; (void)shmem;
    const char *name = "?";
    for (int i = 0; i < nkernels; ++i)
        if (kernels[i].host == f) name = kernels[i].name;
    const size_t n = strlen(name);
    if (log_len + n + 2 < sizeof fake_log) {
        memcpy(fake_log + log_len, name, n);
        log_len += n;
        memcpy(fake_log + log_len++, "\n", 2);
    }
    if (s && *(int *)s != current) ++fake_wrong_device;
    /* a pull costs ten of the others, so that a push is the fastest choice */
    now += strstr(name, "k_pull") ? 10 : 1;
    if (strstr(name, "k_select")) select_level(args);
    if (strstr(name, "k_words_to_queueILb1") && fake_finalizes < MAX_LEVELS * 64)
        fake_build_max[fake_finalizes++] = *(const long long *)args[4];
    return hipSuccess;
}

/* ---- memory ---- */
typedef struct {
    size_t bytes;
    int device;
} head_t;
#define HEAD 4096
#define BIG (1u << 20)

API hipError_t hipMalloc(void **p, size_t bytes)
{
    *p = NULL;
    if (fake_malloc_us) usleep((useconds_t)fake_malloc_us);
    if (fake_live_bytes[current] + (long long)bytes > fake_capacity) return hipErrorOutOfMemory;
    /* (large ones by mmap, so that what is not touched takes no memory) */
    char *m = bytes < BIG ? (char *)calloc(1, bytes + HEAD) : (char *)mmap(NULL, bytes + HEAD, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
    if (!m || m == MAP_FAILED) return hipErrorOutOfMemory;
    ((head_t *)m)->bytes = bytes;
    ((head_t *)m)->device = current;
    fake_live_bytes[current] += (long long)bytes;
    ++fake_live_blocks[current];
    *p = m + HEAD;
    return hipSuccess;
}
API hipError_t hipFree(void *p)
{
    if (!p) return hipSuccess;
    head_t *h = (head_t *)((char *)p - HEAD);
    fake_live_bytes[h->device] -= (long long)h->bytes;
    --fake_live_blocks[h->device];
    if (h->bytes < BIG) free(h);
    else munmap(h, h->bytes + HEAD);
    return hipSuccess;
}
API hipError_t hipHostMalloc(void **p, size_t bytes, unsigned f)
{
    (void)f;
    *p = (long long)bytes > fake_pinned_max ? NULL : calloc(1, bytes);
    return *p ? hipSuccess : hipErrorOutOfMemory;
}
API hipError_t hipHostFree(void *p)
{
    free(p);
    return hipSuccess;
}
API hipError_t hipHostGetDevicePointer(void **d, void *h, unsigned f)
{
    (void)f;
    *d = h;
    return hipSuccess;
}
API hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind k, hipStream_t st)
{
    (void)k; (void)st;
    memcpy(d, s, n);
    return hipSuccess;
}
API hipError_t hipMemcpyWithStream(void *d, const void *s, size_t n, hipMemcpyKind k, hipStream_t st)
{
    return hipMemcpyAsync(d, s, n, k, st);
}
API hipError_t hipMemsetAsync(void *d, int v, size_t n, hipStream_t st)
{
    (void)st;
    memset(d, v, n);
    return hipSuccess;
}
API hipError_t hipGetSymbolAddress(void **p, const void *sym)
{
    (void)sym;
    static char scratch[1 << 20];
    *p = scratch;
    return hipSuccess;
}

/* ---- devices, streams, events ---- */
API hipError_t hipGetDeviceCount(int *n)
{
    *n = DEVICES;
    return hipSuccess;
}
API hipError_t hipGetDevice(int *d)
{
    *d = current;
    return hipSuccess;
}
API hipError_t hipSetDevice(int d)
{
    current = d;
    return hipSuccess;
}
API hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600 *p, int d)
{
    (void)d;
    memset(p, 0, sizeof *p);
    p->multiProcessorCount = 256;
    p->warpSize = 64;
    strcpy(p->gcnArchName, "gfx950");
    return hipSuccess;
}
API hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t a, int d)
{
    (void)a; (void)d;
    *v = 100000; /* a clock rate in kHz */
    return hipSuccess;
}
API hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int *n, const void *f, int b, size_t s)
{
    (void)f; (void)b; (void)s;
    *n = 2;
    return hipSuccess;
}
API hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned f)
{
    (void)f;
    int *x = (int *)malloc(sizeof *x);
    *x = current;
    *s = (hipStream_t)x;
    return hipSuccess;
}
API hipError_t hipStreamDestroy(hipStream_t s)
{
    free((void *)s);
    return hipSuccess;
}
API hipError_t hipStreamQuery(hipStream_t s)
{
    (void)s;
    return hipSuccess;
}
API hipError_t hipStreamSynchronize(hipStream_t s)
{
    (void)s;
    return hipSuccess;
}
API int hipGetStreamDeviceId(hipStream_t s) { return s ? *(int *)s : current; }
API hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned f)
{
    (void)f;
    *e = (hipEvent_t)calloc(1, sizeof(double));
    return hipSuccess;
}
API hipError_t hipEventCreate(hipEvent_t *e) { return hipEventCreateWithFlags(e, 0); }
API hipError_t hipEventDestroy(hipEvent_t e)
{
    free((void *)e);
    return hipSuccess;
}
API hipError_t hipEventRecord(hipEvent_t e, hipStream_t s)
{
    (void)s;
    *(double *)e = now;
    return hipSuccess;
}
API hipError_t hipEventSynchronize(hipEvent_t e)
{
    (void)e;
    return hipSuccess;
}
API hipError_t hipEventElapsedTime(float *ms, hipEvent_t a, hipEvent_t b)
{
    *ms = (float)(*(double *)b - *(double *)a);
    return hipSuccess;
}
API hipError_t hipGetLastError(void) { return hipSuccess; }
API const char *hipGetErrorString(hipError_t e) { return e == hipErrorOutOfMemory ? "out of memory" : "?"; }

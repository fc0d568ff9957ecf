/* A stand-in for the HIP runtime calls the library's host code makes, for
 * tests of that code without a GPU (loaded before the library, into the global
 * symbol scope).  Device memory is host memory, handed out page after page
 * without gaps, so that two allocations can touch; a copy that leaves its
 * allocation fails; kernels do not run, but their first argument is noted.
 * Allocations can be made to fail. */
#define _GNU_SOURCE
#include <stddef.h>
#include <stdint.h>
#include <stdlib.h>
#include <string.h>
#include <sys/mman.h>

enum { kOk = 0, kInvalid = 1, kOutOfMemory = 2, kPage = 4096, kMaxBlocks = 65536 };

struct block {
    char *base;
    size_t bytes;
    int live, launched; /* launched: kernels whose first argument is its base */
};
static struct block blocks[kMaxBlocks];
static int nblocks;
static char *arena, *arena_end, *top;
static int fail_in;        /* > 0: this many allocations from now, one fails */
static const void *table;  /* where the last copy of exactly table_bytes went */
static size_t table_bytes;

static struct block *block_of(const void *p)
{
    for (int k = nblocks - 1; k >= 0; --k)
        if (blocks[k].live && (const char *)p >= blocks[k].base && (const char *)p < blocks[k].base + blocks[k].bytes)
            return &blocks[k];
    return NULL;
}

static int inside(const void *p, size_t n)
{
    const struct block *b = block_of(p);
    return n == 0 || (b && (const char *)p + n <= b->base + b->bytes);
}

/* ---- what the tests ask for */
void fake_fail_in(int k) { fail_in = k; }
int fake_pending_failure(void) { return fail_in; }
void fake_watch_table(size_t bytes) { table_bytes = bytes; table = NULL; }
/* 1: the allocation the last watched copy went to is still there, and unchanged at its start */
int fake_table_holds(const void *expected)
{
    return table && inside(table, table_bytes) && memcmp(table, expected, table_bytes) == 0;
}
/* live allocations of `bytes`, and how many of them were a kernel's first argument */
int fake_launched(size_t bytes)
{
    int n = 0;
    for (int k = 0; k < nblocks; ++k)
        n += blocks[k].live && blocks[k].bytes == bytes && blocks[k].launched;
    return n;
}

/* ---- memory */
int hipMalloc(void **p, size_t n)
{
    if (!arena) {
        const size_t room = 64ull << 30;
        arena = mmap(NULL, room, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
        if (arena == MAP_FAILED)
            abort();
        arena_end = arena + room;
        top = arena;
    }
    if (fail_in > 0 && --fail_in == 0)
        return kOutOfMemory;
    const size_t pages = (n + kPage - 1) / kPage * kPage;
    if (nblocks == kMaxBlocks || top + pages > arena_end)
        return kOutOfMemory;
    blocks[nblocks++] = (struct block){top, n, 1, 0};
    *p = top;
    memset(top, 0xA5, n < kPage ? n : kPage); /* not what it was before, nor zero */
    top += pages;
    return kOk;
}
int hipFree(void *p)
{
    struct block *b = p ? block_of(p) : NULL;
    if (p && (!b || b->base != p))
        return kInvalid;
    if (b)
        b->live = 0;
    return kOk;
}
int hipHostMalloc(void **p, size_t n, unsigned flags) { (void)flags; *p = malloc(n); return *p ? kOk : kOutOfMemory; }
int hipHostFree(void *p) { free(p); return kOk; }
int hipMemset(void *p, int v, size_t n) { if (!inside(p, n)) return kInvalid; memset(p, v, n); return kOk; }
int hipMemcpyAsync(void *dst, const void *src, size_t n, int kind, void *st)
{
    (void)st;
    if ((kind != 1 && !inside(src, n)) || (kind != 2 && !inside(dst, n))) /* 1: to, 2: from the device */
        return kInvalid;
    memcpy(dst, src, n);
    if (kind == 1 && n == table_bytes)
        table = dst;
    return kOk;
}
int hipMemGetInfo(size_t *f, size_t *t) { *f = *t = 64ull << 30; return kOk; }
int hipGetSymbolAddress(void **p, const void *s) { (void)p; (void)s; return kInvalid; }

/* ---- launches */
struct dim3_ { uint32_t x, y, z; };
int __hipPushCallConfiguration(struct dim3_ g, struct dim3_ b, size_t lds, void *st)
{
    (void)g; (void)b; (void)lds; (void)st;
    return kOk;
}
int __hipPopCallConfiguration(struct dim3_ *g, struct dim3_ *b, size_t *lds, void **st)
{
    *g = *b = (struct dim3_){1, 1, 1};
    *lds = 0;
    *st = NULL;
    return kOk;
}
int hipLaunchKernel(const void *f, struct dim3_ g, struct dim3_ b, void **args, size_t lds, void *st)
{
    (void)f; (void)g; (void)b; (void)lds; (void)st;
    const void *first;
    memcpy(&first, args[0], sizeof first);
    for (int k = 0; k < nblocks; ++k)
        if (blocks[k].live && blocks[k].base == first)
            blocks[k].launched = 1;
    return kOk;
}

/* ---- devices, streams, events, graphs */
int hipGetDeviceCount(int *n) { *n = 1; return kOk; }
int hipGetDevice(int *d) { *d = 0; return kOk; }
int hipDeviceGetAttribute(int *v, int a, int d) { (void)a; (void)d; *v = 256; return kOk; }
int hipOccupancyMaxActiveBlocksPerMultiprocessor(int *n, const void *f, int b, size_t lds)
{
    (void)f; (void)b; (void)lds;
    *n = 2;
    return kOk;
}
int hipGetLastError(void) { return kOk; }
const char *hipGetErrorString(int e) { return e ? "an error of the stand-in runtime" : "no error"; }
static int handle;
int hipStreamCreateWithFlags(void **s, unsigned f) { (void)f; *s = &handle; return kOk; }
int hipStreamDestroy(void *s) { (void)s; return kOk; }
int hipStreamSynchronize(void *s) { (void)s; return kOk; }
int hipStreamBeginCapture(void *s, int m) { (void)s; (void)m; return kOk; }
int hipStreamEndCapture(void *s, void **g) { (void)s; *g = &handle; return kOk; }
int hipThreadExchangeStreamCaptureMode(int *m) { (void)m; return kOk; }
int hipGraphInstantiate(void **e, void *g, void *n, char *b, size_t s)
{
    (void)g; (void)n; (void)b; (void)s;
    *e = &handle;
    return kOk;
}
int hipGraphLaunch(void *e, void *s) { (void)e; (void)s; return kOk; }
int hipGraphDestroy(void *g) { (void)g; return kOk; }
int hipGraphExecDestroy(void *e) { (void)e; return kOk; }
int hipEventCreate(void **e) { *e = &handle; return kOk; }
int hipEventCreateWithFlags(void **e, unsigned f) { (void)f; *e = &handle; return kOk; }
int hipEventDestroy(void *e) { (void)e; return kOk; }
int hipEventRecord(void *e, void *s) { (void)e; (void)s; return kOk; }
int hipEventSynchronize(void *e) { (void)e; return kOk; }
int hipEventElapsedTime(float *ms, void *a, void *b) { (void)a; (void)b; *ms = 1.0f; return kOk; }

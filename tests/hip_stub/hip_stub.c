/*
 * A stand-in of the HIP runtime for libclm's host code, so that its launches and
 * copies can be looked at on a machine without a GPU.  Test infrastructure only.
 *
 * Device memory is host memory, kernels do nothing and are recorded (name,
 * grid, block, the first bytes of their first argument).  A copy to the device
 * from pageable memory is taken at its word: the source is read when the stream
 * is waited for, and one that no longer holds its bytes by then is counted
 * (stub_lost).  stub_int: what copies of one int back from the device return.
 * Loaded with RTLD_GLOBAL before libclm.so, its symbols come first.
 */
#define _GNU_SOURCE
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>
#include <sys/mman.h>

typedef struct { uint32_t x, y, z; } dim3;
enum { ARG = 256, NAMES = 4096, LAUNCHES = 4096, COPIES = 4096 };

static struct { const void *fn; const char *name; } g_names[NAMES];
static int g_nnames;
static struct { const char *name; dim3 grid, block; unsigned char arg[ARG]; } g_launch[LAUNCHES];
static int g_nlaunch;
static struct { void *dst; const void *src; size_t n; uint64_t sum; } g_copy[COPIES];
static int g_ncopy;
static long g_lost;
static int g_int = 0;

static uint64_t sum_of(const void *p, size_t n)
{
    const unsigned char *c = p;
    uint64_t h = 1469598103934665603ull;
    for (size_t i = 0; i < n; i++) h = (h ^ c[i]) * 1099511628211ull;
    return h;
}

static void finish_copies(void)
{
    for (int i = 0; i < g_ncopy; i++) {
        if (sum_of(g_copy[i].src, g_copy[i].n) != g_copy[i].sum) g_lost++;
        memcpy(g_copy[i].dst, g_copy[i].src, g_copy[i].n);
    }
    g_ncopy = 0;
}

/* ------------------------------------------------------- what a test reads */
int stub_launches(void) { return g_nlaunch; }
const char *stub_name(int i) { return g_launch[i].name; }
const void *stub_arg(int i) { return g_launch[i].arg; }
uint32_t stub_block(int i) { return g_launch[i].block.x; }
uint32_t stub_grid(int i) { return g_launch[i].grid.x; }
long stub_lost(void) { return g_lost; }
void stub_int(int v) { g_int = v; }
void stub_reset(void) { g_nlaunch = 0; g_lost = 0; }

/* ------------------------------------------------------------- the runtime */
void **__hipRegisterFatBinary(const void *d) { static void *h; (void)d; return &h; }
void __hipUnregisterFatBinary(void **m) { (void)m; }
void __hipRegisterFunction(void **m, const void *fn, char *dev, const char *name, unsigned lim, void *t, void *b,
                           void *bd, void *gd, int *ws)
{
    (void)m; (void)dev; (void)lim; (void)t; (void)b; (void)bd; (void)gd; (void)ws;
    if (g_nnames < NAMES) {
        g_names[g_nnames].fn = fn;
        g_names[g_nnames++].name = name;
    }
}
void __hipRegisterVar(void **m, void *v, char *h, char *d, int e, size_t n, int c, int g)
{
    (void)m; (void)v; (void)h; (void)d; (void)e; (void)n; (void)c; (void)g;
}

static dim3 g_cfg_grid, g_cfg_block;
static size_t g_cfg_lds;
static void *g_cfg_stream;
int __hipPushCallConfiguration(dim3 grid, dim3 block, size_t lds, void *stream)
{
    g_cfg_grid = grid;
    g_cfg_block = block;
    g_cfg_lds = lds;
    g_cfg_stream = stream;
    return 0;
}
int __hipPopCallConfiguration(dim3 *grid, dim3 *block, size_t *lds, void **stream)
{
    *grid = g_cfg_grid;
    *block = g_cfg_block;
    *lds = g_cfg_lds;
    *stream = g_cfg_stream;
    return 0;
}
int hipLaunchKernel(const void *fn, dim3 grid, dim3 block, void **args, size_t lds, void *stream)
{
    (void)lds; (void)stream;
    if (g_nlaunch == LAUNCHES) return 0;
    const char *name = "?";
    for (int i = 0; i < g_nnames; i++)
        if (g_names[i].fn == fn) name = g_names[i].name;
    g_launch[g_nlaunch].name = name;
    g_launch[g_nlaunch].grid = grid;
    g_launch[g_nlaunch].block = block;
    memcpy(g_launch[g_nlaunch].arg, args[0], ARG); /* on the caller's stack */
    g_nlaunch++;
    return 0;
}

int hipGetDeviceCount(int *n) { *n = 1; return 0; }
int hipSetDevice(int d) { (void)d; return 0; }
int hipGetDevicePropertiesR0600(void *p, int d) { (void)p; (void)d; return 1; }
int hipGetLastError(void) { return 0; }
const char *hipGetErrorString(int e) { return e ? "error" : "no error"; }
int hipFuncSetAttribute(const void *f, int a, int v) { (void)f; (void)a; (void)v; return 0; }
int hipOccupancyMaxActiveBlocksPerMultiprocessor(int *n, const void *f, int b, size_t l)
{
    (void)f; (void)b; (void)l;
    *n = 1;
    return 0;
}
int hipGetSymbolAddress(void **p, const void *s)
{
    (void)s;
    *p = mmap(NULL, (size_t)1 << 30, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
    return *p == MAP_FAILED;
}
int hipMalloc(void **p, size_t n) { *p = calloc(1, n); return *p ? 0 : 2; }
int hipFree(void *p) { finish_copies(); free(p); return 0; }
int hipMemsetAsync(void *p, int v, size_t n, void *s) { (void)s; memset(p, v, n); return 0; }
int hipMemcpyAsync(void *dst, const void *src, size_t n, int kind, void *s)
{
    (void)s;
    if (kind == 1 && g_ncopy < COPIES) {
        g_copy[g_ncopy].dst = dst;
        g_copy[g_ncopy].src = src;
        g_copy[g_ncopy].n = n;
        g_copy[g_ncopy++].sum = sum_of(src, n);
        return 0;
    }
    finish_copies();
    memcpy(dst, src, n);
    if (kind == 2 && n == sizeof g_int && g_int) memcpy(dst, &g_int, n);
    return 0;
}
int hipMemcpy(void *dst, const void *src, size_t n, int kind) { (void)kind; finish_copies(); memcpy(dst, src, n); return 0; }
int hipStreamCreateWithFlags(void **s, unsigned f) { (void)f; *s = (void *)8; return 0; }
int hipStreamDestroy(void *s) { (void)s; return 0; }
int hipStreamSynchronize(void *s) { (void)s; finish_copies(); return 0; }
int hipEventCreate(void **e) { *e = (void *)16; return 0; }
int hipEventDestroy(void *e) { (void)e; return 0; }
int hipEventRecord(void *e, void *s) { (void)e; (void)s; return 0; }
int hipEventSynchronize(void *e) { (void)e; finish_copies(); return 0; }
int hipEventElapsedTime(float *ms, void *a, void *b) { (void)a; (void)b; *ms = 0.f; return 0; }
int hipStreamBeginCapture(void *s, int m) { (void)s; (void)m; return 0; }
int hipStreamEndCapture(void *s, void **g) { (void)s; *g = (void *)24; return 0; }
int hipGraphInstantiate(void **e, void *g, void **n, char *l, size_t z) { (void)g; (void)n; (void)l; (void)z; *e = (void *)32; return 0; }
int hipGraphLaunch(void *e, void *s) { (void)e; (void)s; return 0; }
int hipGraphExecDestroy(void *e) { (void)e; return 0; }
int hipGraphDestroy(void *g) { (void)g; return 0; }

/* A HIP runtime for host-path tests on a machine without a GPU: it stands in
 * for libamdhip64 under libb40c_hip.so, gives "device" memory from the host
 * heap within a budget, copies and fills at once, and launches nothing.
 *
 * What it checks is what the host code may rely on: hipMemset fills device
 * memory by the null stream and may return before the fill is done, and
 * streams created non-blocking do not wait for the null stream.  A kernel
 * launched on such a stream while a fill by the null stream is outstanding
 * counts as unordered (stub_unordered). */
#include <stdlib.h>
#include <string.h>

enum { kSuccess = 0, kInvalidValue = 1, kOutOfMemory = 2 };

struct block {
    struct block *next;
    size_t bytes;
    void *ptr;
};

static struct block *g_blocks;
static size_t g_used, g_budget = (size_t) 1 << 40, g_refuse_lo = 1, g_refuse_hi = 0;
static int g_last, g_fill_outstanding, g_unordered, g_launches;

void stub_budget(size_t bytes) { g_budget = bytes; }
/* allocations of lo to hi bytes fail (none: lo > hi) */
void stub_refuse(size_t lo, size_t hi) { g_refuse_lo = lo; g_refuse_hi = hi; }
size_t stub_used(void) { return g_used; }
int stub_unordered(void) { return g_unordered; }
int stub_launches(void) { return g_launches; }

static int fail(int e) { return g_last = e; }

int hipMalloc(void **out, size_t bytes)
{
    struct block *b;
    if (g_used + bytes > g_budget || (bytes >= g_refuse_lo && bytes <= g_refuse_hi)) return fail(kOutOfMemory);
    b = malloc(sizeof *b);
    b->ptr = calloc(1, bytes ? bytes : 1);
    b->bytes = bytes;
    b->next = g_blocks;
    g_blocks = b;
    g_used += bytes;
    *out = b->ptr;
    return kSuccess;
}

int hipFree(void *p)
{
    struct block **at = &g_blocks, *b;
    if (!p) return kSuccess;
    g_fill_outstanding = 0; /* (waits for the device) */
    while (*at && (*at)->ptr != p) at = &(*at)->next;
    if (!*at) return fail(kInvalidValue);
    b = *at;
    *at = b->next;
    g_used -= b->bytes;
    free(b->ptr);
    free(b);
    return kSuccess;
}

int hipHostMalloc(void **out, size_t bytes, unsigned flags)
{
    (void) flags;
    *out = calloc(1, bytes);
    return kSuccess;
}
int hipHostFree(void *p) { free(p); return kSuccess; }
int hipHostGetDevicePointer(void **out, void *p, unsigned flags) { (void) flags; *out = p; return kSuccess; }

int hipMemcpy(void *dst, const void *src, size_t n, int kind)
{
    (void) kind;
    memcpy(dst, src, n);
    g_fill_outstanding = 0; /* (a blocking call on the null stream) */
    return kSuccess;
}
int hipMemcpyAsync(void *dst, const void *src, size_t n, int kind, void *stream)
{
    (void) kind;
    (void) stream;
    memcpy(dst, src, n);
    return kSuccess;
}
int hipMemset(void *dst, int value, size_t n)
{
    memset(dst, value, n);
    g_fill_outstanding = 1;
    return kSuccess;
}
int hipMemsetAsync(void *dst, int value, size_t n, void *stream)
{
    memset(dst, value, n);
    if (!stream) g_fill_outstanding = 1;
    return kSuccess;
}

static int launched(void *stream)
{
    g_launches++;
    if (stream && g_fill_outstanding) g_unordered++;
    return kSuccess;
}
struct dim3 { unsigned x, y, z; };
int hipLaunchKernel(const void *f, struct dim3 g, struct dim3 b, void **args, size_t lds, void *stream)
{
    (void) f; (void) g; (void) b; (void) args; (void) lds;
    return launched(stream);
}
int hipLaunchCooperativeKernel(const void *f, struct dim3 g, struct dim3 b, void **args, unsigned lds, void *stream)
{
    (void) f; (void) g; (void) b; (void) args; (void) lds;
    return launched(stream);
}

static struct dim3 g_cfg_grid, g_cfg_block;
static size_t g_cfg_lds;
static void *g_cfg_stream;
int __hipPushCallConfiguration(struct dim3 g, struct dim3 b, size_t lds, void *stream)
{
    g_cfg_grid = g;
    g_cfg_block = b;
    g_cfg_lds = lds;
    g_cfg_stream = stream;
    return kSuccess;
}
int __hipPopCallConfiguration(struct dim3 *g, struct dim3 *b, size_t *lds, void **stream)
{
    *g = g_cfg_grid;
    *b = g_cfg_block;
    *lds = g_cfg_lds;
    *stream = g_cfg_stream;
    return kSuccess;
}

static int g_module;
void **__hipRegisterFatBinary(const void *data) { (void) data; return (void **) &g_module; }
void __hipUnregisterFatBinary(void **m) { (void) m; }
void __hipRegisterFunction(void **m, const void *f, char *name, const char *dname, unsigned threads, void *a, void *b,
                           void *c, void *d, int *e)
{
    (void) m; (void) f; (void) name; (void) dname; (void) threads; (void) a; (void) b; (void) c; (void) d; (void) e;
}
void __hipRegisterVar(void **m, void *var, char *name, char *dname, int ext, size_t size, int constant, int global)
{
    (void) m; (void) var; (void) name; (void) dname; (void) ext; (void) size; (void) constant; (void) global;
}

int hipGetDeviceCount(int *n) { *n = 1; return kSuccess; }
int hipSetDevice(int d) { return d == 0 ? kSuccess : fail(kInvalidValue); }
int hipDeviceGetAttribute(int *v, int attr, int d) { (void) attr; (void) d; *v = 256; return kSuccess; }
int hipDeviceSynchronize(void) { g_fill_outstanding = 0; return kSuccess; }
int hipGetLastError(void) { int e = g_last; g_last = kSuccess; return e; }
const char *hipGetErrorString(int e) { return e == kOutOfMemory ? "out of memory" : "error"; }
int hipGetSymbolAddress(void **p, const void *s) { (void) s; *p = NULL; return fail(kInvalidValue); }
int hipOccupancyMaxActiveBlocksPerMultiprocessor(int *n, const void *f, int block, size_t lds)
{
    (void) f; (void) block; (void) lds;
    *n = 2;
    return kSuccess;
}

int hipStreamCreateWithFlags(void **s, unsigned flags) { (void) flags; *s = malloc(1); return kSuccess; }
int hipStreamDestroy(void *s) { free(s); return kSuccess; }
int hipStreamSynchronize(void *s) { if (!s) g_fill_outstanding = 0; return kSuccess; }
int hipStreamBeginCapture(void *s, int mode) { (void) s; (void) mode; return kSuccess; }
int hipStreamEndCapture(void *s, void **g) { (void) s; *g = NULL; return kSuccess; }
int hipGraphDestroy(void *g) { (void) g; return kSuccess; }
int hipGraphExecDestroy(void *g) { (void) g; return kSuccess; }
int hipGraphInstantiate(void **e, void *g, void *n, char *log, size_t bytes)
{
    (void) g; (void) n; (void) log; (void) bytes;
    *e = NULL;
    return kSuccess;
}
int hipGraphLaunch(void *e, void *s) { (void) e; (void) s; return kSuccess; }
int hipEventCreate(void **e) { *e = malloc(1); return kSuccess; }
int hipEventDestroy(void *e) { free(e); return kSuccess; }
int hipEventRecord(void *e, void *s) { (void) e; (void) s; return kSuccess; }
int hipEventSynchronize(void *e) { (void) e; return kSuccess; }
int hipEventElapsedTime(float *ms, void *a, void *b) { (void) a; (void) b; *ms = 0.f; return kSuccess; }

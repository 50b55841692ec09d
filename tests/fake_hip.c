#define _DEFAULT_SOURCE
/* A HIP runtime for tests of host code without a GPU, preloaded in front of libamdhip64: two devices, streams and
 * events that belong to one of them, device memory that is an address only, launches that are counted and
 * not run. It refuses what HIP refuses: an event recorded and a kernel launched on another device's stream, and a launch of
 * 2^32 or more threads in a dimension. Prototypes are written out, so no HIP header is needed. */
#include <stdint.h>
#include <stdlib.h>
#include <string.h>
#include <unistd.h>

typedef struct { uint32_t x, y, z; } dim3;
typedef struct { int device; } handle;
enum { OK = 0, INVALID_VALUE = 1, OUT_OF_MEMORY = 2, INVALID_CONFIGURATION = 9, INVALID_HANDLE = 400 };

static __thread int current;
static __thread int last_error;
static uintptr_t next_address = 0x100000000000ull;
static uint32_t totals[4];
static uint64_t kept;
static int no_memory;
static long device_syncs, allocations, launches;
static struct { const void *host; char name[200]; long launches; uint64_t threads; } kernels[512];
static int kernel_count;
static struct { dim3 grid, block; size_t shared; void *stream; } config;

static int set(int e) { if(e != OK) last_error = e; return e; }
static int device_of(void *stream) { return stream == NULL ? current : ((handle *)stream)->device; }
static handle *make(void) { handle *h = malloc(sizeof *h); h->device = current; return h; }

/* what a test asks and sets */
long fake_device_syncs(void) { return device_syncs; }
long fake_allocations(void) { return allocations; }
long fake_launches(void) { return launches; }
/* launches of the kernels whose (mangled) name holds `part`, and the most threads along x of one */
long fake_launches_of(const char *part)
{
    long n = 0;
    for(int i = 0; i < kernel_count; ++i) if(strstr(kernels[i].name, part)) n += kernels[i].launches;
    return n;
}
uint64_t fake_threads_of(const char *part)
{
    uint64_t t = 0;
    for(int i = 0; i < kernel_count; ++i) if(strstr(kernels[i].name, part) && kernels[i].threads > t) t = kernels[i].threads;
    return t;
}
/* what a scan_partials_kernel leaves in the totals that it is given */
void fake_set_totals(uint32_t a, uint32_t b) { totals[0] = a; totals[1] = b; }
/* the word that a preprocess_kernel leaves for its first workgroup; whether hipMalloc fails */
void fake_set_kept(uint64_t word) { kept = word; }
void fake_set_no_memory(int yes) { no_memory = yes; }

int hipGetDeviceCount(int *n) { *n = 2; return OK; }
int hipGetDevice(int *d) { *d = current; return OK; }
int hipSetDevice(int d) { if(d < 0 || d > 1) return set(INVALID_VALUE); current = d; return OK; }
int hipDeviceSynchronize(void) { ++device_syncs; usleep(20000); return OK; }
int hipGetLastError(void) { int e = last_error; last_error = OK; return e; }
const char *hipGetErrorString(int e) { return e == INVALID_CONFIGURATION ? "invalid configuration" : "fake HIP error"; }

int hipMalloc(void **p, size_t n)
{
    if(no_memory) return set(OUT_OF_MEMORY);
    ++allocations;
    *p = (void *)next_address;
    next_address += (n + 4095) / 4096 * 4096;
    return OK;
}
int hipFree(void *p) { (void)p; return OK; }
int hipHostMalloc(void **p, size_t n, unsigned flags) { (void)flags; *p = calloc(1, n); return OK; }
int hipHostFree(void *p) { free(p); return OK; }
int hipHostGetDevicePointer(void **d, void *h, unsigned flags) { (void)flags; *d = h; return OK; }
int hipGetSymbolAddress(void **p, const void *s) { (void)s; *p = (void *)next_address; next_address += 1 << 20; return OK; }
int hipMemcpy(void *d, const void *s, size_t n, int k) { (void)d; (void)s; (void)n; (void)k; return OK; }
int hipMemcpyAsync(void *d, const void *s, size_t n, int k, void *st) { (void)st; return hipMemcpy(d, s, n, k); }

int hipStreamCreateWithFlags(void **s, unsigned flags) { (void)flags; *s = make(); return OK; }
int hipStreamDestroy(void *s) { free(s); return OK; }
int hipStreamSynchronize(void *s) { (void)s; return OK; }
int hipStreamWaitEvent(void *s, void *e, unsigned flags) { (void)s; (void)e; (void)flags; return OK; }
int hipEventCreateWithFlags(void **e, unsigned flags) { (void)flags; *e = make(); return OK; }
int hipEventDestroy(void *e) { free(e); return OK; }
int hipEventRecord(void *e, void *s) { return ((handle *)e)->device == device_of(s) ? OK : set(INVALID_HANDLE); }
int hipEventSynchronize(void *e) { (void)e; return OK; }
int hipEventElapsedTime(float *ms, void *a, void *b) { (void)a; (void)b; *ms = 0.0f; return OK; }

void **__hipRegisterFatBinary(const void *data) { (void)data; return (void **)&config; }
void __hipUnregisterFatBinary(void **m) { (void)m; }
void __hipRegisterVar(void **m, void *v, char *h, char *d, int ext, size_t n, int c, int g)
{
    (void)m; (void)v; (void)h; (void)d; (void)ext; (void)n; (void)c; (void)g;
}
void __hipRegisterFunction(void **m, const void *host, char *name, const char *device, unsigned limit, void *t, void *b,
    dim3 *bd, dim3 *gd, int *w)
{
    (void)m; (void)device; (void)limit; (void)t; (void)b; (void)bd; (void)gd; (void)w;
    if(kernel_count == 512) abort();
    kernels[kernel_count].host = host;
    strncpy(kernels[kernel_count++].name, name, sizeof kernels[0].name - 1);
}
int __hipPushCallConfiguration(dim3 grid, dim3 block, size_t shared, void *stream)
{
    config.grid = grid; config.block = block; config.shared = shared; config.stream = stream;
    return OK;
}
int __hipPopCallConfiguration(dim3 *grid, dim3 *block, size_t *shared, void **stream)
{
    *grid = config.grid; *block = config.block; *shared = config.shared; *stream = config.stream;
    return OK;
}
int hipLaunchKernel(const void *host, dim3 grid, dim3 block, void **args, size_t shared, void *stream)
{
    (void)shared;
    const uint64_t x = (uint64_t)grid.x * block.x, y = (uint64_t)grid.y * block.y, z = (uint64_t)grid.z * block.z;
    if(x == 0 || y == 0 || z == 0 || x >> 32 || y >> 32 || z >> 32) return set(INVALID_CONFIGURATION);
    if(device_of(stream) != current) return set(INVALID_HANDLE);
    ++launches;
    for(int i = 0; i < kernel_count; ++i) {
        if(kernels[i].host != host) continue;
        kernels[i].launches += 1;
        if(x > kernels[i].threads) kernels[i].threads = x;
        if(strstr(kernels[i].name, "scan_partials_kernel") && *(uint32_t **)args[2] != NULL)
            for(uint32_t b = 0; b < grid.x; ++b) (*(uint32_t **)args[2])[b] = totals[b];
        if(strstr(kernels[i].name, "preprocess_kernel")) **(uint64_t **)args[18] = kept;
    }
    return OK;
}

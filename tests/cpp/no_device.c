// The HIP runtime calls that the library makes, without a device: memory is counted against a budget and never read or
// written, launches do nothing.  Loaded before the library, so that its host code can be driven on the CPU as far as it waits for no
// result: what a call allocates, and what it does when an allocation fails.
#include <stdint.h>
#include <stdlib.h>
#include <string.h>

typedef struct {
    uint32_t x, y, z;
} dim3;
static int64_t in_use, most, budget = INT64_MAX;
void no_device_budget(int64_t bytes) { budget = bytes; }
void no_device_most_from_now(void) { most = in_use; }
int64_t no_device_in_use(void) { return in_use; }
int64_t no_device_most(void) { return most; }

int hipMalloc(void **p, size_t n)
{
    if (in_use + (int64_t)n > budget) return 2;  // hipErrorOutOfMemory
    char *q = aligned_alloc(256, 256 + (n + 255) / 256 * 256);
    if (!q) return 2;
    *(size_t *)q = n;
    in_use += (int64_t)n;
    if (in_use > most) most = in_use;
    *p = q + 256;
    return 0;
}
int hipFree(void *p)
{
    if (!p) return 0;
    in_use -= (int64_t) * (size_t *)((char *)p - 256);
    free((char *)p - 256);
    return 0;
}
int hipHostMalloc(void **p, size_t n, unsigned flags)
{
    (void)flags;
    *p = aligned_alloc(256, (n + 255) / 256 * 256);
    return *p ? 0 : 2;
}
int hipHostFree(void *p)
{
    free(p);
    return 0;
}
int hipHostGetDevicePointer(void **d, void *h, unsigned flags)
{
    (void)flags;
    *d = h;
    return 0;
}
int hipGetDeviceCount(int *n) { return *n = 1, 0; }
int hipGetDevice(int *d) { return *d = 0, 0; }
int hipSetDevice(int d) { return d ? 101 : 0; }
int hipDeviceGetAttribute(int *v, int attribute, int device)
{
    (void)attribute, (void)device;
    return *v = 256, 0;
}
static int some_handle;
int hipStreamCreate(void **s) { return *s = &some_handle, 0; }
int hipStreamDestroy(void *s) { return (void)s, 0; }
int hipStreamQuery(void *s) { return (void)s, 0; }
int hipStreamSynchronize(void *s) { return (void)s, 0; }
int hipEventCreate(void **e) { return *e = &some_handle, 0; }
int hipEventCreateWithFlags(void **e, unsigned flags) { return (void)flags, *e = &some_handle, 0; }
int hipEventDestroy(void *e) { return (void)e, 0; }
int hipEventElapsedTime(float *ms, void *a, void *b) { return (void)a, (void)b, *ms = 0, 0; }
int hipEventRecord(void *e, void *s) { return (void)e, (void)s, 0; }
int hipEventSynchronize(void *e) { return (void)e, 0; }
int hipMemcpy(void *d, const void *s, size_t n, int kind) { return (void)d, (void)s, (void)n, (void)kind, 0; }
int hipMemcpyAsync(void *d, const void *s, size_t n, int kind, void *stream) { return (void)d, (void)s, (void)n, (void)kind, (void)stream, 0; }
int hipMemset(void *d, int v, size_t n) { return (void)d, (void)v, (void)n, 0; }
int hipMemsetAsync(void *d, int v, size_t n, void *stream) { return (void)d, (void)v, (void)n, (void)stream, 0; }
int hipFuncSetAttribute(const void *f, int attribute, int value) { return (void)f, (void)attribute, (void)value, 0; }
int hipOccupancyMaxActiveBlocksPerMultiprocessor(int *n, const void *f, int block, size_t lds) { return (void)f, (void)block, (void)lds, *n = 1, 0; }
// the last launch's first argument: its first word (a pointer, in structures that begin with one)
static uint64_t launches, first_word;
uint64_t no_device_launches(void) { return launches; }
uint64_t no_device_first_word(void) { return first_word; }
int hipLaunchKernel(const void *f, dim3 grid, dim3 block, void **args, size_t lds, void *stream)
{
    launches++;
    memcpy(&first_word, args[0], 8);
    return (void)f, (void)grid, (void)block, (void)lds, (void)stream, 0;
}
int hipGetLastError(void) { return 0; }
const char *hipGetErrorString(int e) { return (void)e, "no device"; }

// what the compiler's launch syntax and its registration of kernels call
static struct {
    dim3 grid, block;
    size_t lds;
    void *stream;
} pushed;
int __hipPushCallConfiguration(dim3 grid, dim3 block, size_t lds, void *stream)
{
    pushed.grid = grid, pushed.block = block, pushed.lds = lds, pushed.stream = stream;
    return 0;
}
int __hipPopCallConfiguration(dim3 *grid, dim3 *block, size_t *lds, void **stream)
{
    *grid = pushed.grid, *block = pushed.block, *lds = pushed.lds, *stream = pushed.stream;
    return 0;
}
void **__hipRegisterFatBinary(const void *data) { return (void)data, (void **)&pushed.stream; }
void __hipUnregisterFatBinary(void **modules) { (void)modules; }
void __hipRegisterFunction(void **modules, const void *f, char *a, const char *b, unsigned c, void *d, void *e, void *g, void *h, int *i)
{
    (void)modules, (void)f, (void)a, (void)b, (void)c, (void)d, (void)e, (void)g, (void)h, (void)i;
}

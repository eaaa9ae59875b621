/* Host stand-ins for the HIP runtime calls of libtopefft.so: nothing runs on a
 * device, the calls are counted.  Loaded into a process of its own, with global
 * symbols, ahead of the library (test_host_calls.py).  An event keeps its
 * creation flags and the number of launches made before it was recorded; the time
 * between two events is the number of launches between them, in milliseconds. */
#define __HIP_PLATFORM_AMD__
#include <hip/hip_runtime_api.h>
#include <stdlib.h>
#include <string.h>

struct ev {
    unsigned flags;
    long launches;
};

static long launches, copies;
static unsigned last_flags[4096];
static int records;

static unsigned long sequence;

long log_launches(void) { return launches; }
/* Stands for the kernels launched since the last call, in their order. */
unsigned long log_sequence(void)
{
    const unsigned long s = sequence;
    sequence = 0;
    return s;
}
long log_copies(void) { return copies; }
/* Events recorded since the last call: their creation flags. */
int log_records(unsigned *flags, int max)
{
    const int n = records < max ? records : max;
    memcpy(flags, last_flags, (size_t)n * sizeof *flags);
    records = 0;
    return n;
}

static struct {
    dim3 grid, block;
    size_t shmem;
    hipStream_t stream;
} config;
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t m, hipStream_t s)
{
    config.grid = g;
    config.block = b;
    config.shmem = m;
    config.stream = s;
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *m, hipStream_t *s)
{
    *g = config.grid;
    *b = config.block;
    *m = config.shmem;
    *s = config.stream;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void *f, dim3 g, dim3 b, void **a, size_t m, hipStream_t s)
{
    ++launches;
    sequence = sequence * 1000003 + (unsigned long)f;
    return hipSuccess;
}

hipError_t hipGetDeviceCount(int *n) { return *n = 1, hipSuccess; }
hipError_t hipGetDevice(int *d) { return *d = 0, hipSuccess; }
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t a, int d) { return *v = 256, hipSuccess; }
hipError_t hipGetLastError(void) { return hipSuccess; }
hipError_t hipGetSymbolAddress(void **p, const void *s) { return *p = malloc(16), hipSuccess; }

hipError_t hipMalloc(void **p, size_t n) { return *p = malloc(n), *p ? hipSuccess : hipErrorOutOfMemory; }
hipError_t hipFree(void *p) { return free(p), hipSuccess; }
hipError_t hipHostMalloc(void **p, size_t n, unsigned f) { return *p = calloc(1, n), hipSuccess; }
hipError_t hipHostFree(void *p) { return free(p), hipSuccess; }
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind k, hipStream_t t)
{
    ++copies;
    return hipSuccess;
}

hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned f) { return *s = malloc(1), hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t s) { return free(s), hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t s) { return hipSuccess; }

hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned flags)
{
    struct ev *v = calloc(1, sizeof *v);
    v->flags = flags;
    *e = (hipEvent_t)v;
    return hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t *e) { return hipEventCreateWithFlags(e, hipEventDefault); }
hipError_t hipEventDestroy(hipEvent_t e) { return free(e), hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s)
{
    struct ev *v = (struct ev *)e;
    v->launches = launches;
    if (records < (int)(sizeof last_flags / sizeof *last_flags)) last_flags[records++] = v->flags;
    return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t e) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t a, hipEvent_t b)
{
    *ms = (float)(((struct ev *)b)->launches - ((struct ev *)a)->launches);
    return hipSuccess;
}

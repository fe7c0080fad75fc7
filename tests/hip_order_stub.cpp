// A HIP runtime without a device, for test_stream_order.py: memory is the
// host's, kernels do nothing, and work that a non-blocking stream is given
// while a clear on the null stream may still run is counted.  (The null stream
// is ordered with blocking streams only, and hipMemset returns before the
// device is through; a synchronous copy on the null stream waits for it.)
#include <hip/hip_runtime_api.h>

#include <cstdlib>
#include <cstring>

static bool pending = false;   // a clear on the null stream nothing has waited for
static int violations = 0, launches = 0;
static void on_stream(hipStream_t st)
{
    if (st && pending) ++violations;
}

extern "C" {
int order_violations(void) { return violations; }
int order_launches(void) { return launches; }

hipError_t hipGetDeviceCount(int *n) { *n = 1; return hipSuccess; }
hipError_t hipGetDevice(int *d) { *d = 0; return hipSuccess; }
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t, int) { *v = 65536; return hipSuccess; }
hipError_t hipMalloc(void **p, size_t n) { *p = std::calloc(n ? n : 1, 1); return *p ? hipSuccess : hipErrorOutOfMemory; }
hipError_t hipFree(void *p) { std::free(p); return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) { *s = (hipStream_t)std::malloc(8); return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t s) { std::free(s); return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t s) { if (!s) pending = false; return hipSuccess; }
hipError_t hipDeviceSynchronize(void) { pending = false; return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t *e) { *e = (hipEvent_t)std::malloc(8); return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t e) { std::free(e); return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) { *ms = 1.f; return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipGetLastError(void) { return hipSuccess; }
hipError_t hipMemset(void *p, int v, size_t n) { std::memset(p, v, n); pending = true; return hipSuccess; }
hipError_t hipMemsetAsync(void *p, int v, size_t n, hipStream_t s)
{
    on_stream(s);
    std::memset(p, v, n);
    if (!s) pending = true;
    return hipSuccess;
}
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind)
{
    std::memcpy(d, s, n);
    pending = false;
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t st)
{
    on_stream(st);
    std::memcpy(d, s, n);
    return hipSuccess;
}

static dim3 grid_, block_;
static size_t lds_;
static hipStream_t stream_;
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t lds, hipStream_t s)
{
    grid_ = g;
    block_ = b;
    lds_ = lds;
    stream_ = s;
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *lds, hipStream_t *s)
{
    *g = grid_;
    *b = block_;
    *lds = lds_;
    *s = stream_;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void *, dim3, dim3, void **, size_t, hipStream_t s)
{
    on_stream(s);
    ++launches;
    return hipSuccess;
}
}

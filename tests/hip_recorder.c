/* The HIP runtime functions libgfl_moe.so calls, as a recorder for the CPU: device memory is host memory that no kernel
 * touches (hip_recorder_limit bounds it), and each launch appends its kernel's name and dynamic LDS bytes to a log. Loaded with RTLD_GLOBAL before
 * the library, so that the library's own launch code runs against it. */
#include <hip/hip_runtime_api.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

static struct { const void* fn; const char* name; } kernels[1024];
static int n_kernels;
static char launches[1 << 20];
static size_t log_len, left = (size_t)-1;
static hipError_t last = hipSuccess;

static hipError_t done(hipError_t e)
{
    if (e != hipSuccess) last = e;
    return e;
}

void hip_recorder_limit(size_t bytes) { left = bytes; }
void hip_recorder_clear(void) { launches[log_len = 0] = 0; }
const char* hip_recorder_log(void) { return launches; }

static hipError_t launched(const void* fn, size_t lds)
{
    for (int i = 0; i < n_kernels; ++i)
        if (kernels[i].fn == fn)
        {
            log_len += (size_t)snprintf(launches + log_len, sizeof launches - log_len, "%s %zu\n", kernels[i].name,
                                        lds);
            return done(log_len < sizeof launches ? hipSuccess : hipErrorOutOfMemory);
        }
    return done(hipErrorInvalidDeviceFunction);
}

void** __hipRegisterFatBinary(const void* data) { (void)data; return (void**)kernels; }
void __hipUnregisterFatBinary(void** m) { (void)m; }
void __hipRegisterVar(void** m, void* var, char* host, char* dev, int ext, size_t size, int c, int g)
{
    (void)m; (void)var; (void)host; (void)dev; (void)ext; (void)size; (void)c; (void)g;
}
void __hipRegisterFunction(void** m, const void* fn, char* dev, const char* name, unsigned tl, void* t, void* b, void* bd,
                           void* gd, int* ws)
{
    (void)m; (void)dev; (void)tl; (void)t; (void)b; (void)bd; (void)gd; (void)ws;
    if (n_kernels < 1024)
    {
        kernels[n_kernels].fn = fn;
        kernels[n_kernels++].name = name;
    }
}

static dim3 grid, block;
static size_t shared;
static hipStream_t stream;
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t s, hipStream_t st)
{
    grid = g; block = b; shared = s; stream = st;
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t* s, hipStream_t* st)
{
    *g = grid; *b = block; *s = shared; *st = stream;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void* fn, dim3 g, dim3 b, void** args, size_t s, hipStream_t st)
{
    (void)args; (void)st;
    return g.x && g.y && g.z && b.x * b.y * b.z <= 1024 && s <= 163840 ? launched(fn, s) : done(hipErrorInvalidConfiguration);
}

hipError_t hipMalloc(void** p, size_t n)
{
    if (n > left) return done(hipErrorOutOfMemory);
    left -= left == (size_t)-1 ? 0 : n;
    *p = aligned_alloc(256, (n + 255) / 256 * 256);
    return done(*p ? hipSuccess : hipErrorOutOfMemory);
}
hipError_t hipFree(void* p) { free(p); return hipSuccess; }
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind k) { (void)k; memcpy(d, s, n); return hipSuccess; }
hipError_t hipMemset(void* d, int v, size_t n) { (void)d; (void)v; (void)n; return hipSuccess; }
hipError_t hipGetLastError(void) { const hipError_t e = last; last = hipSuccess; return e; }
const char* hipGetErrorString(hipError_t e) { return e == hipErrorOutOfMemory ? "out of memory" : "recorded error"; }
hipError_t hipGetDeviceCount(int* n) { *n = 1; return hipSuccess; }
hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
hipError_t hipSetDevice(int d) { return done(d ? hipErrorInvalidDevice : hipSuccess); }
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t a, int d) { (void)a; (void)d; *v = 256; return hipSuccess; }
hipError_t hipDeviceSynchronize(void) { return hipSuccess; }
hipError_t hipFuncSetAttribute(const void* f, hipFuncAttribute a, int v) { (void)f; (void)a; (void)v; return hipSuccess; }
hipError_t hipFuncGetAttributes(struct hipFuncAttributes* a, const void* f)
{
    (void)f;
    memset(a, 0, sizeof *a);
    a->numRegs = 80;
    return hipSuccess;
}
hipError_t hipStreamIsCapturing(hipStream_t s, hipStreamCaptureStatus* c)
{
    (void)s;
    *c = hipStreamCaptureStatusNone;
    return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned f) { (void)f; *e = (hipEvent_t)kernels; return hipSuccess; }

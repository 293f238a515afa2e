/* fake_hip.c -- the HIP calls of libncmhip.so without a device, for tests of
 * the host code on the CPU: loaded before the library, it takes their place
 * (device addresses are numbers, nothing is copied or run), writes the name of
 * every launch, allocation and synchronisation to a log, and can make the n-th
 * launch fail or report the stream as being captured. */
#define __HIP_PLATFORM_AMD__
#include <hip/hip_runtime_api.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#define LAUNCH_ERROR ((hipError_t)719)

static char log_text[1 << 20];
static size_t log_len;
static int fail_at, capturing;
static size_t next_address = 1u << 20, limit = (size_t)1 << 40;

static void put(const char *s) {
    const size_t n = strlen(s);
    if (log_len + n + 2 > sizeof log_text) return;
    memcpy(log_text + log_len, s, n);
    log_len += n;
    log_text[log_len++] = '\n';
    log_text[log_len] = 0;
}

const char *fake_log(void) { return log_text; }
/* Empties the log; the n-th launch from here on fails (0: none), the stream
 * reports itself as captured or not, and an allocation beyond `max` bytes is
 * refused (0: none is). */
void fake_reset(int n, int capture, size_t max) {
    log_text[log_len = 0] = 0;
    fail_at = n;
    capturing = capture;
    limit = max ? max : (size_t)1 << 40;
}

hipError_t hipGetDeviceCount(int *n) { *n = 1; return hipSuccess; }
hipError_t hipSetDevice(int d) { (void)d; return hipSuccess; }
hipError_t hipGetDeviceProperties(hipDeviceProp_t *p, int d) {   /* (the header's name for its current version) */
    (void)d;
    memset(p, 0, sizeof *p);
    strcpy(p->gcnArchName, "gfx950");
    p->multiProcessorCount = 256;
    return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned f) { (void)f; *s = (hipStream_t)16; return hipSuccess; }
hipError_t hipModuleLoadData(hipModule_t *m, const void *image) { (void)image; *m = (hipModule_t)32; return hipSuccess; }
hipError_t hipModuleGetFunction(hipFunction_t *f, hipModule_t m, const char *name) {
    (void)m;
    *f = (hipFunction_t)strdup(name);
    return hipSuccess;
}
hipError_t hipModuleOccupancyMaxActiveBlocksPerMultiprocessor(int *n, hipFunction_t f, int block, size_t lds) {
    (void)f, (void)block, (void)lds;
    *n = 5;
    return hipSuccess;
}
hipError_t hipModuleLaunchKernel(hipFunction_t f, unsigned gx, unsigned gy, unsigned gz, unsigned bx, unsigned by,
                                 unsigned bz, unsigned lds, hipStream_t s, void **args, void **extra) {
    (void)gx, (void)gy, (void)gz, (void)bx, (void)by, (void)bz, (void)lds, (void)s, (void)args, (void)extra;
    put((const char *)f);
    return fail_at && --fail_at == 0 ? LAUNCH_ERROR : hipSuccess;
}
hipError_t hipMalloc(void **p, size_t n) {
    put("hipMalloc");
    *p = NULL;
    if (n > limit) return hipErrorOutOfMemory;
    *p = (void *)next_address;
    next_address += (n + 4095) & ~(size_t)4095;
    return hipSuccess;
}
hipError_t hipFree(void *p) { (void)p; put("hipFree"); return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t s) { (void)s; put("hipStreamSynchronize"); return hipSuccess; }
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind k, hipStream_t st) {
    (void)d, (void)s, (void)n, (void)k, (void)st;
    put("hipMemcpyAsync");
    return hipSuccess;
}
hipError_t hipMemsetAsync(void *d, int v, size_t n, hipStream_t st) {
    (void)d, (void)v, (void)n, (void)st;
    put("hipMemsetAsync");
    return hipSuccess;
}
hipError_t hipStreamIsCapturing(hipStream_t s, hipStreamCaptureStatus *st) {
    (void)s;
    *st = capturing ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
    return hipSuccess;
}
hipError_t hipGetSymbolAddress(void **p, const void *sym) { (void)sym; *p = (void *)4096; return hipSuccess; }
hipError_t hipGetLastError(void) { return hipSuccess; }
const char *hipGetErrorString(hipError_t e) { return e == LAUNCH_ERROR ? "launch failure" : "error"; }

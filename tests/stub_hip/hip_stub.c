/* A HIP runtime without a device, preloaded by tests/test_host_paths.py under
 * liblbmhip.so: device memory is host memory out of a budget, copies are
 * memcpy, and a kernel launch only adds the kernel's name to a log.  It lets
 * the CPU tests follow the library's host side -- which launches a call makes,
 * what it allocates, what it does when an allocation or a launch fails.
 *
 * Small device-to-host copies (4 or 8 bytes: the counts that Init reads back)
 * deliver stub_count in every word, since no kernel computed them. */
#define _GNU_SOURCE
#include <pthread.h>
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>
#include <hip/hip_runtime_api.h>

#undef hipGetDeviceProperties

/* ---- control, from the test ---------------------------------------------- */
size_t stub_free = (size_t)1 << 40;     /* bytes of device memory left */
uint32_t stub_count = 0;
int stub_devices = 1;
char stub_fail_launch[128] = "";        /* launches of kernels with this in their name fail */
char stub_fail_call[64] = "";           /* so does this runtime call ("memset") */

void (*stub_hook)(void) = NULL;         /* called by every hipStreamSynchronize */

static pthread_mutex_t g_lock = PTHREAD_MUTEX_INITIALIZER;
static char g_log[1 << 22];
static size_t g_logLen = 0;
static __thread hipError_t t_error = hipSuccess;
static __thread int t_device = 0;

static void note(const char * word, const char * name)
{
	pthread_mutex_lock(&g_lock);
	if (g_logLen + strlen(name) + 32 < sizeof(g_log))
		g_logLen += (size_t)sprintf(g_log + g_logLen, "%s %s\n", word, name);
	pthread_mutex_unlock(&g_lock);
}

const char * stub_log(void) { g_log[g_logLen] = '\0'; return g_log; }
void stub_clear(void) { g_logLen = 0; g_log[0] = '\0'; }

static hipError_t result(hipError_t e)
{
	if (e != hipSuccess) t_error = e;
	return e;
}

/* ---- registration and launches ------------------------------------------- */
static struct { const void * fn; char name[256]; } g_fn[4096];
static int g_nFn = 0;

void ** __hipRegisterFatBinary(const void * data) { (void)data; static void * h; return &h; }
void __hipUnregisterFatBinary(void ** h) { (void)h; }
void __hipRegisterVar(void ** m, void * v, char * a, char * b, int e, size_t s, int c, int g)
{
	(void)m; (void)v; (void)a; (void)b; (void)e; (void)s; (void)c; (void)g;
}
void __hipRegisterFunction(void ** m, const void * fn, char * a, const char * name, unsigned n, void * t, void * b,
                           void * bd, void * gd, int * w)
{
	(void)m; (void)a; (void)n; (void)t; (void)b; (void)bd; (void)gd; (void)w;
	if (g_nFn == 4096) return;
	g_fn[g_nFn].fn = fn;
	snprintf(g_fn[g_nFn].name, sizeof(g_fn[0].name), "%s", name);
	++g_nFn;
}
static __thread dim3 t_grid, t_block;
static __thread size_t t_shared;
static __thread hipStream_t t_stream;
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t s, hipStream_t st)
{
	t_grid = g; t_block = b; t_shared = s; t_stream = st;
	return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 * g, dim3 * b, size_t * s, hipStream_t * st)
{
	*g = t_grid; *b = t_block; *s = t_shared; *st = t_stream;
	return hipSuccess;
}
hipError_t hipLaunchKernel(const void * fn, dim3 g, dim3 b, void ** args, size_t s, hipStream_t st)
{
	(void)g; (void)b; (void)args; (void)s; (void)st;
	const char * name = "?";
	for (int i = 0; i < g_nFn; ++i)
		if (g_fn[i].fn == fn) name = g_fn[i].name;
	note("launch", name);
	return result(stub_fail_launch[0] && strstr(name, stub_fail_launch) ? hipErrorLaunchFailure : hipSuccess);
}
hipError_t hipGetLastError(void) { const hipError_t e = t_error; t_error = hipSuccess; return e; }
const char * hipGetErrorName(hipError_t e) { return e == hipErrorOutOfMemory ? "hipErrorOutOfMemory" : "hipError"; }
const char * hipGetErrorString(hipError_t e) { return e == hipErrorOutOfMemory ? "out of memory" : "stub error"; }

/* ---- devices -------------------------------------------------------------- */
hipError_t hipGetDeviceCount(int * n) { *n = stub_devices; return hipSuccess; }
hipError_t hipGetDevice(int * d) { *d = t_device; return hipSuccess; }
hipError_t hipSetDevice(int d) { t_device = d; return hipSuccess; }
hipError_t hipDeviceGetAttribute(int * v, hipDeviceAttribute_t a, int d)
{
	(void)d;
	*v = a == hipDeviceAttributeMultiprocessorCount ? 256 : 163840;
	return hipSuccess;
}
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600 * p, int d)
{
	(void)d;
	memset(p, 0, sizeof(*p));
	strcpy(p->name, "stub");
	return hipSuccess;
}
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int * n, const void * f, int b, size_t s)
{
	(void)f; (void)b; (void)s;
	*n = 4;
	return hipSuccess;
}
hipError_t hipGetSymbolAddress(void ** p, const void * s) { (void)s; *p = NULL; return result(hipErrorInvalidValue); }

/* ---- memory ---------------------------------------------------------------- */
typedef struct { size_t bytes, device; } Head;      /* in front of every allocation */

hipError_t hipMalloc(void ** p, size_t n)
{
	char text[64];
	pthread_mutex_lock(&g_lock);
	const int fits = n <= stub_free;
	if (fits) stub_free -= n;
	pthread_mutex_unlock(&g_lock);
	if (!fits) { note("refused", "hipMalloc"); *p = NULL; return result(hipErrorOutOfMemory); }
	Head * h = (Head *)calloc(1, sizeof(Head) + n);
	h->bytes = n;
	h->device = (size_t)t_device;
	snprintf(text, sizeof(text), "%zu on %d", n, t_device);
	note("malloc", text);
	*p = h + 1;
	return hipSuccess;
}
hipError_t hipFree(void * p)
{
	if (!p) return hipSuccess;
	char text[64];
	Head * h = (Head *)p - 1;
	snprintf(text, sizeof(text), "%zu", h->bytes);
	note("free", text);
	pthread_mutex_lock(&g_lock);
	stub_free += h->bytes;
	pthread_mutex_unlock(&g_lock);
	free(h);
	return hipSuccess;
}
hipError_t hipMemGetInfo(size_t * f, size_t * t) { *f = stub_free; *t = (size_t)1 << 40; return hipSuccess; }
hipError_t hipHostMalloc(void ** p, size_t n, unsigned flags) { (void)flags; *p = calloc(1, n); return hipSuccess; }
hipError_t hipHostFree(void * p) { free(p); return hipSuccess; }
hipError_t hipMemcpyAsync(void * d, const void * s, size_t n, hipMemcpyKind k, hipStream_t st)
{
	(void)st;
	char text[64];
	snprintf(text, sizeof(text), "%zu kind %d", n, (int)k);
	note("copy", text);
	if (k == hipMemcpyDeviceToHost && (n == 4 || n == 8))
		for (size_t i = 0; i < n / 4; ++i) ((uint32_t *)d)[i] = stub_count;
	else
		memcpy(d, s, n);
	return hipSuccess;
}
hipError_t hipMemcpy(void * d, const void * s, size_t n, hipMemcpyKind k) { return hipMemcpyAsync(d, s, n, k, NULL); }
hipError_t hipMemcpy2DAsync(void * d, size_t dp, const void * s, size_t sp, size_t w, size_t h, hipMemcpyKind k, hipStream_t st)
{
	(void)st;
	char text[64];
	snprintf(text, sizeof(text), "%zu x %zu kind %d", h, w, (int)k);
	note("copy2d", text);
	for (size_t i = 0; i < h; ++i) memcpy((char *)d + i * dp, (const char *)s + i * sp, w);
	return hipSuccess;
}
hipError_t hipMemsetAsync(void * d, int v, size_t n, hipStream_t st)
{
	(void)st;
	if (!strcmp(stub_fail_call, "memset")) return result(hipErrorInvalidValue);
	memset(d, v, n);
	return hipSuccess;
}
hipError_t hipMemset(void * d, int v, size_t n) { return hipMemsetAsync(d, v, n, NULL); }

/* ---- streams, events, graphs ---------------------------------------------- */
hipError_t hipStreamCreateWithFlags(hipStream_t * s, unsigned f) { (void)f; *s = (hipStream_t)calloc(1, 8); return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t s) { free(s); return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t s) { (void)s; if (stub_hook) stub_hook(); return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t * e) { *e = (hipEvent_t)calloc(1, 8); return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t * e, unsigned f) { (void)f; return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t e) { free(e); return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) { (void)e; (void)s; return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t e) { (void)e; return hipSuccess; }
hipError_t hipEventElapsedTime(float * ms, hipEvent_t a, hipEvent_t b) { (void)a; (void)b; *ms = 1.0f; return hipSuccess; }
hipError_t hipStreamBeginCapture(hipStream_t s, hipStreamCaptureMode m) { (void)s; (void)m; note("graph", "capture"); return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t s, hipGraph_t * g) { (void)s; *g = (hipGraph_t)calloc(1, 8); return hipSuccess; }
hipError_t hipGraphInstantiate(hipGraphExec_t * x, hipGraph_t g, hipGraphNode_t * n, char * b, size_t s)
{
	(void)g; (void)n; (void)b; (void)s;
	*x = (hipGraphExec_t)calloc(1, 8);
	return hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t x, hipStream_t s) { (void)x; (void)s; note("graph", "replay"); return hipSuccess; }
hipError_t hipGraphDestroy(hipGraph_t g) { free(g); return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t x) { free(x); return hipSuccess; }

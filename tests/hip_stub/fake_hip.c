/* Stand-in for the HIP runtime in CPU tests of the library's host code.
 *
 * Loaded with RTLD_GLOBAL before libfdkhip.so, whose calls then come here:
 * device memory is host memory (filled with fake_fill's byte), kernels do not
 * run, and every call that matters to a test is a line of fake_log():
 *   launch <device> <gx> <gy> <gz> <threads> <lds bytes> <stream>
 *   memcpy <device> <bytes> <kind> <stream>      sync <device>
 *   streamsync <stream>   graphlaunch <stream>
 * fake_fail(name, n) lets the n calls of a function that follow fail.
 * hipEventElapsedTime takes 1 ms for launches of fake_fast_lds bytes of LDS
 * (the last launch before the later event) and 2 ms for all others.
 */
#define __HIP_PLATFORM_AMD__ 1
#include <hip/hip_runtime_api.h>

#include <stdarg.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

static char log_[1 << 20], fail_name[64];
static size_t log_len, fast_lds, last_lds;
static int fail_count, device, fill = 0, capturing;

struct fake_event {
	size_t lds;
};

static void note(const char *fmt, ...)
{
	va_list ap;
	va_start(ap, fmt);
	if (log_len + 256 < sizeof log_)
		log_len += (size_t) vsnprintf(log_ + log_len, 256, fmt, ap);
	va_end(ap);
}

static int failing(const char *name)
{
	if (fail_count > 0 && strcmp(name, fail_name) == 0) {
		--fail_count;
		return 1;
	}
	return 0;
}
#define MAY_FAIL do { if (failing(__func__)) return hipErrorUnknown; } while (0)

const char *fake_log(void) { log_[log_len] = 0; return log_; }
void fake_clear(void) { log_len = 0; }
void fake_fail(const char *name, int n) { snprintf(fail_name, sizeof fail_name, "%s", name); fail_count = n; }
void fake_fill(int byte) { fill = byte; }
void fake_fast_lds(size_t n) { fast_lds = n; }
void fake_capturing(int on) { capturing = on; }

hipError_t hipGetDevice(int *d) { *d = device; return hipSuccess; }
hipError_t hipSetDevice(int d) { MAY_FAIL; device = d; return hipSuccess; }
hipError_t hipGetDeviceCount(int *n) { *n = 2; return hipSuccess; }
hipError_t hipDeviceSynchronize(void) { MAY_FAIL; note("sync %d\n", device); return hipSuccess; }
hipError_t hipGetLastError(void) { return hipSuccess; }
const char *hipGetErrorString(hipError_t e) { return e == hipSuccess ? "no error" : "fake error"; }

hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t a, int d)
{
	(void) d;
	*v = a == hipDeviceAttributeMaxSharedMemoryPerBlock ? 160 * 1024 : 256;
	return hipSuccess;
}

hipError_t hipMalloc(void **p, size_t n)
{
	MAY_FAIL;
	*p = malloc(n ? n : 1);
	if (*p)
		memset(*p, fill, n);
	return *p ? hipSuccess : hipErrorOutOfMemory;
}
hipError_t hipFree(void *p) { free(p); return hipSuccess; }

hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind k, hipStream_t st)
{
	MAY_FAIL;
	note("memcpy %d %zu %d %zu\n", device, n, (int) k, (size_t) st);
	memcpy(d, s, n);
	return hipSuccess;
}
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind k)
{
	return hipMemcpyAsync(d, s, n, k, NULL);
}
hipError_t hipMemset(void *d, int v, size_t n) { memset(d, v, n); return hipSuccess; }

/* a launch's configuration, between the call and the kernel's host stub */
static struct {
	dim3 g, b;
	size_t lds;
	hipStream_t st;
} config;

hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t lds, hipStream_t st)
{
	config.g = g;
	config.b = b;
	config.lds = lds;
	config.st = st;
	return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *lds, hipStream_t *st)
{
	*g = config.g;
	*b = config.b;
	*lds = config.lds;
	*st = config.st;
	return hipSuccess;
}

hipError_t hipLaunchKernel(const void *f, dim3 g, dim3 b, void **args, size_t lds, hipStream_t st)
{
	(void) f;
	(void) args;
	MAY_FAIL;
	last_lds = lds;
	note("launch %d %u %u %u %u %zu %zu\n", device, g.x, g.y, g.z, b.x * b.y * b.z, lds, (size_t) st);
	return hipSuccess;
}
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int *n, const void *f, int b, size_t lds)
{
	(void) f;
	(void) b;
	(void) lds;
	*n = 1;
	return hipSuccess;
}

hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned f)
{
	static size_t next = 1000;
	(void) f;
	*s = (hipStream_t) ++next;
	return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t s) { (void) s; return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t s)
{
	MAY_FAIL;
	note("streamsync %zu\n", (size_t) s);
	return hipSuccess;
}
hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned f)
{
	(void) s;
	(void) e;
	(void) f;
	return hipSuccess;
}
hipError_t hipStreamIsCapturing(hipStream_t s, hipStreamCaptureStatus *c)
{
	(void) s;
	*c = capturing ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
	return hipSuccess;
}
hipError_t hipThreadExchangeStreamCaptureMode(hipStreamCaptureMode *m)
{
	static hipStreamCaptureMode now = hipStreamCaptureModeGlobal;
	const hipStreamCaptureMode was = now;
	now = *m;
	*m = was;
	note("capturemode %d\n", (int) now);
	return hipSuccess;
}
hipError_t hipStreamBeginCapture(hipStream_t s, hipStreamCaptureMode m)
{
	(void) s;
	(void) m;
	return hipSuccess;
}
hipError_t hipStreamEndCapture(hipStream_t s, hipGraph_t *g)
{
	(void) s;
	*g = (hipGraph_t) 1;
	return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t *e, hipGraph_t g, hipGraphNode_t *n, char *l, size_t z)
{
	(void) g;
	(void) n;
	(void) l;
	(void) z;
	*e = (hipGraphExec_t) 1;
	return hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t e, hipStream_t s)
{
	(void) e;
	note("graphlaunch %zu\n", (size_t) s);
	return hipSuccess;
}
hipError_t hipGraphDestroy(hipGraph_t g) { (void) g; return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t e) { (void) e; return hipSuccess; }

hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned f)
{
	(void) f;
	*e = (hipEvent_t) calloc(1, sizeof(struct fake_event));
	return hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t *e) { return hipEventCreateWithFlags(e, 0); }
hipError_t hipEventDestroy(hipEvent_t e) { free((void *) e); return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s)
{
	(void) s;
	((struct fake_event *) e)->lds = last_lds;
	return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t e) { (void) e; return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t a, hipEvent_t b)
{
	(void) a;
	*ms = ((struct fake_event *) b)->lds == fast_lds ? 1.f : 2.f;
	return hipSuccess;
}

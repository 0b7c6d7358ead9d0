/* fake_hip.c -- the HIP runtime calls that libpp_hip.so makes, without a GPU:
 * preloaded into a process, it lets the library's host side run on the CPU.
 * Device memory is host memory (zero, and untouched pages cost nothing), copies
 * copy, and kernels do nothing; allocations and launches are written down, one
 * line each:
 *   malloc BYTES / hostmalloc BYTES
 *   launch KERNEL GRID_X GRID_Y GRID_Z BLOCK_X BLOCK_Y BLOCK_Z
 * As in HIP, a launch of 2^32 threads or more along an axis, of no workgroup,
 * or of more than 1024 threads per workgroup is refused, and device memory ends
 * at fake_hip_limit bytes. */
#define _GNU_SOURCE
#include <stdarg.h>
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>
#include <sys/mman.h>

typedef struct { uint32_t x, y, z; } dim3;
typedef void *stream_t;
enum { OK = 0, OUT_OF_MEMORY = 2, BAD_CONFIGURATION = 9 };

static char *log_text;
static size_t log_len, log_cap;
static int last_error;
static size_t mem_used, mem_limit = (size_t) 288 << 30;

static void note(const char *fmt, ...) {
	if(log_cap - log_len < 4096) log_text = realloc(log_text, log_cap += 1 << 20);
	va_list ap;
	va_start(ap, fmt);
	log_len += (size_t) vsnprintf(log_text + log_len, log_cap - log_len, fmt, ap);
	va_end(ap);
}

const char *fake_hip_log(void) { return log_text ? log_text : ""; }
void fake_hip_clear(void) {
	log_len = 0;
	if(log_text) log_text[0] = 0;
}
void fake_hip_limit(size_t more) { mem_limit = mem_used + more; }

static int failed(int e) { return last_error = e; }

/* memory: a header page holds the size */
enum { PAGE = 4096 };
static void *take(size_t n) {
	char *p = mmap(NULL, n + PAGE, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
	if(p == MAP_FAILED) return NULL;
	*(size_t *) p = n;
	return p + PAGE;
}
static size_t give(void *q) {
	char *p = (char *) q - PAGE;
	const size_t n = *(size_t *) p;
	munmap(p, n + PAGE);
	return n;
}
int hipMalloc(void **p, size_t n) {
	if(n > mem_limit || mem_used > mem_limit - n || !(*p = take(n))) return failed(OUT_OF_MEMORY);
	mem_used += n;
	note("malloc %zu\n", n);
	return OK;
}
int hipFree(void *p) {
	if(p) mem_used -= give(p);
	return OK;
}
int hipHostMalloc(void **p, size_t n, unsigned flags) {
	(void) flags;
	if(!(*p = take(n))) return failed(OUT_OF_MEMORY);
	note("hostmalloc %zu\n", n);
	return OK;
}
int hipHostFree(void *p) {
	if(p) give(p);
	return OK;
}
int hipHostGetDevicePointer(void **d, void *h, unsigned flags) {
	(void) flags;
	*d = h;
	return OK;
}
int hipMemcpy(void *d, const void *s, size_t n, int kind) {
	(void) kind;
	memmove(d, s, n);
	return OK;
}
int hipMemcpyAsync(void *d, const void *s, size_t n, int kind, stream_t st) {
	(void) st;
	return hipMemcpy(d, s, n, kind);
}

/* kernels */
static struct { const void *f; const char *name; } kernels[512];
static int n_kernels;
static void *module;
void **__hipRegisterFatBinary(const void *data) {
	(void) data;
	return &module;
}
void __hipUnregisterFatBinary(void **m) { (void) m; }
void __hipRegisterFunction(void **m, const void *f, char *df, const char *name, unsigned lim, void *a, void *b, void *c, void *d,
                           int *w) {
	(void) m, (void) df, (void) lim, (void) a, (void) b, (void) c, (void) d, (void) w;
	if(n_kernels < 512) {
		kernels[n_kernels].f = f;
		kernels[n_kernels++].name = name;
	}
}
void __hipRegisterVar(void **m, void *v, char *h, char *d, int ext, size_t n, int c, int g) {
	(void) m, (void) v, (void) h, (void) d, (void) ext, (void) n, (void) c, (void) g;
}
static struct { dim3 grid, block; size_t lds; stream_t s; } call;
int __hipPushCallConfiguration(dim3 grid, dim3 block, size_t lds, stream_t s) {
	call.grid = grid, call.block = block, call.lds = lds, call.s = s;
	return OK;
}
int __hipPopCallConfiguration(dim3 *grid, dim3 *block, size_t *lds, stream_t *s) {
	*grid = call.grid, *block = call.block, *lds = call.lds, *s = call.s;
	return OK;
}
int hipLaunchKernel(const void *f, dim3 g, dim3 b, void **args, size_t lds, stream_t s) {
	(void) args, (void) lds, (void) s;
	const char *name = "?";
	for(int k = 0; k < n_kernels; k++)
		if(kernels[k].f == f) name = kernels[k].name;
	note("launch %s %u %u %u %u %u %u\n", name, g.x, g.y, g.z, b.x, b.y, b.z);
	const uint64_t lim = (uint64_t) 1 << 32;
	if((uint64_t) g.x * b.x >= lim || (uint64_t) g.y * b.y >= lim || (uint64_t) g.z * b.z >= lim || !g.x || !g.y || !g.z ||
	   (uint64_t) b.x * b.y * b.z > 1024 || !b.x || !b.y || !b.z)
		return failed(BAD_CONFIGURATION);
	return OK;
}
int hipLaunchCooperativeKernel(const void *f, dim3 g, dim3 b, void **args, unsigned lds, stream_t s) {
	return hipLaunchKernel(f, g, b, args, lds, s);
}

/* the rest answers as a device that is always done */
int hipDeviceGetAttribute(int *v, int what, int dev) {
	(void) what, (void) dev;
	*v = 256;
	return OK;
}
int hipOccupancyMaxActiveBlocksPerMultiprocessor(int *n, const void *f, int block, size_t lds) {
	(void) f, (void) block, (void) lds;
	*n = 2;
	return OK;
}
int hipGetDeviceCount(int *n) {
	*n = 1;
	return OK;
}
int hipGetSymbolAddress(void **p, const void *sym) { return *p = (void *) sym, OK; }
int hipSetDevice(int d) { return (void) d, OK; }
int hipDeviceSynchronize(void) { return OK; }
int hipGetLastError(void) {
	const int e = last_error;
	last_error = OK;
	return e;
}
const char *hipGetErrorString(int e) {
	return e == OK ? "no error" : (e == OUT_OF_MEMORY ? "out of memory" : "invalid configuration argument");
}
int hipStreamCreateWithFlags(stream_t *s, unsigned f) { return (void) f, *s = &module, OK; }
int hipStreamDestroy(stream_t s) { return (void) s, OK; }
int hipStreamQuery(stream_t s) { return (void) s, OK; }
int hipStreamSynchronize(stream_t s) { return (void) s, OK; }
int hipStreamWaitEvent(stream_t s, void *e, unsigned f) { return (void) s, (void) e, (void) f, OK; }
int hipEventCreate(void **e) { return *e = &module, OK; }
int hipEventCreateWithFlags(void **e, unsigned f) { return (void) f, hipEventCreate(e); }
int hipEventDestroy(void *e) { return (void) e, OK; }
int hipEventRecord(void *e, stream_t s) { return (void) e, (void) s, OK; }
int hipEventSynchronize(void *e) { return (void) e, OK; }
int hipEventElapsedTime(float *ms, void *a, void *b) { return (void) a, (void) b, *ms = 0.f, OK; }

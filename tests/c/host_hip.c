/*
 * A HIP runtime in host memory for tests of the host code without a GPU:
 * device memory is malloc'd, copies are checked against the live
 * allocations and end the program when they leave them, launches do
 * nothing, and the n-th allocation from now can be made to fail.  Loaded
 * ahead of the library with global symbols, so that the library binds to
 * it.
 */
#define __HIP_PLATFORM_AMD__ 1
#include <hip/hip_runtime_api.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#define MAX_LIVE 4096
static struct {
	char *p;
	size_t n;
} live[MAX_LIVE];
static long n_live, n_allocs, fail_in, n_launches;
static int fail_pinned;
static hipError_t last;	/* kept until it is asked for */

/* the n-th device allocation from now fails (0: none does) */
void host_hip_fail(long n) { fail_in = n; }
/* every pinned allocation fails while on */
void host_hip_fail_pinned(int on) { fail_pinned = on; }
long host_hip_live(void) { return n_live; }
long host_hip_allocs(void) { return n_allocs; }
long host_hip_launches(void) { return n_launches; }

static void check(const char *what, const void *p, size_t n)
{
	for(int i = 0; i < MAX_LIVE; i++)
		if(live[i].p && (const char *) p >= live[i].p && (const char *) p + n <= live[i].p + live[i].n)
			return;
	fprintf(stderr, "%s: %zu bytes at %p are not inside a live device allocation\n", what, n, p);
	fflush(stderr);
	_Exit(70);
}

hipError_t hipMalloc(void **p, size_t n)
{
	n_allocs++;
	if(fail_in && !--fail_in) {
		*p = NULL;
		return last = hipErrorOutOfMemory;
	}
	for(int i = 0; i < MAX_LIVE; i++)
		if(!live[i].p) {
			live[i].p = calloc(1, n ? n : 1);
			live[i].n = n;
			n_live++;
			*p = live[i].p;
			return live[i].p ? hipSuccess : hipErrorOutOfMemory;
		}
	return hipErrorOutOfMemory;
}

hipError_t hipFree(void *p)
{
	for(int i = 0; p && i < MAX_LIVE; i++)
		if(live[i].p == (char *) p) {
			free(live[i].p);
			live[i].p = NULL;
			n_live--;
			return hipSuccess;
		}
	if(p)
		check("hipFree", NULL, 1);
	return hipSuccess;
}

hipError_t hipMemcpy(void *dst, const void *src, size_t n, hipMemcpyKind kind)
{
	if(kind != hipMemcpyDeviceToHost)
		check("copy to the device", dst, n);
	if(kind != hipMemcpyHostToDevice)
		check("copy from the device", src, n);
	memmove(dst, src, n);
	return hipSuccess;
}

hipError_t hipMemcpyAsync(void *dst, const void *src, size_t n, hipMemcpyKind kind, hipStream_t st)
{
	(void) st;
	return hipMemcpy(dst, src, n, kind);
}

hipError_t hipMemset(void *dst, int v, size_t n)
{
	check("fill", dst, n);
	memset(dst, v, n);
	return hipSuccess;
}

/* the launch syntax pushes its configuration, the kernel's stub pops it */
static struct {
	dim3 grid, block;
	size_t lds;
	hipStream_t st;
} config;

hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t lds, hipStream_t st)
{
	config.grid = grid;
	config.block = block;
	config.lds = lds;
	config.st = st;
	return hipSuccess;
}

hipError_t __hipPopCallConfiguration(dim3 *grid, dim3 *block, size_t *lds, hipStream_t *st)
{
	*grid = config.grid;
	*block = config.block;
	*lds = config.lds;
	*st = config.st;
	return hipSuccess;
}

hipError_t hipLaunchKernel(const void *f, dim3 grid, dim3 block, void **args, size_t lds, hipStream_t st)
{
	(void) f, (void) args, (void) st;
	n_launches++;
	if(grid.x && grid.y && grid.z && block.x * block.y * block.z <= 1024 && lds <= 160 * 1024)
		return hipSuccess;
	return last = hipErrorInvalidConfiguration;
}

hipError_t hipGetDeviceProperties(hipDeviceProp_t *prop, int dev)
{
	(void) dev;
	memset(prop, 0, sizeof(*prop));
	strcpy(prop->gcnArchName, "host");
	prop->sharedMemPerBlock = 160 * 1024;
	prop->multiProcessorCount = 256;
	return hipSuccess;
}

hipError_t hipGetDeviceCount(int *n) { *n = 1; return hipSuccess; }
hipError_t hipGetDevice(int *dev) { *dev = 0; return hipSuccess; }
hipError_t hipGetLastError(void) { const hipError_t e = last; last = hipSuccess; return e; }
const char *hipGetErrorString(hipError_t e) { return e == hipSuccess ? "no error" : "host error"; }
hipError_t hipDeviceSynchronize(void) { return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t *st, unsigned flags) { (void) flags; *st = (hipStream_t) malloc(1); return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t st) { (void) st; return hipSuccess; }
hipError_t hipHostMalloc(void **p, size_t n, unsigned flags)
{
	(void) flags;
	*p = fail_pinned ? NULL : calloc(1, n);
	return *p ? hipSuccess : (last = hipErrorOutOfMemory);
}

hipError_t hipHostFree(void *p) { free(p); return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned flags) { (void) flags; *e = (hipEvent_t) malloc(1); return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t e) { free((void *) e); return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t st) { (void) e, (void) st; return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t e) { (void) e; return hipSuccess; }

/* A stand-in for the HIP runtime on a machine without a GPU: launches are noted, not run, and refused where HIP refuses them
 * (2^32 threads or more in a dimension, over 160 KB of LDS).  Memory is address space without access.  A test that loads this
 * library first, with its symbols global, sees what the library's entry points would launch. */
#include <stddef.h>
#include <stdint.h>
#include <stdio.h>
#include <sys/mman.h>

enum { ERROR_MEMORY = 2, ERROR_CONFIGURATION = 9, MAX_KERNELS = 4096, MAX_LAUNCHES = 4096 };
typedef struct { uint32_t x, y, z; } dim3_t;

static struct { const void* host; const char* name; } kernels[MAX_KERNELS];
static struct { const char* name; uint64_t dims[5]; } launches[MAX_LAUNCHES];  /* grid x, y, z, threads, bytes of LDS */
static int kernel_count, launch_count, last_error;
static struct { dim3_t grid, block; size_t lds; void* stream; } pushed;
static void* module;

void** __hipRegisterFatBinary(const void* data) { (void)data; return &module; }
void __hipUnregisterFatBinary(void** m) { (void)m; }
void __hipRegisterVar(void) {}
void __hipRegisterFunction(void** m, const void* host, char* device, const char* name)
{
	(void)m; (void)device;
	if (kernel_count == MAX_KERNELS) return;
	kernels[kernel_count].host = host;
	kernels[kernel_count++].name = name;
}
int __hipPushCallConfiguration(dim3_t grid, dim3_t block, size_t lds, void* stream)
{
	pushed.grid = grid; pushed.block = block; pushed.lds = lds; pushed.stream = stream;
	return 0;
}
int __hipPopCallConfiguration(dim3_t* grid, dim3_t* block, size_t* lds, void** stream)
{
	*grid = pushed.grid; *block = pushed.block; *lds = pushed.lds; *stream = pushed.stream;
	return 0;
}

int hipGetDevice(int* d) { *d = 0; return 0; }
int hipSetDevice(int d) { (void)d; return 0; }
int hipGetDeviceCount(int* d) { *d = 1; return 0; }
int hipMalloc(void** p, size_t bytes)
{
	*p = mmap(NULL, bytes, PROT_NONE, MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
	return *p == MAP_FAILED ? ERROR_MEMORY : 0;
}
int hipFree(void* p) { (void)p; return 0; }
int hipMemset(void* p, int v, size_t bytes) { (void)p; (void)v; (void)bytes; return 0; }
int hipStreamCreate(void** s) { *s = &module; return 0; }
int hipStreamSynchronize(void* s) { (void)s; return 0; }
int hipGetSymbolAddress(void** p, const void* symbol) { (void)symbol; *p = &module; return 0; }
int hipGetLastError(void)
{
	const int e = last_error;
	last_error = 0;
	return e;
}
const char* hipGetErrorString(int e) { return e == 0 ? "no error" : e == ERROR_CONFIGURATION ? "invalid configuration argument" : "error"; }

int hipLaunchKernel(const void* host, dim3_t grid, dim3_t block, void** args, size_t lds, void* stream)
{
	(void)args; (void)stream;
	const char* name = "?";
	for (int k = 0; k < kernel_count; k++)
		if (kernels[k].host == host) name = kernels[k].name;
	if (launch_count < MAX_LAUNCHES) {
		const uint64_t dims[5] = { grid.x, grid.y, grid.z, (uint64_t)block.x * block.y * block.z, lds };
		launches[launch_count].name = name;
		for (int i = 0; i < 5; i++) launches[launch_count].dims[i] = dims[i];
		launch_count++;
	}
	if (grid.x == 0 || grid.y == 0 || grid.z == 0 || (uint64_t)grid.x * block.x >= 1ull << 32 || (uint64_t)grid.y * block.y >= 1ull << 32 ||
	    (uint64_t)grid.z * block.z >= 1ull << 32 || lds > 160 * 1024) last_error = ERROR_CONFIGURATION;
	return last_error;
}

int stub_launches(void) { return launch_count; }
void stub_forget(void) { launch_count = 0; }
const char* stub_name(int i) { return launches[i].name; }
void stub_dims(int i, uint64_t* out)
{
	for (int k = 0; k < 5; k++) out[k] = launches[i].dims[k];
}

/* A stand-in for the HIP runtime calls of a shape set's batches, for tests of the host code without a
 * GPU: device memory is host memory (zeroed), allocations above stub_limit bytes fail, and launches are
 * counted instead of being run, those of the fill kernel at address zero by themselves. */
#include <stdlib.h>
#include <string.h>

size_t stub_limit = (size_t)-1;
int stub_null_fills = 0;
int stub_launches = 0;
static const void* fill_kernel = NULL;
typedef struct { unsigned x, y, z; } dim3_;
static dim3_ cfg_grid, cfg_block;
static int last_error = 0;

void __hipRegisterFunction(void* m, const void* host, char* dev, const char* name, unsigned t, void* a, void* b, void* c,
                           void* d, int* e) {
  if (strstr(name, "k_fill_u32")) fill_kernel = host;
}
int hipMalloc(void** p, size_t n) {
  *p = NULL;
  if (n > stub_limit || !(*p = calloc(1, n))) return last_error = 2;
  return 0;
}
int hipFree(void* p) { free(p); return 0; }
int hipMemcpyAsync(void* d, const void* s, size_t n, int kind, void* stream) { memmove(d, s, n); return 0; }
int hipMemcpy(void* d, const void* s, size_t n, int kind) { memmove(d, s, n); return 0; }
int hipStreamSynchronize(void* s) { return 0; }
int hipGetLastError(void) { int e = last_error; last_error = 0; return e; }
int hipEventCreate(void** e) { *e = NULL; return 0; }
int hipEventDestroy(void* e) { return 0; }
const char* hipGetErrorString(int e) { return e == 2 ? "out of memory" : "error"; }
int __hipPushCallConfiguration(dim3_ g, dim3_ b, size_t sh, void* s) { cfg_grid = g; cfg_block = b; return 0; }
int __hipPopCallConfiguration(dim3_* g, dim3_* b, size_t* sh, void** s) {
  *g = cfg_grid; *b = cfg_block; *sh = 0; *s = NULL;
  return 0;
}
int hipLaunchKernel(const void* f, dim3_ g, dim3_ b, void** args, size_t sh, void* s) {
  ++stub_launches;
  if (f == fill_kernel && *(void**)args[0] == NULL) ++stub_null_fills;
  return 0;
}

/* A HIP runtime that runs no kernel: the calls libyahmc.so makes, with device
 * memory that is only counted and kernel launches that are only recorded.
 * Loaded into a process before libyahmc.so (RTLD_GLOBAL), it lets host logic -
 * which kernel a call launches, with which grid and arguments, and how much
 * memory it takes - be tested without a GPU.  Copies to the host yield zeros. */
#include <stddef.h>
#include <stdint.h>
#include <stdlib.h>
#include <string.h>

typedef struct { uint32_t x, y, z; } dim3_t;
typedef int err_t;
enum { MAX_KERNELS = 4096, MAX_LAUNCHES = 1 << 16, MAX_ALLOCS = 1 << 14 };

static struct { const void* host; const char* name; } kernels[MAX_KERNELS];
static int nkernels;
static struct { const char* name; dim3_t grid, block; int arg; } launches[MAX_LAUNCHES];
static int nlaunches;
static struct { uintptr_t addr; size_t size; } allocs[MAX_ALLOCS];
static int nallocs;
static size_t in_use, peak;
static uintptr_t next_addr = (uintptr_t)1 << 44;
static const char* watch_name = "";
static int watch_arg = -1;

/* what the tests read */
void stub_reset(void) { nlaunches = 0; peak = in_use; }
int stub_launches(void) { return nlaunches; }
const char* stub_name(int i) { return launches[i].name; }
void stub_grid(int i, uint32_t* out) { memcpy(out, &launches[i].grid, sizeof(dim3_t)); }
int stub_arg(int i) { return launches[i].arg; }
size_t stub_in_use(void) { return in_use; }
size_t stub_peak(void) { return peak; }
/* record the int argument `arg` of the kernels whose name contains `name` */
void stub_watch(const char* name, int arg) { watch_name = strdup(name); watch_arg = arg; }

void** __hipRegisterFatBinary(const void* d) { static void* h; (void)d; return &h; }
void __hipUnregisterFatBinary(void** m) { (void)m; }
void __hipRegisterFunction(void** m, const void* host, char* dev, const char* name, unsigned lim, void* tid, void* bid,
                           void* bd, void* gd, int* ws) {
  (void)m; (void)dev; (void)lim; (void)tid; (void)bid; (void)bd; (void)gd; (void)ws;
  if (nkernels < MAX_KERNELS) { kernels[nkernels].host = host; kernels[nkernels++].name = name; }
}
void __hipRegisterVar(void** m, void* var, char* hv, char* dv, int ext, size_t size, int con, int glob) {
  (void)m; (void)var; (void)hv; (void)dv; (void)ext; (void)size; (void)con; (void)glob;
}

static dim3_t cfg_grid, cfg_block;
static size_t cfg_lds;
static void* cfg_stream;
err_t __hipPushCallConfiguration(dim3_t g, dim3_t b, size_t lds, void* s) {
  cfg_grid = g; cfg_block = b; cfg_lds = lds; cfg_stream = s;
  return 0;
}
err_t __hipPopCallConfiguration(dim3_t* g, dim3_t* b, size_t* lds, void** s) {
  *g = cfg_grid; *b = cfg_block; *lds = cfg_lds; *s = cfg_stream;
  return 0;
}
err_t hipLaunchKernel(const void* f, dim3_t g, dim3_t b, void** args, size_t lds, void* s) {
  (void)lds; (void)s;
  if (nlaunches == MAX_LAUNCHES) abort();
  const char* name = "?";
  for (int i = 0; i < nkernels; i++)
    if (kernels[i].host == f) name = kernels[i].name;
  launches[nlaunches].name = name;
  launches[nlaunches].grid = g;
  launches[nlaunches].block = b;
  launches[nlaunches].arg = watch_arg >= 0 && strstr(name, watch_name) ? *(int*)args[watch_arg] : 0;
  nlaunches++;
  return 0;
}

err_t hipMalloc(void** p, size_t n) {
  if (nallocs == MAX_ALLOCS) abort();
  *p = (void*)next_addr;
  allocs[nallocs].addr = next_addr;
  allocs[nallocs++].size = n;
  next_addr += (n + 4095) / 4096 * 4096 + 4096;
  in_use += n;
  if (in_use > peak) peak = in_use;
  return 0;
}
err_t hipFree(void* p) {
  for (int i = 0; i < nallocs; i++)
    if (allocs[i].addr == (uintptr_t)p) {
      in_use -= allocs[i].size;
      allocs[i] = allocs[--nallocs];
      return 0;
    }
  return p ? 1 : 0;
}
err_t hipHostMalloc(void** p, size_t n, unsigned f) { (void)f; *p = calloc(1, n); return 0; }
err_t hipHostFree(void* p) { free(p); return 0; }
err_t hipMemcpyAsync(void* d, const void* s, size_t n, int kind, void* st) {
  (void)s; (void)st;
  if (kind == 2) memset(d, 0, n); /* device to host */
  return 0;
}
err_t hipMemcpyToSymbol(const void* d, const void* s, size_t n, size_t o, int kind) {
  (void)d; (void)s; (void)n; (void)o; (void)kind;
  return 0;
}
err_t hipMemset(void* p, int v, size_t n) { (void)p; (void)v; (void)n; return 0; }
err_t hipMemsetAsync(void* p, int v, size_t n, void* st) { (void)p; (void)v; (void)n; (void)st; return 0; }
err_t hipGetSymbolAddress(void** p, const void* s) { (void)s; *p = (void*)((uintptr_t)1 << 43); return 0; }
err_t hipFuncSetAttribute(const void* f, int a, int v) { (void)f; (void)a; (void)v; return 0; }
err_t hipGetDeviceCount(int* n) { *n = 1; return 0; }
err_t hipGetDevice(int* d) { *d = 0; return 0; }
err_t hipSetDevice(int d) { (void)d; return 0; }
err_t hipDeviceSynchronize(void) { return 0; }
err_t hipGetLastError(void) { return 0; }
const char* hipGetErrorString(err_t e) { return e ? "error" : "no error"; }
err_t hipStreamCreateWithFlags(void** s, unsigned f) { (void)f; *s = (void*)1; return 0; }
err_t hipStreamDestroy(void* s) { (void)s; return 0; }
err_t hipStreamSynchronize(void* s) { (void)s; return 0; }
err_t hipStreamBeginCapture(void* s, int m) { (void)s; (void)m; return 1; }
err_t hipStreamEndCapture(void* s, void** g) { (void)s; *g = NULL; return 1; }
err_t hipGraphInstantiate(void** e, void* g, void* n, char* b, size_t sz) {
  (void)e; (void)g; (void)n; (void)b; (void)sz;
  return 1;
}
err_t hipGraphLaunch(void* e, void* s) { (void)e; (void)s; return 1; }
err_t hipGraphDestroy(void* g) { (void)g; return 0; }
err_t hipGraphExecDestroy(void* e) { (void)e; return 0; }
err_t hipEventCreate(void** e) { *e = (void*)1; return 0; }
err_t hipEventCreateWithFlags(void** e, unsigned f) { (void)f; *e = (void*)1; return 0; }
err_t hipEventDestroy(void* e) { (void)e; return 0; }
err_t hipEventRecord(void* e, void* s) { (void)e; (void)s; return 0; }
err_t hipEventSynchronize(void* e) { (void)e; return 0; }
err_t hipEventElapsedTime(float* ms, void* a, void* b) { (void)a; (void)b; *ms = 1.0f; return 0; }

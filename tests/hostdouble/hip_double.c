/* A stand-in for the HIP runtime's host interface, for tests of the library's
 * host code on a machine without a GPU: device memory is reserved address
 * space within a budget, allocations can be made to fail, kernel launches are
 * reported and not run. */
#define _GNU_SOURCE
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>
#include <sys/mman.h>

typedef struct {
  uint32_t x, y, z;
} dim3;
typedef void (*launch_cb)(const char* name, dim3 grid, dim3 block, size_t shmem, void** args);

#define MAXFN 4096
#define MAXMEM 65536
static struct {
  const void* fn;
  char name[512];
} fns[MAXFN];
static int nfns;
static struct {
  void* p;
  size_t n;
} mem[MAXMEM];
static int nmem;
static size_t held, budget = (size_t)288 << 30;
static long countdown = -1, nmalloc;
static launch_cb callback;

void double_on_launch(launch_cb cb) { callback = cb; }
void double_fail_after(long n) { countdown = n; } /* the n-th allocation from now fails (0: the next); -1: none */
void double_budget(size_t bytes) { budget = bytes; }
size_t double_held(void) { return held; }
long double_mallocs(void) { return nmalloc; }

int hipMalloc(void** p, size_t n) {
  *p = NULL;
  ++nmalloc;
  if (countdown >= 0 && countdown-- == 0) return 2;
  if (held + n > budget || nmem >= MAXMEM) return 2;
  void* q = mmap(NULL, n ? n : 1, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
  if (q == MAP_FAILED) return 2;
  mem[nmem].p = q;
  mem[nmem++].n = n;
  held += n;
  *p = q;
  return 0;
}

int hipFree(void* p) {
  for (int i = 0; i < nmem; ++i)
    if (mem[i].p == p) {
      munmap(p, mem[i].n ? mem[i].n : 1);
      held -= mem[i].n;
      mem[i] = mem[--nmem];
      return 0;
    }
  return p ? 1 : 0;
}

size_t double_size(const void* p) {
  for (int i = 0; i < nmem; ++i)
    if (mem[i].p == p) return mem[i].n;
  return 0;
}

/* copies of tables are made, whole maps are not */
static int copy(void* d, const void* s, size_t n) {
  if (n <= ((size_t)64 << 20)) memcpy(d, s, n);
  return 0;
}
int hipMemcpy(void* d, const void* s, size_t n, int kind) { return copy(d, s, n); }
int hipMemcpyAsync(void* d, const void* s, size_t n, int kind, void* st) { return copy(d, s, n); }
int hipMemcpy2DAsync(void* d, size_t dp, const void* s, size_t sp, size_t w, size_t h, int kind, void* st) { return 0; }
int hipMemset(void* d, int v, size_t n) {
  if (n <= ((size_t)64 << 20)) memset(d, v, n);
  return 0;
}
int hipMemsetAsync(void* d, int v, size_t n, void* st) { return hipMemset(d, v, n); }
int hipMemcpyToSymbol(void* sym, const void* s, size_t n, size_t off, int kind) { return copy((char*)sym + off, s, n); }
int hipMemcpyFromSymbol(void* d, const void* sym, size_t n, size_t off, int kind) {
  return copy(d, (const char*)sym + off, n);
}
int hipGetSymbolAddress(void** p, const void* sym) {
  *p = (void*)sym;
  return 0;
}
int hipMemGetInfo(size_t* f, size_t* t) {
  *f = budget - held;
  *t = budget;
  return 0;
}

int hipGetDeviceCount(int* n) {
  *n = 1;
  return 0;
}
int hipSetDevice(int d) { return 0; }
int hipDeviceSynchronize(void) { return 0; }
int hipGetLastError(void) { return 0; }
const char* hipGetErrorString(int e) { return e == 2 ? "out of memory" : "error"; }
int hipFuncSetAttribute(const void* f, int attr, int v) { return 0; }
static int event;
int hipEventCreate(void** e) {
  *e = &event;
  return 0;
}
int hipEventCreateWithFlags(void** e, unsigned f) { return hipEventCreate(e); }
int hipEventDestroy(void* e) { return 0; }
int hipEventRecord(void* e, void* st) { return 0; }
int hipEventSynchronize(void* e) { return 0; }
int hipEventElapsedTime(float* ms, void* a, void* b) {
  *ms = 1.0f;
  return 0;
}
int hipStreamCreateWithFlags(void** s, unsigned f) {
  *s = &event;
  return 0;
}
int hipStreamDestroy(void* s) { return 0; }
int hipStreamSynchronize(void* s) { return 0; }
int hipStreamWaitEvent(void* s, void* e, unsigned f) { return 0; }

/* the compiler's registration of kernels and the <<<>>> call sequence */
static void* module;
void** __hipRegisterFatBinary(const void* data) { return &module; }
void __hipUnregisterFatBinary(void** m) {}
void __hipRegisterVar(void** m, void* var, char* host, char* dev, int ext, size_t size, int constant, int global) {}
void __hipRegisterFunction(void** m, const void* fn, char* dev, const char* name, unsigned tl, void* tid, void* bid,
                           void* bd, void* gd, int* ws) {
  if (nfns >= MAXFN) return;
  fns[nfns].fn = fn;
  snprintf(fns[nfns++].name, sizeof(fns[0].name), "%s", name);
}
static dim3 cgrid, cblock;
static size_t cshmem;
static void* cstream;
int __hipPushCallConfiguration(dim3 g, dim3 b, size_t sh, void* st) {
  cgrid = g;
  cblock = b;
  cshmem = sh;
  cstream = st;
  return 0;
}
int __hipPopCallConfiguration(dim3* g, dim3* b, size_t* sh, void** st) {
  *g = cgrid;
  *b = cblock;
  *sh = cshmem;
  *st = cstream;
  return 0;
}
int hipLaunchKernel(const void* fn, dim3 g, dim3 b, void** args, size_t sh, void* st) {
  const char* name = "?";
  for (int i = 0; i < nfns; ++i)
    if (fns[i].fn == fn) name = fns[i].name;
  if (callback) callback(name, g, b, sh, args);
  return 0;
}

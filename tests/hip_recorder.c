// Stand-ins for the HIP runtime calls of libwanferenz_amd.so that record instead of running, so
// that the host side (which kernel, what grid and LDS, on which device) can be checked without a
// GPU.  Loaded with RTLD_GLOBAL ahead of the library (tests/launch_recorder.py).
#include <pthread.h>
#include <stddef.h>
#include <stdio.h>

typedef struct {
  unsigned x, y, z;
} dim3_t;

enum { kMaxKernels = 4096, kMaxEvents = 1 << 16 };
enum { kEvGrant = 0, kEvLaunch = 1 };

typedef struct {
  int kind, device, kernel;
  unsigned long bytes;  // a grant's LDS, or a launch's dynamic LDS
  unsigned grid, block;
} event_t;

static struct {
  const void* host;
  const char* name;
} kernels[kMaxKernels];
static int n_kernels;
static event_t events[kMaxEvents];
static int n_events;
static pthread_mutex_t mu = PTHREAD_MUTEX_INITIALIZER;
static __thread int device;
static __thread struct {
  dim3_t grid, block;
  size_t lds;
  void* stream;
} conf;

static int kernel_of(const void* host) {
  for (int i = 0; i < n_kernels; ++i)
    if (kernels[i].host == host) return i;
  return -1;
}

static void add(int kind, const void* host, unsigned long bytes, unsigned grid, unsigned block) {
  pthread_mutex_lock(&mu);
  if (n_events < kMaxEvents) {
    const event_t e = {kind, device, kernel_of(host), bytes, grid, block};
    events[n_events++] = e;
  }
  pthread_mutex_unlock(&mu);
}

// ------------------------------------------------------ the test's side ----
void rec_set_device(int d) { device = d; }
int rec_kernels(void) { return n_kernels; }
const char* rec_kernel_name(int i) { return kernels[i].name; }
int rec_events(void) { return n_events; }
void rec_event(int i, long* out) {
  const event_t* e = &events[i];
  out[0] = e->kind, out[1] = e->device, out[2] = e->kernel;
  out[3] = (long)e->bytes, out[4] = e->grid, out[5] = e->block;
}

// ------------------------------------------------------- the HIP runtime ----
void** __hipRegisterFatBinary(const void* data) {
  static void* handle;
  return &handle;
}
void __hipUnregisterFatBinary(void** m) {}
void __hipRegisterVar(void** m, void* var, char* host, char* name, int ext, size_t size, int constant, int global) {}
void __hipRegisterFunction(void** m, const void* host, char* dev, const char* name, unsigned limit, void* tid,
                           void* bid, void* bd, void* gd, int* ws) {
  if (n_kernels < kMaxKernels) {
    kernels[n_kernels].host = host;
    kernels[n_kernels++].name = name;
  }
}
int __hipPushCallConfiguration(dim3_t grid, dim3_t block, size_t lds, void* stream) {
  conf.grid = grid, conf.block = block, conf.lds = lds, conf.stream = stream;
  return 0;
}
int __hipPopCallConfiguration(dim3_t* grid, dim3_t* block, size_t* lds, void** stream) {
  *grid = conf.grid, *block = conf.block, *lds = conf.lds, *stream = conf.stream;
  return 0;
}
int hipLaunchKernel(const void* f, dim3_t grid, dim3_t block, void** args, size_t lds, void* stream) {
  add(kEvLaunch, f, lds, grid.x * grid.y * grid.z, block.x * block.y * block.z);
  return 0;
}
int hipFuncSetAttribute(const void* f, int attr, int value) {
  add(kEvGrant, f, (unsigned long)value, 0, 0);
  return 0;
}
int hipGetDevice(int* d) {
  *d = device;
  return 0;
}
int hipDeviceGetAttribute(int* v, int attr, int d) {
  *v = 256;  // compute units of an MI355X: the only attribute the library asks for
  return 0;
}
int hipOccupancyMaxActiveBlocksPerMultiprocessor(int* n, const void* f, int block, size_t lds) {
  *n = 1;
  return 0;
}
int hipGetLastError(void) { return 0; }
int hipStreamIsCapturing(void* s, int* status) {
  *status = 0;
  return 0;
}
int hipMemcpyAsync(void* d, const void* s, size_t n, int kind, void* stream) { return 0; }
int hipGetSymbolAddress(void** p, const void* s) {
  *p = (void*)256;
  return 0;
}

/* A host program with a HIP runtime of its own (no device: memory is malloc'ed, a
 * kernel launch only checks its arguments) around libsomaxhip.so, for what the library
 * does on the host: which kernels have their dynamic LDS limit raised on which
 * device, and how much workspace a plan asks for.
 *
 *   host_driver LIB nx ny nl precision
 *
 * creates a plan on device 0 and one on device 1, runs an inversion, a right-hand side
 * and a step on device 1, and prints "workspace BYTES", "launches N", "refused N" (the
 * launches on a device that ask for more than the 64 KiB of dynamic LDS that a
 * kernel has unless hipFuncSetAttribute raised it there) and "allocations N" (C++
 * allocations of the three calls). */
#include <dlfcn.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include "somaxhip.h"

typedef struct {
  unsigned x, y, z;
} grid3;

static int device, launches, refused, allocations;
static struct {
  const void* f;
  int device, bytes;
} raised[1024];
static int nraised;
static struct {
  grid3 g, b;
  size_t lds;
  void* stream;
} call;

void** __hipRegisterFatBinary(const void* d) { return (void**)calloc(1, sizeof(void*)); }
void __hipUnregisterFatBinary(void** m) {}
void __hipRegisterFunction(void** m, const void* f, char* n, const char* d, unsigned l, void* a, void* b, void* c,
                           void* e, int* w) {}
void __hipRegisterVar(void** m, void* v, char* n, char* d, int e, size_t s, int c, int g) {}
int __hipPushCallConfiguration(grid3 g, grid3 b, size_t lds, void* stream) {
  call.g = g;
  call.b = b;
  call.lds = lds;
  call.stream = stream;
  return 0;
}
int __hipPopCallConfiguration(grid3* g, grid3* b, size_t* lds, void** stream) {
  *g = call.g;
  *b = call.b;
  *lds = call.lds;
  *stream = call.stream;
  return 0;
}
int hipLaunchKernel(const void* f, grid3 g, grid3 b, void** args, size_t lds, void* stream) {
  size_t limit = 65536;
  for (int i = 0; i < nraised; ++i)
    if (raised[i].f == f && raised[i].device == device && (size_t)raised[i].bytes > limit) limit = raised[i].bytes;
  ++launches;
  refused += lds > limit;
  return 0;
}
int hipFuncSetAttribute(const void* f, int attribute, int value) {
  if (nraised == 1024) return 1;
  raised[nraised].f = f;
  raised[nraised].device = device;
  raised[nraised++].bytes = value;
  return 0;
}
int hipGetDevice(int* d) {
  *d = device;
  return 0;
}
int hipDeviceGetAttribute(int* v, int a, int d) {
  *v = 256;
  return 0;
}
int hipMalloc(void** p, size_t n) { return (*p = malloc(n ? n : 1)) ? 0 : 2; }
int hipFree(void* p) {
  free(p);
  return 0;
}
int hipMemcpy(void* d, const void* s, size_t n, int k) {
  memcpy(d, s, n);
  return 0;
}
int hipMemcpyAsync(void* d, const void* s, size_t n, int k, void* st) { return hipMemcpy(d, s, n, k); }
int hipGetSymbolAddress(void** p, const void* s) {
  static char scratch[1];
  *p = scratch;
  return 0;
}
/* operator new and delete */
void* _Znwm(size_t n) {
  ++allocations;
  return malloc(n);
}
void _ZdlPv(void* p) { free(p); }
void _ZdlPvm(void* p, size_t n) { free(p); }
int hipGetLastError(void) { return 0; }
const char* hipGetErrorString(int e) { return "error"; }
int hipStreamSynchronize(void* s) { return 0; }
int hipDeviceSynchronize(void) { return 0; }

int main(int argc, char** argv) {
  if (argc != 6) return 2;
  void* lib = dlopen(argv[1], RTLD_NOW);
  if (!lib) {
    fprintf(stderr, "%s\n", dlerror());
    return 2;
  }
  const int nx = atoi(argv[2]), ny = atoi(argv[3]), nl = atoi(argv[4]), precision = atoi(argv[5]);
  int (*create)(const somaxhip_qg_desc*, somaxhip_qg_plan*) = dlsym(lib, "somaxhip_qg_plan_create");
  size_t (*bytes)(somaxhip_qg_plan) = dlsym(lib, "somaxhip_qg_workspace_bytes");
  const int f64 = precision == SOMAXHIP_PREC_FP64;
  int (*invert)(somaxhip_qg_plan, void*, void*, int, void*, void*) =
      dlsym(lib, f64 ? "somaxhip_qg_invert_f64" : "somaxhip_qg_invert");
  int (*rhs)(somaxhip_qg_plan, void*, void*, void*, const somaxhip_qg_params*, int, void*, void*) =
      dlsym(lib, f64 ? "somaxhip_qg_rhs_f64" : "somaxhip_qg_rhs");
  int (*step)(somaxhip_qg_plan, void*, void*, int, double, const somaxhip_qg_params*, void*, void*) =
      dlsym(lib, f64 ? "somaxhip_qg_step_f64" : "somaxhip_qg_step");
  double* rows = calloc(ny + 2, sizeof(double));
  double eye[64] = {0}, lambdas[8] = {0};
  for (int i = 0; i < nl; ++i) eye[i * nl + i] = 1.0;
  somaxhip_qg_desc d = {0};
  d.nx = nx;
  d.ny = ny;
  d.nl = nl;
  d.dx = d.dy = 1e4;
  d.cl2m = d.cm2l = eye;
  d.lambdas = d.wind_scale = lambdas;
  d.beta_y_row = d.wind_row = rows;
  d.precision = precision;
  somaxhip_qg_plan plan[2];
  for (device = 0; device < 2; ++device)
    if (create(&d, &plan[device])) return 3;
  device = 1;
  launches = refused = allocations = 0;
  const somaxhip_qg_params prm = {1.0, 0.0, 0.0, 0.0};
  static double q[1];  /* no launch reads memory */
  if (invert(plan[1], q, q + 1, 0, q, NULL) || rhs(plan[1], q, q + 1, NULL, &prm, 1, q, NULL) ||
      step(plan[1], q, NULL, 1, 1.0, &prm, q, NULL))
    return 4;
  printf("workspace %zu\nlaunches %d\nrefused %d\nallocations %d\n", bytes(plan[1]), launches, refused,
         allocations);
  return 0;
}

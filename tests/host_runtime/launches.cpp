// Runs the library's host side against a HIP runtime of its own: device memory
// is host memory, kernels are not run, and every launch is compared with what
// its function was granted on the current device.  This program exports the
// runtime's symbols (-rdynamic), so the library that it opens binds to them.
//
//   launches LIBRARY SCENARIO...
//
// A scenario prints what it finds wrong; the exit status is the count (at most
// 99).  Results of projections mean nothing here: no kernel has written them.
#include <dlfcn.h>
#include <hip/hip_runtime_api.h>

#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <string>
#include <utility>
#include <vector>

#include "fluid_projection.h"

namespace {

constexpr int kDevices = 2;
constexpr int kBlockLds = 160 * 1024;    // gfx950
constexpr size_t kUngranted = 64 * 1024; // dynamic LDS of a function whose limit was never raised

constexpr size_t kCounters = 24 * 1024;  // of an extrapolation, spread over cache lines

int g_wrong = 0;
thread_local int g_device = 0;
std::map<const void*, std::string> g_functions;
std::map<std::pair<int, const void*>, size_t> g_granted;
std::map<std::string, int> g_launches;
std::map<void*, size_t> g_blocks;  // live device allocations
struct Launch {
  dim3 grid, block;
  size_t lds;
  hipStream_t stream;
} g_config;

void wrong(const std::string& what) {
  ++g_wrong;
  std::printf("%s\n", what.c_str());
}

}  // namespace

extern "C" {

void** __hipRegisterFatBinary(const void*) {
  static void* handle;
  return &handle;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned, uint3*, uint3*, dim3*, dim3*,
                           int*) {
  g_functions[host] = name;
}
void __hipRegisterVar(void**, void* var, char*, char*, int, size_t, int, int) { (void)var; }
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t lds, hipStream_t s) {
  g_config = Launch{grid, block, lds, s};
  return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* grid, dim3* block, size_t* lds, hipStream_t* s) {
  *grid = g_config.grid;
  *block = g_config.block;
  *lds = g_config.lds;
  *s = g_config.stream;
  return hipSuccess;
}

hipError_t hipGetDeviceCount(int* n) {
  *n = kDevices;
  return hipSuccess;
}
hipError_t hipSetDevice(int d) {
  g_device = d;
  return hipSuccess;
}
hipError_t hipGetDevice(int* d) {
  *d = g_device;
  return hipSuccess;
}
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t a, int) {
  if (a != hipDeviceAttributeMaxSharedMemoryPerBlock) return hipErrorInvalidValue;
  *v = kBlockLds;
  return hipSuccess;
}
hipError_t hipFuncSetAttribute(const void* f, hipFuncAttribute a, int v) {
  if (a != hipFuncAttributeMaxDynamicSharedMemorySize || v < 0 || v > kBlockLds) return hipErrorInvalidValue;
  g_granted[{g_device, f}] = (size_t)v;
  return hipSuccess;
}
hipError_t hipLaunchKernel(const void* f, dim3, dim3, void**, size_t lds, hipStream_t) {
  const std::string& name = g_functions[f];
  ++g_launches[name];
  const auto it = g_granted.find({g_device, f});
  const size_t most = it == g_granted.end() ? kUngranted : it->second;
  if (lds > most)
    wrong("device " + std::to_string(g_device) + ": " + name + " launched with " + std::to_string(lds) +
          " bytes of dynamic LDS, granted " + std::to_string(most));
  return hipSuccess;
}

hipError_t hipMalloc(void** p, size_t n) {
  *p = std::calloc(n ? n : 1, 1);
  if (!*p) return hipErrorOutOfMemory;
  g_blocks[*p] = n;
  return hipSuccess;
}
hipError_t hipFree(void* p) {
  g_blocks.erase(p);
  std::free(p);
  return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
  *p = std::calloc(n ? n : 1, 1);
  return *p ? hipSuccess : hipErrorOutOfMemory;
}
hipError_t hipHostFree(void* p) {
  std::free(p);
  return hipSuccess;
}
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) {
  std::memmove(d, s, n);
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) {
  std::memmove(d, s, n);
  return hipSuccess;
}
hipError_t hipMemset(void* p, int v, size_t n) {
  std::memset(p, v, n);
  return hipSuccess;
}
hipError_t hipMemsetAsync(void* p, int v, size_t n, hipStream_t) {
  std::memset(p, v, n);
  return hipSuccess;
}
hipError_t hipGetSymbolAddress(void** p, const void*) {
  static unsigned char symbol[1 << 16];
  *p = symbol;
  return hipSuccess;
}

hipError_t hipGetLastError() { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "error"; }
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) {
  *s = nullptr;
  return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) {
  *e = nullptr;
  return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
  *e = nullptr;
  return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) {
  *ms = 0.0f;
  return hipSuccess;
}
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t* g) {
  *g = nullptr;
  return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t* e, hipGraph_t, hipGraphNode_t*, char*, size_t) {
  *e = nullptr;
  return hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipSuccess; }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }

}  // extern "C"

namespace {

void* g_lib;
template <class F>
F* entry(F*, const char* name) {
  F* f = reinterpret_cast<F*>(dlsym(g_lib, name));
  if (!f) {
    std::printf("no %s\n", name);
    std::exit(99);
  }
  return f;
}
#define FP(name) entry(static_cast<decltype(name)*>(nullptr), #name)

void must(int rc, const char* what) {
  if (rc == FP_OK) return;
  wrong(std::string(what) + ": " + std::to_string(rc) + " " + FP(fp_last_error)());
}

fp_ctx* context(int device, uint64_t budget = 0) {
  fp_ctx* c = nullptr;
  must(FP(fp_ctx_create)(device, budget, &c), "fp_ctx_create");
  return c;
}

struct Uniform {
  fp_grid* g = nullptr;
  std::vector<float> phi, u, v, w;
  Uniform(fp_ctx* c, int nx, int ny, int nz)
      : phi((size_t)nx * ny * nz, -1.0f), u((size_t)(nx + 1) * ny * nz), v((size_t)nx * (ny + 1) * nz),
        w((size_t)nx * ny * (nz + 1)) {
    fp_grid_desc d;
    std::memset(&d, 0, sizeof(d));
    d.layout = FP_LAYOUT_UNIFORM;
    d.nx = nx;
    d.ny = ny;
    d.nz = nz;
    d.h = 1.0 / nx;
    must(FP(fp_grid_create)(c, &d, &g), "fp_grid_create");
  }
  int project(int solver, int precision) {
    fp_options o;
    must(FP(fp_default_options)(&o), "fp_default_options");
    o.solver = solver;
    o.precision = precision;
    fp_inputs in;
    std::memset(&in, 0, sizeof(in));
    in.memory = FP_MEMORY_HOST;
    in.phi = phi.data();
    in.u = u.data();
    in.v = v.data();
    in.w = w.data();
    in.dt = 0.01;
    in.rho = 1000.0;
    fp_outputs out{nullptr, u.data(), v.data(), w.data()};
    fp_report r;
    return FP(fp_project)(g, &in, &out, &o, &r);
  }
  int vcycle(int precision) {
    fp_options o;
    must(FP(fp_default_options)(&o), "fp_default_options");
    o.precision = precision;
    std::vector<float> z(phi.size());
    return FP(fp_probe_vcycle)(g, phi.data(), &o, phi.data(), z.data());
  }
  void destroy() { must(FP(fp_grid_destroy)(g), "fp_grid_destroy"); }
};

int launches_of(const char* part) {
  int n = 0;
  for (const auto& kv : g_launches)
    if (kv.first.find(part) != std::string::npos) n += kv.second;
  return n;
}
void must_launch(const char* part) {
  if (launches_of(part) == 0) wrong(std::string("no launch of ") + part);
}

// A CM11a grid with a large tail, then one with a small tail, then the first again.
void cm11a_two_grids() {
  fp_ctx* c = context(0);
  Uniform big(c, 64, 64, 64), small(c, 16, 16, 16);
  must(big.project(FP_SOLVER_CM11A, FP_PRECISION_MIXED_FP16), "64^3");
  must(small.project(FP_SOLVER_CM11A, FP_PRECISION_MIXED_FP16), "16^3");
  must(big.project(FP_SOLVER_CM11A, FP_PRECISION_MIXED_FP16), "64^3 again");
  must_launch("k_cm_tail");
  big.destroy();
  small.destroy();
  must(FP(fp_ctx_destroy)(c), "fp_ctx_destroy");
}

// A finest level whose passes work in place holds no second pressure, and the
// bytes that a call is refused by are those it takes.
void cm11a_bytes() {
  const size_t n = 98, level = (n * n * n * 4 + 255) & ~(size_t)255;  // 96^3 with its halo
  fp_ctx* c = context(0);
  Uniform g(c, 96, 96, 96);
  const std::map<void*, size_t> before = g_blocks;
  must(g.project(FP_SOLVER_CM11A, FP_PRECISION_MIXED_FP16), "96^3");
  int arrays = 0;
  for (const auto& b : g_blocks) arrays += before.count(b.first) == 0 && b.second == level;
  // level sets, pressure, right-hand sides, p_min; b, p_min, its shift and the backup
  if (arrays != 10) wrong(std::to_string(arrays) + " arrays of the finest level, 10 expected");
  uint64_t used = 0;
  must(FP(fp_ctx_bytes_in_use)(c, &used), "fp_ctx_bytes_in_use");
  g.destroy();
  must(FP(fp_ctx_destroy)(c), "fp_ctx_destroy");
  for (int less = 0; less < 2; ++less) {
    fp_ctx* b = context(0, used - less);
    Uniform q(b, 96, 96, 96);
    const int rc = q.project(FP_SOLVER_CM11A, FP_PRECISION_MIXED_FP16);
    if (rc != (less ? FP_ERR_BUDGET : FP_OK)) wrong("budget of " + std::to_string(used - less) + ": " + std::to_string(rc));
    q.destroy();
    must(FP(fp_ctx_destroy)(b), "fp_ctx_destroy");
  }
}

// An extrapolation's state and host staging stay within 48 bytes a cell for two
// sides of values and distances, 5 for flags, classes and masks, 4 for the list,
// 4 a cell and 4 a face for host arrays, and the hierarchy: budgets that held
// those hold the call.
void extrapolate_bytes() {
  const int shapes[][3] = {{2, 40, 33}, {33, 2, 40}, {16, 16, 16}, {48, 31, 50}};
  for (const auto& d : shapes)
    for (int memory = 0; memory < 2; ++memory)
      for (int pass = 0; pass < 2; ++pass) {  // without a budget, then with that one
        const size_t nx = d[0], ny = d[1], nz = d[2], n = nx * ny * nz;
        auto up = [](size_t b) { return (b + 255) & ~(size_t)255; };
        const size_t faces = (nx + 1) * ny * nz + nx * (ny + 1) * nz + nx * ny * (nz + 1);
        size_t most = 13 * up(4 * n) + 5 * up(n) + up(4 * n) + up(4 * faces) + 256;
        for (size_t a = nx, b = ny, c = nz; a > 1 && b > 1 && c > 1;) {
          a = (a + 1) / 2;
          b = (b + 1) / 2;
          c = (c + 1) / 2;
          most += 6 * up(4 * a * b * c) + 2 * up(a * b * c);
        }
        static uint64_t grid;  // of the pass before
        fp_ctx* c = context(0, pass ? grid + most + kCounters : 0);
        Uniform g(c, d[0], d[1], d[2]);
        must(FP(fp_ctx_bytes_in_use)(c, &grid), "fp_ctx_bytes_in_use");
        fp_extrapolate_args a;
        std::memset(&a, 0, sizeof(a));
        a.memory = memory;
        a.phi = g.phi.data();
        a.u = a.u_out = g.u.data();
        a.v = a.v_out = g.v.data();
        a.w = a.w_out = g.w.data();
        const std::string what = std::to_string(nx) + "x" + std::to_string(ny) + "x" + std::to_string(nz) +
                                 (memory == FP_MEMORY_HOST ? " host" : " device");
        for (int call = 0; call < 2; ++call) must(FP(fp_extrapolate_velocity)(g.g, &a, nullptr), what.c_str());
        uint64_t used = 0;
        must(FP(fp_ctx_bytes_in_use)(c, &used), "fp_ctx_bytes_in_use");
        if (pass && used > grid + most + kCounters)
          wrong(what + ": " + std::to_string(used - grid) + " bytes, at most " + std::to_string(most));
        g.destroy();
        must(FP(fp_ctx_bytes_in_use)(c, &used), "fp_ctx_bytes_in_use");
        if (used != 0) wrong(what + ": " + std::to_string(used) + " bytes in use after the grid");
        must(FP(fp_ctx_destroy)(c), "fp_ctx_destroy");
      }
}

// The same FP32 grid, its V-cycle's bottom above 64 KB, on a context per device.
void two_devices() {
  fp_ctx* c[kDevices];
  for (int d = 0; d < kDevices; ++d) c[d] = context(d);
  for (int round = 0; round < 2; ++round)
    for (int d = 0; d < kDevices; ++d) {
      Uniform g(c[d], 30, 30, 30);
      must(g.vcycle(FP_PRECISION_FP32), "30^3");
      g.destroy();
    }
  must_launch("k_bottom_lds");
  for (fp_ctx* x : c) must(FP(fp_ctx_destroy)(x), "fp_ctx_destroy");
}

}  // namespace

int main(int argc, char** argv) {
  if (argc < 3 || !(g_lib = dlopen(argv[1], RTLD_NOW | RTLD_LOCAL))) {
    std::printf("usage: launches LIBRARY SCENARIO... (%s)\n", argc < 3 ? "arguments" : dlerror());
    return 99;
  }
  const std::map<std::string, void (*)()> scenarios{{"cm11a_bytes", cm11a_bytes},
                                                        {"cm11a_two_grids", cm11a_two_grids},
                                                        {"extrapolate_bytes", extrapolate_bytes},
                                                        {"two_devices", two_devices}};
  for (int k = 2; k < argc; ++k) scenarios.at(argv[k])();
  std::printf("%d wrong\n", g_wrong);
  std::fflush(stdout);
  _Exit(g_wrong < 99 ? g_wrong : 99);  // (the library's own static state may not end against this runtime)
}

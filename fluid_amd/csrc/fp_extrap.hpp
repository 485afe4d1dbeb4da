// fp_extrap.hpp -- velocity extrapolation of a uniform grid (host side).
//
// The step after the projection in the reference's uniform solver
// (lib/methods/uniform/webgpu-uniform-velocity-extrapolation{,.wgsl}.ts): every
// velocity component is extended from the faces next to liquid into the air,
// first by Jeong-Ross-Whitaker passes of the Godunov distance clipped to a
// two-cell band with the first-order upwind extension of CM11b Eq. 7, then
// into the far field by a restrict / prolong hierarchy of renormalised
// trilinear interpolation of known values.  FP32 in the reference's operation
// order without contraction: results equal oracle/fp_oracle_extrap.c bit for
// bit.
#pragma once

#include "fluid_projection.h"

#include <hip/hip_runtime.h>

#include <vector>

namespace fp {

// One ping-pong side of the narrow-band state (per cell, z fastest).
struct ExState {
  float* val[3];
  float* dist[3];
  uint8_t* flags;  // bits 0-2 known(c)
  uint8_t* stat;   // bits 2c, 2c+1: the face's part in the front (kQuiet ...)
};

// One level of the far-field hierarchy.
struct ExLevel {
  int d[3];
  long long n;
  float* val[3];
  uint8_t* known;
  float* up_val[3];
  uint8_t* up_known;
};

// Counters are spread over kExSpread cache lines by workgroup: thousands of
// atomics on one address take about 11 ns each.
constexpr int kExSpread = 16;
struct ExCounters {
  int active[20][kExSpread][16];                     // [0] the seed's, [k] before pass k + 1
  unsigned long long unknown[kExSpread][8];          // open faces left unknown
  unsigned long long band_known[kExSpread][8];       // faces known after the band
  int latest;                                        // side holding the band result
  int list_count;                                    // cells of the band list
};

// Their sums, for the host.
struct ExTotals {
  int active[20];
  unsigned long long unknown, band_known;
};

class Extrapolator {
 public:
  ~Extrapolator();
  // Bytes of create(), and those that the first host-memory run adds.
  static size_t estimate_bytes(int nx, int ny, int nz);
  static size_t host_bytes(int nx, int ny, int nz);
  bool host_ready() const { return in_ != nullptr; }
  int create(int nx, int ny, int nz, double h);
  // One extrapolation of a->phi / a->density and a->u, a->v, a->w into the
  // outputs; synchronous on s.
  // same_band: the field (phi / density) and open_top are those of this
  // object's previous run, whose classes, list mask and band list are reused
  // (a second extrapolation over the same surface, as a MacCormack step makes)
  int run(hipStream_t s, const fp_extrapolate_args* a, fp_extrapolate_report* rep, bool same_band = false);
  size_t bytes() const { return bytes_; }

 private:
  int alloc(void** p, size_t bytes);
  int stage_host();
  std::vector<void*> allocations_;
  std::vector<ExLevel> levels_;
  size_t bytes_ = 0;
  int d_[3] = {0, 0, 0};
  long long n_ = 0;
  float h_ = 0.0f;
  ExState st_[2];
  uint8_t* cls_ = nullptr;
  uint8_t* cand_[2] = {nullptr, nullptr};
  int band_count_ = -1;  // band list length of the previous run (-1: none)
  int* list_ = nullptr;
  float* in_ = nullptr;  // host-memory staging of u, v, w
  ExCounters* counters_ = nullptr;
  ExTotals* totals_ = nullptr;  // behind the counters
};

}  // namespace fp

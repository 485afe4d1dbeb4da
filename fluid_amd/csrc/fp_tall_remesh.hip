// fp_tall_remesh.hip -- re-laying a restricted tall-cell grid out around its
// current surface, on the device (fp_tall_remesh).
//
// Per column (one thread): the lowest and highest fine rows where the liquid
// (phi < 0) meets air along the column, with phi read from the current
// layout -- linear in the row inside the tall cell (the reconstruction of
// representedInitialPhiVolumeCells, lib/core/tall-cell-grid.ts:220-238), the
// band samples above it, air beyond the band -- and a surface cell being one
// whose wetness differs from the row below or above (isInitialSurfaceCell,
// tall-cell-grid.ts:263-279); the base from them (chooseTallCellBase,
// tall-cell-grid.ts:61-82; a dry column takes the highest base, :378-386);
// then Jacobi passes of base <= min(neighbour) + D until no base changes
// (limitNeighboringTallCellBases, :84-106, run to convergence as the layout
// builder's nx + nz passes do, :395).  The quantities move to the new layout
// as tallCells.txt:240-252 states: band cells copy the old value at their
// fine row (read linearly from the old tall cell where it covered the row),
// the new tall cell's bottom and top samples are the least-squares line
// through the old values of its rows; vertical face slots likewise (the tall
// cell's interior faces share the mean), horizontal ones refit their affine
// part over the rows both columns' tall cells share.  A column (pair) whose
// base(s) did not change is copied as is.  FP64 sums in row order without
// contraction, so a CPU restatement gives the same bits.
#pragma clang fp contract(off)

#include "fp_tall.hpp"

#include <algorithm>
#include <cstring>

namespace fp {

namespace {

struct RemeshGeo {
  int nx, ny, nz, B, P, S, D;
  double air;  // phi of the rows beyond the band (5 h, buildInitialPhi's limit)
};

// phi of fine row y of a column with base b inside its tall cell: linear
// between the bottom and top samples.  y / (b - 1) is made from the correctly
// rounded reciprocal `inv` of d = b - 1 with one residual step (Markstein):
// the correctly rounded quotient in three operations instead of a division
// per row (compared with the division for every y <= d <= 20000).
struct TallLine {
  double bottom, span, d, inv;
  __device__ __forceinline__ TallLine(float bot, float top, int b)
      : bottom((double)bot), span((double)top - (double)bot), d((double)max(b - 1, 1)), inv(1.0 / d) {}
  __device__ __forceinline__ double at(int y) const {
    const double q = (double)y * inv;
    const double t = __builtin_fma(__builtin_fma(-q, d, (double)y), inv, q);
    return bottom + span * t;
  }
};

// phi of fine row y of column c in a layout with base b
__device__ __forceinline__ double column_phi(const RemeshGeo& g, const float* __restrict__ col, const TallLine& line,
                                             int b, int y) {
  const int py = 2 + y - b;
  const double band = (double)col[(size_t)min(max(py, 0), g.P - 1) * g.nz];
  return y < b ? line.at(y) : py < g.P ? band : g.air;
}

// v at fine face f (between rows f-1 and f) of a column with base b: slot 0
// inside the tall cell, slot f - b + 1 from the tall top up
__device__ __forceinline__ double column_v(const RemeshGeo& g, const float* __restrict__ v, int x, int z, int b,
                                           int f) {
  if (f <= 0 || f >= g.ny) return 0.0;
  if (f < b) return v[((size_t)x * g.P + 0) * g.nz + z];
  const int s = f - b + 1;
  return s < g.P ? (double)v[((size_t)x * g.P + s) * g.nz + z] : 0.0;
}

// horizontal slots of one face: the affine part over rows 0..m-1 (mean, slope
// about (m-1)/2), then one slot per row from m
__device__ __forceinline__ double face_value(const RemeshGeo& g, const float* __restrict__ a, size_t base_index,
                                             size_t stride, int m, int y) {
  if (y < m) {
    const double mean = a[base_index];
    const double slope = a[base_index + stride];
    return mean + slope * ((double)y - 0.5 * (double)(m - 1));
  }
  const int s = 2 + y - m;
  return s < g.S ? (double)a[base_index + (size_t)s * stride] : 0.0;
}

// chooseTallCellBase (tall-cell-grid.ts:61-82) with Math.round
__device__ __forceinline__ int choose_base(int lowest, int highest, int fine_ny, int B, int liquid_halo,
                                           int air_halo) {
  const int maximum_base = max(0, fine_ny - B);
  const int lower = highest + 1 + air_halo - B;
  const int upper = lowest + 1 - liquid_halo;
  const int desired = lower <= upper ? (int)floor((double)(lower + upper) / 2.0 + 0.5) : lower;
  const int clamped = max(0, min(maximum_base, desired));
  return maximum_base >= 2 ? max(2, clamped) : 0;
}

// Surface rows and base of each column.  The rows above the tall cell are
// walked (band + 2 of them); inside it phi is monotone in the row (each
// rounded operation of TallLine::at is), so its wetness changes at most once
// and a bisection finds where.  Walking every fine row took 189 us for 512^2
// columns of 512 rows.
__global__ __launch_bounds__(256) void k_remesh_bases(RemeshGeo g, const float* __restrict__ phi,
                                                      const int* __restrict__ bases, int* __restrict__ raw,
                                                      int liquid_halo, int air_halo, unsigned long long* moved) {
  const int ncol = g.nx * g.nz;
  if (blockIdx.x == 0 && threadIdx.x == 0) *moved = 0;  // k_remesh_column counts
  for (int c = blockIdx.x * blockDim.x + threadIdx.x; c < ncol; c += gridDim.x * blockDim.x) {
    const int x = c / g.nz, z = c - (c / g.nz) * g.nz;
    const int b = bases[c];
    const float* __restrict__ col = phi + (size_t)x * g.P * g.nz + z;
    const float bot = col[0], top = col[g.nz];
    const TallLine line(bot, top, b);
    int lowest = g.ny, highest = -1;
    const bool bounded = isfinite(bot) && isfinite(top);  // else the line is not monotone: walk it
    int y0 = 0;                                           // first row of the walk
    if (bounded && b > 1) {
      const bool first = line.at(0) < 0.0, last = line.at(b - 1) < 0.0;
      if (first != last) {
        int lo = 0, hi = b - 1;  // wetness `first` at lo, `last` at hi
        while (hi - lo > 1) {
          const int mid = (lo + hi) >> 1;
          if ((line.at(mid) < 0.0) == first) lo = mid;
          else hi = mid;
        }
        lowest = lo;
        highest = hi;
      }
      y0 = b - 1;
    }
    // rows y0 .. y1: the tall cell's last row, the band, the first row beyond it
    const int y1 = min(g.ny - 1, b + g.B);
    bool here = column_phi(g, col, line, b, y0) < 0.0;
    bool below = here;  // row 0: itself; row b - 1: the bisection holds its change from below
#pragma unroll 8
    for (int y = y0; y <= y1; ++y) {
      const bool above = y + 1 < g.ny && column_phi(g, col, line, b, y + 1) < 0.0;
      if (here != below || here != above) {
        lowest = min(lowest, y);
        highest = max(highest, y);
      }
      below = here;
      here = above;
    }
    const int maximum_base = max(0, g.ny - g.B);
    const int lh = min(liquid_halo, g.B), ah = min(air_halo, g.B);
    const int surface = highest >= 0 ? choose_base(lowest, highest, g.ny, g.B, lh, ah)
                                     : (maximum_base <= 3 ? min(2, maximum_base) : maximum_base);
    raw[c] = maximum_base >= 2 ? max(2, surface) : 0;
  }
}

// The limit base <= min(4-neighbour) + D run to its fixed point is
// min over columns j of raw_j + D |i - j|_1, and that minimum separates: lines
// along z, then lines along x.  One wave per line takes it 64 columns at a
// time, a prefix minimum of raw_j - D j up and of raw_j + D j down with the
// carry of the chunks before: 11 us for both directions of 512^2 columns
// (Jacobi passes to convergence took 8.6 us each, sixteen of them there, with
// a host check every eight).
__global__ __launch_bounds__(256) void k_remesh_limit(int lines, int n, int line_stride, int stride, int D,
                                                      const int* __restrict__ in, int* out) {
  const int line = (int)((blockIdx.x * blockDim.x + threadIdx.x) >> 6), lane = (int)(threadIdx.x & 63);
  if (line >= lines) return;
  const size_t l0 = (size_t)line * line_stride;
  constexpr int kFar = 1 << 29;
  const int chunks = (n + 63) / 64;
  int carry = kFar;
  for (int k = 0; k < chunks; ++k) {  // prefix minima, upward
    const int j = 64 * k + lane;
    int v = min(j < n ? in[l0 + (size_t)j * stride] - D * j : kFar, carry);
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int p = __shfl_up(v, o, 64);
      v = lane >= o ? min(v, p) : v;
    }
    carry = __shfl(v, 63, 64);
    if (j < n) out[l0 + (size_t)j * stride] = v + D * j;
  }
  carry = kFar;
  for (int k = chunks - 1; k >= 0; --k) {  // downward, over what the same lane wrote
    const int j = 64 * k + lane;
    int v = min(j < n ? out[l0 + (size_t)j * stride] + D * j : kFar, carry);
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int p = __shfl_down(v, o, 64);
      v = lane + o < 64 ? min(v, p) : v;
    }
    carry = __shfl(v, 0, 64);
    if (j < n) out[l0 + (size_t)j * stride] = v - D * j;
  }
}

// Rows (or slots) that one lane of the transfer kernels moves; blockIdx.y 0
// makes a column's least-squares part, the others kRemeshRows rows each.
constexpr int kRemeshRows = 8;

// sum of t^2 over t = y - (n - 1)/2, y < n: every partial sum is a multiple of
// 1/4 below 2^53, so the running sum is exact and equals this
__device__ __forceinline__ double centred_squares(int n) {
  const double m = (double)n;
  return m * (m * m - 1.0) / 12.0;
}

// New samples and vertical slots of one column.  The sums over the tall cell's
// rows are a serial FP64 chain in row order (64 us alone for 290 rows of 512^2
// columns); the rows above it only move (47 us alone), so blockIdx.y gives
// them lanes of their own that stream while the sums run: 103 us together,
// 271 us when one lane did a whole column with a division per row.
__global__ __launch_bounds__(256) void k_remesh_column(RemeshGeo g, const int* __restrict__ ob,
                                                       const int* __restrict__ nb, const float* __restrict__ phi,
                                                       const float* __restrict__ v, float* __restrict__ phi_o,
                                                       float* __restrict__ v_o, unsigned long long* changed) {
  const int ncol = g.nx * g.nz;
  unsigned long long moved = 0;
  for (int c = blockIdx.x * blockDim.x + threadIdx.x; c < ncol; c += gridDim.x * blockDim.x) {
    const int x = c / g.nz, z = c - (c / g.nz) * g.nz;
    const int bo = ob[c], bn = nb[c];
    const size_t i0 = (size_t)x * g.P * g.nz + z;
    const float* __restrict__ pc = phi + i0;
    const float* __restrict__ vc = v + i0;
    float* __restrict__ po = phi_o + i0;
    float* __restrict__ vo = v_o + i0;
    const TallLine line(pc[0], pc[g.nz], bo);
    if (blockIdx.y == 0) {
      if (bo == bn) {
        po[0] = pc[0];
        po[g.nz] = pc[g.nz];
        vo[0] = vc[0];
        continue;
      }
      ++moved;
      // least-squares line through rows 0..bn-1, in t = y - (bn - 1)/2
      const double mid = 0.5 * (double)(bn - 1);
      double sf = 0.0, stf = 0.0, t = -mid;  // t + 1 is exact: a half-integer
      const int inside = min(bo, bn);
#pragma unroll 4
      for (int y = 0; y < inside; ++y) {
        const double f = line.at(y);
        sf += f;
        stf += t * f;
        t += 1.0;
      }
      for (int y = inside; y < bn; ++y) {
        const double f = column_phi(g, pc, line, bo, y);
        sf += f;
        stf += t * f;
        t += 1.0;
      }
      const double stt = centred_squares(bn);
      const double mean = sf / (double)bn, slope = stt > 0.0 ? stf / stt : 0.0;
      po[0] = (float)(mean - slope * mid);
      po[g.nz] = (float)(mean + slope * mid);
      // vertical faces: the tall cell's interior faces 1..bn-1 share their
      // mean; the old tall cell's part of the sum is a multiple of one FP32
      // value, exact in FP64 however it is added up
      double sv = inside > 1 ? 0.0 + (double)(inside - 1) * (double)vc[0] : 0.0;
      for (int f = max(inside, 1); f < bn; ++f) sv += column_v(g, v, x, z, bo, f);
      vo[0] = (float)(sv / (double)max(bn - 1, 1));
      continue;
    }
    const int r0 = 1 + ((int)blockIdx.y - 1) * kRemeshRows;
#pragma unroll
    for (int k = 0; k < kRemeshRows; ++k) {
      const int s = r0 + k;
      if (s >= g.P) break;
      const size_t o = (size_t)s * g.nz;
      if (bo == bn) {
        if (s >= 2) po[o] = pc[o];
        vo[o] = vc[o];
        continue;
      }
      if (s >= 2) {
        const int y = bn + s - 2;
        po[o] = y < g.ny ? (float)column_phi(g, pc, line, bo, y) : (float)g.air;
      }
      vo[o] = (float)column_v(g, v, x, z, bo, bn + s - 1);
    }
  }
  if (moved) atomicAdd(changed, moved);
}

// New horizontal slots of the faces between columns (axis 0: x faces, 1: z
// faces), split as k_remesh_column is: 55 us per axis for 512^2 columns (81.9
// MB read and written), 131 us before.
__global__ __launch_bounds__(256) void k_remesh_faces(RemeshGeo g, int axis, const int* __restrict__ ob,
                                                      const int* __restrict__ nb, const float* __restrict__ a,
                                                      float* __restrict__ a_o) {
  // u: (nx+1, S, nz); w: (nx, S, nz+1)
  const int fx = axis == 0 ? g.nx + 1 : g.nx, fz = axis == 0 ? g.nz : g.nz + 1;
  const int nf = fx * fz;
  for (int k = blockIdx.x * blockDim.x + threadIdx.x; k < nf; k += gridDim.x * blockDim.x) {
    const int x = k / fz, z = k - (k / fz) * fz;
    const size_t stride = (size_t)fz;
    const size_t i0 = (size_t)x * g.S * fz + z;
    const bool wall = axis == 0 ? (x == 0 || x == g.nx) : (z == 0 || z == g.nz);
    int ca = 0, cn = 0;
    if (!wall) {
      ca = axis == 0 ? (x - 1) * g.nz + z : x * g.nz + z - 1;
      cn = axis == 0 ? x * g.nz + z : x * g.nz + z;
    }
    const bool keep = wall || (ob[ca] == nb[ca] && ob[cn] == nb[cn]);
    const int mo = min(ob[ca], ob[cn]), mn = min(nb[ca], nb[cn]);
    if (blockIdx.y == 0) {
      const float mean0 = a[i0], slope0 = a[i0 + stride];
      if (keep) {
        a_o[i0] = mean0;
        a_o[i0 + stride] = slope0;
        continue;
      }
      const double mean = mean0, slope = slope0;
      const double mid = 0.5 * (double)(mn - 1);
      double sf = 0.0, stf = 0.0, t = -mid, to = -0.5 * (double)(mo - 1);  // both exact half-integers
      const int inside = min(mo, mn);
#pragma unroll 4
      for (int y = 0; y < inside; ++y) {
        const double f = mean + slope * to;
        sf += f;
        stf += t * f;
        t += 1.0;
        to += 1.0;
      }
      for (int y = inside; y < mn; ++y) {
        const double f = face_value(g, a, i0, stride, mo, y);
        sf += f;
        stf += t * f;
        t += 1.0;
      }
      const double stt = centred_squares(mn);
      a_o[i0] = (float)(sf / (double)mn);
      a_o[i0 + stride] = (float)(stt > 0.0 ? stf / stt : 0.0);
      continue;
    }
    const int top = min(g.ny, max(nb[ca], nb[cn]) + g.B);
    const int r0 = 2 + ((int)blockIdx.y - 1) * kRemeshRows;
#pragma unroll
    for (int q = 0; q < kRemeshRows; ++q) {
      const int s = r0 + q;
      if (s >= g.S) break;
      const size_t o = i0 + (size_t)s * stride;
      if (keep) {
        a_o[o] = a[o];
        continue;
      }
      const int y = mn + s - 2;
      a_o[o] = y < top ? (float)face_value(g, a, i0, stride, mo, y) : 0.0f;
    }
  }
}

constexpr int kRemeshHead = 16;  // ints before the bases: the changed-column counter

int grid_of(long long n) { return (int)std::min<long long>(std::max<long long>((n + 255) / 256, 1), 4096); }

}  // namespace

size_t TallGrid::remesh_bytes(int nx, int nz, int band, int max_delta) {
  const size_t P = (size_t)band + 2, S = P + (size_t)max_delta;
  const size_t state = (size_t)nx * P * nz * 2 + (size_t)(nx + 1) * S * nz + (size_t)nx * S * (nz + 1);
  auto round = [](size_t b) { return (b + 255) & ~(size_t)255; };
  return 2 * round(state * 4) + round((size_t)nx * nz * 8 + 64);
}

int TallGrid::remesh(hipStream_t s, const fp_tall_remesh_args* a, int64_t* changed_columns) {
  TallRec& R = *rec_;
  if (R.ny - R.band < 2) {
    set_error("fp_tall_remesh: fine_ny %d - band %d < 2 leaves no tall cell to re-lay", R.ny, R.band);
    return FP_ERR_LAYOUT;
  }
  const long long ncol = (long long)R.nx * R.nz;
  const size_t state = (size_t)(R.n + R.nu + R.nv + R.nw);
  if (!rm_host_) {
    int rc = rm_in_ ? FP_OK : alloc((void**)&rm_in_, state * 4);
    if (!rc && !rm_out_) rc = alloc((void**)&rm_out_, state * 4);
    if (!rc && !rm_b_) rc = alloc((void**)&rm_b_, (size_t)ncol * 8 + 64);
    if (rc) return rc;
    HIPCHK(hipHostMalloc((void**)&rm_host_, (size_t)ncol * 4 + 64, hipHostMallocDefault));
  }
  const size_t bytes[4] = {(size_t)R.n * 4, (size_t)R.nu * 4, (size_t)R.nv * 4, (size_t)R.nw * 4};
  const void* in[4] = {a->phi, a->u, a->v, a->w};
  void* out[4] = {a->phi_out, a->u_out, a->v_out, a->w_out};
  float* stage_in[4];
  float* stage_out[4];
  stage_in[0] = rm_in_;
  stage_out[0] = rm_out_;
  for (int k = 1; k < 4; ++k) {
    stage_in[k] = stage_in[k - 1] + bytes[k - 1] / 4;
    stage_out[k] = stage_out[k - 1] + bytes[k - 1] / 4;
  }
  const float* src[4];
  float* dst[4];
  if (a->memory == FP_MEMORY_HOST) {
    for (int k = 0; k < 4; ++k) {
      HIPCHK(hipMemcpyAsync(stage_in[k], in[k], bytes[k], hipMemcpyHostToDevice, s));
      src[k] = stage_in[k];
      dst[k] = stage_out[k];
    }
  } else {
    // device arrays are read in place; an output is written directly unless
    // it overlaps an input that a later kernel still reads
    for (int k = 0; k < 4; ++k) {
      src[k] = (const float*)in[k];
      bool overlaps = false;
      for (int j = 0; j < 4 && out[k]; ++j) {
        const char *o0 = (const char*)out[k], *i0 = (const char*)in[j];
        overlaps = overlaps || (o0 < i0 + bytes[j] && i0 < o0 + bytes[k]);
      }
      dst[k] = out[k] && !overlaps ? (float*)out[k] : stage_out[k];
    }
  }
  const float *ip = src[0], *iu = src[1], *iv = src[2], *iw = src[3];
  float *op = dst[0], *ou = dst[1], *ov = dst[2], *ow = dst[3];
  // counter, then the bases: they reach the host in one copy
  unsigned long long* moved = (unsigned long long*)rm_b_;
  int* raw = rm_b_ + kRemeshHead;
  int* tmp = raw + ncol;
  const RemeshGeo g{R.nx, R.ny, R.nz, R.band, R.P, R.S, R.D, 5.0 * R.h};
  // tallCellSettings.high halos (tall-cell-grid.ts:57)
  const int lh = a->liquid_halo > 0 ? a->liquid_halo : 16, ah = a->air_halo > 0 ? a->air_halo : 8;
  const int blocks = grid_of(ncol);
  hipLaunchKernelGGL(k_remesh_bases, dim3(blocks), dim3(256), 0, s, g, (const float*)ip, R.bases, raw, lh, ah,
                     moved);
  // the neighbour limit: lines along z, then along x
  hipLaunchKernelGGL(k_remesh_limit, dim3((unsigned)((R.nx + 3) / 4)), dim3(256), 0, s, R.nx, R.nz, R.nz, 1, R.D,
                     (const int*)raw, tmp);
  hipLaunchKernelGGL(k_remesh_limit, dim3((unsigned)((R.nz + 3) / 4)), dim3(256), 0, s, R.nz, R.nx, 1, R.nz, R.D,
                     (const int*)tmp, raw);
  const int* nb = raw;
  auto parts = [](int rows) { return (unsigned)(1 + (rows + kRemeshRows - 1) / kRemeshRows); };
  hipLaunchKernelGGL(k_remesh_column, dim3(blocks, parts(g.P - 1)), dim3(256), 0, s, g, R.bases, nb, (const float*)ip,
                     (const float*)iv, op, ov, moved);
  hipLaunchKernelGGL(k_remesh_faces, dim3(grid_of((long long)(R.nx + 1) * R.nz), parts(g.S - 2)), dim3(256), 0, s, g, 0, R.bases, nb,
                     (const float*)iu, ou);
  hipLaunchKernelGGL(k_remesh_faces, dim3(grid_of((long long)R.nx * (R.nz + 1)), parts(g.S - 2)), dim3(256), 0, s, g, 1, R.bases, nb,
                     (const float*)iw, ow);
  // the grid takes the new layout; its resident pressure belonged to the old one
  HIPCHK(hipMemcpyAsync(const_cast<int*>(R.bases), nb, (size_t)ncol * 4, hipMemcpyDeviceToDevice, s));
  HIPCHK(hipMemsetAsync(R.x, 0, (size_t)R.n * 8, s));
  const hipMemcpyKind kout = a->memory == FP_MEMORY_HOST ? hipMemcpyDeviceToHost : hipMemcpyDeviceToDevice;
  for (int k = 0; k < 4; ++k)
    if (out[k] && dst[k] != out[k]) HIPCHK(hipMemcpyAsync(out[k], dst[k], bytes[k], kout, s));
  HIPCHK(hipMemcpyAsync(rm_host_, rm_b_, ((size_t)kRemeshHead + (size_t)ncol) * 4, hipMemcpyDeviceToHost, s));
  HIPCHK(hipStreamSynchronize(s));
  const int* hb = rm_host_ + kRemeshHead;
  if (a->column_bases_out) std::memcpy(a->column_bases_out, hb, (size_t)ncol * 4);
  // every column's band reaching the lid leaves the pressure unanchored
  const long long anchored = R.ns_liquid;
  R.ns_liquid = 0;
  for (long long i = 0; i < ncol && R.ns_liquid >= 0; ++i)
    R.ns_liquid = hb[(size_t)i] + R.band >= R.ny ? R.ns_liquid + 2 + (R.ny - hb[(size_t)i]) : -1;
  // the state machine reads ns_liquid from the device record
  if (R.ns_liquid != anchored) {
    int rc = upload(s);
    if (rc) return rc;
    HIPCHK(hipStreamSynchronize(s));
  }
  if (changed_columns) {
    unsigned long long h_moved = 0;
    std::memcpy(&h_moved, rm_host_, sizeof(h_moved));
    *changed_columns = (int64_t)h_moved;
  }
  return FP_OK;
}

}  // namespace fp

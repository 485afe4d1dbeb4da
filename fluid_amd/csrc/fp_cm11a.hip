// fp_cm11a.hip -- the CM11a separating-wall LCP pressure solve on MI355X.
//
// Kernels restate lib/methods/uniform/webgpu-uniform-pressure-multigrid.wgsl.ts
// (cited per kernel) and the schedule of …multigrid.ts:488-576.  Every level
// is a halo-padded FP32 lattice in HBM, z fastest, with packed float4
// dual volumes and coefficients (one 16-byte word per cell).  A colour pass reads only the
// other colour, so a sweep of both is what the reference's ping-pong textures
// compute, whether it goes from one buffer to another or in place.  The whole
// file is compiled without floating-point contraction, and sums follow the
// reference's D4 order, so results equal oracle/fp_oracle_cm11a.c bit for bit.
#pragma clang fp contract(off)

#include "fp_cm11a.hpp"
#include "fp_common.hpp"
#include "fp_uniform.hpp"

#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstring>

namespace fp {

namespace {

constexpr float kNegBig = -3.402823e38f;  // the reference's "no constraint" p_min
constexpr float kThetaMin = 0.05f;
constexpr int kCoarseLanes = 1024;        // most padded cells of the coarsest level

__device__ __forceinline__ float d4s6(const float* t) { return ((t[0] + t[1]) + (t[4] + t[5])) + (t[2] + t[3]); }
__device__ __forceinline__ float d4s8(const float* t) {
  const float y0 = (t[0] + t[5]) + (t[1] + t[4]);
  const float y1 = (t[2] + t[7]) + (t[3] + t[6]);
  return y0 + y1;
}
__device__ __forceinline__ float cm_theta(float l, float a, float eps) {
  const float r = fabsf(l) / fmaxf(fabsf(l) + fabsf(a), eps);
  return fminf(1.0f, fmaxf(kThetaMin, r));
}
__constant__ int kNb[6][3] = {{-1, 0, 0}, {1, 0, 0}, {0, -1, 0}, {0, 1, 0}, {0, 0, -1}, {0, 0, 1}};

__device__ __forceinline__ int cidx(const CmLevel& L, int x, int y, int z) { return (x * L.D1 + y) * L.D2 + z; }
__device__ __forceinline__ bool cvalid(const CmLevel& L, int x, int y, int z) {
  return x >= 0 && y >= 0 && z >= 0 && x < L.D0 && y < L.D1 && z < L.D2;
}
__device__ __forceinline__ bool cinterior(const CmLevel& L, int x, int y, int z) {
  return x >= 1 && y >= 1 && z >= 1 && x < L.D0 - 1 && y < L.D1 - 1 && z < L.D2 - 1;
}
__device__ __forceinline__ void cdecode(const CmLevel& L, int i, int& x, int& y, int& z) {
  z = i % L.D2;
  const int t = i / L.D2;
  y = t % L.D1;
  x = t / L.D1;
}
__device__ __forceinline__ float hof(const CmLevel& L, int a) { return a == 0 ? L.h0 : (a == 1 ? L.h1 : L.h2); }
__device__ __forceinline__ float comp(const float4& v, int k) {
  return k == 0 ? v.x : (k == 1 ? v.y : (k == 2 ? v.z : v.w));
}

__device__ __forceinline__ int wave_sum_int(int v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_down(v, o, 64);
  return v;
}

#define CM_FOR(i, n) for (int i = (int)(blockIdx.x * blockDim.x + threadIdx.x); i < (n); i += (int)(gridDim.x * blockDim.x))

// ---- double-single arithmetic (…multigrid.wgsl.ts:364-381) ----
struct DS {
  float x, y;
};
__device__ __forceinline__ DS two_sum(float a, float b) {
  const float s = a + b;
  const float bb = s - a;
  return DS{s, (a - (s - bb)) + (b - bb)};
}
__device__ __forceinline__ DS ds_add(DS a, DS b) {
  const DS s = two_sum(a.x, b.x), t = two_sum(a.y, b.y), u = two_sum(s.y, t.x), v = two_sum(s.x, u.x);
  return DS{v.x, (v.y + u.y) + t.y};
}
__device__ __forceinline__ DS ds_neg(DS a) { return DS{-a.x, -a.y}; }
__device__ __forceinline__ DS ds_scale(DS a, float b) {
  const float product = a.x * b;
  const float error = __fmaf_rn(a.x, b, -product) + a.y * b;
  return two_sum(product, error);
}
__device__ __forceinline__ DS ds_divide(DS a, float b) {
  const float q = a.x / b;
  const DS remainder = ds_add(a, ds_neg(ds_scale(DS{q, 0.0f}, b)));
  const float correction = (remainder.x + remainder.y) / b;
  return two_sum(q, correction);
}
__device__ __forceinline__ DS d4s6_ds(const DS* v) {
  return ds_add(ds_add(ds_add(v[0], v[1]), ds_add(v[4], v[5])), ds_add(v[2], v[3]));
}

// dual volume of the positive face of an interior finest cell
// (webgpu-uniform-reference.wgsl.ts:536-561): 1 inside, 1/2 at a box wall, 1 at the open top
__device__ __forceinline__ float face_volume(int n, int c, int axis, int open_top) {
  if (c + 1 < n) return 1.0f;
  if (axis == 1 && open_top) return 1.0f;
  return 0.5f;
}

// mgBuildFinestTopology + mgBuildFinestRhs (…multigrid.wgsl.ts:135-167), the
// divergence of divergenceAt (webgpu-uniform-reference.wgsl.ts:1010-1027)
__global__ void k_cm_finest(CmLevel L, int nx, int ny, int nz, const float* __restrict__ phi,
                            const float* __restrict__ u, const float* __restrict__ v, const float* __restrict__ w,
                            const float* __restrict__ q, float dt, float rho, int open_top, float* __restrict__ b,
                            float* __restrict__ pmin, CmStats* stats) {
  const float hmin = fminf(L.h0, fminf(L.h1, L.h2));
  int liquid = 0;
  CM_FOR(i, L.n) {
    int X, Y, Z;
    cdecode(L, i, X, Y, Z);
    L.p[i] = 0.0f;
    if (cinterior(L, X, Y, Z)) {
      const int x = X - 1, y = Y - 1, z = Z - 1;
      const size_t s = ((size_t)x * ny + y) * nz + z;
      const float ph = phi[s];
      L.topo[i] = make_float4(1.0f, face_volume(nx, x, 0, open_top), face_volume(ny, y, 1, open_top),
                              face_volume(nz, z, 2, open_top));
      L.phi_raw[i] = ph;
      pmin[i] = kNegBig;
      float rhs = 0.0f;
      if (ph < 0.0f) {
        ++liquid;
        const float vi = 1.0f;
        const int c[3] = {x, y, z}, n[3] = {nx, ny, nz};
        float terms[6];
#pragma unroll
        for (int a = 0; a < 3; ++a) {
          const float vp = face_volume(n[a], c[a], a, open_top);
          const float vm = c[a] == 0 ? 0.5f : 1.0f;
          float up, um;
          if (a == 0) {
            up = u[((size_t)(x + 1) * ny + y) * nz + z];
            um = u[((size_t)x * ny + y) * nz + z];
          } else if (a == 1) {
            up = v[((size_t)x * (ny + 1) + y + 1) * nz + z];
            um = v[((size_t)x * (ny + 1) + y) * nz + z];
          } else {
            up = w[((size_t)x * ny + y) * (nz + 1) + z + 1];
            um = w[((size_t)x * ny + y) * (nz + 1) + z];
          }
          const float h = hof(L, a);
          terms[2 * a] = (vp * up) / h + (vp - vi) * 0.0f;
          terms[2 * a + 1] = -(vm * um) / h - (vm - vi) * 0.0f;
        }
        const float div = d4s6(terms);
        const float corr = q ? q[s] : 0.0f;
        rhs = rho * (div - corr) / dt;
      }
      b[i] = -rhs;
    } else {
      const bool xi = X > 0 && X < L.D0 - 1, yi = Y > 0 && Y < L.D1 - 1, zi = Z > 0 && Z < L.D2 - 1;
      const bool open = open_top && Y == L.D1 - 1 && xi && zi;
      const float o = open ? 1.0f : 0.0f;
      float4 t = make_float4(o, o, o, o);
      if (X == 0 && yi && zi) t.y = 0.5f;
      if (Y == 0 && xi && zi) t.z = 0.5f;
      if (Z == 0 && xi && yi) t.w = 0.5f;
      L.topo[i] = t;
      L.phi_raw[i] = 0.5f * hmin;
      b[i] = 0.0f;
      pmin[i] = open ? kNegBig : 0.0f;
    }
  }
  liquid = wave_sum_int(liquid);
  if ((threadIdx.x & 63) == 0 && liquid) atomicAdd(&stats->liquid, liquid);
}

// mgFineChild (…multigrid.wgsl.ts:71-76)
__device__ __forceinline__ int fine_child(const CmLevel& F, const CmLevel& C, int X, int Y, int Z, int o) {
  const int c[3] = {X, Y, Z}, fd[3] = {F.D0, F.D1, F.D2}, cd[3] = {C.D0, C.D1, C.D2};
  int out[3];
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    const int fp = fd[a] - 2;
    const int cp = max(cd[a] - 2, 1);
    const int stride = max(fp / cp, 1);
    const int oa = (o >> a) & 1;
    out[a] = min(max(stride * (c[a] - 1) + oa * (stride - 1), -1), fp) + 1;
  }
  return cidx(F, out[0], out[1], out[2]);
}

// mgDownsampleTopology (…multigrid.wgsl.ts:169-195)
__global__ void k_cm_down_topology(CmLevel F, CmLevel C, int dest, int levels, int preserve, int open_top) {
  CM_FOR(i, C.n) {
    int X, Y, Z;
    cdecode(C, i, X, Y, Z);
    float t0[8], t1[8], t2[8], t3[8], ph[8], pos[8], pf[8], nf[8];
#pragma unroll
    for (int o = 0; o < 8; ++o) {
      const int j = fine_child(F, C, X, Y, Z, o);
      const float4 t = F.topo[j];
      t0[o] = t.x;
      t1[o] = t.y;
      t2[o] = t.z;
      t3[o] = t.w;
      const float phi = F.phi_raw[j];
      ph[o] = phi;
      pos[o] = phi >= 0.0f ? phi : 0.0f;
      pf[o] = phi >= 0.0f ? 1.0f : 0.0f;
      nf[o] = phi >= 0.0f ? 0.0f : 1.0f;
    }
    const float phi_sum = d4s8(ph), pos_sum = d4s8(pos), pc = d4s8(pf), nc = d4s8(nf);
    const bool mixed = pc > 0.0f && nc > 0.0f;
    const bool use_positive = mixed && (levels - dest) >= (levels - preserve);
    float4 t = make_float4(d4s8(t0) / 8.0f, d4s8(t1) / 8.0f, d4s8(t2) / 8.0f, d4s8(t3) / 8.0f);
    if (X == C.D0 - 2) t.y = 0.5f;
    if (Y == C.D1 - 2) t.z = open_top ? 1.0f : 0.5f;
    if (Z == C.D2 - 2) t.w = 0.5f;
    C.topo[i] = t;
    C.phi_raw[i] = use_positive ? pos_sum / fmaxf(pc, 1.0f) : phi_sum / 8.0f;
  }
}

// mgExtrapolatePhiOneCell (…multigrid.wgsl.ts:288-300)
__global__ void k_cm_extrapolate(CmLevel L) {
  CM_FOR(i, L.n) {
    if (L.topo[i].x > 1e-5f) {
      L.phi[i] = L.phi_raw[i];
      continue;
    }
    int X, Y, Z;
    cdecode(L, i, X, Y, Z);
    float terms[6], wts[6];
#pragma unroll
    for (int nb = 0; nb < 6; ++nb) {
      const int x = X + kNb[nb][0], y = Y + kNb[nb][1], z = Z + kNb[nb][2];
      terms[nb] = 0.0f;
      wts[nb] = 0.0f;
      if (!cvalid(L, x, y, z)) continue;
      const int j = cidx(L, x, y, z);
      const float vq = L.topo[j].x, pq = L.phi_raw[j];
      if (vq > 1e-5f && pq < 0.0f) {
        terms[nb] = vq * pq;
        wts[nb] = vq;
      }
    }
    const float sum = d4s6(terms), weight = d4s6(wts);
    L.phi[i] = weight > 0.0f ? sum / fmaxf(weight, 1e-9f) : L.phi_raw[i];
  }
}

// mgCoefficientRaw (…multigrid.wgsl.ts:93-115), +axis face
__device__ __forceinline__ float coefficient_raw(const CmLevel& L, int i, int X, int Y, int Z, int axis,
                                                 int open_top) {
  int q[3] = {X, Y, Z};
  q[axis] += 1;
  const float h = hof(L, axis);
  if (!cvalid(L, q[0], q[1], q[2])) {
    if (axis == 1 && Y == L.D1 - 1 && open_top) {
      const float theta = cm_theta(L.phi[i], 0.5f * h, 1e-9f);
      return L.topo[i].z / (h * h * theta);
    }
    return 0.0f;
  }
  const float vf = comp(L.topo[i], 1 + axis);
  if (vf <= 1e-6f) return 0.0f;
  const int j = cidx(L, q[0], q[1], q[2]);
  const float pi = L.phi[i], pj = L.phi[j];
  const bool il = pi < 0.0f, ql = pj < 0.0f;
  float theta = 1.0f;
  if (il && !ql) theta = cm_theta(pi, pj, 1e-9f);
  if (!il && ql) theta = cm_theta(pj, pi, 1e-9f);
  return vf / (h * h * theta);
}

// A cell's stencil: its six coefficients (mgCoefficient,
// …multigrid.wgsl.ts:116-122), their sum and the liquid flags (bits 0-5 the
// neighbours, bit 6 the cell).  The level stores the three positive faces and
// the flags in one 16-byte word; the negative faces are the positive ones of
// the cells behind, so a stencil is one word and three floats, and neither
// those loads nor the neighbours' pressures wait for another.  (All six
// coefficients in 32 bytes a cell took 47.0 ms for a 256^3 projection against
// 43.7, both in sweeps: memory bounds them there.)
struct CmRecord {
  float a[6], diag;
  unsigned liq;
};
__device__ __forceinline__ CmRecord record_at(const CmLevel& L, int i, int X, int Y, int Z) {
  const float4 own = L.coef[i];
  const float* c = reinterpret_cast<const float*>(L.coef);
  const bool hx = X > 0, hy = Y > 0, hz = Z > 0;
  const float mx = c[4 * (size_t)(hx ? i - L.D1 * L.D2 : i)], my = c[4 * (size_t)(hy ? i - L.D2 : i) + 1],
              mz = c[4 * (size_t)(hz ? i - 1 : i) + 2];
  CmRecord r{{hx ? mx : 0.0f, own.x, hy ? my : 0.0f, own.y, hz ? mz : 0.0f, own.z}, 0.0f, __float_as_uint(own.w)};
  r.diag = d4s6(r.a);
  return r;
}
__device__ __forceinline__ CmRecord record_at(const CmLevel& L, int i) {
  int X, Y, Z;
  cdecode(L, i, X, Y, Z);
  return record_at(L, i, X, Y, Z);
}
constexpr unsigned kSelfLiquid = 64u;

// mgBakeCoefficients (…multigrid.wgsl.ts:302-309)
__global__ void k_cm_bake(CmLevel L, int open_top) {
  CM_FOR(i, L.n) {
    int X, Y, Z;
    cdecode(L, i, X, Y, Z);
    unsigned liq = L.phi[i] < 0.0f ? kSelfLiquid : 0u;
#pragma unroll
    for (int nb = 0; nb < 6; ++nb) {
      const int x = X + kNb[nb][0], y = Y + kNb[nb][1], z = Z + kNb[nb][2];
      if (cvalid(L, x, y, z) && L.phi[cidx(L, x, y, z)] < 0.0f) liq |= 1u << nb;
    }
    L.coef[i] = make_float4(coefficient_raw(L, i, X, Y, Z, 0, open_top), coefficient_raw(L, i, X, Y, Z, 1, open_top),
                            coefficient_raw(L, i, X, Y, Z, 2, open_top), __uint_as_float(liq));
  }
}

// The liquid neighbours' pressures of cell i (0 elsewhere)
__device__ __forceinline__ void neighbour_pressures(const CmLevel& L, const float* p, int i, unsigned liq, float* v) {
  const int off[6] = {-L.D1 * L.D2, L.D1 * L.D2, -L.D2, L.D2, -1, 1};
#pragma unroll
  for (int nb = 0; nb < 6; ++nb) {
    const bool l = liq >> nb & 1;
    const float x = p[l ? i + off[nb] : i];
    v[nb] = l ? x : 0.0f;
  }
}
// A p at a cell
__device__ __forceinline__ float apply_record(const CmRecord& r, float centre, const float* v) {
  float terms[6];
#pragma unroll
  for (int nb = 0; nb < 6; ++nb) terms[nb] = r.a[nb] * (centre - v[nb]);
  return d4s6(terms);
}
// mgSmoothColour's value of a cell (…multigrid.wgsl.ts:325-344)
__device__ __forceinline__ float smoothed(const float* a, float diag, unsigned liq, const float* v, float rhs,
                                          float centre, float pmin) {
  if (!(liq & kSelfLiquid)) return fmaxf(centre, pmin);
  float st[6];
#pragma unroll
  for (int nb = 0; nb < 6; ++nb) st[nb] = (liq >> nb & 1) ? a[nb] * v[nb] : 0.0f;
  const float sum = d4s6(st);
  const float pn = diag > 0.0f ? (sum + rhs) / diag : 0.0f;
  return fmaxf(pn, pmin);
}

// One red-black sweep of a level in one launch, from p into p2: a workgroup
// takes an 8 x 8 x 16 tile, updates the first colour on the tile and its ring
// from the old pressure, passes it through LDS and updates the second colour
// of the tile, as (even z, odd z) pairs of one cell of each colour.  The ring
// makes half the first-colour work twice, but a colour pass as a launch of its
// own is only latency on small levels: a sweep of a 34^3 level takes 7.0 us, two
// passes 8 and a gap more.  (Larger levels: kSweepCells.)
constexpr int kSweepX = 8, kSweepY = 8, kSweepZ = 16, kSweepLanes = 512;
__global__ __launch_bounds__(kSweepLanes) void k_cm_sweep(CmLevel L, const float* __restrict__ rhs,
                                                          const float* __restrict__ pmin) {
  constexpr int WX = kSweepX + 2, WY = kSweepY + 2, WP = kSweepZ / 2 + 2;  // ring 1, one pair on either side in z
  constexpr int NP = WX * WY * WP, S = (NP + kSweepLanes - 1) / kSweepLanes;
  static_assert(kSweepX * kSweepY * kSweepZ / 2 == kSweepLanes, "a lane per second-colour cell of the tile");
  __shared__ float s_first[NP];
  const float* __restrict__ p = L.p;
  float* __restrict__ out = L.p2;
  const int tz = (L.D2 + kSweepZ - 1) / kSweepZ, ty = (L.D1 + kSweepY - 1) / kSweepY;
  const int b = (int)blockIdx.x, x0 = b / (tz * ty) * kSweepX, y0 = b / tz % ty * kSweepY, z0 = b % tz * kSweepZ;
  // first colour: slots of window pairs
  int fi[S];
  CmRecord fr[S];
  float fv[S][6], frhs[S], fp[S], fmin_[S];
#pragma unroll
  for (int s = 0; s < S; ++s) {
    const int q = (int)threadIdx.x + kSweepLanes * s;
    const int wp = q % WP, t = q / WP, X = x0 - 1 + t / WY, Y = y0 - 1 + t % WY;
    const int Z = z0 - 2 + 2 * wp + ((X + Y) & 1);
    const bool in = q < NP && cvalid(L, X, Y, Z);
    const int i = in ? cidx(L, X, Y, Z) : 0;
    fi[s] = in ? i : -1;
    fr[s] = record_at(L, i, in ? X : 0, in ? Y : 0, in ? Z : 0);
    if (!in) fr[s].liq = 0;
    frhs[s] = rhs[i];
    fp[s] = p[i];
    fmin_[s] = pmin[i];
    neighbour_pressures(L, p, i, fr[s].liq, fv[s]);
  }
  // second colour: this lane's cell of the tile
  const int lp = (int)threadIdx.x % (kSweepZ / 2), lt = (int)threadIdx.x / (kSweepZ / 2);
  const int lx = lt / kSweepY, ly = lt % kSweepY, X = x0 + lx, Y = y0 + ly, odd = (X + Y + 1) & 1;
  const int Z = z0 + 2 * lp + odd;
  const bool mine = cvalid(L, X, Y, Z);
  const int i = mine ? cidx(L, X, Y, Z) : 0;
  const CmRecord r = record_at(L, i, mine ? X : 0, mine ? Y : 0, mine ? Z : 0);
  const float sr = rhs[i], sp = p[i], sm = pmin[i];
#pragma unroll
  for (int s = 0; s < S; ++s) {
    if (fi[s] < 0) continue;
    const int q = (int)threadIdx.x + kSweepLanes * s;
    const float v = smoothed(fr[s].a, fr[s].diag, fr[s].liq, fv[s], frhs[s], fp[s], fmin_[s]);
    s_first[q] = v;
    const int wp = q % WP, t = q / WP, wx = t / WY, wy = t % WY;
    if (wx >= 1 && wx <= kSweepX && wy >= 1 && wy <= kSweepY && wp >= 1 && wp <= kSweepZ / 2) out[fi[s]] = v;
  }
  __syncthreads();
  if (!mine) return;
  // every neighbour is a first-colour cell: the pair of the row beside this
  // one, or this row's pair and the one before or after it
  const int c = ((lx + 1) * WY + ly + 1) * WP + lp + 1;
  const int at[6] = {c - WY * WP, c + WY * WP, c - WP, c + WP, odd ? c : c - 1, odd ? c + 1 : c};
  float v[6];
#pragma unroll
  for (int nb = 0; nb < 6; ++nb) v[nb] = (r.liq >> nb & 1) ? s_first[at[nb]] : 0.0f;
  out[i] = smoothed(r.a, r.diag, r.liq, v, sr, sp, sm);
}

// The cells of one colour, in place, for the levels with more than kSweepCells:
// there the bytes count, k_cm_sweep reads its ring's stencils twice and those of
// air cells, and this reads an air cell's own word, pressure and p_min.
__global__ void k_cm_colour(CmLevel L, const float* __restrict__ rhs, const float* __restrict__ pmin, int colour) {
  CM_FOR(i, L.n) {
    int X, Y, Z;
    cdecode(L, i, X, Y, Z);
    if (((X + Y + Z) & 1) != colour) continue;
    if (!(__float_as_uint(L.coef[i].w) & kSelfLiquid)) {
      L.p[i] = fmaxf(L.p[i], pmin[i]);
      continue;
    }
    const CmRecord r = record_at(L, i, X, Y, Z);
    float v[6];
    neighbour_pressures(L, L.p, i, r.liq, v);
    L.p[i] = smoothed(r.a, r.diag, r.liq, v, rhs[i], L.p[i], pmin[i]);
  }
}
// Above this many padded cells: 64^3 (66^3 padded) takes 2.70 ms in colour passes
// on its finest level and 2.99 in sweeps, 96^3 4.2 and 5.1, 384^3 at rest 85 and
// 139 (105 with the passes and stencils of 32 bytes a neighbour); a 34^3 level
// in colour passes too makes the 64^3 grid's 2.90.  Between: 32 x 64 x 64 (148 K
// padded) 2.53 either way, 48 x 48 x 96 (245 K) 2.79 and 3.04; the grids of 76 K and
// 125 K, in sweeps on every level, 2.28 and 2.48, in colour passes 2.60 and 2.74.
constexpr int kSweepCells = 1 << 17;

// mgResidual (…multigrid.wgsl.ts:197-205)
__global__ void k_cm_residual(CmLevel L, const float* __restrict__ rhs, float* __restrict__ out) {
  CM_FOR(i, L.n) {
    const CmRecord r = record_at(L, i);
    float v[6];
    neighbour_pressures(L, L.p, i, r.liq, v);
    out[i] = (r.liq & kSelfLiquid) ? rhs[i] - apply_record(r, L.p[i], v) : 0.0f;
  }
}

// mgTrilinearPressure (…multigrid.wgsl.ts:217-241) at fine cell i
__device__ __forceinline__ float trilinear(const CmLevel& C, const float* cp, const CmLevel& F, int i) {
  int id[3];
  cdecode(F, i, id[0], id[1], id[2]);
  const int fd[3] = {F.D0, F.D1, F.D2}, cd[3] = {C.D0, C.D1, C.D2};
  float f[3];
  int base[3];
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    const float fine_phys = (float)(fd[a] - 2), coarse_phys = (float)(cd[a] - 2);
    const float scale = coarse_phys / fmaxf(fine_phys, 1.0f);
    const float q = ((float)id[a] - 0.5f) * scale + 0.5f;
    const float fl = floorf(q);
    base[a] = (int)fl;
    f[a] = q - fl;
  }
  float values[8], weights[8];
#pragma unroll
  for (int o = 0; o < 8; ++o) {
    const int ox = o & 1, oy = (o >> 1) & 1, oz = (o >> 2) & 1;
    const int px = base[0] + ox, py = base[1] + oy, pz = base[2] + oz;
    values[o] = 0.0f;
    weights[o] = 0.0f;
    if (!cinterior(C, px, py, pz)) continue;
    const float w = ((ox ? f[0] : 1.0f - f[0]) * (oy ? f[1] : 1.0f - f[1])) * (oz ? f[2] : 1.0f - f[2]);
    values[o] = w * cp[cidx(C, px, py, pz)];
    weights[o] = w;
  }
  const float value = d4s8(values), total = d4s8(weights);
  return total > 0.0f ? value / total : 0.0f;
}

// mgProlongateAdd / Assign (…multigrid.wgsl.ts:243-253)
__global__ void k_cm_prolong(CmLevel C, CmLevel F, int add) {
  CM_FOR(i, F.n) {
    const float t = trilinear(C, C.p, F, i);
    F.p[i] = add ? F.p[i] + t : t;
  }
}

__global__ void k_cm_fill(float* __restrict__ a, int n, float v) {
  CM_FOR(i, n) a[i] = v;
}
// mgCopyPressure + mgShiftMinimum at the start of a full cycle
__global__ void k_cm_backup_shift(const float* __restrict__ p, const float* __restrict__ pmin0,
                                  float* __restrict__ backup, float* __restrict__ shift, int n) {
  CM_FOR(i, n) {
    const float v = p[i];
    backup[i] = v;
    shift[i] = pmin0[i] - v;
  }
}
// mgAddPressure
__global__ void k_cm_add(float* __restrict__ p, const float* __restrict__ backup, int n) {
  CM_FOR(i, n) p[i] = p[i] + backup[i];
}

// mgCoarseCoefficient (…multigrid.wgsl.ts:384-397): from the coarse level set and dual volumes
__device__ __forceinline__ float coarse_coefficient(const CmLevel& L, int i, int X, int Y, int Z, int nb,
                                                    int open_top) {
  const int axis = nb / 2, x = X + kNb[nb][0], y = Y + kNb[nb][1], z = Z + kNb[nb][2];
  const float h = hof(L, axis);
  if (!cvalid(L, x, y, z)) {
    if (axis == 1 && Y == L.D1 - 1 && y == L.D1 && open_top) {
      const float theta = cm_theta(L.phi[i], 0.5f * h, 1e-9f);
      return L.topo[i].z / (h * h * theta);
    }
    return 0.0f;
  }
  const int j = cidx(L, x, y, z);
  const float vf = (nb & 1) ? comp(L.topo[i], 1 + axis) : comp(L.topo[j], 1 + axis);
  if (vf <= 1e-6f) return 0.0f;
  float theta = 1.0f;
  if (L.phi[j] >= 0.0f) theta = cm_theta(L.phi[i], L.phi[j], 1e-9f);
  return vf / (h * h * theta);
}

// mgSolveCoarsest (…multigrid.wgsl.ts:404-471): one workgroup, a lane per
// padded cell, double-single projected red-black sweeps in LDS until the
// projected residual (1/s) is at most tol, or cap sweeps.  p, rhs and pmin may
// lie in LDS.
__device__ __forceinline__ void coarsest_solve(const CmLevel& L, float* p, const float* rhs, const float* pmin,
                                               float dt, float rho, float tol, int cap, int open_top, CmStats* stats,
                                               float* sx, float* sy, unsigned& s_max) {
  const int lane = threadIdx.x;
  const bool live = lane < L.n;
  int X = 0, Y = 0, Z = 0;
  float a[6] = {0, 0, 0, 0, 0, 0};
  int j[6] = {0, 0, 0, 0, 0, 0};
  bool nl[6] = {false, false, false, false, false, false};
  bool liquid = false;
  float r = 0.0f, pm = 0.0f;
  int colour = 0;
  if (live) {
    cdecode(L, lane, X, Y, Z);
    colour = (X + Y + Z) & 1;
    liquid = L.phi[lane] < 0.0f;
    r = rhs[lane];
    pm = pmin[lane];
    sx[lane] = p[lane];
    sy[lane] = 0.0f;
    if (liquid)
#pragma unroll
      for (int nb = 0; nb < 6; ++nb) {
        a[nb] = coarse_coefficient(L, lane, X, Y, Z, nb, open_top);
        const int x = X + kNb[nb][0], y = Y + kNb[nb][1], z = Z + kNb[nb][2];
        if (cvalid(L, x, y, z)) {
          j[nb] = cidx(L, x, y, z);
          nl[nb] = L.phi[j[nb]] < 0.0f;
        }
      }
  }
  const float diag = d4s6(a);
  __syncthreads();
  int iterations = 0;
  bool converged = false;
  float worst = 0.0f;
  for (int it = 0; it < cap; ++it) {
    iterations = it + 1;
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      if (live && liquid && colour == c) {
        DS st[6];
#pragma unroll
        for (int nb = 0; nb < 6; ++nb) st[nb] = nl[nb] ? ds_scale(DS{sx[j[nb]], sy[j[nb]]}, a[nb]) : DS{0.0f, 0.0f};
        const DS sum = d4s6_ds(st);
        if (diag > 0.0f) {
          const DS next = ds_divide(ds_add(sum, DS{r, 0.0f}), diag);
          if (next.x + next.y < pm) {
            sx[lane] = pm;
            sy[lane] = 0.0f;
          } else {
            sx[lane] = next.x;
            sy[lane] = next.y;
          }
        }
      }
      __syncthreads();
    }
    if (live && sx[lane] + sy[lane] < pm) {
      sx[lane] = pm;
      sy[lane] = 0.0f;
    }
    if (lane == 0) s_max = 0u;
    __syncthreads();
    if (live && liquid && diag > 0.0f) {
      const DS P{sx[lane], sy[lane]};
      DS ap[6];
#pragma unroll
      for (int nb = 0; nb < 6; ++nb) {
        const DS nv = nl[nb] ? DS{sx[j[nb]], sy[j[nb]]} : DS{0.0f, 0.0f};
        ap[nb] = ds_scale(ds_add(P, ds_neg(nv)), a[nb]);
      }
      const DS applied = d4s6_ds(ap);
      const DS lrp = ds_add(DS{r, 0.0f}, ds_neg(applied));
      const float lr = lrp.x + lrp.y;
      const float pressure = P.x + P.y;
      const float gap = fmaxf(0.0f, pressure - pm);
      const bool projects = lr < 0.0f && -lr >= gap * diag;
      const float lcp = projects ? gap * diag : fabsf(lr);
      const float divres = lcp * dt / rho;
      atomicMax(&s_max, __float_as_uint(divres));
    }
    __syncthreads();
    worst = __uint_as_float(s_max);
    if (worst <= tol) {
      converged = true;
      break;
    }
    __syncthreads();  // s_max is reset by the next iteration
  }
  if (live) p[lane] = sx[lane] + sy[lane];
  if (lane == 0) {
    stats->coarse_sweeps = max(stats->coarse_sweeps, iterations);
    stats->coarse_residual_bits = max(stats->coarse_residual_bits, __float_as_uint(worst));
    stats->coarse_failed += converged ? 0 : 1;
    stats->coarse_solves += 1;
  }
}

__global__ __launch_bounds__(kCoarseLanes) void k_cm_coarse(CmLevel L, const float* __restrict__ rhs,
                                                            const float* __restrict__ pmin, float dt, float rho,
                                                            float tol, int cap, int open_top, CmStats* stats) {
  __shared__ float sx[kCoarseLanes], sy[kCoarseLanes];
  __shared__ unsigned s_max;
  coarsest_solve(L, L.p, rhs, pmin, dt, rho, tol, cap, open_top, stats, sx, sy, s_max);
}

// mgResidual, mgRestrictResidual (…multigrid.wgsl.ts:197-215), the zero start
// and mgDownsampleSubtract (:311-323) of the next level in one launch: a lane per
// coarse cell evaluates the stencils of its eight children (a child away from
// the halo belongs to one coarse cell, so hardly any residual is made twice).
__global__ void k_cm_descend(CmLevel F, const float* __restrict__ rhs, const float* __restrict__ fmin, int constrained,
                             CmLevel C) {
  CM_FOR(i, C.n) {
    int X, Y, Z;
    cdecode(C, i, X, Y, Z);
    float t[8];
    float lower = kNegBig;
#pragma unroll
    for (int o = 0; o < 8; ++o) {
      const int j = fine_child(F, C, X, Y, Z, o);
      const CmRecord r = record_at(F, j);
      const float centre = F.p[j];
      if (constrained) lower = fmaxf(lower, fmin[j] - centre);
      float v[6];
      neighbour_pressures(F, F.p, j, r.liq, v);
      t[o] = (r.liq & kSelfLiquid) ? rhs[j] - apply_record(r, centre, v) : 0.0f;
    }
    C.rhs0[i] = d4s8(t) / 8.0f;
    C.p[i] = 0.0f;
    C.pmin[i] = lower;
  }
}

// mgRestrictResidual and mgDownsampleMinimum of a full cycle's way down
__global__ void k_cm_full_down(CmLevel F, const float* __restrict__ fmin, int constrained, CmLevel C) {
  CM_FOR(i, C.n) {
    int X, Y, Z;
    cdecode(C, i, X, Y, Z);
    float t[8];
    float lower = kNegBig;
#pragma unroll
    for (int o = 0; o < 8; ++o) {
      const int j = fine_child(F, C, X, Y, Z, o);
      t[o] = F.rhs1[j];
      if (constrained) lower = fmaxf(lower, fmin[j]);
    }
    C.rhs1[i] = d4s8(t) / 8.0f;
    C.pmin[i] = lower;
  }
}

// ---------------------------------------------------------------------------
// The tail of the schedule in one workgroup: every level from `first` on (at
// most kTailCells padded cells in all) keeps its pressure, right-hand sides
// and p_min in LDS, so a colour pass is a barrier instead of a launch.  On a
// 64^3 grid 1152 of the 1560 colour passes are on these levels, and a launch
// of one took 4 to 5 us with its gap; a V-cycle from 18^3 takes 63 us here, one
// of 72 passes and 3 transfers, or about one us a pass.  A lane owns (even z,
// odd z) pairs of cells, one of each colour, and holds their coefficients in
// registers for a whole smoothing leg.  The arithmetic is that of k_cm_sweep,
// k_cm_descend, k_cm_full_down, k_cm_prolong and k_cm_coarse.
// ---------------------------------------------------------------------------
constexpr int kTailLanes = 1024;
constexpr int kTailSlots = 3;       // pairs per lane on the first level
constexpr int kTailCells = 7424;    // 16 bytes of LDS each, and 4 for the first level's residuals
constexpr int kTailLevels = kMaxLevels;
constexpr size_t kTailLds = (size_t)kTailCells * 20;  // beside the coarsest solve's static LDS, within a CU's 160 KB
static_assert(kTailLds + kCoarseLanes * 8 + 256 <= 160 * 1024, "the tail fits a CU");

struct CmTail {
  CmLevel lv[kTailLevels];
  int first, levels, constraint_levels;
  int sweeps;
  float dt, rho, tol;
  int cap, open_top;
};

template <int S>
struct TailCells {
  CmRecord r[2][S];
  float rhs[2][S], pm[2][S];
  int i[2][S];             // LDS index, -1: no cell
  __device__ __forceinline__ void load(const CmLevel& L, const float* rhs_, const float* pmin_) {
    const int PZ = (L.D2 + 1) / 2, pairs = L.D0 * L.D1 * PZ;
#pragma unroll
    for (int s = 0; s < S; ++s) {
      const int q = (int)threadIdx.x + kTailLanes * s;
      const int pz = q % PZ, t = q / PZ, Y = t % L.D1, X = t / L.D1;
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        const int Z = 2 * pz + ((X + Y + c) & 1);
        const bool in = q < pairs && Z < L.D2;
        const int j = in ? cidx(L, X, Y, Z) : 0;
        i[c][s] = in ? j : -1;
        r[c][s] = record_at(L, j, in ? X : 0, in ? Y : 0, in ? Z : 0);
        rhs[c][s] = rhs_[j];
        pm[c][s] = pmin_[j];
      }
    }
  }
  // mgSmoothColour of one colour
  __device__ __forceinline__ void smooth(const CmLevel& L, float* p, int c) const {
#pragma unroll
    for (int s = 0; s < S; ++s) {
      if (i[c][s] < 0) continue;
      float v[6];
      neighbour_pressures(L, p, i[c][s], r[c][s].liq, v);
      p[i[c][s]] = smoothed(r[c][s].a, r[c][s].diag, r[c][s].liq, v, rhs[c][s], p[i[c][s]], pm[c][s]);
    }
  }
  __device__ __forceinline__ void residual(const CmLevel& L, const float* p, float* out) const {
#pragma unroll
    for (int c = 0; c < 2; ++c)
#pragma unroll
      for (int s = 0; s < S; ++s) {
        if (i[c][s] < 0) continue;
        float v[6];
        neighbour_pressures(L, p, i[c][s], r[c][s].liq, v);
        out[i[c][s]] = (r[c][s].liq & kSelfLiquid) ? rhs[c][s] - apply_record(r[c][s], p[i[c][s]], v) : 0.0f;
      }
  }
};

// A level's arrays in LDS: p, rhs0, rhs1, pmin.
struct TailArrays {
  float *p, *rhs0, *rhs1, *pmin;
};
__device__ __forceinline__ TailArrays tail_arrays(const CmTail& T, float* base, int l) {
  for (int k = T.first; k < l; ++k) base += 4 * T.lv[k].n;
  const int n = T.lv[l].n;
  return TailArrays{base, base + n, base + 2 * n, base + 3 * n};
}

template <int S>
__device__ __forceinline__ void tail_smooth(const CmTail& T, int l, const TailArrays& A, const float* rhs, float* res) {
  const CmLevel& L = T.lv[l];
  TailCells<S> cells;
  cells.load(L, rhs, A.pmin);
  for (int k = 0; k < T.sweeps; ++k)
    for (int c = 0; c < 2; ++c) {
      cells.smooth(L, A.p, c);
      __syncthreads();
    }
  if (res) {
    cells.residual(L, A.p, res);
    __syncthreads();
  }
}

__device__ __forceinline__ void tail_prolong(const CmLevel& C, const float* cp, const CmLevel& F, float* fp, int add) {
  for (int i = (int)threadIdx.x; i < F.n; i += kTailLanes) {
    const float t = trilinear(C, cp, F, i);
    fp[i] = add ? fp[i] + t : t;
  }
}

// full: 1 the part of a full cycle on these levels (in: the first level's rhs1
// and p_min; out: its pressure after its V-cycle), 0 one V-cycle from the
// first level (in: its rhs0 and p_min, pressure zero).
__global__ __launch_bounds__(kTailLanes) void k_cm_tail(CmTail T, int full, CmStats* stats) {
  extern __shared__ float s_tail[];
  __shared__ float sx[kCoarseLanes], sy[kCoarseLanes];
  __shared__ unsigned s_max;
  const int tid = (int)threadIdx.x, first = T.first, last = T.levels - 1;
  float* res = s_tail;  // the first level's cells, reused by the levels below it
  float* base = s_tail + T.lv[first].n;
  {
    const CmLevel& L = T.lv[first];
    const TailArrays A = tail_arrays(T, base, first);
    const float* __restrict__ src = full ? L.rhs1 : L.rhs0;
    float* dst = full ? A.rhs1 : A.rhs0;
    for (int i = tid; i < L.n; i += kTailLanes) {
      A.p[i] = 0.0f;
      dst[i] = src[i];
      A.pmin[i] = L.pmin[i];
    }
  }
  __syncthreads();
  // one V-cycle from level l0 with its right-hand side
  auto vcycle = [&](int l0, bool first_rhs1) {
    for (int l = l0; l < last; ++l) {
      const TailArrays A = tail_arrays(T, base, l), N = tail_arrays(T, base, l + 1);
      const float* rhs = l == l0 && first_rhs1 ? A.rhs1 : A.rhs0;
      if (l == first) tail_smooth<kTailSlots>(T, l, A, rhs, res);
      else tail_smooth<1>(T, l, A, rhs, res);
      const CmLevel &F = T.lv[l], &C = T.lv[l + 1];
      for (int i = tid; i < C.n; i += kTailLanes) {
        int X, Y, Z;
        cdecode(C, i, X, Y, Z);
        float t[8], lower = kNegBig;
#pragma unroll
        for (int o = 0; o < 8; ++o) {
          const int j = fine_child(F, C, X, Y, Z, o);
          t[o] = res[j];
          if (l < T.constraint_levels) lower = fmaxf(lower, A.pmin[j] - A.p[j]);
        }
        N.rhs0[i] = d4s8(t) / 8.0f;
        N.p[i] = 0.0f;
        N.pmin[i] = lower;
      }
      __syncthreads();
    }
    {
      const TailArrays A = tail_arrays(T, base, last);
      coarsest_solve(T.lv[last], A.p, l0 == last && first_rhs1 ? A.rhs1 : A.rhs0, A.pmin, T.dt, T.rho, T.tol, T.cap,
                     T.open_top, stats, sx, sy, s_max);
      __syncthreads();
    }
    for (int l = last - 1; l >= l0; --l) {
      const TailArrays A = tail_arrays(T, base, l), N = tail_arrays(T, base, l + 1);
      tail_prolong(T.lv[l + 1], N.p, T.lv[l], A.p, 1);
      __syncthreads();
      const float* rhs = l == l0 && first_rhs1 ? A.rhs1 : A.rhs0;
      if (l == first) tail_smooth<kTailSlots>(T, l, A, rhs, nullptr);
      else tail_smooth<1>(T, l, A, rhs, nullptr);
    }
  };
  if (full) {
    for (int l = first; l < last; ++l) {
      const TailArrays A = tail_arrays(T, base, l), N = tail_arrays(T, base, l + 1);
      const CmLevel &F = T.lv[l], &C = T.lv[l + 1];
      for (int i = tid; i < C.n; i += kTailLanes) {
        int X, Y, Z;
        cdecode(C, i, X, Y, Z);
        float t[8], lower = kNegBig;
#pragma unroll
        for (int o = 0; o < 8; ++o) {
          const int j = fine_child(F, C, X, Y, Z, o);
          t[o] = A.rhs1[j];
          if (l < T.constraint_levels) lower = fmaxf(lower, A.pmin[j]);
        }
        N.rhs1[i] = d4s8(t) / 8.0f;
        N.p[i] = 0.0f;
        N.pmin[i] = lower;
      }
      __syncthreads();
    }
    for (int l = last; l >= first; --l) {
      if (l < last) {
        tail_prolong(T.lv[l + 1], tail_arrays(T, base, l + 1).p, T.lv[l], tail_arrays(T, base, l).p, 0);
        __syncthreads();
      }
      vcycle(l, true);
    }
  } else {
    vcycle(first, false);
  }
  const CmLevel& L = T.lv[first];
  const TailArrays A = tail_arrays(T, base, first);
  for (int i = tid; i < L.n; i += kTailLanes) L.p[i] = A.p[i];
}

// Max of non-negative floats (as bits) into *out: one atomic per workgroup, and
// only where it can raise the value.  One per wave on a single address, 4096
// of them at 64^3, was 48 us of a 4 us pass.
__device__ __forceinline__ void max_bits(float v, unsigned* out) {
  const unsigned m = __float_as_uint(block_max(v));
  if (threadIdx.x == 0 && m > __hip_atomic_load(out, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) atomicMax(out, m);
}

// mgMeasureFineResidual (…multigrid.wgsl.ts:473-481): max projected residual
// (1/s) and, per workgroup, the sum of squares of the projected residual and
// of b (the relative LCP residual of the report)
__global__ void k_cm_measure(CmLevel L, const float* __restrict__ b, const float* __restrict__ pmin, float dt,
                             float rho, CmStats* stats, double* partials) {
  double acc[2] = {0.0, 0.0};
  float mx = 0.0f;
  CM_FOR(i, L.n) {
    const CmRecord c = record_at(L, i);
    if (!(c.liq & kSelfLiquid)) continue;
    const float diag = c.diag;
    if (diag <= 0.0f) continue;
    float v[6];
    neighbour_pressures(L, L.p, i, c.liq, v);
    const float r = b[i] - apply_record(c, L.p[i], v);
    const float gap = fmaxf(0.0f, L.p[i] - pmin[i]);
    const bool projects = r < 0.0f && -r >= gap * diag;
    const float pr = projects ? gap * diag : fabsf(r);
    mx = fmaxf(mx, pr * dt / rho);
    acc[0] += (double)pr * (double)pr;
    acc[1] += (double)b[i] * (double)b[i];
  }
  max_bits(mx, &stats->lcp_residual_bits);
  block_sum<2>(acc);
  if (threadIdx.x == 0) {
    partials[2 * blockIdx.x] = acc[0];
    partials[2 * blockIdx.x + 1] = acc[1];
  }
}

// max |div u| over liquid cells with the dual-volume divergence (1/s)
__global__ void k_cm_max_div(int nx, int ny, int nz, float h, const float* __restrict__ phi,
                             const float* __restrict__ u, const float* __restrict__ v, const float* __restrict__ w,
                             int open_top, unsigned* out_bits) {
  const int n = nx * ny * nz;
  float mx = 0.0f;
  CM_FOR(s, n) {
    if (!(phi[s] < 0.0f)) continue;
    const int z = s % nz, t = s / nz, y = t % ny, x = t / ny;
    const int c[3] = {x, y, z}, nn[3] = {nx, ny, nz};
    float terms[6];
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      const float vp = face_volume(nn[a], c[a], a, open_top);
      const float vm = c[a] == 0 ? 0.5f : 1.0f;
      float up, um;
      if (a == 0) {
        up = u[((size_t)(x + 1) * ny + y) * nz + z];
        um = u[((size_t)x * ny + y) * nz + z];
      } else if (a == 1) {
        up = v[((size_t)x * (ny + 1) + y + 1) * nz + z];
        um = v[((size_t)x * (ny + 1) + y) * nz + z];
      } else {
        up = w[((size_t)x * ny + y) * (nz + 1) + z + 1];
        um = w[((size_t)x * ny + y) * (nz + 1) + z];
      }
      terms[2 * a] = (vp * up) / h;
      terms[2 * a + 1] = -(vm * um) / h;
    }
    mx = fmaxf(mx, fabsf(d4s6(terms)));
  }
  max_bits(mx, out_bits);
}

// project (webgpu-uniform-reference.wgsl.ts:1052-1099) on a box container:
// each face is written by the thread of the cell below it (and the low wall
// faces by the cells at index 0), so outputs may alias the inputs
__global__ void k_cm_project(CmLevel L, int nx, int ny, int nz, const float* __restrict__ phi, const float* uin,
                             const float* vin, const float* win, float* uo, float* vo, float* wo, float dt, float rho,
                             int open_top) {
  const float scale = dt / rho;
  const float hmin = fminf(L.h0, fminf(L.h1, L.h2));
  const int n = nx * ny * nz;
  CM_FOR(s, n) {
    const int z = s % nz, t = s / nz, y = t % ny, x = t / ny;
    const int c[3] = {x, y, z}, nn[3] = {nx, ny, nz};
    const float ph = phi[s];
    const bool liquid = ph < 0.0f;
    const float p0 = liquid ? L.p[cidx(L, x + 1, y + 1, z + 1)] : 0.0f;
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      const float* fin = a == 0 ? uin : (a == 1 ? vin : win);
      float* fo = a == 0 ? uo : (a == 1 ? vo : wo);
      if (!fo) continue;
      size_t lo, hi;
      if (a == 0) {
        lo = ((size_t)x * ny + y) * nz + z;
        hi = ((size_t)(x + 1) * ny + y) * nz + z;
      } else if (a == 1) {
        lo = ((size_t)x * (ny + 1) + y) * nz + z;
        hi = ((size_t)x * (ny + 1) + y + 1) * nz + z;
      } else {
        lo = ((size_t)x * ny + y) * (nz + 1) + z;
        hi = ((size_t)x * ny + y) * (nz + 1) + z + 1;
      }
      const float h = hof(L, a);
      if (c[a] == 0) {
        int hc[3] = {x + 1, y + 1, z + 1};
        hc[a] = 0;
        fo[lo] = liquid ? fin[lo] - scale * (p0 - L.p[cidx(L, hc[0], hc[1], hc[2])]) / h : 0.0f;
      }
      if (c[a] == nn[a] - 1) {
        if (a == 1 && open_top) {
          if (liquid) {
            const float theta = cm_theta(ph, 0.5f * hmin, 1e-6f);
            fo[hi] = fin[hi] - scale * (0.0f - p0) / (h * theta);
          } else {
            fo[hi] = 0.0f;
          }
        } else if (liquid) {
          int hc[3] = {x + 1, y + 1, z + 1};
          hc[a] = nn[a] + 1;
          fo[hi] = fin[hi] - scale * (L.p[cidx(L, hc[0], hc[1], hc[2])] - p0) / h;
        } else {
          fo[hi] = 0.0f;
        }
        continue;
      }
      int d[3] = {x, y, z};
      d[a] += 1;
      const size_t sn = ((size_t)d[0] * ny + d[1]) * nz + d[2];
      const float pn = phi[sn];
      const bool nlq = pn < 0.0f;
      if (liquid || nlq) {
        const float p1 = nlq ? L.p[cidx(L, d[0] + 1, d[1] + 1, d[2] + 1)] : 0.0f;
        float theta = 1.0f;
        if (liquid && !nlq) theta = cm_theta(ph, pn, 1e-6f);
        if (!liquid && nlq) theta = cm_theta(pn, ph, 1e-6f);
        fo[hi] = fin[hi] - scale * (p1 - p0) / (h * theta);
      } else {
        fo[hi] = 0.0f;
      }
    }
  }
}

// interior pressure of the liquid cells (0 elsewhere) into the caller's array
__global__ void k_cm_pressure_out(CmLevel L, int nx, int ny, int nz, const float* __restrict__ phi,
                                  float* __restrict__ out) {
  const int n = nx * ny * nz;
  CM_FOR(s, n) {
    const int z = s % nz, t = s / nz, y = t % ny, x = t / ny;
    out[s] = phi[s] < 0.0f ? L.p[cidx(L, x + 1, y + 1, z + 1)] : 0.0f;
  }
}

int grid_for(long long n) { return (int)std::min<long long>(std::max<long long>((n + 255) / 256, 1), 65536); }
constexpr int kMeasureBlocks = 1024;

}  // namespace

#define CM_LAUNCH(kern, n, s, ...) hipLaunchKernelGGL(kern, dim3(grid_for(n)), dim3(256), 0, s, ##__VA_ARGS__)

Cm11a::~Cm11a() {
  for (void* p : allocations_) (void)hipFree(p);
}

int Cm11a::alloc(void** p, size_t bytes) {
  bytes = (bytes + 255) & ~(size_t)255;
  if (hipMalloc(p, bytes) != hipSuccess) {
    set_error("CM11a: hipMalloc(%zu) failed", bytes);
    return FP_ERR_OUT_OF_MEMORY;
  }
  allocations_.push_back(*p);
  bytes_ += bytes;
  return FP_OK;
}

size_t Cm11a::estimate_bytes(int nx, int ny, int nz) {
  int dims[kMaxLevels][3], strides[kMaxLevels][3];
  const int L = plan_uniform_levels(nx, ny, nz, dims, strides);
  size_t total = 0;
  auto up = [](size_t b) { return (b + 255) & ~(size_t)255; };
  for (int l = 0; l < L; ++l) {
    const size_t n = (size_t)(dims[l][0] + 2) * (dims[l][1] + 2) * (dims[l][2] + 2);
    total += (n > kSweepCells ? 6 : 7) * up(n * 4) + 2 * up(n * 16);
    if (l == 0) total += 4 * up(n * 4);
  }
  return total + up((size_t)kMeasureBlocks * 16) + up(sizeof(CmStats));
}

int Cm11a::create(int nx, int ny, int nz, double h) {
  int dims[kMaxLevels][3], strides[kMaxLevels][3];
  const int L = plan_uniform_levels(nx, ny, nz, dims, strides);
  if (L <= 0) {
    set_error("CM11a: no level plan for %dx%dx%d", nx, ny, nz);
    return FP_ERR_LAYOUT;
  }
  // the reference's hierarchy halves axes exactly (mgFineChild's stride): a
  // lattice its planner rejects (the library ceil-halves those) has no CM11a form
  for (int l = 1; l < L; ++l)
    for (int a = 0; a < 3; ++a)
      if (dims[l][a] != dims[l - 1][a] && 2 * dims[l][a] != dims[l - 1][a]) {
        set_error("CM11a: %dx%dx%d has no hierarchy of exact halvings (planUniformCM11aHierarchy rejects it)", nx,
                  ny, nz);
        return FP_ERR_LAYOUT;
      }
  const long long coarsest = (long long)(dims[L - 1][0] + 2) * (dims[L - 1][1] + 2) * (dims[L - 1][2] + 2);
  if (coarsest > kCoarseLanes) {
    set_error("CM11a: the coarsest level of %dx%dx%d has %lld cells with its halo (at most %d)", nx, ny, nz,
              coarsest, kCoarseLanes);
    return FP_ERR_UNSUPPORTED;
  }
  nx_ = nx, ny_ = ny, nz_ = nz, h_ = h;
  const int n[3] = {nx, ny, nz};
  lv_.resize(L);
  for (int l = 0; l < L; ++l) {
    CmLevel& c = lv_[l];
    c.D0 = dims[l][0] + 2;
    c.D1 = dims[l][1] + 2;
    c.D2 = dims[l][2] + 2;
    c.n = c.D0 * c.D1 * c.D2;
    // spacing of the level: h * (finest cells / level cells) per axis (…multigrid.ts:583-588)
    c.h0 = (float)(h * ((double)n[0] / (double)dims[l][0]));
    c.h1 = (float)(h * ((double)n[1] / (double)dims[l][1]));
    c.h2 = (float)(h * ((double)n[2] / (double)dims[l][2]));
    const size_t b4 = (size_t)c.n * 4, b16 = (size_t)c.n * 16;
    int rc = alloc((void**)&c.phi_raw, b4);
    if (!rc) rc = alloc((void**)&c.phi, b4);
    if (!rc) rc = alloc((void**)&c.topo, b16);
    if (!rc) rc = alloc((void**)&c.coef, b16);
    if (!rc) rc = alloc((void**)&c.p, b4);
    if (!rc && c.n <= kSweepCells) rc = alloc((void**)&c.p2, b4);  // k_cm_colour works in place
    if (!rc) rc = alloc((void**)&c.rhs0, b4);
    if (!rc) rc = alloc((void**)&c.rhs1, b4);
    if (!rc) rc = alloc((void**)&c.pmin, b4);
    if (rc) return rc;
  }
  const size_t b0 = (size_t)lv_[0].n * 4;
  int rc = alloc((void**)&b_, b0);
  if (!rc) rc = alloc((void**)&pmin0_, b0);
  if (!rc) rc = alloc((void**)&pshift_, b0);
  if (!rc) rc = alloc((void**)&backup_, b0);
  if (!rc) rc = alloc((void**)&partials_, (size_t)kMeasureBlocks * 16);
  if (!rc) rc = alloc((void**)&stats_, sizeof(CmStats));
  if (rc) return rc;
  // the tail starts at the first level (not the finest) whose levels fit; a
  // device that gives a workgroup less LDS keeps one launch per pass.  The limit
  // belongs to the kernel on this device and not to a grid: every grid asks for
  // the same, the most that a tail takes.
  for (int l = 1; l + 1 < L && tail_ == 0; ++l)
    if (tail_lds(l)) tail_ = l;
  if (tail_ > 0 && hipFuncSetAttribute(reinterpret_cast<const void*>(&k_cm_tail),
                                       hipFuncAttributeMaxDynamicSharedMemorySize, (int)kTailLds) != hipSuccess) {
    (void)hipGetLastError();
    tail_ = 0;
  }
  return FP_OK;
}

void Cm11a::coarse_solve(hipStream_t s, const float* rhs, const float* pmin) {
  const CmLevel& c = lv_.back();
  const int threads = std::max(64, ((c.n + 63) / 64) * 64);
  hipLaunchKernelGGL(k_cm_coarse, dim3(1), dim3(threads), 0, s, c, rhs, pmin, dt_, rho_, tol_, cap_, open_top_,
                     stats_);
}

// Bytes of k_cm_tail's dynamic LDS for the levels from `first` on, 0 when they
// do not fit its lanes and LDS.
size_t Cm11a::tail_lds(int first) const {
  const int L = (int)lv_.size();
  long long cells = 0;
  for (int l = first; l < L; ++l) cells += lv_[l].n;
  auto pairs = [&](int l) { return (long long)lv_[l].D0 * lv_[l].D1 * ((lv_[l].D2 + 1) / 2); };
  if (pairs(first) > (long long)kTailSlots * kTailLanes) return 0;
  if (first + 1 < L - 1 && pairs(first + 1) > kTailLanes) return 0;
  if (cells > kTailCells || L > kTailLevels) return 0;
  return ((size_t)cells * 4 + (size_t)lv_[first].n) * sizeof(float);
}

void Cm11a::tail(hipStream_t s, int full) {
  CmTail t;
  std::memset(&t, 0, sizeof(t));
  const int L = (int)lv_.size();
  for (int l = 0; l < L; ++l) t.lv[l] = lv_[l];
  t.first = tail_;
  t.levels = L;
  t.constraint_levels = constraint_levels_;
  t.sweeps = pre_;
  t.dt = dt_;
  t.rho = rho_;
  t.tol = tol_;
  t.cap = cap_;
  t.open_top = open_top_;
  hipLaunchKernelGGL(k_cm_tail, dim3(1), dim3(kTailLanes), tail_lds(tail_), s, t, full, stats_);
}

// `count` red-black sweeps; each writes the level's other pressure buffer,
// which then is the level's pressure.
void Cm11a::sweeps(hipStream_t s, CmLevel& c, int count, const float* rhs, const float* pmin) {
  if (c.n > kSweepCells) {
    for (int i = 0; i < count; ++i)
      for (int colour = 0; colour < 2; ++colour) CM_LAUNCH(k_cm_colour, c.n, s, c, rhs, pmin, colour);
    return;
  }
  auto tiles = [](int n, int t) { return (n + t - 1) / t; };
  const int groups = tiles(c.D0, kSweepX) * tiles(c.D1, kSweepY) * tiles(c.D2, kSweepZ);
  for (int i = 0; i < count; ++i) {
    hipLaunchKernelGGL(k_cm_sweep, dim3(groups), dim3(kSweepLanes), 0, s, c, rhs, pmin);
    std::swap(c.p, c.p2);
  }
}

// vCycle (…multigrid.ts:518-533); pmin0: the finest level's current p_min
void Cm11a::vcycle(hipStream_t s, int l, const float* rhs, const float* pmin0) {
  const int L = (int)lv_.size();
  CmLevel& c = lv_[l];
  const float* pmin = l == 0 ? pmin0 : c.pmin;
  if (l == L - 1) {
    coarse_solve(s, rhs, pmin);
    return;
  }
  CmLevel& d = lv_[l + 1];
  sweeps(s, c, pre_, rhs, pmin);
  CM_LAUNCH(k_cm_descend, d.n, s, c, rhs, pmin, l < constraint_levels_ ? 1 : 0, d);
  if (l + 1 == tail_) tail(s, 0);
  else vcycle(s, l + 1, d.rhs0, pmin0);
  CM_LAUNCH(k_cm_prolong, c.n, s, d, c, 1);
  sweeps(s, c, post_, rhs, pmin);
}

// fullCycle (…multigrid.ts:534-557)
void Cm11a::full_cycle(hipStream_t s, const float* pmin0) {
  const int L = (int)lv_.size();
  CmLevel& f = lv_[0];
  CM_LAUNCH(k_cm_backup_shift, f.n, s, (const float*)f.p, pmin0, backup_, pshift_, f.n);
  CM_LAUNCH(k_cm_residual, f.n, s, f, (const float*)b_, f.rhs1);
  const int deep = tail_ > 0 ? tail_ : L - 1;  // the levels below run in the tail, or are the coarsest
  for (int l = 0; l < deep; ++l)
    CM_LAUNCH(k_cm_full_down, lv_[l + 1].n, s, lv_[l], (const float*)(l == 0 ? pshift_ : lv_[l].pmin),
              l < constraint_levels_ ? 1 : 0, lv_[l + 1]);
  if (tail_ > 0) {
    tail(s, 1);
  } else {
    CmLevel& cc = lv_[L - 1];
    CM_LAUNCH(k_cm_fill, cc.n, s, cc.p, cc.n, 0.0f);
    coarse_solve(s, cc.rhs1, L == 1 ? pshift_ : cc.pmin);
  }
  for (int l = deep - 1; l >= 0; --l) {
    CM_LAUNCH(k_cm_prolong, lv_[l].n, s, lv_[l + 1], lv_[l], 0);
    vcycle(s, l, lv_[l].rhs1, pshift_);
  }
  CM_LAUNCH(k_cm_add, f.n, s, f.p, (const float*)backup_, f.n);
}

int Cm11a::run(hipStream_t s, UniformGrid* g, const fp_options* opt, double dt, double rho, fp_report* rep) {
  const auto t0 = std::chrono::steady_clock::now();
  GridRec& R = *g->host_rec();
  const int L = (int)lv_.size();
  pre_ = opt->lcp_sweeps > 0 ? opt->lcp_sweeps : 6;
  post_ = pre_;
  const int full = opt->full_cycles > 0 ? opt->full_cycles : 3;
  const int vcyc = opt->v_cycles > 0 ? opt->v_cycles : 4;
  open_top_ = opt->open_top ? 1 : 0;
  dt_ = (float)dt;
  rho_ = (float)rho;
  const float* phi = R.lv[0].phi;  // the staged level set
  HIPCHK(hipMemsetAsync(stats_, 0, sizeof(CmStats), s));
  CmLevel& f = lv_[0];
  CM_LAUNCH(k_cm_max_div, (long long)nx_ * ny_ * nz_, s, nx_, ny_, nz_, (float)h_, phi, R.in_u, R.in_v, R.in_w,
            open_top_, &stats_->div_before_bits);
  CM_LAUNCH(k_cm_finest, f.n, s, f, nx_, ny_, nz_, phi, R.in_u, R.in_v, R.in_w, R.in_q, dt_, rho_, open_top_, b_,
            pmin0_, stats_);
  for (int l = 0; l + 1 < L; ++l)
    CM_LAUNCH(k_cm_down_topology, lv_[l + 1].n, s, lv_[l], lv_[l + 1], l + 1, L, 2, open_top_);
  for (int l = 0; l < L; ++l) {
    CM_LAUNCH(k_cm_extrapolate, lv_[l].n, s, lv_[l]);
    CM_LAUNCH(k_cm_bake, lv_[l].n, s, lv_[l], open_top_);
  }
  for (int k = 0; k < full; ++k) full_cycle(s, pmin0_);
  for (int k = 0; k < vcyc; ++k) vcycle(s, 0, b_, pmin0_);
  hipLaunchKernelGGL(k_cm_measure, dim3(kMeasureBlocks), dim3(256), 0, s, f, (const float*)b_, (const float*)pmin0_,
                     dt_, rho_, stats_, partials_);
  // outputs: the projected velocities (in place when they alias the inputs) and the pressure
  hipLaunchKernelGGL(k_cm_project, dim3(grid_for((long long)nx_ * ny_ * nz_)), dim3(256), 0, s, f, nx_, ny_, nz_,
                     phi, R.in_u, R.in_v, R.in_w, R.out_u, R.out_v, R.out_w, dt_, rho_, open_top_);
  if (R.out_p)
    CM_LAUNCH(k_cm_pressure_out, (long long)nx_ * ny_ * nz_, s, f, nx_, ny_, nz_, phi, R.out_p);
  if (R.out_u && R.out_v && R.out_w)
    CM_LAUNCH(k_cm_max_div, (long long)nx_ * ny_ * nz_, s, nx_, ny_, nz_, (float)h_, phi, (const float*)R.out_u,
              (const float*)R.out_v, (const float*)R.out_w, open_top_, &stats_->div_after_bits);
  CmStats st;
  std::vector<double> part(2 * kMeasureBlocks);
  HIPCHK(hipMemcpyAsync(&st, stats_, sizeof(CmStats), hipMemcpyDeviceToHost, s));
  HIPCHK(hipMemcpyAsync(part.data(), partials_, part.size() * 8, hipMemcpyDeviceToHost, s));
  HIPCHK(hipStreamSynchronize(s));
  HIPCHK(hipGetLastError());
  if (rep) {
    std::memset(rep, 0, sizeof(*rep));
    double rr = 0.0, bb = 0.0;
    for (int k = 0; k < kMeasureBlocks; ++k) {
      rr += part[2 * k];
      bb += part[2 * k + 1];
    }
    float lcp, cres, db, da;
    std::memcpy(&lcp, &st.lcp_residual_bits, 4);
    std::memcpy(&cres, &st.coarse_residual_bits, 4);
    std::memcpy(&db, &st.div_before_bits, 4);
    std::memcpy(&da, &st.div_after_bits, 4);
    rep->iterations = full + vcyc;
    rep->outer_iterations = 0;
    rep->levels = L;
    rep->relative_residual = bb > 0.0 ? std::sqrt(rr / bb) : 0.0;
    rep->rhs_norm = std::sqrt(bb);
    rep->max_div_before = db;
    rep->max_div_after = (R.out_u && R.out_v && R.out_w) ? (double)da : std::nan("");
    rep->lcp_residual = lcp;
    rep->coarse_sweeps = st.coarse_sweeps;
    rep->coarse_failures = st.coarse_failed;
    if (st.coarse_failed > 0) rep->flags |= FP_FLAG_NONCONVERGENCE;
    if (!std::isfinite(lcp) || !std::isfinite(rep->relative_residual)) rep->flags |= FP_FLAG_NONFINITE;
    rep->samples = (int64_t)nx_ * ny_ * nz_;
    rep->liquid_samples = st.liquid;
    (void)cres;
  }
  const double ms = std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
  if (rep) rep->device_ms = ms;
  return FP_OK;
}

}  // namespace fp

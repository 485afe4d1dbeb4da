// fp_advect.hip -- velocity advection and body forces of a uniform grid on MI355X.
//
// Kernels restate lib/methods/uniform/webgpu-uniform-reference.wgsl.ts (cited
// per function) for box containers without solids, inflow or surface tension.
// One thread per cell advances the cell's three positive faces; each face's
// characteristic is an RK2 trace through the transported (extrapolated)
// field with trilinear samples in D4 corner order.  The face arrays keep this
// library's layout (z fastest, u (nx+1,ny,nz) ...): the reference's padded
// transport shell is the same data with the outside read as 0.  No
// contraction: results equal oracle/fp_oracle_advect.c bit for bit.
#pragma clang fp contract(off)

#include "fp_advect.hpp"
#include "fp_extrap.hpp"
#include "fp_uniform.hpp"

#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstring>

namespace fp {

namespace {

constexpr int kThreads = 256;

struct AdGeo {
  int d[3];
  float h, inv_h;  // cell size and its correctly rounded reciprocal
  float far;       // below it a quotient by h is far from overflow (div_h)
  int open_top;
  int no_slip;
  float dt, gravity, nu;
};

constexpr float kTinyCell = 1e-22f;  // smaller cells divide (div_h)

struct Faces {
  const float* f[3];
};
struct FacesOut {
  float* f[3];
};

// v clamped into [lo, hi] (lo < hi) in one instruction.  For finite v this
// equals v < lo ? lo : (v > hi ? hi : v) up to the sign of a zero result;
// positions are only ever used as p - off with off >= 1/2, or compared, so
// that sign never reaches a result.
__device__ __forceinline__ float med3(float v, float lo, float hi) { return __builtin_amdgcn_fmed3f(v, lo, hi); }

// a * b for a, b < 2^24 and a product below 2^32: one full-rate 24-bit
// multiply (written out: the compiler keeps a quarter-rate 32-bit multiply
// when the operands' ranges are not visible inside the trace loop)
__device__ __forceinline__ unsigned mul24(unsigned a, unsigned b) {
  unsigned r;
  asm("v_mul_u32_u24 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
  return r;
}

// Two neighbouring faces of a row in one load (a vector: two floats would be
// loaded one by one where both are used apart).
typedef float Pair __attribute__((ext_vector_type(2), aligned(4)));
__device__ __forceinline__ Pair pair_at(const float* base, unsigned byte) {
  return *reinterpret_cast<const Pair*>(reinterpret_cast<const char*>(base) + byte);
}

// face (x, y, z) of component c (fewer than 2^24 rows and 2^30 faces per
// component, checked at set-up)
__device__ __forceinline__ unsigned fidx(const AdGeo& g, int c, int x, int y, int z) {
  const unsigned ey = g.d[1] + (c == 1), ez = g.d[2] + (c == 2);
  return mul24(mul24((unsigned)x, ey) + (unsigned)y, ez) + (unsigned)z;
}

// x / h, correctly rounded, from the reciprocal: two residual steps
// (Markstein 1990: the first quotient is within 1.5 ulp, the second faithful,
// the third rounded as the division) in five full-rate operations, where the
// division takes eleven and a quarter-rate reciprocal, 21 times a cell and
// step.  A residual, 2^-48 of x, underflows for quotients below 2^-101 / h: with
// h of kTinyCell or more those never reach a position of 1/2 or more, and zero
// keeps its value, not its sign (subtracted or compared only).  For |x| < g.far:
// beyond it a quotient may overflow.
__device__ __forceinline__ float div_h(const AdGeo& g, float x) {
  const float q0 = x * g.inv_h;
  const float q1 = __builtin_fmaf(__builtin_fmaf(-q0, g.h, x), g.inv_h, q0);
  return __builtin_fmaf(__builtin_fmaf(-q1, g.h, x), g.inv_h, q1);
}
// every x / h; where a lane has one of g.far or more the wave divides (a NaN
// stays one either way)
template <int N>
__device__ __forceinline__ void div_h_all(const AdGeo& g, float* x) {
  float big = 0.0f;
#pragma unroll
  for (int i = 0; i < N; ++i) big = fmaxf(big, fabsf(x[i]));
  if (__any(!(big < g.far))) {
#pragma unroll
    for (int i = 0; i < N; ++i) x[i] = x[i] / g.h;
  } else {
#pragma unroll
    for (int i = 0; i < N; ++i) x[i] = div_h(g, x[i]);
  }
}

// d4Sum8 (…wgsl.ts:103-106) of the weighted corners; with bounds also the
// range of the donors (boundedMacCormack, …wgsl.ts:963-991): the corners that
// carry weight, a corner below the domain along c (low) counting as 0
// (sampledFaceVelocity, :247-250; the sample reads the wall face there).  A
// corner past the top of an axis has no weight.
template <bool BOUNDS>
__device__ __forceinline__ float corner_sum(const float* fr, const float* vals, int c, bool low, float* range) {
  float terms[8];
  float lower = 1e30f, upper = -1e30f;
#pragma unroll
  for (int corner = 0; corner < 8; ++corner) {
    const int o[3] = {corner & 1, corner >> 1 & 1, corner >> 2 & 1};
    float w[3];
#pragma unroll
    for (int a = 0; a < 3; ++a) w[a] = o[a] ? fr[a] : 1.0f - fr[a];
    const float weight = w[0] * w[1] * w[2];
    terms[corner] = weight * vals[corner];
    if constexpr (BOUNDS) {
      const float value = low && !o[c] ? 0.0f : vals[corner];
      if (weight > 0.0f) {
        lower = value < lower ? value : lower;
        upper = value > upper ? value : upper;
      }
    }
  }
  if constexpr (BOUNDS) {
    range[0] = lower;
    range[1] = upper;
  }
  const float y0 = (terms[0] + terms[5]) + (terms[1] + terms[4]);
  const float y1 = (terms[2] + terms[7]) + (terms[3] + terms[6]);
  return y0 + y1;
}

// Where the points of a wave lie: INSIDE, at least half a cell from every
// wall, no sample of theirs is clamped or reads past an array; ZEDGE, that
// holds along x and y; EDGE otherwise.  INSIDE takes 51 instructions a sample
// and EDGE 90 (clamps, selects, and an address per row); a row's last cell is
// in every sixth wave at nz = 384 and in every other at 128, so the z edge has
// a path of its own (62).
enum Where { INSIDE, ZEDGE, EDGE };
__device__ __forceinline__ Where where_are(const AdGeo& g, const float (*p)[3]) {
  bool xy = true, z = true;
#pragma unroll
  for (int f = 0; f < 3; ++f) {
    xy = xy && p[f][0] >= 0.5f && p[f][0] < (float)g.d[0] - 0.5f && p[f][1] >= 0.5f && p[f][1] < (float)g.d[1] - 0.5f;
    z = z && p[f][2] >= 0.5f && p[f][2] < (float)g.d[2] - 0.5f;
  }
  if (!__all(xy)) return EDGE;
  return __all(z) ? INSIDE : ZEDGE;
}

// sampleVelocityComponent (…wgsl.ts:261-270)
template <Where W, bool BOUNDS = false>
__device__ __forceinline__ float sample_comp(const AdGeo& g, const Faces& t, const float* p, int c,
                                             float* range = nullptr) {
  float q[3];
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    const float off = a == c ? 1.0f : 0.5f, lo = a == c ? -1.0f : 0.0f, hi = (float)(g.d[a] - 1);
    const float v = p[a] - off;
    q[a] = W == EDGE || (W == ZEDGE && a == 2) ? med3(v, lo, hi) : v;
  }
  int b[3];
  float fr[3];
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    const float f = floorf(q[a]);
    b[a] = (int)f;
    // q lies in [lo, hi], so this clamp changes nothing; it keeps the
    // indices below inside the arrays whatever the input
    if (W == EDGE || (W == ZEDGE && a == 2)) b[a] = min(max(b[a], a == c ? -1 : 0), g.d[a] - 1);
    fr[a] = q[a] - f;
  }
  // All eight corners' values first, then the weights.  Corner o is face
  // array element e = b + o (+1 along c): e >= 0 always, and only an o = 1
  // corner at the top of an axis lies past the array (it reads 0, as the
  // reference's padded shell does; its weight is 0).  Corners k and k + 4
  // differ only in z and come from one 8-byte load at a row index clamped so
  // that both words lie in the row (every row holds at least 2 faces: grids
  // are at least 2 cells on each axis).  Byte offsets fit 32 bits (fewer than
  // 2^30 faces per component), so the loads take a scalar base.
  const int ex = g.d[0] + (c == 0), ey = g.d[1] + (c == 1), ez = g.d[2] + (c == 2);
  const int ix0 = b[0] + (c == 0), iy0 = b[1] + (c == 1), iz0 = b[2] + (c == 2);
  const bool topz = W != INSIDE && iz0 > ez - 2;
  const int zb = W != INSIDE ? min(iz0, ez - 2) : iz0;
  const float* base = t.f[c];
  Pair pair[4];
  bool inx1 = true, iny1 = true;
  if constexpr (W == EDGE) {
    inx1 = ix0 + 1 < ex;
    iny1 = iy0 + 1 < ey;
    const int ix1 = min(ix0 + 1, ex - 1), iy1 = min(iy0 + 1, ey - 1);
    // (24-bit multiplies: fewer than 2^24 rows per component)
    const unsigned r0 = mul24((unsigned)ix0, (unsigned)ey), r1 = mul24((unsigned)ix1, (unsigned)ey);
    const unsigned rows[4] = {r0 + iy0, r1 + iy0, r0 + iy1, r1 + iy1};
#pragma unroll
    for (int k = 0; k < 4; ++k)
      pair[k] = pair_at(base, (mul24(rows[k], (unsigned)ez) + (unsigned)zb) << 2);
  } else {
    // one offset per sample: the rows beside it are scalar bases of their own
    const unsigned at = (mul24(mul24((unsigned)ix0, (unsigned)ey) + (unsigned)iy0, (unsigned)ez) + (unsigned)zb) << 2;
    const size_t dy = (size_t)ez, dx = (size_t)ey * dy;
    pair[0] = pair_at(base, at);
    pair[1] = pair_at(base + dx, at);
    pair[2] = pair_at(base + dy, at);
    pair[3] = pair_at(base + dx + dy, at);
  }
  float vals[8];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const bool in = ((k & 1) == 0 || inx1) && ((k & 2) == 0 || iny1);
    vals[k] = in ? (topz ? pair[k].y : pair[k].x) : 0.0f;
    vals[k + 4] = in && !topz ? pair[k].y : 0.0f;
  }
  return corner_sum<BOUNDS>(fr, vals, c, b[c] < 0, range);
}

// The samples of every component at three points, all their loads in flight
// together.
template <Where W>
__device__ __forceinline__ void sample9(const AdGeo& g, const Faces& t, const float (*p)[3], float (*out)[3]) {
#pragma unroll
  for (int f = 0; f < 3; ++f)
#pragma unroll
    for (int c = 0; c < 3; ++c) out[f][c] = sample_comp<W>(g, t, p[f], c);
}
__device__ __forceinline__ void sample_all(const AdGeo& g, const Faces& t, const float (*p)[3], float (*out)[3]) {
  switch (where_are(g, p)) {
    case INSIDE: sample9<INSIDE>(g, t, p, out); break;
    case ZEDGE: sample9<ZEDGE>(g, t, p, out); break;
    default: sample9<EDGE>(g, t, p, out);
  }
}

// The samples of the first stage, at the three positive faces of cell (x, y,
// z) themselves: a face's own component is one array element (its other
// corners have no weight) and each other component the mean of four (of two at
// the top of the face's axis).  The 20 loads cover all corners of the nine
// samples, the ones without weight too: 0 times an infinity is not 0, so where
// any of them is not finite the samples are made in full.  Nine samples are 36
// loads and 460 to 810 instructions, this is 20 and 150.
__device__ __forceinline__ bool first_samples(const AdGeo& g, const Faces& t, int x, int y, int z, float (*out)[3]) {
  const int p[3] = {x, y, z};
  bool up[3];  // a cell above along the axis
#pragma unroll
  for (int a = 0; a < 3; ++a) up[a] = p[a] + 1 < g.d[a];
  // weights of the lower and upper corner along an axis of the face's own
  float wl[3], wh[3];
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    wl[a] = up[a] ? 0.5f : 1.0f;
    wh[a] = up[a] ? 0.5f : 0.0f;
  }
  unsigned worst = 0;
  auto seen = [&](float v) {
    const unsigned m = __float_as_uint(v) & 0x7fffffffu;
    worst = m > worst ? m : worst;
  };
  auto row = [&](int c, int X, int Y) {
    return mul24(mul24((unsigned)X, (unsigned)(g.d[1] + (c == 1))) + (unsigned)Y, (unsigned)(g.d[2] + (c == 2)));
  };
  // u: three along x, two along y and z; v: three along y
  float u[3][2][2], v[2][3][2], w[2][2][3];
  const int x1 = x + (up[0] ? 1 : 0), y1 = y + (up[1] ? 1 : 0), z1 = z + (up[2] ? 1 : 0);
  const unsigned zb = (unsigned)min(z, g.d[2] - 2);
  auto row_pair = [&](int c, int X, int Y, float* o) {
    const Pair f = pair_at(t.f[c], (row(c, X, Y) + zb) << 2);
    o[0] = up[2] ? f.x : f.y;
    o[1] = f.y;  // at the top of z: the row's last face again, without weight
  };
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) row_pair(0, i < 2 ? x + i : x1 + 1, j ? y1 : y, u[i][j]);
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 3; ++j) row_pair(1, i ? x1 : x, j < 2 ? y + j : y1 + 1, v[i][j]);
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const unsigned r = row(2, i ? x1 : x, j ? y1 : y);
      const Pair f = pair_at(t.f[2], (r + (unsigned)z) << 2);
      w[i][j][0] = f.x;
      w[i][j][1] = f.y;
      w[i][j][2] = t.f[2][r + (unsigned)(z1 + 1)];
    }
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        seen(u[i][j][k]);
        seen(v[j][i][k]);
        seen(w[j][k][i]);
      }
  // terms in corner_sum's order; the absent corners add zeros
  auto mean = [](float a, float wa, float b, float wb, float c, float wc, float d, float wd) {
    return (wa * a + wb * b) + (wc * c + wd * d);
  };
  out[0][0] = u[1][0][0];
  out[1][1] = v[0][1][0];
  out[2][2] = w[0][0][1];
  // component c at face f: weights 1/2 along c, wl and wh along f
  out[0][1] = mean(v[0][0][0], wl[0] * 0.5f, v[1][0][0], wh[0] * 0.5f, v[0][1][0], wl[0] * 0.5f, v[1][1][0],
                   wh[0] * 0.5f);
  out[0][2] = mean(w[0][0][0], wl[0] * 0.5f, w[1][0][1], wh[0] * 0.5f, w[1][0][0], wh[0] * 0.5f, w[0][0][1],
                   wl[0] * 0.5f);
  out[1][0] = mean(u[0][0][0], 0.5f * wl[1], u[1][0][0], 0.5f * wl[1], u[0][1][0], 0.5f * wh[1], u[1][1][0],
                   0.5f * wh[1]);
  out[1][2] = mean(w[0][0][0], wl[1] * 0.5f, w[0][0][1], wl[1] * 0.5f, w[0][1][0], wh[1] * 0.5f, w[0][1][1],
                   wh[1] * 0.5f);
  out[2][0] = mean(u[0][0][0], 0.5f * wl[2], u[1][0][1], 0.5f * wh[2], u[1][0][0], 0.5f * wl[2], u[0][0][1],
                   0.5f * wh[2]);
  out[2][1] = mean(v[0][0][0], 0.5f * wl[2], v[0][0][1], 0.5f * wh[2], v[0][1][0], 0.5f * wl[2], v[0][1][1],
                   0.5f * wh[2]);
  return worst < 0x7f800000u;
}

// clampVelocityTraceToDomain (…wgsl.ts:317-322)
__device__ __forceinline__ void clamp_trace(const AdGeo& g, float* q) {
  q[0] = med3(q[0], 0.0f, (float)g.d[0]);
  q[2] = med3(q[2], 0.0f, (float)g.d[2]);
  q[1] = g.open_top ? fmaxf(q[1], 0.0f) : med3(q[1], 0.0f, (float)g.d[1]);
}

__device__ __forceinline__ void face_position(int x, int y, int z, int c, float* pos) {
  pos[0] = (float)x + 0.5f;
  pos[1] = (float)y + 0.5f;
  pos[2] = (float)z + 0.5f;
  pos[c] = (float)(c == 0 ? x : c == 1 ? y : z) + 1.0f;
}

// departurePoint (…wgsl.ts:324-334), RK2 in pieces of at most 1.5 cells, for
// the cell's three faces at once: the same operations per face, the three
// traces advanced together (a finished trace keeps its point), so each round
// of samples serves three faces
__device__ __forceinline__ void departure3(const AdGeo& g, const Faces& t, int x, int y, int z, float dt,
                                           float (*point)[3]) {
  float remaining[3];
#pragma unroll
  for (int f = 0; f < 3; ++f) {
    face_position(x, y, z, f, point[f]);
    remaining[f] = fabsf(dt);
  }
  const float direction = dt >= 0.0f ? 1.0f : -1.0f;
  for (int step = 0; step < 32; ++step) {
    bool live[3];
#pragma unroll
    for (int f = 0; f < 3; ++f) live[f] = !(remaining[f] <= 1e-7f);
    if (!live[0] && !live[1] && !live[2]) break;
    float first[3][3];
    bool made = false;
    if (step == 0) made = __all(first_samples(g, t, x, y, z, first));
    if (!made) sample_all(g, t, point, first);
    float mid[3][3], rate[3], step_s[3], signed_step[3], q[9];
    bool pieces = false;
#pragma unroll
    for (int f = 0; f < 3; ++f) {
      // max(|u|/h, |v|/h, |w|/h) as max(|u|, |v|, |w|)/h: a correctly rounded
      // division by h > 0 is monotonic, so both pick the same value
      const float ax = fabsf(first[f][0]), ay = fabsf(first[f][1]), az = fabsf(first[f][2]);
      const float myz = ay > az ? ay : az;
      rate[f] = ax > myz ? ax : myz;
    }
    div_h_all<3>(g, rate);
#pragma unroll
    for (int f = 0; f < 3; ++f) {
      rate[f] = rate[f] > 1e-6f ? rate[f] : 1e-6f;
      step_s[f] = remaining[f];
      pieces = pieces || rate[f] * remaining[f] >= 1.49f;
    }
    // a step of less than 1.49 cells is one piece (below 1.5 / rate however
    // the products round): the limit's division only where a lane has more
    if (__any(pieces)) {
#pragma unroll
      for (int f = 0; f < 3; ++f) {
        const float lim = 1.5f / rate[f];
        step_s[f] = remaining[f] < lim ? remaining[f] : lim;
      }
    }
#pragma unroll
    for (int f = 0; f < 3; ++f) {
      signed_step[f] = direction * step_s[f];
#pragma unroll
      for (int a = 0; a < 3; ++a) q[3 * f + a] = 0.5f * first[f][a] * signed_step[f];
    }
    div_h_all<9>(g, q);
#pragma unroll
    for (int f = 0; f < 3; ++f) {
#pragma unroll
      for (int a = 0; a < 3; ++a) mid[f][a] = point[f][a] - q[3 * f + a];
      clamp_trace(g, mid[f]);
    }
    float second[3][3];
    sample_all(g, t, mid, second);
#pragma unroll
    for (int f = 0; f < 3; ++f)
#pragma unroll
      for (int a = 0; a < 3; ++a) q[3 * f + a] = second[f][a] * signed_step[f];
    div_h_all<9>(g, q);
#pragma unroll
    for (int f = 0; f < 3; ++f) {
      float next[3];
#pragma unroll
      for (int a = 0; a < 3; ++a) next[a] = point[f][a] - q[3 * f + a];
      clamp_trace(g, next);
#pragma unroll
      for (int a = 0; a < 3; ++a) point[f][a] = live[f] ? next[a] : point[f][a];
      remaining[f] = live[f] ? remaining[f] - step_s[f] : remaining[f];
    }
  }
}

// each face's own component at its point
template <Where W, bool BOUNDS>
__device__ __forceinline__ void sample_own(const AdGeo& g, const Faces& t, const float (*p)[3], float* val,
                                           float (*range)[2]) {
#pragma unroll
  for (int c = 0; c < 3; ++c) val[c] = sample_comp<W, BOUNDS>(g, t, p[c], c, range[c]);
}

// advectVelocityComponent (…wgsl.ts:415-423) without solids or the
// liquid-only toggle, for the three faces of cell (x,y,z) together; with BOUNDS
// also the range of each face's donors at its departure point
template <bool BOUNDS>
__device__ __forceinline__ void advect3(const AdGeo& g, const Faces& t, int x, int y, int z, float dt, float* val,
                                        float (*range)[2]) {
  float dep[3][3];
  departure3(g, t, x, y, z, dt, dep);
  switch (where_are(g, dep)) {
    case INSIDE: sample_own<INSIDE, BOUNDS>(g, t, dep, val, range); break;
    case ZEDGE: sample_own<ZEDGE, BOUNDS>(g, t, dep, val, range); break;
    default: sample_own<EDGE, BOUNDS>(g, t, dep, val, range);
  }
}

__device__ __forceinline__ float occupancy(const AdGeo& g, const float* phi, const float* dens, int x, int y, int z) {
  if (x < 0 || y < 0 || z < 0 || x >= g.d[0] || y >= g.d[1] || z >= g.d[2]) return 0.0f;
  const unsigned i = mul24(mul24((unsigned)x, (unsigned)g.d[1]) + (unsigned)y, (unsigned)g.d[2]) + (unsigned)z;
  const float v = phi ? 0.5f - phi[i] / (4.0f * g.h) : dens[i];
  return v < 0.0f ? 0.0f : (v > 1.0f ? 1.0f : v);
}

// diffusionVelocity (…wgsl.ts:860): the cell's positive faces, clamped into
// the domain, reflected outside it for no-slip walls
__device__ __forceinline__ void diff_vel(const AdGeo& g, const Faces& cur, int x, int y, int z, float* out) {
  const bool inside = x >= 0 && y >= 0 && z >= 0 && x < g.d[0] && y < g.d[1] && z < g.d[2];
  const int cx = min(max(x, 0), g.d[0] - 1), cy = min(max(y, 0), g.d[1] - 1), cz = min(max(z, 0), g.d[2] - 1);
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    const float v = cur.f[c][fidx(g, c, cx + (c == 0), cy + (c == 1), cz + (c == 2))];
    out[c] = g.no_slip && !inside ? -v : v;
  }
}

// applyVelocityForces (…wgsl.ts:872-915) without surface tension or inflow
__device__ void forces(const AdGeo& g, const Faces& cur, const float* phi, const float* dens, int x, int y, int z,
                       float* v) {
  const float occ = occupancy(g, phi, dens, x, y, z);
  if (occ > 0.0f && g.nu > 0.0f) {
    float ce[3], xp[3], xm[3], yp[3], ym[3], zp[3], zm[3];
    diff_vel(g, cur, x, y, z, ce);
    diff_vel(g, cur, x + 1, y, z, xp);
    diff_vel(g, cur, x - 1, y, z, xm);
    diff_vel(g, cur, x, y + 1, z, yp);
    diff_vel(g, cur, x, y - 1, z, ym);
    diff_vel(g, cur, x, y, z + 1, zp);
    diff_vel(g, cur, x, y, z - 1, zm);
    const float h2 = g.h * g.h;
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      const float lap = ((xp[c] - 2.0f * ce[c] + xm[c]) / h2 + (yp[c] - 2.0f * ce[c] + ym[c]) / h2) +
                        (zp[c] - 2.0f * ce[c] + zm[c]) / h2;
      v[c] += g.dt * g.nu * lap;
    }
  }
  const float occ_y = occupancy(g, phi, dens, x, y + 1, z);
  if (occ > 1e-5f || occ_y > 1e-5f) v[1] += g.gravity * g.dt;
}

__device__ __forceinline__ bool cell_of(const AdGeo& g, int& x, int& y, int& z) {
  const unsigned i = blockIdx.x * kThreads + threadIdx.x;
  const unsigned n = (unsigned)g.d[0] * g.d[1] * g.d[2];
  if (i >= n) return false;
  z = (int)(i % (unsigned)g.d[2]);
  const unsigned t = i / (unsigned)g.d[2];
  y = (int)(t % (unsigned)g.d[1]);
  x = (int)(t / (unsigned)g.d[1]);
  return true;
}

// the negative domain faces carry over (carryBoundaryVelocity, …wgsl.ts:196)
__device__ __forceinline__ void carry_walls(const AdGeo& g, const Faces& cur, float* const* out, int x, int y, int z) {
  if (x == 0) out[0][fidx(g, 0, 0, y, z)] = cur.f[0][fidx(g, 0, 0, y, z)];
  if (y == 0) out[1][fidx(g, 1, x, 0, z)] = cur.f[1][fidx(g, 1, x, 0, z)];
  if (z == 0) out[2][fidx(g, 2, x, y, 0)] = cur.f[2][fidx(g, 2, x, y, 0)];
}

// The traces are bound by the samples' instructions and loads (four waves a
// SIMD: 128 registers; at three 2.60 ms for the 384^3 pass of a flow of one to
// three pieces, at five the same, at six, with spills, 2.45): 3.02 -> 2.28 ms with
// the paths by position, the first stage's few corners and the divisions by h
// as products; 1 TB/s of inputs and outputs (a block order by XCD: 2.35 ms).

// semiLagrangianAdvection (…wgsl.ts:922-936)
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(4, 4))) void k_adv_sl(
    AdGeo g, Faces t, Faces cur, const float* __restrict__ phi, const float* __restrict__ dens, float* uo, float* vo,
    float* wo) {
  int x, y, z;
  if (!cell_of(g, x, y, z)) return;
  float* out[3] = {uo, vo, wo};
  const int p[3] = {x, y, z};
  float val[3], unused[3][2];
  advect3<false>(g, t, x, y, z, g.dt, val, unused);
  for (int c = 0; c < 3; ++c) {
    if (p[c] == g.d[c] - 1 && !(c == 1 && g.open_top)) {
      const float old = cur.f[c][fidx(g, c, x + (c == 0), y + (c == 1), z + (c == 2))];
      val[c] = val[c] < old ? val[c] : old;
    }
  }
  forces(g, cur, phi, dens, x, y, z, val);
  for (int c = 0; c < 3; ++c) out[c][fidx(g, c, x + (c == 0), y + (c == 1), z + (c == 2))] = val[c];
  carry_walls(g, cur, out, x, y, z);
}

// advect (prediction, …wgsl.ts:938-952): the wall faces keep the field the
// trace starts from.  The donors' range at the departure point, which the
// correction limits to, is made here, where the corners are in registers: 24
// bytes a cell written and read instead of the same trace again.
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(4, 4))) void k_adv_predict(
    AdGeo g, Faces t, Faces walls, float* uo, float* vo, float* wo, FacesOut lower, FacesOut upper) {
  int x, y, z;
  if (!cell_of(g, x, y, z)) return;
  float* out[3] = {uo, vo, wo};
  const int p[3] = {x, y, z};
  float adv[3], range[3][2];
  advect3<true>(g, t, x, y, z, g.dt, adv, range);
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    const unsigned fi = fidx(g, c, x + (c == 0), y + (c == 1), z + (c == 2));
    float val = adv[c];
    if (p[c] == g.d[c] - 1 && !(c == 1 && g.open_top)) val = walls.f[c][fi];
    out[c][fi] = val;
    lower.f[c][fi] = range[c][0];
    upper.f[c][fi] = range[c][1];
  }
  carry_walls(g, walls, out, x, y, z);
}

// reverseAdvection (…wgsl.ts:954-961) through the prediction's extrapolation
// te, correctAdvection (:993-1004) with boundedMacCormack (:963-991) and the
// forces in one pass: a face's correction needs the reverse trace of that face
// only.  160 x 117 x 143 in MacCormack with its extrapolations: 1.18 ->
// 0.98 ms with one forward trace instead of two and no field of reversed or
// corrected faces.
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(4, 4))) void k_adv_correct(
    AdGeo g, Faces te, Faces cur, Faces pred, Faces lower, Faces upper, const float* __restrict__ phi,
    const float* __restrict__ dens, float* uo, float* vo, float* wo) {
  int x, y, z;
  if (!cell_of(g, x, y, z)) return;
  float* out[3] = {uo, vo, wo};
  const int p[3] = {x, y, z};
  float val[3], rev[3], unused[3][2];
  advect3<false>(g, te, x, y, z, -g.dt, rev, unused);
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    const unsigned fi = fidx(g, c, x + (c == 0), y + (c == 1), z + (c == 2));
    const float predicted = pred.f[c][fi];
    const float reversed = p[c] == g.d[c] - 1 && !(c == 1 && g.open_top) ? predicted : rev[c];
    const float corrected = predicted + 0.5f * (cur.f[c][fi] - reversed);
    const bool revert = corrected < lower.f[c][fi] || corrected > upper.f[c][fi];
    val[c] = revert ? predicted : corrected;
  }
  forces(g, cur, phi, dens, x, y, z, val);
  for (int c = 0; c < 3; ++c) out[c][fidx(g, c, x + (c == 0), y + (c == 1), z + (c == 2))] = val[c];
  carry_walls(g, cur, out, x, y, z);
}

}  // namespace

Advector::~Advector() {
  for (void* p : allocations_) (void)hipFree(p);
}

int Advector::alloc(void** p, size_t bytes) {
  bytes = (bytes + 255) & ~(size_t)255;
  if (hipMalloc(p, bytes) != hipSuccess) {
    set_error("velocity advection: hipMalloc(%zu) failed", bytes);
    return FP_ERR_OUT_OF_MEMORY;
  }
  allocations_.push_back(*p);
  bytes_ += bytes;
  return FP_OK;
}

size_t Advector::estimate_bytes(int nx, int ny, int nz) {
  const size_t faces = (size_t)(nx + 1) * ny * nz + (size_t)nx * (ny + 1) * nz + (size_t)nx * ny * (nz + 1);
  return 5 * ((faces * 4 + 255) & ~(size_t)255);
}

int Advector::create(int nx, int ny, int nz, double h) {
  // the paired z loads need 2 faces per row; byte offsets of 32 bits
  if (nx < 2 || ny < 2 || nz < 2) return FP_ERR_UNSUPPORTED;
  const size_t most = (size_t)(std::max(nx, std::max(ny, nz)) + 1) * nx * ny * nz / std::min(nx, std::min(ny, nz));
  if (most >= ((size_t)1 << 30) || (size_t)(nx + 1) * (ny + 1) >= ((size_t)1 << 24)) {
    set_error("velocity advection: %d x %d x %d has 2^30 or more faces or 2^24 or more rows per component", nx, ny,
              nz);
    return FP_ERR_UNSUPPORTED;
  }
  d_[0] = nx;
  d_[1] = ny;
  d_[2] = nz;
  h_ = (float)h;
  nf_[0] = (size_t)(nx + 1) * ny * nz;
  nf_[1] = (size_t)nx * (ny + 1) * nz;
  nf_[2] = (size_t)nx * ny * (nz + 1);
  const size_t faces = nf_[0] + nf_[1] + nf_[2];
  int rc;
  if ((rc = alloc((void**)&transport_, faces * 4))) return rc;
  if ((rc = alloc((void**)&pred_, faces * 4))) return rc;
  if ((rc = alloc((void**)&lower_, faces * 4))) return rc;
  if ((rc = alloc((void**)&upper_, faces * 4))) return rc;
  if ((rc = alloc((void**)&out_, faces * 4))) return rc;
  return FP_OK;
}

int Advector::stage_host(size_t floats) {
  if (host_floats_ >= floats) return FP_OK;
  int rc = alloc((void**)&host_, floats * 4);
  if (!rc) host_floats_ = floats;
  return rc;
}

int Advector::run(hipStream_t s, Extrapolator* ex, const fp_advect_args* a, fp_advect_report* rep) {
  const auto t0 = std::chrono::steady_clock::now();
  const int nx = d_[0], ny = d_[1], nz = d_[2];
  const size_t n = (size_t)nx * ny * nz;
  const bool host = a->memory == FP_MEMORY_HOST;
  const float* field = a->phi ? a->phi : a->density;
  const float* cur_in[3] = {a->u, a->v, a->w};
  const float* tr_in[3] = {a->tu, a->tv, a->tw};
  const bool have_transport = a->tu && a->tv && a->tw;
  // inputs on the device
  const float* f = field;
  const float* cur[3] = {cur_in[0], cur_in[1], cur_in[2]};
  const float* tr[3] = {tr_in[0], tr_in[1], tr_in[2]};
  if (host) {
    const size_t need = n + 2 * (nf_[0] + nf_[1] + nf_[2]);
    int rc = stage_host(need);
    if (rc) return rc;
    float* p = host_;
    HIPCHK(hipMemcpyAsync(p, field, n * 4, hipMemcpyHostToDevice, s));
    f = p;
    p += n;
    for (int c = 0; c < 3; ++c) {
      HIPCHK(hipMemcpyAsync(p, cur_in[c], nf_[c] * 4, hipMemcpyHostToDevice, s));
      cur[c] = p;
      p += nf_[c];
    }
    for (int c = 0; c < 3; ++c) {
      if (have_transport) HIPCHK(hipMemcpyAsync(p, tr_in[c], nf_[c] * 4, hipMemcpyHostToDevice, s));
      tr[c] = p;
      p += nf_[c];
    }
  }
  float* split[4][3];
  float* bases[4] = {transport_, pred_, lower_, upper_};
  for (int k = 0; k < 4; ++k) {
    split[k][0] = bases[k];
    split[k][1] = bases[k] + nf_[0];
    split[k][2] = bases[k] + nf_[0] + nf_[1];
  }
  const int open_top = a->open_top ? 1 : 0;
  if (!have_transport) {
    fp_extrapolate_args e;
    std::memset(&e, 0, sizeof(e));
    e.memory = FP_MEMORY_DEVICE;
    e.open_top = open_top;
    e.phi = a->phi ? f : nullptr;
    e.density = a->phi ? nullptr : f;
    e.u = cur[0];
    e.v = cur[1];
    e.w = cur[2];
    e.u_out = split[0][0];
    e.v_out = split[0][1];
    e.w_out = split[0][2];
    int rc = ex->run(s, &e, nullptr);
    if (rc) return rc;
    for (int c = 0; c < 3; ++c) tr[c] = split[0][c];
  }
  // outputs: written directly unless host memory or an overlap with an input
  float* out[3] = {a->u_out, a->v_out, a->w_out};
  float* dst[3];
  float* stage[3] = {out_, out_ + nf_[0], out_ + nf_[0] + nf_[1]};
  for (int c = 0; c < 3; ++c) {
    bool overlaps = host;
    const size_t ob = nf_[c] * 4;
    const void* ins[7] = {field, cur_in[0], cur_in[1], cur_in[2], tr_in[0], tr_in[1], tr_in[2]};
    const size_t ib[7] = {n * 4, nf_[0] * 4, nf_[1] * 4, nf_[2] * 4, nf_[0] * 4, nf_[1] * 4, nf_[2] * 4};
    for (int k = 0; k < 7 && !overlaps; ++k) {
      if (!ins[k]) continue;
      const char *o0 = (const char*)out[c], *i0 = (const char*)ins[k];
      overlaps = o0 < i0 + ib[k] && i0 < o0 + ob;
    }
    dst[c] = overlaps ? stage[c] : out[c];
  }
  AdGeo g;
  g.d[0] = nx;
  g.d[1] = ny;
  g.d[2] = nz;
  g.h = h_;
  g.inv_h = 1.0f / h_;
  g.far = h_ >= kTinyCell && std::isnormal(g.inv_h) ? std::min(1e38f * h_, 3e38f) : 0.0f;
  g.open_top = open_top;
  g.no_slip = a->no_slip ? 1 : 0;
  g.dt = (float)a->dt;
  g.gravity = (float)a->gravity;
  g.nu = (float)a->viscosity;
  const Faces T{{tr[0], tr[1], tr[2]}}, C{{cur[0], cur[1], cur[2]}};
  const float* phi = a->phi ? f : nullptr;
  const float* dens = a->phi ? nullptr : f;
  const dim3 grid((unsigned)((n + kThreads - 1) / kThreads)), block(kThreads);
  if (a->scheme == FP_ADVECT_SEMI_LAGRANGIAN) {
    hipLaunchKernelGGL(k_adv_sl, grid, block, 0, s, g, T, C, phi, dens, dst[0], dst[1], dst[2]);
  } else {
    const Faces P{{split[1][0], split[1][1], split[1][2]}}, Lo{{split[2][0], split[2][1], split[2][2]}},
        Hi{{split[3][0], split[3][1], split[3][2]}};
    hipLaunchKernelGGL(k_adv_predict, grid, block, 0, s, g, T, C, split[1][0], split[1][1], split[1][2],
                       FacesOut{{split[2][0], split[2][1], split[2][2]}},
                       FacesOut{{split[3][0], split[3][1], split[3][2]}});
    // the transport is not read again: the prediction's extrapolation takes its place
    fp_extrapolate_args e;
    std::memset(&e, 0, sizeof(e));
    e.memory = FP_MEMORY_DEVICE;
    e.open_top = open_top;
    e.phi = phi;
    e.density = dens;
    e.u = split[1][0];
    e.v = split[1][1];
    e.w = split[1][2];
    e.u_out = split[0][0];
    e.v_out = split[0][1];
    e.w_out = split[0][2];
    // the same surface as the transport's extrapolation when this call made it
    int rc = ex->run(s, &e, nullptr, !have_transport);
    if (rc) return rc;
    const Faces PE{{split[0][0], split[0][1], split[0][2]}};
    hipLaunchKernelGGL(k_adv_correct, grid, block, 0, s, g, PE, C, P, Lo, Hi, phi, dens, dst[0], dst[1], dst[2]);
  }
  for (int c = 0; c < 3; ++c)
    if (dst[c] != out[c])
      HIPCHK(hipMemcpyAsync(out[c], dst[c], nf_[c] * 4, host ? hipMemcpyDeviceToHost : hipMemcpyDeviceToDevice, s));
  HIPCHK(hipStreamSynchronize(s));
  if (rep) {
    std::memset(rep, 0, sizeof(*rep));
    rep->device_ms = std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
  }
  return FP_OK;
}

}  // namespace fp

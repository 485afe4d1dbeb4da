// fp_leg.hpp -- one leg of the V-cycle on a cache-resident level as one launch.
//
// On levels of up to about a million cells (leg_cells) a column march
// (fp_sweep.hpp, fp_march.hpp) is bound by the latency of its chain of plane
// steps and by the launches themselves: at 32^3 two pre-smoothing sweeps, the
// residual and the restriction take 8.1 + 8.7 + 7.6 + 6.7 us although the
// level's data sit in the caches.  Here a 1024-lane workgroup takes an 8 x 8 x
// 16 tile of cells with the ring that the whole leg reaches into, loads every
// coefficient it needs once into registers, and runs all of the leg's passes
// on it:
//
//   down   pre-smoothing sweeps from zero, residual, restriction of the
//          tile's coarse cells (ring 2 kLegSweeps + 1): 31 -> 13.7 us at 32^3,
//          17.6 us at 64^3
//   up     prolongation of the coarse correction, post-smoothing sweeps
//          (ring 2 kLegSweeps): 22 -> 13.6 us at 32^3, 17.4 us at 64^3
//
// A pass spoils one ring of the window's edge (it reads cells that the window
// does not hold), so values that are needed further in stay exact; nothing is
// tested per pass.  The redundant ring work (an 18 x 18 x 28 window for 1024
// cells) is the price of one launch instead of four, which is why the legs
// stop at leg_cells.  1024 lanes with five pairs each keep the window's
// coefficients in 128 registers; 512 lanes need 256 and spill.
//
// The two colours of the window live in LDS arrays of their own, indexed by
// (even z, odd z) pair: each pair holds one cell of each colour, so every
// neighbour of a cell is in the other array at the pair's index or one pair,
// row or plane beside it, and a wave's reads are contiguous.  Every update
// has the arithmetic of sweep3_body, OpResidualW, k_restrict_march and
// k_prolong_march in their order, so a leg gives the same bits as those
// launches.
#pragma once

#include "fp_march.hpp"
#include "fp_sweep.hpp"
#include "fp_uniform.hpp"

namespace fp {

constexpr int kLegThreads = 1024;
constexpr int kLegX = 8, kLegY = 8, kLegZ = 16;  // tile of fine cells
constexpr int kLegSweeps = 2;                    // most sweeps per side

// Window of a leg: ring HX in x and y, HZ (even) in z; slots of one (even z,
// odd z) pair per lane.
template <int HX, int HZ>
struct LegWindow {
  static constexpr int WX = kLegX + 2 * HX, WY = kLegY + 2 * HX, PZ = (kLegZ + 2 * HZ) / 2;
  static constexpr int ROW = PZ, PLANE = WY * PZ, NP = WX * PLANE;
  static constexpr int SLOTS = (NP + kLegThreads - 1) / kLegThreads;
  static constexpr int PAD = PLANE;  // neighbours of the window's edge read the padding
  static constexpr int LDS = NP + 2 * PAD;
};

// Coefficients of one cell: its packed record and the positive-face weights
// of its three negative neighbours.  Two-byte storage keeps them packed two to
// a register.
template <typename T, int N = sizeof(T)>
struct LegCell {
  float v[7];
  __device__ __forceinline__ void set(W4<T> w, T xm, T ym, T zm) {
    v[0] = wf(w.wx); v[1] = wf(w.wy); v[2] = wf(w.wz); v[3] = wf(w.id);
    v[4] = wf(xm); v[5] = wf(ym); v[6] = wf(zm);
  }
  template <int I> __device__ __forceinline__ float get() const { return v[I]; }
};
template <typename T>
struct LegCell<T, 2> {
  unsigned v[4];
  __device__ __forceinline__ void set(W4<T> w, T xm, T ym, T zm) {
    const fp_u32x2 b = __builtin_bit_cast(fp_u32x2, w);
    v[0] = b.x;
    v[1] = b.y;
    v[2] = (unsigned)__builtin_bit_cast(unsigned short, xm) | (unsigned)__builtin_bit_cast(unsigned short, ym) << 16;
    v[3] = (unsigned)__builtin_bit_cast(unsigned short, zm);
  }
  template <int I> __device__ __forceinline__ float get() const {
    const unsigned short h = (unsigned short)((I & 1) ? v[I / 2] >> 16 : v[I / 2] & 0xffffu);
    return wf(__builtin_bit_cast(T, h));
  }
};
// indices of LegCell::get
constexpr int kLegWX = 0, kLegWY = 1, kLegWZ = 2, kLegID = 3, kLegXM = 4, kLegYM = 5, kLegZM = 6;

template <typename T>
__device__ __forceinline__ W4<T> leg_zero() {
  const T z = to_store<T>(0.0f);
  return W4<T>{z, z, z, z};
}

// The tile of workgroup blk, and whether its cells can hold liquid (its 32 x
// 8 hull tile covers the 8 x 16 column).
struct LegTile {
  int x0, y0, z0;
  bool wet;
};
__device__ __forceinline__ LegTile leg_tile(const LevelRec& lv, int blk) {
  LegTile t;
  const int tz = (lv.d[2] + kLegZ - 1) / kLegZ, ty = (lv.d[1] + kLegY - 1) / kLegY;
  t.z0 = (blk % tz) * kLegZ;
  const int r = blk / tz;
  t.y0 = (r % ty) * kLegY;
  t.x0 = (r / ty) * kLegX;
  static_assert(kHullTZ % kLegZ == 0 && kHullTY == kLegY, "a leg tile lies in one hull tile");
  const int* hp = lv.hull + 2 * ((t.y0 / kHullTY) * lv.mg.tz + t.z0 / kHullTZ);
  t.wet = max(t.x0, cload(hp)) < min(t.x0 + kLegX, cload(hp + 1) + 1);
  return t;
}

// Loads of one window: per slot the two cells ordered by colour (first: the
// colour (x + y + z) & 1 == first), the raw right-hand sides and whether the
// first-colour cell is the odd one of its pair.
template <class W, int HX, int HZ, typename TR, typename T>
struct LegLoad {
  LegCell<T> c[2][W::SLOTS];
  TR r[2][W::SLOTS];
  unsigned odd;  // bit k: slot k's first-colour cell is its odd one
  __device__ __forceinline__ void load(const LevelRec& lv, const LegTile& t, const TR* __restrict__ rhs, int first) {
    static_assert(W::SLOTS <= 32, "one bit per slot");
    const int nx = lv.d[0], ny = lv.d[1], nz = lv.d[2];
    const T* __restrict__ wt = (const T*)lv.w;
    const long long plane = (long long)ny * nz;
    odd = 0;
#pragma unroll
    for (int k = 0; k < W::SLOTS; ++k) {
      const int q = (int)threadIdx.x + kLegThreads * k;
      const int wx = q / W::PLANE, wr = q - wx * W::PLANE, wy = wr / W::ROW, pz = wr - wy * W::ROW;
      const int gx = t.x0 - HX + wx, gy = t.y0 - HX + wy, gz = t.z0 - HZ + 2 * pz;
      W4<T> we = leg_zero<T>(), wo = leg_zero<T>();
      const T z = to_store<T>(0.0f);
      T exm = z, eym = z, ezm = z, oxm = z, oym = z;
      TR re = to_store<TR>(0.0f), ro = to_store<TR>(0.0f);
      const bool in = q < W::NP && gx >= 0 && gx < nx && gy >= 0 && gy < ny && gz >= 0;
      const size_t i = in ? (size_t)(gx * plane) + (size_t)gy * nz + gz : 0;
      if (in && gz < nz) {
        we = ldg((const W4<T>*)wt, i);
        re = ldg(rhs, i);
        if (gx > 0) exm = ldg(wt, 4 * (i - plane));
        if (gy > 0) eym = ldg(wt, 4 * (i - nz) + 1);
        if (gz > 0) ezm = ldg(wt, 4 * (i - 1) + 2);
      }
      if (in && gz + 1 < nz) {
        wo = ldg((const W4<T>*)wt, i + 1);
        ro = ldg(rhs, i + 1);
        if (gx > 0) oxm = ldg(wt, 4 * (i + 1 - plane));
        if (gy > 0) oym = ldg(wt, 4 * (i + 1 - nz) + 1);
      }
      const bool sw = ((gx + gy + gz) & 1) != first;  // the odd cell has the first colour
      odd |= sw ? 1u << k : 0u;
      LegCell<T> e, o;
      e.set(we, exm, eym, ezm);
      o.set(wo, oxm, oym, we.wz);
      c[0][k] = sw ? o : e;
      c[1][k] = sw ? e : o;
      r[0][k] = sw ? ro : re;
      r[1][k] = sw ? re : ro;
    }
  }
};

// One colour pass over the window: dst the colour updated, src the other.
// ZERO: the other colour is zero (the first pass of a sweep from e = 0).
template <class W, bool ZERO, typename TR, typename T>
__device__ __forceinline__ void leg_pass(const LegCell<T> (&c)[W::SLOTS], const TR (&r)[W::SLOTS], unsigned odd,
                                         float rm, T* dst, const T* src) {
#pragma unroll
  for (int k = 0; k < W::SLOTS; ++k) {
    const int q = (int)threadIdx.x + kLegThreads * k;
    if ((k + 1) * kLegThreads > W::NP && q >= W::NP) continue;
    const int p = W::PAD + q, s = (int)(odd >> k & 1);
    // the sweeps stage the scaled right-hand side in storage precision
    const T rs = to_store<T>(f32_rounded(Store<TR>::ld(&r[k], 0) * rm));
    float acc = wf(rs);
    if constexpr (!ZERO) {
      acc += c[k].template get<kLegWX>() * wf(src[p + W::PLANE]);
      acc += c[k].template get<kLegXM>() * wf(src[p - W::PLANE]);
      acc += c[k].template get<kLegWY>() * wf(src[p + W::ROW]);
      acc += c[k].template get<kLegYM>() * wf(src[p - W::ROW]);
      acc += c[k].template get<kLegWZ>() * wf(src[p + s]);
      acc += c[k].template get<kLegZM>() * wf(src[p - 1 + s]);
    }
    const float id = c[k].template get<kLegID>();
    dst[p] = to_store<T>(id > 0.0f ? f32_rounded(acc * id) : 0.0f);
  }
}

// Writes the tile's cells of the window to a level buffer.
template <class W, int HX, int HZ, typename T>
__device__ __forceinline__ void leg_store(const LevelRec& lv, const LegTile& t, unsigned odd, const T* a, const T* b,
                                          T* __restrict__ out) {
  const int nx = lv.d[0], ny = lv.d[1], nz = lv.d[2];
#pragma unroll
  for (int k = 0; k < W::SLOTS; ++k) {
    const int q = (int)threadIdx.x + kLegThreads * k;
    const int wx = q / W::PLANE, wr = q - wx * W::PLANE, wy = wr / W::ROW, pz = wr - wy * W::ROW;
    const int lx = wx - HX, ly = wy - HX, lz = 2 * pz - HZ;
    const int gx = t.x0 + lx, gy = t.y0 + ly, gz = t.z0 + lz;
    if (lx < 0 || lx >= kLegX || ly < 0 || ly >= kLegY || lz < 0 || lz >= kLegZ) continue;
    if (gx >= nx || gy >= ny || gz >= nz) continue;
    const T va = a[W::PAD + q], vb = b[W::PAD + q];
    const bool sw = odd >> k & 1;
    const T ev = sw ? vb : va, ov = sw ? va : vb;
    const size_t i = ((size_t)gx * ny + gy) * nz + gz;
    if ((nz & 1) == 0) {
      struct alignas(2 * sizeof(T)) Two { T lo, hi; };
      stg(reinterpret_cast<Two*>(out), i >> 1, Two{ev, ov});
    } else {
      stg(out, i, ev);
      if (gz + 1 < nz) stg(out, i + 1, ov);
    }
  }
}

// e after `pre` sweeps from zero (in the buffer that the cycle's last sweep
// does not write), and the restricted residual of the tile's coarse cells.
template <typename TR, typename T>
__global__ __launch_bounds__(kLegThreads) void k_leg_down(const Part* parts, int np, int level, int pre) {
  constexpr int HX = 2 * kLegSweeps + 1, HZ = HX + 1;
  using W = LegWindow<HX, HZ>;
  constexpr int TX = kLegX + 2, TY = kLegY + 2, TZ = kLegZ + 2;  // residual on the tile and its ring
  __shared__ T s_a[W::LDS], s_b[W::LDS];
  __shared__ T s_t[TX * TY * TZ];
  FP_PART(parts, np);
  const State* st = cload(&Gp->st);
  if (cload(&st->done)) return;
  const LevelRec lv = cload(&Gp->lv[level]);
  const LevelRec cl = cload(&Gp->lv[level + 1]);
  const bool top = level == 0;
  const TR* __restrict__ rhs = (const TR*)(top ? (const void*)cload(&Gp->r) : lv.r);
  const float rsc = top ? cload(&st->rscale) : 1.0f;
  const float rm = (top ? 1.0f : lv.Sr) / lv.Se * rsc;
  const float rmt = (top ? 1.0f : lv.Sr) / lv.St * rsc;
  const float emul = lv.Se / lv.St;
  const LegTile t = leg_tile(lv, blk);
  const int sx = cl.s[0], sy = cl.s[1], sz = cl.s[2];
  const int cnx = cl.d[0], cny = cl.d[1], cnz = cl.d[2];
  const int fnx = lv.d[0], fny = lv.d[1], fnz = lv.d[2];
  // coarse cells of the tile: four lanes per cell, one per fine plane of its
  // 4-tap x stencil
  const int CX = kLegX / sx, CY = kLegY / sy, CZ = kLegZ / sz;
  const int nc = CX * CY * CZ;
  const int X0 = t.x0 / sx, Y0 = t.y0 / sy, Z0 = t.z0 / sz;
  T* __restrict__ rc = (T*)cl.r;
  T* __restrict__ e = (T*)(lv.efinal ? lv.e : lv.e2);
  if (!t.wet) {
    // no liquid: the coarse cells over it are air
    for (int c = (int)threadIdx.x; c < nc; c += kLegThreads) {
      const int I = X0 + c / (CY * CZ), J = Y0 + c / CZ % CY, K = Z0 + c % CZ;
      if (I < cnx && J < cny && K < cnz) stg(rc, ((size_t)I * cny + J) * cnz + K, to_store<T>(0.0f));
    }
    return;
  }
  LegLoad<W, HX, HZ, TR, T> L;
  L.load(lv, t, rhs, 0);
  for (int sw = 0; sw < pre; ++sw) {
    if (sw == 0) leg_pass<W, true>(L.c[0], L.r[0], L.odd, rm, s_a, s_b);
    else leg_pass<W, false>(L.c[0], L.r[0], L.odd, rm, s_a, s_b);
    __syncthreads();
    leg_pass<W, false>(L.c[1], L.r[1], ~L.odd, rm, s_b, s_a);
    __syncthreads();
  }
  leg_store<W, HX, HZ>(lv, t, L.odd, s_a, s_b, e);
  // residual on the tile and its ring
#pragma unroll
  for (int k = 0; k < W::SLOTS; ++k) {
    const int q = (int)threadIdx.x + kLegThreads * k;
    const int wx = q / W::PLANE, wr = q - wx * W::PLANE, wy = wr / W::ROW, pz = wr - wy * W::ROW;
    const int lx = wx - HX + 1, ly = wy - HX + 1;
    if (lx < 0 || lx >= TX || ly < 0 || ly >= TY) continue;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int s = (int)(L.odd >> k & 1) ^ h;  // this cell is the odd one of its pair
      const int lz = 2 * pz - HZ + 1 + s;
      if (lz < 0 || lz >= TZ) continue;
      const int p = W::PAD + q;
      const T* own = h ? s_b : s_a;
      const T* src = h ? s_a : s_b;
      const LegCell<T>& c = L.c[h][k];
      float res = 0.0f;
      if (c.template get<kLegID>() > 0.0f) {
        const float ce = wf(own[p]);
        const float ap = c.template get<kLegWX>() * (ce - wf(src[p + W::PLANE])) + c.template get<kLegXM>() * (ce - wf(src[p - W::PLANE])) +
                         c.template get<kLegWY>() * (ce - wf(src[p + W::ROW])) + c.template get<kLegYM>() * (ce - wf(src[p - W::ROW])) +
                         c.template get<kLegWZ>() * (ce - wf(src[p + s])) + c.template get<kLegZM>() * (ce - wf(src[p - 1 + s]));
        res = Store<TR>::ld(&L.r[h][k], 0) * rmt - emul * ap;
      }
      s_t[(lx * TY + ly) * TZ + lz] = to_store<T>(res);
    }
  }
  __syncthreads();
  const int k2 = (sx == 2) + (sy == 2) + (sz == 2);
  const float fac = (1.0f / (float)(1 << k2)) * lv.St / cl.Sr;
  auto taps = [](int I, int s_, int nf, int n, int l, int* tt, float* w) {
    if (s_ == 1) {
      tt[0] = tt[1] = tt[2] = tt[3] = l + 1;
      w[0] = 1.0f;
      w[1] = w[2] = w[3] = 0.0f;
      return;
    }
    for (int q = 0; q < 4; ++q) tt[q] = 2 * l + q;  // fine 2I-1+q
    w[0] = I >= 1 ? 0.25f : 0.0f;
    w[1] = I >= 1 ? 0.75f : 1.0f;
    w[2] = 2 * I + 1 < nf ? (I + 1 >= n ? 1.0f : 0.75f) : 0.0f;
    w[3] = 2 * I + 2 < nf ? 0.25f : 0.0f;
  };
  for (int it = (int)threadIdx.x; it < 4 * nc; it += kLegThreads) {  // 4 nc: whole waves take part together
    const int c = it >> 2, b = it & 3;
    const int lx = c / (CY * CZ), ly = c / CZ % CY, lz = c % CZ;
    const int I = X0 + lx, J = Y0 + ly, K = Z0 + lz;
    const bool mine = I < cnx && J < cny && K < cnz;
    const size_t o = mine ? ((size_t)I * cny + J) * cnz + K : 0;
    const float phc = mine ? ldg(cl.phi, o) : 1.0f;
    int tx[4], ty[4], tz[4];
    float wx[4], wy[4], wz[4];
    taps(I, sx, fnx, cnx, lx, tx, wx);
    taps(J, sy, fny, cny, ly, ty, wy);
    taps(K, sz, fnz, cnz, lz, tz, wz);
    const T* pl = s_t + (sx == 1 ? lx + 1 : 2 * lx + b) * TY * TZ;
    float v = 0.0f;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const T* row = pl + ty[j] * TZ;
      const float rowsum = wz[0] * Store<T>::ld(row, tz[0]) + wz[1] * Store<T>::ld(row, tz[1]) +
                           wz[2] * Store<T>::ld(row, tz[2]) + wz[3] * Store<T>::ld(row, tz[3]);
      v += wy[j] * rowsum;
    }
    const int lane = (int)(threadIdx.x & 60);
    float acc = 0.0f;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float vj = __shfl(v, lane + j, 64);
      acc += wx[j] * vj;
    }
    if (b == 0 && mine) stg(rc, o, to_store<T>(phc < 0.0f ? acc * fac : 0.0f));
  }
}

// `post` sweeps (second colour first) of e + P e_coarse, into the buffer
// where the cycle's last sweep leaves its result.
template <typename TR, typename T>
__global__ __launch_bounds__(kLegThreads) void k_leg_up(const Part* parts, int np, int level, int post) {
  constexpr int HX = 2 * kLegSweeps, HZ = HX;
  using W = LegWindow<HX, HZ>;
  // coarse cells under the window: at most 2 HX + kLegX cells on an axis that
  // is not coarsened, half of that and a tap either side on one that is (at
  // least one is)
  constexpr int NX1 = kLegX + 2 * HX, NX2 = NX1 / 2 + 2, NZ1 = kLegZ + 2 * HZ, NZ2 = NZ1 / 2 + 2;
  constexpr int NCW = NX1 * NX1 * NZ2 > NX2 * NX1 * NZ1 ? NX1 * NX1 * NZ2 : NX2 * NX1 * NZ1;
  __shared__ T s_a[W::LDS], s_b[W::LDS];
  __shared__ T s_c[NCW];
  FP_PART(parts, np);
  const State* st = cload(&Gp->st);
  if (cload(&st->done)) return;
  const LevelRec lv = cload(&Gp->lv[level]);
  const LevelRec cl = cload(&Gp->lv[level + 1]);
  const bool top = level == 0;
  const TR* __restrict__ rhs = (const TR*)(top ? (const void*)cload(&Gp->r) : lv.r);
  const float rm = (top ? 1.0f : lv.Sr) / lv.Se * (top ? cload(&st->rscale) : 1.0f);
  const float fac = cl.Se / lv.Se;
  const LegTile t = leg_tile(lv, blk);
  const int nx = lv.d[0], ny = lv.d[1], nz = lv.d[2];
  T* __restrict__ out = (T*)(lv.efinal ? lv.e2 : lv.e);
  const T* __restrict__ e = (const T*)(lv.efinal ? lv.e : lv.e2);
  if (!t.wet) {
    // the finest level's correction is never read on such a tile; a coarse
    // level's is, as the zero of its air cells
    if (!top)
      for (int q = (int)threadIdx.x; q < kLegX * kLegY * kLegZ; q += kLegThreads) {
        const int gx = t.x0 + q / (kLegY * kLegZ), gy = t.y0 + q / kLegZ % kLegY, gz = t.z0 + q % kLegZ;
        if (gx < nx && gy < ny && gz < nz) stg(out, ((size_t)gx * ny + gy) * nz + gz, to_store<T>(0.0f));
      }
    return;
  }
  const int s3[3] = {cl.s[0], cl.s[1], cl.s[2]};
  const int cd[3] = {cl.d[0], cl.d[1], cl.d[2]};
  const int b0 = s3[0] == 2 ? t.x0 / 2 - HX / 2 - 1 : t.x0 - HX, m0 = s3[0] == 2 ? NX2 : NX1;
  const int b1 = s3[1] == 2 ? t.y0 / 2 - HX / 2 - 1 : t.y0 - HX, m1 = s3[1] == 2 ? NX2 : NX1;
  const int b2 = s3[2] == 2 ? t.z0 / 2 - HZ / 2 - 1 : t.z0 - HZ, m2 = s3[2] == 2 ? NZ2 : NZ1;
  {
    const T* __restrict__ ec = (const T*)(cl.efinal ? cl.e2 : cl.e);
    for (int q = (int)threadIdx.x; q < m0 * m1 * m2; q += kLegThreads) {
      const int a = q / (m1 * m2), r = q - a * (m1 * m2), b = r / m2, c = r - b * m2;
      const int I = b0 + a, J = b1 + b, K = b2 + c;
      const bool in = I >= 0 && I < cd[0] && J >= 0 && J < cd[1] && K >= 0 && K < cd[2];
      s_c[q] = in ? ldg(ec, ((size_t)I * cd[1] + J) * cd[2] + K) : to_store<T>(0.0f);
    }
  }
  LegLoad<W, HX, HZ, TR, T> L;
  L.load(lv, t, rhs, 1);
  T ev[W::SLOTS][2];
#pragma unroll
  for (int k = 0; k < W::SLOTS; ++k) {
    const int q = (int)threadIdx.x + kLegThreads * k;
    const int wx = q / W::PLANE, wr = q - wx * W::PLANE, wy = wr / W::ROW, pz = wr - wy * W::ROW;
    const int gx = t.x0 - HX + wx, gy = t.y0 - HX + wy, gz = t.z0 - HZ + 2 * pz;
    const bool in = q < W::NP && gx >= 0 && gx < nx && gy >= 0 && gy < ny && gz >= 0;
    const size_t i = in ? ((size_t)gx * ny + gy) * nz + gz : 0;
    ev[k][0] = in && gz < nz ? ldg(e, i) : to_store<T>(0.0f);
    ev[k][1] = in && gz + 1 < nz ? ldg(e, i + 1) : to_store<T>(0.0f);
  }
  __syncthreads();
  auto taps2 = [](int f, int s_, int n, int* c, float* w) {
    const int m = ptaps(f, s_, n, c, w);
    if (m == 1) {
      c[1] = c[0];
      w[1] = 0.0f;
    }
  };
#pragma unroll
  for (int k = 0; k < W::SLOTS; ++k) {
    const int q = (int)threadIdx.x + kLegThreads * k;
    if ((k + 1) * kLegThreads > W::NP && q >= W::NP) continue;
    const int wx = q / W::PLANE, wr = q - wx * W::PLANE, wy = wr / W::ROW, pz = wr - wy * W::ROW;
    const int gx = t.x0 - HX + wx, gy = t.y0 - HX + wy, gz = t.z0 - HZ + 2 * pz;
    const bool sw = L.odd >> k & 1;
    const float id0 = L.c[0][k].template get<kLegID>(), id1 = L.c[1][k].template get<kLegID>();
    T val[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      // h: the even (0) or odd (1) cell of the pair; air keeps zero
      const bool wet = ((h != 0) != sw ? id1 : id0) > 0.0f;
      T v = to_store<T>(0.0f);
      if (wet) {
        int cx[2], cy[2], cz[2];
        float fx[2], fy[2], fz[2];
        taps2(gx, s3[0], cd[0], cx, fx);
        taps2(gy, s3[1], cd[1], cy, fy);
        taps2(gz + h, s3[2], cd[2], cz, fz);
        auto at = [&](int a, int b, int c) { return wf(s_c[((cx[a] - b0) * m1 + (cy[b] - b1)) * m2 + (cz[c] - b2)]); };
        const float a0 = fy[0] * (fz[0] * at(0, 0, 0) + fz[1] * at(0, 0, 1)) +
                         fy[1] * (fz[0] * at(0, 1, 0) + fz[1] * at(0, 1, 1));
        const float a1 = fy[0] * (fz[0] * at(1, 0, 0) + fz[1] * at(1, 0, 1)) +
                         fy[1] * (fz[0] * at(1, 1, 0) + fz[1] * at(1, 1, 1));
        const float acc = fx[0] * a0 + fx[1] * a1;
        v = to_store<T>(wf(ev[k][h]) + fac * acc);
      }
      val[h] = v;
    }
    const T vf = sw ? val[1] : val[0], vs = sw ? val[0] : val[1];
    s_a[W::PAD + q] = vf;
    s_b[W::PAD + q] = vs;
  }
  __syncthreads();
  for (int sw = 0; sw < post; ++sw) {
    leg_pass<W, false>(L.c[0], L.r[0], L.odd, rm, s_a, s_b);
    __syncthreads();
    leg_pass<W, false>(L.c[1], L.r[1], ~L.odd, rm, s_b, s_a);
    __syncthreads();
  }
  leg_store<W, HX, HZ>(lv, t, L.odd, s_a, s_b, out);
}

}  // namespace fp

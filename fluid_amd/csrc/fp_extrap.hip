// fp_extrap.hip -- velocity extrapolation of a uniform grid on MI355X.
//
// Kernels restate lib/methods/uniform/webgpu-uniform-velocity-extrapolation.wgsl.ts
// (cited per kernel) and its schedule (…extrapolation.ts:312-392).  The
// narrow band runs only where it can change anything: a face whose lattice
// (L1) distance to every source face exceeds 3 never activates, since each
// Godunov step adds at least h/sqrt(3) and the band ends at 2h, so after the
// seed three dilations of the source masks and one compaction give the list
// of cells the passes visit.  The seed writes the whole state, on both
// ping-pong sides, at those cells and their neighbours; elsewhere only side A's
// known flags and known values, and nothing else there may be read.  Each pass is
// one launch over the list that returns at once when an earlier pass left no face active (the
// reference's indirect dispatch chain).  The hierarchy and the seed stream
// the whole grid in XCD-contiguous chunks.  No contraction anywhere: results
// equal oracle/fp_oracle_extrap.c bit for bit.
#pragma clang fp contract(off)

#include "fp_extrap.hpp"
#include "fp_uniform.hpp"

#include <algorithm>
#include <array>
#include <chrono>
#include <cmath>
#include <cstring>

namespace fp {

namespace {

constexpr float kInf = 65504.0f;  // DISTANCE_INFINITY (…extrapolation.wgsl.ts:61)
constexpr int kThreads = 256;
// A face's part in the front between two passes (ExState::stat).
constexpr unsigned kQuiet = 0, kEligible = 1,  // inactive; eligible: its candidate distance lies in the band
    kActive = 2, kConverged = 3;               // converged in the last pass, and inactive since

// Division by a launch-invariant divisor: floor(n / d) = (n * m) >> s for
// every n < 2^31 with s = 31 + ceil(log2 d), m = ceil(2^s / d) < 2^32
// (Granlund and Montgomery, "Division by invariant integers using
// multiplication", PLDI 1994, Thm 4.2).  Cell indices stay below 2^31.
struct FastDiv {
  unsigned m;
  int s;
};
FastDiv make_div(unsigned d) {
  int l = 0;
  while ((1ull << l) < d) ++l;
  const unsigned long long m = ((1ull << (31 + l)) + d - 1) / d;
  return FastDiv{(unsigned)m, 31 + l};
}
__device__ __forceinline__ unsigned fdiv(unsigned n, FastDiv f) {
  return (unsigned)(((unsigned long long)n * f.m) >> f.s);
}

struct ExGeo {
  int d[3];
  float h;
  int open_top;
  float eps_min, eps_max;  // fimConvergenceEpsilon's clamp (…wgsl.ts:114-119)
  FastDiv dz, dy;          // division by nz and by ny
};

__device__ __forceinline__ unsigned eidx(const ExGeo& g, int x, int y, int z) {
  return ((unsigned)x * g.d[1] + y) * g.d[2] + z;
}
__device__ __forceinline__ bool ein(const int* d, int x, int y, int z) {
  return x >= 0 && y >= 0 && z >= 0 && x < d[0] && y < d[1] && z < d[2];
}
// cell index -> (x, y, z) of a lattice with divisors dz = nz, dy = ny
__device__ __forceinline__ void decode3(unsigned i, int ny, int nz, FastDiv dz, FastDiv dy, int& x, int& y, int& z) {
  const unsigned t = fdiv(i, dz);
  z = (int)(i - t * (unsigned)nz);
  const unsigned xx = fdiv(t, dy);
  y = (int)(t - xx * (unsigned)ny);
  x = (int)xx;
}
__device__ __forceinline__ void edecode(const ExGeo& g, unsigned i, int& x, int& y, int& z) {
  decode3(i, g.d[1], g.d[2], g.dz, g.dy, x, y, z);
}
// positive face of cell (x,y,z) along c in the (n_c + 1)-long face array
__device__ __forceinline__ unsigned face_of(const ExGeo& g, int c, int x, int y, int z) {
  return c == 0 ? ((unsigned)(x + 1) * g.d[1] + y) * g.d[2] + z
       : c == 1 ? ((unsigned)x * (g.d[1] + 1) + y + 1) * g.d[2] + z
                : ((unsigned)x * g.d[1] + y) * (g.d[2] + 1) + z + 1;
}
// XCD-contiguous chunk of a streaming launch: workgroup b runs on XCD b mod 8
__device__ __forceinline__ unsigned chunk_of(unsigned chunks) {
  const unsigned per = (chunks + 7) / 8;
  return (blockIdx.x & 7) * per + (blockIdx.x >> 3);
}
__device__ __forceinline__ float eps_of(const ExGeo& g, float reference) {
  float a = fabsf(reference);
  a = a < g.eps_min ? g.eps_min : (a > g.eps_max ? g.eps_max : a);
  return a * 1.1920929e-7f;
}
__device__ __forceinline__ int block_sum(int v) {
  __shared__ int part[kThreads / 64];
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_down(v, o, 64);
  if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = v;
  __syncthreads();
  int s = 0;
  if (threadIdx.x == 0)
    for (int k = 0; k < kThreads / 64; ++k) s += part[k];
  return s;
}

// ---- classes: open (bits 0-2) and source (bits 3-5) per component ----
// faceOpenFraction (webgpu-uniform-reference.wgsl.ts:511-519) without solids,
// sourceFace (…extrapolation.wgsl.ts:100-104)
// Streaming kernels take kCells cells per thread (kCells x kThreads per
// workgroup, the cells of one pass kThreads apart) and issue every load of
// their cells before the first store: neighbour loads are clamped to the cell
// itself at the domain edge and masked afterwards, so no branch separates
// them.  One cell per thread, or loads behind bounds branches, left these
// kernels waiting on one memory round trip at a time.
constexpr int kCells = 4;

__device__ __forceinline__ unsigned cell_of(unsigned n, int j) {
  const unsigned per_group = kThreads * kCells;
  return chunk_of((n + per_group - 1) / per_group) * per_group + j * kThreads + threadIdx.x;
}

// exclusive prefix of v over the workgroup, and the workgroup total
__device__ __forceinline__ int block_scan(int v, int* total) {
  __shared__ int wsum[kThreads / 64];
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  int x = v;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int y = __shfl_up(x, o, 64);
    if (lane >= o) x += y;
  }
  if (lane == 63) wsum[wid] = x;
  __syncthreads();
  int before = 0, all = 0;
#pragma unroll
  for (int k = 0; k < kThreads / 64; ++k) {
    before += k < wid ? wsum[k] : 0;
    all += wsum[k];
  }
  *total = all;
  return before + x - v;
}

__global__ __launch_bounds__(kThreads) void k_ex_classify(ExGeo g, const float* __restrict__ field, int is_phi,
                                                         uint8_t* __restrict__ cls, uint8_t* __restrict__ cand,
                                                         unsigned n) {
  const unsigned sx = (unsigned)g.d[1] * g.d[2], sy = (unsigned)g.d[2];
  float f[kCells][4];
  int pos[kCells][3];
#pragma unroll
  for (int j = 0; j < kCells; ++j) {
    const unsigned i = min(cell_of(n, j), n - 1);
    int x, y, z;
    edecode(g, i, x, y, z);
    pos[j][0] = x;
    pos[j][1] = y;
    pos[j][2] = z;
    f[j][0] = field[i];
    f[j][1] = field[i + (x + 1 < g.d[0] ? sx : 0u)];
    f[j][2] = field[i + (y + 1 < g.d[1] ? sy : 0u)];
    f[j][3] = field[i + (z + 1 < g.d[2] ? 1u : 0u)];
  }
#pragma unroll
  for (int j = 0; j < kCells; ++j) {
    const unsigned i = cell_of(n, j);
    if (i >= n) break;
    bool wet[4];
    for (int k = 0; k < 4; ++k) wet[k] = is_phi ? f[j][k] < 0.0f : f[j][k] > 0.5f;
    unsigned b = 0;
    for (int c = 0; c < 3; ++c) {
      const bool inside = pos[j][c] + 1 < g.d[c];
      const bool open = inside || (c == 1 && g.open_top);
      if (!open) continue;
      b |= 1u << c;
      if (wet[0] || (inside && wet[1 + c])) b |= 8u << c;
    }
    cls[i] = (uint8_t)b;
    cand[i] = (uint8_t)(b >> 3);
  }
}

// ---- four cells in a word ----
// The byte arrays (classes, candidates) are worked on four consecutive cells
// to a lane: the cells' bytes are one word and so are those of each neighbour
// offset, loaded unaligned, with the bytes of cells that have no neighbour
// there masked off.  Seven word loads serve four cells where a load per byte
// took twenty-eight (the dilations and the seed were bound by them: at 384^3
// the dilations take 32 to 69 us for 62 to 100, the seed, which also writes
// less, 198 for 650).  A quad may run over a row's or a plane's end, so
// nothing depends on the row length; the arrays carry quad_pad bytes on either
// side for the words that reach past the grid.
struct Quad {
  unsigned i;         // first cell
  unsigned in;        // mask of the cells below n
  unsigned ok[6];     // mask of the cells that have the neighbour (-x, +x, -y, +y, -z, +z)
  int x, y, z;        // of the first cell
  bool row;           // the cells are one row's
  __device__ __forceinline__ Quad(const ExGeo& g, unsigned n) {
    const unsigned per_group = kThreads * 4;
    i = chunk_of((n + per_group - 1) / per_group) * per_group + 4 * threadIdx.x;
    in = 0;
    row = false;
#pragma unroll
    for (int k = 0; k < 6; ++k) ok[k] = 0;
    if (i >= n) return;
    edecode(g, i, x, y, z);
    row = z + 3 < g.d[2];
    if (row) {  // (so every cell is below n)
      in = ~0u;
      ok[0] = x > 0 ? ~0u : 0u;
      ok[1] = x + 1 < g.d[0] ? ~0u : 0u;
      ok[2] = y > 0 ? ~0u : 0u;
      ok[3] = y + 1 < g.d[1] ? ~0u : 0u;
      ok[4] = z > 0 ? ~0u : ~0u << 8;
      ok[5] = z + 4 < g.d[2] ? ~0u : ~0u >> 8;
      return;
    }
    int a = x, b = y, c = z;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const unsigned m = i + j < n ? 0xffu << 8 * j : 0u;
      in |= m;
      ok[0] |= a > 0 ? m : 0u;
      ok[1] |= a + 1 < g.d[0] ? m : 0u;
      ok[2] |= b > 0 ? m : 0u;
      ok[3] |= b + 1 < g.d[1] ? m : 0u;
      ok[4] |= c > 0 ? m : 0u;
      ok[5] |= c + 1 < g.d[2] ? m : 0u;
      if (++c == g.d[2]) {
        c = 0;
        if (++b == g.d[1]) {
          b = 0;
          ++a;
        }
      }
    }
  }
};
__device__ __forceinline__ unsigned word_at(const uint8_t* p, int i) {
  unsigned w;
  __builtin_memcpy(&w, p + i, 4);
  return w;
}
// the OR of the six neighbours' bytes, per cell
__device__ __forceinline__ unsigned around(const ExGeo& g, const Quad& q, const uint8_t* __restrict__ a) {
  const int sx = g.d[1] * g.d[2], sy = g.d[2], i = (int)q.i;
  const int off[6] = {-sx, sx, -sy, sy, -1, 1};
  unsigned w[6], m = 0;
#pragma unroll
  for (int k = 0; k < 6; ++k) w[k] = word_at(a, i + off[k]);
#pragma unroll
  for (int k = 0; k < 6; ++k) m |= w[k] & q.ok[k];
  return m;
}
constexpr unsigned kBits3 = 0x07070707u, kBit = 0x01010101u;

// seedActiveFront (…extrapolation.wgsl.ts:148-170).  Flags everywhere; the
// rest only where it is read: a known face's value (the hierarchy selects by
// the flags), and the whole state, on both sides, where a pass can read it
// before writing it: the band list's cells (listed) and their 6-neighbours (a
// pass writes every list cell of its destination side, and reads its source
// side at list cells and their neighbours only).  At 384^3 the list holds 1% of
// the cells: inside the liquid the seed copies 12 bytes a cell, in the air
// beyond the band it writes one, where it wrote 25 and 50.
__global__ __launch_bounds__(kThreads) void k_ex_seed(ExGeo g, const uint8_t* __restrict__ cls,
                                                     const uint8_t* __restrict__ listed,
                                                     const float* __restrict__ u, const float* __restrict__ v,
                                                     const float* __restrict__ w, ExState a, ExState b,
                                                     ExCounters* cnt, unsigned n) {
  const Quad q(g, n);
  int active = 0;
  if (q.in) {
    const unsigned me = word_at(cls, (int)q.i) & q.in;
    const unsigned nr = (word_at(listed, (int)q.i) | around(g, q, listed)) & q.in;
    const unsigned open = me & kBits3, known = me >> 3 & kBits3;
    const unsigned act = open & ~known & (around(g, q, cls) >> 3 & kBits3);
    const unsigned stat = (act & kBit) << 1 | (act >> 1 & kBit) << 3 | (act >> 2 & kBit) << 5;
    static_assert(kActive == 2, "an active face's state is the upper of its two bits");
    active = __popc(act);
    reinterpret_cast<unsigned*>(a.flags)[q.i >> 2] = known;
    if (nr) {
      reinterpret_cast<unsigned*>(a.stat)[q.i >> 2] = stat;
      reinterpret_cast<unsigned*>(b.flags)[q.i >> 2] = known;
      reinterpret_cast<unsigned*>(b.stat)[q.i >> 2] = stat;
    }
    if (known || nr) {
      // the positive face of every cell exists in the face arrays, four of a
      // row side by side
      float in[3][4], val[3][4], dist[3][4];
      if (q.row) {
        __builtin_memcpy(in[0], u + face_of(g, 0, q.x, q.y, q.z), 16);
        __builtin_memcpy(in[1], v + face_of(g, 1, q.x, q.y, q.z), 16);
        __builtin_memcpy(in[2], w + face_of(g, 2, q.x, q.y, q.z), 16);
      } else {
        int x = q.x, y = q.y, z = q.z;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const bool there = q.in >> 8 * j & 1u;
          in[0][j] = there ? u[face_of(g, 0, x, y, z)] : 0.0f;
          in[1][j] = there ? v[face_of(g, 1, x, y, z)] : 0.0f;
          in[2][j] = there ? w[face_of(g, 2, x, y, z)] : 0.0f;
          if (++z == g.d[2]) {
            z = 0;
            if (++y == g.d[1]) {
              y = 0;
              ++x;
            }
          }
        }
      }
#pragma unroll
      for (int c = 0; c < 3; ++c)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const bool k = known >> (8 * j + c) & 1u;
          val[c][j] = k ? in[c][j] : 0.0f;
          dist[c][j] = k ? 0.0f : kInf;
        }
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        const float4 vc = make_float4(val[c][0], val[c][1], val[c][2], val[c][3]);
        const float4 dc = make_float4(dist[c][0], dist[c][1], dist[c][2], dist[c][3]);
        reinterpret_cast<float4*>(a.val[c])[q.i >> 2] = vc;
        if (nr) {
          reinterpret_cast<float4*>(a.dist[c])[q.i >> 2] = dc;
          reinterpret_cast<float4*>(b.val[c])[q.i >> 2] = vc;
          reinterpret_cast<float4*>(b.dist[c])[q.i >> 2] = dc;
        }
      }
    }
  }
  const int s = block_sum(active);
  if (threadIdx.x == 0 && s) atomicAdd(&cnt->active[0][blockIdx.x % kExSpread][0], s);
}

// one 6-neighbour OR of the candidate bits; the last one appends the cells
// with an open non-source candidate face to the band list (one atomic per
// workgroup) and stores which they are
__global__ __launch_bounds__(kThreads) void k_ex_dilate(ExGeo g, const uint8_t* __restrict__ cls,
                                                       const uint8_t* __restrict__ in, uint8_t* __restrict__ out,
                                                       int last, int* __restrict__ list, ExCounters* cnt,
                                                       unsigned n) {
  const Quad q(g, n);
  unsigned takes = 0;
  if (q.in) {
    const unsigned me = last ? word_at(cls, (int)q.i) : 0u;
    unsigned m = (word_at(in, (int)q.i) | around(g, q, in)) & q.in;
    if (last) {
      takes = m & me & ~(me >> 3) & kBits3;
      takes = (takes | takes >> 1 | takes >> 2) & kBit;
      m = takes;
    }
    reinterpret_cast<unsigned*>(out)[q.i >> 2] = m;
  }
  if (!last) return;
  int total;
  int at = block_scan(__popc(takes), &total);
  __shared__ int base;
  if (threadIdx.x == 0) base = total ? atomicAdd(&cnt->list_count, total) : 0;
  __syncthreads();
  at += base;
#pragma unroll
  for (int j = 0; j < 4; ++j)
    if (takes >> 8 * j & 1u) list[at++] = (int)(q.i + j);
}

// ---- the band pass (updateActiveFront and helpers, …extrapolation.wgsl.ts:172-331) ----
// godunovDistance (…extrapolation.wgsl.ts:188-215), cubic cells, from the
// distances of the neighbours (-x, +x, -y, +y, -z, +z; kInf where there is no
// open face)
__device__ __forceinline__ float godunov(const float* nd, float h) {
  float m[3];
#pragma unroll
  for (int a = 0; a < 3; ++a) m[a] = nd[2 * a] < nd[2 * a + 1] ? nd[2 * a] : nd[2 * a + 1];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = i + 1; j < 3; ++j)
      if (m[j] < m[i]) {
        const float t = m[i];
        m[i] = m[j];
        m[j] = t;
      }
  if (m[0] >= 0.5f * kInf) return kInf;
  float root = m[0] + h;
#pragma unroll
  for (int count = 2; count <= 3; ++count) {
    if (m[count - 1] >= 0.5f * kInf || root <= m[count - 1]) break;
    float A = 0.0f, B = 0.0f, C = -1.0f;
    for (int k = 0; k < count; ++k) {
      const float inv = 1.0f / (h * h);
      A += inv;
      B += m[k] * inv;
      C += m[k] * m[k] * inv;
    }
    const float disc = B * B - A * C;
    root = (B + sqrtf(disc > 0.0f ? disc : 0.0f)) / A;
  }
  return root;
}

// upwindExtensionValue (…extrapolation.wgsl.ts:221-248); nv: the neighbours'
// values (0 where unknown)
__device__ __forceinline__ float upwind(const ExGeo& g, const float* nd, const float* nv, float solved) {
  const float h = g.h;
  float wt[3], ws[3];
  const float eps = eps_of(g, solved);
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    wt[a] = 0.0f;
    ws[a] = 0.0f;
    const float dl = nd[2 * a], dh = nd[2 * a + 1];
    const float mn = dl < dh ? dl : dh;
    if (mn >= solved - eps) continue;
    float mv = 0.0f, mc = 0.0f;
    if (fabsf(dl - mn) <= eps) {
      mv += nv[2 * a];
      mc += 1.0f;
    }
    if (fabsf(dh - mn) <= eps) {
      mv += nv[2 * a + 1];
      mc += 1.0f;
    }
    if (mc <= 0.0f) continue;
    const float weight = (solved - mn) / (h * h);
    wt[a] = weight * mv / mc;
    ws[a] = weight;
  }
  const float value = (wt[0] + wt[2]) + wt[1], sum = (ws[0] + ws[2]) + ws[1];
  return sum > 0.0f ? value / sum : 0.0f;
}

// One pass over the band list.  A pass of the reference updates the active
// faces and activates the inactive ones beside a face that converges in that
// pass (activatedByConvergedUpwindNeighbor, …wgsl.ts:266-283, which evaluates
// activeNodeConverges, :253-265, of each neighbour again from the neighbours
// of that).  Here a face that converges says so in its state, and the faces
// beside it are activated when the next pass starts: whether one is depends
// on its own candidate distance before the pass, which it computes there and
// keeps as kEligible, on the converged neighbour's new distance, which is
// that neighbour's state, and on its own distance, which did not change.  So
// a face reads its six neighbours and nothing further, where one of seven
// Godunov updates was its own before: 90 -> 33 us a pass on the 654 K cells
// under 384^3, 39 -> 8.3 us at 160 x 117 x 143.
//
// The pass therefore counts the faces active before it; `last` only counts
// (the faces that the pass before left active).  A wave takes one component of
// 64 list cells: three times the waves of a lane per cell, each a third as
// long.  A face's distance is kInf and its value 0 where it is not open or not
// known yet (the seed's state), so neither needs its class or flags.
__global__ __launch_bounds__(3 * 64) void k_ex_pass(ExGeo g, const uint8_t* __restrict__ cls,
                                                    const int* __restrict__ list, int count, ExState src, ExState dst,
                                                    ExCounters* cnt, int pass, int last) {
  __shared__ unsigned s_bits[3][64];
  __shared__ int s_active[3];
  const int lane = (int)(threadIdx.x & 63), c = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  {
    // nothing was active before the previous pass (the first: after the seed)
    const int seen = cnt->active[max(pass - 2, 0)][lane % kExSpread][0];
    if (!__any(seen != 0)) return;
  }
  if (!last && blockIdx.x == 0 && threadIdx.x == 0) cnt->latest = pass & 1;
  const int k = (int)blockIdx.x * 64 + lane;
  const bool mine = k < count;
  const unsigned i = mine ? (unsigned)list[k] : 0u;
  bool act = false;
  unsigned bits = 0;  // known(c) in bit c, the new state in bits 3 + 2c
  if (mine) {
    int x, y, z;
    edecode(g, i, x, y, z);
    const unsigned sx = (unsigned)g.d[1] * g.d[2], sy = (unsigned)g.d[2];
    const bool ok[6] = {x > 0, x + 1 < g.d[0], y > 0, y + 1 < g.d[1], z > 0, z + 1 < g.d[2]};
    const unsigned at[6] = {ok[0] ? i - sx : i, ok[1] ? i + sx : i, ok[2] ? i - sy : i,
                            ok[3] ? i + sy : i, ok[4] ? i - 1 : i,  ok[5] ? i + 1 : i};
    const unsigned me = cls[i], own = src.stat[i] >> 2 * c & 3u, flags = src.flags[i];
    float dist = src.dist[c][i], val = src.val[c][i], nd[6], nv[6];
    unsigned ns[6];
#pragma unroll
    for (int q = 0; q < 6; ++q) {
      nd[q] = src.dist[c][at[q]];
      nv[q] = src.val[c][at[q]];
      ns[q] = src.stat[at[q]];
    }
#pragma unroll
    for (int q = 0; q < 6; ++q) {
      nd[q] = ok[q] ? nd[q] : kInf;
      nv[q] = ok[q] ? nv[q] : 0.0f;
      ns[q] = ok[q] ? ns[q] >> 2 * c & 3u : kQuiet;
    }
    unsigned known = flags >> c & 1u, state = kQuiet;
    if ((me >> c & 1) && !(me >> (3 + c) & 1)) {
      const float eps = eps_of(g, dist);
      act = own == kActive;
      if (own == kEligible)
#pragma unroll
        for (int q = 0; q < 6; ++q) act = act || (ns[q] == kConverged && dist > nd[q] + eps);
      bool stirring = act;  // a neighbour may be active, so may converge in this pass
#pragma unroll
      for (int q = 0; q < 6; ++q) stirring = stirring || ns[q] == kActive || ns[q] == kEligible;
      if (!last && stirring) {
        const float cand = godunov(nd, g.h);
        if (act) {
          const float old = dist;
          const float upd = old < cand ? old : cand;
          const bool conv = old < 0.5f * kInf && fabsf(upd - old) <= eps;
          if (upd <= 2.0f * g.h) {
            dist = upd;
            val = upwind(g, nd, nv, upd);
            known = 1u;
            state = conv ? kConverged : kActive;
          }
        } else if (!(cand > 2.0f * g.h)) {
          state = kEligible;
        }
      }
    }
    if (!last) {
      dst.val[c][i] = val;
      dst.dist[c][i] = dist;
      bits = known << c | state << (3 + 2 * c);
    }
  }
  s_bits[c][lane] = bits;
  const unsigned long long who = __ballot(act);
  if (lane == 0) s_active[c] = __popcll(who);
  __syncthreads();
  if (c != 0) return;
  if (mine && !last) {
    const unsigned all = s_bits[0][lane] | s_bits[1][lane] | s_bits[2][lane];
    dst.flags[i] = (uint8_t)(all & 7u);
    dst.stat[i] = (uint8_t)(all >> 3);
  }
  const int total = s_active[0] + s_active[1] + s_active[2];
  if (lane == 0 && total && pass > 1) atomicAdd(&cnt->active[pass - 1][blockIdx.x % kExSpread][0], total);
}

// the counters' sums
__global__ void k_ex_totals(const ExCounters* __restrict__ cnt, ExTotals* __restrict__ t) {
  const int k = (int)threadIdx.x;
  if (k < 20) {
    int s = 0;
    for (int q = 0; q < kExSpread; ++q) s += cnt->active[k][q][0];
    t->active[k] = s;
  } else if (k < 22) {
    unsigned long long s = 0;
    for (int q = 0; q < kExSpread; ++q) s += k == 20 ? cnt->unknown[q][0] : cnt->band_known[q][0];
    (k == 20 ? t->unknown : t->band_known) = s;
  }
}

// ---- hierarchy (…extrapolation.wgsl.ts:385-488) ----
struct ExSrc {
  int d[3];
  const float* val[3];
  const uint8_t* known;
};

// hierarchyComponentSample: renormalised trilinear sample of known values,
// the component axis face-centred; returns the weight sum
__device__ float hier_sample(const ExSrc& S, const int* T, const int* p, int c, float* value) {
  float pos[3];
  for (int a = 0; a < 3; ++a) pos[a] = ((float)p[a] + 0.5f) * (float)S.d[a] / (float)T[a] - 0.5f;
  pos[c] = (float)(p[c] + 1) * (float)S.d[c] / (float)T[c] - 1.0f;
  int lower[3];
  float fr[3];
  for (int a = 0; a < 3; ++a) {
    const float f = floorf(pos[a]);
    lower[a] = (int)f;
    fr[a] = pos[a] - f;
  }
  float cx[8], cw[8];
#pragma unroll
  for (int corner = 0; corner < 8; ++corner) {
    const int off[3] = {corner & 1, corner >> 1 & 1, corner >> 2 & 1};
    int q[3];
    float wgt[3];
    for (int a = 0; a < 3; ++a) {
      q[a] = min(max(lower[a] + off[a], 0), S.d[a] - 1);
      wgt[a] = off[a] ? fr[a] : 1.0f - fr[a];
    }
    const float weight = wgt[0] * wgt[1] * wgt[2];
    const unsigned i = ((unsigned)q[0] * S.d[1] + q[1]) * S.d[2] + q[2];
    // load every corner (the clamped index is always valid) and select:
    // branch-free, so the eight corners' loads are in flight together
    const unsigned kn = S.known[i];
    const float val = S.val[c][i];
    const bool use = weight > 0.0f && (kn >> c & 1);
    cx[corner] = use ? weight * val : 0.0f;
    cw[corner] = use ? weight : 0.0f;
  }
  const float xs = ((cx[0] + cx[5]) + (cx[1] + cx[4])) + ((cx[2] + cx[7]) + (cx[3] + cx[6]));
  const float wsum = ((cw[0] + cw[5]) + (cw[1] + cw[4])) + ((cw[2] + cw[7]) + (cw[3] + cw[6]));
  *value = wsum > 0.0f ? xs / wsum : 0.0f;
  return wsum;
}

__device__ __forceinline__ void known_at(const ExSrc& S, int x, int y, int z, int c, float* v, float* w) {
  *v = 0.0f;
  *w = 0.0f;
  if (!ein(S.d, x, y, z)) return;
  const unsigned i = ((unsigned)x * S.d[1] + y) * S.d[2] + z;
  if (S.known[i] >> c & 1) {
    *v = S.val[c][i];
    *w = 1.0f;
  }
}

// hierarchyCorrespondingCellSample (…wgsl.ts:430-447)
__device__ float corresponding_sample(const ExSrc& S, const int* p, int c, float* value) {
  const int lx = 2 * p[0], ly = 2 * p[1], lz = 2 * p[2];
  float sx = 0.0f, sw = 0.0f;
  for (int oy = 0; oy <= 1; ++oy) {
    float v00, w00, v11, w11, v10, w10, v01, w01;
    known_at(S, lx, ly + oy, lz, c, &v00, &w00);
    known_at(S, lx + 1, ly + oy, lz + 1, c, &v11, &w11);
    known_at(S, lx + 1, ly + oy, lz, c, &v10, &w10);
    known_at(S, lx, ly + oy, lz + 1, c, &v01, &w01);
    sx += (v00 + v11) + (v10 + v01);
    sw += (w00 + w11) + (w10 + w01);
  }
  *value = sw > 0.0f ? sx / sw : 0.0f;
  return sw;
}

// resolveConvergedFront (…wgsl.ts:359-369): the band cells' final state,
// on the side the last pass wrote, back into side A, which then holds the
// band result of every cell
__global__ __launch_bounds__(kThreads) void k_ex_resolve(const int* __restrict__ list, int count, ExState a,
                                                        ExState b, const ExCounters* cnt) {
  const int k = blockIdx.x * kThreads + threadIdx.x;
  if (k >= count || cnt->latest == 0) return;
  const unsigned i = (unsigned)list[k];
  for (int c = 0; c < 3; ++c) a.val[c][i] = b.val[c][i];
  a.flags[i] = b.flags[i];
}

// restrictKnownVelocity (…wgsl.ts:450-471); level 1 samples the band result
__global__ __launch_bounds__(kThreads) void k_ex_restrict(ExSrc src, ExLevel tgt, FastDiv tz, FastDiv ty) {
  const unsigned n = (unsigned)tgt.n;
  const unsigned i = chunk_of((n + kThreads - 1) / kThreads) * kThreads + threadIdx.x;
  if (i >= n) return;
  int p[3];
  decode3(i, tgt.d[1], tgt.d[2], tz, ty, p[0], p[1], p[2]);
  unsigned known = 0;
  for (int c = 0; c < 3; ++c) {
    float v;
    float w = hier_sample(src, tgt.d, p, c, &v);
    if (w <= 0.0f && c == 1) w = corresponding_sample(src, p, c, &v);
    tgt.val[c][i] = w > 0.0f ? v : 0.0f;
    if (w > 0.0f) known |= 1u << c;
  }
  tgt.known[i] = (uint8_t)known;
}

// ---- prolongation of a tile ----
// The target level in tiles of kTileX x kTileY x kTileZ cells, a lane per
// (y, z) column.  hier_sample reads eight corners per component from the
// coarser level, and neighbouring cells read the same ones: 48 gathers a cell,
// and nine divisions for the sample positions, bound the prolongations.  Here
// the coarse cells under the tile are staged in LDS once, per component as
// (value or 0, known 1 or 0), with the coarse index clamped at staging; a
// lane's y and z positions are made once for its kTileX cells.  A sample is
// then eight LDS reads at fixed offsets and the sums of hier_sample, in its
// order.
constexpr int kTileX = 4, kTileY = 8, kTileZ = 32;
// coarse cells under a tile: about half its extent, the far corner, the one
// cell between the centred and the face sample, and one for odd levels' ratio
constexpr int kWinX = 6, kWinY = 8, kWinZ = 20, kWin = kWinX * kWinY * kWinZ;

struct TilePos {  // one axis of a sample: window index of the lower corner, fraction
  int lo;
  float fr;
};
__device__ __forceinline__ float sample_pos(int p, int S, int T, bool face) {
  return face ? (float)(p + 1) * (float)S / (float)T - 1.0f : ((float)p + 0.5f) * (float)S / (float)T - 0.5f;
}
__device__ __forceinline__ TilePos tile_pos(int p, int S, int T, bool face, int base) {
  const float pos = sample_pos(p, S, T, face), f = floorf(pos);
  return TilePos{(int)f - base, pos - f};
}
// First coarse cell under target cells p0 .. p1 of an axis and their number
__device__ __forceinline__ void tile_window(int p0, int p1, int S, int T, int& base, int& count) {
  base = (int)floorf(fminf(sample_pos(p0, S, T, false), sample_pos(p0, S, T, true)));
  count = (int)floorf(fmaxf(sample_pos(p1, S, T, false), sample_pos(p1, S, T, true))) + 2 - base;
}

// The sample of component c (hier_sample's corners and sums)
__device__ __forceinline__ float tile_sample(const float2* win, const TilePos* ax, float* value) {
  const float2* w = win + (ax[0].lo * kWinY + ax[1].lo) * kWinZ + ax[2].lo;
  float cx[8], cw[8];
#pragma unroll
  for (int corner = 0; corner < 8; ++corner) {
    const int o0 = corner & 1, o1 = corner >> 1 & 1, o2 = corner >> 2 & 1;
    const float weight = (o0 ? ax[0].fr : 1.0f - ax[0].fr) * (o1 ? ax[1].fr : 1.0f - ax[1].fr) *
                         (o2 ? ax[2].fr : 1.0f - ax[2].fr);
    const float2 v = w[(o0 * kWinY + o1) * kWinZ + o2];
    cx[corner] = weight > 0.0f ? weight * v.x : 0.0f;  // (a corner without weight may hold an infinity)
    cw[corner] = weight * v.y;
  }
  const float xs = ((cx[0] + cx[5]) + (cx[1] + cx[4])) + ((cx[2] + cx[7]) + (cx[3] + cx[6]));
  const float wsum = ((cw[0] + cw[5]) + (cw[1] + cw[4])) + ((cw[2] + cw[7]) + (cw[3] + cw[6]));
  *value = wsum > 0.0f ? xs / wsum : 0.0f;
  return wsum;
}

// Samples the unknown components of a lane's kTileX cells: known bits and
// values (c, cell) in and out.  need: some lane of the workgroup has one (the
// whole workgroup calls this with the same).  T: the target level.
__device__ __forceinline__ void tile_fill(const ExSrc& S, const int* T, int x0, int y0, int z0, float2* win,
                                          unsigned (&known)[kTileX], float (&val)[kTileX][3]) {
  int base[3], m[3];
  const int p0[3] = {x0, y0, z0};
  const int tile[3] = {kTileX, kTileY, kTileZ};
#pragma unroll
  for (int a = 0; a < 3; ++a) tile_window(p0[a], min(p0[a] + tile[a], T[a]) - 1, S.d[a], T[a], base[a], m[a]);
  const int tid = (int)threadIdx.x;
  const int y = y0 + (tid / kTileZ), z = z0 + tid % kTileZ;
  if (m[0] > kWinX || m[1] > kWinY || m[2] > kWinZ) {  // no level ratio makes such a window; sampled directly
    for (int j = 0; j < kTileX; ++j) {
      const int p[3] = {x0 + j, y, z};
      if (p[0] >= T[0] || y >= T[1] || z >= T[2]) continue;
      for (int c = 0; c < 3; ++c) {
        float v;
        if (!(known[j] >> c & 1) && hier_sample(S, T, p, c, &v) > 0.0f) {
          val[j][c] = v;
          known[j] |= 1u << c;
        }
      }
    }
    return;
  }
  for (int q = tid; q < m[0] * m[1] * m[2]; q += kThreads) {
    const int d = q % m[2], t = q / m[2], b = t % m[1], a = t / m[1];
    const int X = min(max(base[0] + a, 0), S.d[0] - 1), Y = min(max(base[1] + b, 0), S.d[1] - 1),
              Z = min(max(base[2] + d, 0), S.d[2] - 1);
    const unsigned i = ((unsigned)X * S.d[1] + Y) * S.d[2] + Z;
    const unsigned kn = S.known[i];
    const float v[3] = {S.val[0][i], S.val[1][i], S.val[2][i]};
    const int o = (a * kWinY + b) * kWinZ + d;
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      const bool k = kn >> c & 1;
      win[c * kWin + o] = make_float2(k ? v[c] : 0.0f, k ? 1.0f : 0.0f);
    }
  }
  __syncthreads();
  if (y >= T[1] || z >= T[2]) return;
  const TilePos py[2] = {tile_pos(y, S.d[1], T[1], false, base[1]), tile_pos(y, S.d[1], T[1], true, base[1])};
  const TilePos pz[2] = {tile_pos(z, S.d[2], T[2], false, base[2]), tile_pos(z, S.d[2], T[2], true, base[2])};
#pragma unroll
  for (int j = 0; j < kTileX; ++j) {
    if (x0 + j >= T[0] || known[j] == 7u) continue;
    const TilePos px[2] = {tile_pos(x0 + j, S.d[0], T[0], false, base[0]),
                           tile_pos(x0 + j, S.d[0], T[0], true, base[0])};
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      if (known[j] >> c & 1) continue;
      const TilePos ax[3] = {px[c == 0], py[c == 1], pz[c == 2]};
      float v;
      if (tile_sample(win + c * kWin, ax, &v) > 0.0f) {
        val[j][c] = v;
        known[j] |= 1u << c;
      }
    }
  }
}

// tile of a launch over the level's tiles (z fastest), in XCD-contiguous runs
__device__ __forceinline__ bool tile_of(const int* T, int& x0, int& y0, int& z0) {
  const unsigned tz = (T[2] + kTileZ - 1) / kTileZ, ty = (T[1] + kTileY - 1) / kTileY, tx = (T[0] + kTileX - 1) / kTileX;
  const unsigned t = chunk_of(tx * ty * tz);
  if (t >= tx * ty * tz) return false;
  z0 = (int)(t % tz) * kTileZ;
  y0 = (int)(t / tz % ty) * kTileY;
  x0 = (int)(t / (tz * ty)) * kTileX;
  return true;
}

// prolongUnknownVelocity (…wgsl.ts:473-488) into a level's up arrays, a lane
// per cell: for levels too small to fill the chip with tiles, where a tile's
// staging is one more round trip (kTileCells)
__global__ __launch_bounds__(kThreads) void k_ex_prolong_cells(ExSrc src, ExLevel tgt, FastDiv tz, FastDiv ty) {
  const unsigned n = (unsigned)tgt.n;
  const unsigned i = chunk_of((n + kThreads - 1) / kThreads) * kThreads + threadIdx.x;
  if (i >= n) return;
  int p[3];
  decode3(i, tgt.d[1], tgt.d[2], tz, ty, p[0], p[1], p[2]);
  unsigned known = tgt.known[i];
  for (int c = 0; c < 3; ++c) {
    float out = tgt.val[c][i];
    if (!(known >> c & 1)) {
      float v;
      if (hier_sample(src, tgt.d, p, c, &v) > 0.0f) {
        out = v;
        known |= 1u << c;
      }
    }
    tgt.up_val[c][i] = out;
  }
  tgt.up_known[i] = (uint8_t)known;
}
// Levels of this many cells take tiles.  A lane per cell against tiles, cubic
// levels: 48^3 7.0 / 8.3 us, 64^3 8.2 / 8.6, 72^3 10.2 / 9.8, 80^3 12.0 / 12.1, 88^3
// 15.4 / 13.8, 96^3 17.3 / 15.9, 104^3 (1.1 M) 21.7 / 20.2, 128^3 34.8 / 25.1; 80 x 59 x
// 72, whose last tiles are thin, 11.6 / 15.9.  Between 0.4 and 1 M cells the two
// are within 1.6 us on cubes and tiles lose where they divide a level badly.
constexpr long long kTileCells = 1 << 20;

// The same in tiles: 113 us -> 70 on the 192^3 level.
__global__ __launch_bounds__(kThreads) void k_ex_prolong(ExSrc src, ExLevel tgt) {
  __shared__ float2 win[3 * kWin];
  int x0, y0, z0;
  if (!tile_of(tgt.d, x0, y0, z0)) return;
  const int y = y0 + (int)threadIdx.x / kTileZ, z = z0 + (int)threadIdx.x % kTileZ;
  const bool column = y < tgt.d[1] && z < tgt.d[2];
  unsigned known[kTileX];
  float val[kTileX][3];
  bool need = false;
#pragma unroll
  for (int j = 0; j < kTileX; ++j) {
    const bool in = column && x0 + j < tgt.d[0];
    const unsigned i = in ? ((unsigned)(x0 + j) * tgt.d[1] + y) * tgt.d[2] + z : 0u;
    known[j] = in ? tgt.known[i] : 7u;
#pragma unroll
    for (int c = 0; c < 3; ++c) val[j][c] = tgt.val[c][i];
    need = need || known[j] != 7u;
  }
  if (__syncthreads_or(need)) tile_fill(src, tgt.d, x0, y0, z0, win, known, val);
#pragma unroll
  for (int j = 0; j < kTileX; ++j) {
    if (!column || x0 + j >= tgt.d[0]) continue;
    const unsigned i = ((unsigned)(x0 + j) * tgt.d[1] + y) * tgt.d[2] + z;
#pragma unroll
    for (int c = 0; c < 3; ++c) tgt.up_val[c][i] = val[j][c];
    tgt.up_known[i] = (uint8_t)known[j];
  }
}

// the last prolongation onto the band result, packed into the face arrays
// (packTransportShell, …wgsl.ts:491-512): known values on open faces, 0 else.
// 990 us at 384^3 with a lane per cell, 654 in tiles, 52 -> 39.7 at
// 160 x 117 x 143, and in tiles at every size, as most tiles need no samples: 32^3
// 22 -> 11 us, 64^3 21 -> 12, 128^3 46 -> 29; 24 bytes a cell at most, 2.1 TB/s: what is left is the sums.
__global__ __launch_bounds__(kThreads) void k_ex_finish(ExGeo g, ExSrc src, int have_src, ExState r,
                                                       const uint8_t* __restrict__ cls, ExCounters* cnt,
                                                       float* __restrict__ uo, float* __restrict__ vo,
                                                       float* __restrict__ wo) {
  __shared__ float2 win[3 * kWin];
  int x0 = 0, y0 = 0, z0 = 0;
  if (!tile_of(g.d, x0, y0, z0)) return;
  const int y = y0 + (int)threadIdx.x / kTileZ, z = z0 + (int)threadIdx.x % kTileZ;
  const bool column = y < g.d[1] && z < g.d[2];
  int unknown = 0, band = 0;
  unsigned me[kTileX], known[kTileX];
  float val[kTileX][3];
  bool need = false;
#pragma unroll
  for (int j = 0; j < kTileX; ++j) {
    const bool in = column && x0 + j < g.d[0];
    const unsigned i = in ? eidx(g, x0 + j, y, z) : 0u;
    me[j] = in ? cls[i] : 0u;
    known[j] = in ? r.flags[i] & 7u : 0u;
  }
  // (the band result holds no values in the far air, most of a tank)
#pragma unroll
  for (int j = 0; j < kTileX; ++j) {
    const unsigned i = column && x0 + j < g.d[0] ? eidx(g, x0 + j, y, z) : 0u;
#pragma unroll
    for (int c = 0; c < 3; ++c) val[j][c] = 0.0f;
    if (known[j])
#pragma unroll
      for (int c = 0; c < 3; ++c) val[j][c] = r.val[c][i];
    band += __popc(known[j]);
    // a closed face is written 0 whatever the hierarchy holds
    known[j] |= ~me[j] & 7u;
    need = need || known[j] != 7u;
  }
  if (__syncthreads_or(need) && have_src) tile_fill(src, g.d, x0, y0, z0, win, known, val);
#pragma unroll
  for (int j = 0; j < kTileX; ++j) {
    const int x = x0 + j;
    if (!column || x >= g.d[0]) continue;
    const unsigned open = me[j] & 7u;
    unknown += __popc(open & ~known[j]);
    float* out[3] = {uo, vo, wo};
#pragma unroll
    for (int c = 0; c < 3; ++c) out[c][face_of(g, c, x, y, z)] = (open & known[j]) >> c & 1u ? val[j][c] : 0.0f;
    // the negative domain faces are walls
    if (x == 0) uo[(unsigned)y * g.d[2] + z] = 0.0f;
    if (y == 0) vo[(unsigned)x * (g.d[1] + 1) * g.d[2] + z] = 0.0f;
    if (z == 0) wo[((unsigned)x * g.d[1] + y) * (g.d[2] + 1)] = 0.0f;
  }
  const int su = block_sum(unknown);
  __syncthreads();
  const int sb = block_sum(band);
  if (threadIdx.x == 0) {
    if (su) atomicAdd(&cnt->unknown[blockIdx.x % kExSpread][0], (unsigned long long)su);
    if (sb) atomicAdd(&cnt->band_known[blockIdx.x % kExSpread][0], (unsigned long long)sb);
  }
}

// workgroups of a launch over a level's tiles
int tiled_grid(const int* d) {
  auto up = [](int n, int t) { return (n + t - 1) / t; };
  const int tiles = up(d[0], kTileX) * up(d[1], kTileY) * up(d[2], kTileZ);
  return 8 * ((tiles + 7) / 8);
}

// workgroups of a streaming launch over n < 2^31 items, cells per thread k
int chunked_grid(long long n, int k = 1) {
  const long long chunks = (n + (long long)kThreads * k - 1) / ((long long)kThreads * k);
  return (int)(8 * ((chunks + 7) / 8));
}

}  // namespace

Extrapolator::~Extrapolator() {
  for (void* p : allocations_) (void)hipFree(p);
}

int Extrapolator::alloc(void** p, size_t bytes) {
  bytes = (bytes + 255) & ~(size_t)255;
  if (hipMalloc(p, bytes) != hipSuccess) {
    set_error("velocity extrapolation: hipMalloc(%zu) failed", bytes);
    return FP_ERR_OUT_OF_MEMORY;
  }
  allocations_.push_back(*p);
  bytes_ += bytes;
  return FP_OK;
}

static void level_dims(int nx, int ny, int nz, std::vector<std::array<int, 3>>* out) {
  int d[3] = {nx, ny, nz};
  while (std::min(d[0], std::min(d[1], d[2])) > 1) {
    for (int a = 0; a < 3; ++a) d[a] = (d[a] + 1) / 2;
    out->push_back({d[0], d[1], d[2]});
  }
}

// Bytes on either side of a byte array that a quad's neighbour words reach
// into (one plane and a word), aligned as the array is.
static size_t quad_pad(int ny, int nz) { return ((size_t)ny * nz + 8 + 255) & ~(size_t)255; }

size_t Extrapolator::estimate_bytes(int nx, int ny, int nz) {
  auto round = [](size_t b) { return (b + 255) & ~(size_t)255; };
  const size_t n = (size_t)nx * ny * nz;
  const size_t padded = n + 2 * quad_pad(ny, nz);
  size_t total = 2 * 6 * round(n * 4) + 3 * round(n) + 3 * round(padded) + round(n * 4) +
                 round(sizeof(ExCounters) + sizeof(ExTotals));
  std::vector<std::array<int, 3>> dims;
  level_dims(nx, ny, nz, &dims);
  for (const auto& d : dims) {
    const size_t m = (size_t)d[0] * d[1] * d[2];
    total += 6 * round(m * 4) + 2 * round(m);
  }
  return total;
}

int Extrapolator::create(int nx, int ny, int nz, double h) {
  d_[0] = nx;
  d_[1] = ny;
  d_[2] = nz;
  n_ = (long long)nx * ny * nz;
  h_ = (float)h;
  const size_t n = (size_t)n_;
  int rc;
  for (int k = 0; k < 2; ++k) {
    for (int c = 0; c < 3; ++c) {
      if ((rc = alloc((void**)&st_[k].val[c], n * 4))) return rc;
      if ((rc = alloc((void**)&st_[k].dist[c], n * 4))) return rc;
    }
    if ((rc = alloc((void**)&st_[k].flags, n))) return rc;
  }
  if ((rc = alloc((void**)&st_[1].stat, n))) return rc;
  const size_t pad = quad_pad(ny, nz);
  for (uint8_t** p : {&cls_, &cand_[0], &cand_[1]}) {
    if ((rc = alloc((void**)p, n + 2 * pad))) return rc;
    *p += pad;
  }
  st_[0].stat = cand_[0];  // the last dilation is its last reader, the seed this one's first writer
  if ((rc = alloc((void**)&list_, n * 4))) return rc;
  if ((rc = alloc((void**)&counters_, sizeof(ExCounters) + sizeof(ExTotals)))) return rc;
  totals_ = reinterpret_cast<ExTotals*>(counters_ + 1);
  std::vector<std::array<int, 3>> dims;
  level_dims(nx, ny, nz, &dims);
  for (const auto& d : dims) {
    ExLevel L;
    std::memset(&L, 0, sizeof(L));
    L.d[0] = d[0];
    L.d[1] = d[1];
    L.d[2] = d[2];
    L.n = (long long)d[0] * d[1] * d[2];
    for (int c = 0; c < 3; ++c) {
      if ((rc = alloc((void**)&L.val[c], (size_t)L.n * 4))) return rc;
      if ((rc = alloc((void**)&L.up_val[c], (size_t)L.n * 4))) return rc;
    }
    if ((rc = alloc((void**)&L.known, (size_t)L.n))) return rc;
    if ((rc = alloc((void**)&L.up_known, (size_t)L.n))) return rc;
    levels_.push_back(L);
  }
  return FP_OK;
}

int Extrapolator::stage_host() { return in_ ? FP_OK : alloc((void**)&in_, host_bytes(d_[0], d_[1], d_[2])); }

size_t Extrapolator::host_bytes(int nx, int ny, int nz) {
  const size_t faces = (size_t)(nx + 1) * ny * nz + (size_t)nx * (ny + 1) * nz + (size_t)nx * ny * (nz + 1);
  return (faces * 4 + 255) & ~(size_t)255;
}

int Extrapolator::run(hipStream_t s, const fp_extrapolate_args* a, fp_extrapolate_report* rep, bool same_band) {
  const auto t0 = std::chrono::steady_clock::now();
  const int nx = d_[0], ny = d_[1], nz = d_[2];
  const long long n = n_;
  const size_t nu = (size_t)(nx + 1) * ny * nz, nv = (size_t)nx * (ny + 1) * nz, nw = (size_t)nx * ny * (nz + 1);
  if ((long long)(nx + 1) * ny * nz >= (1ll << 31) || (long long)nx * (ny + 1) * nz >= (1ll << 31) ||
      (long long)nx * ny * (nz + 1) >= (1ll << 31)) {
    set_error("fp_extrapolate_velocity: grids of 2^31 or more faces per component are not supported");
    return FP_ERR_UNSUPPORTED;
  }
  const float* field = a->phi ? a->phi : a->density;
  const float *u = a->u, *v = a->v, *w = a->w;
  // kernels write device memory only: host outputs go through the input
  // staging (free once the seed has read the inputs) and are copied back
  float *uo = a->u_out, *vo = a->v_out, *wo = a->w_out;
  if (a->memory == FP_MEMORY_HOST) {
    const int rc = stage_host();
    if (rc) return rc;
    float* f = st_[1].val[0];  // read by the classification only, written by the seed after it
    float* hu = in_;
    float* hv = hu + nu;
    float* hw = hv + nv;
    HIPCHK(hipMemcpyAsync(f, field, (size_t)n * 4, hipMemcpyHostToDevice, s));
    HIPCHK(hipMemcpyAsync(hu, u, nu * 4, hipMemcpyHostToDevice, s));
    HIPCHK(hipMemcpyAsync(hv, v, nv * 4, hipMemcpyHostToDevice, s));
    HIPCHK(hipMemcpyAsync(hw, w, nw * 4, hipMemcpyHostToDevice, s));
    field = f;
    u = hu;
    v = hv;
    w = hw;
    uo = hu;
    vo = hv;
    wo = hw;
  }
  ExGeo g;
  g.d[0] = nx;
  g.d[1] = ny;
  g.d[2] = nz;
  g.h = h_;
  g.open_top = a->open_top ? 1 : 0;
  g.dz = make_div((unsigned)nz);
  g.dy = make_div((unsigned)ny);
  g.eps_min = 2.0f * h_;
  {
    const float dx = (float)nx * h_, dy = (float)ny * h_, dz = (float)nz * h_;
    g.eps_max = std::sqrt((dx * dx + dy * dy) + dz * dz);
  }
  int ceiling = std::min(std::max(nx, std::max(ny, nz)), 16);
  if (a->max_passes > 0) ceiling = std::min(a->max_passes, 19);
  const dim3 grid(chunked_grid(n, kCells)), block(kThreads);
  HIPCHK(hipMemsetAsync(counters_, 0, sizeof(ExCounters), s));
  const unsigned un = (unsigned)n;
  same_band = same_band && band_count_ >= 0;
  if (!same_band) {
    hipLaunchKernelGGL(k_ex_classify, grid, block, 0, s, g, field, a->phi ? 1 : 0, cls_, cand_[0], un);
    hipLaunchKernelGGL(k_ex_dilate, grid, block, 0, s, g, (const uint8_t*)cls_, (const uint8_t*)cand_[0], cand_[1],
                       0, list_, counters_, un);
    hipLaunchKernelGGL(k_ex_dilate, grid, block, 0, s, g, (const uint8_t*)cls_, (const uint8_t*)cand_[1], cand_[0],
                       0, list_, counters_, un);
    hipLaunchKernelGGL(k_ex_dilate, grid, block, 0, s, g, (const uint8_t*)cls_, (const uint8_t*)cand_[0], cand_[1],
                       1, list_, counters_, un);
  }
  hipLaunchKernelGGL(k_ex_seed, grid, block, 0, s, g, (const uint8_t*)cls_, (const uint8_t*)cand_[1], u, v, w,
                     st_[0], st_[1], counters_, un);
  if (!same_band) {
    int listed = 0;
    HIPCHK(hipMemcpyAsync(&listed, &counters_->list_count, sizeof(int), hipMemcpyDeviceToHost, s));
    HIPCHK(hipStreamSynchronize(s));
    band_count_ = listed;
  }
  const int count = band_count_;
  if (count > 0) {
    // one launch more than passes: it counts the faces left active
    for (int pass = 1; pass <= ceiling + 1; ++pass)
      hipLaunchKernelGGL(k_ex_pass, dim3((count + 63) / 64), dim3(3 * 64), 0, s, g, (const uint8_t*)cls_,
                         (const int*)list_, count, st_[(pass - 1) & 1], st_[pass & 1], counters_, pass,
                         pass > ceiling ? 1 : 0);
    hipLaunchKernelGGL(k_ex_resolve, dim3((count + kThreads - 1) / kThreads), block, 0, s, (const int*)list_, count,
                       st_[0], st_[1], (const ExCounters*)counters_);
  }
  // hierarchy: restrict down, prolong up, the last prolongation fused with the packing
  const int L = (int)levels_.size();
  const ExSrc none{{0, 0, 0}, {nullptr, nullptr, nullptr}, nullptr};
  for (int l = 0; l < L; ++l) {
    const ExLevel& T = levels_[l];
    ExSrc src{{nx, ny, nz}, {st_[0].val[0], st_[0].val[1], st_[0].val[2]}, st_[0].flags};
    if (l > 0) {
      const ExLevel& S = levels_[l - 1];
      src = ExSrc{{S.d[0], S.d[1], S.d[2]}, {S.val[0], S.val[1], S.val[2]}, S.known};
    }
    hipLaunchKernelGGL(k_ex_restrict, dim3(chunked_grid(T.n)), block, 0, s, src, T, make_div((unsigned)T.d[2]),
                       make_div((unsigned)T.d[1]));
  }
  ExSrc coarser = none;
  if (L > 0) {
    const ExLevel& C = levels_[L - 1];
    coarser = ExSrc{{C.d[0], C.d[1], C.d[2]}, {C.val[0], C.val[1], C.val[2]}, C.known};
  }
  for (int l = L - 2; l >= 0; --l) {
    const ExLevel& T = levels_[l];
    if (T.n >= kTileCells)
      hipLaunchKernelGGL(k_ex_prolong, dim3(tiled_grid(T.d)), block, 0, s, coarser, T);
    else
      hipLaunchKernelGGL(k_ex_prolong_cells, dim3(chunked_grid(T.n)), block, 0, s, coarser, T,
                         make_div((unsigned)T.d[2]), make_div((unsigned)T.d[1]));
    coarser = ExSrc{{T.d[0], T.d[1], T.d[2]}, {T.up_val[0], T.up_val[1], T.up_val[2]}, T.up_known};
  }
  hipLaunchKernelGGL(k_ex_finish, dim3(tiled_grid(d_)), block, 0, s, g, coarser, L > 0 ? 1 : 0, st_[0],
                     (const uint8_t*)cls_, counters_, uo, vo, wo);
  if (a->memory == FP_MEMORY_HOST) {
    HIPCHK(hipMemcpyAsync(a->u_out, uo, nu * 4, hipMemcpyDeviceToHost, s));
    HIPCHK(hipMemcpyAsync(a->v_out, vo, nv * 4, hipMemcpyDeviceToHost, s));
    HIPCHK(hipMemcpyAsync(a->w_out, wo, nw * 4, hipMemcpyDeviceToHost, s));
  }
  ExTotals host;
  hipLaunchKernelGGL(k_ex_totals, dim3(1), dim3(64), 0, s, (const ExCounters*)counters_, totals_);
  HIPCHK(hipMemcpyAsync(&host, totals_, sizeof(ExTotals), hipMemcpyDeviceToHost, s));
  HIPCHK(hipStreamSynchronize(s));
  if (rep) {
    std::memset(rep, 0, sizeof(*rep));
    int passes = 0;
    for (int k = 1; k <= ceiling; ++k)
      if (host.active[k - 1] > 0) passes = k;
    rep->passes = count > 0 ? passes : 0;
    rep->active_left = rep->passes > 0 ? host.active[rep->passes] : host.active[0];
    rep->levels = L;
    rep->band_faces = (int64_t)host.band_known;
    rep->unknown_faces = (int64_t)host.unknown;
    rep->device_ms = std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
  }
  return FP_OK;
}

}  // namespace fp

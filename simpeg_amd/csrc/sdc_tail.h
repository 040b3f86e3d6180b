// The coarse end of the multigrid cycle in one launch.
//
// The coarse levels are small (38,088 + 7,406 + 1,352 + 245 + 48 nodes below a 932,137-node mesh),
// so launches of their own for each smoothing step, residual and transfer cost 4-10 us apiece
// whatever they do.  Here one work-group of 1,024 owns one right-hand-side column and runs the
// cycle of every level from the first with at most SDC_TAIL_NODES nodes on (the finest itself on
// small meshes), the W step included, as one launch; the column's rhs is read once from HBM, the
// solution written once.  The arithmetic is the multi-launch cycle's: Chebyshev steps on the same
// interval (three-term form), the same P and the 27-point P^T, the dense inverse on the coarsest
// level.
//
// What bounds it is latency: a step is a few hundred LDS reads per wave between two barriers, so
// no step may wait for L2.  The top level's coefficients stay in registers from the first step to
// the last (up to 8 nodes a work-item; 1,024 work-items fill the register file at 128 each, and the
// form of 8 nodes, for top levels of more than 4,096, is over it by 6 to 16 registers that live
// in scratch memory), with the rows scaled by the inverse diagonal: six weights,
// A' x = x - sum w x_nbr.  Its iterate is the only top-level vector in LDS.  The lower levels'
// scaled coefficients, their interpolation weights and the transfers' tables come into LDS with
// one copy of an image that k_tail_pack lays out when the operator is set.  With the coefficients read from L2 in every step (the form
// before) the levels of 7,406 + 1,352 + 245 + 48 nodes took 59-86 us per launch, now 33 (3 columns)
// to 38 (128); of that 5 us load the 350 KB of image and coefficients, 2-3 us go to each step of
// the top level and 1-2 us to each step of a lower one.
#pragma once
#include "sdc_kernels.h"

#define SDC_TAIL_MAX 6
#define SDC_TAIL_THREADS 1024
#define SDC_TAIL_NODES 8192  // most nodes of the top level (8 per work-item)
#define SDC_TAIL_PROG 80     // most steps of a cycle: 5 levels, the W step's coarse part twice

// One level: shape and LDS offsets (in floats).  x and y point at node 0 with a zeroed halo of one
// plane on either side, so a missing neighbour (weight 0) reads a finite value.  The top level
// (index 0) has x only.
struct TailLev {
  uint32_t nN, n1x, plane;
  uint32_t coef;  // wxm, wxp, wym, wyp, wzm, wzp, 1/diagonal: 7 arrays of nN
  uint32_t b, x, y;
};

// Transfer between level l and l + 1: strides of the grids, the LDS offset of its table (two
// words per coarse node, tail_table_entry; the top level's is read from global memory) and where
// its interpolation weights start (Xfer::wx, wy, wz one after the other): LDS offset w.  The top
// level's weights are laid out per coarse node in the image instead (SDC_TAIL_WR for the
// restriction, SDC_TAIL_WP for the interpolation, each an array over the coarse nodes): read from
// L2 point by point, 9 gathers of stride 2 per work-item, they took 20,000 of a launch's 77,000
// clocks on 7,406 + 1,352 nodes.
#define SDC_TAIL_WR 27
#define SDC_TAIL_WP 12
struct TailXf {
  uint32_t fn1x, fplane, cn1x, cplane, cN;
  uint32_t ys;         // cn1x * fn1y: plane stride of the Py grid
  uint32_t nwx, nwy;   // sizes of the first two weight arrays
  uint32_t tab, w;
};

// Table entry of a coarse node: its fine index and six flags (the fine neighbour below / above it
// along x, y, z exists and lies between coarse nodes), and its index on the Py and Pz grids.  The
// transfers decode positions from it: with divisions and lookups per axis instead they were bound
// by 16-cycle integer multiplies (20,000 of a cycle's 85,000 clocks on 7,406 + 1,352 nodes).
__host__ __device__ inline uint2 tail_table_entry(uint32_t fine, uint32_t flags, uint32_t py,
                                                  uint32_t pz) {
  return uint2{fine | flags << 13, py | pz << 16};
}

// a step of the cycle: what, on which level
enum TailOp : uint8_t {
  TAIL_PRE,     // pre-smoothing from a zero guess
  TAIL_DOWN,    // residual and its restriction into the next level's rhs
  TAIL_DENSE,   // coarsest level
  TAIL_UP,      // interpolate the next level's solution into this one's
  TAIL_MID,     // smoothing between the two coarse corrections of the W step
  TAIL_POST     // post-smoothing
};

struct TailDesc {
  TailLev lv[SDC_TAIL_MAX];
  TailXf xf[SDC_TAIL_MAX - 1];
  uint8_t op[SDC_TAIL_PROG], lev[SDC_TAIL_PROG];
  int nop;
  // operator image (per set, imgs floats apart): 8 arrays of NPT * SDC_TAIL_THREADS floats of the
  // top level (the six weights, 1/diagonal, diagonal; entries past its nodes are 0, so the kernel
  // needs no bounds), then nimg floats for LDS offset 0, then the top transfer's weights
  // (SDC_TAIL_WR + SDC_TAIL_WP arrays).  Tables: the top transfer's (ntop words), then ntab words
  // for LDS offset nimg.  The rest of the nlds floats is cleared.  nimg, ntop, ntab and nlds are
  // multiples of 4.
  const float* img;
  size_t imgs;
  const float* tab;
  uint32_t nimg, ntop, ntab, nlds;
  const float* ainv;  // coarsest dense inverse, nn x nn, symmetric
  uint32_t astride;
  int nn;
  const int32_t* cset;  // operator sets: column c uses set cset[c] (null: one set)
  int nu_pre, nu_post, nu_mid;
  float c1[16], c2[16];
};

// What k_tail_pack lays out: the non-coarsest levels' operators and the weights of their
// transfers: operator-dependent, a weight per grid point (d0 = 1, d1 beyond the grid), or geometric,
// the axis table spread over the same grid (d0, d1: strides that give the axis coordinate).
struct TailPack {
  Sten<float> s[SDC_TAIL_MAX - 1];
  uint32_t coef[SDC_TAIL_MAX - 1];  // image offset of the level's coefficients
  struct W {
    const float* src;  // of set z at src + z * stride, point i at entry (i / d0) % d1
    uint32_t n, stride, dst, d0, d1;
    // no branch: with the choice between the two forms and between the axes made here, the
    // compiler left the base register of one path undefined
    __device__ __forceinline__ float at(size_t set, uint32_t i) const {
      const uint32_t c = i / d0;
      return src[set * stride + (c - c / d1 * d1)];
    }
  } w[3 * (SDC_TAIL_MAX - 1)];
  int nlev, nw;   // levels (without the coarsest), weight arrays (the first three: top transfer)
  const uint2* tab;  // the top transfer's table and strides
  TailXf x0;
  uint32_t top;      // image offset of its weights
  uint32_t rows;  // length of the top level's arrays
  float* img;
  size_t imgs;
};

// Grid: (blocks of 256; levels, the top transfer, the lower ones' weight arrays; operator sets)
__global__ __launch_bounds__(SDC_BLOCK) void k_tail_pack(TailPack p) {
  const uint32_t n = blockIdx.x * SDC_BLOCK + threadIdx.x;
  const int y = (int)blockIdx.y;
  const size_t set = blockIdx.z;
  float* img = p.img + set * p.imgs;
  if (y < p.nlev) {
    Sten<float> s = p.s[y];
    float* dst = img + p.coef[y];
    const size_t len = y == 0 ? p.rows : s.nN;
    if (n >= len) return;
    if (n >= s.nN) {
#pragma unroll
      for (int k = 0; k < 8; ++k) dst[k * len + n] = 0.0f;
      return;
    }
    const size_t o = set * s.sstride;
    s.cx += o;
    s.cy += o;
    s.cz += o;
    s.rd += o;
    s.idg += o;
    const NodeC<float> c = node_coef(s, n);
    const float g = s.idg[n];
    const float w[6] = {c.wxm * g, c.wxp * g, c.wym * g, c.wyp * g, c.wzm * g, c.wzp * g};
#pragma unroll
    for (int k = 0; k < 6; ++k) dst[k * len + n] = w[k];
    dst[6 * len + n] = g;
    if (y == 0) dst[7 * len + n] = 1.0f / g;
    return;
  }
  if (y > p.nlev) {
    const TailPack::W& a = p.w[y - p.nlev + 2];
    if (n < a.n) img[a.dst + n] = a.at(set, n);
    return;
  }
  // the top transfer per coarse node: the 27 restriction weights (plane by plane, row by row), then
  // the weights of the owned nodes along x (4 rows), y (2 planes x 2 x parents) and z (4 parents)
  if (n >= p.x0.cN) return;
  const TailXf& X = p.x0;
  const TailPack::W &wx = p.w[0], &wy = p.w[1], &wz = p.w[2];
  const uint2 t = p.tab[n];
  const bool lo[3] = {(t.x >> 13 & 1u) != 0, (t.x >> 15 & 1u) != 0, (t.x >> 17 & 1u) != 0};
  const bool hi[3] = {(t.x >> 14 & 1u) != 0, (t.x >> 16 & 1u) != 0, (t.x >> 18 & 1u) != 0};
  const uint32_t f = t.x & 8191u, py = t.y & 65535u, pz = t.y >> 16;
  float* dst = img + p.top + n;
  for (int c = 0; c < 3; ++c) {
    const bool oz = c == 0 ? lo[2] : c == 1 || hi[2];
    const int dk = oz ? c - 1 : 0;
    const float z = c == 1 ? 1.0f : !oz ? 0.0f : c == 0 ? wz.at(set, pz - X.cplane)
                                                       : 1.0f - wz.at(set, pz + X.cplane);
    for (int b = 0; b < 3; ++b) {
      const bool oy = b == 0 ? lo[1] : b == 1 || hi[1];
      const int dj = oy ? b - 1 : 0;
      const uint32_t yi = py + (uint32_t)(dk * (int)X.ys + dj * (int)X.cn1x);
      const float yv = b == 1 ? 1.0f : !oy ? 0.0f : b == 0 ? wy.at(set, yi) : 1.0f - wy.at(set, yi);
      const uint32_t row = f + (uint32_t)(dk * (int)X.fplane + dj * (int)X.fn1x);
      const float x0 = lo[0] ? wx.at(set, row - 1) : 0.0f;
      const float x2 = hi[0] ? 1.0f - wx.at(set, row + 1) : 0.0f;
      dst[(size_t)(9 * c + 3 * b) * X.cN] = z * yv * x0;
      dst[(size_t)(9 * c + 3 * b + 1) * X.cN] = z * yv;
      dst[(size_t)(9 * c + 3 * b + 2) * X.cN] = z * yv * x2;
    }
  }
  dst += (size_t)SDC_TAIL_WR * X.cN;
  const uint32_t dx = hi[0] ? 1u : 0u, dy = hi[1] ? X.cn1x : 0u, dz = hi[2] ? X.cplane : 0u;
  const uint32_t f1 = hi[1] ? X.fn1x : 0u, f2 = hi[2] ? X.fplane : 0u, y2 = hi[2] ? X.ys : 0u;
  const float v[SDC_TAIL_WP] = {
      wx.at(set, f + dx),           wx.at(set, f + f1 + dx),      wx.at(set, f + f2 + dx),
      wx.at(set, f + f1 + f2 + dx), wy.at(set, py + dy),          wy.at(set, py + dy + dx),
      wy.at(set, py + dy + y2),     wy.at(set, py + dy + y2 + dx), wz.at(set, pz + dz),
      wz.at(set, pz + dz + dx),     wz.at(set, pz + dz + dy),     wz.at(set, pz + dz + dy + dx)};
#pragma unroll
  for (int k = 0; k < SDC_TAIL_WP; ++k) dst[(size_t)k * X.cN] = v[k];
}

namespace tail {

// element i of an array in global memory, addressed by a 32-bit byte offset from its start
__device__ __forceinline__ float at(const float* p, uint32_t i) {
  return *(const float*)((const char*)p + (uint32_t)(i * 4u));
}

// bc = P^T r: the 27 fine nodes around every coarse node, those that lie between coarse nodes
// with their interpolation weight (restrict_weights).  One work-item per coarse node and fine
// plane (9 points), the planes' sums in bc, p1 and p2 added afterwards.  w: the transfer's
// weights, in LDS, or per coarse node in the image (TOP).
template <bool TOP>
__device__ __forceinline__ void restrict_to(const TailXf& X, const uint2* tab, const float* r,
                                            float* bc, float* p1, float* p2, const float* w) {
  const float* wy = w + X.nwx;
  const float* wz = wy + X.nwy;
  for (uint32_t e = threadIdx.x; e < 3 * X.cN; e += SDC_TAIL_THREADS) {
    const uint32_t c = (uint32_t)(e >= X.cN) + (uint32_t)(e >= 2 * X.cN);
    const uint32_t n = e - c * X.cN;
    const uint2 t = tab[n];
    const bool xl = t.x & 1u << 13, xh = t.x & 1u << 14, yl = t.x & 1u << 15,
               yh = t.x & 1u << 16, zl = t.x & 1u << 17, zh = t.x & 1u << 18;
    uint32_t f = t.x & 8191u, py = t.y & 65535u, pz = t.y >> 16;
    const bool on = c == 0 ? zl : c == 1 || zh;
    if (c == 0 && zl) {
      f -= X.fplane;
      py -= X.ys;
      pz -= X.cplane;
    } else if (c == 2 && zh) {
      f += X.fplane;
      py += X.ys;
      pz += X.cplane;
    }
    const uint32_t f0 = yl ? f - X.fn1x : f, f2 = yh ? f + X.fn1x : f;
    const uint32_t il = xl ? 1u : 0u, ih = xh ? 1u : 0u;
    const uint32_t row[3] = {f0, f, f2};
    float acc = 0.0f;
    if (TOP) {
      const uint32_t g0 = 9 * c * X.cN + n;
      float g[9];
#pragma unroll
      for (int q = 0; q < 9; ++q) g[q] = at(w, g0 + q * X.cN);
#pragma unroll
      for (int q = 0; q < 3; ++q)
        acc += g[3 * q] * r[row[q] - il] + g[3 * q + 1] * r[row[q]] + g[3 * q + 2] * r[row[q] + ih];
    } else if (on) {
      const float wv = wz[pz], y0 = wy[yl ? py - X.cn1x : py], y2 = wy[yh ? py + X.cn1x : py];
      float a[3], b[3], v[3];
#pragma unroll
      for (int q = 0; q < 3; ++q) {
        a[q] = w[row[q] - il];
        b[q] = w[row[q] + ih];
      }
#pragma unroll
      for (int q = 0; q < 3; ++q)
        v[q] = r[row[q]] + (xl ? a[q] * r[row[q] - il] : 0.0f) +
               (xh ? (1.0f - b[q]) * r[row[q] + ih] : 0.0f);
      const float z = c == 0 ? wv : c == 1 ? 1.0f : 1.0f - wv;
      acc = z * (v[1] + (yl ? y0 * v[0] : 0.0f) + (yh ? (1.0f - y2) * v[2] : 0.0f));
    }
    (c == 0 ? bc : c == 1 ? p1 : p2)[n] = acc;
  }
  __syncthreads();
  for (uint32_t n = threadIdx.x; n < X.cN; n += SDC_TAIL_THREADS) bc[n] += p1[n] + p2[n];
  __syncthreads();
}

// xf += P xc, one work-item per coarse node updating the up to 8 fine nodes it owns (as
// k_prolong_own).
template <bool TOP>
__device__ __forceinline__ void prolong_add(const TailXf& X, const uint2* tab, const float* xc,
                                            float* xf, const float* w) {
  const float* wy = w + X.nwx;
  const float* wz = wy + X.nwy;
  for (uint32_t n = threadIdx.x; n < X.cN; n += SDC_TAIL_THREADS) {
    const uint2 t = tab[n];
    // owned nodes per axis: 2 where the coarse cell spans 2 fine cells; elsewhere the second one
    // (and the next coarse node) is the first again and its update is left out
    const bool ox = t.x & 1u << 14, oy = t.x & 1u << 16, oz = t.x & 1u << 18;
    const uint32_t f = t.x & 8191u, py = t.y & 65535u, pz = t.y >> 16;
    const uint32_t dx = ox ? 1u : 0u, dy = oy ? X.cn1x : 0u, dz = oz ? X.cplane : 0u;
    const float* c = xc + n;
    const float v[8] = {c[0],  c[dx],      c[dy],      c[dy + dx],
                        c[dz], c[dz + dx], c[dz + dy], c[dz + dy + dx]};
    const uint32_t fy1 = oy ? X.fn1x : 0u, fz1 = oz ? X.fplane : 0u;
    const uint32_t row[4] = {f, f + fy1, f + fz1, f + fy1 + fz1};
    const uint32_t ya = py + dy, yb = ya + (oz ? X.ys : 0u), za = pz + dz;
    float fx[4], fy[2][2], fz[4];
    if (TOP) {
      const uint32_t g0 = SDC_TAIL_WR * X.cN + n;
#pragma unroll
      for (int m = 0; m < 4; ++m) {
        fx[m] = at(w, g0 + m * X.cN);
        fy[m >> 1][m & 1] = at(w, g0 + (4 + m) * X.cN);
        fz[m] = at(w, g0 + (8 + m) * X.cN);
      }
    } else {
#pragma unroll
      for (int m = 0; m < 4; ++m) fx[m] = w[row[m] + dx];
      fy[0][0] = wy[ya];
      fy[0][1] = wy[ya + dx];
      fy[1][0] = wy[yb];
      fy[1][1] = wy[yb + dx];
      fz[0] = wz[za];
      fz[1] = wz[za + dx];
      fz[2] = wz[za + dy];
      fz[3] = wz[za + dy + dx];
    }
#pragma unroll
    for (int cz = 0; cz < 2; ++cz) {
      if (cz && !oz) break;
      // the four (x, y) parents at this fine z
      float p[4];
#pragma unroll
      for (int m = 0; m < 4; ++m) p[m] = cz ? v[m] + fz[m] * (v[m + 4] - v[m]) : v[m];
#pragma unroll
      for (int by = 0; by < 2; ++by) {
        if (by && !oy) continue;
        const float q0 = by ? p[0] + fy[cz][0] * (p[2] - p[0]) : p[0];
        const float q1 = by ? p[1] + fy[cz][1] * (p[3] - p[1]) : p[1];
        const uint32_t i = row[by + 2 * cz];
        xf[i] += q0;
        if (ox) xf[i + 1] += q0 + fx[by + 2 * cz] * (q1 - q0);
      }
    }
  }
}

// sum of w x_nbr at node n of a lower level (weights: 6 LDS arrays of nN from w)
__device__ __forceinline__ float nbr_sum(const TailLev& L, const float* w, const float* x,
                                         uint32_t n) {
  const float* xn = x + n;
  const int n1 = (int)L.n1x, pl = (int)L.plane;
  return w[n] * xn[-1] + w[L.nN + n] * xn[1] + w[2 * L.nN + n] * xn[-n1] +
         w[3 * L.nN + n] * xn[n1] + w[4 * L.nN + n] * xn[-pl] + w[5 * L.nN + n] * xn[pl];
}

}  // namespace tail

// One cycle of the tail levels per column: x = M^-1 b, b and x column blockIdx.x of the top
// level's blocks (types B, O, column stride ld).  NPT: top-level nodes per work-item.  partial
// non-null: also b.x (with x as stored) per column, one partial each.
template <typename B, typename O, int NPT>
__global__ __launch_bounds__(SDC_TAIL_THREADS) void k_tail_cycle(TailDesc d,
                                                                 const B* __restrict__ b,
                                                                 O* __restrict__ x, size_t ld,
                                                                 double* __restrict__ partial,
                                                                 const int* __restrict__ done) {
  if (done && ld_flag(done)) return;
  extern __shared__ __align__(16) float lds[];
  typedef float f4 __attribute__((ext_vector_type(4)));
  constexpr uint32_t NT = SDC_TAIL_THREADS;
  const uint32_t tid = threadIdx.x;
  const size_t col = blockIdx.x;
  const size_t set = d.cset ? (size_t)d.cset[col] : (size_t)0;
  const float* img = d.img + set * d.imgs;
  const uint32_t nN = d.lv[0].nN;
  const float* ainv = d.ainv + set * d.astride;
  const B* bc = b + col * ld;

  constexpr uint32_t ROWS = NPT * NT;
  // lower levels' image and all tables into LDS, the vectors' part cleared
  {
    const f4* src = (const f4*)(img + 8 * ROWS);
    const f4* tab = (const f4*)(d.tab + d.ntop);
    f4* dst = (f4*)lds;
    const uint32_t ni = d.nimg / 4, nt = ni + d.ntab / 4, nl = d.nlds / 4;
    for (uint32_t e0 = tid; e0 < nt; e0 += 4 * NT) {
      f4 v[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const uint32_t e = e0 + u * NT;
        if (e < nt) v[u] = e < ni ? src[e] : tab[e - ni];
      }
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const uint32_t e = e0 + u * NT;
        if (e < nt) dst[e] = v[u];
      }
    }
    for (uint32_t e = nt + tid; e < nl; e += NT) dst[e] = f4(0.0f);
  }
  // top level: scaled weights and scaled rhs into registers; xs holds the previous iterate while
  // smoothing (the current one is in X) and the current one while X holds something else
  float wxm[NPT], wxp[NPT], wym[NPT], wyp[NPT], wzm[NPT], wzp[NPT], bs[NPT], xs[NPT];
#pragma unroll
  for (int k = 0; k < NPT; ++k) {
    const float* im = img + k * NT;
    wxm[k] = im[tid];
    wxp[k] = im[ROWS + tid];
    wym[k] = im[2 * ROWS + tid];
    wyp[k] = im[3 * ROWS + tid];
    wzm[k] = im[4 * ROWS + tid];
    wzp[k] = im[5 * ROWS + tid];
    bs[k] = im[6 * ROWS + tid] * (float)bc[min(tid + k * NT, nN - 1)];
    xs[k] = 0.0f;
  }
  __syncthreads();

  const float* const topw = img + 8 * ROWS + d.nimg;
  float* const X = lds + d.lv[0].x;
  const int n1 = (int)d.lv[0].n1x, pl = (int)d.lv[0].plane;

  // b' - A' x of the top level at this work-item's nodes
  auto top_res = [&](float(&t)[NPT]) {
#pragma unroll
    for (int k = 0; k < NPT; ++k) {
      const float* xn = X + tid + k * NT;
      t[k] = bs[k] - xn[0] + wxm[k] * xn[-1] + wxp[k] * xn[1] + wym[k] * xn[-n1] +
             wyp[k] * xn[n1] + wzm[k] * xn[-pl] + wzp[k] * xn[pl];
      // at most two nodes' reads in flight: all 56 at once moved the weights to scratch memory
      if (k & 1) asm volatile("" ::: "memory");
    }
  };
  auto top_store = [&](const float(&v)[NPT]) {
    __syncthreads();
#pragma unroll
    for (int k = 0; k < NPT; ++k) X[tid + k * NT] = v[k];
    __syncthreads();
  };
  auto top_step = [&](float c1, float c2) {
    float t[NPT];
    top_res(t);
#pragma unroll
    for (int k = 0; k < NPT; ++k) {
      const float xc = X[tid + k * NT];
      t[k] = xc + c1 * (xc - xs[k]) + c2 * t[k];
      xs[k] = xc;
    }
    top_store(t);
  };
  // lower levels: which of x, y holds the current iterate (bit l: y)
  uint32_t cur = 0;
  auto low_x = [&](int l) { return lds + ((cur >> l) & 1u ? d.lv[l].y : d.lv[l].x); };
  auto low_o = [&](int l) { return lds + ((cur >> l) & 1u ? d.lv[l].x : d.lv[l].y); };
  auto low_step = [&](int l, float c1, float c2, bool prev) {
    const TailLev& L = d.lv[l];
    const float* w = lds + L.coef;
    const float* B_ = lds + L.b;
    const float* xc = low_x(l);
    float* o = low_o(l);
    for (uint32_t n = tid; n < L.nN; n += NT) {
      const float v = xc[n];
      const float g = w[6 * L.nN + n];
      const float t = g * B_[n] - v + tail::nbr_sum(L, w, xc, n);
      o[n] = v + c1 * (v - (prev ? o[n] : 0.0f)) + c2 * t;
    }
    __syncthreads();
    cur ^= 1u << l;
  };

  for (int pc = 0; pc < d.nop; ++pc) {
    const int op = d.op[pc], l = d.lev[pc];
    if (op == TAIL_PRE) {
      if (l == 0) {
        float t[NPT];
#pragma unroll
        for (int k = 0; k < NPT; ++k) {
          xs[k] = 0.0f;
          t[k] = d.c2[0] * bs[k];
        }
        top_store(t);
        for (int k = 1; k < d.nu_pre; ++k) top_step(d.c1[k], d.c2[k]);
      } else {
        const TailLev& L = d.lv[l];
        cur &= ~(1u << l);
        float* xl = lds + L.x;
        for (uint32_t n = tid; n < L.nN; n += NT)
          xl[n] = d.c2[0] * lds[L.coef + 6 * L.nN + n] * lds[L.b + n];
        __syncthreads();
        for (int k = 1; k < d.nu_pre; ++k) low_step(l, d.c1[k], d.c2[k], k >= 2);
      }
    } else if (op == TAIL_DOWN) {
      const TailXf& T = d.xf[l];
      // the next level's iterates are not in use yet: two of the restriction's partial sums
      float* bn = lds + d.lv[l + 1].b;
      float* p1 = lds + d.lv[l + 1].x;
      float* p2 = lds + d.lv[l + 1].y;
      if (l == 0) {
        float t[NPT];
        top_res(t);
#pragma unroll
        for (int k = 0; k < NPT; ++k) {
          t[k] *= img[7 * ROWS + k * NT + tid];
          xs[k] = X[tid + k * NT];
        }
        top_store(t);
        tail::restrict_to<true>(T, (const uint2*)d.tab, X, bn, p1, p2, topw);
      } else {
        const TailLev& L = d.lv[l];
        const float* w = lds + L.coef;
        const float* xc = low_x(l);
        float* o = low_o(l);
        for (uint32_t n = tid; n < L.nN; n += NT) {
          const float g = w[6 * L.nN + n];
          o[n] = (g * lds[L.b + n] - xc[n] + tail::nbr_sum(L, w, xc, n)) / g;
        }
        __syncthreads();
        tail::restrict_to<false>(T, (const uint2*)(lds + T.tab), o, bn, p1, p2, lds + T.w);
      }
    } else if (op == TAIL_DENSE) {
      // 16 work-items per row, partial sums over columns m = part + 16 j
      const float* bl = lds + d.lv[l].b;
      float* xl = lds + d.lv[l].x;
      const int part = (int)(tid & 15u);
      for (int r0 = 0; r0 < d.nn; r0 += (int)(NT / 16)) {
        const int r = r0 + (int)(tid >> 4);
        float acc = 0.0f;
        if (r < d.nn) {
#pragma unroll 4
          for (int m = part; m < d.nn; m += 16) acc += ainv[(size_t)r * d.nn + m] * bl[m];
        }
#pragma unroll
        for (int s = 8; s > 0; s >>= 1) acc += __shfl_xor(acc, s, 64);
        if (part == 0 && r < d.nn) xl[r] = acc;
      }
      __syncthreads();
    } else if (op == TAIL_UP) {
      const TailXf& T = d.xf[l];
      const float* xc = low_x(l + 1);
      if (l == 0) {
        top_store(xs);
        tail::prolong_add<true>(T, (const uint2*)d.tab, xc, X, topw);
        __syncthreads();
      } else {
        tail::prolong_add<false>(T, (const uint2*)(lds + T.tab), xc, low_x(l), lds + T.w);
        __syncthreads();
      }
    } else {
      const int ns = op == TAIL_MID ? d.nu_mid : d.nu_post;
      for (int k = 0; k < ns; ++k) {
        const float c1 = k == 0 ? 0.0f : d.c1[k];
        if (l == 0)
          top_step(c1, d.c2[k]);
        else
          low_step(l, c1, d.c2[k], k >= 1);
      }
    }
  }

  O* xcol = x + col * ld;
  double acc = 0.0;
#pragma unroll
  for (int k = 0; k < NPT; ++k) {
    const uint32_t n = tid + k * NT;
    if (n < nN) {
      const O v = (O)X[n];
      xcol[n] = v;
      if (partial) acc += (double)(float)bc[n] * (double)(float)v;
    }
  }
  if (partial) {
    double* red = (double*)lds;  // free: nothing but X is read after the last step
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) acc += __shfl_down(acc, off, 64);
    __syncthreads();
    if ((tid & 63u) == 0) red[tid >> 6] = acc;
    __syncthreads();
    if (tid == 0) {
      double t = 0.0;
      for (uint32_t w = 0; w < NT / 64; ++w) t += red[w];
      partial[col] = t;
    }
  }
}

// The xy slab transform on matrix cores: one wavefront takes one z plane of
// one band from its sticks to its sticks, every intermediate in registers.
//
// r(x, y) real is split by parity in x and in y.  With th_x = 2 pi / n1,
// th_y = 2 pi / n2, E = Y(kx, ky) + Y(kx, -ky), O = Y(kx, ky) - Y(kx, -ky)
// and c = 1 for kx = 0 and kx = n1 / 2, else 2, the four class matrices
//   ee = c Re E,  oe = -c Im E,  eo = -c Im O,  oo = -c Re O   (x, y parity)
// over 0 <= kx <= kxmax, 0 <= ky <= kymax give r as four REAL products
//   r_ab = Ca_x A_ab Cb_y^T,   Ce = cos(th h k), Co = sin(th h k),
//   r(+-x, +-y) = r_ee (+-)x r_oe (+-)y r_eo (+-)x(+-)y r_oo
// over the quarter plane 0 <= x <= n1/2, 0 <= y <= n2/2, and the forward
// transform is the transpose.  Against a dense transform that is a quarter
// of the multiplications, and the sphere's pruning (kmax about n / 4) halves
// the inner lengths again: at 60 x 60 with kmax 14 the padded products are
// 394 kflop per plane against 167 kflop of butterflies, on units that do
// twice (FP32) to eight times what the butterflies reached.
//
// Chain of v_mfma_*_16x16x4 per 16-row y tile, no LDS and no barrier between
// the products: an accumulator (register i, lane group g) is the operand of
// the next product's k-step i as it stands, as B operand or, transposed, as
// A operand (both put the inner index in the lane group).
//   1  D1[kx][y]  = A[kx][ky]   C_y[ky][y]      A = the class matrix
//   2  D2[x][y]   = C_x[x][kx]  D1[kx][y]       B = D1
//      pointwise: times V, itself split into its classes W (the product of
//      classes a and b is of class a b, so out_a = sum_b W_ab r_b: 16
//      multiply-adds per point of the quarter plane)
//   3  D3[y][kx] += D2^T[y][x]  C_x[x][kx]      A = D2, over the x tiles
//   4  D4[ky][kx] += C_y[ky][y] D3[y][kx]       B = D3, over the y tiles
// Row r of an accumulator sits at (i, g) = (r / 4, r % 4) in FP64 but
// (r % 4, r / 4) in FP32, so FP32 lanes carry the indices in the permuted
// order perm(): then (i, g) holds index 4 i + g of its tile in both.
//
// Bound by the matrix pipes.  Constants (tables of {cos, sin}) come from LDS,
// one read per four products; V from a copy in operand order.
#pragma once
#include <algorithm>
#include <cmath>
#include <type_traits>
#include <vector>

#include "pw_fft.h"
#include "pw_internal.h"

namespace pw {

template <typename T> struct MmV;
template <> struct MmV<double> { typedef double t __attribute__((ext_vector_type(4))); };
template <> struct MmV<float> { typedef float t __attribute__((ext_vector_type(4))); };

__device__ __forceinline__ MmV<double>::t mm16(double a, double b, MmV<double>::t c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ MmV<float>::t mm16(float a, float b, MmV<float>::t c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// index within a 16-tile carried by lane c % 16
template <typename T>
__host__ __device__ __forceinline__ int mm_perm(int c) {
  return sizeof(T) == 8 ? c : 4 * (c & 3) + (c >> 2);
}

// {cos, sin} of 2 pi m / n, m = 0 .. n - 1, the quadrant taken exactly
inline std::vector<double2> roots_of(int n) {
  std::vector<double2> w(n);
  for (long m = 0; m < n; m++) {
    const long q = 4 * m / n, rem = 4 * m - q * n;
    const long double a = (long double)rem / (long double)n * 1.57079632679489661923132169163975144L;
    const double c = (double)cosl(a), s = (double)sinl(a);
    w[m] = q == 0 ? double2{c, s} : q == 1 ? double2{-s, c} : q == 2 ? double2{-c, -s} : double2{s, -c};
  }
  return w;
}

// The two tables of one axis: kt [T][KS][64] = {cos, sin}(2 pi h k / n) at
// k = 4 s + lane / 16, h = 16 tile + perm(lane % 16); ht [TK][4 T][64] at h =
// 4 u + lane / 16, k = 16 tile + perm(lane % 16); zero beyond kmax and n / 2.
template <typename T>
inline typename cx<T>::t* axis_tables(int n, int kmax, int KS, int tiles, typename cx<T>::t* out) {
  const int TK = (KS + 3) / 4, H = n / 2 + 1;
  const std::vector<double2> w = roots_of(n);
  auto put = [&](int k, int h) {
    const double2 e = k <= kmax && h < H ? w[(long)k * h % n] : double2{0, 0};
    *out++ = typename cx<T>::t{(T)e.x, (T)e.y};
  };
  for (int a = 0; a < tiles; a++)
    for (int s = 0; s < KS; s++)
      for (int l = 0; l < 64; l++) put(4 * s + l / 16, 16 * a + mm_perm<T>(l % 16));
  for (int a = 0; a < TK; a++)
    for (int u = 0; u < 4 * tiles; u++)
      for (int l = 0; l < 64; l++) put(16 * a + mm_perm<T>(l % 16), 4 * u + l / 16);
  return out;
}

// Stick entry of (kx, ky >= 0): x = stick of +ky, y = stick of -ky; kMmNone
// where there is none, kMmConj set where the value is the conjugate of that
// stick (the kx = 0 column, which stores one of each pair).
constexpr int kMmNone = -1;
constexpr int kMmConj = 1 << 30;

// Device pointers and lengths of one context's plan in one precision.
template <typename T>
struct MmArgs {
  const typename cx<T>::t *kx_t, *hx_t;  // x: [TX][KS][64] (k inner), [TK][4 TX][64] (h inner)
  const typename cx<T>::t *ky_t, *hy_t;  // y, the same pointers where the tables agree
  const int2* sp;                        // [TK][KS][64]
  const typename MmV<T>::t* v;           // [z][TY][TX][4][64]: V / N as W_ee, W_oe, W_eo, W_oo
  int TX, TY, XS, YS;                    // tiles and k-steps of the quarter plane
  int n3, nstick, nb, half;              // half: n1 / 2 where n1 is even, else -1 (the kx with weight 1)
  int shared;                            // the y tables are the x tables
};

// LDS bytes of the tables
template <typename T>
inline size_t mm_lds(int KS, int TX, int TY, bool shared) {
  const int TK = (KS + 3) / 4;
  const size_t tab = (size_t)(KS + 4 * TK) * (TX + (shared ? 0 : TY));
  return 64 * (sizeof(typename cx<T>::t) * tab + sizeof(int2) * TK * KS);
}

// KS: k-steps (of 4) that cover kxmax + 1 and kymax + 1; NW waves per
// workgroup, each with its own band of plane z.  A workgroup walks over
// (plane, band group) items; a wave asks for the sticks of its next item
// before the last products of the current one, when the registers of the
// first products are free.
template <typename T, int KS, int NW, int LB>
__global__ void __launch_bounds__(64 * NW, LB)
k_slab_mm(const typename cx<T>::t* __restrict__ t1, typename cx<T>::t* __restrict__ t2, const MmArgs<T> g_) {
  typedef typename cx<T>::t C;
  typedef typename MmV<T>::t V;
  constexpr int TK = (KS + 3) / 4;
  extern __shared__ __align__(16) unsigned char smem_raw[];
  C* kxt = reinterpret_cast<C*>(smem_raw);
  C* hxt = kxt + 64 * KS * g_.TX;
  C* kyt = g_.shared ? kxt : hxt + 64 * 4 * TK * g_.TX;
  C* hyt = g_.shared ? hxt : kyt + 64 * KS * g_.TY;
  int2* spt = reinterpret_cast<int2*>(hyt + 64 * 4 * TK * g_.TY);
  const int t = threadIdx.x, lane = t & 63, w = t >> 6, c = lane & 15;
  // consecutive items: the band groups of one plane.  XCD x takes one
  // contiguous run of items (one L2 copy of a plane of V) and its blocks step
  // through that run together.
  const int ngrp = (g_.nb + NW - 1) / NW, items = g_.n3 * ngrp;
  const int xcd = blockIdx.x & 7, step = (gridDim.x + 7 - xcd) >> 3;
  const int q8 = items >> 3, r8 = items & 7;
  const int last = (xcd + 1) * q8 + min(xcd + 1, r8);
  int item = xcd * q8 + min(xcd, r8) + (blockIdx.x >> 3);
  {
    const int nk = 64 * KS * g_.TX, nh = 64 * 4 * TK * g_.TX;
    for (int e = t; e < nk; e += 64 * NW) kxt[e] = g_.kx_t[e];
    for (int e = t; e < nh; e += 64 * NW) hxt[e] = g_.hx_t[e];
    if (!g_.shared) {
      const int mk = 64 * KS * g_.TY, mh = 64 * 4 * TK * g_.TY;
      for (int e = t; e < mk; e += 64 * NW) kyt[e] = g_.ky_t[e];
      for (int e = t; e < mh; e += 64 * NW) hyt[e] = g_.hy_t[e];
    }
    for (int e = t; e < 64 * TK * KS; e += 64 * NW) spt[e] = g_.sp[e];
  }
  __syncthreads();

  // the sticks +-ky of this lane, as loaded (absent ones: any stick)
  C rp[TK][KS], rm[TK][KS];
  auto fetch = [&](int it) {
    const int z = it / ngrp, band = min((it - z * ngrp) * NW + w, g_.nb - 1);
    const C* src = t1 + ((size_t)band * g_.n3 + z) * g_.nstick;
#pragma unroll
    for (int k = 0; k < TK; k++)
#pragma unroll
      for (int s = 0; s < KS; s++) {
        const int2 e = spt[(k * KS + s) * 64 + lane];
        rp[k][s] = src[e.x == kMmNone ? 0 : (e.x & ~kMmConj)];
        rm[k][s] = src[e.y == kMmNone ? 0 : (e.y & ~kMmConj)];
      }
  };
  if (item < last) fetch(item);

  for (; item < last; item += step) {
  const int z = item / ngrp, band = (item - z * ngrp) * NW + w;
  // the plane's sticks into the four class matrices
  T ee[TK][KS], oe[TK][KS], eo[TK][KS], oo[TK][KS];
#pragma unroll
  for (int k = 0; k < TK; k++) {
    const int kx = 16 * k + mm_perm<T>(c);
    const T wt = (kx == 0 || kx == g_.half) ? (T)1 : (T)2;
#pragma unroll
    for (int s = 0; s < KS; s++) {
      const int2 e = spt[(k * KS + s) * 64 + lane];
      C p = rp[k][s], m = rm[k][s];
      if (e.x & kMmConj) p.y = -p.y;
      if (e.y & kMmConj) m.y = -m.y;
      if (e.x == kMmNone) p = C{0, 0};
      if (e.y == kMmNone) m = C{0, 0};
      ee[k][s] = wt * (p.x + m.x);
      oe[k][s] = -wt * (p.y + m.y);
      eo[k][s] = -wt * (p.y - m.y);
      oo[k][s] = -wt * (p.x - m.x);
    }
  }

  const V zero = {0, 0, 0, 0};
  V zee[TK][TK], zoe[TK][TK], zeo[TK][TK], zoo[TK][TK];  // [ky tile][kx tile]
#pragma unroll
  for (int a = 0; a < TK; a++)
#pragma unroll
    for (int b = 0; b < TK; b++) zee[a][b] = zoe[a][b] = zeo[a][b] = zoo[a][b] = zero;

  auto ytile = [&](int yt, bool prefetch) {
    V dee[TK], doe[TK], deo[TK], doo[TK];
#pragma unroll
    for (int k = 0; k < TK; k++) dee[k] = doe[k] = deo[k] = doo[k] = zero;
    {
      C q[KS];
#pragma unroll
      for (int s = 0; s < KS; s++) q[s] = kyt[(yt * KS + s) * 64 + lane];
#pragma unroll
      for (int s = 0; s < KS; s++)
#pragma unroll
        for (int k = 0; k < TK; k++) {
          dee[k] = mm16(ee[k][s], q[s].x, dee[k]);
          deo[k] = mm16(eo[k][s], q[s].y, deo[k]);
          doe[k] = mm16(oe[k][s], q[s].x, doe[k]);
          doo[k] = mm16(oo[k][s], q[s].y, doo[k]);
        }
    }
    V fee[TK], foe[TK], feo[TK], foo[TK];  // D3
#pragma unroll
    for (int k = 0; k < TK; k++) fee[k] = foe[k] = feo[k] = foo[k] = zero;
    const V* vp = g_.v + ((size_t)(z * g_.TY + yt) * g_.TX * 4) * 64 + lane;
    // one x tile of NI k-steps in its second product.  Everything it reads is
    // issued first (left alone, the compiler sinks the loads behind the
    // products and waits for each)
    auto tile = [&](int xt, auto ni) {
      constexpr int NI = decltype(ni)::value;
      V v[4];
      C q[KS], h[TK][NI];
#pragma unroll
      for (int i = 0; i < NI; i++) v[i] = vp[(xt * 4 + i) * 64];
#pragma unroll
      for (int s = 0; s < KS; s++) q[s] = kxt[(xt * KS + s) * 64 + lane];
      if constexpr (TK == 1) {
#pragma unroll
        for (int i = 0; i < NI; i++) h[0][i] = hxt[(4 * xt + i) * 64 + lane];
      }
      __builtin_amdgcn_sched_barrier(0);
      V ree = zero, roe = zero, reo = zero, roo = zero;
#pragma unroll
      for (int s = 0; s < KS; s++) {
        ree = mm16(q[s].x, dee[s / 4][s % 4], ree);
        roe = mm16(q[s].y, doe[s / 4][s % 4], roe);
        reo = mm16(q[s].x, deo[s / 4][s % 4], reo);
        roo = mm16(q[s].y, doo[s / 4][s % 4], roo);
      }
      if constexpr (TK > 1) {
#pragma unroll
        for (int k = 0; k < TK; k++)
#pragma unroll
          for (int i = 0; i < NI; i++) h[k][i] = hxt[(k * 4 * g_.TX + 4 * xt + i) * 64 + lane];
      }
#pragma unroll
      for (int i = 0; i < NI; i++) {
        const T e0 = ree[i], e1 = roe[i], e2 = reo[i], e3 = roo[i];
        const T w0 = v[i][0], w1 = v[i][1], w2 = v[i][2], w3 = v[i][3];
        ree[i] = w0 * e0 + w1 * e1 + w2 * e2 + w3 * e3;
        roe[i] = w1 * e0 + w0 * e1 + w3 * e2 + w2 * e3;
        reo[i] = w2 * e0 + w3 * e1 + w0 * e2 + w1 * e3;
        roo[i] = w3 * e0 + w2 * e1 + w1 * e2 + w0 * e3;
#pragma unroll
        for (int k = 0; k < TK; k++) {
          fee[k] = mm16(ree[i], h[k][i].x, fee[k]);
          foe[k] = mm16(roe[i], h[k][i].y, foe[k]);
          feo[k] = mm16(reo[i], h[k][i].x, feo[k]);
          foo[k] = mm16(roo[i], h[k][i].y, foo[k]);
        }
      }
    };
    const int full = g_.XS >> 2;
    for (int xt = 0; xt < full; xt++) tile(xt, std::integral_constant<int, 4>{});
    switch (g_.XS & 3) {
      case 1: tile(full, std::integral_constant<int, 1>{}); break;
      case 2: tile(full, std::integral_constant<int, 2>{}); break;
      case 3: tile(full, std::integral_constant<int, 3>{}); break;
      default: break;
    }
    if (prefetch) {
      __builtin_amdgcn_sched_barrier(0);
      fetch(min(item + step, last - 1));  // unconditional: a branch would keep the old values in registers
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int a = 0; a < TK; a++) {
      C q[4];
#pragma unroll
      for (int i = 0; i < 4; i++) q[i] = hyt[(a * 4 * g_.TY + 4 * yt + i) * 64 + lane];
#pragma unroll
      for (int i = 0; i < 4; i++)
        if (i == 0 || 4 * yt + i < g_.YS) {
#pragma unroll
          for (int k = 0; k < TK; k++) {
            zee[a][k] = mm16(q[i].x, fee[k][i], zee[a][k]);
            zeo[a][k] = mm16(q[i].y, feo[k][i], zeo[a][k]);
            zoe[a][k] = mm16(q[i].x, foe[k][i], zoe[a][k]);
            zoo[a][k] = mm16(q[i].y, foo[k][i], zoo[a][k]);
          }
        }
    }
  };
  for (int yt = 0; yt + 1 < g_.TY; yt++) ytile(yt, false);
  ytile(g_.TY - 1, true);
  if (band >= g_.nb) continue;
  // Z(kx, +-ky): Re = ee -+ oo, Im = -(oe +- eo)
  C* dst = t2 + ((size_t)band * g_.n3 + z) * g_.nstick;
#pragma unroll
  for (int k = 0; k < TK; k++) {
    int2 e[KS];
#pragma unroll
    for (int s = 0; s < KS; s++) e[s] = spt[(k * KS + s) * 64 + lane];
#pragma unroll
    for (int s = 0; s < KS; s++) {
      const T a = zee[s / 4][k][s % 4], b = zoo[s / 4][k][s % 4], p = zoe[s / 4][k][s % 4], q = zeo[s / 4][k][s % 4];
      if (e[s].x >= 0 && !(e[s].x & kMmConj)) dst[e[s].x] = C{a - b, -(p + q)};
      if (e[s].y >= 0 && !(e[s].y & kMmConj)) dst[e[s].y] = C{a + b, q - p};
    }
  }
  }
}

// The same transform for spheres of more than 16 columns, where one wavefront
// would need the whole register file for its tiles: a workgroup takes NB bands
// of a plane, wavefront (band, y tile) runs products 1 to 3 for its tile with
// the class matrices in LDS, and the third products' results go through LDS
// (two classes at a time, in the class matrices' place) to the fourth, whose
// (ky, kx) tiles the band's wavefronts share out.  The x tables stay in LDS
// for all items of a workgroup.
//
// Bound by the matrix pipes: a 180 x 180 plane of 45 columns is 5076 products
// in FP32, 69 ns of the chip; it takes 113 ns, against 173 ns of butterflies in
// LDS (k_slab_xy), 120 x 120 planes of 30 columns 40 ns against 329.
template <typename T>
inline size_t mm_wg_band(int KS, int TY) {  // LDS bytes of one band
  const int TK = (KS + 3) / 4;
  return 64 * sizeof(T) * (size_t)TK * std::max(4 * KS, 8 * TY);
}
template <typename T>
inline size_t mm_wg_tables(int KS, int TX) {
  return 64 * sizeof(typename cx<T>::t) * (size_t)TX * (KS + 4 * ((KS + 3) / 4));
}
template <typename T, int TK, int MAXT>
__global__ void __launch_bounds__(MAXT)
k_slab_mm_wg(const typename cx<T>::t* __restrict__ t1, typename cx<T>::t* __restrict__ t2, const MmArgs<T> g_, int KS,
             int NB) {
  typedef typename cx<T>::t C;
  typedef typename MmV<T>::t V;
  extern __shared__ __align__(16) unsigned char smem_raw[];
  C* kxt = reinterpret_cast<C*>(smem_raw);
  C* hxt = kxt + 64 * KS * g_.TX;
  const C* kyt = g_.shared ? kxt : g_.ky_t;
  const C* hyt = g_.shared ? hxt : g_.hy_t;
  const int t = threadIdx.x, lane = t & 63, w = t >> 6, c = lane & 15, TY = g_.TY;
  const int bl = w / TY, yt = w - bl * TY;
  T* buf = reinterpret_cast<T*>(hxt + 64 * 4 * TK * g_.TX) + (size_t)bl * 64 * TK * max(4 * KS, 8 * TY);
  for (int e = t; e < 64 * KS * g_.TX; e += blockDim.x) kxt[e] = g_.kx_t[e];
  for (int e = t; e < 64 * 4 * TK * g_.TX; e += blockDim.x) hxt[e] = g_.hx_t[e];
  const int ngrp = (g_.nb + NB - 1) / NB, items = g_.n3 * ngrp;
  const int xcd = blockIdx.x & 7, step = (gridDim.x + 7 - xcd) >> 3;
  const int q8 = items >> 3, r8 = items & 7;
  const int last = (xcd + 1) * q8 + min(xcd + 1, r8);
  const V zero = {0, 0, 0, 0};
  for (int item = xcd * q8 + min(xcd, r8) + (blockIdx.x >> 3); item < last; item += step) {
    const int z = item / ngrp, band = (item - z * ngrp) * NB + bl;
    const bool live = band < g_.nb;
    const size_t base = ((size_t)(live ? band : 0) * g_.n3 + z) * g_.nstick;
    const C* src = t1 + base;
    // class matrices [kx tile][k-step][class][64]
    for (int e = yt * 64 + lane; e < 64 * TK * KS; e += 64 * TY) {
      const int kx = 16 * ((e >> 6) / KS) + mm_perm<T>(c);
      const T wt = (kx == 0 || kx == g_.half) ? (T)1 : (T)2;
      const int2 se = g_.sp[e];
      C p = src[se.x == kMmNone ? 0 : (se.x & ~kMmConj)], m = src[se.y == kMmNone ? 0 : (se.y & ~kMmConj)];
      if (se.x & kMmConj) p.y = -p.y;
      if (se.y & kMmConj) m.y = -m.y;
      if (se.x == kMmNone) p = C{0, 0};
      if (se.y == kMmNone) m = C{0, 0};
      T* o = buf + (size_t)(e >> 6) * 256 + lane;
      o[0] = wt * (p.x + m.x);
      o[64] = -wt * (p.y + m.y);
      o[128] = -wt * (p.y - m.y);
      o[192] = -wt * (p.x - m.x);
    }
    __syncthreads();
    V dee[TK], doe[TK], deo[TK], doo[TK];
#pragma unroll
    for (int k = 0; k < TK; k++) dee[k] = doe[k] = deo[k] = doo[k] = zero;
#pragma unroll 2
    for (int s = 0; s < KS; s++) {
      const C q = kyt[(yt * KS + s) * 64 + lane];
#pragma unroll
      for (int k = 0; k < TK; k++) {
        const T* a = buf + (size_t)(k * KS + s) * 256 + lane;
        dee[k] = mm16(a[0], q.x, dee[k]);
        doe[k] = mm16(a[64], q.x, doe[k]);
        deo[k] = mm16(a[128], q.y, deo[k]);
        doo[k] = mm16(a[192], q.y, doo[k]);
      }
    }
    V fee[TK], foe[TK], feo[TK], foo[TK];
#pragma unroll
    for (int k = 0; k < TK; k++) fee[k] = foe[k] = feo[k] = foo[k] = zero;
    const V* vp = g_.v + ((size_t)(z * TY + yt) * g_.TX * 4) * 64 + lane;
    for (int xt = 0; xt < g_.TX; xt++) {
      V v[4];
#pragma unroll
      for (int i = 0; i < 4; i++) v[i] = vp[(xt * 4 + i) * 64];
      V ree = zero, roe = zero, reo = zero, roo = zero;
#pragma unroll
      for (int k = 0; k < TK; k++)
#pragma unroll
        for (int i = 0; i < 4; i++)
          if (k + 1 < TK || 4 * k + i < KS) {
            const C q = kxt[(xt * KS + 4 * k + i) * 64 + lane];
            ree = mm16(q.x, dee[k][i], ree);
            roe = mm16(q.y, doe[k][i], roe);
            reo = mm16(q.x, deo[k][i], reo);
            roo = mm16(q.y, doo[k][i], roo);
          }
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const T e0 = ree[i], e1 = roe[i], e2 = reo[i], e3 = roo[i];
        const T w0 = v[i][0], w1 = v[i][1], w2 = v[i][2], w3 = v[i][3];
        ree[i] = w0 * e0 + w1 * e1 + w2 * e2 + w3 * e3;
        roe[i] = w1 * e0 + w0 * e1 + w3 * e2 + w2 * e3;
        reo[i] = w2 * e0 + w3 * e1 + w0 * e2 + w1 * e3;
        roo[i] = w3 * e0 + w2 * e1 + w1 * e2 + w0 * e3;
      }
#pragma unroll
      for (int i = 0; i < 4; i++)
        if (i == 0 || 4 * xt + i < g_.XS) {
#pragma unroll
          for (int k = 0; k < TK; k++) {
            const C q = hxt[(k * 4 * g_.TX + 4 * xt + i) * 64 + lane];
            fee[k] = mm16(ree[i], q.x, fee[k]);
            foe[k] = mm16(roe[i], q.y, foe[k]);
            feo[k] = mm16(reo[i], q.x, feo[k]);
            foo[k] = mm16(roo[i], q.y, foo[k]);
          }
        }
    }
    // Re (ee, oo), then Im (oe, eo): [class of the pair][kx tile][4 TY][64]
    T* pa = buf;
    T* pb = buf + (size_t)TK * 4 * TY * 64;
#pragma unroll
    for (int im = 0; im < 2; im++) {
      __syncthreads();  // the class matrices, then the first pair, have been read
#pragma unroll
      for (int k = 0; k < TK; k++)
#pragma unroll
        for (int i = 0; i < 4; i++) {
          const int at = (k * 4 * TY + 4 * yt + i) * 64 + lane;
          pa[at] = im ? foe[k][i] : fee[k][i];
          pb[at] = im ? feo[k][i] : foo[k][i];
        }
      __syncthreads();
      for (int u = yt; u < TK * TK; u += TY) {
        const int ky = u / TK, kx = u - ky * TK;
        V za = zero, zb = zero;
#pragma unroll 4
        for (int s = 0; s < g_.YS; s++) {
          const C q = hyt[(ky * 4 * TY + s) * 64 + lane];
          za = mm16(q.x, pa[(kx * 4 * TY + s) * 64 + lane], za);
          zb = mm16(q.y, pb[(kx * 4 * TY + s) * 64 + lane], zb);
        }
        if (!live) continue;
        T* dst = reinterpret_cast<T*>(t2 + base) + im;
#pragma unroll
        for (int i = 0; i < 4; i++)
          if (4 * ky + i < KS) {
            const int2 e = g_.sp[(kx * KS + 4 * ky + i) * 64 + lane];
            if (e.x >= 0 && !(e.x & kMmConj)) dst[2 * e.x] = im ? -(za[i] + zb[i]) : za[i] - zb[i];
            if (e.y >= 0 && !(e.y & kMmConj)) dst[2 * e.y] = im ? zb[i] - za[i] : za[i] + zb[i];
          }
      }
    }
    __syncthreads();  // before the next item's class matrices
  }
}

// Density of nb bands on one 16 x 16 tile of the quarter plane: products 1 and
// 2 of k_slab_mm per band, then acc += f r(+-x, +-y)^2 in FP64 registers.  A
// wave takes (plane, tile, every nsplit-th band) and writes its tile once to
// part[split] (N doubles each), so the sums over splits are in a fixed order.
// The first product is repeated for each x tile (16 products beside the 16 of
// the second): with the tile fixed the sums stay in 32 registers at any size.
template <typename T, int KS, int NW>
__global__ void __launch_bounds__(64 * NW, sizeof(T) == 8 && KS > 4 ? 1 : 2)
k_density_mm(const typename cx<T>::t* __restrict__ t1, const MmArgs<T> g_, const double* __restrict__ f, double invN,
             int nsplit, int n1, int n2, double* __restrict__ part) {
  typedef typename cx<T>::t C;
  typedef typename MmV<T>::t V;
  constexpr int TK = (KS + 3) / 4;
  const int lane = threadIdx.x & 63, c = lane & 15, gq = lane >> 4;
  const int per_z = g_.TX * g_.TY * nsplit;
  const int unit = blockIdx.x * NW + (threadIdx.x >> 6);
  if (unit >= per_z * g_.n3) return;
  const int z = unit / per_z, r = unit - z * per_z, split = r / (g_.TX * g_.TY);
  const int xt = r % g_.TX, yt = r / g_.TX % g_.TY;
  C ky[KS], kx[KS];
#pragma unroll
  for (int s = 0; s < KS; s++) {
    ky[s] = g_.ky_t[(yt * KS + s) * 64 + lane];
    kx[s] = g_.kx_t[(xt * KS + s) * 64 + lane];
  }
  double acc[4][4];
#pragma unroll
  for (int i = 0; i < 4; i++)
#pragma unroll
    for (int s = 0; s < 4; s++) acc[i][s] = 0.0;
  const V zero = {0, 0, 0, 0};
  for (int band = split; band < g_.nb; band += nsplit) {
    const C* src = t1 + ((size_t)band * g_.n3 + z) * g_.nstick;
    const double fb = f[band] * invN;
    V dee[TK], doe[TK], deo[TK], doo[TK];
#pragma unroll
    for (int k = 0; k < TK; k++) {
      dee[k] = doe[k] = deo[k] = doo[k] = zero;
      const int kxi = 16 * k + mm_perm<T>(c);
      const T wt = (kxi == 0 || kxi == g_.half) ? (T)1 : (T)2;
#pragma unroll
      for (int s = 0; s < KS; s++) {
        const int2 e = g_.sp[(k * KS + s) * 64 + lane];
        C p = src[e.x == kMmNone ? 0 : (e.x & ~kMmConj)], m = src[e.y == kMmNone ? 0 : (e.y & ~kMmConj)];
        if (e.x & kMmConj) p.y = -p.y;
        if (e.y & kMmConj) m.y = -m.y;
        if (e.x == kMmNone) p = C{0, 0};
        if (e.y == kMmNone) m = C{0, 0};
        dee[k] = mm16(wt * (p.x + m.x), ky[s].x, dee[k]);
        doe[k] = mm16(-wt * (p.y + m.y), ky[s].x, doe[k]);
        deo[k] = mm16(-wt * (p.y - m.y), ky[s].y, deo[k]);
        doo[k] = mm16(-wt * (p.x - m.x), ky[s].y, doo[k]);
      }
    }
    V ree = zero, roe = zero, reo = zero, roo = zero;
#pragma unroll
    for (int s = 0; s < KS; s++) {
      ree = mm16(kx[s].x, dee[s / 4][s % 4], ree);
      roe = mm16(kx[s].y, doe[s / 4][s % 4], roe);
      reo = mm16(kx[s].x, deo[s / 4][s % 4], reo);
      roo = mm16(kx[s].y, doo[s / 4][s % 4], roo);
    }
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const T ep = ree[i] + reo[i], em = ree[i] - reo[i], op = roe[i] + roo[i], om = roe[i] - roo[i];
      const double r0 = ep + op, r1 = ep - op, r2 = em + om, r3 = em - om;
      acc[i][0] += r0 * r0 * fb;
      acc[i][1] += r1 * r1 * fb;
      acc[i][2] += r2 * r2 * fb;
      acc[i][3] += r3 * r3 * fb;
    }
  }
  double* o = part + ((size_t)split * g_.n3 + z) * n1 * n2;
  const int y = 16 * yt + mm_perm<T>(c);
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const int x = 16 * xt + 4 * i + gq;
    if (x > n1 / 2 || y > n2 / 2) continue;
    const bool mx = x != 0 && 2 * x != n1, my = y != 0 && 2 * y != n2;
    o[(size_t)y * n1 + x] = acc[i][0];
    if (mx) o[(size_t)y * n1 + n1 - x] = acc[i][1];
    if (my) o[(size_t)(n2 - y) * n1 + x] = acc[i][2];
    if (mx && my) o[(size_t)(n2 - y) * n1 + n1 - x] = acc[i][3];
  }
}

}  // namespace pw

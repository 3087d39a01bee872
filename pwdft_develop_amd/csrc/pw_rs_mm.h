// Dual-grid transforms of the real-space path on FP64 matrix cores.
//
// Planes: a real n1 x n2 plane to and from its half spectrum at kx <= kmax_x,
// |ky| <= kmax_y, as the four parity classes of pw_slab_mm.h (the same
// tables); the fine grid's planes are pruned to the coarse band by the short
// k axis alone.  Pencils: complex transforms along z as P = sum E cos, Q =
// sum O sin with E, O = X(k) +- X(-k) and G(+-z) = P +- i Q, 16 neighbouring
// columns per wavefront as the product's columns, streaming over the inner
// index.  Any length goes, prime factors included, and one pass replaces the
// y and x passes of butterflies through LDS.
//
// Bound by memory: a 124 x 124 plane of 32 x 63 entries is 768 products of
// 2048 flops each way (0.47 ms of a 170-band launch) and 155 kB.
// Accumulator layouts and operand identities: pw_slab_mm.h.
#pragma once
#include "pw_slab_mm.h"

namespace pw {

typedef MmV<double>::t RsV;

// One axis: kt [T][KS][64], ht [TK][4 T][64] of {cos, sin} (axis_tables).
struct RsAxis {
  const double2 *kt, *ht;
  int n, H, T;  // length, quarter rows n / 2 + 1, their 16-row tiles
};

struct RsPlane {
  RsAxis x, y;
  const int *rp, *rm;  // spectrum row of +ky and of -ky (-1: none), 4 KS entries each
  int hw, nrow;        // kx entries per spectrum row, rows per plane
  int nplane, nb;      // planes per band, bands
};

// LDS bytes of the inverse plane kernel: the class matrices and the x table
inline size_t rs_plane_inv_lds(int KS, int TX) {
  const int TK = (KS + 3) / 4;
  return 64 * (sizeof(double) * 4 * TK * KS + sizeof(double2) * (size_t)TX * KS);
}

// spectrum [band][plane][row][kx] -> real [band][plane][y][x].  One workgroup
// of four wavefronts per plane; a wavefront takes every fourth y tile.  The
// lanes of a product's columns are neighbouring x, so stores are 128-byte
// runs.
template <int KS>
__global__ void __launch_bounds__(256, 2)
k_rs_plane_inv(const double2* __restrict__ in, RsPlane g, double* __restrict__ out) {
  constexpr int TK = (KS + 3) / 4;
  extern __shared__ __align__(16) unsigned char smem_raw[];
  double2* kxt = reinterpret_cast<double2*>(smem_raw);
  double* cls = reinterpret_cast<double*>(kxt + 64 * KS * g.x.T);  // [TK][KS][class][64]
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, c = lane & 15, q4 = lane >> 4;
  const int item = xcd_item(blockIdx.x, gridDim.x);
  const int band = item / g.nplane, z = item - band * g.nplane;
  const double2* src = in + ((size_t)band * g.nplane + z) * g.nrow * g.hw;
  for (int e = threadIdx.x; e < 64 * TK * KS; e += 256) {
    const int l = e & 63, s = (e >> 6) % KS, k = (e >> 6) / KS;
    const int kx = 16 * k + (l & 15), ky = 4 * s + (l >> 4);
    const int rp = g.rp[ky], rm = g.rm[ky];
    const bool in_x = kx < g.hw;
    double2 p = src[(size_t)max(rp, 0) * g.hw + (in_x ? kx : 0)], m = src[(size_t)max(rm, 0) * g.hw + (in_x ? kx : 0)];
    if (!in_x || rp < 0) p = make_double2(0.0, 0.0);
    if (!in_x || rm < 0) m = make_double2(0.0, 0.0);
    const double wt = (kx == 0 || 2 * kx == g.x.n) ? 1.0 : 2.0;
    double* o = cls + (size_t)(k * KS + s) * 256 + l;
    o[0] = wt * (p.x + m.x);
    o[64] = -wt * (p.y + m.y);
    o[128] = -wt * (p.y - m.y);
    o[192] = -wt * (p.x - m.x);
  }
  for (int e = threadIdx.x; e < 64 * KS * g.x.T; e += 256) kxt[e] = g.x.kt[e];
  __syncthreads();
  const RsV zero = {0, 0, 0, 0};
  out += ((size_t)band * g.nplane + z) * g.y.n * g.x.n;
  for (int yt = w; yt < g.y.T; yt += 4) {
    RsV dee[TK], doe[TK], deo[TK], doo[TK];
#pragma unroll
    for (int k = 0; k < TK; k++) dee[k] = doe[k] = deo[k] = doo[k] = zero;
#pragma unroll
    for (int s = 0; s < KS; s++) {
      const double2 q = g.y.kt[(yt * KS + s) * 64 + lane];
#pragma unroll
      for (int k = 0; k < TK; k++) {
        const double* a = cls + (size_t)(k * KS + s) * 256 + lane;
        dee[k] = mm16(a[0], q.x, dee[k]);
        doe[k] = mm16(a[64], q.x, doe[k]);
        deo[k] = mm16(a[128], q.y, deo[k]);
        doo[k] = mm16(a[192], q.y, doo[k]);
      }
    }
    for (int xt = 0; xt < g.x.T; xt++) {
      RsV ree = zero, roe = zero, reo = zero, roo = zero;
#pragma unroll
      for (int s = 0; s < KS; s++) {
        const double2 q = kxt[(xt * KS + s) * 64 + lane];
        ree = mm16(dee[s / 4][s % 4], q.x, ree);
        roe = mm16(doe[s / 4][s % 4], q.y, roe);
        reo = mm16(deo[s / 4][s % 4], q.x, reo);
        roo = mm16(doo[s / 4][s % 4], q.y, roo);
      }
      const int x = 16 * xt + c;
      const bool ok = x < g.x.H, mx = ok && x != 0 && 2 * x != g.x.n;
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const int y = 16 * yt + 4 * i + q4;
        if (y >= g.y.H) continue;
        const bool my = y != 0 && 2 * y != g.y.n;
        const double ep = ree[i] + reo[i], em = ree[i] - reo[i], op = roe[i] + roo[i], om = roe[i] - roo[i];
        double *r0 = out + y * g.x.n, *r1 = out + (g.y.n - y) * g.x.n;
        if (ok) r0[x] = ep + op;
        if (mx) r0[g.x.n - x] = ep - op;
        if (ok && my) r1[x] = em + om;
        if (mx && my) r1[g.x.n - x] = em - om;
      }
    }
  }
}

// real [band][plane][y][x], times vloc [plane][y][x] with kV -> spectrum rows
// at kx < hw, ky of the row tables.
// One wavefront per plane, NW planes (neighbouring bands) per workgroup.
// Contracts y first: a lane's loads are neighbouring x (A operand: row x, k
// y), then x against the tables with the first result as A operand, so that
// the lanes of the stores are neighbouring kx.
template <int KS, int NW, bool kV>
__global__ void __launch_bounds__(64 * NW, 2)
k_rs_plane_fwd(const double* __restrict__ in, RsPlane g, const double* __restrict__ vloc, double2* __restrict__ out) {
  constexpr int TK = (KS + 3) / 4;
  extern __shared__ __align__(16) unsigned char smem_raw[];
  double2* hyt = reinterpret_cast<double2*>(smem_raw);  // [TK][4 TY][64]
  double2* hxt = g.x.ht == g.y.ht ? hyt : hyt + 64 * 4 * TK * g.y.T;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, c = lane & 15, q4 = lane >> 4;
  const int ngrp = (g.nb + NW - 1) / NW;
  const int item = xcd_item(blockIdx.x, gridDim.x);
  const int z = item / ngrp, band = (item - z * ngrp) * NW + w;
  for (int e = threadIdx.x; e < 64 * 4 * TK * g.y.T; e += 64 * NW) hyt[e] = g.y.ht[e];
  if (hxt != hyt)
    for (int e = threadIdx.x; e < 64 * 4 * TK * g.x.T; e += 64 * NW) hxt[e] = g.x.ht[e];
  __syncthreads();
  if (band >= g.nb) return;
  const double* src = in + ((size_t)band * g.nplane + z) * g.y.n * g.x.n;
  const double* vz = kV ? vloc + (size_t)z * g.y.n * g.x.n : nullptr;
  const RsV zero = {0, 0, 0, 0};
  RsV zee[TK][TK], zoe[TK][TK], zeo[TK][TK], zoo[TK][TK];  // [ky tile][kx tile]
#pragma unroll
  for (int a = 0; a < TK; a++)
#pragma unroll
    for (int b = 0; b < TK; b++) zee[a][b] = zoe[a][b] = zeo[a][b] = zoo[a][b] = zero;
  const int YS = (g.y.H + 3) / 4;
  for (int xt = 0; xt < g.x.T; xt++) {
    const int x = 16 * xt + c;
    const bool ok = x < g.x.H, mx = ok && x != 0 && 2 * x != g.x.n;
    const int xp = ok ? x : 0, xm = mx ? g.x.n - x : 0;
    RsV fee[TK], foe[TK], feo[TK], foo[TK];
#pragma unroll
    for (int k = 0; k < TK; k++) fee[k] = foe[k] = feo[k] = foo[k] = zero;
    // the four signs of (x, y = 4 u + lane / 16), one step ahead
    double n[4], v[4];
    auto load = [&](int u) {
      const int y = min(4 * u + q4, g.y.H - 1), ym = (y != 0 && 2 * y != g.y.n) ? g.y.n - y : y;
      const int at[4] = {y * g.x.n + xp, y * g.x.n + xm, ym * g.x.n + xp, ym * g.x.n + xm};
#pragma unroll
      for (int s = 0; s < 4; s++) {
        n[s] = src[at[s]];
        if constexpr (kV) v[s] = vz[at[s]];
      }
    };
    load(0);
    for (int u = 0; u < YS; u++) {
      const int y = 4 * u + q4;
      const bool oy = y < g.y.H, my = oy && y != 0 && 2 * y != g.y.n;
      if constexpr (kV) {
#pragma unroll
        for (int s = 0; s < 4; s++) n[s] *= v[s];
      }
      const double s0 = ok && oy ? n[0] : 0.0, s1 = mx && oy ? n[1] : 0.0, s2 = ok && my ? n[2] : 0.0,
                   s3 = mx && my ? n[3] : 0.0;
      if (u + 1 < YS) load(u + 1);
      const double sp = s0 + s1, dp = s0 - s1, sm = s2 + s3, dm = s2 - s3;
#pragma unroll
      for (int k = 0; k < TK; k++) {
        const double2 q = hyt[(k * 4 * g.y.T + u) * 64 + lane];
        fee[k] = mm16(sp + sm, q.x, fee[k]);
        foe[k] = mm16(dp + dm, q.x, foe[k]);
        feo[k] = mm16(sp - sm, q.y, feo[k]);
        foo[k] = mm16(dp - dm, q.y, foo[k]);
      }
    }
#pragma unroll
    for (int i = 0; i < 4; i++) {
#pragma unroll
      for (int b = 0; b < TK; b++) {
        const double2 q = hxt[(b * 4 * g.x.T + 4 * xt + i) * 64 + lane];
#pragma unroll
        for (int a = 0; a < TK; a++) {
          zee[a][b] = mm16(fee[a][i], q.x, zee[a][b]);
          zoe[a][b] = mm16(foe[a][i], q.y, zoe[a][b]);
          zeo[a][b] = mm16(feo[a][i], q.x, zeo[a][b]);
          zoo[a][b] = mm16(foo[a][i], q.y, zoo[a][b]);
        }
      }
    }
  }
  double2* dst = out + ((size_t)band * g.nplane + z) * g.nrow * g.hw;
#pragma unroll
  for (int a = 0; a < TK; a++)
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const int ky = 16 * a + 4 * i + q4;
      if (ky >= 4 * KS) continue;
      const int rp = g.rp[ky], rm = g.rm[ky];
#pragma unroll
      for (int b = 0; b < TK; b++) {
        const int kx = 16 * b + c;
        if (kx >= g.hw) continue;
        const double e = zee[a][b][i], o = zoo[a][b][i], p = zoe[a][b][i], q = zeo[a][b][i];
        if (rp >= 0) dst[(size_t)rp * g.hw + kx] = make_double2(e - o, -(p + q));
        if (rm >= 0) dst[(size_t)rm * g.hw + kx] = make_double2(e + o, q - p);
      }
    }
}

// Complex transform along the slowest axis of [band][a2][column]: input entry
// j >= 0 of index +j at ip[j], of -j at im[j] (-1: none), output entry h at
// op[h] / om[h]; tab [TH][KS][64] with row h = 16 tile + lane % 16 and inner
// index 4 s + lane / 16.  sg = +1 backward, -1 forward.  kC2f: the input is
// the coarse spectrum [k][j][i] read by the coarse-to-fine rules (columns l hc
// + i of live rows l; IP_c2f, src/utility.cpp:3150-3212), times scale.
struct RsPencil {
  const double2* in;
  double2* out;
  const double2* tab;
  const int *ip, *im, *op, *om;
  int KS, steps, nin, nout;  // k-steps in the table and in use; valid input / output entries (j, h)
  int ncol;                // columns
  long in_bs, out_bs;      // band strides
  long in_s, out_s;        // strides of the transformed axis
  double sg, scale;
  int c0, c1, c2, hc;      // kC2f
  int eqy, eqz;            // kC2f: the fine axis is the coarse one
};
template <int TH, bool kC2f, int NW>
__global__ void __launch_bounds__(64 * NW, 2) k_rs_pencil_mm(RsPencil g, int ngrp, long groups) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  double2* tab = reinterpret_cast<double2*>(smem_raw);
  const int lane = threadIdx.x & 63, c = lane & 15, q4 = lane >> 4;
  for (int e = threadIdx.x; e < 64 * TH * g.KS; e += 64 * NW) tab[e] = g.tab[e];
  __syncthreads();
  const RsV zero = {0, 0, 0, 0};
  for (long u = (long)blockIdx.x * NW + (threadIdx.x >> 6); u < groups; u += (long)gridDim.x * NW) {
    const long band = u / ngrp;
    const int col = (int)(u - band * ngrp) * 16 + c;
    const bool ok = col < g.ncol;
    const int cc = ok ? col : g.ncol - 1;
    const double2* src = g.in + band * g.in_bs;
    // kC2f: the coarse column (j, i) and which of its axes sit on Nyquist
    int l = 0, i = 0, j = 0;
    bool ni = false, nj = false, dj = false;
    if constexpr (kC2f) {
      l = cc / g.hc;
      i = cc - l * g.hc;
      dj = l >= g.c1;
      j = dj ? g.c1 / 2 : l;
      ni = i == g.c0 / 2;
      nj = j == g.c1 / 2;
      src += (long)j * g.hc + i;
    } else {
      src += cc;
    }
    RsV pr[TH], pi[TH], qr[TH], qi[TH];
#pragma unroll
    for (int t = 0; t < TH; t++) pr[t] = pi[t] = qr[t] = qi[t] = zero;
    double2 a, b;
    auto load = [&](int s) {
      const int k = min(4 * s + q4, g.nin - 1);
      a = src[(long)max(g.ip[k], 0) * g.in_s];
      b = src[(long)max(g.im[k], 0) * g.in_s];
    };
    load(0);
    for (int s = 0; s < g.steps; s++) {
      const int k = 4 * s + q4;
      double fa = 1.0, fb = 1.0;
      if constexpr (kC2f) {
        const bool nk = 2 * k == g.c2;
        // +k (dk = 0) and -k (dk = 1 on the Nyquist plane); an unrefined axis
        // keeps its Nyquist entry and has no second one
        if (!dj) {
          fa = (ni || nj || nk) ? 0.5 : 1.0;
          fb = nk ? ((!ni && (!nj || g.eqy)) ? 0.5 : 0.0) : fa;
        } else {
          fa = (!ni && (!nk || g.eqz)) ? 0.5 : 0.0;
          fb = nk ? (!ni ? 0.5 : 0.0) : fa;
        }
        fa *= g.scale;
        fb *= g.scale;
      }
      const bool va = k < g.nin && g.ip[min(k, g.nin - 1)] >= 0, vb = k < g.nin && g.im[min(k, g.nin - 1)] >= 0;
      const double2 p = va ? make_double2(a.x * fa, a.y * fa) : make_double2(0.0, 0.0);
      const double2 m = vb ? make_double2(b.x * fb, b.y * fb) : make_double2(0.0, 0.0);
      if (s + 1 < g.steps) load(s + 1);
#pragma unroll
      for (int t = 0; t < TH; t++) {
        const double2 q = tab[(t * g.KS + s) * 64 + lane];
        pr[t] = mm16(q.x, p.x + m.x, pr[t]);
        pi[t] = mm16(q.x, p.y + m.y, pi[t]);
        qr[t] = mm16(q.y, p.x - m.x, qr[t]);
        qi[t] = mm16(q.y, p.y - m.y, qi[t]);
      }
    }
    if (!ok) continue;
    double2* dst = g.out + band * g.out_bs + col;
#pragma unroll
    for (int t = 0; t < TH; t++)
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const int h = 16 * t + 4 * r + q4;
        if (h >= g.nout) continue;
        const int op = g.op[h], om = g.om[h];
        const double x = g.sg * qi[t][r], y = g.sg * qr[t][r];  // G(+-h) = P +- i sg Q
        if (op >= 0) dst[op * g.out_s] = make_double2(pr[t][r] - x, pi[t][r] + y);
        if (om >= 0) dst[om * g.out_s] = make_double2(pr[t][r] + x, pi[t][r] - y);
      }
  }
}

}  // namespace pw

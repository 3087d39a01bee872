// Tall-skinny GEMMs of the hot path on MFMA (gfx950), FP64 and FP32.
//
//   TN:  C(n1 x n2) = A^T B, A: K x n1, B: K x n2, K = 2 npw long
//        (Gram blocks Re(X^H Y), projections Re(beta^H X); blas.cpp:997-1029,
//        eigensolver.cpp:471-515, lobpcg.cpp:227-419).  Split-K: each
//        workgroup reduces one K chunk of one tile into a partial buffer; a
//        second kernel sums the partials in a fixed order, so the result is
//        deterministic.
//   NN:  Y(m x n) = alpha A(m x k) B(k x n) + beta Y  (subspace rotations,
//        beta * W; blas.cpp:1031-1067, lobpcg.cpp:445-526);
//        the projector apply inside H Y takes an epilogue that adds H's
//        other terms or forms a Chebyshev step.
//
// Both use the 16x16x4 MFMA (v_mfma_f64_16x16x4f64 / v_mfma_f32_16x16x4f32)
// on operands in registers, or products of split BF16 terms: in registers
// (TN, and NN on an operand split ahead of time) or on tiles in LDS (NN on
// operands that are not).  Lane layout of the 16x16x4 MFMA: A operand lane l = (row l%16, k l/16), B operand lane l =
// (k l/16, col l%16).  Accumulator lane l register i holds column l%16 and
// row 4(l/16)+i for the FP32 MFMA but row 4i + l/16 for the FP64 one
// (checked on gfx950 with a known 16x16x4 product).
#include <algorithm>
#include <cstdlib>
#include <string>

#include "pw_internal.h"

namespace pw {

typedef double d4v __attribute__((ext_vector_type(4)));
typedef float f4v __attribute__((ext_vector_type(4)));

template <typename T> struct acc4;
template <> struct acc4<double> { typedef d4v t; };
template <> struct acc4<float> { typedef f4v t; };

__device__ __forceinline__ d4v mfma16(double a, double b, d4v c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ f4v mfma16(float a, float b, f4v c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

constexpr int BM = 64, BN = 64, BK = 32;

// Block -> (row tile, column tile, K split) for the split-K products, which
// launch ti x tj tiles x nsplit splits as one row of blocks.  Blocks are
// dispatched round-robin over the 8 XCDs (block b to XCD b % 8), each with
// its own L2; giving every XCD one contiguous range of (split, tile) pairs
// puts the ti x tj tiles of a K chunk, which read the same A and B rows, in
// one L2 instead of spreading them over all eight.
struct TnBlock {
  int i, j, split;
};
__device__ __forceinline__ TnBlock tn_block(int n1, int n2, int K, int kc, int t1, int t2) {
  const int ti = (n1 + t1 - 1) / t1, tj = (n2 + t2 - 1) / t2, tiles = ti * tj;
  const int n = tiles * ((K + kc - 1) / kc), b = blockIdx.x;
  const int q = n >> 3, r = n & 7, x = b & 7;
  const int L = x * q + min(x, r) + (b >> 3);
  const int tile = L % tiles;
  return TnBlock{tile % ti, tile / ti, L / tiles};
}

// Four consecutive values of a matrix, at any element's alignment (global
// loads and stores of 16 bytes need 4-byte alignment only).
template <typename T> struct run4;
template <> struct run4<double> { typedef double t __attribute__((ext_vector_type(4), aligned(8))); };
template <> struct run4<float> { typedef float t __attribute__((ext_vector_type(4), aligned(4))); };

// Both native products keep a wavefront's operands in registers, straight
// from global memory: a 64 x 64 tile takes 64 MFMAs per 16 k (4096 cycles in
// FP64, 2048 in FP32) for 8 loads of four values a lane, 8 KiB (4 KiB), so
// the next 16 k arrive during the current ones from L2 with no LDS, no
// barrier and one address step.  The k of an MFMA are any four as long as A
// and B agree: lane group g = lane / 16 takes k = 16 q + 4 g + i for MFMA i,
// four consecutive values where k is the contiguous dimension.  The tiles are
// mfma(b, a) = (A B)^T: accumulator register r holds row lane % 16 (of the
// MFMA's 16) and column acc_col.
template <typename T>
__device__ __forceinline__ int acc_col(int lane, int r) {
  return sizeof(T) == 8 ? 4 * r + (lane >> 4) : 4 * (lane >> 4) + r;
}

// The four wavefronts' tiles of one workgroup, added in LDS in the order of
// their rows, into P (n1 x n2).
template <typename T, int NI, int NJ>
__device__ __forceinline__ void tn_store(const typename acc4<T>::t (&acc)[NI][NJ], int i0, int j0, int n1, int n2,
                                         T* __restrict__ P) {
  typedef typename acc4<T>::t V;
  extern __shared__ __align__(16) unsigned char gemm_smem[];
  V* const red = (V*)gemm_smem;  // [4][NI * NJ][64]
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
#pragma unroll
  for (int a = 0; a < NI; a++)
#pragma unroll
    for (int b = 0; b < NJ; b++) red[((w * NI + a) * NJ + b) * 64 + lane] = acc[a][b];
  __syncthreads();
  for (int e = w; e < NI * NJ; e += 4) {
    V s = red[e * 64 + lane];
#pragma unroll
    for (int v = 1; v < 4; v++) s += red[(v * NI * NJ + e) * 64 + lane];
    const int row = i0 + 16 * (e / NJ) + (lane & 15);
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const int col = j0 + 16 * (e % NJ) + acc_col<T>(lane, r);
      if (row < n1 && col < n2) P[row + (size_t)n1 * col] = s[r];
    }
  }
}

// Partial C tile of A^T B over K rows [kb, ke): P[split](n1 x n2, ld n1), a
// 16 NI x 16 NJ tile per workgroup whose four wavefronts take a quarter of
// the rows each and meet in LDS (4 NI NJ KiB a wavefront in FP64, half in
// FP32), summed in the order of the rows: a quarter of the partials that
// tiles split over the wavefronts write.
template <typename T, int NI, int NJ>
__global__ void __launch_bounds__(256, (int)sizeof(T) * NI * NJ > 96 ? 1 : 2)
k_gemm_tn_partial(const T* __restrict__ A, int lda, const T* __restrict__ B, int ldb, int K, int n1, int n2,
                  int kc, T* __restrict__ P, const T* const* __restrict__ Ab, const T* const* __restrict__ Bb,
                  long sP) {
  typedef typename acc4<T>::t V;
  typedef typename run4<T>::t R;
  if (Ab) {  // product blockIdx.y of a batch: operands from the pointer tables
    A = Ab[blockIdx.y];
    B = Bb[blockIdx.y];
    P += blockIdx.y * sP;
  }
  const TnBlock tb = tn_block(n1, n2, K, kc, 16 * NI, 16 * NJ);
  const int i0 = tb.i * 16 * NI, j0 = tb.j * 16 * NJ, split = tb.split;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, c = lane & 15, g = lane >> 4;
  const int kw = kc >> 2, kb = min(K, split * kc + w * kw), ke = min(K, kb + kw);
  V acc[NI][NJ];
#pragma unroll
  for (int a = 0; a < NI; a++)
#pragma unroll
    for (int b = 0; b < NJ; b++) acc[a][b] = V{0, 0, 0, 0};
  const T *pa[NI], *pb[NJ];  // columns beyond the matrix repeat its last one
#pragma unroll
  for (int a = 0; a < NI; a++) pa[a] = A + (size_t)min(i0 + 16 * a + c, n1 - 1) * lda;
#pragma unroll
  for (int b = 0; b < NJ; b++) pb[b] = B + (size_t)min(j0 + 16 * b + c, n2 - 1) * ldb;
  auto mm = [&](const R (&ra)[NI], const R (&rb)[NJ]) {
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
      for (int a = 0; a < NI; a++)
#pragma unroll
        for (int b = 0; b < NJ; b++) acc[a][b] = mfma16(rb[b][i], ra[a][i], acc[a][b]);
  };
  const int nq = (ke - kb) >> 4;  // full chunks of 16 rows
  if (nq > 0) {
    auto load = [&](R (&ra)[NI], R (&rb)[NJ], int q) {
      const int k = kb + 16 * min(q, nq - 1) + 4 * g;  // (the chunk past the end: read and dropped)
#pragma unroll
      for (int a = 0; a < NI; a++) ra[a] = *(const R*)(pa[a] + k);
#pragma unroll
      for (int b = 0; b < NJ; b++) rb[b] = *(const R*)(pb[b] + k);
    };
    R a0[NI], b0[NJ], a1[NI], b1[NJ];
    load(a0, b0, 0);
    int q = 0;
    for (; q + 2 <= nq; q += 2) {
      load(a1, b1, q + 1);
      mm(a0, b0);
      load(a0, b0, q + 2);
      mm(a1, b1);
    }
    if (q < nq) mm(a0, b0);
  }
  if (kb + 16 * nq < ke) {  // the last, incomplete chunk
    R ra[NI], rb[NJ];
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const int k = kb + 16 * nq + 4 * g + i, kk = min(k, ke - 1);
#pragma unroll
      for (int a = 0; a < NI; a++) ra[a][i] = k < ke ? pa[a][kk] : (T)0;
#pragma unroll
      for (int b = 0; b < NJ; b++) rb[b][i] = k < ke ? pb[b][kk] : (T)0;
    }
    mm(ra, rb);
  }
  tn_store<T, NI, NJ>(acc, i0, j0, n1, n2, P + (size_t)split * n1 * n2);
}

// ---- split BF16 products (FP32 data, FP32 accumulation) ----
// Each FP32 operand x is split into NS BF16 terms rounded to nearest even:
// NS = 2: x = hi + lo (16 significant bits), NS = 3: x = hi + mid + lo (24
// bits, FP32's).  A product a b is the sum of the term products down to
// 2^-8 (NS - 1) relative: NS = 2: a_lo b_hi + a_hi b_lo + a_hi b_hi; NS = 3:
// a_lo b_hi + a_hi b_lo + a_mid b_mid + a_mid b_hi + a_hi b_mid + a_hi b_hi
// (smallest first), on v_mfma_f32_16x16x32_bf16, whose operand lane l holds
// row (or column) l % 16 and k = 8 (l / 16) .. 8 (l / 16) + 7 and whose
// accumulator is laid out as v_mfma_f32_16x16x4f32's.
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

// Round to nearest even: one v_cvt_pk_bf16_f32 per pair of values on
// gfx950; x - hi is exact in FP32, so the terms sum to x up to the last
// term's rounding.
template <int NS>
__device__ __forceinline__ void bf16_split(float x, unsigned short (&t)[NS]) {
  float r = x;
#pragma unroll
  for (int i = 0; i < NS; i++) {
    const __bf16 h = (__bf16)r;
    t[i] = __builtin_bit_cast(unsigned short, h);
    r -= (float)h;
  }
}
// Four values (two pairs) into NS packed BF16 term pairs: term i of x0, x1
// in t[i].x (x0 in the low half), of x2, x3 in t[i].y; the same terms as
// bf16_split (one v_cvt_pk_bf16_f32 per pair and term).
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
template <int NS>
__device__ __forceinline__ void bf16_split4(float2 p, float2 q, uint2 (&t)[NS]) {
  float r0 = p.x, r1 = p.y, r2 = q.x, r3 = q.y;
#pragma unroll
  for (int i = 0; i < NS; i++) {
    const bf16x2 h01 = {(__bf16)r0, (__bf16)r1}, h23 = {(__bf16)r2, (__bf16)r3};
    const unsigned u = __builtin_bit_cast(unsigned, h01), v = __builtin_bit_cast(unsigned, h23);
    t[i].x = u;
    t[i].y = v;
    if (i + 1 < NS) {  // residuals from the packed words (a BF16 is the top half of its FP32)
      r0 -= __uint_as_float(u << 16);
      r1 -= __uint_as_float(u & 0xffff0000u);
      r2 -= __uint_as_float(v << 16);
      r3 -= __uint_as_float(v & 0xffff0000u);
    }
  }
}
__device__ __forceinline__ f4v mfma_b16(const unsigned short* a, const unsigned short* b, f4v acc) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(*reinterpret_cast<const bf16x8*>(a),
                                                 *reinterpret_cast<const bf16x8*>(b), acc, 0, 0, 0);
}
// a[i], b[i]: the i-th BF16 term tiles (16 x 32 operands at the lane's
// offset); NS term tiles each, at a common offset.
template <int NS>
__device__ __forceinline__ f4v mfma_split(const unsigned short* const (&a)[NS], const unsigned short* const (&b)[NS],
                                          f4v acc) {
  if constexpr (NS == 3) {
    acc = mfma_b16(a[2], b[0], acc);
    acc = mfma_b16(a[0], b[2], acc);
    acc = mfma_b16(a[1], b[1], acc);
  }
  acc = mfma_b16(a[1], b[0], acc);
  acc = mfma_b16(a[0], b[1], acc);
  return mfma_b16(a[0], b[0], acc);
}
constexpr int BKP = 40;  // LDS row stride of the bf16 tiles (80 bytes: 16-byte aligned rows)
// The term pairs of mfma_split in its order (smallest first): NS = 3 uses
// all six, NS = 2 the last three.  Loops over (pair, tile) in this order
// give every tile the same sequence of products while consecutive MFMAs
// write different accumulators.
__device__ constexpr int kSplitPairA[6] = {2, 0, 1, 1, 0, 0};
__device__ constexpr int kSplitPairB[6] = {0, 2, 1, 0, 1, 0};

// k_gemm_tn_partial with FP32 inputs split into NS BF16 terms: a lane loads
// eight consecutive rows of a column per 32-row chunk (its operand of one
// 16x16x32 product per kept pairing of terms, in place of eight 16x16x4 FP32
// products) and splits them in registers.  The splitting (about 50 VALU
// operations an operand tile) costs as much as the products; the two
// wavefronts of a SIMD overlap one's with the other's.  13134 x 256 x 256:
// 21.5 us (28.1 through LDS tiles of 64 x 64 split over the wavefronts).
template <int NS>
__device__ __forceinline__ void split8(const f4v& lo, const f4v& hi, bf16x8 (&t)[NS]) {
  uint2 u[NS], v[NS];
  bf16_split4<NS>(float2{lo[0], lo[1]}, float2{lo[2], lo[3]}, u);
  bf16_split4<NS>(float2{hi[0], hi[1]}, float2{hi[2], hi[3]}, v);
#pragma unroll
  for (int i = 0; i < NS; i++) t[i] = __builtin_bit_cast(bf16x8, uint4{u[i].x, u[i].y, v[i].x, v[i].y});
}
template <int NI, int NJ, int NS>
__global__ void __launch_bounds__(256, 2)
k_gemm_tn_partial_bf(const float* __restrict__ A, int lda, const float* __restrict__ B, int ldb, int K, int n1,
                     int n2, int kc, float* __restrict__ P) {
  typedef run4<float>::t R;
  const TnBlock tb = tn_block(n1, n2, K, kc, 16 * NI, 16 * NJ);
  const int i0 = tb.i * 16 * NI, j0 = tb.j * 16 * NJ, split = tb.split;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, c = lane & 15, g = lane >> 4;
  const int kw = kc >> 2, kb = min(K, split * kc + w * kw), ke = min(K, kb + kw);
  f4v acc[NI][NJ];
#pragma unroll
  for (int a = 0; a < NI; a++)
#pragma unroll
    for (int b = 0; b < NJ; b++) acc[a][b] = f4v{0, 0, 0, 0};
  const float *pa[NI], *pb[NJ];  // columns beyond the matrix repeat its last one
#pragma unroll
  for (int a = 0; a < NI; a++) pa[a] = A + (size_t)min(i0 + 16 * a + c, n1 - 1) * lda;
#pragma unroll
  for (int b = 0; b < NJ; b++) pb[b] = B + (size_t)min(j0 + 16 * b + c, n2 - 1) * ldb;
  auto mm = [&](const f4v (&ra)[NI][2], const f4v (&rb)[NJ][2]) {
    bf16x8 fa[NI][NS];
#pragma unroll
    for (int a = 0; a < NI; a++) split8<NS>(ra[a][0], ra[a][1], fa[a]);
#pragma unroll
    for (int b = 0; b < NJ; b++) {
      bf16x8 fb[NS];
      split8<NS>(rb[b][0], rb[b][1], fb);
      // term pair outer, tiles inner: mfma_split's order per tile
#pragma unroll
      for (int p = 6 - (NS == 3 ? 6 : 3); p < 6; p++)
#pragma unroll
        for (int a = 0; a < NI; a++)
          acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fb[kSplitPairB[p]], fa[a][kSplitPairA[p]], acc[a][b],
                                                               0, 0, 0);
    }
  };
  f4v ra[NI][2], rb[NJ][2];
  const int nq = (ke - kb) >> 5;  // full chunks of 32 rows
  if (nq > 0) {
    auto load = [&](f4v (&xa)[NI][2], f4v (&xb)[NJ][2], int q) {
      const int k = kb + 32 * min(q, nq - 1) + 8 * g;  // (the chunk past the end: read and dropped)
#pragma unroll
      for (int h = 0; h < 2; h++) {
#pragma unroll
        for (int a = 0; a < NI; a++) xa[a][h] = *(const R*)(pa[a] + k + 4 * h);
#pragma unroll
        for (int b = 0; b < NJ; b++) xb[b][h] = *(const R*)(pb[b] + k + 4 * h);
      }
    };
    load(ra, rb, 0);
    for (int q = 0; q < nq; q++) {
      f4v xa[NI][2], xb[NJ][2];
      load(xa, xb, q + 1);
      mm(ra, rb);
#pragma unroll
      for (int h = 0; h < 2; h++) {
#pragma unroll
        for (int a = 0; a < NI; a++) ra[a][h] = xa[a][h];
#pragma unroll
        for (int b = 0; b < NJ; b++) rb[b][h] = xb[b][h];
      }
    }
  }
  if (kb + 32 * nq < ke) {  // the last, incomplete chunk
#pragma unroll
    for (int i = 0; i < 8; i++) {
      const int k = kb + 32 * nq + 8 * g + i, kk = min(k, ke - 1);
#pragma unroll
      for (int a = 0; a < NI; a++) ra[a][i >> 2][i & 3] = k < ke ? pa[a][kk] : 0.f;
#pragma unroll
      for (int b = 0; b < NJ; b++) rb[b][i >> 2][i & 3] = k < ke ? pb[b][kk] : 0.f;
    }
    mm(ra, rb);
  }
  tn_store<float, NI, NJ>(acc, i0, j0, n1, n2, P + (size_t)split * n1 * n2);
}

// C[i + ldc j] = rowscale[i] * sum_s P[s][i + n1 j] (+ beta C), rowscale may
// be null.  The partials are summed in split order (deterministic), 16
// loads in flight at a time.
template <typename T>
__global__ void k_gemm_tn_reduce(const T* __restrict__ P, int nsplit, int n1, int n2, T* __restrict__ C, int ldc,
                                 const T* __restrict__ rowscale, T beta, T* const* __restrict__ Cb, long sP) {
  if (Cb) {  // product blockIdx.y of a batch
    C = Cb[blockIdx.y];
    P += blockIdx.y * sP;
  }
  const long total = (long)n1 * n2;
  for (long e = blockIdx.x * (long)blockDim.x + threadIdx.x; e < total; e += (long)gridDim.x * blockDim.x) {
    const int i = (int)(e % n1), j = (int)(e / n1);
    T s = 0;
    for (int q0 = 0; q0 < nsplit; q0 += 16) {
      T v[16];
#pragma unroll
      for (int u = 0; u < 16; u++) v[u] = (q0 + u < nsplit) ? P[(size_t)(q0 + u) * total + e] : (T)0;
#pragma unroll
      for (int u = 0; u < 16; u++) s += v[u];
    }
    if (rowscale) s *= rowscale[i];
    T* c = C + i + (size_t)ldc * j;
    *c = (beta == (T)0) ? s : s + beta * *c;
  }
}

// Tile origin of block blockIdx.x in the one-row grid of ti x tj BM x BN
// output tiles of the NN products: the tj column tiles of a row tile, which
// read the same rows of A, are consecutive items, and xcd_item puts runs of
// consecutive items on one XCD (one L2).
__device__ __forceinline__ void nn_tile_origin(int m, int n, int& i0, int& j0) {
  const int ti = (m + BM - 1) / BM, tj = (n + BN - 1) / BN;
  const int item = xcd_item(blockIdx.x, ti * tj), i = item / tj;
  i0 = i * BM;
  j0 = (item - i * tj) * BN;
}

// Epilogue of the projector apply inside H Y (acc = (beta w) W for one
// output element e = row + ld col):
//   kCheb == false: out[e] = H[e] + acc                    (H Y += beta w W)
//   kCheb == true:  out[e] = s1 (H[e] + acc - c Yc[e]) - s2 Yp[e]
// with (c, s1, s2) = coef[3 step ..] and Yp == null meaning s2 = 0: one step
// of the scaled Chebyshev three-term recurrence fused with H Y's last term.
// out may alias H or Yp, not Yc.
// The plain product uses the same kernels with out[e] = alpha acc + beta H[e]
// (H read only when beta != 0; H may alias out).
template <typename T>
struct NnEpilogue {
  const T* H;
  const T* Yc;
  const T* Yp;
  T* out;
  int ld;
  const T* coef;
  int step;
  T alpha, beta;
};

template <typename T, bool kCheb>
__device__ __forceinline__ void nn_epilogue(const NnEpilogue<T>& ep, size_t e, T acc) {
  if constexpr (kCheb) {
    const T h = ep.H[e] + acc;
    const T c = ep.coef[3 * ep.step], s1 = ep.coef[3 * ep.step + 1], s2 = ep.coef[3 * ep.step + 2];
    T v = (h - c * ep.Yc[e]) * s1;
    if (ep.Yp) v -= s2 * ep.Yp[e];
    ep.out[e] = v;
  } else {
    const T v = ep.alpha * acc;
    ep.out[e] = ep.beta == (T)0 ? v : v + ep.beta * ep.H[e];
  }
}

// The same for four consecutive rows.
template <typename T, bool kCheb>
__device__ __forceinline__ void nn_epilogue4(const NnEpilogue<T>& ep, size_t e, typename run4<T>::t acc) {
  typedef typename run4<T>::t R;
  if constexpr (kCheb) {
    const R h = *(const R*)(ep.H + e) + acc;
    const T c = ep.coef[3 * ep.step], s1 = ep.coef[3 * ep.step + 1], s2 = ep.coef[3 * ep.step + 2];
    R v = (h - c * *(const R*)(ep.Yc + e)) * s1;
    if (ep.Yp) v -= s2 * *(const R*)(ep.Yp + e);
    *(R*)(ep.out + e) = v;
  } else {
    R v = ep.alpha * acc;
    if (ep.beta != (T)0) v += ep.beta * *(const R*)(ep.H + e);
    *(R*)(ep.out + e) = v;
  }
}

// Y-tile product A (m x k) B (k x n) with FP32 inputs split into NS BF16
// terms, FP32 accumulation, and the epilogue above.  64 x 64 tiles, four
// waves of 32 x 32, 32-deep K chunks: A chunk loads are 64-row runs (lane =
// row, 8 k per thread), B chunk loads 8 contiguous k of one column per
// thread; both are split and stored as k-contiguous BF16 rows so that one
// 16-byte LDS read is one MFMA operand.  The finished tile goes through LDS
// so that the epilogue reads and writes 16 contiguous rows per thread.
template <bool kCheb, int NS>
__global__ void __launch_bounds__(256)
k_gemm_nn_bf(const float* __restrict__ A, int lda, const float* __restrict__ B, int ldb, int m, int n, int k,
             NnEpilogue<float> ep) {
  __shared__ __align__(16) unsigned short Sh[2 * NS * 64 * BKP > 64 * 65 * 2 ? 2 * NS * 64 * BKP : 64 * 65 * 2];
  unsigned short* As = Sh;                 // NS term tiles of A (64 rows x 32 k)
  unsigned short* Bs = Sh + NS * 64 * BKP;  // NS term tiles of B (64 columns x 32 k)
  int i0, j0;
  nn_tile_origin(m, n, i0, j0);
  const int t = threadIdx.x, lane = t & 63, w = t >> 6;
  const int wi = (w & 1) * 32, wj = (w >> 1) * 32;
  f4v acc[2][2];
#pragma unroll
  for (int a = 0; a < 2; a++)
#pragma unroll
    for (int b = 0; b < 2; b++) acc[a][b] = f4v{0, 0, 0, 0};
  const int arow = i0 + (t & 63), ak = 8 * (t >> 6);
  const int bcol = j0 + (t >> 2), bk = 8 * (t & 3);
  const int fr = lane & 15, fk = 8 * (lane >> 4);
  auto pack = [](const unsigned short* v) {
    return uint4{v[0] | ((unsigned)v[1] << 16), v[2] | ((unsigned)v[3] << 16), v[4] | ((unsigned)v[5] << 16),
                 v[6] | ((unsigned)v[7] << 16)};
  };
  for (int k0 = 0; k0 < k; k0 += BK) {
    unsigned short ta[NS][8], tb[NS][8];
#pragma unroll
    for (int j = 0; j < 8; j++) {
      const int ka = k0 + ak + j, kb2 = k0 + bk + j;
      const float x = (arow < m && ka < k) ? A[(size_t)ka * lda + arow] : 0.f;
      const float y = (bcol < n && kb2 < k) ? B[(size_t)bcol * ldb + kb2] : 0.f;
      unsigned short sx[NS], sy[NS];
      bf16_split<NS>(x, sx);
      bf16_split<NS>(y, sy);
#pragma unroll
      for (int i = 0; i < NS; i++) {
        ta[i][j] = sx[i];
        tb[i][j] = sy[i];
      }
    }
#pragma unroll
    for (int i = 0; i < NS; i++) {
      *reinterpret_cast<uint4*>(As + i * 64 * BKP + (t & 63) * BKP + ak) = pack(ta[i]);
      *reinterpret_cast<uint4*>(Bs + i * 64 * BKP + (t >> 2) * BKP + bk) = pack(tb[i]);
    }
    __syncthreads();
#pragma unroll
    for (int a = 0; a < 2; a++)
#pragma unroll
      for (int b = 0; b < 2; b++) {
        const int oa = (wi + a * 16 + fr) * BKP + fk, ob = (wj + b * 16 + fr) * BKP + fk;
        const unsigned short* pa[NS];
        const unsigned short* pb[NS];
#pragma unroll
        for (int i = 0; i < NS; i++) {
          pa[i] = As + i * 64 * BKP + oa;
          pb[i] = Bs + i * 64 * BKP + ob;
        }
        acc[a][b] = mfma_split<NS>(pa, pb, acc[a][b]);
      }
    __syncthreads();
  }
  // tile (64 x 64 floats, column stride 65) through LDS
  float* Ct = reinterpret_cast<float*>(Sh);
#pragma unroll
  for (int a = 0; a < 2; a++)
#pragma unroll
    for (int b = 0; b < 2; b++)
#pragma unroll
      for (int i = 0; i < 4; i++)
        Ct[(wj + b * 16 + (lane & 15)) * 65 + wi + a * 16 + acc_col<float>(lane, i)] = acc[a][b][i];
  __syncthreads();
  const int col = j0 + (t >> 2), r0 = 16 * (t & 3);
  if (col < n) {
    for (int rr = 0; rr < 16; rr++) {
      const int row = i0 + r0 + rr;
      if (row < m) nn_epilogue<float, kCheb>(ep, (size_t)col * ep.ld + row, Ct[(t >> 2) * 65 + r0 + rr]);
    }
  }
}

// ---- products with operands split ahead of time ----
// Operand tile layout (both operands): for a 16-row (or 16-column) tile r
// and a 32-deep K chunk q, the NS_MAX = 3 term blocks of 64 lanes x 8 BF16
// (one 16-byte v_mfma_f32_16x16x32_bf16 operand per lane: row / column
// l % 16, k = 32 q + 8 (l / 16) .. + 7) sit at ((r nkc + q) 3 + i) 512
// BF16 elements, so that a wave loads an operand with one 1 KiB read.  Rows,
// columns and k beyond the matrix are zero.  The 2-term split is the first
// two terms of the 3-term one.
constexpr int kSplitTerms = 3;
typedef unsigned short u16x8 __attribute__((ext_vector_type(8)));

// One operand group (r, q) per lane-block: A column-major (ld lda): rows
// of A are the tile dimension (transpose = false), or columns of B
// (transpose = true, B column-major with ld ldb: B(k, col) at col ldb + k).
template <bool kCols>
__global__ void k_split_operand(const float* __restrict__ X, int ldx, int nr, int K, int nkc,
                                unsigned short* __restrict__ out, long ngroups) {
  const long g = (long)blockIdx.x * (blockDim.x / 64) + (threadIdx.x >> 6);
  if (g >= ngroups) return;
  const int lane = threadIdx.x & 63;
  const int r = (int)(g / nkc), q = (int)(g - (long)r * nkc);
  const int idx = 16 * r + (lane & 15), k0 = 32 * q + 8 * (lane >> 4);
  unsigned short t[kSplitTerms][8];
#pragma unroll
  for (int j = 0; j < 8; j++) {
    const int k = k0 + j;
    float x = 0.f;
    if (idx < nr && k < K) x = kCols ? X[(size_t)idx * ldx + k] : X[(size_t)k * ldx + idx];
    unsigned short v[kSplitTerms];
    bf16_split<kSplitTerms>(x, v);
#pragma unroll
    for (int i = 0; i < kSplitTerms; i++) t[i][j] = v[i];
  }
#pragma unroll
  for (int i = 0; i < kSplitTerms; i++) {
    u16x8 v;
#pragma unroll
    for (int j = 0; j < 8; j++) v[j] = t[i][j];
    *reinterpret_cast<u16x8*>(out + ((size_t)g * kSplitTerms + i) * 512 + 8 * lane) = v;
  }
}


// out = epilogue(A B) with both operands split ahead of time (layout above;
// A: nrt = ceil(m / 16) row tiles, B: ceil(n / 16) column tiles, nkc
// chunks).  A workgroup takes 64 rows x 256 columns: wave w the 64 x 64
// block of columns 64 w .., as 4 x 4 MFMA tiles whose operands come
// straight from global memory (A from HBM, shared by the four waves through
// the caches; B from L2), the next chunk's operands in flight during the
// current chunk's products.  (Staging the A slab in LDS measured slower:
// 42 against 38 us at 13134 x 256 x 256.)  The epilogue works on the
// accumulator layout: a lane's four rows of one column are contiguous, read
// and written as two float pairs (m and ld even).
template <bool kCheb, int NS, int RT = 4>
__global__ void __launch_bounds__(256, 1)
k_gemm_nn_pre(const unsigned short* __restrict__ Ab, const unsigned short* __restrict__ Bb, int m, int n, int nkc,
              NnEpilogue<float> ep) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int nrt = (m + 15) >> 4, nct = (n + 15) >> 4;
  const int rt0 = RT * blockIdx.x, ct0 = 16 * blockIdx.y + 4 * w;
  const int na = min(RT, nrt - rt0), nbt = min(4, nct - ct0);
  if (nbt <= 0) return;
  const bf16x8* A8 = reinterpret_cast<const bf16x8*>(Ab);
  const bf16x8* B8 = reinterpret_cast<const bf16x8*>(Bb);
  f4v acc[RT][4];
#pragma unroll
  for (int a = 0; a < RT; a++)
#pragma unroll
    for (int b = 0; b < 4; b++) acc[a][b] = f4v{0, 0, 0, 0};
  bf16x8 av[RT][NS], bv[4][NS];
  auto load = [&](int q, bf16x8 (&xa)[RT][NS], bf16x8 (&xb)[4][NS]) {
#pragma unroll
    for (int a = 0; a < RT; a++)
#pragma unroll
      for (int i = 0; i < NS; i++)
        xa[a][i] = a < na ? A8[((size_t)((rt0 + a) * nkc + q) * kSplitTerms + i) * 64 + lane] : bf16x8{};
#pragma unroll
    for (int b = 0; b < 4; b++)
#pragma unroll
      for (int i = 0; i < NS; i++)
        xb[b][i] = b < nbt ? B8[((size_t)((ct0 + b) * nkc + q) * kSplitTerms + i) * 64 + lane] : bf16x8{};
  };
  load(0, av, bv);
  for (int q = 0; q < nkc; q++) {
    bf16x8 an[RT][NS], bn[4][NS];
    if (q + 1 < nkc) load(q + 1, an, bn);
    // term pair outer, tiles inner: the order of mfma_split per tile, while
    // consecutive MFMAs write different accumulators
#pragma unroll
    for (int p = 6 - (NS == 3 ? 6 : 3); p < 6; p++)
#pragma unroll
      for (int a = 0; a < RT; a++)
#pragma unroll
        for (int b = 0; b < 4; b++)
          acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av[a][kSplitPairA[p]], bv[b][kSplitPairB[p]],
                                                               acc[a][b], 0, 0, 0);
    if (q + 1 < nkc) {
#pragma unroll
      for (int a = 0; a < 4; a++)
#pragma unroll
        for (int i = 0; i < NS; i++) {
          if (a < RT) av[a][i] = an[a][i];
          bv[a][i] = bn[a][i];
        }
    }
  }
  float cc = 0.f, s1 = 0.f, s2 = 0.f;
  if constexpr (kCheb) {
    cc = ep.coef[3 * ep.step];
    s1 = ep.coef[3 * ep.step + 1];
    s2 = ep.coef[3 * ep.step + 2];
  }
#pragma unroll
  for (int b = 0; b < 4; b++) {
    const int col = 16 * (ct0 + b) + (lane & 15);
    if (b >= nbt || col >= n) continue;
#pragma unroll
    for (int a = 0; a < RT; a++) {
      const int r0 = 16 * (rt0 + a) + 4 * (lane >> 4);
      if (a >= na) continue;
#pragma unroll
      for (int h = 0; h < 2; h++) {
        const int row = r0 + 2 * h;
        if (row >= m) continue;
        const size_t e = (size_t)col * ep.ld + row;
        const float x0 = acc[a][b][2 * h], x1 = acc[a][b][2 * h + 1];
        float2 o;
        if constexpr (kCheb) {
          const float2 hv = *reinterpret_cast<const float2*>(ep.H + e);
          const float2 yc = *reinterpret_cast<const float2*>(ep.Yc + e);
          o.x = (hv.x + x0 - cc * yc.x) * s1;
          o.y = (hv.y + x1 - cc * yc.y) * s1;
          if (ep.Yp) {
            const float2 yp = *reinterpret_cast<const float2*>(ep.Yp + e);
            o.x -= s2 * yp.x;
            o.y -= s2 * yp.y;
          }
        } else {
          o.x = ep.alpha * x0;
          o.y = ep.alpha * x1;
          if (ep.beta != 0.f) {
            const float2 hv = *reinterpret_cast<const float2*>(ep.H + e);
            o.x += ep.beta * hv.x;
            o.y += ep.beta * hv.y;
          }
        }
        *reinterpret_cast<float2*>(ep.out + e) = o;
      }
    }
  }
}

// The same product in the operands' own precision: a wavefront takes 64 rows
// x 16 NJ columns, the four of a workgroup consecutive (row, column) tiles,
// so that where n > 16 NJ they read the same rows of A.  MFMA row c of row
// tile t is row 4 c + t: one load of four consecutive rows per lane and k
// feeds four MFMAs, and a lane's results are four consecutive rows too.  The
// last rows' lanes start early enough to stay inside the matrix and write
// only what no other lane does.
template <typename T, int NJ, bool kCheb>
__global__ void __launch_bounds__(256, 2)
k_gemm_nn_ep(const T* __restrict__ A, int lda, const T* __restrict__ B, int ldb, int m, int n, int k,
             NnEpilogue<T> ep) {
  typedef typename acc4<T>::t V;
  typedef typename run4<T>::t R;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, c = lane & 15, g = lane >> 4;
  const int ti = (m + 63) / 64, tj = (n + 16 * NJ - 1) / (16 * NJ);
  const int item = 4 * xcd_item(blockIdx.x, gridDim.x) + w;
  if (item >= ti * tj) return;
  const int i = item / tj, j0 = 16 * NJ * (item - i * tj);
  const int r0 = 64 * i + 4 * c, rb0 = max(0, min(r0, m - 4));
  V acc[4][NJ];
#pragma unroll
  for (int t = 0; t < 4; t++)
#pragma unroll
    for (int b = 0; b < NJ; b++) acc[t][b] = V{0, 0, 0, 0};
  const T *pa = A + rb0, *pb[NJ];
#pragma unroll
  for (int b = 0; b < NJ; b++) pb[b] = B + (size_t)min(j0 + 16 * b + c, n - 1) * ldb;
  auto mm = [&](const R (&ra)[4], const R (&rb)[NJ]) {
#pragma unroll
    for (int q = 0; q < 4; q++)
#pragma unroll
      for (int b = 0; b < NJ; b++)
#pragma unroll
        for (int t = 0; t < 4; t++) acc[t][b] = mfma16(rb[b][q], ra[q][t], acc[t][b]);
  };
  const int nq = m >= 4 ? k >> 4 : 0;
  if (nq > 0) {
    auto load = [&](R (&ra)[4], R (&rb)[NJ], int q) {
      const int k0 = 16 * min(q, nq - 1) + 4 * g;
#pragma unroll
      for (int u = 0; u < 4; u++) ra[u] = *(const R*)(pa + (size_t)(k0 + u) * lda);
#pragma unroll
      for (int b = 0; b < NJ; b++) rb[b] = *(const R*)(pb[b] + k0);
    };
    R a0[4], b0[NJ], a1[4], b1[NJ];
    load(a0, b0, 0);
    int q = 0;
    for (; q + 2 <= nq; q += 2) {
      load(a1, b1, q + 1);
      mm(a0, b0);
      load(a0, b0, q + 2);
      mm(a1, b1);
    }
    if (q < nq) mm(a0, b0);
  }
  for (int k1 = 16 * nq; k1 < k; k1 += 16) {  // the last, incomplete chunk (all of them where m < 4)
    R ra[4], rb[NJ];
#pragma unroll
    for (int u = 0; u < 4; u++) {
      const int kq = k1 + 4 * g + u, kk = min(kq, k - 1);
#pragma unroll
      for (int t = 0; t < 4; t++) ra[u][t] = kq < k ? A[(size_t)kk * lda + min(rb0 + t, m - 1)] : (T)0;
#pragma unroll
      for (int b = 0; b < NJ; b++) rb[b][u] = kq < k ? pb[b][kk] : (T)0;
    }
    mm(ra, rb);
  }
#pragma unroll
  for (int b = 0; b < NJ; b++)
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const int col = j0 + 16 * b + acc_col<T>(lane, r);
      if (col >= n || r0 >= m) continue;
      const size_t e = (size_t)col * ep.ld + rb0;
      if (rb0 == r0 && m >= 4)
        nn_epilogue4<T, kCheb>(ep, e, R{acc[0][b][r], acc[1][b][r], acc[2][b][r], acc[3][b][r]});
      else
#pragma unroll
        for (int t = 0; t < 4; t++)
          if (rb0 + t >= r0 && rb0 + t < m) nn_epilogue<T, kCheb>(ep, e + t, acc[t][b][r]);
    }
}

// Elementwise form of the epilogue (no projectors: acc = 0).
template <typename T, bool kCheb>
__global__ void k_nn_epilogue_only(long m, int n, NnEpilogue<T> ep) {
  const long total = m * n;
  for (long e = blockIdx.x * (long)blockDim.x + threadIdx.x; e < total; e += (long)gridDim.x * blockDim.x) {
    const long col = e / m, row = e - col * m;
    nn_epilogue<T, kCheb>(ep, (size_t)col * ep.ld + row, (T)0);
  }
}

// Single-column products (the one-band H x of Lanczos): GEMV kernels.
// C(n1) = A^T b over K: workgroup (i, split) sums column i of A against b
// over one K range, 256 threads with 8 loads in flight each; partials go
// through k_gemm_tn_reduce like the split-K GEMM.
template <typename T>
__global__ void __launch_bounds__(256)
k_gemv_t_partial(const T* __restrict__ A, int lda, const T* __restrict__ b, int K, int kc, int n1,
                 T* __restrict__ P) {
  const int i = blockIdx.x, split = blockIdx.y;
  const int kb = split * kc, ke = min(K, kb + kc);
  const T* a = A + (size_t)i * lda;
  T s = 0;
  for (int r0 = kb + threadIdx.x; r0 < ke; r0 += 8 * 256) {
    T x[8], y[8];
#pragma unroll
    for (int u = 0; u < 8; u++) {
      const int r = r0 + 256 * u;
      x[u] = r < ke ? a[r] : (T)0;
      y[u] = r < ke ? b[r] : (T)0;
    }
#pragma unroll
    for (int u = 0; u < 8; u++) s += x[u] * y[u];
  }
  __shared__ T red[256];
  red[threadIdx.x] = s;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) P[(size_t)split * n1 + i] = red[0];
}

// y = alpha A x + beta y, A m x k: workgroup of NW waves per 64 rows; wave
// w sums columns j = w (mod NW) for its 64 rows (16 loads in flight per
// lane), the NW partial rows meet in LDS in a fixed order.  NW = 16 for
// k >= 128: one round of loads per wave, four times the waves in flight
// (the single-column products of the Lanczos steps are latency-bound).
template <typename T, int NW>
__global__ void __launch_bounds__(64 * NW)
k_gemv_n(const T* __restrict__ A, int lda, const T* __restrict__ x, T* __restrict__ y, int m, int k, T alpha,
         T beta) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int row = blockIdx.x * 64 + lane;
  T s = 0;
  if (row < m) {
    for (int j0 = w; j0 < k; j0 += 16 * NW) {
      T a[16];
#pragma unroll
      for (int u = 0; u < 16; u++) {
        const int j = j0 + NW * u;
        a[u] = j < k ? A[(size_t)j * lda + row] : (T)0;
      }
#pragma unroll
      for (int u = 0; u < 16; u++) {
        const int j = j0 + NW * u;
        if (j < k) s += a[u] * x[j];
      }
    }
  }
  __shared__ T red[NW][64];
  red[w][lane] = s;
  __syncthreads();
  if (w == 0 && row < m) {
    T v = 0;
#pragma unroll
    for (int q = 0; q < NW; q++) v += red[q][lane];
    v *= alpha;
    y[row] = (beta == (T)0) ? v : v + beta * y[row];
  }
}

template <typename T>
static void launch_gemv_n(pw_ctx* c, const T* A, int lda, const T* x, T* y, int m, int k, T alpha, T beta) {
  if (k >= 128)
    hipLaunchKernelGGL((k_gemv_n<T, 16>), dim3((m + 63) / 64), dim3(1024), 0, c->stream, A, lda, x, y, m, k, alpha,
                       beta);
  else
    hipLaunchKernelGGL((k_gemv_n<T, 4>), dim3((m + 63) / 64), dim3(256), 0, c->stream, A, lda, x, y, m, k, alpha,
                       beta);
}

// The context's split-K partial buffer, grown to need bytes (allocates).
static int grow_gemm_ws(pw_ctx* c, size_t need) {
  if (need <= c->gemm_ws_bytes) return PW_OK;
  invalidate_graph(c);
  if (c->d_gemm_ws) (void)hipFree(c->d_gemm_ws);
  c->d_gemm_ws = nullptr;
  c->gemm_ws_bytes = 0;
  PW_HIP(hipMalloc(&c->d_gemm_ws, need));
  c->gemm_ws_bytes = need;
  return PW_OK;
}

// 16-wide tiles of a workgroup along a dimension of n: as few workgroups of
// up to most tiles as cover it, evenly filled (77 columns are two of 48, not
// of 64).
static int tiles16(int n, int most) {
  const int t = (n + 15) / 16, nb = (t + most - 1) / most;
  return std::max(2, (t + nb - 1) / nb);
}

template <typename T>
using TnKernel = void (*)(const T*, int, const T*, int, int, int, int, int, T*, const T* const*, const T* const*, long);

template <typename T>
static TnKernel<T> tn_kernel(int ni, int nj) {
  static const TnKernel<T> k[3][3] = {
      {k_gemm_tn_partial<T, 2, 2>, k_gemm_tn_partial<T, 2, 3>, k_gemm_tn_partial<T, 2, 4>},
      {k_gemm_tn_partial<T, 3, 2>, k_gemm_tn_partial<T, 3, 3>, k_gemm_tn_partial<T, 3, 4>},
      {k_gemm_tn_partial<T, 4, 2>, k_gemm_tn_partial<T, 4, 3>, k_gemm_tn_partial<T, 4, 4>}};
  return k[ni - 2][nj - 2];
}

using TnKernelBf = void (*)(const float*, int, const float*, int, int, int, int, int, float*);

template <int NS>
static TnKernelBf tn_kernel_bf(int ni, int nj) {
  static const TnKernelBf k[3][3] = {
      {k_gemm_tn_partial_bf<2, 2, NS>, k_gemm_tn_partial_bf<2, 3, NS>, k_gemm_tn_partial_bf<2, 4, NS>},
      {k_gemm_tn_partial_bf<3, 2, NS>, k_gemm_tn_partial_bf<3, 3, NS>, k_gemm_tn_partial_bf<3, 4, NS>},
      {k_gemm_tn_partial_bf<4, 2, NS>, k_gemm_tn_partial_bf<4, 3, NS>, k_gemm_tn_partial_bf<4, 4, NS>}};
  return k[ni - 2][nj - 2];
}

// Tiles, splits and rows per split of nbatch products K x n1 x n2: as many
// workgroups as the CUs hold (cap: aimed at instead), so that all of them run
// at once; at least 128 rows a split, and at most 64 splits, whose partials
// the reduction reads one after the other.  Tiles of up to 64 x 64, or 32 x 32
// where those leave most CUs without work.  us, FP64: 13134 x 256 x 256 with
// 64 x 64 tiles 43.3 (256 workgroups; 512: 53.4), 32 x 64 46.5, 48 x 48 55.5,
// 32 x 32 57.0 (through LDS, 64 x 64 split over the wavefronts: 58.9); 7550 x
// 76 x 77 7.9, 8.7 with 32 x 48 tiles; 2944 x 48 x 64 8.2, 4.5 with 32 x 32.
// FP32, 152400 x 256 x 256: 195 with two 64 x 64 workgroups a CU, 235 with one,
// 217 with 32 x 64, 274 with 32 x 32 (through LDS: 240).
struct TnShape {
  int ni, nj, tiles, nsplit, kc;
  size_t lds;
};
template <typename T>
static TnShape tn_shape(int K, int n1, int n2, int nbatch, int cap, int max_split, int rows4 = 64) {
  TnShape s;
  const int rows = std::min(64, (K + 127) / 128);
  const int most = (long)((n1 + 63) / 64) * ((n2 + 63) / 64) * nbatch * rows >= 192 ? 4 : 2;
  s.ni = tiles16(n1, most);
  s.nj = tiles16(n2, most);
  s.lds = 4 * sizeof(T) * 256 * (size_t)s.ni * s.nj;
  s.tiles = ((n1 + 16 * s.ni - 1) / (16 * s.ni)) * ((n2 + 16 * s.nj - 1) / (16 * s.nj));
  if (cap <= 0) cap = sizeof(T) * s.ni * s.nj > 96 ? 256 : 512;
  const long all = (long)s.tiles * nbatch;
  s.nsplit = (int)std::max(1L, std::min({cap / all, (long)(K + 127) / 128, 64L, (long)max_split}));
  s.kc = ((K + s.nsplit - 1) / s.nsplit + rows4 - 1) / rows4 * rows4;  // whole chunks a wavefront
  s.nsplit = std::max(1, (K + s.kc - 1) / s.kc);
  return s;
}

// ws == null: the partials go to the context's buffer (grown on demand);
// else to ws (ws_bytes long), with fewer K splits when the usual count does
// not fit and PW_ERR_UNSUPPORTED when not even one split does.
template <typename T>
int gemm_tn_ws(pw_ctx* c, int K, int n1, int n2, const T* A, int lda, const T* B, int ldb, T* C, int ldc,
               const T* rowscale, T beta, int split, void* ws, size_t ws_bytes) {
  if (n1 <= 0 || n2 <= 0) return PW_OK;
  if (n2 == 1) {
    int nsplit = std::max(1, std::min(64, (K + 2047) / 2048));
    if (ws) nsplit = (int)std::min<size_t>(nsplit, ws_bytes / (sizeof(T) * (size_t)n1));
    if (nsplit < 1) return fail(PW_ERR_UNSUPPORTED, "projection of %d columns exceeds the %zu-byte scratch", n1, ws_bytes);
    const int kc = (K + nsplit - 1) / nsplit;
    const size_t need = sizeof(T) * (size_t)nsplit * n1;
    if (!ws) PW_TRY(grow_gemm_ws(c, need));
    T* P = (T*)(ws ? ws : c->d_gemm_ws);
    hipLaunchKernelGGL(k_gemv_t_partial<T>, dim3(n1, nsplit), dim3(256), 0, c->stream, A, lda, B, K, kc, n1, P);
    const int g = std::max(1, std::min((n1 + 255) / 256, 4096));
    hipLaunchKernelGGL(k_gemm_tn_reduce<T>, dim3(g), dim3(256), 0, c->stream, (const T*)P, nsplit, n1, 1, C, ldc,
                       rowscale, beta, (T* const*)nullptr, 0L);
    PW_HIP(hipGetLastError());
    return PW_OK;
  }
  const pw_ctx::Plan& pl = c->plan[sizeof(T) == 8 ? PW_F64 : PW_F32];
  const size_t per_split = sizeof(T) * (size_t)n1 * n2;
  if (ws && per_split > ws_bytes)
    return fail(PW_ERR_UNSUPPORTED, "a %d x %d projection exceeds the %zu-byte scratch", n1, n2, ws_bytes);
  const int max_split = ws ? (int)std::min<size_t>(ws_bytes / per_split, 1 << 20) : 1 << 20;
  const long total = (long)n1 * n2;
  const int g = (int)std::min<long>((total + 255) / 256, 4096);
  T* P = nullptr;
  int nsplit = 0;
  const TnShape s = tn_shape<T>(K, n1, n2, 1, pl.tn_cap, max_split, sizeof(T) == 4 && split >= 2 ? 128 : 64);
  nsplit = s.nsplit;
  // The buffer is sized by the shape, not by the kind of product: the native
  // product's 64-row splits are at least as many as the 128-row ones, and a
  // filter and an H X of the same bands then never move it under each other.
  if (!ws) PW_TRY(grow_gemm_ws(c, per_split * tn_shape<T>(K, n1, n2, 1, pl.tn_cap, max_split, 64).nsplit));
  P = (T*)(ws ? ws : c->d_gemm_ws);
  bool done = false;
  if constexpr (sizeof(T) == 4) {
    if (split == 2 || split == 3) {
      const auto kern = split == 3 ? tn_kernel_bf<3>(s.ni, s.nj) : tn_kernel_bf<2>(s.ni, s.nj);
      PW_TRY(ensure_lds((const void*)kern, s.lds));
      hipLaunchKernelGGL(kern, dim3(s.tiles * nsplit), dim3(256), s.lds, c->stream, A, lda, B, ldb, K, n1, n2, s.kc,
                         P);
      done = true;
    }
  }
  if (!done) {
    const auto kern = tn_kernel<T>(s.ni, s.nj);
    PW_TRY(ensure_lds((const void*)kern, s.lds));
    hipLaunchKernelGGL(kern, dim3(s.tiles * nsplit), dim3(256), s.lds, c->stream, A, lda, B, ldb, K, n1, n2, s.kc, P,
                       (const T* const*)nullptr, (const T* const*)nullptr, 0L);
  }
  hipLaunchKernelGGL(k_gemm_tn_reduce<T>, dim3(g), dim3(256), 0, c->stream, (const T*)P, nsplit, n1, n2, C, ldc,
                     rowscale, beta, (T* const*)nullptr, 0L);
  PW_HIP(hipGetLastError());
  return PW_OK;
}

template <typename T>
int gemm_tn(pw_ctx* c, int K, int n1, int n2, const T* A, int lda, const T* B, int ldb, T* C, int ldc,
            const T* rowscale, T beta, int split) {
  return gemm_tn_ws<T>(c, K, n1, n2, A, lda, B, ldb, C, ldc, rowscale, beta, split, nullptr, 0);
}

// 16 columns a wavefront where that takes fewer rounds of the chip's 1024 SIMDs
// than 32 (few rows, or the ragged end of n), else 32.  us with 16 / 32 / 48 /
// 64 columns: FP64 13134 x 256 x 256 50.6 / 47.2 / 77.2 / 55.2 (through LDS:
// 65.8), 7550 x 77 x 76 12.5 / 21.6 / 29.1 / 36.9; FP32 152400 x 256 x 256
// 269 / 235 / 235 / 239 (through LDS: 302).
template <typename T, bool kCheb>
static void launch_nn(pw_ctx* c, const T* A, int lda, const T* B, int ldb, int m, int n, int k,
                      const NnEpilogue<T>& ep) {
  const int ti = (m + 63) / 64, it1 = ti * ((n + 15) / 16), it2 = ti * ((n + 31) / 32);
  const bool one = (it1 + 1023) / 1024 < 2 * ((it2 + 1023) / 1024);
  const int items = one ? it1 : it2;
  const auto kern = one ? k_gemm_nn_ep<T, 1, kCheb> : k_gemm_nn_ep<T, 2, kCheb>;
  hipLaunchKernelGGL(kern, dim3((items + 3) / 4), dim3(256), 0, c->stream, A, lda, B, ldb, m, n, k, ep);
}

template <typename T>
int gemm_nn(pw_ctx* c, int m, int n, int k, T alpha, const T* A, int lda, const T* B, int ldb, T beta, T* Y,
            int ldy) {
  if (m <= 0 || n <= 0) return PW_OK;
  if (n == 1) {
    launch_gemv_n<T>(c, A, lda, B, Y, m, k, alpha, beta);
    PW_HIP(hipGetLastError());
    return PW_OK;
  }
  launch_nn<T, false>(c, A, lda, B, ldb, m, n, k, NnEpilogue<T>{Y, nullptr, nullptr, Y, ldy, nullptr, 0, alpha, beta});
  PW_HIP(hipGetLastError());
  return PW_OK;
}

// out (m x n) = epilogue(H, A B) for the projector apply of H Y: FP32 on
// split-BF16 MFMA (FP32 MFMA when the context's split products are off), FP64
// on FP64 MFMA; A = beta w (m x k), B = W (k x n).
template <typename T>
int gemm_nn_ep(pw_ctx* c, int m, int n, int k, const T* A, int lda, const T* B, int ldb, const T* H, const T* Yc,
               const T* Yp, T* out, int ld, const T* coef, int step, bool cheb, int split) {
  if (m <= 0 || n <= 0) return PW_OK;
  NnEpilogue<T> ep{H, Yc, Yp, out, ld, coef, step, (T)1, (T)1};
  const dim3 grid(((m + BM - 1) / BM) * ((n + BN - 1) / BN));  // nn_tile_origin's order
  bool done = false;
  if (!cheb && n == 1 && k > 0 && H == out) {
    // one column (the Lanczos vector): out += A b
    launch_gemv_n<T>(c, A, lda, B, out, m, k, (T)1, (T)1);
    done = true;
  }
  if (k <= 0) {
    const int g = (int)std::min<long>(((long)m * n + 255) / 256, 8192);
    if (cheb)
      hipLaunchKernelGGL((k_nn_epilogue_only<T, true>), dim3(g), dim3(256), 0, c->stream, (long)m, n, ep);
    else
      hipLaunchKernelGGL((k_nn_epilogue_only<T, false>), dim3(g), dim3(256), 0, c->stream, (long)m, n, ep);
    done = true;
  }
  if constexpr (sizeof(T) == 4) {
    if (!done && (split == 2 || split == 3)) {
      if (cheb && split == 3)
        hipLaunchKernelGGL((k_gemm_nn_bf<true, 3>), grid, dim3(256), 0, c->stream, A, lda, B, ldb, m, n, k, ep);
      else if (split == 3)
        hipLaunchKernelGGL((k_gemm_nn_bf<false, 3>), grid, dim3(256), 0, c->stream, A, lda, B, ldb, m, n, k, ep);
      else if (cheb)
        hipLaunchKernelGGL((k_gemm_nn_bf<true, 2>), grid, dim3(256), 0, c->stream, A, lda, B, ldb, m, n, k, ep);
      else
        hipLaunchKernelGGL((k_gemm_nn_bf<false, 2>), grid, dim3(256), 0, c->stream, A, lda, B, ldb, m, n, k, ep);
      done = true;
    }
  }
  if (!done) {
    if (cheb)
      launch_nn<T, true>(c, A, lda, B, ldb, m, n, k, ep);
    else
      launch_nn<T, false>(c, A, lda, B, ldb, m, n, k, ep);
  }
  PW_HIP(hipGetLastError());
  return PW_OK;
}

// A (m x k, column-major, ld lda) split ahead of time into the caller's
// split_a_bytes(m, k) bytes at out (the tile layout of k_gemm_nn_pre).
size_t split_a_bytes(int m, int k) {
  return sizeof(unsigned short) * (size_t)((m + 15) / 16) * ((k + 31) / 32) * kSplitTerms * 512;
}

int split_a_operand(pw_ctx* c, const float* A, int lda, int m, int k, unsigned short* out) {
  if (m <= 0 || k <= 0) return PW_OK;
  const int nrt = (m + 15) / 16, nkc = (k + 31) / 32;
  const long ng = (long)nrt * nkc;
  hipLaunchKernelGGL(k_split_operand<false>, dim3((unsigned)((ng + 3) / 4)), dim3(256), 0, c->stream, A, lda, m, k,
                     nkc, out, ng);
  PW_HIP(hipGetLastError());
  return PW_OK;
}

size_t split_b_bytes(int n, int k) {
  return sizeof(unsigned short) * (size_t)((n + 15) / 16) * ((k + 31) / 32) * kSplitTerms * 512;
}

// out (m x n) = epilogue(A B) on k_gemm_nn_pre: Ab = A split by
// split_a_operand, B (k x n, ld ldb) split here into Bws (split_b_bytes(n,
// k) bytes); NS = split terms (2 or 3).  m and ld even, H / Yc / Yp / out
// 8-byte aligned.
int gemm_nn_pre(pw_ctx* c, int m, int n, int k, const unsigned short* Ab, const float* B, int ldb,
                unsigned short* Bws, const float* H, const float* Yc, const float* Yp, float* out, int ld,
                const float* coef, int step, bool cheb, int split) {
  if (m <= 0 || n <= 0) return PW_OK;
  if ((m & 1) || (ld & 1)) return fail(PW_ERR_ARG, "gemm_nn_pre: odd row count or leading dimension");
  const int nkc = (k + 31) / 32, nct = (n + 15) / 16, nrt = (m + 15) / 16;
  const long ng = (long)nct * nkc;
  hipLaunchKernelGGL(k_split_operand<true>, dim3((unsigned)((ng + 3) / 4)), dim3(256), 0, c->stream, B, ldb, n, k,
                     nkc, Bws, ng);
  NnEpilogue<float> ep{H, Yc, Yp, out, ld, coef, step, 1.f, 1.f};
  // 16 RT rows per workgroup: RT = 2 doubles the grid of RT = 4 (206 -> 411
  // workgroups at 13134 rows x 256 columns) at fewer registers per wave, for
  // grids that would give fewer than two workgroups per CU; larger ones keep
  // RT = 4 (twice the reuse of each B fragment)
  const char* rte = std::getenv("PW_NNPRE_RT");
  int ncu = 256;
  PW_HIP(hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, c->device));
  const long g4 = (long)((nrt + 3) / 4) * ((nct + 15) / 16);
  const int rt = (rte && std::atoi(rte) == 4) ? 4 : (rte && std::atoi(rte) == 2) ? 2 : (g4 < 2L * ncu ? 2 : 4);
  const dim3 grid((nrt + rt - 1) / rt, (nct + 15) / 16);
  auto kern = rt == 4 ? (cheb ? (split == 3 ? k_gemm_nn_pre<true, 3, 4> : k_gemm_nn_pre<true, 2, 4>)
                              : (split == 3 ? k_gemm_nn_pre<false, 3, 4> : k_gemm_nn_pre<false, 2, 4>))
                      : (cheb ? (split == 3 ? k_gemm_nn_pre<true, 3, 2> : k_gemm_nn_pre<true, 2, 2>)
                              : (split == 3 ? k_gemm_nn_pre<false, 3, 2> : k_gemm_nn_pre<false, 2, 2>));
  hipLaunchKernelGGL(kern, grid, dim3(256), 0, c->stream, Ab, Bws, m, n, nkc, ep);
  PW_HIP(hipGetLastError());
  return PW_OK;
}

template int gemm_nn_ep<double>(pw_ctx*, int, int, int, const double*, int, const double*, int, const double*,
                                const double*, const double*, double*, int, const double*, int, bool, int);
template int gemm_nn_ep<float>(pw_ctx*, int, int, int, const float*, int, const float*, int, const float*,
                               const float*, const float*, float*, int, const float*, int, bool, int);
// nbatch products C_b = A_b^T B_b (n1 x n2, K rows; A_b, B_b, C_b from
// device pointer tables dA, dB, dC, one leading dimension each): one
// launch of split-K partial tiles for all products and one fixed-order
// reduction.
template <typename T>
int gemm_tn_batched(pw_ctx* c, int K, int n1, int n2, const T* const* dA, int lda, const T* const* dB, int ldb,
                    T* const* dC, int ldc, int nbatch) {
  if (n1 <= 0 || n2 <= 0 || nbatch <= 0) return PW_OK;
  const TnShape s = tn_shape<T>(K, n1, n2, nbatch, 0, 1 << 20);
  const long per = (long)n1 * n2 * s.nsplit;  // partials of one product
  PW_TRY(grow_gemm_ws(c, sizeof(T) * (size_t)per * nbatch));
  T* P = (T*)c->d_gemm_ws;
  const auto kern = tn_kernel<T>(s.ni, s.nj);
  PW_TRY(ensure_lds((const void*)kern, s.lds));
  hipLaunchKernelGGL(kern, dim3(s.tiles * s.nsplit, nbatch), dim3(256), s.lds, c->stream, (const T*)nullptr, lda,
                     (const T*)nullptr, ldb, K, n1, n2, s.kc, P, dA, dB, per);
  const long total = (long)n1 * n2;
  const int g = (int)std::max<long>(1, std::min<long>((total + 255) / 256, 4096));
  hipLaunchKernelGGL(k_gemm_tn_reduce<T>, dim3(g, nbatch), dim3(256), 0, c->stream, (const T*)P, s.nsplit, n1, n2,
                     (T*)nullptr, ldc, (const T*)nullptr, (T)0, dC, per);
  PW_HIP(hipGetLastError());
  return PW_OK;
}
template int gemm_tn_batched<double>(pw_ctx*, int, int, int, const double* const*, int, const double* const*, int,
                                     double* const*, int, int);

template int gemm_tn_ws<double>(pw_ctx*, int, int, int, const double*, int, const double*, int, double*, int,
                                const double*, double, int, void*, size_t);
template int gemm_tn_ws<float>(pw_ctx*, int, int, int, const float*, int, const float*, int, float*, int,
                               const float*, float, int, void*, size_t);
template int gemm_tn<double>(pw_ctx*, int, int, int, const double*, int, const double*, int, double*, int,
                             const double*, double, int);
template int gemm_tn<float>(pw_ctx*, int, int, int, const float*, int, const float*, int, float*, int,
                            const float*, float, int);
template int gemm_nn<double>(pw_ctx*, int, int, int, double, const double*, int, const double*, int, double,
                             double*, int);
template int gemm_nn<float>(pw_ctx*, int, int, int, float, const float*, int, const float*, int, float, float*,
                            int);

}  // namespace pw

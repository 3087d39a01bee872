// Host side of the matrix-core slab transform (pw_slab_mm.h): tables, stick
// entries and the potential in operand order per context, and the launch.
#include "pw_slab_mm.h"

#include <algorithm>
#include <cmath>
#include <cstring>
#include <vector>

#include "pw_internal.h"

namespace pw {

struct SlabMm {
  int KS = 0, TX = 0, TY = 0, XS = 0, YS = 0, half = -1, shared = 0;
  struct Grid { int blocks = 0; } grid[2], wgrid[2][2];  // resident workgroups, asked for once
  size_t off_hx = 0, off_ky = 0, off_hy = 0;
  void* buf = nullptr;                // tables and stick entries of both precisions
  const void* tab[2];                 // [PW_F64], [PW_F32]: x and y tables
  const int2* sp[2];
  void* v[2] = {nullptr, nullptr};    // V / N in operand order (one allocation, at v[PW_F64])
};

// V / N in operand order: [z][y tile][x tile][i][lane], the four classes
// W = sum over the signs of (x, y) of V(+-x, +-y) times the class's signs at
// (x, y) = (16 xt + 4 i + lane / 16, 16 yt + perm(lane % 16)); a point that is
// its own mirror counts once.  Formed in FP64 in both precisions.
template <typename T>
__global__ void k_mm_potential(const double* __restrict__ vtot, typename MmV<T>::t* __restrict__ out, int n1, int n2,
                               int TX, int TY, long total) {
  for (long e = blockIdx.x * (long)blockDim.x + threadIdx.x; e < total; e += (long)gridDim.x * blockDim.x) {
    const int lane = (int)(e & 63), i = (int)(e >> 6) & 3;
    const long q = e >> 8;
    const int xt = (int)(q % TX), yt = (int)(q / TX % TY);
    const long z = q / TX / TY;
    const int x = 16 * xt + 4 * i + lane / 16, y = 16 * yt + mm_perm<T>(lane % 16);
    typename MmV<T>::t w = {0, 0, 0, 0};
    if (x <= n1 / 2 && y <= n2 / 2) {
      const double* p = vtot + z * n1 * n2;
      const bool mx = x != 0 && 2 * x != n1, my = y != 0 && 2 * y != n2;
      const double a = p[(long)y * n1 + x];
      const double b = mx ? p[(long)y * n1 + n1 - x] : 0.0;
      const double c = my ? p[(long)(n2 - y) * n1 + x] : 0.0;
      const double d = mx && my ? p[(long)(n2 - y) * n1 + n1 - x] : 0.0;
      w[0] = (T)((a + b) + (c + d));
      w[1] = (T)((a - b) + (c - d));
      w[2] = (T)((a + b) - (c + d));
      w[3] = (T)((a - b) - (c - d));
    }
    out[e] = w;
  }
}

void mm_free(pw_ctx* c) {
  if (!c->mm) return;
  if (c->mm->buf) (void)hipFree(c->mm->buf);
  if (c->mm->v[PW_F64]) (void)hipFree(c->mm->v[PW_F64]);
  delete c->mm;
  c->mm = nullptr;
}

// one precision's tables and stick entries at host (and their device place)
template <typename T>
static void fill_plan(const pw_ctx* c, SlabMm* m, int kymax, const std::vector<int>& plus,
                      const std::vector<int>& minus, unsigned char* host, size_t tab_bytes, const unsigned char* dev) {
  typedef typename cx<T>::t C;
  const int d = sizeof(T) == 8 ? PW_F64 : PW_F32, TK = (m->KS + 3) / 4, nk = 16 * TK;
  C* end = axis_tables<T>(c->n1, c->sp.kxmax, m->KS, m->TX, (C*)host);
  if (!m->shared) axis_tables<T>(c->n2, kymax, m->KS, m->TY, end);
  int2* sp = (int2*)(host + tab_bytes);
  for (int k = 0; k < TK; k++)
    for (int s = 0; s < m->KS; s++)
      for (int l = 0; l < 64; l++) {
        const int kx = 16 * k + mm_perm<T>(l % 16), ky = 4 * s + l / 16;
        *sp++ = int2{plus[ky * nk + kx], minus[ky * nk + kx]};
      }
  m->tab[d] = dev;
  m->sp[d] = (const int2*)(dev + tab_bytes);
}

// The plan of a context, where the transform covers its sphere: at most 64
// kx and 64 ky, and one stick of each conjugate pair of the kx = 0 column.
int mm_plan(pw_ctx* c) {
  const StickPlan& st = c->sp;
  int kymax = 0;
  for (int s = 0; s < st.nstick; s++) kymax = std::max(kymax, std::abs(kgrid(st.ky[s], c->n2)));
  const int K = std::max(st.kxmax, kymax) + 1, KS = (K + 3) / 4;
  if (KS > 16) return PW_OK;
  SlabMm* m = new SlabMm();
  m->KS = KS <= 2 ? 2 : (KS == 7 ? 8 : KS);
  m->TX = (c->n1 / 2 + 16) / 16;
  m->TY = (c->n2 / 2 + 16) / 16;
  m->XS = (c->n1 / 2 + 4) / 4;
  m->YS = (c->n2 / 2 + 4) / 4;
  m->half = c->n1 % 2 == 0 ? c->n1 / 2 : -1;
  m->shared = c->n1 == c->n2 && st.kxmax == kymax;
  const int TK = (m->KS + 3) / 4, nk = 16 * TK;
  std::vector<int> plus((size_t)nk * 4 * m->KS, kMmNone), minus(plus);
  bool ok = true;
  for (int s = 0; s < st.nstick; s++) {
    const int ky = kgrid(st.ky[s], c->n2), at = std::abs(ky) * nk + st.kx[s];
    (ky >= 0 ? plus : minus)[at] = s;
  }
  for (int s = 0; s < st.nstick; s++) {
    const int ky = kgrid(st.ky[s], c->n2), at = std::abs(ky) * nk;
    if (st.kx[s] != 0 || ky == 0 || 2 * ky == c->n2) continue;
    int& other = (ky > 0 ? minus : plus)[at];
    if (other != kMmNone && !(other & kMmConj)) ok = false;
    else other = s | kMmConj;
  }
  m->off_hx = 64 * (size_t)m->KS * m->TX;
  m->off_ky = m->shared ? 0 : m->off_hx + 64 * (size_t)4 * TK * m->TX;
  m->off_hy = m->shared ? m->off_hx : m->off_ky + 64 * (size_t)m->KS * m->TY;
  if (!ok) {
    delete m;
    return PW_OK;
  }
  c->mm = m;
  const size_t entries = 64 * (size_t)(m->KS + 4 * TK) * (m->TX + (m->shared ? 0 : m->TY));
  const size_t sp_bytes = sizeof(int2) * 64 * TK * m->KS, tab64 = sizeof(double2) * entries, tab32 = tab64 / 2;
  std::vector<unsigned char> host(tab64 + tab32 + 2 * sp_bytes);
  PW_HIP(hipMalloc(&m->buf, host.size()));
  unsigned char* dev = (unsigned char*)m->buf;
  fill_plan<double>(c, m, kymax, plus, minus, host.data(), tab64, dev);
  const size_t second = tab64 + sp_bytes;
  fill_plan<float>(c, m, kymax, plus, minus, host.data() + second, tab32, dev + second);
  PW_HIP(hipMemcpy(m->buf, host.data(), host.size(), hipMemcpyHostToDevice));
  const size_t vn = 4 * 64 * 4 * (size_t)m->TX * m->TY * c->n3;
  PW_HIP(hipMalloc(&m->v[PW_F64], (sizeof(double) + sizeof(float)) * vn));
  m->v[PW_F32] = (double*)m->v[PW_F64] + vn;
  return PW_OK;
}

// After the potential has been set (on the context's stream, waited for).
int mm_potential(pw_ctx* c) {
  if (!c->mm) return PW_OK;
  SlabMm* m = c->mm;
  const long total = 256L * m->TX * m->TY * c->n3;
  const int blocks = (int)std::min<long>((total + 255) / 256, 8192);
  hipLaunchKernelGGL(k_mm_potential<double>, dim3(blocks), dim3(256), 0, c->stream, c->d_vtot,
                     (MmV<double>::t*)m->v[PW_F64], c->n1, c->n2, m->TX, m->TY, total);
  hipLaunchKernelGGL(k_mm_potential<float>, dim3(blocks), dim3(256), 0, c->stream, c->d_vtot,
                     (MmV<float>::t*)m->v[PW_F32], c->n1, c->n2, m->TX, m->TY, total);
  PW_HIP(hipGetLastError());
  PW_HIP(hipStreamSynchronize(c->stream));
  return PW_OK;
}

constexpr int kMmWaves = 4;

// waves per SIMD of an instantiation: the registers of its accumulators
template <typename T, int KS> constexpr int mm_lb() {
  return sizeof(T) == 8 ? (KS <= 4 ? 2 : 1) : (KS <= 4 ? 4 : 2);
}
template <typename T>
using mm_fn = decltype(&k_slab_mm<T, 4, kMmWaves, mm_lb<T, 4>()>);
template <typename T>
static mm_fn<T> mm_kernel(int KS) {
  switch (KS) {
    case 2: return &k_slab_mm<T, 2, kMmWaves, mm_lb<T, 2>()>;
    case 3: return &k_slab_mm<T, 3, kMmWaves, mm_lb<T, 3>()>;
    case 4: return &k_slab_mm<T, 4, kMmWaves, mm_lb<T, 4>()>;
    case 5: return &k_slab_mm<T, 5, kMmWaves, mm_lb<T, 5>()>;
    case 6: return &k_slab_mm<T, 6, kMmWaves, mm_lb<T, 6>()>;
    case 8: return &k_slab_mm<T, 8, kMmWaves, mm_lb<T, 8>()>;
    default: return nullptr;
  }
}

// The workgroup kernel beyond four k-steps: threads at most (12 wavefronts
// where 168 registers hold the tiles, else 8), bands per workgroup (the fewest
// that reach the most resident wavefronts), LDS.  nb = 0: it does not fit.
struct WgShape {
  int maxt = 0, nb = 0;
  size_t lds = 0;
};
template <typename T>
static WgShape wg_shape(const SlabMm* m) {
  WgShape w;
  const int TK = (m->KS + 3) / 4;
  if (sizeof(T) == 8 && TK > 2) return w;  // 384 registers of tiles a wavefront
  w.maxt = sizeof(T) == 4 && TK <= 3 ? 768 : 512;
  int best = 0;
  for (int nb = 1; nb * m->TY * 64 <= w.maxt; nb++) {
    const size_t lds = mm_wg_tables<T>(m->KS, m->TX) + nb * mm_wg_band<T>(m->KS, m->TY);
    if (lds > 160 * 1024) break;
    const int waves = std::min<int>((160 * 1024) / lds * nb * m->TY, w.maxt / 64 / (nb * m->TY) * nb * m->TY);
    if (waves > best) {
      best = waves;
      w.nb = nb;
      w.lds = lds;
    }
  }
  return w;
}
// Bands too few to fill the chip: one a workgroup, in more workgroups.
static bool wg_few(const pw_ctx* c, const WgShape& w, int nb) {
  return (long)c->n3 * ((nb + w.nb - 1) / w.nb) < 256;
}
template <typename T>
static WgShape wg_one(const SlabMm* m, WgShape w) {
  w.lds -= (w.nb - 1) * mm_wg_band<T>(m->KS, m->TY);
  w.nb = 1;
  return w;
}
template <typename T>
using wg_fn = decltype(&k_slab_mm_wg<T, 2, 512>);
template <typename T>
static wg_fn<T> wg_kernel(int KS) {
  if constexpr (sizeof(T) == 4) {
    switch ((KS + 3) / 4) {
      case 2: return &k_slab_mm_wg<T, 2, 768>;
      case 3: return &k_slab_mm_wg<T, 3, 768>;
      default: return &k_slab_mm_wg<T, 4, 512>;
    }
  } else {
    return &k_slab_mm_wg<T, 2, 512>;
  }
}

// The workgroup kernel rather than one wavefront per plane: always beyond eight
// k-steps (the tiles of 33 columns no longer fit a wavefront), never up to four.
// Between, us of wavefront / workgroup kernel:
//   FP32, 128 bands: 72^3 128 / 259, 96 x 96 x 24 81 / 99, 120 x 120 x 24 106 /
//   122; 8 bands 22 / 26, 31 / 18, 39 / 20: the workgroup where the planes are
//   too few to fill the chip and a plane has four y tiles to split;
//   FP64, 128 bands: 72^3 350 / 392, 96 x 54 x 24 119 / 103, 96 x 96 x 24 192 /
//   163, 120 x 120 x 24 289 / 211; 8 bands 46 / 44, 38 / 35, 60 / 31, 86 / 38:
//   the workgroup from four tiles on (the wavefront spills at one per SIMD).
template <typename T>
static bool use_wg(const pw_ctx* c, int nb) {
  const SlabMm* m = c->mm;
  if (m->KS <= 4) return false;
  if (wg_shape<T>(m).nb == 0) return false;
  if (m->KS > 8 || mm_lds<T>(m->KS, m->TX, m->TY, m->shared) > 160 * 1024) return true;
  if (sizeof(T) == 8) return std::max(m->TX, m->TY) >= 4;
  return m->TY >= 4 && (long)nb * c->n3 < 1024;
}

template <typename T>
bool mm_slab_ready(const pw_ctx* c) {
  if (!c->mm) return false;
  const SlabMm* m = c->mm;
  return (m->KS <= 8 && mm_lds<T>(m->KS, m->TX, m->TY, m->shared) <= 160 * 1024) ||
         (m->KS > 4 && wg_shape<T>(m).nb > 0);
}

int mm_ksteps(const pw_ctx* c) { return c->mm ? c->mm->KS : 0; }

// The matrix-core kernel's time in us beyond launch and stick traffic, which the
// LDS kernel has too: a wavefront's products (32 cycles each in FP32, 64 in
// FP64), the first round and the further ones of what the CUs hold at once; in
// the workgroup kernel the fourth product, two chains long, and a cost per item
// by themselves.  Planes of one or two y tiles give the workgroup kernel as few
// wavefronts a band: never the faster with one (180 x 24 FP32, 24 bands of 24
// planes, 109 us for 40 in LDS), 1.6 times the estimate in FP32 with two.
template <typename T>
double mm_slab_us(const pw_ctx* c, int nb) {
  const SlabMm* m = c->mm;
  const int KS = m->KS, TK = (KS + 3) / 4, TX = m->TX, TY = m->TY;
  const double cyc = (sizeof(T) == 8 ? 64.0 : 32.0) / 2400.0;
  auto rounds = [](double r) { return r < 8 ? std::max(1.0, std::ceil(r)) : r; };
  if (!use_wg<T>(c, nb)) {
    const double w = 4.0 * cyc * (TY * (TK * KS + TX * KS + m->XS * TK) + m->YS * TK * TK);
    const double r = rounds((double)c->n3 * ((nb + 3) / 4) / 256);
    return sizeof(T) == 4 ? w * (1.48 + 0.934 * (r - 1)) : w * (1.75 + 1.76 * (r - 1));
  }
  if (TY == 1) return 1e30;
  WgShape w = wg_shape<T>(m);
  if (wg_few(c, w, nb)) w = wg_one<T>(m, w);
  const double items = (double)c->n3 * ((nb + w.nb - 1) / w.nb);
  const int per_cu = std::max(1, std::min((int)(160 * 1024 / w.lds), w.maxt / (64 * w.nb * TY)));
  const double q = (w.nb * TY + 3) / 4, r = rounds(items / (256.0 * per_cu));
  const double p3 = 4.0 * cyc * q * (TK * KS + TX * KS + m->XS * TK);
  const double p4 = 4.0 * cyc * q * m->YS * ((TK * TK + TY - 1) / TY);
  if (sizeof(T) == 8) return p3 * (1.0 + 1.15 * (r - 1)) + 9.6 * r;
  return (TY == 2 ? 1.6 : 1.0) * (p3 * (1.31 + 1.49 * (r - 1)) + 2.51 * p4 * r + 4.4 * r);
}

template <typename T>
static MmArgs<T> mm_args(const pw_ctx* c, int nb) {
  typedef typename cx<T>::t C;
  const SlabMm* m = c->mm;
  const int d = sizeof(T) == 8 ? PW_F64 : PW_F32;
  const C* tab = (const C*)m->tab[d];
  return MmArgs<T>{tab, tab + m->off_hx, tab + m->off_ky, tab + m->off_hy, m->sp[d], (const typename MmV<T>::t*)m->v[d],
                   m->TX, m->TY, m->XS, m->YS, c->n3, c->sp.nstick, nb, m->half, m->shared};
}

template <typename T>
int mm_slab(pw_ctx* c, int nb, const void* t1, void* t2) {
  typedef typename cx<T>::t C;
  const SlabMm* m = c->mm;
  const int d = sizeof(T) == 8 ? PW_F64 : PW_F32;
  if (use_wg<T>(c, nb)) {
    const auto kwg = wg_kernel<T>(m->KS);
    WgShape w = wg_shape<T>(m);
    const bool few = wg_few(c, w, nb);
    if (few) w = wg_one<T>(m, w);
    const int threads = 64 * w.nb * m->TY;
    PW_TRY(ensure_lds((const void*)kwg, w.lds));
    SlabMm::Grid& gw = c->mm->wgrid[d][few];
    if (gw.blocks == 0) {
      int per_cu = 0, ncu = 0;
      PW_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, (const void*)kwg, threads, w.lds));
      PW_HIP(hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, c->device));
      gw.blocks = std::max(1, per_cu) * std::max(8, ncu);
    }
    const int nitem = c->n3 * ((nb + w.nb - 1) / w.nb);
    hipLaunchKernelGGL(kwg, dim3((unsigned)std::max(8, std::min(nitem, gw.blocks))), dim3(threads), w.lds, c->stream,
                       (const C*)t1, (C*)t2, mm_args<T>(c, nb), m->KS, w.nb);
    PW_HIP(hipGetLastError());
    return PW_OK;
  }
  const auto kern = mm_kernel<T>(m->KS);
  const size_t lds = mm_lds<T>(m->KS, m->TX, m->TY, m->shared);
  PW_TRY(ensure_lds((const void*)kern, lds));
  // as many workgroups as the device holds at once, at most one per item
  SlabMm::Grid& gr = c->mm->grid[d];
  if (gr.blocks == 0) {
    int per_cu = 0, ncu = 0;
    PW_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, (const void*)kern, 64 * kMmWaves, lds));
    PW_HIP(hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, c->device));
    gr.blocks = std::max(1, per_cu) * std::max(8, ncu);
  }
  const int items = c->n3 * ((nb + kMmWaves - 1) / kMmWaves);
  // (8 at least: every XCD's run of items needs a workgroup)
  hipLaunchKernelGGL(kern, dim3((unsigned)std::max(8, std::min(items, gr.blocks))), dim3(64 * kMmWaves), lds,
                     c->stream, (const C*)t1, (C*)t2, mm_args<T>(c, nb));
  PW_HIP(hipGetLastError());
  return PW_OK;
}

// Splits of the bands that give the density about four waves per SIMD.
int mm_density_splits(const pw_ctx* c, int nb) {
  if (!c->mm || c->mm->KS > 8) return 0;
  const long tiles = (long)c->n3 * c->mm->TX * c->mm->TY;
  return (int)std::max<long>(1, std::min<long>({(long)nb, 16, (4096 + tiles - 1) / tiles}));
}

template <typename T>
int mm_density(pw_ctx* c, int nb, const void* t1, const double* f, int nsplit, double* part) {
  typedef typename cx<T>::t C;
  const SlabMm* m = c->mm;
  const long units = (long)c->n3 * m->TX * m->TY * nsplit;
  const dim3 grid((unsigned)((units + kMmWaves - 1) / kMmWaves)), block(64 * kMmWaves);
#define PW_MM_DENSITY(K)                                                                                       \
  case K:                                                                                                      \
    hipLaunchKernelGGL((k_density_mm<T, K, kMmWaves>), grid, block, 0, c->stream, (const C*)t1, mm_args<T>(c, nb), f, \
                       1.0 / (double)c->N, nsplit, c->n1, c->n2, part);                                        \
    break;
  switch (m->KS) {
    PW_MM_DENSITY(2)
    PW_MM_DENSITY(3)
    PW_MM_DENSITY(4)
    PW_MM_DENSITY(5)
    PW_MM_DENSITY(6)
    PW_MM_DENSITY(8)
    default: return fail(PW_ERR_STATE, "mm_density: no kernel for %d k-steps", m->KS);
  }
#undef PW_MM_DENSITY
  PW_HIP(hipGetLastError());
  return PW_OK;
}
template int mm_density<double>(pw_ctx*, int, const void*, const double*, int, double*);
template int mm_density<float>(pw_ctx*, int, const void*, const double*, int, double*);
template bool mm_slab_ready<double>(const pw_ctx*);
template bool mm_slab_ready<float>(const pw_ctx*);
template int mm_slab<double>(pw_ctx*, int, const void*, void*);
template double mm_slab_us<double>(const pw_ctx*, int);
template double mm_slab_us<float>(const pw_ctx*, int);
template int mm_slab<float>(pw_ctx*, int, const void*, void*);

}  // namespace pw

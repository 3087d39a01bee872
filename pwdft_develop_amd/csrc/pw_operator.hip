// The operator's data on the device: local potential and projectors, from host
// arrays or formed on the device.
//
// A step of the adjoint (new potential, moved atoms) needs 4 npw nbeta values
// of projectors in four forms.  Formed and converted on one host core and
// copied form by form they cost 8 ms of a 9 ms band-energy gradient at 48^3
// with 64 projectors (128 bands; 0.49 ms now), against 12 us for the kernels
// here, which are bound by their stores (36 bytes per coefficient).
#include <algorithm>
#include <cmath>
#include <vector>

#include "pw_fft.h"
#include "pw_internal.h"

namespace pw {

// V -> V / N in both precisions (the C2R normalisation of spinor.cpp:620-621)
// (out may be v)
__global__ void k_scale_potential(const double* v, double* out, float* outf, long n, double inv) {
  for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x) {
    const double x = v[i] * inv;
    out[i] = x;
    outf[i] = (float)x;
  }
}

// betaw = beta diag(w) and the FP32 copies of both; m rows, columns by blockIdx.y
__global__ void k_projector_forms(const double* __restrict__ beta, const double* __restrict__ w, int m, int nbeta,
                                  double* __restrict__ betaw, float* __restrict__ bf, float* __restrict__ bwf) {
  for (int p = blockIdx.y; p < nbeta; p += gridDim.y) {
    const size_t at = (size_t)p * m;
    const double wp = w[p];
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < m; i += gridDim.x * blockDim.x) {
      const double b = beta[at + i], bw = b * wp;
      betaw[at + i] = bw;
      bf[at + i] = (float)b;
      bwf[at + i] = (float)bw;
    }
  }
}

// pw_gaussian_projectors on the device: sphere point i of atoms blockIdx.y,
// ..., all their projectors (one sincos for the four of s, pz, px, py).
struct GaussArgs {
  double recip[9], sigma2, c0, c1;  // c0, c1: the radial factors of l = 0, 1
  int n1, n2, n3, h1, npw, npa, natom;
};
__global__ void k_gaussian_projectors(GaussArgs a, const int* __restrict__ idx, const double* __restrict__ pos,
                                      double2* __restrict__ beta) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= a.npw) return;
  const int g = idx[i], kx = g % a.h1, ky = g / a.h1 % a.n2, kz = g / (a.h1 * a.n2);
  const int m0 = kx <= a.n1 / 2 ? kx : kx - a.n1, m1 = ky <= a.n2 / 2 ? ky : ky - a.n2,
            m2 = kz <= a.n3 / 2 ? kz : kz - a.n3;
  double G[3];
  for (int d = 0; d < 3; d++) G[d] = a.recip[d] * m0 + a.recip[3 + d] * m1 + a.recip[6 + d] * m2;
  const double gauss = exp(-(G[0] * G[0] + G[1] * G[1] + G[2] * G[2]) * a.sigma2 / 2.0);
  const double f = (i == 0 ? 1.0 : 1.4142135623730950488016887242097) * gauss;
  for (int at = blockIdx.y; at < a.natom; at += gridDim.y) {
    const double* R = pos + 3 * at;
    double s, c;
    sincos(-(G[0] * R[0] + G[1] * R[1] + G[2] * R[2]), &s, &c);
    double2* o = beta + (size_t)at * a.npa * a.npw + i;
    o[0] = make_double2(f * a.c0 * c, f * a.c0 * s);
    for (int p = 1; p < a.npa; p++) {
      const double v = f * a.c1 * (p == 1 ? G[2] : p == 2 ? G[0] : G[1]);
      o[(size_t)p * a.npw] = make_double2(v * s, -v * c);  // -i v (c + i s)
    }
  }
}

// Buffers of nbeta projectors: kept when the count stays (the captured graphs
// hold their addresses), else allocated anew.
static int projector_buffers(pw_ctx* c, int nbeta) {
  if (nbeta == c->nbeta && (nbeta == 0 || c->d_W_bf)) return PW_OK;
  invalidate_graph(c);
  void* ptrs[] = {c->d_beta, c->d_betaw, c->d_W, c->d_beta_f, c->d_betaw_f, c->d_W_f, c->d_betaw_bf, c->d_W_bf,
                  c->d_wgt};
  for (void* p : ptrs)
    if (p) (void)hipFree(p);
  c->d_beta = c->d_betaw = c->d_W = c->d_wgt = nullptr;
  c->d_beta_f = c->d_betaw_f = c->d_W_f = nullptr;
  c->d_betaw_bf = c->d_W_bf = nullptr;
  c->nbeta = nbeta;
  if (nbeta == 0) return PW_OK;
  const size_t m = 2 * (size_t)c->npw, blk = m * nbeta;
  PW_HIP(hipMalloc((void**)&c->d_beta, sizeof(double) * blk));
  PW_HIP(hipMalloc((void**)&c->d_betaw, sizeof(double) * blk));
  PW_HIP(hipMalloc((void**)&c->d_beta_f, sizeof(float) * blk));
  PW_HIP(hipMalloc((void**)&c->d_betaw_f, sizeof(float) * blk));
  PW_HIP(hipMalloc((void**)&c->d_wgt, sizeof(double) * nbeta));
  PW_HIP(hipMalloc((void**)&c->d_W, sizeof(double) * (size_t)nbeta * c->max_bands));
  PW_HIP(hipMalloc((void**)&c->d_W_f, sizeof(float) * (size_t)nbeta * c->max_bands));
  PW_HIP(hipMalloc((void**)&c->d_betaw_bf, split_a_bytes((int)m, nbeta)));
  PW_HIP(hipMalloc((void**)&c->d_W_bf, split_b_bytes(c->max_bands, nbeta)));
  return PW_OK;
}

// the other forms of the projectors in d_beta with the weights in d_wgt
static int projector_forms(pw_ctx* c) {
  const int m = 2 * c->npw;
  hipLaunchKernelGGL(k_projector_forms, dim3(std::min((m + 255) / 256, 64), std::min(c->nbeta, 32768)), dim3(256), 0,
                     c->stream, (const double*)c->d_beta, (const double*)c->d_wgt, m, c->nbeta, c->d_betaw, c->d_beta_f, c->d_betaw_f);
  PW_HIP(hipGetLastError());
  // the FP32 filter's projector apply on split BF16 products: betaw split once
  PW_TRY(split_a_operand(c, c->d_betaw_f, m, m, c->nbeta, c->d_betaw_bf));
  PW_HIP(hipStreamSynchronize(c->stream));
  return PW_OK;
}

static int potential_buffers(pw_ctx* c) {
  if (c->d_vtot) return PW_OK;
  invalidate_graph(c);
  PW_HIP(hipMalloc((void**)&c->d_vtot, sizeof(double) * c->N));
  PW_HIP(hipMalloc((void**)&c->d_vtot_f, sizeof(float) * c->N));
  return PW_OK;
}

// V (device) -> d_vtot and its other forms, waited for
static int potential_forms(pw_ctx* c, const double* v) {
  hipLaunchKernelGGL(k_scale_potential, dim3((unsigned)std::min<long>((c->N + 255) / 256, 4096)), dim3(256), 0,
                     c->stream, v, c->d_vtot, c->d_vtot_f, c->N, 1.0 / (double)c->N);
  PW_HIP(hipGetLastError());
  PW_TRY(mm_potential(c));
  PW_HIP(hipStreamSynchronize(c->stream));
  c->have_vtot = true;
  return PW_OK;
}

}  // namespace pw

using namespace pw;

extern "C" int pw_set_vtot(pw_ctx* c, const double* vtot) {
  if (!c || !vtot) return fail(PW_ERR_ARG, "pw_set_vtot: null argument");
  PW_TRY(potential_buffers(c));
  PW_HIP(hipStreamSynchronize(c->stream));  // earlier calls may still read the potential
  PW_HIP(hipMemcpy(c->d_vtot, vtot, sizeof(double) * c->N, hipMemcpyHostToDevice));
  return potential_forms(c, c->d_vtot);
}

extern "C" int pw_set_vtot_device(pw_ctx* c, const double* vtot) {
  if (!c || !vtot) return fail(PW_ERR_ARG, "pw_set_vtot_device: null argument");
  PW_TRY(potential_buffers(c));
  return potential_forms(c, vtot);
}

extern "C" int pw_set_nonlocal(pw_ctx* c, int nbeta, const double* beta, const double* w) {
  if (!c || nbeta < 0 || (nbeta > 0 && (!beta || !w))) return fail(PW_ERR_ARG, "pw_set_nonlocal: bad argument");
  PW_HIP(hipStreamSynchronize(c->stream));  // earlier calls may still read the projectors
  PW_TRY(projector_buffers(c, nbeta));
  if (nbeta == 0) return PW_OK;
  PW_HIP(hipMemcpy(c->d_beta, beta, sizeof(double) * 2 * (size_t)c->npw * nbeta, hipMemcpyHostToDevice));
  PW_HIP(hipMemcpy(c->d_wgt, w, sizeof(double) * nbeta, hipMemcpyHostToDevice));
  return projector_forms(c);
}

extern "C" int pw_set_gaussian_projectors(pw_ctx* c, int natom, const double* pos, double sigma, int lmax,
                                          const double* wgt_channel) {
  if (!c || natom < 0 || (natom > 0 && (!pos || !wgt_channel)))
    return fail(PW_ERR_ARG, "pw_set_gaussian_projectors: bad argument");
  if (lmax < 0 || lmax > 1) return fail(PW_ERR_UNSUPPORTED, "pw_set_gaussian_projectors: lmax must be 0 or 1");
  const int npa = (lmax + 1) * (lmax + 1), nbeta = natom * npa;
  PW_HIP(hipStreamSynchronize(c->stream));
  PW_TRY(projector_buffers(c, nbeta));
  if (nbeta == 0) return PW_OK;
  // weights (as pw_gaussian_projectors) and positions up in one copy: the
  // positions pass through W's buffer, which no pending call reads
  std::vector<double> w(nbeta);
  for (int a = 0; a < natom; a++)
    for (int p = 0; p < npa; p++)
      w[(size_t)a * npa + p] = wgt_channel[a * (lmax + 1) + (p == 0 ? 0 : 1)] * (4.0 * M_PI) * (4.0 * M_PI) / c->vol;
  PW_HIP(hipMemcpy(c->d_wgt, w.data(), sizeof(double) * nbeta, hipMemcpyHostToDevice));
  double* dpos = c->d_W;
  if (npa * c->max_bands < 3) PW_HIP(hipMalloc((void**)&dpos, sizeof(double) * 3 * natom));
  PW_HIP(hipMemcpy(dpos, pos, sizeof(double) * 3 * natom, hipMemcpyHostToDevice));
  GaussArgs a;
  for (int i = 0; i < 9; i++) a.recip[i] = c->recip[i];
  const double rad = std::sqrt(M_PI / 2.0);
  a.sigma2 = sigma * sigma;
  a.c0 = std::sqrt(1.0 / (4.0 * M_PI)) * rad * std::pow(sigma, 3);
  a.c1 = std::sqrt(3.0 / (4.0 * M_PI)) * rad * std::pow(sigma, 5);
  a.n1 = c->n1; a.n2 = c->n2; a.n3 = c->n3; a.h1 = c->h1; a.npw = c->npw; a.npa = npa; a.natom = natom;
  hipLaunchKernelGGL(k_gaussian_projectors, dim3((c->npw + 255) / 256, std::min(natom, 32768)), dim3(256), 0, c->stream, a,
                     (const int*)c->d_idx, (const double*)dpos, (double2*)c->d_beta);
  const hipError_t e = hipGetLastError();
  const int rc = e == hipSuccess ? projector_forms(c) : fail(PW_ERR_HIP, "projectors: %s", hipGetErrorString(e));
  if (dpos != c->d_W) (void)hipFree(dpos);
  return rc;
}

// Many independent cells of uneven grids and band counts in one call (FP32
// H*psi and the scaled Chebyshev filter around it).
//
// The reference runs one cell per MPI job and applies H one band at a time
// (Spinor::AddMultSpinorFineR2C, src/SCF/spinor.cpp:562-677; the
// NonlocalMultX GEMMs, src/EigenSolver/eigensolver.cpp:471-515).  Here a
// batch holds many cells, each a device context of its own (sphere, stick
// plan, potential, projectors, scratch).  A cell's kernels are those of the
// single-cell path; a small cell leaves most of the chip idle in each, so the
// cells are dealt to a few lanes (streams, largest cell first onto the least
// loaded lane) whose kernels overlap, and the whole of it - every step of
// every cell on forked streams - is captured into one hipGraph on the second
// call of a degree and replayed from then on.  The caller's block is copied
// in and out, so the graph does not depend on its address.
//
// 24 cells (24..72 cubed, 1900 bands), degree 8: 29.4 ms with all cells' items
// in the job queues of one persistent kernel (a union of every job's registers
// and LDS at two workgroups per CU, device-wide barriers between stages), 16.0
// ms cell after cell on the kernels used here, see kLanes for the lanes.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <numeric>
#include <string>
#include <vector>

#include "pw_fft.h"
#include "pw_internal.h"

namespace pw {

constexpr int kMaxDegree = 64;
// Lanes by default.  A process has four hardware queues; more lanes than that
// still even out the queues' loads (graph replay, degree 8, 1 / 2 / 3 / 4 / 6 /
// 8 / 12 lanes: 24 cells 15.1 / 11.2 / 9.2 / 8.7 / 8.9 / 8.4 / 8.3 ms, 6 cells
// 3.21 / 2.70 / 1.99 / 2.32 / 1.88 ms, 3 cells 1.78 / 1.36 / 1.29 ms).
constexpr int kLanes = 8;
constexpr int kMaxLanes = 16;

__global__ void k_tune_fill_b(float* __restrict__ x, long n) {
  for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x)
    x[i] = __sinf(0.7548776662f * (float)(i % 100003) + 0.1f);
}

}  // namespace pw

using namespace pw;

struct pw_batch {
  int device = 0;
  hipStream_t stream = nullptr;
  int ncell = 0;
  std::vector<pw_ctx*> ctx;
  std::vector<int> nb;
  std::vector<long> xoff;
  long xtotal = 0;
  std::vector<int> shapes;                // grid, sphere, bands, projectors per cell (the autotuner's key)
  std::vector<std::vector<int>> lane;     // cells of each lane, in order
  std::vector<hipStream_t> lstream;       // made one after the other: neighbours get different hardware queues
  std::vector<hipEvent_t> ljoin;
  hipEvent_t fork = nullptr;
  float2 *d_X = nullptr, *d_Y[3] = {nullptr, nullptr, nullptr}, *d_HY = nullptr;
  float* d_coef = nullptr;                // [cell][3 kMaxDegree]
  std::vector<float> h_coef;
  int nwg_force = 0;
  bool use_graphs = true;
  hipStream_t gstream = nullptr;
  hipEvent_t gev[2] = {nullptr, nullptr};
  hipGraphExec_t gexec = nullptr;
  long gkey = -1, gwarm = -1;
  long gepoch = 0;  // epochs() at the capture
  unsigned long long* d_stamps = nullptr;  // stage timing: [cell][5 kMaxDegree]
  int stamp_steps = 0;
};

namespace pw {

static void drop_graph(pw_batch* b) {
  if (b->gexec) (void)hipGraphExecDestroy(b->gexec);
  b->gexec = nullptr;
  b->gkey = b->gwarm = -1;
}

// Sum of the cells' epochs: another value than at the capture means that a
// buffer the graph's nodes point to has moved (a product of another shape grew
// a cell's partial sums, say), and the graph must not run again.
static long epochs(const pw_batch* b) {
  long n = 0;
  for (const pw_ctx* c : b->ctx) n += c->epoch;
  return n;
}

// Cells onto lanes: the largest first, each to the lane with the least work.
static int batch_plan(pw_batch* b) {
  drop_graph(b);
  const int n = std::max(1, std::min({b->nwg_force > 0 ? b->nwg_force : kLanes, b->ncell, kMaxLanes}));
  std::vector<double> cost(b->ncell), load(n, 0.0);
  for (int i = 0; i < b->ncell; i++) {
    const pw_ctx* c = b->ctx[i];
    cost[i] = 50.0 * 2000.0 + (double)b->nb[i] * (10.0 * (double)c->N + 8.0 * c->npw * c->nbeta);
  }
  std::vector<int> order(b->ncell);
  std::iota(order.begin(), order.end(), 0);
  std::stable_sort(order.begin(), order.end(), [&](int x, int y) { return cost[x] > cost[y]; });
  b->lane.assign(n, {});
  for (int i : order) {
    const int l = (int)(std::min_element(load.begin(), load.end()) - load.begin());
    b->lane[l].push_back(i);
    load[l] += cost[i];
  }
  while ((int)b->lstream.size() < n) {
    hipStream_t s = nullptr;
    PW_HIP(hipStreamCreateWithFlags(&s, hipStreamNonBlocking));
    b->lstream.push_back(s);
  }
  while ((int)b->ljoin.size() < n) {
    hipEvent_t e = nullptr;
    PW_HIP(hipEventCreateWithFlags(&e, hipEventDisableTiming));
    b->ljoin.push_back(e);
  }
  return PW_OK;
}

// One cell's filter steps from block X into *res (a block of d_Y), or H X.
static int cell_run(pw_batch* b, int i, const float2* X, float2* HX, int degree) {
  pw_ctx* c = b->ctx[i];
  const long o = b->xoff[i];
  if (degree == 0) return pw_apply_h(c, PW_F32, b->nb[i], X + o, HX + o);
  const float* coef = b->d_coef + (size_t)3 * kMaxDegree * i;
  const float2 *cur = X + o, *prev = nullptr;
  for (int k = 0; k < degree; k++) {
    float2* next = b->d_Y[k % 3] + o;
    PW_TRY(cheb_step_coef(c, b->nb[i], cur, b->d_HY + o, prev, next, coef, k));
    prev = cur;
    cur = next;
  }
  return PW_OK;
}

// Every cell on its lane, forked from and joined to stream s.
static int batch_body(pw_batch* b, hipStream_t s, const float2* X, float2* HX, int degree) {
  const int n = (int)b->lane.size();
  PW_HIP(hipEventRecord(b->fork, s));
  int rc = PW_OK;
  for (int l = n - 1; l >= 0; l--) {
    hipStream_t ls = b->lstream[l];
    PW_HIP(hipStreamWaitEvent(ls, b->fork, 0));
    for (int i : b->lane[l]) {
      if (rc != PW_OK) break;
      pw_ctx* c = b->ctx[i];
      c->stream = ls;
      c->stamps = b->d_stamps ? b->d_stamps + (size_t)5 * kMaxDegree * i : nullptr;
      c->stamp_calls = 0;
      rc = cell_run(b, i, X, HX, degree);
      c->stream = b->stream;
      c->stamps = nullptr;
    }
    PW_HIP(hipEventRecord(b->ljoin[l], ls));
    PW_HIP(hipStreamWaitEvent(s, b->ljoin[l], 0));
  }
  return rc;
}

static int batch_replay(pw_batch* b) {
  PW_HIP(hipEventRecord(b->gev[0], b->stream));
  PW_HIP(hipStreamWaitEvent(b->gstream, b->gev[0], 0));
  PW_HIP(hipGraphLaunch(b->gexec, b->gstream));
  PW_HIP(hipEventRecord(b->gev[1], b->gstream));
  PW_HIP(hipStreamWaitEvent(b->stream, b->gev[1], 0));
  return PW_OK;
}

// The steps on the batch's own blocks (d_X in; d_Y, or d_HY for degree 0,
// out): eagerly the first time (every scratch buffer gets its size), captured
// the second, replayed from then on.
static int batch_steps(pw_batch* b, int degree) {
  float2* HX = degree == 0 ? b->d_HY : nullptr;
  if (b->d_stamps) b->stamp_steps = std::max(degree, 1);
  if (!b->use_graphs || b->d_stamps) return batch_body(b, b->stream, b->d_X, HX, degree);
  if (b->gexec && b->gepoch != epochs(b)) drop_graph(b);
  if (b->gexec && b->gkey == degree) return batch_replay(b);
  if (b->gwarm != degree) {
    const int rc = batch_body(b, b->stream, b->d_X, HX, degree);
    b->gwarm = rc == PW_OK ? degree : -1;  // (a failed call may have left buffers unsized)
    return rc;
  }
  if (!b->gstream) PW_HIP(hipStreamCreateWithFlags(&b->gstream, hipStreamNonBlocking));
  for (auto& e : b->gev)
    if (!e) PW_HIP(hipEventCreateWithFlags(&e, hipEventDisableTiming));
  if (b->gexec) (void)hipGraphExecDestroy(b->gexec);
  b->gexec = nullptr;
  b->gkey = -1;
  hipGraph_t g = nullptr;
  int rc = PW_OK;
  if (hipStreamBeginCapture(b->gstream, hipStreamCaptureModeThreadLocal) != hipSuccess) {
    rc = fail(PW_ERR_HIP, "batch: hipStreamBeginCapture failed");
  } else {
    rc = batch_body(b, b->gstream, b->d_X, HX, degree);
    const hipError_t e = hipStreamEndCapture(b->gstream, &g);
    if (rc == PW_OK && e != hipSuccess) rc = fail(PW_ERR_HIP, "batch: hipStreamEndCapture: %s", hipGetErrorString(e));
    if (rc == PW_OK && hipGraphInstantiate(&b->gexec, g, nullptr, nullptr, 0) != hipSuccess)
      rc = fail(PW_ERR_HIP, "batch: hipGraphInstantiate failed");
  }
  if (g) (void)hipGraphDestroy(g);
  if (rc != PW_OK) {
    b->gwarm = -1;
    return rc;
  }
  b->gkey = degree;
  b->gepoch = epochs(b);
  return batch_replay(b);
}

static int batch_run(pw_batch* b, const void* X, void* out, int degree) {
  const size_t bytes = sizeof(float2) * b->xtotal;
  PW_HIP(hipMemcpyAsync(b->d_X, X, bytes, hipMemcpyDeviceToDevice, b->stream));
  PW_TRY(batch_steps(b, degree));
  const float2* res = degree == 0 ? b->d_HY : b->d_Y[(degree - 1) % 3];
  PW_HIP(hipMemcpyAsync(out, res, bytes, hipMemcpyDeviceToDevice, b->stream));
  PW_HIP(hipStreamSynchronize(b->stream));
  return PW_OK;
}

}  // namespace pw

extern "C" int pw_batch_destroy(pw_batch* b) {
  if (!b) return PW_OK;
  drop_graph(b);
  void* p[] = {b->d_X, b->d_Y[0], b->d_Y[1], b->d_Y[2], b->d_HY, b->d_coef, b->d_stamps};
  for (void* q : p)
    if (q) (void)hipFree(q);
  for (pw_ctx* c : b->ctx)
    if (c) pw_ctx_destroy(c);
  for (hipStream_t s : b->lstream) (void)hipStreamDestroy(s);
  for (hipEvent_t e : b->ljoin) (void)hipEventDestroy(e);
  if (b->fork) (void)hipEventDestroy(b->fork);
  if (b->gstream) (void)hipStreamDestroy(b->gstream);
  for (auto& e : b->gev)
    if (e) (void)hipEventDestroy(e);
  delete b;
  return PW_OK;
}

extern "C" int pw_batch_create(pw_batch** out, int ncell, const int* grid, const double* supercell, const int* npw,
                               const int* idx, const int* npad, const int* pad_src, const int* pad_dst,
                               const double* ekin, const double* teter, const double* vtot, const int* nbeta,
                               const double* beta, const double* wgt, const int* nb, void* stream) {
  if (!out || ncell < 1 || !grid || !supercell || !npw || !idx || !npad || !ekin || !teter || !vtot || !nbeta ||
      !nb)
    return fail(PW_ERR_ARG, "pw_batch_create: bad argument");
  pw_batch* b = new pw_batch();
  b->stream = (hipStream_t)stream;
  b->ncell = ncell;
  if (hipGetDevice(&b->device) != hipSuccess) {
    delete b;
    return fail(PW_ERR_HIP, "pw_batch_create: no device");
  }
  long io = 0, ip = 0, iv = 0, ib = 0, iw = 0;
  for (int i = 0; i < ncell; i++) {
    if (nb[i] < 1 || npw[i] < 1 || nbeta[i] < 0) {
      pw_batch_destroy(b);
      return fail(PW_ERR_ARG, "pw_batch_create: cell %d: nb %d, npw %d, nbeta %d out of range", i, nb[i], npw[i],
                  nbeta[i]);
    }
    pw_ctx* c = nullptr;
    int rc = pw_ctx_create(&c, grid + 3 * i, supercell + 9 * i, npw[i], idx + io, npad[i], pad_src + ip, pad_dst + ip,
                           ekin + io, teter + io, nb[i], stream);
    if (rc == PW_OK) rc = pw_set_vtot(c, vtot + iv);
    if (rc == PW_OK && nbeta[i] > 0) rc = pw_set_nonlocal(c, nbeta[i], beta + ib, wgt + iw);
    if (rc != PW_OK) {
      if (c) pw_ctx_destroy(c);
      pw_batch_destroy(b);
      return rc;
    }
    b->ctx.push_back(c);
    b->nb.push_back(nb[i]);
    b->xoff.push_back(b->xtotal);
    for (int v : {c->n1, c->n2, c->n3, c->npw, nb[i], nbeta[i]}) b->shapes.push_back(v);
    b->xtotal += (long)npw[i] * nb[i];
    io += npw[i];
    ip += npad[i];
    iv += (long)grid[3 * i] * grid[3 * i + 1] * grid[3 * i + 2];
    ib += 2L * npw[i] * nbeta[i];
    iw += nbeta[i];
  }
  float2** blocks[] = {&b->d_X, &b->d_Y[0], &b->d_Y[1], &b->d_Y[2], &b->d_HY};
  for (float2** p : blocks)
    if (hipMalloc((void**)p, sizeof(float2) * b->xtotal) != hipSuccess) {
      pw_batch_destroy(b);
      return fail(PW_ERR_NOMEM, "batch: cannot allocate the batch buffers");
    }
  int rc = PW_OK;
  if (hipMalloc((void**)&b->d_coef, sizeof(float) * 3 * kMaxDegree * ncell) != hipSuccess ||
      hipEventCreateWithFlags(&b->fork, hipEventDisableTiming) != hipSuccess)
    rc = fail(PW_ERR_HIP, "pw_batch_create: device setup failed");
  if (rc == PW_OK) rc = batch_plan(b);
  if (rc != PW_OK) {
    pw_batch_destroy(b);
    return rc;
  }
  *out = b;
  return PW_OK;
}

extern "C" int pw_batch_info(const pw_batch* b, long* xtotal, int* njobs, int* nwg, int* lds) {
  if (!b) return fail(PW_ERR_ARG, "null batch");
  if (xtotal) *xtotal = b->xtotal;
  if (njobs) *njobs = std::accumulate(b->nb.begin(), b->nb.end(), 0);
  if (nwg) *nwg = (int)b->lane.size();
  if (lds) *lds = 0;
  return PW_OK;
}

extern "C" int pw_batch_tune(pw_batch* b, int rp, int zc, int nwg) {
  if (!b || rp < 0 || zc < 0 || nwg < 0) return fail(PW_ERR_ARG, "pw_batch_tune: bad argument");
  b->nwg_force = nwg;
  return batch_plan(b);
}

// Stage timing: while enabled, calls run eagerly with a wall-clock stamp (100
// MHz) around every stage of every cell's step.
extern "C" int pw_batch_set_timing(pw_batch* b, int enable) {
  if (!b) return fail(PW_ERR_ARG, "null batch");
  if (enable && !b->d_stamps)
    PW_HIP(hipMalloc((void**)&b->d_stamps, sizeof(unsigned long long) * 5 * kMaxDegree * b->ncell));
  if (!enable && b->d_stamps) {
    PW_HIP(hipStreamSynchronize(b->stream));
    (void)hipFree(b->d_stamps);
    b->d_stamps = nullptr;
  }
  b->stamp_steps = 0;
  return PW_OK;
}

extern "C" int pw_batch_timing(pw_batch* b, double* stage_ms) {
  if (!b || !stage_ms) return fail(PW_ERR_ARG, "pw_batch_timing: bad argument");
  for (int i = 0; i < 4; i++) stage_ms[i] = 0.0;
  if (!b->d_stamps || b->stamp_steps == 0) return PW_OK;
  std::vector<unsigned long long> h((size_t)5 * kMaxDegree * b->ncell);
  PW_HIP(hipStreamSynchronize(b->stream));
  PW_HIP(hipMemcpy(h.data(), b->d_stamps, sizeof(unsigned long long) * h.size(), hipMemcpyDeviceToHost));
  for (int c = 0; c < b->ncell; c++)
    for (int k = 0; k < b->stamp_steps; k++) {
      const unsigned long long* t = &h[(size_t)5 * kMaxDegree * c + 5 * k];
      for (int i = 0; i < 4; i++) stage_ms[i] += (double)(t[i + 1] - t[i]) * 1e-5;
    }
  return PW_OK;
}

extern "C" int pw_batch_set_graphs(pw_batch* b, int enable) {
  if (!b) return fail(PW_ERR_ARG, "null batch");
  b->use_graphs = enable != 0;
  return PW_OK;
}

extern "C" int pw_batch_apply_h(pw_batch* b, const void* X, void* HX) {
  if (!b || !X || !HX || X == HX) return fail(PW_ERR_ARG, "pw_batch_apply_h: bad argument");
  return batch_run(b, X, HX, 0);
}

extern "C" int pw_batch_cheb_filter(pw_batch* b, int m, const double* bounds, void* X) {
  if (!b || !X || !bounds || m < 1 || m > kMaxDegree) return fail(PW_ERR_ARG, "pw_batch_cheb_filter: bad argument");
  b->h_coef.assign((size_t)3 * kMaxDegree * b->ncell, 0.f);
  std::vector<double> cf(3 * kMaxDegree);
  for (int i = 0; i < b->ncell; i++) {
    const double a = bounds[3 * i], bu = bounds[3 * i + 1], aL = bounds[3 * i + 2];
    if (!(bu > a) || !(aL < a)) return fail(PW_ERR_ARG, "pw_batch_cheb_filter: cell %d needs aL < a < b", i);
    cheb_coef(a, bu, aL, m, cf.data());
    for (int k = 0; k < 3 * m; k++) b->h_coef[3 * kMaxDegree * i + k] = (float)cf[k];
  }
  PW_HIP(hipMemcpyAsync(b->d_coef, b->h_coef.data(), sizeof(float) * b->h_coef.size(), hipMemcpyHostToDevice,
                        b->stream));
  return batch_run(b, X, X, m);
}

// The same filter cell by cell on each cell's own context (pw_cheb_filter,
// FP32): the one-by-one reference point of the batched launch.
extern "C" int pw_batch_cheb_filter_serial(pw_batch* b, int m, const double* bounds, void* X) {
  if (!b || !X || !bounds || m < 1 || m > kMaxDegree) return fail(PW_ERR_ARG, "pw_batch_cheb_filter_serial: bad argument");
  for (int i = 0; i < b->ncell; i++) {
    pw_ctx* c = b->ctx[i];
    PW_TRY(pw_ctx_set_stream(c, b->stream));
    PW_TRY(pw_cheb_filter(c, PW_F32, b->nb[i], m, bounds[3 * i], bounds[3 * i + 1], bounds[3 * i + 2],
                          (float2*)X + b->xoff[i]));
  }
  return PW_OK;
}

extern "C" int pw_batch_set_stream(pw_batch* b, void* stream) {
  if (!b) return fail(PW_ERR_ARG, "null batch");
  b->stream = (hipStream_t)stream;
  for (pw_ctx* c : b->ctx) PW_TRY(pw_ctx_set_stream(c, stream));
  return PW_OK;
}

// Autotuner of the batched launch (see pw_tune.cpp for the single-cell
// plans): the number of lanes, timed on the batch's own H X over every cell;
// the fastest is kept and recorded in cache_path ("<key> <lanes>") under a key
// of the device and the batch's shapes.
extern "C" int pw_batch_autotune(pw_batch* b, const char* cache_path, char* summary, int len) {
  if (!b) return fail(PW_ERR_ARG, "null batch");
  std::string key;
  {
    hipDeviceProp_t p;
    std::string dev = "dev";
    if (hipGetDeviceProperties(&p, b->device) == hipSuccess) {
      dev = p.gcnArchName;
      const size_t colon = dev.find(':');
      if (colon != std::string::npos) dev = dev.substr(0, colon);
      dev += "-" + std::to_string(p.multiProcessorCount) + "cu";
    }
    unsigned long h = 1469598103934665603UL;  // FNV-1a over the cells' shapes
    for (int v : b->shapes) h = (h ^ (unsigned long)v) * 1099511628211UL;
    char hb[32];
    snprintf(hb, sizeof(hb), "%016lx", h);
    key = dev + "|batch" + std::to_string(b->ncell) + "|" + hb + "|lanes";
  }
  if (cache_path) {
    FILE* f = fopen(cache_path, "r");
    if (f) {
      char line[512];
      int n = 0;
      while (fgets(line, sizeof(line), f)) {
        char k[400];
        int lanes;
        if (sscanf(line, "%399s %d", k, &lanes) == 2 && key == k && lanes >= 1 && lanes <= kMaxLanes) n = lanes;
      }
      fclose(f);
      if (n > 0) {
        b->nwg_force = n;
        PW_TRY(batch_plan(b));
        char s[160];
        snprintf(s, sizeof(s), "batch lanes %d (cached)", n);
        if (summary && len > 0) snprintf(summary, (size_t)len, "%s", s);
        return PW_OK;
      }
    }
  }
  float2 *X = nullptr, *HX = nullptr;
  auto done = [&](int rc) {
    if (X) (void)hipFree(X);
    if (HX) (void)hipFree(HX);
    return rc;
  };
  if (hipMalloc((void**)&X, sizeof(float2) * b->xtotal) != hipSuccess ||
      hipMalloc((void**)&HX, sizeof(float2) * b->xtotal) != hipSuccess)
    return done(fail(PW_ERR_NOMEM, "pw_batch_autotune: cannot allocate the timing blocks"));
  const long n = 2 * b->xtotal;
  hipLaunchKernelGGL(k_tune_fill_b, dim3((int)std::min<long>((n + 255) / 256, 8192)), dim3(256), 0, b->stream,
                     (float*)X, n);
  hipEvent_t e0, e1;
  if (hipEventCreate(&e0) != hipSuccess || hipEventCreate(&e1) != hipSuccess)
    return done(fail(PW_ERR_HIP, "pw_batch_autotune: event creation failed"));
  double tbest = 1e30;
  const int was = b->nwg_force;
  int bn = 0, tried = 0;
  int rc = PW_OK;
  for (int lanes : {1, 2, 3, 4, 6, 8}) {
    if (lanes > b->ncell) continue;
    b->nwg_force = lanes;
    if ((rc = batch_plan(b)) != PW_OK) break;
    float best = 1e30f;
    for (int rep = 0; rep < 5 && rc == PW_OK; rep++) {  // eager, captured, three replays
      (void)hipEventRecord(e0, b->stream);
      rc = batch_run(b, X, HX, 0);
      (void)hipEventRecord(e1, b->stream);
      if (hipEventSynchronize(e1) != hipSuccess && rc == PW_OK) rc = fail(PW_ERR_HIP, "pw_batch_autotune: event wait");
      float ms = 0.f;
      (void)hipEventElapsedTime(&ms, e0, e1);
      if (rep >= 2) best = std::min(best, ms);
    }
    if (rc != PW_OK) break;
    tried++;
    if (best < tbest) {
      tbest = best;
      bn = lanes;
    }
  }
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  b->nwg_force = rc == PW_OK ? bn : was;
  const int rp = batch_plan(b);  // (the lanes of before where timing failed)
  if (rc != PW_OK || rp != PW_OK) return done(rc != PW_OK ? rc : rp);
  if (cache_path) {
    FILE* f = fopen(cache_path, "a");
    if (f) {
      fprintf(f, "%s %d\n", key.c_str(), bn);
      fclose(f);
    }
  }
  char s[200];
  snprintf(s, sizeof(s), "batch lanes %d (%.3f ms H X over %d layouts)", bn, tbest, tried);
  if (summary && len > 0) snprintf(summary, (size_t)len, "%s", s);
  return done(PW_OK);
}

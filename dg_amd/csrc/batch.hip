// Batched ensemble: many independent 1D problems of uneven size and order,
// each advanced by the RK4 loop of RK::RK_integration (rk.cc:132-247) with
// its own CFL time step (rk.cc:250-272), the HR limiter (limiting.cc:11-27)
// and the DG right-hand side of DG_SOLVER::dg_solver (dg_solver.h:292-364).
//
// One launch per step for every problem and order: the host cuts the problems
// into segments of consecutive elements, one workgroup each, and a workgroup
// takes its segment through the whole step in its registers and LDS, window
// by window (step1d.cuh), without a word to the others.  A problem's Dt comes
// from its segments' maxima of |u|+a, which every launch leaves for the next
// one: each segment's workgroup reduces them itself, in the same order.  The
// state moves between the caller's buffer and one of the same size, the
// maxima between two slots.
//
// Measured on MI355X, 256 two-fluid problems (200-4000 elements, orders 1-3,
// HR limiter, 128 threads): the former kernel, which kept a problem's chunks
// resident for all steps and exchanged their ends through agent-scope atomics
// eight times a step, moved the state through memory at every stage (24 state
// vectors a step) and took 0.49 ms a step; see k_batch for this one.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <numeric>
#include <string>
#include <type_traits>
#include <vector>

#include "dgx_internal.h"
#include "step1d.cuh"

namespace dgx {

// A workgroup's segment: the elements [c0, c1) of problem pid, whose segments
// are the workgroups wg0 .. wg0+n-1.
struct BatchSeg {
  int pid, c0, c1, wg0, n;
};

struct BatchArgs {
  Tab1D tab[3];             // orders 1..3 (Minv per problem, below)
  const BatchSeg* seg;      // [workgroup]
  const int* order;         // [problem] 1..3
  const int* n_elem;        // [problem]
  const long* state_off;    // [problem] doubles into the packed state
  const long* elem_off;     // [problem] elements into the packed per-element arrays
  const double* J;          // [element]
  const double* ij;         // [element]
  const double* normals;    // [elem_off + problem + face]
  const double* minv;       // [problem*16 + k]: Minv of the problem's element 0 (N_s x N_s)
  const double* J0;         // [problem] Jacobian of that element
  const double* dx;         // [problem] Dx
  int bc[2];
  const double* In;
  double* Out;              // null: only the maxima
  double* T;                // [problem] accumulated time
  int* status;              // [problem] 0 ok, 1 Dt too small or NaN
  const double* part_in;    // [workgroup] maxima of |u|+a; NaN: the problem has stopped
  double* part_out;
  double cfl;               // the deck's CFL number
  int limiter, stages;      // stages 0: only the limiter, and the maxima
};

// max that keeps a NaN: a problem whose state holds a NaN gets a NaN Dt and
// stops with status 1 at once (the reference's idamax skips NaNs that are
// not first and stops only once its Dt turns NaN, rk.cc:147-148)
__device__ inline double nanmax(double a, double b) { return (b != b || b > a) ? b : a; }

__device__ inline double block_nanmax(double v, double* red) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v = nanmax(v, __shfl_xor(v, off));
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  double m = red[0];
  for (int k = 1; k < (int)(blockDim.x >> 6); ++k) m = nanmax(m, red[k]);
  __syncthreads();  // red is used again
  return m;
}

// One workgroup's segment through one launch (order P).
template <int P, int PH, int FL, int R, int LB>
__device__ __forceinline__ void batch_segment(const BatchArgs& a, const BatchSeg sg, double* lds, double* red) {
  constexpr int NU = Fields<1, PH>::NF * (P + 1);
  const int tid = threadIdx.x, nthr = blockDim.x, pid = sg.pid;
  const long so = a.state_off[pid], eo = a.elem_off[pid];
  const double* In = a.In + so;
  double* Out = a.Out ? a.Out + so : nullptr;
  // Whether the problem has stopped.  Every thread of its workgroups must come
  // to the same answer, since barriers follow: a run's first launch takes it
  // from the caller's status, which no launch of that kind writes; the steps
  // take it from the maxima alone, of which a stopped segment leaves a NaN.
  bool stopped;
  double dt = 0.0;
  if (a.stages) {
    double v = 0.0;
    for (int k = tid; k < sg.n; k += nthr) v = nanmax(v, a.part_in[sg.wg0 + k]);
    dt = a.cfl * a.dx[pid] / (2 * P + 1) / block_nanmax(v, red);  // main.cc:896-897, rk.cc:268
    stopped = !(dt >= 1e-14);
    if (tid == 0 && sg.c0 == 0) {  // the only thread that reads or writes the problem's status in a step
      if (!stopped) a.T[pid] = a.T[pid] + dt;
      else if (a.status[pid] == 0) a.status[pid] = 1;
    }
  } else {
    stopped = a.status[pid] != 0;
  }
  if (stopped) {  // the state moves on as it is
    if (Out)
      for (long k = (long)sg.c0 * NU + tid; k < (long)sg.c1 * NU; k += nthr) Out[k] = In[k];
    if (tid == 0) a.part_out[blockIdx.x] = __builtin_nan("");
    return;
  }
  Tab1D t = a.tab[P - 1];
  t.Minv = a.minv + (long)pid * 16;
  const Mesh1D m{a.n_elem[pid], {a.bc[0], a.bc[1]}, a.J + eo, a.ij + eo, a.normals + eo + pid, 1, 1, a.J0[pid]};
  const int W = window_1d(nthr, R, P), own = W - 2 * halo_1d(true);
  // windows of equal length
  const int len = sg.c1 - sg.c0, nwin = len + 2 * halo_1d(true) <= W || len == m.NE && len <= W ? 1 : (len + own - 1) / own;
  double mx = 0.0;
  for (int w = 0; w < nwin; ++w) {
    const int c0 = sg.c0 + (int)((long)len * w / nwin), c1 = sg.c0 + (int)((long)len * (w + 1) / nwin);
    if (w) __syncthreads();  // the last window's state was read
    step_window<P, PH, FL, R, row_1d(window_1d(LB, R, P))>(t, m, c0, c1, In, Out, [&](double& d) { d = dt; return true; }, a.limiter != 0, a.stages,
                              lds, W, [&](const double* u, int, int) { mx = nanmax(mx, upa<1, PH>(u)); });
  }
  mx = block_nanmax(mx, red);
  if (tid == 0) a.part_out[blockIdx.x] = mx;
}

// LB: the launch bound, WPE: the waves per SIMD the registers must allow.
// Bound by issue and latency, not by memory (two state vectors a step): 256
// two-fluid problems (540k elements, 128 threads): 0.238 ms a step against
// 0.49 ms of the kernel it replaced, 0.197 at 256 threads.
template <int PH, int FL, int R, int LB, int WPE>
__global__ __launch_bounds__(LB) __attribute__((amdgpu_waves_per_eu(WPE))) void k_batch(BatchArgs a) {
  extern __shared__ __align__(16) double lds[];
  __shared__ double red[LB / 64];
  const BatchSeg sg = a.seg[blockIdx.x];
  switch (a.order[sg.pid]) {
    case 1: batch_segment<1, PH, FL, R, LB>(a, sg, lds, red); break;
    case 2: batch_segment<2, PH, FL, R, LB>(a, sg, lds, red); break;
    default: batch_segment<3, PH, FL, R, LB>(a, sg, lds, red); break;
  }
}

__global__ void k_fill_zero_batch(double* T, int* status, int n) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k < n) {
    T[k] = 0.0;
    status[k] = 0;
  }
}

// ------------------------------------------------------------------- host
template <typename Fn>
static hipError_t dispatch_batch(const dgx_config& c, Fn&& fn) {
  using I0 = std::integral_constant<int, 0>;
  using I1 = std::integral_constant<int, 1>;
  auto by_flux = [&](auto ph) -> hipError_t { return c.flux == 0 ? fn(ph, I0{}) : fn(ph, I1{}); };
  return c.physics == 0 ? by_flux(I0{}) : by_flux(I1{});
}

// Elements per lane by workgroup size: three, and registers for two waves per
// SIMD (one where the launch has no more, kLoneWaves), up to 128 threads; two and
// three waves up to 256; one and four above.
// A segment is cut to no less than 64 elements, which at order 3 and 128
// threads takes one window of three elements a lane and two of two (all with
// registers for two waves per SIMD): 16 problems
// of up to 400 elements 66 us a step against 80, 48 of 2000 53 against 70, 256
// of 4000 239 against 244 (four and two 349, one and four 316).  256 threads 197
// (one and four 248, three and two 229), 512 threads 207 (two waves 302), 1024
// threads 230.
static int batch_R(int block) { return block <= 128 ? 3 : (block <= 256 ? 2 : 1); }
// Waves of a launch up to which workgroups of up to 128 threads take the
// instance for one wave per SIMD (262 registers, no spills; the other is held to
// 256, spills and has less room to reorder): the card has 1024 SIMDs, so no wave
// has to share one.  us a step with the two forced: 16 problems
// of up to 400 elements (34 workgroups) 58 against 66, 150 of 600 (500) 60
// against 68, 48 of 2000 (441) 40 against 52; past the line 64 of 2000 (581) 71
// against 69, 128 of 2000 (1221) 109 against 85.
constexpr int kLoneWaves = 1024;
// The launch bound of the instance that runs workgroups of `block` threads.
static int batch_LB(int block) { return block <= 128 ? 128 : (block <= 256 ? 256 : (block <= 512 ? 512 : 1024)); }

}  // namespace dgx

using namespace dgx;

struct dgx_batch {
  dgx_config cfg{};
  int n = 0;
  int bc[2] = {2, 2};
  std::vector<int> ne, order;
  std::vector<long> state_off, elem_off;
  Tab1D tab[3] = {};
  int block = 512;      // workgroup size
  int min_chunk = 64;   // elements per segment of a cut problem at least (0: no problem is cut)
  // the segments, for part_block and part_min_chunk
  int part_block = -1, part_min_chunk = -1, G = 0, nsplit = 0;
  BatchSeg* d_seg = nullptr;
  double* part = nullptr;  // [2][G] maxima of |u|+a
  std::vector<void*> part_allocs;
  int *d_ne = nullptr, *d_order = nullptr;
  long *d_state_off = nullptr, *d_elem_off = nullptr;
  double *d_J = nullptr, *d_ij = nullptr, *d_normals = nullptr, *d_minv = nullptr, *d_J0 = nullptr, *d_dx = nullptr;
  double* S = nullptr;  // the state every second step is written to
  double *tuneU = nullptr, *tuneT = nullptr;
  int* tune_status = nullptr;
  std::vector<void*> allocs;
};

namespace {

template <typename T>
bool bupload(dgx_batch* b, T** dst, const T* src, size_t n) {
  if (n == 0) n = 1;
  void* p = nullptr;
  if (!hip_ok(hipMalloc(&p, n * sizeof(T)), "hipMalloc")) return false;
  b->allocs.push_back(p);
  *dst = static_cast<T*>(p);
  if (src) return hip_ok(hipMemcpy(p, src, n * sizeof(T), hipMemcpyHostToDevice), "hipMemcpy H2D");
  return true;
}

void free_partition(dgx_batch* b) {
  for (void* p : b->part_allocs) (void)hipFree(p);
  b->part_allocs.clear();
  b->d_seg = nullptr;
  b->part = nullptr;
  b->part_block = -1;
}

void free_batch(dgx_batch* b) {
  free_partition(b);
  for (void* p : b->allocs) (void)hipFree(p);
  b->allocs.clear();
}

dgx_status bfail(int code, const std::string& msg) {
  set_error(msg);
  return code;
}

template <typename T>
bool palloc(dgx_batch* b, T** dst, const T* src, size_t n) {
  if (n == 0) n = 1;
  void* p = nullptr;
  if (!hip_ok(hipMalloc(&p, n * sizeof(T)), "hipMalloc")) return false;
  b->part_allocs.push_back(p);
  *dst = static_cast<T*>(p);
  if (src) return hip_ok(hipMemcpy(p, src, n * sizeof(T), hipMemcpyHostToDevice), "hipMemcpy H2D");
  return true;
}

// The segments for workgroups of `block` threads: a problem of more elements
// than a window owns is cut into windows' worth, but not into pieces of less
// than min_chunk elements.  The highest orders (the longest workgroups) come
// first, so that the launch ends on short ones.
bool make_partition(dgx_batch* b, int block) {
  if (b->part_block == block && b->part_min_chunk == b->min_chunk && b->d_seg) return true;
  free_partition(b);  // hipFree waits for the launches that read it
  std::vector<int> ids(b->n);
  std::iota(ids.begin(), ids.end(), 0);
  std::stable_sort(ids.begin(), ids.end(), [&](int x, int y) { return b->order[x] > b->order[y]; });
  std::vector<BatchSeg> seg;
  int nsplit = 0;
  for (int k : ids) {
    const int ne = b->ne[k], W = window_1d(block, batch_R(block), b->order[k]), own = W - 2 * halo_1d(true);
    int c = 1;
    if (b->min_chunk > 0 && ne > W) c = std::max(1, std::min((ne + own - 1) / own, ne / b->min_chunk));
    if (c > 1) ++nsplit;
    const int wg0 = (int)seg.size();
    for (int i = 0; i < c; ++i)
      seg.push_back(BatchSeg{k, (int)((long)i * ne / c), (int)((long)(i + 1) * ne / c), wg0, c});
  }
  const int G = (int)seg.size();
  const bool ok = palloc(b, &b->d_seg, seg.data(), seg.size()) && palloc<double>(b, &b->part, nullptr, (size_t)2 * G);
  if (!ok) {
    free_partition(b);
    return false;
  }
  b->G = G;
  b->nsplit = nsplit;
  b->part_block = block;
  b->part_min_chunk = b->min_chunk;
  return true;
}

// One launch over every segment: the limiter alone (stages 0) or a step.
hipError_t launch_batch(dgx_batch* b, int block, const double* In, double* Out, int parity, double cfl, int limiter,
                        int stages, double* T, int* status, hipStream_t st) {
  BatchArgs a{};
  for (int q = 0; q < 3; ++q) a.tab[q] = b->tab[q];
  a.seg = b->d_seg; a.order = b->d_order; a.n_elem = b->d_ne; a.state_off = b->d_state_off; a.elem_off = b->d_elem_off;
  a.J = b->d_J; a.ij = b->d_ij; a.normals = b->d_normals; a.minv = b->d_minv; a.J0 = b->d_J0; a.dx = b->d_dx;
  a.bc[0] = b->bc[0]; a.bc[1] = b->bc[1];
  a.In = In; a.Out = Out; a.T = T; a.status = status;
  a.part_in = b->part + (size_t)parity * b->G;
  a.part_out = b->part + (size_t)(parity ^ 1) * b->G;
  a.cfl = cfl; a.limiter = limiter; a.stages = stages;
  const int R = batch_R(block), LB = batch_LB(block), NF = 3 + b->cfg.physics;
  size_t lds = 0;
  for (int p = 1; p <= 3; ++p)
    lds = std::max(lds, sizeof(double) * lds_doubles_1d(window_1d(LB, R, p), p, NF, b->cfg.physics));
  return dispatch_batch(b->cfg, [&](auto ph, auto fl) -> hipError_t {
    constexpr int PH = decltype(ph)::value, FL = decltype(fl)::value;
    const dim3 g(b->G), t(block);
    if (LB == 128 && b->G * (block / 64) <= kLoneWaves) hipLaunchKernelGGL((k_batch<PH, FL, 3, 128, 1>), g, t, lds, st, a);
    else if (LB == 128) hipLaunchKernelGGL((k_batch<PH, FL, 3, 128, 2>), g, t, lds, st, a);
    else if (LB == 256) hipLaunchKernelGGL((k_batch<PH, FL, 2, 256, 3>), g, t, lds, st, a);
    else if (LB == 512) hipLaunchKernelGGL((k_batch<PH, FL, 1, 512, 4>), g, t, lds, st, a);
    else hipLaunchKernelGGL((k_batch<PH, FL, 1, 1024, 4>), g, t, lds, st, a);
    return hipGetLastError();
  });
}

// The initial limit (or the maxima alone), nsteps steps, and the state back in U.
bool run_batch(dgx_batch* b, int block, double* U, double cfl, int nsteps, int limiter, bool limit_initial, double* T,
               int* status, hipStream_t st) {
  if (!make_partition(b, block)) return false;
  double* cur = U;
  const bool lim0 = limiter && limit_initial;
  if (!hip_ok(launch_batch(b, block, U, lim0 ? b->S : nullptr, 1, cfl, lim0 ? limiter : 0, 0, T, status, st), "batch"))
    return false;
  if (lim0) cur = b->S;
  for (int k = 0; k < nsteps; ++k) {
    double* out = cur == U ? b->S : U;
    if (!hip_ok(launch_batch(b, block, cur, out, k & 1, cfl, limiter, 4, T, status, st), "batch")) return false;
    cur = out;
  }
  return cur == U || hip_ok(hipMemcpyAsync(U, cur, sizeof(double) * b->state_off[b->n], hipMemcpyDeviceToDevice, st),
                            "batch copy");
}

}  // namespace

extern "C" {

dgx_status dgx_batch_create(const dgx_config* cfg, int n, const int* n_elem, const int* order, double x0, double x1,
                            const int* bc, dgx_batch** out) {
  if (!cfg || !n_elem || !order || !bc || !out || n <= 0) return bfail(DGX_EINVAL, "dgx_batch_create: bad arguments");
  if (cfg->dim != 1) return bfail(DGX_EUNSUPPORTED, "dgx_batch_create: the ensemble runs 1D problems");
  if (cfg->physics < 0 || cfg->physics > 1 || cfg->flux < 0 || cfg->flux > 1)
    return bfail(DGX_EINVAL, "dgx_batch_create: unknown physics or flux");
  for (int k = 0; k < 2; ++k)
    if (bc[k] != BC_FARFIELD && bc[k] != BC_REFLECTIVE)
      return bfail(DGX_EUNSUPPORTED, "dgx_batch_create: boundary tags must be 2 (farfield) or 3 (wall)");
  dgx_batch* b = new dgx_batch;
  b->cfg = *cfg;
  b->n = n;
  b->bc[0] = bc[0];
  b->bc[1] = bc[1];
  const int NF = 2 + 1 + cfg->physics;
  std::vector<double> J, ij, nrm, minv((size_t)n * 16, 0.0), J0(n), dx(n);
  long so = 0, eo = 0;
  auto bail = [&](int code, const std::string& msg) {
    free_batch(b);
    delete b;
    return msg.empty() ? code : bfail(code, msg);
  };
  for (int k = 0; k < n; ++k) {
    if (n_elem[k] < 2 || order[k] < 1 || order[k] > 3)
      return bail(DGX_EINVAL, "dgx_batch_create: problems need >= 2 elements and order 1..3");
    MeshSpec ms;
    ms.dim = 1;
    ms.order = order[k];
    ms.nx = n_elem[k];
    ms.x0 = x0;
    ms.x1 = x1;
    ms.bc[0] = bc[0];
    ms.bc[1] = bc[1];
    ms.nfields = NF;
    Tables t;
    std::string err = build_tables(ms, t);
    if (!err.empty()) return bail(DGX_EINVAL, "dgx_batch_create: " + err);
    const int Ns = t.N_s, NE = t.N_E;
    b->ne.push_back(NE);
    b->order.push_back(order[k]);
    b->state_off.push_back(so);
    b->elem_off.push_back(eo);
    so += (long)NE * NF * Ns;
    eo += NE;
    for (int e = 0; e < NE; ++e) {
      J.push_back(t.J[e]);
      ij.push_back(t.invJac[(size_t)e * t.N_G]);
    }
    // normals in geometric face order: face j between elements j-1 and j
    std::vector<double> nk(NE + 1, 0.0);
    std::vector<char> seen(NE + 1, 0);
    for (int f = 0; f < t.M_T; ++f) {
      const int e = t.face_elem[2 * f], c = t.face_closure[2 * f];
      const int j = (c == 1) ? e + 1 : e;
      if (!(c == 0 && e == 0) && c != 1) return bail(DGX_EINVAL, "dgx_batch_create: unexpected face layout");
      nk[j] = t.normals[f];
      seen[j] = 1;
    }
    for (char v : seen)
      if (!v) return bail(DGX_EINVAL, "dgx_batch_create: unexpected face layout");
    nrm.insert(nrm.end(), nk.begin(), nk.end());
    // one inverse mass matrix per problem, scaled by J_0/J_e (affine elements)
    double mmax = 0.0;
    for (int q = 0; q < Ns * Ns; ++q) mmax = std::max(mmax, std::fabs(t.Minv[q]));
    for (int e = 1; e < NE; ++e) {
      const double r = t.J[0] / t.J[e];
      for (int q = 0; q < Ns * Ns; ++q)
        if (!(std::fabs(t.Minv[(size_t)e * Ns * Ns + q] - t.Minv[q] * r) <= 1e-13 * mmax * std::max(1.0, r)))
          return bail(DGX_EUNSUPPORTED, "dgx_batch_create: element mass matrices are not J-scaled copies");
    }
    for (int q = 0; q < Ns * Ns; ++q) minv[(size_t)k * 16 + q] = t.Minv[q];
    J0[k] = t.J[0];
    dx[k] = t.Dx;
    Tab1D& g = b->tab[order[k] - 1];
    if (!g.phi) {
      double *phi, *dphi, *phi_w, *dphi_w, *L2M, *M2L;
      const bool ok = bupload(b, &phi, t.phi.data(), t.phi.size()) && bupload(b, &dphi, t.dphi.data(), t.dphi.size()) &&
                      bupload(b, &phi_w, t.phi_w.data(), t.phi_w.size()) &&
                      bupload(b, &dphi_w, t.dphi_w.data(), t.dphi_w.size()) &&
                      bupload(b, &L2M, t.Lag2Mono.data(), t.Lag2Mono.size()) &&
                      bupload(b, &M2L, t.Mono2Lag.data(), t.Mono2Lag.size());
      if (!ok) return bail(DGX_EDEVICE, "");
      g = Tab1D{phi, dphi, phi_w, dphi_w, nullptr, L2M, M2L};
    }
  }
  b->state_off.push_back(so);
  b->elem_off.push_back(eo);
  const bool ok = bupload(b, &b->d_ne, b->ne.data(), n) && bupload(b, &b->d_order, b->order.data(), n) &&
                  bupload(b, &b->d_state_off, b->state_off.data(), n + 1) &&
                  bupload(b, &b->d_elem_off, b->elem_off.data(), n + 1) && bupload(b, &b->d_J, J.data(), J.size()) &&
                  bupload(b, &b->d_ij, ij.data(), ij.size()) && bupload(b, &b->d_normals, nrm.data(), nrm.size()) &&
                  bupload(b, &b->d_J0, J0.data(), n) && bupload(b, &b->d_dx, dx.data(), n) &&
                  bupload(b, &b->d_minv, minv.data(), minv.size()) && bupload<double>(b, &b->S, nullptr, so) &&
                  bupload<double>(b, &b->tuneU, nullptr, so) && bupload<double>(b, &b->tuneT, nullptr, n) &&
                  bupload<int>(b, &b->tune_status, nullptr, n);
  if (!ok) return bail(DGX_EDEVICE, "");
  *out = b;
  return DGX_OK;
}

void dgx_batch_free(dgx_batch* b) {
  if (!b) return;
  free_batch(b);
  delete b;
}

long dgx_batch_state_offset(const dgx_batch* b, int k) {
  if (!b || k < 0 || k > b->n) return -1;
  return b->state_off[k];
}

dgx_status dgx_batch_block_sizes(dgx_batch* b, int* sizes) {
  if (!b || !sizes) return bfail(DGX_EINVAL, "dgx_batch_block_sizes: null argument");
  if (!make_partition(b, b->block)) return DGX_EDEVICE;
  sizes[0] = b->block;
  sizes[1] = b->G;
  sizes[2] = b->nsplit;
  return DGX_OK;
}

dgx_status dgx_batch_set_min_chunk(dgx_batch* b, int min_chunk) {
  if (!b) return bfail(DGX_EINVAL, "dgx_batch_set_min_chunk: null argument");
  if (min_chunk != 0 && min_chunk < 8) return bfail(DGX_EINVAL, "dgx_batch_set_min_chunk: 0 or at least 8 elements");
  b->min_chunk = min_chunk;
  return DGX_OK;
}

dgx_status dgx_batch_set_block_sizes(dgx_batch* b, const int* sizes) {
  if (!b || !sizes) return bfail(DGX_EINVAL, "dgx_batch_set_block_sizes: null argument");
  if (sizes[0] < 64 || sizes[0] > 1024 || sizes[0] % 64)
    return bfail(DGX_EINVAL, "dgx_batch_set_block_sizes: workgroup size a multiple of 64 in [64, 1024]");
  b->block = sizes[0];
  return DGX_OK;
}

dgx_status dgx_batch_autotune(dgx_batch* b, const double* U, double cfl, int limiter, void* stream) {
  if (!b || !U) return bfail(DGX_EINVAL, "dgx_batch_autotune: null argument");
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  hipEvent_t t0, t1;
  if (!hip_ok(hipEventCreate(&t0), "hipEventCreate") || !hip_ok(hipEventCreate(&t1), "hipEventCreate"))
    return DGX_EDEVICE;
  const int sizes[5] = {64, 128, 256, 512, 1024};
  float best = 1e30f;
  int best_b = b->block;
  dgx_status r = DGX_OK;
  // per size: a warm-up run, then the fastest of two timed runs of kTuneSteps
  // steps
  constexpr int kTuneSteps = 10;
  for (int bs : sizes) {
    float tot = 1e30f;
    for (int rep = 0; rep < 3 && r == DGX_OK; ++rep) {
      // scratch copies: the caller's state and times are left untouched
      if (!hip_ok(hipMemcpyAsync(b->tuneU, U, sizeof(double) * b->state_off[b->n], hipMemcpyDeviceToDevice, st),
                  "autotune copy")) { r = DGX_EDEVICE; break; }
      hipLaunchKernelGGL(k_fill_zero_batch, dim3((b->n + 255) / 256), dim3(256), 0, st, b->tuneT, b->tune_status,
                         b->n);
      if (!make_partition(b, bs)) { r = DGX_EDEVICE; break; }
      (void)hipEventRecord(t0, st);
      if (!run_batch(b, bs, b->tuneU, cfl, kTuneSteps, limiter, false, b->tuneT, b->tune_status, st)) {
        r = DGX_EDEVICE;
        break;
      }
      (void)hipEventRecord(t1, st);
      if (!hip_ok(hipEventSynchronize(t1), "autotune sync")) { r = DGX_EDEVICE; break; }
      float ms = 0.0f;
      (void)hipEventElapsedTime(&ms, t0, t1);
      if (rep > 0) tot = std::min(tot, ms);  // the first run warms the code object and caches
    }
    if (r != DGX_OK) break;
    if (tot < best) {
      best = tot;
      best_b = bs;
    }
  }
  (void)hipEventDestroy(t0);
  (void)hipEventDestroy(t1);
  b->block = best_b;
  return r;
}

dgx_status dgx_batched_rk4(dgx_batch* b, double* U, double cfl, int nsteps, int limiter, int limit_initial, double* T,
                           int* status, void* stream) {
  if (!b || !U || !T || !status || nsteps < 0) return bfail(DGX_EINVAL, "dgx_batched_rk4: bad arguments");
  if (limiter != 0 && limiter != 1) return bfail(DGX_EUNSUPPORTED, "dgx_batched_rk4: limiter must be 0 or 1 (hrl)");
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  return run_batch(b, b->block, U, cfl, nsteps, limiter, limit_initial != 0, T, status, st) ? DGX_OK : DGX_EDEVICE;
}

}  // extern "C"

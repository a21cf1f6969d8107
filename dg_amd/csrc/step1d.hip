// 1D solver: one launch per RK4 step (step1d.cuh), with the step's Dt and the
// run's time control inside it.
//
// Each block forms the step's Dt from the per-block maxima of |u|+a that the
// previous launch left (the same values in the same order, so every block
// gets the same Dt), and block 0 writes the new time and run state.  Maxima,
// time and state are double-buffered by step parity: a launch reads one slot
// and writes the other, so no block can see a value of its own launch.
// Measured on MI355X, CFL steps with the HR limiter: 1000 single-fluid
// elements, p = 2, Rusanov: 45 us a step as ten launches (four stages, four
// limiter applications, two for Dt) with their gaps, 17 us as one; 4001
// two-fluid elements, p = 3, Roe: 71 us as fourteen launches, 24 us.  What
// bounds a step now is its chain of 20 barrier-separated phases (about 0.6 us
// each); loading the Dt operands and the window together gave 1.3 us of it, a
// wave of its own for the faces 0.5 us.
#include <algorithm>
#include <type_traits>

#include "dgx_internal.h"
#include "step1d.cuh"

namespace dgx {

struct Step1DArgs {
  Tab1D t;
  Mesh1D m;
  const double* In;
  double* Out;
  int own;  // elements per block
  int limited, stages;
  // either: this Dt ...
  const double* dt_fixed;
  // ... or Dt = cfl / max(part_in), clamped to the final time
  const double* part_in;  // [npart] maxima, then node 0's value
  int npart;
  double cfl, tf;
  const double* in;  // {Dt, T} of the previous step
  double* out;
  const int* st_in;  // {stopped, last step taken, Dt error, steps}
  int* st_out;
  double* part_out;  // [gridDim.x] maxima, then node 0's value; or null
};

// idamax's way with NaNs, as k_upa_max: see rhs.hip
__device__ inline double skip_nan(double a, double b) { return b > a ? b : a; }

__device__ inline double block_skip_nan(double v, double* red) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v = skip_nan(v, __shfl_xor(v, off));
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  double m = red[0];
  for (int k = 1; k < (int)(blockDim.x >> 6); ++k) m = skip_nan(m, red[k]);
  return m;
}

template <int P, int PH, int FL, int LANES, int R>
__global__ __launch_bounds__(256) void k_step1d(Step1DArgs a) {
  extern __shared__ __align__(16) double lds[];
  __shared__ double red[4], red_out[4];
  const int tid = threadIdx.x;
  // the step's Dt and the run's time control, the window's loads in flight
  auto get_dt = [&](double& dt) -> bool {
    const bool first = blockIdx.x == 0 && tid == 0;
    if (a.dt_fixed) {
      dt = *a.dt_fixed;
      return true;
    }
    if (!a.stages) {
      if (a.st_out && first) {  // the start of a run
        for (int k = 0; k < 4; ++k) a.st_out[k] = 0;
        a.out[0] = a.out[1] = 0.0;
      }
      return true;
    }
    const int stopped = a.st_in[0], last = a.st_in[1], err = a.st_in[2], steps = a.st_in[3];
    const double dt_prev = a.in[0], T = a.in[1], n0 = a.part_in[a.npart];
    double v = 0.0;
    for (int k = tid; k < a.npart; k += blockDim.x) v = skip_nan(v, a.part_in[k]);
    const double mx = block_skip_nan(v, red);
    dt = a.cfl / (n0 != n0 ? n0 : mx);
    const bool done = stopped || last;
    const bool bad = !done && (dt < 1e-14 || dt != dt);  // rk.cc:147-148
    const bool clamp = dt > (a.tf - T);                  // rk.cc:149
    if (clamp) dt = a.tf - T;
    const bool go = !done && !bad;
    if (first) {
      a.st_out[0] = go ? 0 : 1;
      a.st_out[1] = done ? last : (go && clamp ? 1 : 0);
      a.st_out[2] = bad ? 1 : err;
      a.st_out[3] = steps + (go ? 1 : 0);
      a.out[0] = go ? dt : dt_prev;
      a.out[1] = go ? T + dt : T;
    }
    return go;
  };
  const int c0 = blockIdx.x * a.own, c1 = min(a.m.NE, c0 + a.own);
  double v = 0.0;
  const bool taken = step_window<P, PH, FL, R, row_1d(window_1d(LANES, R, P))>(
      a.t, a.m, c0, c1, a.In, a.Out, get_dt, a.limited != 0, a.stages, lds, window_1d(LANES, R, P),
      [&](const double* u, int e, int q) {
        if (!a.part_out) return;
        const double s = upa<1, PH>(u);
        if (e == 0 && q == 0) a.part_out[gridDim.x] = s;
        v = skip_nan(v, s);
      });
  if (taken && a.part_out) {  // the same for every thread; a step that was left out leaves no maxima
    const double mx = block_skip_nan(v, red_out);
    if (tid == 0) a.part_out[blockIdx.x] = mx;
  }
}

// part_in's n maxima and node 0's value into out[0], out[1], where there are
// so many that every block of a step reading them all would cost more than
// this launch
__global__ __launch_bounds__(256) void k_part_max(const double* __restrict__ part, int n, double* __restrict__ out) {
  __shared__ double red[4];
  double v = 0.0;
  for (int k = threadIdx.x; k < n; k += 256) v = skip_nan(v, part[k]);
  const double m = block_skip_nan(v, red);
  if (threadIdx.x == 0) {
    out[0] = m;
    out[1] = part[n];
  }
}

// ------------------------------------------------------------------- host
template <typename Fn>
static hipError_t dispatch_1d(const dgx_config& c, Fn&& fn) {
  using I0 = std::integral_constant<int, 0>;
  using I1 = std::integral_constant<int, 1>;
  using I2 = std::integral_constant<int, 2>;
  using I3 = std::integral_constant<int, 3>;
  auto by_flux = [&](auto p, auto ph) -> hipError_t { return c.flux == 0 ? fn(p, ph, I0{}) : fn(p, ph, I1{}); };
  auto by_phys = [&](auto p) -> hipError_t {
    switch (c.physics) {
      case 0: return by_flux(p, I0{});
      case 1: return by_flux(p, I1{});
      case 2: return by_flux(p, I2{});
      default: return by_flux(p, I3{});
    }
  };
  switch (c.order) {
    case 1: return by_phys(I1{});
    case 2: return by_phys(I2{});
    default: return by_phys(I3{});
  }
}

// Launch shape: two waves of nodes and one for the faces while that gives at
// most two blocks per CU (the chip is idle: the fewer waves a block has to
// bring together, the shorter a step), then four waves, then four with two
// elements per lane (a wider window computes its halo less often: 112 of 128
// elements owned at p = 3 against 48 of 64 and 16 of 32).  Two-fluid, us a
// step with the three shapes forced: 4001 elements p = 2 20, 23 and 31;
// 16000 elements p = 3 29, 28 and 32; 100000 elements p = 3 141, 104 and 74.
Step1DShape step1d_shape(int P, int NE, bool limited) {
  const int H = halo_1d(limited);
  Step1DShape s{};
  auto fit = [&](int lanes, int threads, int R) {
    const int cap = window_1d(lanes, R, P) - 2 * H;
    s.lanes = lanes;
    s.threads = threads;
    s.R = R;
    s.blocks = (NE + cap - 1) / cap;
    s.own = (NE + s.blocks - 1) / s.blocks;
    s.blocks = (NE + s.own - 1) / s.own;
  };
  fit(128, 192, 1);
  if (s.blocks > 512) fit(256, 256, 1);
  if (s.blocks > 1536) fit(256, 256, 2);
  return s;
}

// Blocks up to which every block of a step reads all the maxima itself (16 KB
// from the L2 at most); beyond, k_part_max does first.
constexpr int kSelfReduced = 2048;

hipError_t launch_step1d(const Solver& s, const Step1DRun& r, hipStream_t st) {
  const Step1DShape sh = step1d_shape(s.P, s.N_E, r.limited);
  Step1DArgs a{};
  a.t = Tab1D{s.t.phi, s.t.dphi, s.t.phi_w, s.t.dphi_w, s.t.Minv, s.t.Lag2Mono, s.t.Mono2Lag};
  a.m = Mesh1D{s.N_E, {s.cart.bc[0], s.cart.bc[1]}, s.t.J, s.t.invJac, s.t.face_geo_x, s.t.geo_stride, 4, s.t.J0};
  a.In = r.In; a.Out = r.Out;
  a.own = sh.own;
  a.limited = r.limited ? 1 : 0;
  a.stages = r.stages;
  a.dt_fixed = r.dt_fixed;
  a.part_in = r.part_in; a.npart = r.npart;
  if (r.part_in && r.npart > kSelfReduced) {
    double* red = s.part1d + 2 * (size_t)s.part1d_len;
    hipLaunchKernelGGL(k_part_max, dim3(1), dim3(256), 0, st, r.part_in, r.npart, red);
    a.part_in = red;
    a.npart = 1;
  }
  a.cfl = r.cfl; a.tf = r.tf;
  a.in = r.in; a.out = r.out; a.st_in = r.st_in; a.st_out = r.st_out; a.part_out = r.part_out;
  return dispatch_1d(s.cfg, [&](auto p, auto ph, auto fl) -> hipError_t {
    constexpr int P = decltype(p)::value, PH = decltype(ph)::value, FL = decltype(fl)::value;
    auto go = [&](auto lanes, auto R) {
      constexpr int L = decltype(lanes)::value, RR = decltype(R)::value;
      constexpr size_t lds =
          sizeof(double) * lds_doubles_1d(window_1d(L, RR, P), P, Fields<1, PH>::NF, Fields<1, PH>::NNC);
      hipLaunchKernelGGL((k_step1d<P, PH, FL, L, RR>), dim3(sh.blocks), dim3(sh.threads), lds, st, a);
    };
    using One = std::integral_constant<int, 1>;
    using L256 = std::integral_constant<int, 256>;
    if (sh.lanes == 128) go(std::integral_constant<int, 128>{}, One{});
    else if (sh.R == 1) go(L256{}, One{});
    else go(L256{}, std::integral_constant<int, 2>{});
    return hipGetLastError();
  });
}

}  // namespace dgx

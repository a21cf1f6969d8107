// A whole RK4 step of 1D elements in one workgroup (RK::RK_integration,
// rk.cc:132-247, with DG_SOLVER::dg_solver, dg_solver.h:292-364, and the HR
// limiter, limiting.cc:11-27), shared by the 1D solver (step1d.hip) and the
// ensemble (batch.hip).
//
// A 1D step is short of work, not of bandwidth: run as one launch per stage,
// limiter application and Dt reduction it was ten dependent launches of 2.5-5
// us each (1000 elements, p = 2: 39 us a step), and run with the chunks of a
// problem exchanging their ends inside one launch it waited for neighbours
// eight times a step.  Here a workgroup owns a run of consecutive elements
// and loads a halo wide enough for the whole step: a stage reads one element
// further on each side (its faces), a limiter application one more, so four
// limited stages need 8 elements on each side and four plain ones 4.  The
// halo elements are computed again by both neighbours, the same arithmetic
// on the same values, and nothing is exchanged within a step.  The trade pays
// from the smallest problem, where the chip is idle anyway, to ensembles that
// fill it (a window of 128 elements owns 112); the kernels that use it state
// what they measured.
//
// A lane owns one node (and Gauss point: there are as many) of R elements:
// U^n, the RK accumulator and the stage state stay in its registers for the
// whole step.  LDS only carries what lanes exchange, two buffers of N_F*N_s
// rows (row = field and node or point, the window's elements along it, so
// that every access of a wave is to consecutive words) whose roles swap from
// phase to phase, and one of face fluxes.
#pragma once
#include "hr.cuh"
#include "physics.cuh"
#include "volume.cuh"

namespace dgx {

// reference-element tables of one order, in device memory
struct Tab1D {
  const double* __restrict__ phi;
  const double* __restrict__ dphi;
  const double* __restrict__ phi_w;
  const double* __restrict__ dphi_w;
  const double* __restrict__ Minv;  // of the element with Jacobian J0, N_s x N_s
  const double* __restrict__ L2M;   // Lag2Mono, column-major N_s x N_s
  const double* __restrict__ M2L;   // Mono2Lag
};

// the mesh of one problem
struct Mesh1D {
  int NE;
  int bc[2];
  const double* __restrict__ J;
  const double* __restrict__ ij;
  const double* __restrict__ nrm;  // [face * nrm_stride], face j between elements j-1 and j
  int geo_stride, nrm_stride;
  double J0;
};

constexpr int halo_1d(bool limited) { return limited ? 8 : 4; }

// Window capacity (elements) of `lanes` node lanes with R elements each at
// order p.
__host__ __device__ constexpr int window_1d(int lanes, int R, int p) { return R * (lanes / (p + 1)); }
// Row length of a window's LDS buffers, by the most elements it may have (a
// constant of the kernel: the row offsets then fold into the LDS
// instructions): room for the faces, and odd so that the transposing load
// spreads over the banks.
__host__ __device__ constexpr int row_1d(int window) { return (window + 1) | 1; }
__host__ __device__ constexpr int lds_doubles_1d(int window, int p, int nf, int nnc) {
  return 6 * (p + 1) * (p + 1) + row_1d(window) * (2 * nf * (p + 1) + nf + nnc);
}
// The tables in LDS, [table][q * N_s + l]: a lane reads its row q of one table
// in one phase of a stage (in registers for the whole step they cost 48 of
// them at p = 3, a third wave per SIMD).
enum { T_L2M, T_PHI, T_DPHI, T_DW, T_PW, T_MINV };

// The HR limiter of a window: nodal values in A (rows f*Ns + node) become
// limited ones, through their Taylor coefficients in B.  Column (field,
// element) by lane: the lane of node q takes fields q, q + Ns, ...
// (hrl1D, limiting_kernels.cu:245-319; the order of k_apply and k_hr_sweep,
// without contraction: the same bits).
template <int P, int PH, int R, int LS>
__device__ __forceinline__ void window_limit(const Tab1D& t, const Mesh1D& m, int w0, int n, double* A, double* B,
                                             const double* sT, int q, const int (&e)[R]) {
#pragma clang fp contract(off)
  constexpr int NF = Fields<1, PH>::NF, Ns = P + 1;
  int ec[R];
#pragma unroll
  for (int r = 0; r < R; ++r) ec[r] = e[r] < n ? e[r] : n - 1;  // lanes without an element compute along
  {
    double l2m[Ns];
#pragma unroll
    for (int l = 0; l < Ns; ++l) l2m[l] = sT[(T_L2M * Ns + q) * Ns + l];
#pragma unroll
    for (int r = 0; r < R; ++r) {
      double y[NF];
#pragma unroll
      for (int f = 0; f < NF; ++f) {
        y[f] = 0.0;
#pragma unroll
        for (int l = 0; l < Ns; ++l) y[f] = y[f] + A[(f * Ns + l) * LS + ec[r]] * l2m[l];
      }
      if (e[r] < n)
#pragma unroll
        for (int f = 0; f < NF; ++f) B[(f * Ns + q) * LS + e[r]] = y[f];
    }
  }
  __syncthreads();
  const bool periodic = m.bc[0] == BC_PERIODIC;
#pragma unroll
  for (int f0 = 0; f0 < NF; f0 += Ns) {
    const int f = f0 + q;
    if (f >= NF) break;
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int ee = ec[r];
      int physical = 0;
      if (!periodic && w0 + ee == 0) physical = m.bc[0];
      if (!periodic && w0 + ee == m.NE - 1) physical = m.bc[1];
      const int el = ee > 0 ? ee - 1 : 0, er = ee < n - 1 ? ee + 1 : ee;  // beyond the window: not used by its valid part
      double al[Ns], ac[Ns], ar[Ns], lim[Ns], out[Ns];
#pragma unroll
      for (int k = 0; k < Ns; ++k) {
        al[k] = B[(f * Ns + k) * LS + el];
        ac[k] = B[(f * Ns + k) * LS + ee];
        ar[k] = B[(f * Ns + k) * LS + er];
        lim[k] = 0.0;
      }
      limit_monomial_d<P>(al, ac, ar, lim);
      if (physical != 0) {
        if (physical == BC_FARFIELD || (physical == BC_REFLECTIVE && f != 1)) {
          average_monomial_d<P>(ac, lim);
        } else {  // the wall-normal momentum, and every field of other boundaries, stays
#pragma unroll
          for (int k = 0; k < Ns; ++k) lim[k] = ac[k];
        }
      }
#pragma unroll
      for (int k = 0; k < Ns; ++k) out[k] = 0.0;
#pragma unroll
      for (int l = 0; l < Ns; ++l)
#pragma unroll
        for (int k = 0; k < Ns; ++k) out[k] = out[k] + lim[l] * t.M2L[k + l * Ns];
      if (e[r] < n)
#pragma unroll
        for (int k = 0; k < Ns; ++k) A[(f * Ns + k) * LS + ee] = out[k];
    }
  }
  __syncthreads();
}

// One RK4 step (stages == 4) or only a limiter application (stages == 0) of
// the owned elements [c0, c1), In -> Out (element-major states of the whole
// problem; In != Out; a null Out: only umax).  The window, [c0, c1) and its
// halo, may not exceed W elements, a multiple of R; the halo is cut at the ends
// of a problem that is not periodic.  get_dt(dt) is called once by every thread,
// the window's loads in flight, and gives the step's Dt (it may synchronise the
// block); when it returns false the step is left out and step_window returns
// false.  umax(u, e, q) is called with the fields of every owned node of the new
// state.  Every thread of the block
// calls it (a multiple of 64 threads, W/R*N_s of them with nodes); LS =
// row_1d of W or more, lds holds 6*N_s*N_s + LS*(2*N_F*N_s + N_F + NNC)
// doubles.
template <int P, int PH, int FL, int R, int LS, typename GetDt, typename UMax>
__device__ __forceinline__ bool step_window(const Tab1D& t, const Mesh1D& m, int c0, int c1, const double* In,
                                            double* Out, GetDt&& get_dt, bool limited, int stages, double* lds,
                                            int W, UMax&& umax) {
  using V = Vol<1, P, PH>;
  constexpr int NF = V::NF, Ns = V::Ns, NG = V::NG, NU = V::NU, NFX = V::NFX, NNC = V::NNC;
  static_assert(NG == Ns && V::NQ == NF, "a lane is a node and a Gauss point");
  const int tid = threadIdx.x, nthr = blockDim.x;
  double* sT = lds;
  double* X = lds + 6 * Ns * Ns;
  double* Y = X + NU * LS;
  double* FF = Y + NU * LS;  // per face: F, then the non-conservative terms of the last NNC fields
  const bool periodic = m.bc[0] == BC_PERIODIC;
  const int H = stages ? halo_1d(limited) : 1;
  const int w0 = periodic ? c0 - H : max(0, c0 - H), w1 = periodic ? c1 + H : min(m.NE, c1 + H), n = w1 - w0;
  auto gel = [&](int e) {  // the element at window place e
    int g = w0 + e;
    if (periodic) {
      g %= m.NE;
      if (g < 0) g += m.NE;
    }
    return g;
  };
  // lane: node q of the elements e0 + r*WR; lanes left over hold none
  const int WR = W / R;
  int q = tid / WR, e[R];
#pragma unroll
  for (int r = 0; r < R; ++r) e[r] = q < Ns ? tid - q * WR + r * WR : n;
  if (q >= Ns) q = 0;
  int ec[R];
#pragma unroll
  for (int r = 0; r < R; ++r) ec[r] = e[r] < n ? e[r] : n - 1;  // lanes without an element compute along
  // consecutive loads of the window's states, the lane's geometry and its row
  // of each table, all in flight before the first is used
  constexpr int KL = NF * R;  // W * NU <= R * nthr * NF: one round
  const int total = n * NU;
  double v[KL];
#pragma unroll
  for (int k = 0; k < KL; ++k) {
    const int i = tid + k * nthr;
    v[k] = 0.0;
    if (i < total) v[k] = In[(long)gel(i / NU) * NU + i % NU];
  }
  double Je[R], ije[R];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int g = (e[r] < n ? gel(e[r]) : 0) * m.geo_stride;
    Je[r] = stages ? m.J[g] : 1.0;
    ije[r] = stages ? m.ij[g] : 1.0;
  }
  for (int k = tid; k < 6 * Ns * Ns; k += nthr) {
    const int tab = k / (Ns * Ns), row = k % (Ns * Ns) / Ns, l = k % Ns;
    double x = 0.0;
    if (tab == T_L2M) x = t.L2M[row + l * Ns];
    if (tab == T_PHI) x = t.phi[row + l * NG];
    if (tab == T_DW) x = t.dphi_w[l + row * NG];  // at Gauss point l, test function `row`
    if (tab == T_MINV) x = t.Minv[l * Ns + row];
    if (NNC > 0 && tab == T_DPHI) x = t.dphi[row + l * NG];
    if (NNC > 0 && tab == T_PW) x = t.phi_w[l + row * NG];
    sT[k] = x;
  }
  double dt = 0.0;
  if (!get_dt(dt)) return false;
#pragma unroll
  for (int k = 0; k < KL; ++k) {
    const int i = tid + k * nthr;
    if (i < total) X[(i % NU) * LS + i / NU] = v[k];
  }
  double* A = X;  // nodal values of the present state
  double* B = Y;
  if (stages) {
    double dte[R], un[R][NF], acc[R][NF], s[R][NF];
#pragma unroll
    for (int r = 0; r < R; ++r) dte[r] = dt * (m.J0 / Je[r]);
    // faces: one lane each, from wave fw0 on: the waves without nodes where
    // there are any, else other waves (of a four-wave block: another SIMD)
    // from block to block
    const int nw = nthr >> 6, nodew = (WR * Ns + 63) >> 6;
    const int shift = 64 * (nodew < nw ? nodew : (int)(blockIdx.x % nw));
    const int j0 = !periodic && w0 == 0 ? 0 : 1, j1 = !periodic && w1 == m.NE ? n : n - 1;
    const int fl0 = tid >= shift ? tid - shift : tid + nthr - shift;
    __syncthreads();
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
      for (int f = 0; f < NF; ++f) {
        un[r][f] = A[(f * Ns + q) * LS + ec[r]];
        acc[r][f] = s[r][f] = 0.0;
      }
#pragma unroll 1
    for (int k = 0; k < 4; ++k) {
      if (k > 0) {
#pragma unroll
        for (int r = 0; r < R; ++r)
          if (e[r] < n)
#pragma unroll
            for (int f = 0; f < NF; ++f) A[(f * Ns + q) * LS + e[r]] = s[r][f];
        __syncthreads();
        if (limited) window_limit<P, PH, R, LS>(t, m, w0, n, A, B, sT, q, e);
      }
      // ---- faces (the window's outermost ones only at the domain's ends)
      for (int j = j0 + fl0; j <= j1; j += nthr) {
        const bool lb = j == 0, rb = j == n;
        double ul[NF], ur[NF], F[NF], nc[NF];
#pragma unroll
        for (int f = 0; f < NF; ++f) {
          ul[f] = lb ? A[(f * Ns) * LS] : A[(f * Ns + 1) * LS + j - 1];
          ur[f] = rb ? A[(f * Ns + 1) * LS + j - 1] : A[(f * Ns) * LS + j];
        }
        if ((lb && m.bc[0] == BC_REFLECTIVE) || (rb && m.bc[1] == BC_REFLECTIVE)) ur[1] = -ur[1];  // boundaries.cu:20-35
        int g = w0 + j;
        if (periodic) {  // the wrap face is the last one
          g %= m.NE;
          if (g <= 0) g += m.NE;
        }
        riemann<1, PH, FL>(ul, ur, m.nrm[(long)g * m.nrm_stride], 0.0, F, nc);
#pragma unroll
        for (int f = 0; f < NF; ++f) FF[f * LS + j] = F[f];
#pragma unroll
        for (int c = 0; c < NNC; ++c) FF[(NF + c) * LS + j] = nc[NF - NNC + c];
      }
      // ---- fluxes and sources at the Gauss points (vol_phase1's arithmetic)
      {
        double phi[Ns], dphi[Ns];
#pragma unroll
        for (int i = 0; i < Ns; ++i) {
          phi[i] = sT[(T_PHI * Ns + q) * Ns + i];
          if (NNC > 0) dphi[i] = sT[(T_DPHI * Ns + q) * Ns + i];
        }
#pragma unroll
        for (int r = 0; r < R; ++r) {
          double ug[NF], dua[NNC ? NNC : 1], fx[NF], snc[NNC ? NNC : 1], fe[NF];
#pragma unroll
          for (int f = 0; f < NF; ++f) {
            double a = 0.0, d = 0.0;
#pragma unroll
            for (int i = 0; i < Ns; ++i) {
              const double u = A[(f * Ns + i) * LS + ec[r]];
              a += u * phi[i];
              if (f >= NFX) d += u * dphi[i];
            }
            ug[f] = a;
            if (f >= NFX) dua[f - NFX] = d;
          }
          volume_flux<1, PH>(ug, dua, &ije[r], fx, snc);
#pragma unroll
          for (int f = 0; f < NFX; ++f) {
            double sol = 0.0;
            sol += ije[r] * fx[f] * Je[r];
            fe[f] = sol;
          }
#pragma unroll
          for (int c = 0; c < NNC; ++c) fe[NFX + c] = snc[c] * Je[r];
          if (e[r] < n)
#pragma unroll
            for (int f = 0; f < NF; ++f) B[(f * Ns + q) * LS + e[r]] = fe[f];
        }
      }
      __syncthreads();
      // ---- integration against the test functions and the face terms
      // (vol_phase2's order); the state in A is spent
      {
        double dw[NG], pw[NG];
#pragma unroll
        for (int g = 0; g < NG; ++g) {
          dw[g] = sT[(T_DW * Ns + q) * Ns + g];
          if (NNC > 0) pw[g] = sT[(T_PW * Ns + q) * Ns + g];
        }
#pragma unroll
        for (int r = 0; r < R; ++r) {
          double a[NF];
#pragma unroll
          for (int f = 0; f < NF; ++f) a[f] = 0.0;
#pragma unroll
          for (int g = 0; g < NG; ++g) {
#pragma unroll
            for (int f = 0; f < NFX; ++f) a[f] += dw[g] * B[(f * Ns + g) * LS + ec[r]];
#pragma unroll
            for (int c = 0; c < NNC; ++c) a[NFX + c] += pw[g] * B[((NFX + c) * Ns + g) * LS + ec[r]];
          }
          // node 0 takes face e as its right side (its left one at the left
          // domain end, where the element is side 0), node 1 face e+1 as left
          if (q < 2) {
            const int j = ec[r] + q;
            const double sgn = (q == 0 && (periodic || w0 + ec[r] != 0)) ? 1.0 : -1.0;
#pragma unroll
            for (int f = 0; f < NF; ++f) {
              const double nc = f >= NFX ? FF[(NF + f - NFX) * LS + j] : 0.0;
              a[f] += __builtin_fma(sgn, FF[f * LS + j], nc);
            }
          }
          if (e[r] < n)
#pragma unroll
            for (int f = 0; f < NF; ++f) A[(f * Ns + q) * LS + e[r]] = a[f];
        }
      }
      __syncthreads();
      // ---- Dt * Minv and the RK4 combination
      {
        double mi[Ns];
#pragma unroll
        for (int ii = 0; ii < Ns; ++ii) mi[ii] = sT[(T_MINV * Ns + q) * Ns + ii];
#pragma unroll
        for (int r = 0; r < R; ++r)
#pragma unroll
          for (int f = 0; f < NF; ++f) {
            double sol = 0.0, an;
#pragma unroll
            for (int ii = 0; ii < Ns; ++ii) sol += mi[ii] * A[(f * Ns + ii) * LS + ec[r]];
            rk_values(k, dte[r] * sol, un[r][f], acc[r][f], an, s[r][f]);
            acc[r][f] = an;
          }
      }
      // the next state goes where the fluxes were (read before the last barrier)
      double* sw = A;
      A = B;
      B = sw;
    }
#pragma unroll
    for (int r = 0; r < R; ++r)
      if (e[r] < n)
#pragma unroll
        for (int f = 0; f < NF; ++f) A[(f * Ns + q) * LS + e[r]] = s[r][f];
  }
  __syncthreads();
  if (limited) window_limit<P, PH, R, LS>(t, m, w0, n, A, B, sT, q, e);
  // ---- the owned elements: consecutive stores, and |u|+a of every node
  const int o0 = c0 - w0;
  if (Out) {
    const int total = (c1 - c0) * NU;
    for (int i = tid; i < total; i += nthr) Out[(long)c0 * NU + i] = A[(i % NU) * LS + o0 + i / NU];
  }
#pragma unroll
  for (int r = 0; r < R; ++r)
    if (e[r] >= o0 && e[r] < c1 - w0) {
      double u[NF];
#pragma unroll
      for (int f = 0; f < NF; ++f) u[f] = A[(f * Ns + q) * LS + e[r]];
      umax(u, w0 + e[r], q);
    }
  return true;
}

}  // namespace dgx

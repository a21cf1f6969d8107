// Element-local DG work shared by the element kernel (general meshes) and
// the fused stage kernel (Cartesian meshes): volume fluxes at the Gauss
// points (evaluate_sf + redistribute_sf), their integration against the test
// functions plus the face contributions (the GEMMs of dg_solver.h:336-340,
// mapToElement, addSFQ), and Dt*Minv with the RK4 stage update
// (rk_kernels.cu:22-56, rk.cc:164-198).  All data is in LDS; one 256-thread
// block processes batches of EPB elements.
#pragma once
#include <type_traits>

#include "physics.cuh"

namespace dgx {

__device__ constexpr double kRkBeta[4] = {0.0, 0.5, 0.5, 1.0};
__device__ constexpr double kRkGamma[4] = {1.0 / 6.0, 2.0 / 6.0, 2.0 / 6.0, 1.0 / 6.0};

constexpr int pow2ceil(int n) { return n <= 1 ? 1 : 2 * pow2ceil((n + 1) / 2); }

template <int D, int P, int PH>
struct Vol {
  using S = Shape<D, P>;
  static constexpr int NF = Fields<D, PH>::NF, Ns = S::Ns, NG = S::NG, Ms = S::Ms, NN = S::NN;
  static constexpr int NNC = Fields<D, PH>::NNC;  // non-conservative fields (the last NNC; no volume flux)
  static constexpr int NFX = NF - NNC;            // fields that carry a volume flux
  static constexpr int NU = NF * Ns;        // state doubles per element
  static constexpr int NQE = NN * NF * Ms;  // face-contribution doubles per element
  static constexpr int NQ = NFX * D + NNC;  // per-point values handed from phase 1 to phase 2
  static constexpr int TPE = pow2ceil(NG);  // lanes per element in phase 1
  static constexpr int EPB = 256 / TPE;     // elements per 256-thread batch
  static constexpr int NTAB_PHI = NG * Ns, NTAB_D = NG * D * Ns;
};

// Reference-element tables staged in LDS (derivative tables transposed so
// that lanes over nodes read consecutive banks).
template <int D, int P, int PH>
struct VolTables {
  double* phi;    // [g + i*NG]
  double* dphi;   // [(g*D+al) + i*NG*D]           (multifluid only)
  double* dw;     // [(g*D+al)*Ns + i]  = dphi_w transposed
  double* pw;     // [g*Ns + i]         = phi_w transposed (multifluid only)
  double* minv;   // [ii*Ns + i]        (uniform Minv only)
};

template <int D, int P, int PH>
__device__ inline void load_vol_tables(const VolTables<D, P, PH>& t, const double* phi, const double* dphi,
                                       const double* phi_w, const double* dphi_w, const double* Minv,
                                       bool uniform_minv, int tid, int nthr = 256) {
  using V = Vol<D, P, PH>;
  for (int k = tid; k < V::NTAB_PHI; k += nthr) t.phi[k] = phi[k];
  for (int k = tid; k < V::NTAB_D; k += nthr) {
    const int i = k / (V::NG * D), r = k % (V::NG * D);
    t.dw[r * V::Ns + i] = dphi_w[k];
    if constexpr (V::NNC > 0) t.dphi[k] = dphi[k];
  }
  if constexpr (V::NNC > 0)
    for (int k = tid; k < V::NTAB_PHI; k += nthr) t.pw[(k % V::NG) * V::Ns + k / V::NG] = phi_w[k];
  if (uniform_minv && Minv)
    for (int k = tid; k < V::Ns * V::Ns; k += nthr) t.minv[k] = Minv[k];
}

// The same tables for 256-thread blocks in two steps: fetch() issues every
// global load into registers and store() writes them to LDS, so that a
// caller can issue its own loads in between and wait once for all of them.
template <int D, int P, int PH>
struct VolTableFetch {
  using V = Vol<D, P, PH>;
  static constexpr int RP = (V::NTAB_PHI + 255) / 256, RD = (V::NTAB_D + 255) / 256;
  static constexpr int RM = (V::Ns * V::Ns + 255) / 256;
  static constexpr bool NC = V::NNC > 0;
  double phi[RP], pw[NC ? RP : 1], dw[RD], dphi[NC ? RD : 1], minv[RM];
  __device__ inline void fetch(const double* phi_g, const double* dphi_g, const double* phi_w, const double* dphi_w,
                               const double* Minv, bool with_minv, int tid) {
#pragma unroll
    for (int r = 0; r < RP; ++r) {
      const int k = tid + r * 256;
      if (k < V::NTAB_PHI) {
        phi[r] = phi_g[k];
        if constexpr (NC) pw[r] = phi_w[k];
      }
    }
#pragma unroll
    for (int r = 0; r < RD; ++r) {
      const int k = tid + r * 256;
      if (k < V::NTAB_D) {
        dw[r] = dphi_w[k];
        if constexpr (NC) dphi[r] = dphi_g[k];
      }
    }
#pragma unroll
    for (int r = 0; r < RM; ++r) {
      const int k = tid + r * 256;
      if (with_minv && k < V::Ns * V::Ns) minv[r] = Minv[k];
    }
  }
  __device__ inline void store(const VolTables<D, P, PH>& t, bool with_minv, int tid) const {
#pragma unroll
    for (int r = 0; r < RP; ++r) {
      const int k = tid + r * 256;
      if (k < V::NTAB_PHI) {
        t.phi[k] = phi[r];
        if constexpr (NC) t.pw[(k % V::NG) * V::Ns + k / V::NG] = pw[r];
      }
    }
#pragma unroll
    for (int r = 0; r < RD; ++r) {
      const int k = tid + r * 256;
      if (k < V::NTAB_D) {
        const int i = k / (V::NG * D), q = k % (V::NG * D);
        t.dw[q * V::Ns + i] = dw[r];
        if constexpr (NC) t.dphi[k] = dphi[r];
      }
    }
#pragma unroll
    for (int r = 0; r < RM; ++r) {
      const int k = tid + r * 256;
      if (with_minv && k < V::Ns * V::Ns) t.minv[k] = minv[r];
    }
  }
};

// Phase 1 for lane (element u, Gauss point g): fluxes with metric terms.
template <int D, int P, int PH>
__device__ inline void vol_phase1(const VolTables<D, P, PH>& t, int g, const double* u, double Je, const double* ij,
                                  double* out) {
  using V = Vol<D, P, PH>;
  constexpr int NF = V::NF, Ns = V::Ns, NG = V::NG, NFX = V::NFX, NNC = V::NNC;
  double ug[NF];
#pragma unroll
  for (int f = 0; f < NF; ++f) {
    double s = 0.0;
#pragma unroll
    for (int i = 0; i < Ns; ++i) s += u[f * Ns + i] * t.phi[g + i * NG];
    ug[f] = s;
  }
  double dua[(NNC ? NNC : 1) * D];
#pragma unroll
  for (int m = 0; m < NNC; ++m)
#pragma unroll
    for (int al = 0; al < D; ++al) {
      double s = 0.0;
#pragma unroll
      for (int i = 0; i < Ns; ++i) s += u[(NFX + m) * Ns + i] * t.dphi[(g * D + al) + i * NG * D];
      dua[m * D + al] = s;
    }
  double fx[NF * D];
  double snc[NNC ? NNC : 1];
  volume_flux<D, PH>(ug, dua, ij, fx, snc);
#pragma unroll
  for (int f = 0; f < NFX; ++f)
#pragma unroll
    for (int al = 0; al < D; ++al) {
      double sol = 0.0;
#pragma unroll
      for (int k = 0; k < D; ++k) sol += ij[al * D + k] * fx[f * D + k] * Je;
      out[f * D + al] = sol;
    }
#pragma unroll
  for (int m = 0; m < NNC; ++m) out[NFX * D + m] = snc[m] * Je;
}

// Phase 2 for lane (element, node i): S+F from the per-point values fe
// (NG x NQ) plus the face contributions qe (N_N x N_F x M_s, forward closure
// order per local edge).  At most two face terms land on a node, so their
// sum does not depend on the order.
template <int D, int P, int PH>
__device__ inline void vol_phase2(const VolTables<D, P, PH>& t, int i, const double* fe, const double* qe,
                                  double* rhs) {
  using V = Vol<D, P, PH>;
  constexpr int NF = V::NF, Ns = V::Ns, NG = V::NG, NFX = V::NFX, NQ = V::NQ, NN = V::NN, Ms = V::Ms, NNC = V::NNC;
  double acc[NF];
#pragma unroll
  for (int f = 0; f < NF; ++f) acc[f] = 0.0;
#pragma unroll 4
  for (int g = 0; g < NG; ++g) {
#pragma unroll
    for (int al = 0; al < D; ++al) {
      const double w = t.dw[(g * D + al) * Ns + i];
#pragma unroll
      for (int f = 0; f < NFX; ++f) acc[f] += w * fe[g * NQ + f * D + al];
    }
#pragma unroll
    for (int m = 0; m < NNC; ++m) acc[NFX + m] += t.pw[g * Ns + i] * fe[g * NQ + NFX * D + m];
  }
  double q[NF];
#pragma unroll
  for (int f = 0; f < NF; ++f) q[f] = 0.0;
#pragma unroll
  for (int kk = 0; kk < NN; ++kk)
#pragma unroll
    for (int jj = 0; jj < Ms; ++jj)
      if (closure_node<D, P>(kk, jj) == i)
#pragma unroll
        for (int f = 0; f < NF; ++f) q[f] += qe[(kk * NF + f) * Ms + jj];
#pragma unroll
  for (int f = 0; f < NF; ++f) rhs[f] = acc[f] + q[f];
}

// RK4 stage combination for one state entry (rk.cc:164-198 with DU fused):
// un = U^n, acc = accumulator (read for stages 1-3), du = Dt*Minv*f.
// The values rk_combine stores: the new accumulator (stages 0-2) and the
// stage output.
__device__ inline void rk_values(int st, double du, double un, double acc, double& acc_new, double& out) {
  const double gk = kRkGamma[st];
  if (st == 0) {
    acc_new = un + gk * du;
    out = un + kRkBeta[1] * du;
  } else if (st < 3) {
    acc_new = acc + gk * du;
    out = un + kRkBeta[st + 1] * du;
  } else {
    acc_new = acc;
    out = acc + gk * du;
  }
}

__device__ inline double rk_combine(int st, double du, double un, double acc, double* acc_out, double* out) {
  double an, o;
  rk_values(st, du, un, acc, an, o);
  if (st < 3) *acc_out = an;
  *out = o;
  return o;  // the stage output written
}

// Phase 3 for one state entry r = f*Ns + i of an element whose right-hand
// side R (NF x Ns) is in LDS: du = Dt * Minv * R, then the RK4 stage update
// at global index idx.
template <int D, int P, int PH>
__device__ inline void rk_update(const VolTables<D, P, PH>& t, const double* Mglob, bool uniform_minv, int r,
                                 const double* R, double dt, int st, size_t idx, const double* Un, double* Uacc,
                                 double* Uout) {
  using V = Vol<D, P, PH>;
  constexpr int Ns = V::Ns;
  const int f = r / Ns, i = r % Ns;
  const double* Rf = R + f * Ns;
  double sol = 0.0;
  if (uniform_minv) {
#pragma unroll
    for (int ii = 0; ii < Ns; ++ii) sol += t.minv[ii * Ns + i] * Rf[ii];
  } else {
#pragma unroll
    for (int ii = 0; ii < Ns; ++ii) sol += Mglob[ii * Ns + i] * Rf[ii];
  }
  const double un = st < 3 ? Un[idx] : 0.0;
  const double acc = st > 0 ? Uacc[idx] : 0.0;
  rk_combine(st, dt * sol, un, acc, Uacc + idx, Uout + idx);
}

}  // namespace dgx

namespace dgx {

typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef double f64x4_t __attribute__((ext_vector_type(4)));

// 16x16x4 matrix-core step in T, and where its result rows land.  Operands
// (both precisions): A lane l = row l%16, k = l/16; B lane l = column l%16,
// k = l/16.  Result register v of lane l holds column l%16 of row
//   v_mfma_f64_16x16x4f64: l/16 + 4v        v_mfma_f32_16x16x4f32: 4(l/16) + v
// Rows are (element, field) pairs of four elements x four fields, numbered
// by row(el, f) so that in both cases register v of lane l is field v of
// element l/16.
template <typename T>
struct Mfma16;
template <>
struct Mfma16<double> {
  using V4 = f64x4_t;
  static __device__ inline int row(int el, int f) { return el + 4 * f; }
  static __device__ inline int el(int r) { return r & 3; }
  static __device__ inline int field(int r) { return r >> 2; }
  static __device__ inline V4 mma(double a, double b, V4 c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
  }
};
template <>
struct Mfma16<float> {
  using V4 = f32x4_t;
  static __device__ inline int row(int el, int f) { return 4 * el + f; }
  static __device__ inline int el(int r) { return r >> 2; }
  static __device__ inline int field(int r) { return r & 3; }
  static __device__ inline V4 mma(float a, float b, V4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  }
};

// Split-BF16 operands for v_mfma_f32_16x16x16_bf16: x ~ hi + lo, both BF16
// (round to nearest even); a product is taken as hi*hi + hi*lo + lo*hi with
// FP32 accumulation (the lo*lo term, ~2^-16 relative, is dropped).
typedef short bf16x4_t __attribute__((ext_vector_type(4)));
__device__ inline unsigned bf16_rne(unsigned u) { return (u + 0x7fffu + ((u >> 16) & 1u)) & 0xffff0000u; }
__device__ inline void bf16_split(float x, short& hi, short& lo) {
  const unsigned h = bf16_rne(__float_as_uint(x));
  const unsigned l = bf16_rne(__float_as_uint(x - __uint_as_float(h)));
  hi = (short)(h >> 16);
  lo = (short)(l >> 16);
}
__device__ inline f32x4_t mma_bf16x3(const bf16x4_t& ah, const bf16x4_t& al, const bf16x4_t& bh, const bf16x4_t& bl,
                                     f32x4_t c) {
  c = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(ah, bh, c, 0, 0, 0);
  c = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(ah, bl, c, 0, 0, 0);
  return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(al, bh, c, 0, 0, 0);
}

// Shape of the matrix-core element phases of 2D order P with physics PH.
template <int P, int PH>
struct VolMfma {
  using V = Vol<2, P, PH>;
  static constexpr int NF = V::NF, Ns = V::Ns, NG = V::NG, NNC = V::NNC;
  static constexpr int NX = NF - 4;             // fields after rho, momenta and E
  static constexpr int NXC = NX - NNC;          // of them, in conservation form (the first)
  static constexpr int CB = (NG + 15) / 16;     // blocks of 16 Gauss points (columns of the map)
  static constexpr int KN = (Ns + 3) / 4;       // steps over nodes
  static constexpr int KG = (NG + 3) / 4;       // steps over Gauss points
  static constexpr int KP = 4 * KG + 1;         // row of flux values, padded
  static constexpr int NSR = NNC + 2 * NXC;     // row sets staged for the fields after E
};

// Doubles of per-wave LDS that vol_mfma_wave needs: 16 flux rows of one
// direction in T, and, apart, 8 rows for each row set of the fields after E.
template <typename T, int P>
constexpr int vol_wave_flux() { return (16 * VolMfma<P, 0>::KP * (int)sizeof(T) + 7) / 8; }
template <int P, int PH>
constexpr int vol_wave_extra() { return VolMfma<P, PH>::NSR * 8 * VolMfma<P, PH>::KP; }

// The lane's operands of the element phases, from the tables in global
// memory: column (or B-side) index c = l % 16, contraction index 4s + l / 16.
// Loaded before the block barrier that the phases wait at.
template <typename T, int P, int PH, typename TM = T>
struct VolOps {
  using M = VolMfma<P, PH>;
  // row strides of dphi_w and phi_w in LDS: lanes read along a column, which at
  // NG = 16 would lie in one bank (p = 2 with FP32 contractions, two-fluid
  // 1024x512 without limiter: 966 us a step unpadded, 935 so)
  static constexpr int LDD = 2 * M::NG + (M::NG % 16 == 0), LDP = M::NG + (M::NG % 16 == 0);
  TM phi[M::CB][M::KN];
  T dw[2][M::KG];
  double minv[M::KN];
  double xphi[M::NX ? M::CB : 1][M::KN], dphi[M::NNC ? 2 : 1][M::NNC ? M::CB : 1][M::KN], pw[M::NNC ? M::KG : 1];
  __device__ inline void load(const double* __restrict__ phi_g, const double* __restrict__ dphi_g,
                              const double* __restrict__ phi_w, const double* __restrict__ dphi_w,
                              const double* __restrict__ Minv, int tid) {
    constexpr int Ns = M::Ns, NG = M::NG;
    const int l = tid & 63, c = l & 15, q = l >> 4;
    // entries outside a table are 0, read from its first entry: no branch
    auto at = [](const double* __restrict__ t, bool in, int i) {
      const double v = t[in ? i : 0];
      return in ? v : 0.0;
    };
#pragma unroll
    for (int s = 0; s < M::KN; ++s) {
      const int k = 4 * s + q;
#pragma unroll
      for (int b = 0; b < M::CB; ++b) {
        const int g = 16 * b + c;
        const bool in = (Ns % 4 == 0 || k < Ns) && (NG % 16 == 0 || g < NG);
        const double v = at(phi_g, in, g + k * NG);
        phi[b][s] = (TM)v;
        if constexpr (M::NX > 0) xphi[b][s] = v;
        if constexpr (M::NNC > 0)
#pragma unroll
          for (int al = 0; al < 2; ++al) dphi[al][b][s] = at(dphi_g, in, (g * 2 + al) + k * NG * 2);
      }
      minv[s] = Minv ? at(Minv, k < Ns && c < Ns, k * Ns + c) : 0.0;
    }
#pragma unroll
    for (int s = 0; s < M::KG; ++s) {
      const int g = 4 * s + q;
      const bool in = (NG % 4 == 0 || g < NG) && (Ns == 16 || c < Ns);
#pragma unroll
      for (int al = 0; al < 2; ++al) dw[al][s] = (T)at(dphi_w, in, c * LDD + g * 2 + al);
      if constexpr (M::NNC > 0) pw[s] = at(phi_w, in, g + c * LDP);
    }
  }
};

__device__ inline void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Element phases of a tile of 32 2D elements of order P = 2 or 3 (256
// threads) on the matrix cores, contractions of rho, momenta and E in T:
// double for the FP64 path, float for the mixed-precision mode (FP32 inputs
// and accumulation; the pointwise flux, the fields after E, the face sums and
// everything after stay FP64).
//   map        Ug[(el,f)][g]  = sum_i U[el][f][i] phi[g][i]         fields 0..3
//   flux       fe[(el,f)][g,al] = sum_k (J_e invJac)[al][k] f_k(Ug)  in registers
//              (sGeo holds J_e invJac per element)
//   integrate  R[(el,f)][i]   = sum_{al} sum_g fe[(el,f)][g,al] dphi_w[g,al][i]
// Wave w owns elements 4w..4w+3 of both groups of 16.  After the map each
// lane holds the four conserved fields of one element at one Gauss point (two
// at p = 3: 25 points in two column blocks), so the flux needs no exchange;
// the scaled fluxes pass through the wave's own LDS rows, one direction at a
// time, into the integration, whose result registers plus the face sums are
// the right-hand side, written to sU.
//
// The fields after E (alpha; rho phic and phinc; alpha and beta) of the
// wave's eight elements are rows of matrix products of their own, both groups
// at once: row el8 + 8x (el8 = 4*group + element, x the field) puts field x of
// element l/16 of group g into result register 2x + g of lane l.  Their
// values and reference gradients at the points, the sources against phi_w,
// the flux of a conservative one against dphi_w and their share of Dt*Minv
// are 9 + 4 + 3 products of a wave at p = 2 two-fluid; as sums on the vector
// units they took 104 FMAs and 146 LDS reads of a lane (a third of the
// phase's), and their tables 4.6 KB of LDS.
//
// With with_minv the right-hand side is then replaced by du = dte * Minv * R,
// again on the FP64 matrix cores (A = R rows read back from sU).  No block
// barrier: every exchange stays inside the wave.  face(el, q) gives the
// face sums q[0..NF) of the lane's node (c) of tile element el.  sFlux needs
// 4 * vol_wave_flux<T, P>() doubles, sExtra 4 * vol_wave_extra<P, PH>().
// SPLIT (T = TM = float, P = 2): the map and the integration as split-BF16
// products on v_mfma_f32_16x16x16_bf16 (K = 16 per instruction: A lane l =
// row l%16, k = 4(l/16)+0..3; B lane l = column l%16, same k; D as the FP32
// 16x16x4 layout), three instructions per contraction block.
template <typename T, int P, int PH, int SU, typename TM, bool SPLIT, typename Face>
__device__ __forceinline__ void vol_mfma_wave(const VolOps<T, P, PH, TM>& op, const double* __restrict__ phi_g,
                                              const double* __restrict__ dphi_w, double* sU, const double* sGeo,
                                              double* sFlux, double* sExtra, int tid, bool with_minv,
                                              const double* dte, Face&& face) {
  static_assert(!SPLIT || (P == 2 && std::is_same<T, float>::value && std::is_same<TM, float>::value),
                "split-BF16 accumulates in FP32");
  // TM: type of the map (T unless set), T: type of the integration.  On gfx950
  // the FP32 16x16x4 integration measured slower than the FP64 one (volume
  // phase of a 2D p=2 tile: 11.0k against 7.3k cycles), the FP32 map about
  // as fast as the FP64 map.
  using M = Mfma16<T>;
  using MM = Mfma16<TM>;
  using M64 = Mfma16<double>;
  using S = VolMfma<P, PH>;
  constexpr int NF = S::NF, Ns = S::Ns, NG = S::NG, D = 2, KP = S::KP, NX = S::NX, NXC = S::NXC, NNC = S::NNC;
  constexpr int CB = S::CB, KN = S::KN, KG = S::KG;
  const int w = tid >> 6, l = tid & 63, c = l & 15, q = l >> 4;
  T* F = reinterpret_cast<T*>(sFlux + w * vol_wave_flux<T, P>());
  double* X = sExtra + w * vol_wave_extra<P, PH>();
  auto elem = [&](int e8) { return 16 * (e8 >> 2) + 4 * w + (e8 & 3); };  // tile element of this wave's e8-th
  // split-BF16 B operands: phi[g = c][i = 4q+j] for the map, dphi_w[i = c][g = 4q+j][al] for the integration
  bf16x4_t sphi_h = {0, 0, 0, 0}, sphi_l = {0, 0, 0, 0}, sdw_h[2], sdw_l[2];
  if constexpr (SPLIT) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int k = 4 * q + j;
      short h, lo;
      bf16_split(k < Ns ? (float)phi_g[c + k * NG] : 0.0f, h, lo);
      sphi_h[j] = h;
      sphi_l[j] = lo;
#pragma unroll
      for (int al = 0; al < D; ++al) {
        bf16_split(c < Ns ? (float)dphi_w[c * NG * D + k * D + al] : 0.0f, h, lo);
        sdw_h[al][j] = h;
        sdw_l[al][j] = lo;
      }
    }
  }
  // ---- the fields after E at the points, both groups: row c of A
  M64::V4 xv[NX ? CB : 1], xd[NNC ? 2 : 1][NNC ? CB : 1];
  const int xe = elem(c & 7), xf = 4 + (c >> 3);  // this lane's row: element and field (rows of absent fields are 0)
  if constexpr (NX > 0) {
#pragma unroll
    for (int b = 0; b < CB; ++b) {
      xv[b] = {0.0, 0.0, 0.0, 0.0};
      if constexpr (NNC > 0) xd[0][b] = xd[1][b] = {0.0, 0.0, 0.0, 0.0};
    }
#pragma unroll
    for (int s = 0; s < KN; ++s) {
      const int k = 4 * s + q;
      const double a = (Ns % 4 == 0 || k < Ns) && (NX == 2 || c < 8) ? sU[xe * SU + xf * Ns + k] : 0.0;
#pragma unroll
      for (int b = 0; b < CB; ++b) {
        xv[b] = M64::mma(a, op.xphi[b][s], xv[b]);
        if constexpr (NNC > 0)
#pragma unroll
          for (int al = 0; al < D; ++al) xd[al][b] = M64::mma(a, op.dphi[al][b][s], xd[al][b]);
      }
    }
  }
  const int a_el = MM::el(c), a_f = MM::field(c);
#pragma unroll
  for (int grp = 0; grp < 2; ++grp) {
    const int e_base = 16 * grp + 4 * w, el = e_base + q;
    // ---- map
    typename MM::V4 acc[CB];
#pragma unroll
    for (int b = 0; b < CB; ++b) acc[b] = {TM(0), TM(0), TM(0), TM(0)};
    if constexpr (SPLIT) {
      bf16x4_t ah, alo;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int k = 4 * q + j;
        short h, lo;
        bf16_split(k < Ns ? (float)sU[(e_base + a_el) * SU + a_f * Ns + k] : 0.0f, h, lo);
        ah[j] = h;
        alo[j] = lo;
      }
      acc[0] = mma_bf16x3(ah, alo, sphi_h, sphi_l, acc[0]);
    } else {
#pragma unroll
      for (int s = 0; s < KN; ++s) {
        const int k = 4 * s + q;
        const TM a = (Ns % 4 == 0 || k < Ns) ? (TM)sU[(e_base + a_el) * SU + a_f * Ns + k] : TM(0);
#pragma unroll
        for (int b = 0; b < CB; ++b) acc[b] = MM::mma(a, op.phi[b][s], acc[b]);
      }
    }
    // ---- flux of element el at point g = 16b + c with metric terms
    T fe[CB][4][D];
    {
      const double ij[4] = {sGeo[el * 4], sGeo[el * 4 + 1], sGeo[el * 4 + 2], sGeo[el * 4 + 3]};  // J_e invJac
#pragma unroll
      for (int b = 0; b < CB; ++b) {
        double ug[NF], dua[(NNC ? NNC : 1) * D], fx[NF * D], snc[NNC ? NNC : 1];
#pragma unroll
        for (int v = 0; v < 4; ++v) ug[v] = (double)acc[b][v];
        // points past the last (p = 3) repeat element q's first-block point
        const bool in = NG % 16 == 0 || 16 * b + c < NG;
        if constexpr (NG % 16 != 0) {
          if (b == CB - 1)
#pragma unroll
            for (int v = 0; v < 4; ++v) ug[v] = in ? ug[v] : (double)acc[0][v];
        }
#pragma unroll
        for (int x = 0; x < NX; ++x) ug[4 + x] = in ? xv[b][2 * x + grp] : xv[0][2 * x + grp];
#pragma unroll
        for (int m = 0; m < NNC; ++m)
#pragma unroll
          for (int al = 0; al < D; ++al) dua[m * D + al] = xd[al][b][2 * (NXC + m) + grp];
        volume_flux<2, PH>(ug, dua, ij, fx, snc);
        const bool row = NG % 16 == 0 || 16 * b + c < 4 * KG;  // within the padded row
#pragma unroll
        for (int f = 0; f < 4 + NXC; ++f)
#pragma unroll
          for (int al = 0; al < D; ++al) {
            double sol = 0.0;
#pragma unroll
            for (int k = 0; k < D; ++k) sol += ij[al * D + k] * fx[f * D + k];
            if (!in) sol = 0.0;
            if (f < 4) fe[b][f < 4 ? f : 0][al] = (T)sol;
            else if (row) X[((NNC + al) * 8 + 4 * grp + q) * KP + 16 * b + c] = sol;
          }
#pragma unroll
        for (int m = 0; m < NNC; ++m)
          if (row) X[(m * 8 + 4 * grp + q) * KP + 16 * b + c] = in ? snc[m] : 0.0;
      }
    }
    // ---- integration, one direction at a time through this wave's rows
    typename M::V4 r = {T(0), T(0), T(0), T(0)};
#pragma unroll
    for (int al = 0; al < D; ++al) {
#pragma unroll
      for (int b = 0; b < CB; ++b)
#pragma unroll
        for (int f = 0; f < 4; ++f)
          if (NG % 16 == 0 || 16 * b + c < 4 * KG) F[M::row(q, f) * KP + 16 * b + c] = fe[b][f][al];
      wave_sync();
      if constexpr (SPLIT) {
        bf16x4_t ah, alo;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          short h, lo;
          bf16_split((float)F[c * KP + 4 * q + j], h, lo);
          ah[j] = h;
          alo[j] = lo;
        }
        r = mma_bf16x3(ah, alo, sdw_h[al], sdw_l[al], r);
      } else {
#pragma unroll
        for (int s = 0; s < KG; ++s) r = M::mma(F[c * KP + 4 * s + q], op.dw[al][s], r);
      }
      wave_sync();  // the rows are rewritten next
    }
    if (Ns == 16 || c < Ns) {
      double qs[NF];
      face(el, qs);
#pragma unroll
      for (int v = 0; v < 4; ++v) sU[el * SU + v * Ns + c] = (double)r[v] + qs[v];
#pragma unroll
      for (int x = 0; x < NX; ++x) sU[el * SU + (4 + x) * Ns + c] = qs[4 + x];
    }
  }
  // ---- the fields after E: sources and fluxes integrated, both groups
  if constexpr (NX > 0) {
    M64::V4 rx = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int s = 0; s < KG; ++s) {
      const int g = 4 * s + q, x = c >> 3;
      // rows of field x: its source (the last NNC), or nothing here
      const int m = x - NXC;
      const double a = (m >= 0 && m < NNC) ? X[(m * 8 + (c & 7)) * KP + g] : 0.0;
      rx = M64::mma(a, op.pw[s], rx);
    }
    if constexpr (NXC > 0) {
#pragma unroll
      for (int al = 0; al < D; ++al)
#pragma unroll
        for (int s = 0; s < KG; ++s) {
          const double a = c < 8 ? X[((NNC + al) * 8 + c) * KP + 4 * s + q] : 0.0;
          rx = M64::mma(a, (double)op.dw[al][s], rx);
        }
    }
    if (Ns == 16 || c < Ns)
#pragma unroll
      for (int x = 0; x < NX; ++x)
#pragma unroll
        for (int grp = 0; grp < 2; ++grp) {
          double* u = sU + (16 * grp + 4 * w + q) * SU + (4 + x) * Ns + c;
          *u = rx[2 * x + grp] + *u;
        }
  }
  if (with_minv) {
    // du = dte * Minv R: rows (el, f) = el + 4f of the four elements, columns = nodes
    wave_sync();  // the right-hand side of the eight elements is in sU
    M64::V4 du[2], dx = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int grp = 0; grp < 2; ++grp) {
      du[grp] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
      for (int s = 0; s < KN; ++s) {
        const int k = 4 * s + q;
        const double a = (Ns % 4 == 0 || k < Ns)
                             ? sU[(16 * grp + 4 * w + M64::el(c)) * SU + M64::field(c) * Ns + k]
                             : 0.0;
        du[grp] = M64::mma(a, op.minv[s], du[grp]);
      }
    }
    if constexpr (NX > 0) {
#pragma unroll
      for (int s = 0; s < KN; ++s) {
        const int k = 4 * s + q;
        const double a = (Ns % 4 == 0 || k < Ns) && (NX == 2 || c < 8) ? sU[xe * SU + xf * Ns + k] : 0.0;
        dx = M64::mma(a, op.minv[s], dx);
      }
    }
    wave_sync();  // every lane has read the right-hand side
    if (Ns == 16 || c < Ns)
#pragma unroll
      for (int grp = 0; grp < 2; ++grp) {
        const int el = 16 * grp + 4 * w + q;
        const double d = dte[el];
#pragma unroll
        for (int v = 0; v < 4; ++v) sU[el * SU + v * Ns + c] = d * du[grp][v];
#pragma unroll
        for (int x = 0; x < NX; ++x) sU[el * SU + (4 + x) * Ns + c] = d * dx[2 * x + grp];
      }
  }
}

// Node of the 2D p = 2 element (Gmsh order) at the lane's place of
// vol_tensor_wave (column a = l % 4, row b = l / 16 of the lattice), or -1.
__device__ inline int tensor_node(int l) {
  const int a = l & 3, b = (l >> 4) & 3;
  // rows of the lattice: 0 4 1 / 7 8 5 / 3 6 2
  constexpr unsigned long long kNodes = 0xfff'f'f263'f587'f140ull;
  const int n = (int)((kNodes >> (16 * b + 4 * a)) & 15);
  return n == 15 ? -1 : n;
}

// The same phases for P = 2 in FP64 as chains of 4x4 products: three nodes and
// four Gauss points per direction fit v_mfma_f64_4x4x4_4b_f64, four
// independent 4x4x4 products, one element each.  Its operands (lane l = 16r +
// 4e + c: A row c, B column c, contraction index r, D row r, column c, of
// block e) make a result usable as the next product's A with its row index
// contracted, so a field goes through both directions, to the points and
// back, without leaving its registers:
//   u[b][a] -> A1[a][gy] = sum_b u[b][a] V[gy][b] -> A2[gy][gx] = sum_a A1[a][gy] V[gx][a]
// (derivative tables in place of V for the gradients), the flux in the lane of
// its point, the test integrals and the mass matrix the same way.  Lane:
// element e of the wave's group, node (a = c, b = r) or point (gx = c, gy = r).
//
// FP64 matrix and vector instructions share the FP64 units on this chip
// (measured: 64 cycles a 16x16x4 product whatever runs beside it, while the
// vector FMAs beside it drop from one in 2.8 cycles to one in 9.9; 19 cycles a
// 4x4x4), so what counts is their sum: 82 products of 16 cycles a wave against
// 44 of 64 for two-fluid with 16x16 tiles, whose rows and columns padding half
// fills; and no flux rows (8.7 KB), no tables (7.6 KB) and no barriers in LDS.
// tab: the tables in LDS, [table][r*4 + c]: V, V', V*w, V'*w, inverse 1D mass
// matrix (tensor_tables).  dtj: Dt / J per element.
constexpr int kTensorTables = 5;
template <int PH, int SU, typename Face>
__device__ __forceinline__ void vol_tensor_wave(const double* tab, double* sU, const double* sGeo, int tid,
                                                bool with_minv, const double* dtj, Face&& face) {
  using V = Vol<2, 2, PH>;
  constexpr int NF = V::NF, Ns = V::Ns, NFX = V::NFX, NNC = V::NNC, D = 2;
  const int w = tid >> 6, l = tid & 63, r = l >> 4, e = (l >> 2) & 3, c = l & 3;
  auto mma = [](double a, double b, double acc) { return __builtin_amdgcn_mfma_f64_4x4x4f64(a, b, acc, 0, 0, 0); };
  const double bV = tab[r * 4 + c], bD = tab[16 + r * 4 + c], bVw = tab[32 + r * 4 + c], bDw = tab[48 + r * 4 + c],
               bM = tab[64 + r * 4 + c];
  const int node = tensor_node(l);
  const bool on = node >= 0;
#pragma unroll
  for (int grp = 0; grp < 2; ++grp) {
    const int el = 16 * grp + 4 * w + e;
    double* ue = sU + el * SU + (on ? node : 0);
    double u[NF];
#pragma unroll
    for (int f = 0; f < NF; ++f) {
      const double v = ue[f * Ns];
      u[f] = on ? v : 0.0;
    }
    double ug[NF], dua[(NNC ? NNC : 1) * D];
#pragma unroll
    for (int f = 0; f < NF; ++f) {
      const double a1 = mma(u[f], bV, 0.0);
      ug[f] = mma(a1, bV, 0.0);
      if (f >= NFX) {
        dua[(f - NFX) * D] = mma(a1, bD, 0.0);
        dua[(f - NFX) * D + 1] = mma(mma(u[f], bD, 0.0), bV, 0.0);
      }
    }
    const double ij[4] = {sGeo[el * 4], sGeo[el * 4 + 1], sGeo[el * 4 + 2], sGeo[el * 4 + 3]};  // J_e invJac
    double fx[NF * D], snc[NNC ? NNC : 1], R[NF];
    volume_flux<2, PH>(ug, dua, ij, fx, snc);
#pragma unroll
    for (int f = 0; f < NFX; ++f) {
      const double f0 = ij[0] * fx[f * D] + ij[1] * fx[f * D + 1], f1 = ij[2] * fx[f * D] + ij[3] * fx[f * D + 1];
      R[f] = mma(mma(f0, bVw, 0.0), bDw, 0.0);
      R[f] = mma(mma(f1, bDw, 0.0), bVw, R[f]);
    }
#pragma unroll
    for (int m = 0; m < NNC; ++m) R[NFX + m] = mma(mma(snc[m], bVw, 0.0), bVw, 0.0);
    double qs[NF];
    face(el, qs);
#pragma unroll
    for (int f = 0; f < NF; ++f) R[f] = on ? R[f] + qs[f] : 0.0;
    if (with_minv) {
      const double d = dtj[el];
#pragma unroll
      for (int f = 0; f < NF; ++f) R[f] = d * mma(mma(R[f], bM, 0.0), bM, 0.0);
    }
    if (on)
#pragma unroll
      for (int f = 0; f < NF; ++f) ue[f * Ns] = R[f];
  }
}

// Offsets (kk*NF*Ms + jj) of the at most two face slots that land on node i
// (closure_node(kk, jj) == i, edges in order), -1 when absent; field f adds f*Ms.
// Built at compile time; each block copies it into LDS.
template <int NF>
struct NodeQ {
  int v[18];
  constexpr NodeQ() : v{} {
    for (int i = 0; i < 9; ++i) {
      int n = 0, o[2] = {-1, -1};
      for (int kk = 0; kk < 4; ++kk)
        for (int jj = 0; jj < 3; ++jj)
          if (closure_node<2, 2>(kk, jj) == i && n < 2) o[n++] = kk * NF * 3 + jj;
      v[2 * i] = o[0];
      v[2 * i + 1] = o[1];
    }
  }
};
template <int NF>
__device__ constexpr NodeQ<NF> kNodeQ{};

template <int NF>
__device__ inline void node_q_table(int* t, int tid) {
  if (tid < 18) t[tid] = kNodeQ<NF>.v[tid];
}

}  // namespace dgx

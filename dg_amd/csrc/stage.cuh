// Fused RK stage for Cartesian meshes (grid order; sides of whole tiles or, in
// 2D, any): one kernel evaluates the whole right-
// hand side of a tile of elements and applies Dt*Minv and the RK4 update.
//
// A 256-thread block owns a TX x TY tile (TX in 1D).  It stages the tile's
// state and the face traces of its halo in LDS, evaluates every face that
// touches the tile (faces on tile edges are evaluated by both neighbouring
// tiles with identical inputs and code), integrates them against psi_w,
// then runs the element phases of volume.cuh and writes the stage update.
// Face sides, closures, normals and boundary treatment follow the reference
// interface construction (simpleMesh.cc:770-989: side 0 = first element in
// element order, its outward normal; boundary faces contribute to side 0
// only, dg_functions.cc:225-233), so the result equals the general
// face/element kernels.  Tiles are mapped to XCDs in contiguous bands so
// that halo rows are shared through each XCD's L2.
#pragma once
#include <algorithm>
#include <cstdint>
#include <type_traits>

#include "dgx_internal.h"
#include "physics.cuh"
#include "sensor.cuh"
#include "volume.cuh"

namespace dgx {

struct StageArgs {
  const double* __restrict__ phi;
  const double* __restrict__ dphi;
  const double* __restrict__ phi_w;
  const double* __restrict__ dphi_w;
  const double* __restrict__ psi;
  const double* __restrict__ psi_w;
  const double* __restrict__ Minv;    // [e*minv_stride] N_s x N_s
  const double* __restrict__ J;       // [e*geo_stride]
  const double* __restrict__ invJac;  // [(e*geo_stride)*D*D + alpha*D + a]
  const double* __restrict__ gx;      // faces normal to x: [(ey*(nx+1) + fx)*4 + {n_x, n_y, JF0, JF1}]
  const double* __restrict__ gy;      // faces normal to y: [(fy*nx + ex)*4 + {n_x, n_y, JF0, JF1}]
  double J0;                          // Jacobian of the element whose Minv is stored when minv_stride == 0
  int geo_stride, minv_stride;
  int nx, ny;
  int bc[4];  // left, right, bottom, top
  int tiles_x, tiles_y;
  int stage;
  const double* Uin;
  const double* Un;
  double* Uacc;
  double* Uout;
  const double* __restrict__ dt;
  double* fout;
  // 2D p=2 two-fluid RK stages: cell means of rho, p and alpha of the output
  // tile for the learned indicator ([e*3 + k], cell_means_rpa with w0), or null
  double* means;
  const double* __restrict__ w0;
  const double* __restrict__ tensor;  // 2D p=2: 1D tables of vol_tensor_wave
  double* uavg;   // 2D p=2,3 RK stages: the output's sensor averages [e*NF + f] (sensor_nodal_mean), or null
  double* psens;  // with means and uavg: the averages' sensor pressures [e]
  const int* gate;  // set and nonzero: the launch does nothing (a step skipped by the device-side time control)
};

template <int D, int TX, int TY>
struct Tile {
  static constexpr int NT = TX * TY;
  static constexpr int NFX = (D == 1) ? TX + 1 : (TX + 1) * TY;  // faces normal to x
  static constexpr int NFY = (D == 1) ? 0 : TX * (TY + 1);       // faces normal to y
  static constexpr int NFACE = NFX + NFY;
  static constexpr int NH = (D == 1) ? 2 : 2 * TY + 2 * TX;      // halo trace slots: L, R, B, T
};

// Where each side of a tile face reads its trace and where it contributes.
// RAG (2D): the tile may reach past the grid's right and upper ends; faces
// there contribute nowhere and read the tile's first element.
struct FaceDesc {
  int src[2];     // tile slot (>= 0) or halo slot (-1 - h)
  int cl[2];      // closure id used by the side (tile sources)
  int dst[2];     // tile slot receiving this side's contribution, or -1
  int edge[2];    // local edge of the receiving element
  int tag;        // 0 interior, else boundary physical tag
  int geo;        // index of the face in gx (x-faces) or gy (y-faces)
  bool xf;        // face normal to x
};

template <int D, int TX, int TY, bool RAG>
__device__ inline FaceDesc face_desc(int fi, int ex0, int ey0, const StageArgs& a) {
  FaceDesc d;
  d.dst[0] = d.dst[1] = -1;
  d.edge[0] = d.edge[1] = 0;
  if constexpr (D == 1) {
    const int exl = ex0 + fi - 1, exr = ex0 + fi;
    d.xf = true;
    d.geo = ex0 + fi;
    if (exl < 0) {  // left domain boundary: side 0 = element 0, closure 0
      d.tag = a.bc[0];
      d.src[0] = 0; d.cl[0] = 0;
      if (d.tag == BC_PERIODIC) { d.src[1] = -1 - 0; d.cl[1] = 1; } else { d.src[1] = 0; d.cl[1] = 0; }
      d.dst[0] = 0; d.edge[0] = 0;
    } else if (exr >= a.nx) {  // right domain boundary: side 0 = last element, closure 1
      d.tag = a.bc[1];
      d.src[0] = TX - 1; d.cl[0] = 1;
      if (d.tag == BC_PERIODIC) { d.src[1] = -1 - 1; d.cl[1] = 0; } else { d.src[1] = TX - 1; d.cl[1] = 1; }
      d.dst[0] = TX - 1; d.edge[0] = 1;
    } else {
      d.tag = 0;
      d.src[0] = (fi == 0) ? -1 - 0 : fi - 1; d.cl[0] = 1;
      d.src[1] = (fi == TX) ? -1 - 1 : fi; d.cl[1] = 0;
      if (fi > 0) { d.dst[0] = fi - 1; d.edge[0] = 1; }
      if (fi < TX) { d.dst[1] = fi; d.edge[1] = 0; }
    }
  } else {
    if constexpr (RAG) {
      const bool xf = fi < Tile<D, TX, TY>::NFX;
      const int fj = xf ? fi : fi - Tile<D, TX, TY>::NFX, w = xf ? TX + 1 : TX;
      const int y = ey0 + fj / w, x = ex0 + fj % w;
      if (xf ? (y >= a.ny || x > a.nx) : (x >= a.nx || y > a.ny)) {
        d.xf = xf;
        d.tag = 0;
        d.geo = xf ? ey0 * (a.nx + 1) + ex0 : ey0 * a.nx + ex0;
        d.src[0] = d.src[1] = 0;
        d.cl[0] = d.cl[1] = 0;
        return d;
      }
    }
    if (fi < Tile<D, TX, TY>::NFX) {
      const int ty = fi / (TX + 1), fx = fi % (TX + 1);
      const int exl = ex0 + fx - 1, exr = ex0 + fx;
      d.xf = true;
      d.geo = (ey0 + ty) * (a.nx + 1) + ex0 + fx;
      if (exl < 0) {
        d.tag = a.bc[0];
        d.src[0] = ty * TX; d.cl[0] = 3;
        if (d.tag == BC_PERIODIC) { d.src[1] = -1 - ty; d.cl[1] = 5; } else { d.src[1] = ty * TX; d.cl[1] = 3; }
        d.dst[0] = ty * TX; d.edge[0] = 3;
      } else if (exr >= a.nx) {
        d.tag = a.bc[1];
        d.src[0] = ty * TX + fx - 1; d.cl[0] = 1;
        if (d.tag == BC_PERIODIC) { d.src[1] = -1 - (TY + ty); d.cl[1] = 7; } else { d.src[1] = ty * TX + fx - 1; d.cl[1] = 1; }
        d.dst[0] = ty * TX + fx - 1; d.edge[0] = 1;
      } else {
        d.tag = 0;
        d.src[0] = (fx == 0) ? -1 - ty : ty * TX + fx - 1; d.cl[0] = 1;
        d.src[1] = (fx == TX) ? -1 - (TY + ty) : ty * TX + fx; d.cl[1] = 7;
        if (fx > 0) { d.dst[0] = ty * TX + fx - 1; d.edge[0] = 1; }
        if (fx < TX) { d.dst[1] = ty * TX + fx; d.edge[1] = 3; }
      }
    } else {
      const int fj = fi - Tile<D, TX, TY>::NFX;
      const int fy = fj / TX, tx = fj % TX;
      const int eyl = ey0 + fy - 1, eyu = ey0 + fy;
      d.xf = false;
      d.geo = (ey0 + fy) * a.nx + ex0 + tx;
      if (eyl < 0) {
        d.tag = a.bc[2];
        d.src[0] = tx; d.cl[0] = 0;
        if (d.tag == BC_PERIODIC) { d.src[1] = -1 - (2 * TY + tx); d.cl[1] = 6; } else { d.src[1] = tx; d.cl[1] = 0; }
        d.dst[0] = tx; d.edge[0] = 0;
      } else if (eyu >= a.ny) {
        d.tag = a.bc[3];
        d.src[0] = (fy - 1) * TX + tx; d.cl[0] = 2;
        if (d.tag == BC_PERIODIC) { d.src[1] = -1 - (2 * TY + TX + tx); d.cl[1] = 4; }
        else { d.src[1] = (fy - 1) * TX + tx; d.cl[1] = 2; }
        d.dst[0] = (fy - 1) * TX + tx; d.edge[0] = 2;
      } else {
        d.tag = 0;
        d.src[0] = (fy == 0) ? -1 - (2 * TY + tx) : (fy - 1) * TX + tx; d.cl[0] = 2;
        d.src[1] = (fy == TY) ? -1 - (2 * TY + TX + tx) : fy * TX + tx; d.cl[1] = 4;
        if (fy > 0) { d.dst[0] = (fy - 1) * TX + tx; d.edge[0] = 2; }
        if (fy < TY) { d.dst[1] = fy * TX + tx; d.edge[1] = 0; }
      }
    }
  }
  return d;
}

// Global element and closure of halo slot h, or -1 when the slot is unused.
template <int D, int TX, int TY, bool RAG>
__device__ inline int halo_source(int h, int ex0, int ey0, const StageArgs& a, int& cl) {
  if constexpr (D == 1) {
    if (h == 0) {
      cl = 1;
      if (ex0 > 0) return ex0 - 1;
      return a.bc[0] == BC_PERIODIC ? a.nx - 1 : -1;
    }
    cl = 0;
    if (ex0 + TX < a.nx) return ex0 + TX;
    return a.bc[1] == BC_PERIODIC ? 0 : -1;
  } else {
    const int nx = a.nx, ny = a.ny;
    if constexpr (RAG) {  // rows and columns past the grid's ends
      if (h < 2 * TY ? ey0 + (h < TY ? h : h - TY) >= ny : ex0 + (h - 2 * TY < TX ? h - 2 * TY : h - 2 * TY - TX) >= nx)
        return -1;
    }
    if (h < TY) {  // left of row h
      const int row = ey0 + h;
      if (ex0 > 0) { cl = 1; return row * nx + ex0 - 1; }
      cl = 5;
      return a.bc[0] == BC_PERIODIC ? row * nx + nx - 1 : -1;
    }
    if (h < 2 * TY) {  // right of row h - TY
      const int row = ey0 + h - TY;
      cl = 7;
      if (ex0 + TX < nx) return row * nx + ex0 + TX;
      return a.bc[1] == BC_PERIODIC ? row * nx : -1;
    }
    if (h < 2 * TY + TX) {  // below column
      const int col = ex0 + h - 2 * TY;
      if (ey0 > 0) { cl = 2; return (ey0 - 1) * nx + col; }
      cl = 6;
      return a.bc[2] == BC_PERIODIC ? (ny - 1) * nx + col : -1;
    }
    const int col = ex0 + h - 2 * TY - TX;  // above column
    cl = 4;
    if (ey0 + TY < ny) return (ey0 + TY) * nx + col;
    return a.bc[3] == BC_PERIODIC ? col : -1;
  }
}

// Per-element LDS stride for n doubles: with padding, the smallest stride
// >= n whose element starts fall on distinct, non-overlapping 16-byte bank
// groups for the four elements a wave reads at once (2*stride mod 32 dwords
// in [4, 28]).
constexpr bool bank_ok(int n) { return (2 * n) % 32 >= 4 && (2 * n) % 32 <= 28; }
constexpr int lds_stride(int n) { return bank_ok(n) ? n : lds_stride(n + 1); }

// The tile of this block, or -1.  Blocks are dispatched round-robin over the
// 8 XCDs; the tiles of each XCD form a contiguous band of the grid, so that
// halo rows are shared in its L2 (the launch has a multiple of 8 blocks).
__device__ inline int tile_of(const StageArgs& a) {
  const int per = gridDim.x >> 3, t = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
  return t < a.tiles_x * a.tiles_y ? t : -1;
}

// The tile kernel with the element phases as batches on the vector units: 1D,
// and first order in 2D (four nodes and points per element: no matrix shape).
// RAG (2D): the grid's sides need not be whole tiles; the tile's elements past
// its ends repeat the tile's first element and are not stored.  VEC (2D): the
// tile state, the RK operands and the output move as 16-byte pairs (first order
// has an even number of values an element): two-fluid 440x220 with limiter 190 us a
// step against 205 in single doubles.
template <int D, int P, int PH, int FL, int MODE, int TX, int TY, bool VEC, bool RAG>
__global__ __launch_bounds__(256) void k_stage(StageArgs a) {
  if (a.gate && *a.gate) return;
  static_assert(!RAG || D == 2, "ragged tiles: 2D");
  using V = Vol<D, P, PH>;
  using T = Tile<D, TX, TY>;
  constexpr int NF = V::NF, Ns = V::Ns, NG = V::NG, Ms = V::Ms, MG = Shape<D, P>::MG;
  constexpr int NU = V::NU, NQE = V::NQE, NQ = V::NQ, TPE = V::TPE, EPB = V::EPB;
  constexpr int NT = T::NT, NFACE = T::NFACE, NH = T::NH, HT = NF * Ms;
  constexpr int SU = lds_stride(NU), SQ = lds_stride(NQE), SW = lds_stride(NG * NQ);
  constexpr int NNC = V::NNC;    // non-conservative fields: the last NNC
  constexpr int NWP = NF + NNC;  // per face point: F, and the non-conservative terms
  constexpr int NW_FACE = NFACE * MG * NWP, NW_VOL = EPB * SW;
  constexpr int NW = NW_FACE > NW_VOL ? NW_FACE : NW_VOL;
  constexpr int NGEO = 1 + D * D;
  // per-thread counts of the loaded quantities
  constexpr int VW = VEC ? 2 : 1;
  static_assert(!VEC || NU % 2 == 0, "pairs within an element");
  constexpr int R_U = (NT * NU / VW + 255) / 256, R_H = (NH * HT + 255) / 256;
  constexpr int R_G = (NT * NGEO + 255) / 256, R_F = (NFACE * 4 + 255) / 256;

  __shared__ double sU[NT * SU];
  __shared__ double sH[NH * HT];
  __shared__ double sQ[NT * SQ];
  __shared__ double sW[NW];  // face-point fluxes, then per-point volume values
  __shared__ double sPhi[V::NTAB_PHI];
  __shared__ double sDphi[PH ? V::NTAB_D : 1];
  __shared__ double sDw[V::NTAB_D];
  __shared__ double sPw[PH ? V::NTAB_PHI : 1];
  __shared__ double sMinv[Ns * Ns];
  __shared__ double sPsi[MG * Ms], sPsiw[MG * Ms];
  __shared__ double sGeo[NT * NGEO];  // per element: J, invJac
  __shared__ double sDte[NT];         // per element: Dt (J_0/J_e with the shared Minv)
  __shared__ double sFG[NFACE * 4];   // per tile face: n_x, n_y, JF side 0, JF side 1
  __shared__ int sFD[NFACE];          // per tile face: receiving slot, edge and closure of each side (packed)
  __shared__ int sFS[NFACE];          // per tile face: source slot of each side (+128, 8 bits each), boundary tag << 16
  static_assert(NT <= 128 && NH <= 128, "face sources fit 8 bits");
  const VolTables<D, P, PH> tb{sPhi, sDphi, sDw, sPw, sMinv};

  const int tid = threadIdx.x, tile = tile_of(a);
  if (tile < 0) return;
  const bool shared_minv = a.minv_stride == 0;
  // reference tables and the tile's inputs are fetched together (one wait)
  static_assert(MG * Ms <= 256, "face tables fit one pass");
  VolTableFetch<D, P, PH> tf;
  tf.fetch(a.phi, a.dphi, a.phi_w, a.dphi_w, a.Minv, MODE == 1 && shared_minv, tid);
  double psi_r = 0.0, psiw_r = 0.0;
  if (tid < MG * Ms) { psi_r = a.psi[tid]; psiw_r = a.psi_w[tid]; }
  const double dt = (MODE == 1) ? a.dt[0] : 0.0;
  const int ex0 = (tile % a.tiles_x) * TX, ey0 = (tile / a.tiles_x) * TY;
  // Lanes past the tile's entries read its last ones: under a condition the
  // pairs of both rounds became one value, whose copy waited for the first load
  // before any other was issued (a launch of two-fluid 64x32 7.9 us, 7.55 so;
  // 200x100 11.95 and 11.65).
  double pu[R_U * VW], ph[R_H], pg[R_G], pf[R_F];
#pragma unroll
  for (int r = 0; r < R_U; ++r) {
    const int k = min(VW * (tid + r * 256), NT * NU - VW);
    const int ty = k / (TX * NU);
    const double* src = a.Uin + ((size_t)(ey0 + ty) * a.nx + ex0) * NU + (k - ty * TX * NU);
    if constexpr (RAG) {
      if (ey0 + ty >= a.ny || k - ty * TX * NU >= (a.nx - ex0) * NU)
        src = a.Uin + ((size_t)ey0 * a.nx + ex0) * NU + k % NU;
    }
    if constexpr (VEC) {
      const double2 v = *reinterpret_cast<const double2*>(src);
      pu[2 * r] = v.x;
      pu[2 * r + 1] = v.y;
    } else {
      pu[r] = *src;
    }
  }
#pragma unroll
  for (int r = 0; r < R_H; ++r) {
    const int k = tid + r * 256;
    if (k < NH * HT) {
      const int h = k / HT, q = k % HT, f = q / Ms, j = q % Ms;
      int cl = 0;
      const int e = halo_source<D, TX, TY, RAG>(h, ex0, ey0, a, cl);
      ph[r] = (e >= 0) ? a.Uin[((size_t)e * NF + f) * Ns + closure_node<D, P>(cl, j)] : 0.0;
    }
  }
#pragma unroll
  for (int r = 0; r < R_G; ++r) {
    const int k = tid + r * 256;
    if (k < NT * NGEO) {
      const int el = k / NGEO, q = k % NGEO;
      const int ty = RAG ? min(el / TX, a.ny - 1 - ey0) : el / TX, tx = RAG ? min(el % TX, a.nx - 1 - ex0) : el % TX;
      const int eg = ((ey0 + ty) * a.nx + ex0 + tx) * a.geo_stride;
      pg[r] = q == 0 ? a.J[eg] : a.invJac[eg * D * D + q - 1];
    }
  }
#pragma unroll
  for (int r = 0; r < R_F; ++r) {
    const int k = tid + r * 256;
    if (k < NFACE * 4) {
      const int fi = k / 4, q = k % 4;
      const double* src;
      if (D == 1 || fi < T::NFX) {
        int ty = (D == 1) ? 0 : fi / (TX + 1), fx = (D == 1) ? fi : fi % (TX + 1);
        if constexpr (RAG) ty = min(ty, a.ny - 1 - ey0), fx = min(fx, a.nx - ex0);
        src = a.gx + ((size_t)(ey0 + ty) * (a.nx + 1) + ex0 + fx) * 4;
      } else {
        const int fj = fi - T::NFX;
        int fy = fj / TX, tx = fj % TX;
        if constexpr (RAG) fy = min(fy, a.ny - ey0), tx = min(tx, a.nx - 1 - ex0);
        src = a.gy + ((size_t)(ey0 + fy) * a.nx + ex0 + tx) * 4;
      }
      pf[r] = src[q];
    }
  }
  // the descriptor of every tile face, once per face (one lane each, while
  // the tile's loads are in flight); the face and integration phases read it
  for (int fi = tid; fi < NFACE; fi += 256) {
    const FaceDesc fd = face_desc<D, TX, TY, RAG>(fi, ex0, ey0, a);
    sFD[fi] = ((fd.dst[0] + 1) | (fd.edge[0] << 8) | (fd.cl[0] << 10)) |
              (((fd.dst[1] + 1) | (fd.edge[1] << 8) | (fd.cl[1] << 10)) << 16);
    sFS[fi] = (fd.src[0] + 128) | ((fd.src[1] + 128) << 8) | (fd.tag << 16);
  }
  tf.store(tb, MODE == 1 && shared_minv, tid);
  if (tid < MG * Ms) { sPsi[tid] = psi_r; sPsiw[tid] = psiw_r; }
  auto gidx = [&](int k) -> size_t {
    const int ty = k / (TX * NU);
    return ((size_t)(ey0 + ty) * a.nx + ex0) * NU + (k - ty * TX * NU);
  };
  auto in_grid = [&](int k) {  // tile entry k belongs to the grid (its row's end is a whole number of elements)
    const int ty = k / (TX * NU);
    return !RAG || (ey0 + ty < a.ny && k - ty * TX * NU < (a.nx - ex0) * NU);
  };
#pragma unroll
  for (int r = 0; r < R_U; ++r) {
    const int k = VW * (tid + r * 256);
    if (k < NT * NU)
#pragma unroll
      for (int v = 0; v < VW; ++v) sU[(k / NU) * SU + k % NU + v] = pu[r * VW + v];
  }
#pragma unroll
  for (int r = 0; r < R_H; ++r) {
    const int k = tid + r * 256;
    if (k < NH * HT) sH[k] = ph[r];
  }
#pragma unroll
  for (int r = 0; r < R_G; ++r) {
    const int k = tid + r * 256;
    if (k < NT * NGEO) sGeo[k] = pg[r];
  }
#pragma unroll
  for (int r = 0; r < R_F; ++r) {
    const int k = tid + r * 256;
    if (k < NFACE * 4) sFG[k] = pf[r];
  }
  __syncthreads();
  // the output's Dt factor once per element (read after several barriers)
  if (MODE == 1 && tid < NT) sDte[tid] = shared_minv ? dt * (a.J0 / sGeo[tid * NGEO]) : dt;
  // RK operands of this thread's output entries, in flight during the compute below
  double pre_un[R_U * VW], pre_acc[R_U * VW];
#pragma unroll
  for (int r = 0; r < R_U; ++r) {
    const int k = VW * (tid + r * 256);
#pragma unroll
    for (int v = 0; v < VW; ++v) pre_un[r * VW + v] = pre_acc[r * VW + v] = 0.0;
    if (MODE == 1 && k < NT * NU && in_grid(k)) {
      const size_t i = gidx(k);
      auto fetch = [&](const double* from, double* to) {
        if constexpr (VEC) {
          const double2 v = *reinterpret_cast<const double2*>(from + i);
          to[0] = v.x;
          to[1] = v.y;
        } else {
          to[0] = from[i];
        }
      };
      if (a.stage < 3) fetch(a.Un, pre_un + r * VW);
      if (a.stage > 0) fetch(a.Uacc, pre_acc + r * VW);
    }
  }

  // ---- faces: one lane per (face, Gauss point)
  for (int itf = tid; itf < NFACE * MG; itf += 256) {
    const int fi = itf / MG, g = itf % MG;
    // descriptor: per side (dst + 1) | edge << 8 | cl << 10 in sFD, source slot + 128 in sFS
    const int fdw = sFD[fi], fsw = sFS[fi];
    const int fsrc[2] = {(fsw & 255) - 128, ((fsw >> 8) & 255) - 128};
    const int fcl[2] = {(fdw >> 10) & 7, (fdw >> 26) & 7};
    const int ftag = fsw >> 16;
    const double* fg = sFG + fi * 4;
    const double nxv = fg[0], nyv = (D == 2) ? fg[1] : 0.0, jf0 = fg[2], jf1 = fg[3];
    double tr[2][NF][Ms];
#pragma unroll
    for (int d = 0; d < 2; ++d) {
      const int s = fsrc[d];
#pragma unroll
      for (int j = 0; j < Ms; ++j) {
        if (s >= 0) {
          const int node = closure_node<D, P>(fcl[d], j);
#pragma unroll
          for (int f = 0; f < NF; ++f) tr[d][f][j] = sU[s * SU + f * Ns + node];
        } else {
#pragma unroll
          for (int f = 0; f < NF; ++f) tr[d][f][j] = sH[(-1 - s) * HT + f * Ms + j];
        }
      }
    }
    if (ftag == BC_REFLECTIVE) {  // boundaries.cu:20-67 on the nodal face values
#pragma unroll
      for (int j = 0; j < Ms; ++j) {
        if constexpr (D == 1) {
          tr[1][1][j] = -tr[1][1][j];
        } else {
          const double nx2 = nxv * nxv, ny2 = nyv * nyv, m2nxny = -2 * nxv * nyv;
          const double inv = 1.0 / (nx2 + ny2);
          const double vxL = tr[0][1][j], vyL = tr[0][2][j];
          tr[1][1][j] = inv * ((-nx2 + ny2) * vxL + m2nxny * vyL);
          tr[1][2][j] = inv * (m2nxny * vxL + (nx2 - ny2) * vyL);
        }
      }
    }
    double ul[NF], ur[NF], F[NF], nc[NF];
#pragma unroll
    for (int f = 0; f < NF; ++f) {
      double sl = 0.0, sr = 0.0;
#pragma unroll
      for (int j = 0; j < Ms; ++j) {
        sl += tr[0][f][j] * sPsi[g + j * MG];
        sr += tr[1][f][j] * sPsi[g + j * MG];
      }
      ul[f] = sl;
      ur[f] = sr;
    }
    riemann<D, PH, FL>(ul, ur, nxv, nyv, F, nc);
    // the non-conservative terms are zero except for the last NNC fields
    // (alpha; phinc; alpha and beta): keep F and those; sides and face
    // Jacobians at integration
    double* w = sW + (fi * MG + g) * NWP;
#pragma unroll
    for (int f = 0; f < NF; ++f) w[f] = F[f];
#pragma unroll
    for (int m = 0; m < NNC; ++m) w[NF + m] = nc[NF - NNC + m];
  }
  __syncthreads();
  // ---- face integration against psi_w into the receiving elements' slots
  for (int itf = tid; itf < NFACE * 2 * Ms; itf += 256) {
    const int fi = itf / (2 * Ms), d = (itf / Ms) % 2, j = itf % Ms;
    const int side = (sFD[fi] >> (16 * d)) & 0xffff;
    const int dst = (side & 0xff) - 1;
    if (dst < 0) continue;
    const int cl = side >> 10, edge = (side >> 8) & 3;
    const int jf = (D == 2 && cl >= 4) ? reversed_pos<P>(j) : j;
    double* q = sQ + dst * SQ + edge * NF * Ms;
    const double jfd = sFG[fi * 4 + 2 + d];
    // the side's sign: fma(-1, F, nc) is -F + nc rounded once, the same
    // bits as the sum, without computing both sums and selecting per lane
    const double sgn = d ? 1.0 : -1.0;
#pragma unroll
    for (int f = 0; f < NF; ++f) {
      double s = 0.0;
#pragma unroll
      for (int g = 0; g < MG; ++g) {
        const double* w = sW + (fi * MG + g) * NWP;
        const double ncf = f >= NF - NNC ? w[NF + f - (NF - NNC)] : 0.0;
        // q_L = (-F + nc) JF_0, q_R = (F + nc) JF_1 (physics.cu:800-804, kernels.cu:199-228)
        const double qv = __builtin_fma(sgn, w[f], ncf) * jfd;
        s += sPsiw[g + j * MG] * qv;
      }
      q[f * Ms + jf] = s;
    }
  }
  __syncthreads();

  // ---- element phases
  for (int b = 0; b < NT; b += EPB) {
    {
      const int el = b + tid / TPE, g = tid % TPE;
      if (el < NT && g < NG)
        vol_phase1<D, P, PH>(tb, g, sU + el * SU, sGeo[el * NGEO], sGeo + el * NGEO + 1,
                             sW + (el - b) * SW + g * NQ);
    }
    __syncthreads();
    {
      const int el = b + tid / TPE, i = tid % TPE;
      double rhs[NF];
      const bool act = el < NT && i < Ns;
      if (act) vol_phase2<D, P, PH>(tb, i, sW + (el - b) * SW, sQ + el * SQ, rhs);
      __syncthreads();
      if (act)
#pragma unroll
        for (int f = 0; f < NF; ++f) sU[el * SU + f * Ns + i] = rhs[f];
    }
    __syncthreads();
  }

  // ---- stage output (coalesced along the tile rows)
#pragma unroll
  for (int r = 0; r < R_U; ++r) {
    const int k = VW * (tid + r * 256);
    if (k >= NT * NU) break;
    if (!in_grid(k)) continue;
    const size_t gi = gidx(k);
    const int el = k / NU;
    double ov[VW], av[VW];
#pragma unroll
    for (int v = 0; v < VW; ++v) {
      const int rr = k % NU + v;
      if constexpr (MODE == 0) {
        ov[v] = sU[el * SU + rr];
      } else {
        // shared Minv: Minv_e = Minv_0 * J_0 / J_e (affine elements); else per element
        const double dte = sDte[el];
        const double* M = shared_minv ? tb.minv : a.Minv + ((size_t)(ey0 + el / TX) * a.nx + ex0 + el % TX) * Ns * Ns;
        const int f = rr / Ns, i = rr % Ns;
        const double* R = sU + el * SU + f * Ns;
        double sol = 0.0;
#pragma unroll
        for (int ii = 0; ii < Ns; ++ii) sol += M[ii * Ns + i] * R[ii];
        rk_values(a.stage, dte * sol, pre_un[r * VW + v], pre_acc[r * VW + v], av[v], ov[v]);
      }
    }
    double* out = (MODE == 0 ? a.fout : a.Uout) + gi;
    if constexpr (VEC) {
      *reinterpret_cast<double2*>(out) = make_double2(ov[0], ov[1]);
      if (MODE == 1 && a.stage < 3) *reinterpret_cast<double2*>(a.Uacc + gi) = make_double2(av[0], av[1]);
    } else {
      out[0] = ov[0];
      if (MODE == 1 && a.stage < 3) a.Uacc[gi] = av[0];
    }
  }
}

// Where the lane of node c of a 2D element (order P) takes its face sums
// from: the at most two edges whose closure holds the node, and its place
// there (closure_node), or -1.
template <int P>
__device__ inline void node_edges(int c, int* edge, int* pos) {
  edge[0] = edge[1] = -1;
  pos[0] = pos[1] = 0;
  if (c < 0) return;
  if (c < 4) {  // corner c: first node of edge c, second of the edge before it
    edge[0] = c;
    edge[1] = (c + 3) & 3;
    pos[1] = 1;
  } else if (c < 4 * P) {
    edge[0] = (c - 4) / (P - 1);
    pos[0] = 2 + (c - 4) % (P - 1);
  }
}

// The tile kernel for 2D orders 2 and 3, 8 x 4 elements, element phases on the
// matrix cores (vol_mfma_wave).  Phases: the tile's state, halo traces and
// geometry into LDS; face fluxes at the Gauss points, one lane each; element
// phases by wave, whose face sums take the fluxes of an element's four faces
// straight from there; the RK4 combination.  Two block barriers between the
// loads and the output.
//
// Bound by HBM and by how much of a block's serial chain the other blocks of
// its CU hide.  1024x512 two-fluid, p = 2: 214 us a launch (755 MB of states,
// 901 MB measured: 4.2 TB/s of the 4.9 a copy reaches) against 309 us of the
// kernel before it, which summed the faces into per-element edges behind a
// barrier of its own, kept the reference tables in LDS (50.8 KB, three blocks
// a CU; now 30.5 KB and four) and ran 28 16x16x4 products and the fields after
// E on the vector units; 512x512 single fluid 88 against 121 us; 512x256
// stiffened 79 against 147 us and p = 3 two-fluid 138 against 489 us, both
// element phases on the vector units before.  On the way: the RK operands
// fetched before the face phase, and copied where a stage needs only one,
// made every wave wait for them there (3.6k of its 36k cycles), the operands
// of the matrix products read from global memory behind them 4.7k.
//
// PREC: 0 FP64, 1 FP32 and 2 split-BF16 contractions of rho, momenta and E
// (p = 2).  VEC: the tile state, the RK operands and the stage output move as
// 16-byte pairs (every state pointer and row start is 16-byte aligned and,
// with RAG, every row of a tile a whole number of pairs, which the host checks
// before it picks this instance).  RAG: the grid's sides need not be whole
// tiles; the tile's elements past its ends hold values of its first element, in
// its order or, where pairs of an odd number of values an element keep it out,
// shifted (not a state then, so anything may come of them).  They are not
// stored, and nothing of the grid's own elements depends on them: a face past
// the ends contributes nowhere and a row of a matrix product is one element's.
// Waves per SIMD the registers must allow.  Measured, us a step without
// limiter: p = 2 single fluid 512x512 353 with 4 and 5, 473 with 6 (spills);
// two-fluid 1024x512 849 with 3 and 4, 917 with 5; stiffened 512x256 315 with 3
// and 4, 323 with 2; p = 3 single fluid 256x256 202-206 with 2 to 4, two-fluid
// 512x256 554 with 2, 562 with 3.
constexpr int stage_waves(int P, int PH) { return P == 2 ? (PH <= 1 ? 4 : 3) : (PH == 0 ? 3 : (PH == 1 ? 2 : 1)); }

template <int P, int PH, int FL, int MODE, int PREC, bool VEC, bool RAG>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(stage_waves(P, PH)))) void k_stage_mfma(StageArgs a) {
  if (a.gate && *a.gate) return;
  constexpr int D = 2, TX = 8, TY = 4;
  using V = Vol<D, P, PH>;
  using T = Tile<D, TX, TY>;
  using TW = typename std::conditional<PREC >= 1, float, double>::type;
  constexpr int NF = V::NF, Ns = V::Ns, Ms = V::Ms, MG = Shape<D, P>::MG, NU = V::NU, NNC = V::NNC;
  constexpr int NT = T::NT, NFACE = T::NFACE, NFX = T::NFX, NH = T::NH, HT = NF * Ms;
  constexpr int SU = lds_stride(NU);
  constexpr int NWP = NF + NNC;  // per face point: F, and the non-conservative terms
  // P = 2 in FP64: 4x4 products in registers (vol_tensor_wave); else 16x16 ones (vol_mfma_wave)
  constexpr bool TENSOR = P == 2 && PREC == 0;
  constexpr int NXT = TENSOR ? 0 : 4 * vol_wave_extra<P, PH>(), NZ = NH * HT > NXT ? NH * HT : NXT;
  constexpr int VW = VEC ? 2 : 1;
  static_assert(!VEC || ((TX * NU) % 2 == 0 && (SU == NU || (NU % 2 == 0 && SU % 2 == 0))), "paired state rows");
  constexpr int R_U = (NT * NU / VW + 255) / 256, R_H = (HT + 7) / 8;

  __shared__ __align__(16) double sU[NT * SU + NZ];  // the tile's state; then the halo traces, later the extra rows
  __shared__ __align__(16) double sW[NFACE * MG * NWP];  // face-point fluxes
  // TENSOR: the 1D tables; else the reference tables until every wave has taken
  // its operands, then the element phases' flux rows
  constexpr int LDD = VolOps<TW, P, PH>::LDD, LDP = VolOps<TW, P, PH>::LDP, NG = V::NG;
  constexpr int O_DW = V::NTAB_PHI, O_MINV = O_DW + Ns * LDD, O_DPHI = O_MINV + Ns * Ns,
                O_PW = O_DPHI + (NNC ? V::NTAB_D : 0), NTAB = O_PW + (NNC ? Ns * LDP : 0);
  constexpr int NFLUX = 4 * vol_wave_flux<TW, P>(), NFT = NTAB > NFLUX ? NTAB : NFLUX;
  __shared__ double sFlux[TENSOR ? kTensorTables * 16 : NFT];
  __shared__ double sPsi[MG * Ms], sPsiw[MG * Ms];
  __shared__ double sGeo[NT * 4];     // per element: J * invJac
  __shared__ double sDte[NT];         // per element: Dt (J_0/J_e with the shared Minv)
  __shared__ __align__(16) double sFG[NFACE * 4];   // per tile face: n_x, n_y, JF side 0, JF side 1
  // per tile face and side: where its trace starts in sU (12 bits), its nodes'
  // offsets there (4 bits each), the face's boundary tag
  __shared__ unsigned sFS[2 * NFACE];
  static_assert(NT * SU + NH * HT < 4096, "trace starts fit 12 bits");
  double* sH = sU + NT * SU;

  const int tid = threadIdx.x, tile = tile_of(a);
  if (tile < 0) return;
  const bool shared_minv = a.minv_stride == 0;
  const double dt = (MODE == 1) ? a.dt[0] : 0.0;
  const int ex0 = (tile % a.tiles_x) * TX, ey0 = (tile / a.tiles_x) * TY;
  // tile entry k: its offset from the tile's first entry in a state, whether
  // the grid holds it (its row's end is a whole number of elements), and its
  // place in LDS
  const size_t tile0 = ((size_t)ey0 * a.nx + ex0) * NU;
  const unsigned row = (unsigned)a.nx * NU;
  auto offset = [&](int k) -> unsigned {
    const int ty = k / (TX * NU);
    return ty * row + (k - ty * TX * NU);
  };
  auto in_grid = [&](int k) {
    const int ty = k / (TX * NU);
    return !RAG || (ey0 + ty < a.ny && k - ty * TX * NU < (a.nx - ex0) * NU);
  };
  auto lds_at = [&](int k) { return SU == NU ? k : (k / NU) * SU + k % NU; };

  // ---- every load of the tile in flight at once: the state, consecutive; the
  // halo traces, 24 slots of 32 lanes, eight entries at a time; per face (the
  // first lanes) and per element (one wave's) the geometry
  double pu[R_U * VW], ph[R_H];
  unsigned off[R_U];
#pragma unroll
  for (int r = 0; r < R_U; ++r) {
    const int k = VW * (tid + r * 256);
    off[r] = offset(k);
    if (k < NT * NU) {
      unsigned o = off[r];
      if constexpr (RAG) {  // an aligned pair of the first element (k is even)
        if (!in_grid(k)) o = VEC && NU % 2 ? k % (NU - 1) : k % NU;
      }
      const double* src = a.Uin + tile0 + o;
      if constexpr (VEC) {
        const double2 v = *reinterpret_cast<const double2*>(src);
        pu[2 * r] = v.x;
        pu[2 * r + 1] = v.y;
      } else {
        pu[r] = *src;
      }
    }
  }
  const int hs = tid & 31, hq = tid >> 5;
  int hcl = 0;
  const int he = hs < NH ? halo_source<D, TX, TY, RAG>(hs, ex0, ey0, a, hcl) : -1;
  unsigned hnodes = 0;
#pragma unroll
  for (int j = 0; j < Ms; ++j) hnodes |= (unsigned)closure_node<D, P>(hcl, j) << (4 * j);
  if (he >= 0) {
    const double* src = a.Uin + (size_t)he * NU;
#pragma unroll
    for (int r = 0; r < R_H; ++r) {
      const int q = min(hq + 8 * r, HT - 1), f = q / Ms, j = q - f * Ms;
      ph[r] = src[f * Ns + ((hnodes >> (4 * j)) & 15)];
    }
  }
  double2 pf0, pf1;
  double pj = 1.0;
  if (tid < NFACE) {
    const int fj = tid - NFX;
    int x, y;
    if (tid < NFX) {
      x = tid % (TX + 1), y = tid / (TX + 1);
      if constexpr (RAG) y = min(y, a.ny - 1 - ey0), x = min(x, a.nx - ex0);
    } else {
      x = fj % TX, y = fj / TX;
      if constexpr (RAG) y = min(y, a.ny - ey0), x = min(x, a.nx - 1 - ex0);
    }
    const double* src = tid < NFX ? a.gx + ((size_t)(ey0 + y) * (a.nx + 1) + ex0 + x) * 4
                                  : a.gy + ((size_t)(ey0 + y) * a.nx + ex0 + x) * 4;
    pf0 = reinterpret_cast<const double2*>(src)[0];
    pf1 = reinterpret_cast<const double2*>(src)[1];
  } else if (tid >= 128 && tid < 128 + NT) {
    const int el = tid - 128;
    const int ty = RAG ? min(el / TX, a.ny - 1 - ey0) : el / TX, tx = RAG ? min(el % TX, a.nx - 1 - ex0) : el % TX;
    const int eg = ((ey0 + ty) * a.nx + ex0 + tx) * a.geo_stride;
    pj = a.J[eg];
    pf0 = reinterpret_cast<const double2*>(a.invJac + (size_t)eg * 4)[0];
    pf1 = reinterpret_cast<const double2*>(a.invJac + (size_t)eg * 4)[1];
  }
  static_assert(NFACE <= 128 && NT <= 32, "one lane per face, one wave for the elements");
  constexpr int R_T = (V::NTAB_PHI + 255) / 256, R_D = (V::NTAB_D + 255) / 256;
  double tphi[R_T], tdw[R_D], tminv = 0.0, tdphi[R_D], tpw[R_T], tpsi, tpsiw, tten = 0.0;
  if constexpr (TENSOR) {
    tten = a.tensor[min(tid, kTensorTables * 16 - 1)];
  } else {
#pragma unroll
  for (int r = 0; r < R_D; ++r) {
    const int k = min(tid + r * 256, V::NTAB_D - 1);
    tdw[r] = a.dphi_w[k];
    if constexpr (NNC > 0) tdphi[r] = a.dphi[k];
  }
#pragma unroll
  for (int r = 0; r < R_T; ++r) {
    const int k = min(tid + r * 256, V::NTAB_PHI - 1);
    tphi[r] = a.phi[k];
    if constexpr (NNC > 0) tpw[r] = a.phi_w[k];
  }
  static_assert(Ns * Ns <= 256, "one round");
  if (MODE == 1 && shared_minv) tminv = a.Minv[min(tid, Ns * Ns - 1)];
  }
  tpsi = a.psi[min(tid, MG * Ms - 1)];
  tpsiw = a.psi_w[min(tid, MG * Ms - 1)];
  // where each side of every tile face reads its trace, one lane per face
  if (tid < NFACE) {
    const FaceDesc fd = face_desc<D, TX, TY, RAG>(tid, ex0, ey0, a);
#pragma unroll
    for (int d = 0; d < 2; ++d) {
      const int s = fd.src[d];
      unsigned w = s >= 0 ? s * SU : NT * SU + (-1 - s) * HT;
#pragma unroll
      for (int j = 0; j < Ms; ++j) w |= (unsigned)(s >= 0 ? closure_node<D, P>(fd.cl[d], j) : j) << (12 + 4 * j);
      sFS[2 * tid + d] = w | (unsigned)(fd.tag == BC_REFLECTIVE) << 31;
    }
  }
  static_assert(12 + 4 * Ms <= 31, "a side's word");
#pragma unroll
  for (int r = 0; r < R_U; ++r) {
    const int k = VW * (tid + r * 256);
    if (k < NT * NU) {
      if constexpr (VEC)
        *reinterpret_cast<double2*>(sU + lds_at(k)) = make_double2(pu[2 * r], pu[2 * r + 1]);
      else
        sU[lds_at(k)] = pu[r];
    }
  }
  if (he >= 0)
#pragma unroll
    for (int r = 0; r < R_H; ++r)
      if (HT % 8 == 0 || hq + 8 * r < HT) sH[hs * HT + hq + 8 * r] = ph[r];
  if (tid < NFACE) {
    reinterpret_cast<double2*>(sFG)[2 * tid] = pf0;
    reinterpret_cast<double2*>(sFG)[2 * tid + 1] = pf1;
  } else if (tid >= 128 && tid < 128 + NT) {
    double* g = sGeo + (tid - 128) * 4;
    g[0] = pf0.x * pj;
    g[1] = pf0.y * pj;
    g[2] = pf1.x * pj;
    g[3] = pf1.y * pj;
    if (MODE == 1) sDte[tid - 128] = shared_minv ? (TENSOR ? dt / pj : dt * (a.J0 / pj)) : dt;
  }
  if constexpr (TENSOR) {
    if (tid < kTensorTables * 16) sFlux[tid] = tten;
  } else {
#pragma unroll
  for (int r = 0; r < R_D; ++r)
    if (tid + r * 256 < V::NTAB_D) {
      const int k = tid + r * 256;
      sFlux[O_DW + k / (2 * NG) * LDD + k % (2 * NG)] = tdw[r];
      if constexpr (NNC > 0) sFlux[O_DPHI + tid + r * 256] = tdphi[r];
    }
#pragma unroll
  for (int r = 0; r < R_T; ++r)
    if (tid + r * 256 < V::NTAB_PHI) {
      sFlux[tid + r * 256] = tphi[r];
      const int k = tid + r * 256;
      if constexpr (NNC > 0) sFlux[O_PW + k / NG * LDP + k % NG] = tpw[r];
    }
  if (tid < Ns * Ns) sFlux[O_MINV + tid] = tminv;
  }
  if (tid < MG * Ms) {
    sPsi[tid] = tpsi;
    sPsiw[tid] = tpsiw;
  }
  __syncthreads();
  // ---- faces: one lane per (face, Gauss point)
  for (int itf = tid; itf < NFACE * MG; itf += 256) {
    const int fi = itf / MG, g = itf % MG;
    double u[2][NF], tr0[Ms];
    const double nxv = sFG[4 * fi], nyv = sFG[4 * fi + 1];
    double psi[Ms];
#pragma unroll
    for (int j = 0; j < Ms; ++j) psi[j] = sPsi[g + j * MG];
    bool wall = false;
#pragma unroll
    for (int d = 0; d < 2; ++d) {
      const unsigned w = sFS[2 * fi + d];
      const int base = w & 4095, fs = base >= NT * SU ? Ms : Ns;
      wall = w >> 31;
      const double* t[Ms];
#pragma unroll
      for (int j = 0; j < Ms; ++j) t[j] = sU + base + ((w >> (12 + 4 * j)) & 15);
#pragma unroll
      for (int f = 0; f < NF; ++f) {
        double s = 0.0;
#pragma unroll
        for (int j = 0; j < Ms; ++j) s += t[j][f * fs] * psi[j];
        u[d][f] = s;
      }
    }
    if (wall) {  // boundaries.cu:20-67 (the reflection is linear: applied at the point instead of at the nodes)
      const double nx2 = nxv * nxv, ny2 = nyv * nyv, m2nxny = -2 * nxv * nyv;
      const double inv = 1.0 / (nx2 + ny2);
      const double vxL = u[0][1], vyL = u[0][2];
      u[1][1] = inv * ((-nx2 + ny2) * vxL + m2nxny * vyL);
      u[1][2] = inv * (m2nxny * vxL + (nx2 - ny2) * vyL);
    }
    double F[NF], nc[NF];
    riemann<D, PH, FL>(u[0], u[1], nxv, nyv, F, nc);
    // the non-conservative terms are zero except for the last NNC fields
    double* w = sW + (fi * MG + g) * NWP;
#pragma unroll
    for (int f = 0; f < NF; ++f) w[f] = F[f];
#pragma unroll
    for (int m = 0; m < NNC; ++m) w[NF + m] = nc[NF - NNC + m];
  }
  // RK operands of this thread's output entries, in flight during the element
  // phases: base + beta*du is the stage output, acc + gamma*du the accumulator
  // (rk_values; stage 0 starts the accumulator from U^n, stage 3 puts out the
  // accumulator: one operand)
  double pre_base[R_U * VW], pre_acc[R_U * VW];
  const bool two = a.stage == 1 || a.stage == 2;
  if constexpr (MODE == 1) {
    auto fetch = [&](const double* from, double* to) {
#pragma unroll
      for (int r = 0; r < R_U; ++r) {
        const int k = VW * (tid + r * 256);
        if (k < NT * NU && in_grid(k)) {
          if constexpr (VEC) {
            const double2 v = *reinterpret_cast<const double2*>(from + tile0 + off[r]);
            to[2 * r] = v.x;
            to[2 * r + 1] = v.y;
          } else {
            to[r] = from[tile0 + off[r]];
          }
        }
      }
    };
    fetch(a.stage < 3 ? a.Un : a.Uacc, pre_base);
    if (two) fetch(a.Uacc, pre_acc);
  }
  VolOps<TW, P, PH> op;
  if constexpr (!TENSOR) op.load(sFlux, sFlux + O_DPHI, sFlux + O_PW, sFlux + O_DW, sFlux + O_MINV, tid);
  int edge[2], pos[2];
  node_edges<P>(TENSOR ? tensor_node(tid & 63) : tid & 15, edge, pos);
  __syncthreads();

  // ---- element phases, with the face terms of node c of element el: the
  // fluxes of at most two faces against psi_w.  The element is side 0 (the
  // flux leaves, -F + nc) of its right and upper faces and of the domain's
  // left and lower ones, else side 1 (F + nc), whose points run backwards
  // (physics.cu:800-804, kernels.cu:199-228).
  auto face = [&](int el, double* qs) {
#pragma unroll
    for (int f = 0; f < NF; ++f) qs[f] = 0.0;
    const int tx = el % TX, ty = el / TX;
#pragma unroll
    for (int n = 0; n < 2; ++n) {
      const int k = edge[n];
      if (k < 0) continue;
      const int fi = (k & 1) ? ty * (TX + 1) + tx + (k == 1) : NFX + (ty + (k == 2)) * TX + tx;
      const bool side0 = k == 1 || k == 2 || (k == 3 ? ex0 + tx == 0 : ey0 + ty == 0);
      const int j = side0 ? pos[n] : reversed_pos<P>(pos[n]);
      const double jf = sFG[4 * fi + (side0 ? 2 : 3)];
      const double* w = sW + fi * MG * NWP;
#pragma unroll
      for (int g = 0; g < MG; ++g) {
        const double wt = sPsiw[g + j * MG] * jf, ws = side0 ? -wt : wt;
#pragma unroll
        for (int f = 0; f < NF; ++f) qs[f] = __builtin_fma(ws, w[g * NWP + f], qs[f]);
#pragma unroll
        for (int m = 0; m < NNC; ++m) qs[NF - NNC + m] = __builtin_fma(wt, w[g * NWP + NF + m], qs[NF - NNC + m]);
      }
    }
  };
  if constexpr (TENSOR)
    vol_tensor_wave<PH, SU>(sFlux, sU, sGeo, tid, MODE == 1 && shared_minv, sDte, face);
  else
    vol_mfma_wave<TW, P, PH, SU, TW, PREC == 2>(op, a.phi, a.dphi_w, sU, sGeo, sFlux, sH, tid,
                                                MODE == 1 && shared_minv, sDte, face);
  __syncthreads();

  // ---- stage output (coalesced along the tile rows, VW entries per step)
  const double gk = MODE == 1 ? kRkGamma[a.stage] : 0.0;
  const double bk = MODE == 1 ? (a.stage < 3 ? kRkBeta[a.stage + 1] : gk) : 0.0;
#pragma unroll
  for (int r = 0; r < R_U; ++r) {
    const int k0 = VW * (tid + r * 256);
    if (k0 >= NT * NU) break;
    if (!in_grid(k0)) continue;
    double ov[VW], av[VW];
#pragma unroll
    for (int v = 0; v < VW; ++v) {
      const int at = lds_at(k0) + v;
      if constexpr (MODE == 0) {
        ov[v] = sU[at];
      } else {
        double du;
        if (shared_minv) {
          du = sU[at];
        } else {  // one Minv per element
          const int el = (k0 + v) / NU, rr = (k0 + v) % NU, f = rr / Ns, i = rr % Ns;
          const double* M = a.Minv + ((size_t)(ey0 + el / TX) * a.nx + ex0 + el % TX) * Ns * Ns;
          const double* R = sU + el * SU + f * Ns;
          double sol = 0.0;
#pragma unroll
          for (int ii = 0; ii < Ns; ++ii) sol += M[ii * Ns + i] * R[ii];
          du = sDte[el] * sol;
        }
        av[v] = (two ? pre_acc[r * VW + v] : pre_base[r * VW + v]) + gk * du;
        ov[v] = pre_base[r * VW + v] + bk * du;
        // this thread's own entry: kept for the cell means and averages below
        if (PH > 0 && shared_minv && a.uavg) sU[at] = ov[v];
        if (P == 2 && PH == 1 && shared_minv && a.means) sU[at] = ov[v];
      }
    }
    double* out = (MODE == 0 ? a.fout : a.Uout) + tile0 + off[r];
    double* acc = a.Uacc + tile0 + off[r];
    if constexpr (VEC) {
      *reinterpret_cast<double2*>(out) = make_double2(ov[0], ov[1]);
      if (MODE == 1 && a.stage < 3) *reinterpret_cast<double2*>(acc) = make_double2(av[0], av[1]);
    } else {
      out[0] = ov[0];
      if (MODE == 1 && a.stage < 3) acc[0] = av[0];
    }
  }
  if constexpr (MODE == 1 && P == 2 && PH == 1) {
    if (a.means && shared_minv) {
      // cell means (cell_means_rpa) and sensor averages (sensor_averages_2d)
      // of the output tile: one lane per (element, field) forms the field's
      // two means, then one lane per element the derived values (the same
      // functions and order as the one-lane forms, so the same bits)
      static_assert(NFACE * MG * NWP >= 2 * NT * NF, "means staging fits the flux buffer");
      __syncthreads();  // the output tile is in sU, sW is free
      double* sM = sW;            // [el*NF + f] mode-0 means
      double* sA = sW + NT * NF;  // [el*NF + f] sensor nodal means
      for (int k = tid; k < NT * NF; k += 256) {
        const int el = k / NF, f = k % NF;
        if (!in_grid(el * NU)) continue;
        const double* uf = sU + el * SU + f * Ns;
        sM[k] = cell_mode0(uf, a.w0);
        if (a.uavg) {
          const double v = sensor_nodal_mean<Ns>(uf);
          sA[k] = v;
          a.uavg[((size_t)(ey0 + el / TX) * a.nx + ex0 + el % TX) * NF + f] = v;
        }
      }
      __syncthreads();
      if (tid < NT && in_grid(tid * NU)) {
        double a3[3];
        rpa_of_means(sM + tid * NF, a3);
        const size_t eg = (size_t)(ey0 + tid / TX) * a.nx + ex0 + tid % TX;
        double* m = a.means + eg * 3;
        m[0] = a3[0];
        m[1] = a3[1];
        m[2] = a3[2];
        if (a.uavg) a.psens[eg] = sensor_cell<2, 1>(sA + tid * NF, 0).p;
      }
      return;
    }
  }
  if constexpr (MODE == 1 && PH > 0) {
    if (a.uavg && shared_minv) {  // the sensor's averages alone, one lane per (element, field)
      __syncthreads();  // the output tile is in sU
      for (int k = tid; k < NT * NF; k += 256) {
        const int el = k / NF, f = k % NF;
        if (in_grid(el * NU))
          a.uavg[((size_t)(ey0 + el / TX) * a.nx + ex0 + el % TX) * NF + f] = sensor_nodal_mean<Ns>(sU + el * SU + f * Ns);
      }
    }
  }
}

// ------------------------------------------------------------------- host
template <int D>
struct TileShape;
// 1D: 128 elements per tile, or 8 where 128 does not divide the mesh
template <>
struct TileShape<1> { static constexpr int TX = 128, TX_SMALL = 8, TY = 1; };
template <>
struct TileShape<2> { static constexpr int TX = 8, TY = 4; };

// fn(dim, order, flux) with all three as integral constants
template <typename Fn>
static hipError_t dispatch_stage(const dgx_config& c, Fn&& fn) {
  using I0 = std::integral_constant<int, 0>;
  using I1 = std::integral_constant<int, 1>;
  using I2 = std::integral_constant<int, 2>;
  using I3 = std::integral_constant<int, 3>;
  auto by_flux = [&](auto d, auto p) -> hipError_t { return c.flux == 0 ? fn(d, p, I0{}) : fn(d, p, I1{}); };
  auto by_order = [&](auto d) -> hipError_t {
    switch (c.order) {
      case 1: return by_flux(d, I1{});
      case 2: return by_flux(d, I2{});
      default: return by_flux(d, I3{});
    }
  };
  return c.dim == 1 ? by_order(I1{}) : by_order(I2{});
}

// The stage launch of one physics; each is instantiated in a source of its own
// (launch_stage in stage.hip picks).
template <int PH>
hipError_t launch_stage_phys(const Solver& s, int mode, int stage, const double* Uin, const double* Un, double* Uacc,
                             double* Uout, const double* dt_dev, double* f_out, hipStream_t st, double* means,
                             double* uavg, double* psens, bool* means_done) {
  if (means_done) *means_done = false;
  const Cart& c = s.cart;
  StageArgs a{};
  a.phi = s.t.phi; a.dphi = s.t.dphi; a.phi_w = s.t.phi_w; a.dphi_w = s.t.dphi_w;
  a.psi = s.t.psi; a.psi_w = s.t.psi_w; a.Minv = s.t.Minv;
  a.J = s.t.J; a.invJac = s.t.invJac; a.gx = s.t.face_geo_x; a.gy = s.t.face_geo_y;
  a.J0 = s.t.J0; a.geo_stride = s.t.geo_stride; a.minv_stride = s.t.minv_stride;
  a.nx = c.nx; a.ny = c.ny;
  for (int k = 0; k < 4; ++k) a.bc[k] = c.bc[k];
  a.tiles_x = (c.nx + c.tx - 1) / c.tx;
  a.tiles_y = (c.ny + c.ty - 1) / c.ty;
  const bool ragged = !c.on;
  const int ntiles = a.tiles_x * a.tiles_y;
  a.stage = stage; a.Uin = Uin; a.Un = Un; a.Uacc = Uacc; a.Uout = Uout; a.dt = dt_dev; a.fout = f_out;
  a.gate = s.gate;
  a.tensor = s.t.tensor;
  a.w0 = s.t.mlp_vinv;  // first row: the mode-0 weights
  return dispatch_stage(s.cfg, [&](auto d, auto p, auto fl) -> hipError_t {
    constexpr int D = decltype(d)::value;
    constexpr int P = decltype(p)::value, FL = decltype(fl)::value;
    const dim3 grid(8 * ((ntiles + 7) / 8)), block(256);  // whole bands (tile_of)
    auto run = [&](auto kern) {
      hipLaunchKernelGGL(kern, grid, block, 0, st, a);
      return hipGetLastError();
    };
    // 16-byte pairs when every state pointer and row allows them: rows start
    // (and, ragged, end) on pairs when an element is a whole number of them
    // or the grid has an even number of columns
    auto al = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; };
    [[maybe_unused]] const bool vec = (Vol<D, P, PH>::NU % 2 == 0 || c.nx % 2 == 0) && al(Uin) &&
                                      (mode == 0 ? al(f_out) : al(Un) && al(Uacc) && al(Uout));
    if constexpr (D == 2 && P >= 2) {
      if constexpr (P == 2 && PH == 1) {
        // the epilogue's cell means: RK stages with the shared Minv
        if (mode == 1 && means && s.t.mlp_vinv && s.t.minv_stride == 0) {
          a.means = means;
          a.uavg = uavg;
          a.psens = psens;
          if (means_done) *means_done = true;
        }
      }
      // the epilogue's sensor averages alone.  Measured, 1024x512 p = 2
      // two-fluid: a pass over the state for them takes 34 us, the epilogue 7
      if (PH > 0 && mode == 1 && !means && uavg && s.t.minv_stride == 0) {
        a.uavg = uavg;
        if (means_done) *means_done = true;
      }
      if constexpr (P == 2 && PH <= 1) {
        if (s.precision == 1)
          return mode == 0 ? (vec ? run(k_stage_mfma<P, PH, FL, 0, 1, true, false>) : run(k_stage_mfma<P, PH, FL, 0, 1, false, false>))
                           : (vec ? run(k_stage_mfma<P, PH, FL, 1, 1, true, false>) : run(k_stage_mfma<P, PH, FL, 1, 1, false, false>));
        if (s.precision == 2)
          return mode == 0 ? (vec ? run(k_stage_mfma<P, PH, FL, 0, 2, true, false>) : run(k_stage_mfma<P, PH, FL, 0, 2, false, false>))
                           : (vec ? run(k_stage_mfma<P, PH, FL, 1, 2, true, false>) : run(k_stage_mfma<P, PH, FL, 1, 2, false, false>));
      }
      // states that cannot be paired (rare) take the ragged instance on whole tiles too
      if (!vec) return mode == 0 ? run(k_stage_mfma<P, PH, FL, 0, 0, false, true>) : run(k_stage_mfma<P, PH, FL, 1, 0, false, true>);
      if (ragged) return mode == 0 ? run(k_stage_mfma<P, PH, FL, 0, 0, true, true>) : run(k_stage_mfma<P, PH, FL, 1, 0, true, true>);
      return mode == 0 ? run(k_stage_mfma<P, PH, FL, 0, 0, true, false>) : run(k_stage_mfma<P, PH, FL, 1, 0, true, false>);
    } else {
      auto go = [&](auto txc) -> hipError_t {
        constexpr int TX = decltype(txc)::value, TY = TileShape<D>::TY;
        if constexpr (D == 2) {
          if (!vec) return mode == 0 ? run(k_stage<D, P, PH, FL, 0, TX, TY, false, true>) : run(k_stage<D, P, PH, FL, 1, TX, TY, false, true>);
          if (ragged) return mode == 0 ? run(k_stage<D, P, PH, FL, 0, TX, TY, true, true>) : run(k_stage<D, P, PH, FL, 1, TX, TY, true, true>);
          return mode == 0 ? run(k_stage<D, P, PH, FL, 0, TX, TY, true, false>) : run(k_stage<D, P, PH, FL, 1, TX, TY, true, false>);
        } else {
          if (ragged) return hipErrorInvalidValue;  // 1D: the whole-step or the face + element kernels
          return mode == 0 ? run(k_stage<D, P, PH, FL, 0, TX, TY, false, false>) : run(k_stage<D, P, PH, FL, 1, TX, TY, false, false>);
        }
      };
      if constexpr (D == 1) {
        if (c.tx == TileShape<1>::TX_SMALL) return go(std::integral_constant<int, TileShape<1>::TX_SMALL>{});
      }
      return go(std::integral_constant<int, TileShape<D>::TX>{});
    }
  });
}
#define DGX_STAGE_PHYS(PH)                                                                                        \
  template hipError_t launch_stage_phys<PH>(const Solver&, int, int, const double*, const double*, double*, double*, \
                                            const double*, double*, hipStream_t, double*, double*, double*, bool*);

}  // namespace dgx

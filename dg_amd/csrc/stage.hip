// Tile kernel (stage.cuh): the launch's choice of physics, and the
// single-fluid instances.  The others are in stage_multifluid.hip and
// stage_passive_stiffened.hip, so that the four compile side by side.
#include "stage.cuh"

namespace dgx {

DGX_STAGE_PHYS(0)
extern template hipError_t launch_stage_phys<1>(const Solver&, int, int, const double*, const double*, double*, double*,
                                                const double*, double*, hipStream_t, double*, double*, double*, bool*);
extern template hipError_t launch_stage_phys<2>(const Solver&, int, int, const double*, const double*, double*, double*,
                                                const double*, double*, hipStream_t, double*, double*, double*, bool*);
extern template hipError_t launch_stage_phys<3>(const Solver&, int, int, const double*, const double*, double*, double*,
                                                const double*, double*, hipStream_t, double*, double*, double*, bool*);

bool stage_tiles(int D, int nx, int ny, int* tx, int* ty) {
  *tx = D == 1 ? (nx % TileShape<1>::TX == 0 ? TileShape<1>::TX : TileShape<1>::TX_SMALL) : TileShape<2>::TX;
  *ty = D == 1 ? TileShape<1>::TY : TileShape<2>::TY;
  return nx % *tx == 0 && (D == 1 || ny % *ty == 0);
}

// Each face's normal and Jacobians in grid order, from the face tables of a
// mesh whose faces cartesian_layout has found in their places: side 0 is the
// left or lower element, or the boundary element.
__global__ __launch_bounds__(256) void k_face_geometry(int D, int M_T, int nx, const int* __restrict__ face_elem,
                                                       const int* __restrict__ face_closure,
                                                       const double* __restrict__ normals,
                                                       const double* __restrict__ JF, double* __restrict__ gx,
                                                       double* __restrict__ gy) {
  const int f = blockIdx.x * 256 + threadIdx.x;
  if (f >= M_T) return;
  const int e = face_elem[2 * f], c = face_closure[2 * f], ex = e % nx, ey = e / nx;
  const bool xface = D == 1 || c == 1 || c == 3;
  double* g = xface ? gx + ((size_t)ey * (nx + 1) + ex + (c == 1 ? 1 : 0)) * 4
                    : gy + ((size_t)(ey + (c == 2 ? 1 : 0)) * nx + ex) * 4;
  g[0] = normals[(size_t)f * D];
  g[1] = D == 2 ? normals[(size_t)f * D + 1] : 0.0;
  g[2] = JF[2 * f];
  g[3] = JF[2 * f + 1];
}

hipError_t launch_face_geometry(const Solver& s, hipStream_t st) {
  hipLaunchKernelGGL(k_face_geometry, dim3((s.M_T + 255) / 256), dim3(256), 0, st, s.D, s.M_T, s.cart.nx,
                     s.t.face_elem, s.t.face_closure, s.t.normals, s.t.JF, s.t.face_geo_x, s.t.face_geo_y);
  return hipGetLastError();
}

hipError_t launch_stage(const Solver& s, int mode, int stage, const double* Uin, const double* Un, double* Uacc,
                        double* Uout, const double* dt_dev, double* f_out, hipStream_t st, double* means,
                        double* uavg, double* psens, bool* means_done) {
  auto go = [&](auto f) { return f(s, mode, stage, Uin, Un, Uacc, Uout, dt_dev, f_out, st, means, uavg, psens, means_done); };
  switch (s.cfg.physics) {
    case 0: return go(launch_stage_phys<0>);
    case 1: return go(launch_stage_phys<1>);
    case 2: return go(launch_stage_phys<2>);
    default: return go(launch_stage_phys<3>);
  }
}

}  // namespace dgx

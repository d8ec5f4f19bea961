// pipgpu_adjoint.hip -- the adjoint kernels of pip_adjoint.h and their
// launches (pip_adj_launch.h).  Compiled on its own, with the exact build's
// contraction flag (-ffp-contract=off; the VJP bodies enable contraction
// themselves) and the compiler's default instruction scheduling.
#include <hip/hip_runtime.h>

#include "pip_adj_launch.h"
#include "pip_adjoint.h"

namespace pip {

constexpr int kCUs = 256;

hipError_t adj_stage_launch(const AdjArgs& a, hipStream_t stream) {
  const dim3 cells((unsigned)((a.N + 255) / 256));
  if (a.make_V) hipLaunchKernelGGL(k_adj_cell, cells, dim3(256), 0, stream, a);
  const dim3 gf((unsigned)(adj_plasma_face_groups(a.nx, a.ny) + adj_edge_face_blocks(a.nx, a.ny)));
  hipLaunchKernelGGL(k_adj_plasma_faces, gf, dim3(ADJ_PBS), 0, stream, a);
  const int ghost = (a.istep == 1 && !a.make_V) ? adj_ghost_blocks(a.ix, a.jx) : 0;
  // One 8 x 8 tile per CU at most: gather us, split and not, 64^2 19.9 / 29.6,
  // 65x48 22.6 / 37.3, 128^2 (256 tiles) 20.6 / 26.1, 160^2 (400) 29.1 / 27.1,
  // 512^2 160 / 76.
  const int ns = GatherTile<GS, GS>::tiles(a.nx, a.ny), nt = GatherTile<GT_X, GT_Y>::tiles(a.nx, a.ny);
  if (ns <= kCUs) hipLaunchKernelGGL(k_adj_gather_split, dim3((unsigned)(ns + ghost)), dim3(GS_NT), 0, stream, a);
  else hipLaunchKernelGGL(k_adj_gather, dim3((unsigned)(nt + ghost)), dim3(256), 0, stream, a);
  return hipGetLastError();
}

hipError_t adj_seed_launch(double* lam, int nvt, int ix, int jx, long long N, const Bnd& bnd, hipStream_t stream) {
  const dim3 cells((unsigned)((N + 255) / 256));
  hipLaunchKernelGGL(k_adj_fold_seed, cells, dim3(256), 0, stream, lam, nvt, ix, jx, N, bnd);
  hipLaunchKernelGGL(k_zero_ghosts, cells, dim3(256), 0, stream, lam, nvt, ix, jx, N);
  return hipGetLastError();
}

}  // namespace pip

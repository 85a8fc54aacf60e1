// The residual chain on xy planes.
#include "chain_launch.hpp"

#ifndef RISM_T
#error "RISM_T: the working type of this translation unit"
#endif

namespace rism {

template <typename T, int N, int H>
void launch_planes_h(bool inv, dim3 grid, hipStream_t s, const SoluteDesc* sd, const GridArgs& g,
                     const cpx<T>* twh, const cpx<T>* twf) {
  if (inv)
    hipLaunchKernelGGL((c2r_xy_resid<T, N, N, H>), grid, dim3((plane_threads<T, N, N>())), 0, s, sd, g, twh, twf);
  else
    hipLaunchKernelGGL((closure_r2c_xy<T, N, N, H>), grid, dim3((plane_threads<T, N, N>())), 0, s, sd, g, twh, twf);
}
template <typename T, int N>
void launch_planes_n(bool inv, dim3 grid, hipStream_t s, const SoluteDesc* sd, const GridArgs& g,
                     const cpx<T>* twh, const cpx<T>* twf, int hist) {
  if (hist <= 8) launch_planes_h<T, N, 8>(inv, grid, s, sd, g, twh, twf);
  else if (hist <= 10) launch_planes_h<T, N, 10>(inv, grid, s, sd, g, twh, twf);
  else launch_planes_h<T, N, MAX_DIIS>(inv, grid, s, sd, g, twh, twf);
}
// Grid: x = z plane, y = site, z = solute.
template <typename T>
void launch_planes(bool inv, int B, hipStream_t s, const SoluteDesc* sd, const GridArgs& g,
                   const cpx<T>* twh, const cpx<T>* twf, int hist) {
  const dim3 grid(g.N2, g.m, B);
  switch (g.N0) {
    case 32: launch_planes_n<T, 32>(inv, grid, s, sd, g, twh, twf, hist); break;
    case 48: launch_planes_n<T, 48>(inv, grid, s, sd, g, twh, twf, hist); break;
    case 64: launch_planes_n<T, 64>(inv, grid, s, sd, g, twh, twf, hist); break;
    case 96: launch_planes_n<T, 96>(inv, grid, s, sd, g, twh, twf, hist); break;
    case 128: launch_planes_n<T, 128>(inv, grid, s, sd, g, twh, twf, hist); break;
  }
}

template void launch_planes<RISM_T>(bool, int, hipStream_t, const SoluteDesc*, const GridArgs&,
                                    const cpx<RISM_T>*, const cpx<RISM_T>*, int);

}  // namespace rism

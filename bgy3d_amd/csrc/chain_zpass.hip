// The z pass of the residual chain.
#include "chain_launch.hpp"

#ifndef RISM_T
#error "RISM_T: the working type of this translation unit"
#endif

namespace rism {

#define RISM_FOR_N(X) X(32) X(48) X(64) X(96) X(128) X(192) X(256) X(384)

template <typename T, int LINES>
void launch_zstar_l(int N2, dim3 grid, size_t lds, hipStream_t s, const SoluteDesc* sd,
                    const GridArgs& g, const cpx<T>* tw, const T* chi, const T* tau) {
  switch (N2) {
#define X(n) case n: hipLaunchKernelGGL((zstar<T, n, LINES>), grid, dim3(NT), lds, s, sd, g, tw, chi, tau); break;
    RISM_FOR_N(X)
#undef X
  }
}
template <typename T, int N2, int NTZ = NT>
void launch_zreg_n(int NX, int N1, int B, hipStream_t s, const SoluteDesc* sd, const GridArgs& g,
                   const cpx<T>* tw, const T* chi, const T* tau) {
  // NTZ threads: the same points per thread over NTZ / NT times the columns
  constexpr int L = zreg_lines<T, N2>() * (NTZ / NT);
  // In FP32 the Nyquist column kx = N0/2 gets blocks of its own (LINES rows
  // each) when the tiles of LINES columns end just before it, instead of a
  // tile that holds it alone (one workgroup in five at N0 = 128): 1.19 ->
  // 1.08 ms per pass at 64 x 128^3.  In FP64 in rows, and in the y passes,
  // that cost more than the tile it replaced.  RISM3D_NYQ=0 keeps it in the
  // last tile (g.nyq).  Y-major spectra (g.ylay) always have it apart.
  const bool split = g.ylay || (g.nyq && sizeof(T) == 4 && NX > 1 && (NX - 1) % L == 0);
  const int tiles = (split ? NX - 1 + L - 1 : NX + L - 1) / L;
  GridArgs gz = g;
  if (gz.zorder == 2 && (tiles * N1) % 8 != 0) gz.zorder = 1;  // whole tiles per XCD
  if (gz.zorder == 3 && N1 % 16 != 0) gz.zorder = 1;            // whole row pairs per XCD
  gz.zB = B;
  gz.ztiles = tiles;
  gz.nyqb = split ? (N1 + L - 1) / L : 0;
  const dim3 grid(((size_t)tiles * N1 + gz.nyqb) * B);
  if constexpr (sizeof(T) == 8 && NTZ == NT) {
    if (g.special == 1) {
      if (g.msol == 1)
        hipLaunchKernelGGL((zstar_reg<T, N2, L, 1, NTZ, 1>), grid, dim3(NTZ), 0, s, sd, gz, tw, chi, tau);
      else if (g.msol == 2)
        hipLaunchKernelGGL((zstar_reg<T, N2, L, 3, NTZ, 2>), grid, dim3(NTZ), 0, s, sd, gz, tw, chi, tau);
      else
        hipLaunchKernelGGL((zstar_reg<T, N2, L, 6, NTZ, 3>), grid, dim3(NTZ), 0, s, sd, gz, tw, chi, tau);
      return;
    }
  }
  if (g.m == 3) {
    hipLaunchKernelGGL((zstar_reg<T, N2, L, 3, NTZ>), grid, dim3(NTZ), 0, s, sd, gz, tw, chi, tau);
  } else {
    hipLaunchKernelGGL((zstar_reg<T, N2, L, 5, NTZ>), grid, dim3(NTZ), 0, s, sd, gz, tw, chi, tau);
  }
}
template <typename T>
void launch_zstar(int N2, int NX, int N1, int B, hipStream_t s, const SoluteDesc* sd,
                  const GridArgs& g, const cpx<T>* tw, const T* chi, const T* tau) {
  if (use_zreg(g)) {
    if constexpr (sizeof(T) == 4) {
      if (g.zwide && N2 <= 128) {  // 512 threads over 32 kx columns
        switch (N2) {
          case 32: launch_zreg_n<T, 32, 2 * NT>(NX, N1, B, s, sd, g, tw, chi, tau); break;
          case 48: launch_zreg_n<T, 48, 2 * NT>(NX, N1, B, s, sd, g, tw, chi, tau); break;
          case 64: launch_zreg_n<T, 64, 2 * NT>(NX, N1, B, s, sd, g, tw, chi, tau); break;
          case 96: launch_zreg_n<T, 96, 2 * NT>(NX, N1, B, s, sd, g, tw, chi, tau); break;
          case 128: launch_zreg_n<T, 128, 2 * NT>(NX, N1, B, s, sd, g, tw, chi, tau); break;
        }
        return;
      }
    }
    switch (N2) {
#define X(n) case n: launch_zreg_n<T, n>(NX, N1, B, s, sd, g, tw, chi, tau); break;
      RISM_FOR_N(X)
#undef X
    }
    return;
  }
  const int L = zstar_lines<T>(N2, g.m);
  const size_t lds = (size_t)g.m * L * lstride_for(N2) * sizeof(cpx<T>);
  const dim3 grid = g.zorder ? dim3((NX + L - 1) / L, N1, B) : dim3(B, (NX + L - 1) / L, N1);
  switch (L) {
    case 2: launch_zstar_l<T, 2>(N2, grid, lds, s, sd, g, tw, chi, tau); break;
    case 4: launch_zstar_l<T, 4>(N2, grid, lds, s, sd, g, tw, chi, tau); break;
    case 8: launch_zstar_l<T, 8>(N2, grid, lds, s, sd, g, tw, chi, tau); break;
    default: launch_zstar_l<T, 16>(N2, grid, lds, s, sd, g, tw, chi, tau); break;
  }
}

template void launch_zstar<RISM_T>(int, int, int, int, hipStream_t, const SoluteDesc*,
                                   const GridArgs&, const cpx<RISM_T>*, const RISM_T*,
                                   const RISM_T*);

}  // namespace rism

// The x and y passes of the residual chain on rows, and the Gram rows.
#include "chain_launch.hpp"

#ifndef RISM_T
#error "RISM_T: the working type of this translation unit"
#endif

namespace rism {

#define RISM_FOR_N(X) X(32) X(48) X(64) X(96) X(128) X(192) X(256) X(384)

// The history loads of the closure and residual kernels are unrolled over
// H slots held in registers: the smallest of 8, 10 and MAX_DIIS that holds
// every solute's history (at 10 slots the residual kernel keeps 80 fewer
// bytes per lane in flight than at 16).
template <typename T>
void launch_closure_r2c(int N0, dim3 grid, hipStream_t s, const SoluteDesc* sd, const GridArgs& g,
                        const cpx<T>* twh, const cpx<T>* twf, int hist) {
  if (hist <= 8) {
    switch (N0) {
#define X(n) case n: hipLaunchKernelGGL((closure_r2c_x<T, n, 8>), grid, dim3(NT), 0, s, sd, g, twh, twf); break;
      RISM_FOR_N(X)
#undef X
    }
    return;
  }
  if (hist <= 10) {
    switch (N0) {
#define X(n) case n: hipLaunchKernelGGL((closure_r2c_x<T, n, 10>), grid, dim3(NT), 0, s, sd, g, twh, twf); break;
      RISM_FOR_N(X)
#undef X
    }
    return;
  }
  switch (N0) {
#define X(n) case n: hipLaunchKernelGGL((closure_r2c_x<T, n, MAX_DIIS>), grid, dim3(NT), 0, s, sd, g, twh, twf); break;
    RISM_FOR_N(X)
#undef X
  }
}
template <typename T>
void launch_c2r_resid(int N0, dim3 grid, hipStream_t s, const SoluteDesc* sd, const GridArgs& g,
                      const cpx<T>* twh, const cpx<T>* twf, int hist) {
  if (hist <= 8) {
    switch (N0) {
#define X(n) case n: hipLaunchKernelGGL((c2r_x_resid<T, n, 8>), grid, dim3(NT), 0, s, sd, g, twh, twf); break;
      RISM_FOR_N(X)
#undef X
    }
    return;
  }
  if (hist <= 10) {
    switch (N0) {
#define X(n) case n: hipLaunchKernelGGL((c2r_x_resid<T, n, 10>), grid, dim3(NT), 0, s, sd, g, twh, twf); break;
      RISM_FOR_N(X)
#undef X
    }
    return;
  }
  switch (N0) {
#define X(n) case n: hipLaunchKernelGGL((c2r_x_resid<T, n, MAX_DIIS>), grid, dim3(NT), 0, s, sd, g, twh, twf); break;
    RISM_FOR_N(X)
#undef X
  }
}
template <typename T, bool INV>
void launch_fft_y(int N1, dim3 grid, hipStream_t s, const SoluteDesc* sd, const GridArgs& g,
                  const cpx<T>* tw) {
  constexpr int LN = y_lines<T>();
  switch (N1) {
#define X(n) case n: hipLaunchKernelGGL((fft_y<T, n, LN, INV>), grid, dim3(NT), 0, s, sd, g, tw); break;
    RISM_FOR_N(X)
#undef X
  }
}

// n: entries of the solute with the most.
template <typename T>
void launch_gram(dim3 grid, hipStream_t s, const SoluteDesc* sd, int64_t mP, int n) {
  if (n <= 8) hipLaunchKernelGGL((gram_rows<T, 8>), grid, dim3(NT), 0, s, sd, mP);
  else if (n <= 10) hipLaunchKernelGGL((gram_rows<T, 10>), grid, dim3(NT), 0, s, sd, mP);
  else hipLaunchKernelGGL((gram_rows<T, MAX_DIIS>), grid, dim3(NT), 0, s, sd, mP);
}

template void launch_gram<RISM_T>(dim3, hipStream_t, const SoluteDesc*, int64_t, int);
template void launch_closure_r2c<RISM_T>(int, dim3, hipStream_t, const SoluteDesc*, const GridArgs&,
                                         const cpx<RISM_T>*, const cpx<RISM_T>*, int);
template void launch_c2r_resid<RISM_T>(int, dim3, hipStream_t, const SoluteDesc*, const GridArgs&,
                                       const cpx<RISM_T>*, const cpx<RISM_T>*, int);
template void launch_fft_y<RISM_T, false>(int, dim3, hipStream_t, const SoluteDesc*,
                                          const GridArgs&, const cpx<RISM_T>*);
template void launch_fft_y<RISM_T, true>(int, dim3, hipStream_t, const SoluteDesc*,
                                         const GridArgs&, const cpx<RISM_T>*);

}  // namespace rism

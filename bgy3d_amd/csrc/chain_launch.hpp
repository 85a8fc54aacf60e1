// Launchers of the residual chain's kernels (chain.hpp).  Each is compiled
// for one working type in a translation unit of its own (chain_rows.hip,
// chain_zpass.hip, chain_planes.hip, once with RISM_T double and once with
// float), so that the instantiations build in parallel.
#pragma once
#include <algorithm>
#include <cstdlib>

#include "chain.hpp"

namespace rism {

struct HipFailure {
  hipError_t err;
};

// Tuning knobs, read once: RISM3D_ZSTAR_LINES (kx columns per zstar
// workgroup, 2..16) and RISM3D_ZSTAR_ORDER (0..3, see zstar_reg).
inline int env_int(const char* name, int dflt) {
  const char* v = std::getenv(name);
  return v ? std::atoi(v) : dflt;
}

template <typename T> constexpr int y_lines() { return 128 / (int)sizeof(cpx<T>); }

template <typename T>
int zstar_lines(int N2, int m) {
  // 8 kx columns per workgroup (64 B FP32, 128 B FP64 rows): at 128^3 the
  // FP32 pass ran 1.7 ms with 8 against 2.25 ms with 16 and 2.3 ms with 4
  // (64 solutes, m = 3; occupancy against row length)
  int L = 8;
  const int want = env_int("RISM3D_ZSTAR_LINES", 0);
  if (want == 2 || want == 4 || want == 8 || want == 16) L = want;
  while (L > 2 && (size_t)m * L * lstride_for(N2) * sizeof(cpx<T>) > 64 * 1024) L /= 2;
  return L;
}

// zstar_reg for the solute residual with 3 or 5 solvent sites and for the 3D
// solvent of at most 3 sites, whose points fit in registers (6 pairs: 24 to
// 48 registers a thread; 4 sites are 10 pairs); zstar otherwise, and for all
// with RISM3D_ZSTAR_LDS=1.
inline bool use_zreg(const GridArgs& g) {
  static const int lds_only = env_int("RISM3D_ZSTAR_LDS", 0);
  return !lds_only && ((g.special == 0 && (g.m == 3 || g.m == 5)) ||
                       (g.special == 1 && g.msol <= 3));
}

// The residual of B solutes on xy planes (closure_r2c_xy, zstar,
// c2r_xy_resid: three launches, the y transforms inside the plane kernels)
// when the planes are square, otherwise (and with RISM3D_PLANES=0) the
// five-launch chain.  FP32: up to 128 points per side, at 48 from four solutes
// on (us per pass, rows against planes: 48^3 50 and 48 but 68 and 72 with the
// host's part for one solute, 195 and 184 for 24; 32^3 48 and 37, 86 and 61;
// 192^2 planes would fill a CU's LDS: 800 and 800, 481 and 552).  FP64: up to 64
// points always; planes of 96 and 128 points take 78 and 136 KB of LDS, two
// and one workgroup per CU, and need about two and four workgroups per CU to
// fill the chip (us per FP64 pass, rows against planes: 32^3 47 and 30, 64^3 72
// and 59, 24 x 64^3 1006 and 841; 96^3 118 and 123 for one solute, 199 and 195
// for 2, 287 and 270 for 3; 128^3 234 and 261, 423 and 437, 4 solutes 1188
// and 1138).  The plane kernels write W y-major with the Nyquist column apart
// (GridArgs::ylay), which only zstar_reg reads.
inline bool use_planes(const GridArgs& g, int B, bool fp32, int on) {
  if (!on || g.N0 != g.N1 || !use_zreg(g)) return false;
  if (fp32)
    return g.N0 == 32 || g.N0 == 64 || g.N0 == 96 || g.N0 == 128 ||
           (g.N0 == 48 && (int64_t)g.m * g.N2 * B >= 512);
  if (g.N0 <= 64) return true;
  const int64_t wgs = (int64_t)g.m * g.N2 * B;
  return (g.N0 == 96 && wgs >= 512) || (g.N0 == 128 && wgs >= 1024);
}

template <typename T>
void launch_closure_r2c(int N0, dim3 grid, hipStream_t s, const SoluteDesc* sd, const GridArgs& g,
                        const cpx<T>* twh, const cpx<T>* twf, int hist);
template <typename T>
void launch_c2r_resid(int N0, dim3 grid, hipStream_t s, const SoluteDesc* sd, const GridArgs& g,
                      const cpx<T>* twh, const cpx<T>* twf, int hist);
template <typename T, bool INV>
void launch_fft_y(int N1, dim3 grid, hipStream_t s, const SoluteDesc* sd, const GridArgs& g,
                  const cpx<T>* tw);
template <typename T>
void launch_zstar(int N2, int NX, int N1, int B, hipStream_t s, const SoluteDesc* sd,
                  const GridArgs& g, const cpx<T>* tw, const T* chi, const T* tau);
// Workgroups of gram_rows per solute: 4 points or more a thread, 2048 at most
// (192^3 with 5 sites: 122 us, 127 with 4096), and 16384 in all: in a batch only
// the solutes at an extrapolation work, a third of them (us per pass with 8192
// and with 16384: 24 x 64^3 in FP64 104 and 99, 24 x 128^3 in FP32 178 and 173).
inline int gram_blocks(int64_t mP, int B) {
  const int64_t most = std::max(64, std::min(2048, 16384 / B)), fit = mP / (NT * 4);
  return (int)std::max<int64_t>(1, std::min(most, fit));
}
template <typename T>
void launch_gram(dim3 grid, hipStream_t s, const SoluteDesc* sd, int64_t mP, int n);
template <typename T>
void launch_planes(bool inv, int B, hipStream_t s, const SoluteDesc* sd, const GridArgs& g,
                   const cpx<T>* twh, const cpx<T>* twf, int hist);

}  // namespace rism

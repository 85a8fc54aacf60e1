// gfx950 kernels of the 3D-RISM residual F(t) = (chi - 1) * c(t) - t and
// its setup / post-processing.  One residual evaluation is five launches,
// or three on xy planes (closure_r2c_xy, zstar, c2r_xy_resid):
//
//   1. closure_r2c_x : c = closure(beta v, t) fused into the x-axis r2c
//   2. fft_y         : forward c2c along y
//   3. zstar         : forward c2c along z, per-k m x m chi contraction,
//                      tau (or Ng long-range) term, inverse c2c along z
//   4. fft_y         : inverse c2c along y
//   5. c2r_x_resid   : x-axis c2r fused with r = t' - t and its norms
//
// References: iterate_t1 hnc3d.c:1184-1285, star hnc3d.c:1115-1138,
// compute_c hnc3d.c:167-181, closures.f90:107-128 and 248-432,
// interp bgy3d-vec.c:23-46, KFREQ bgy3d.h:162, FFT layout
// bgy3d-fftw3.c:364-385.
#pragma once
#include "fft_device.hpp"
#include "kernels.hpp"
#include "closure_math.hpp"

namespace rism {

// closure_c, closure_dc and their helpers: closure_math.hpp

// ------------------------------------------------------------- row sizes
__host__ __device__ constexpr int rows_for(int M) {
  return M <= 16 ? 64 : M <= 32 ? 32 : M <= 64 ? 16 : M <= 128 ? 8 : 4;
}

// Twiddles: every chain kernel but zstar (which reads them from memory) copies
// its tables to LDS (stw) beside its first loads.  Read from global memory inside the stages they shared the vector
// cache and its wait counter with the streams, and each stage waited on both (us per
// launch, from global memory and from LDS: closure and residual of 24 x 128^3
// in FP32 719 and 667, 597 and 547, its z pass 281 and 241; 192^3 with 5 sites
// in FP32 closure 203 and 186, y 71 and 56, z 140 and 126; 24 x 64^3 in FP64 closure
// and residual 193 and 185, 153 and 133, z 91 and 82).

// 16-byte vectors of the working type: the streaming loops of the x-axis
// kernels move 16 B per lane per array (global_load/store_dwordx4), four
// times fewer memory instructions than scalar accesses.  Every array is
// addressed at multiples of N0 >= 32 elements from a 256-byte aligned base.
template <typename T> struct alignas(16) Vec16 {
  static constexpr int W = 16 / sizeof(T);
  T v[W];
};
// Global-memory accessors.  The array pointers come out of descriptors in
// memory, so the compiler sees generic pointers and emits flat accesses,
// which also count against the LDS wait counter: every wait for an LDS
// access would then wait for the outstanding HBM loads too.  These casts to
// address space 1 (through native vector types; aggregate copies lose the
// address space) give global_load / global_store.
template <typename T> struct VecOf;
template <> struct VecOf<float> {
  typedef float v4 __attribute__((ext_vector_type(4)));
  typedef float v2 __attribute__((ext_vector_type(2)));
};
template <> struct VecOf<double> {
  typedef double v4 __attribute__((ext_vector_type(2)));  // 16 bytes
  typedef double v2 __attribute__((ext_vector_type(2)));
};
template <typename T> __device__ __forceinline__ Vec16<T> ld16(const T* p) {
  typedef typename VecOf<T>::v4 V;
  typedef __attribute__((address_space(1))) const V GV;
  const V x = *(GV*)p;
  Vec16<T> r;
#pragma unroll
  for (int k = 0; k < Vec16<T>::W; ++k) r.v[k] = x[k];
  return r;
}
template <typename T> __device__ __forceinline__ void st16(T* p, const Vec16<T>& r) {
  typedef typename VecOf<T>::v4 V;
  typedef __attribute__((address_space(1))) V GV;
  V x;
#pragma unroll
  for (int k = 0; k < Vec16<T>::W; ++k) x[k] = r.v[k];
  *(GV*)p = x;
}
template <typename T> __device__ __forceinline__ cpx<T> ldc(const cpx<T>* p) {
  typedef typename VecOf<T>::v2 V;
  typedef __attribute__((address_space(1))) const V GV;
  const V x = *(GV*)p;
  return cpx<T>{x[0], x[1]};
}
template <typename T> __device__ __forceinline__ void stc(cpx<T>* p, cpx<T> c) {
  typedef typename VecOf<T>::v2 V;
  typedef __attribute__((address_space(1))) V GV;
  V x;
  x[0] = c.re;
  x[1] = c.im;
  *(GV*)p = x;
}
// base[i] for a base the same in every lane and an element index below
// 2^32 bytes from it: the byte offset stays 32-bit, so the access takes the
// scalar-base form instead of a 64-bit address per lane.
template <typename X> __device__ __forceinline__ X* at32(X* base, uint32_t i) {
  return reinterpret_cast<X*>(reinterpret_cast<char*>(base) + i * (uint32_t)sizeof(X));
}
template <typename X> __device__ __forceinline__ const X* at32(const X* base, uint32_t i) {
  return reinterpret_cast<const X*>(reinterpret_cast<const char*>(base) + i * (uint32_t)sizeof(X));
}
template <typename X> __device__ __forceinline__ X gld(const X* p) {  // scalars
  typedef __attribute__((address_space(1))) const X GX;
  return *(GX*)p;
}
template <typename X> __device__ __forceinline__ void gst(X* p, X v) {
  typedef __attribute__((address_space(1))) X GX;
  *(GX*)p = v;
}

// BF16 storage of the FP32 phase's MDIIS residual history, which enters
// only the Gram products <r_i, r_j>: round to nearest even, four values in
// eight bytes.  The Gram row of a new residual is formed from its rounded
// values, so the Gram matrix stays that of the stored vectors.
struct alignas(8) BF4 { uint32_t lo, hi; };
__device__ __forceinline__ uint32_t bf16_bits(float f) {
  const uint32_t u = __float_as_uint(f);
  return (u + 0x7FFFu + ((u >> 16) & 1u)) >> 16;
}
__device__ __forceinline__ float bf16_val(uint32_t h) { return __uint_as_float(h << 16); }
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ BF4 ldbf4(const uint16_t* p) {
  typedef __attribute__((address_space(1))) const u32x2 G;
  const u32x2 x = *(G*)p;
  return BF4{x[0], x[1]};
}
__device__ __forceinline__ void stbf4(uint16_t* p, BF4 q) {
  typedef __attribute__((address_space(1))) u32x2 G;
  u32x2 x;
  x[0] = q.lo;
  x[1] = q.hi;
  *(G*)p = x;
}
// FP8 e4m3 (OCP: largest finite 448; the conversion does not saturate, so
// values are clamped first) of four points scaled by s, packed in a word.
__device__ __forceinline__ uint32_t to_fp8x4(const Vec16<float>& v, float s) {
  auto c = [s](float x) { return fminf(fmaxf(x * s, -448.f), 448.f); };
  int w = 0;
  w = __builtin_amdgcn_cvt_pk_fp8_f32(c(v.v[0]), c(v.v[1]), w, false);
  w = __builtin_amdgcn_cvt_pk_fp8_f32(c(v.v[2]), c(v.v[3]), w, true);
  return (uint32_t)w;
}
__device__ __forceinline__ Vec16<float> from_fp8x4(uint32_t w, float inv) {
  Vec16<float> x;
  x.v[0] = __builtin_amdgcn_cvt_f32_fp8((int)w, 0) * inv;
  x.v[1] = __builtin_amdgcn_cvt_f32_fp8((int)w, 1) * inv;
  x.v[2] = __builtin_amdgcn_cvt_f32_fp8((int)w, 2) * inv;
  x.v[3] = __builtin_amdgcn_cvt_f32_fp8((int)w, 3) * inv;
  return x;
}
__device__ __forceinline__ BF4 to_bf4(const Vec16<float>& v) {
  BF4 q;
  q.lo = bf16_bits(v.v[0]) | (bf16_bits(v.v[1]) << 16);
  q.hi = bf16_bits(v.v[2]) | (bf16_bits(v.v[3]) << 16);
  return q;
}
// The FP32 phase's residual history (Gram rows only): four points of entry
// j at element idx as one packed word (BF16 pairs, or an FP8 word in lo),
// unpacked to FP32, and the new r stored rounded (returned as rounded, so
// that the Gram row is formed from the values the history keeps).
__device__ __forceinline__ BF4 ld_hist(const SoluteDesc& d, const void* p, int64_t idx) {
  if (d.r8) {
    BF4 q;
    q.lo = *reinterpret_cast<const uint32_t*>(static_cast<const uint8_t*>(p) + idx);
    q.hi = 0;
    return q;
  }
  return ldbf4(static_cast<const uint16_t*>(p) + idx);
}
__device__ __forceinline__ Vec16<float> un_hist(const SoluteDesc& d, int j, BF4 q) {
  if (d.r8) return from_fp8x4(q.lo, d.rhinv[j]);
  Vec16<float> x;
  x.v[0] = bf16_val(q.lo & 0xFFFFu);
  x.v[1] = bf16_val(q.lo >> 16);
  x.v[2] = bf16_val(q.hi & 0xFFFFu);
  x.v[3] = bf16_val(q.hi >> 16);
  return x;
}
__device__ __forceinline__ Vec16<float> st_hist(const SoluteDesc& d, int64_t idx,
                                                const Vec16<float>& r) {
  if (d.r8) {
    const uint32_t w = to_fp8x4(r, d.rsc);
    *reinterpret_cast<uint32_t*>(static_cast<uint8_t*>(d.r) + idx) = w;
    return from_fp8x4(w, 1.0f / d.rsc);
  }
  const BF4 q = to_bf4(r);
  stbf4(static_cast<uint16_t*>(d.r) + idx, q);
  Vec16<float> x;
  x.v[0] = bf16_val(q.lo & 0xFFFFu);
  x.v[1] = bf16_val(q.lo >> 16);
  x.v[2] = bf16_val(q.hi & 0xFFFFu);
  x.v[3] = bf16_val(q.hi >> 16);
  return x;
}

// Index of the k point (kz, ky, kx) in a solute's form factor F(k) s(k):
// z-major rows of NH like the tables in FP64; in FP32 y-major rows of
// N0/2 bins (the layout of the plane chain's spectra) and the Nyquist
// column kx = N0/2 compact behind them, so that the z pass reads it
// as it reads the spectra.  (FP64 has that compact column too, at the same
// place, for the z pass's Nyquist blocks.)
template <typename T>
__device__ __forceinline__ int64_t fs_index(const GridArgs& g, int z, int y, int x) {
  if constexpr (sizeof(T) == 8) return ((int64_t)z * g.N1 + y) * g.NH + x;
  return x == g.NX - 1 ? g.K + (int64_t)z * g.N1 + y : ((int64_t)y * g.N2 + z) * g.NH + x;
}

// One vector of VW points at e (an offset into the slab off of solute d's
// site arrays): the MDIIS step t = sum_j coef_j u_j (written to t) or the
// given t, then c = closure(beta v, t) in the solver mode of d.
template <typename T, int H>
__device__ __forceinline__ Vec16<T> closure_vec(const SoluteDesc& d, const GridArgs& g,
                                                int64_t off, int e, T* __restrict__ t,
                                                const T* __restrict__ bv) {
  constexpr int VW = Vec16<T>::W;
  const int nc = d.ncomb;
  Vec16<T> c;
  Vec16<T> tv;
  const Vec16<T> b = ld16(bv + e);
  if (nc > 0) {
    double acc[VW];
#pragma unroll
    for (int k = 0; k < VW; ++k) acc[k] = 0.0;
    bool summed = false;
    if constexpr (sizeof(T) == 4) {
      if (d.u16) {  // the newest u (FP32) and BF16 differences, loads first
        const Vec16<T> u0 = ld16(static_cast<const T*>(d.u[0]) + off + e);
        BF4 du[H];
#pragma unroll
        for (int j = 1; j < H; ++j)
          if (j < nc) du[j] = ldbf4(static_cast<const uint16_t*>(d.u[j]) + off + e);
#pragma unroll
        for (int k = 0; k < VW; ++k) acc[k] = d.coef[0] * (double)u0.v[k];
#pragma unroll
        for (int j = 1; j < H; ++j)
          if (j < nc) {
            const double cj = d.coef[j];
            acc[0] += cj * (double)bf16_val(du[j].lo & 0xFFFFu);
            acc[1] += cj * (double)bf16_val(du[j].lo >> 16);
            acc[2] += cj * (double)bf16_val(du[j].hi & 0xFFFFu);
            acc[3] += cj * (double)bf16_val(du[j].hi >> 16);
          }
        summed = true;
      }
    }
    if (!summed) {
      // all loads first, then the sums: independent loads in flight
      Vec16<T> u[H];
#pragma unroll
      for (int j = 0; j < H; ++j)
        if (j < nc) u[j] = ld16(static_cast<const T*>(d.u[j]) + off + e);
      Vec16<T> sh;
      if (d.shift_w != 0.0) sh = ld16(static_cast<const T*>(d.shift) + off + e);
#pragma unroll
      for (int j = 0; j < H; ++j)
        if (j < nc) {
          const double cj = d.coef[j];
#pragma unroll
          for (int k = 0; k < VW; ++k) acc[k] += cj * (double)u[j].v[k];
        }
      if (d.shift_w != 0.0) {
#pragma unroll
        for (int k = 0; k < VW; ++k) acc[k] -= d.shift_w * (double)sh.v[k];
      }
    }
#pragma unroll
    for (int k = 0; k < VW; ++k) tv.v[k] = T(acc[k]);
    st16(t + e, tv);
  } else {
    tv = ld16(t + e);
  }
#pragma unroll
  for (int k = 0; k < VW; ++k) {
    if (d.mode == 0) c.v[k] = closure_c<T>(g.closure, g.pse_order, b.v[k], tv.v[k]);
    else if (d.mode == 5)  // bv holds x_b (PY: exp(-beta v) - 1, c linear in t)
      c.v[k] = (g.closure == 2) ? b.v[k] * tv.v[k]
                                : closure_dc<T>(g.closure, g.pse_order, b.v[k], tv.v[k]);
    else if (d.mode == 6)  // J v: dc = (dc/dt) v (compute_c1, hnc3d.c:1307)
      c.v[k] = T(gld(d.dt + off + e + k) * (double)tv.v[k]);
    else if (d.mode == 7)  // flag form: dc + v (hnc3d.c:1310-1320)
      c.v[k] = T((gld(d.dt + off + e + k) + 1.0) * (double)tv.v[k]);
    else if (d.mode == 10)  // rho h for the susceptibility (hnc3d.c:1006-1030)
      c.v[k] = T(g.rho) * (closure_c<T>(g.closure, g.pse_order, b.v[k], tv.v[k]) + tv.v[k]);
    else c.v[k] = tv.v[k];
  }
  return c;
}

// ------------------------------------------- 1. closure fused with x r2c
// t = sum_j coef_j u_j (the MDIIS step; written back as the iterate) or the
// given t, then c = closure(beta v, t), then the x-axis r2c of c.
// Grid: x = ceil(N1 N2 / ROWS), y = site, z = solute.
template <typename T, int N0, int H>
__global__ void __launch_bounds__(NT)
closure_r2c_x(const SoluteDesc* __restrict__ sd, GridArgs g,
              const cpx<T>* __restrict__ tw_half, const cpx<T>* __restrict__ tw_full) {
  constexpr int M = N0 / 2;
  constexpr int ROWS = rows_for(M);
  constexpr int LSM = lstride_for(M);
  __shared__ cpx<T> lds[ROWS * LSM];
  const SoluteDesc& d = sd[blockIdx.z];
  if (!d.active) return;
  // the twiddles in LDS: [M of the rows][M + 1 of the split]
  __shared__ cpx<T> stw[2 * M + 1];
  for (int i = threadIdx.x; i < 2 * M + 1; i += NT) stw[i] = i < M ? tw_half[i] : tw_full[i - M];
  const int site = blockIdx.y;
  const int nrows = g.N1 * g.N2;
  const int row0 = blockIdx.x * ROWS;
  const int64_t off = site * g.P + (int64_t)row0 * N0;
  T* __restrict__ t = static_cast<T*>(d.t) + off;
  const T* __restrict__ bv = static_cast<const T*>(d.bv) + off;
  const int vrows = min(ROWS, nrows - row0);
  const int nvalid = vrows * N0;
  constexpr int VW = Vec16<T>::W;
  for (int e = threadIdx.x * VW; e < ROWS * N0; e += NT * VW) {
    Vec16<T> c;
#pragma unroll
    for (int k = 0; k < VW; ++k) c.v[k] = T(0);
    if (e < nvalid) c = closure_vec<T, H>(d, g, off, e, t, bv);  // whole vectors
    // z_n = c_{2n} + i c_{2n+1} of row e / N0
    cpx<T>* zrow = lds + (e / N0) * LSM;
    const int n0 = (e % N0) / 2;
#pragma unroll
    for (int h = 0; h < VW / 2; ++h) zrow[lpos(n0 + h)] = cpx<T>{c.v[2 * h], c.v[2 * h + 1]};
  }
  __syncthreads();
  fft_lines<T, M, ROWS, NT, false>(lds, LSM, vrows, stw);
  cpx<T>* W = static_cast<cpx<T>*>(d.W) + site * g.K + (int64_t)row0 * g.NH;
  const int nout = min(ROWS, nrows - row0) * (M + 1);
  for (int e = threadIdx.x; e < nout; e += NT) {
    const int row = e / (M + 1);
    const int k = e - row * (M + 1);
    const cpx<T> zk = lds[row * LSM + lpos(k == M ? 0 : k)];
    const cpx<T> zm = cconj(lds[row * LSM + lpos(k == 0 ? 0 : M - k)]);
    const cpx<T> s = cadd(zk, zm);
    const cpx<T> dd = rot90<T, false>(cmul(stw[M + k], csub(zk, zm)));  // -i w (Zk - conj Zm)
    stc(W + row * g.NH + k, cpx<T>{T(0.5) * (s.re + dd.re), T(0.5) * (s.im + dd.im)});
  }
}

// -------------------------------------------------- 2/4. c2c along y
// Grid: x = ceil(NH / LINES), y = site * N2 + z, z = solute.
template <typename T, int N1, int LINES, bool INV>
__global__ void __launch_bounds__(NT)
fft_y(const SoluteDesc* __restrict__ sd, GridArgs g, const cpx<T>* __restrict__ tw) {
  __shared__ cpx<T> lds[LINES * N1];  // interleaved: point y of column l at y * LINES + l
  __shared__ cpx<T> stw[N1];
  const SoluteDesc& d = sd[blockIdx.z];
  if (!d.active) return;
  for (int i = threadIdx.x; i < N1; i += NT) stw[i] = tw[i];
  const int site = blockIdx.y / g.N2;
  const int z = blockIdx.y - site * g.N2;
  const int kx0 = blockIdx.x * LINES;
  cpx<T>* W = static_cast<cpx<T>*>(d.W) + site * g.K + (int64_t)z * g.N1 * g.NH + kx0;
  {
    // all loads first (the row padding keeps every column of a tile in
    // bounds; columns past NX are zeroed after the load)
    constexpr int PTS = N1 * LINES, PT = (PTS + NT - 1) / NT;
    const int nl = min(LINES, g.NX - kx0);
    cpx<T> v[PT];
#pragma unroll
    for (int p = 0; p < PT; ++p) {
      const int e = threadIdx.x + p * NT;
      if (PT * NT == PTS || e < PTS) {
        const int y = e / LINES, l = e - y * LINES;
        // the last tile (the Nyquist column) reads only its valid columns
        if (nl == LINES || l < nl) v[p] = ldc(W + y * g.NH + l);
      }
    }
#pragma unroll
    for (int p = 0; p < PT; ++p) {
      const int e = threadIdx.x + p * NT;
      if (PT * NT == PTS || e < PTS) {
        const int l = e & (LINES - 1);
        lds[e] = (kx0 + l < g.NX) ? v[p] : cpx<T>{T(0), T(0)};
      }
    }
  }
  __syncthreads();
  fft_lines_il<T, N1, LINES, NT, INV>(lds, min(LINES, g.NX - kx0), stw);
  for (int e = threadIdx.x; e < N1 * LINES; e += NT) {
    const int y = e / LINES, l = e - y * LINES;
    if (kx0 + l < g.NX) stc(W + y * g.NH + l, lds[e]);
  }
}

// |k|^2 = (kx^2 + ky^2) + kz^2, rounded exactly as the reference's
// SQR(k[0]) + SQR(k[1]) + SQR(k[2]) (bgy3d-vec.h:664-667): no FMA
// contraction.  interp() below is discontinuous at table midpoints and grid
// k often lands exactly on one, so the last bit selects the neighbour.
__device__ __forceinline__ double kmag2(double kx, double ky, double kz) {
#pragma clang fp contract(off)
  const double a = kx * kx;
  const double b = ky * ky;
  const double c = kz * kz;
  return (a + b) + c;
}

// The per-k solvent-solvent OZ of one k point (iterate_t2, hnc3d.c:376-470;
// compute_t2_m, hnc3d.c:231-324) for g.msol <= MSX sites, the site-site
// pair spectra of the point in LDS (pair p = i(i+1)/2 + j at
// lds[(p LINES + l) LS + lpos(z)]), overwritten with T.  sgn is the corner
// phase of the point, U the unit long-range Coulomb there, kk its index
// into the omega table chi3.
template <typename T, int MSX, int LINES, int LS>
__device__ void oz_pairs(cpx<T>* __restrict__ lds, const GridArgs& g, const T* __restrict__ chi3,
                         int64_t kk, int l, int z, double sgn, double U) {
  // solvent-solvent OZ (iterate_t2, hnc3d.c:376-470; compute_t2_m,
  // hnc3d.c:231-324): C = h^3 c s - beta q_i q_j U at the corner,
  // X = (1 - rho W C)^-1 W C W, T = ((X - C) - beta q_i q_j U) s / L^3
  const int ms = g.msol;
  double Cr[MSX][MSX], Ci[MSX][MSX], Wm[MSX][MSX];
  for (int i = 0; i < ms; ++i)
    for (int j = 0; j <= i; ++j) {
      const int p = i * (i + 1) / 2 + j;
      const cpx<T> c = lds[(p * LINES + l) * LS + lpos(z)];
      const double q2 = g.q[i] * g.q[j];
      const double re = (double)c.re * g.h3 * sgn - g.beta * q2 * U;
      const double im = (double)c.im * g.h3 * sgn;
      Cr[i][j] = Cr[j][i] = re;
      Ci[i][j] = Ci[j][i] = im;
      Wm[i][j] = Wm[j][i] = (i == j) ? 1.0 : (double)chi3[p * g.KT + kk];
    }
  // WC, A = 1 - rho WC, B = WC W
  double WCr[MSX][MSX], WCi[MSX][MSX], Ar[MSX][MSX], Ai[MSX][MSX], Br[MSX][MSX],
      Bi[MSX][MSX];
  for (int i = 0; i < ms; ++i)
    for (int j = 0; j < ms; ++j) {
      double ar = 0.0, ai = 0.0;
      for (int q = 0; q < ms; ++q) { ar += Wm[i][q] * Cr[q][j]; ai += Wm[i][q] * Ci[q][j]; }
      WCr[i][j] = ar;
      WCi[i][j] = ai;
      Ar[i][j] = (i == j ? 1.0 : 0.0) - g.rho * ar;
      Ai[i][j] = -g.rho * ai;
    }
  for (int i = 0; i < ms; ++i)
    for (int j = 0; j < ms; ++j) {
      double br = 0.0, bi = 0.0;
      for (int q = 0; q < ms; ++q) { br += WCr[i][q] * Wm[q][j]; bi += WCi[i][q] * Wm[q][j]; }
      Br[i][j] = br;
      Bi[i][j] = bi;
    }
  // Gaussian elimination with partial pivoting, A X = B
  for (int col = 0; col < ms; ++col) {
    int piv = col;
    double best = Ar[col][col] * Ar[col][col] + Ai[col][col] * Ai[col][col];
    for (int r = col + 1; r < ms; ++r) {
      const double a2 = Ar[r][col] * Ar[r][col] + Ai[r][col] * Ai[r][col];
      if (a2 > best) { best = a2; piv = r; }
    }
    if (piv != col)
      for (int q = 0; q < ms; ++q) {
        double tr = Ar[col][q], ti = Ai[col][q];
        Ar[col][q] = Ar[piv][q]; Ai[col][q] = Ai[piv][q]; Ar[piv][q] = tr; Ai[piv][q] = ti;
        tr = Br[col][q]; ti = Bi[col][q];
        Br[col][q] = Br[piv][q]; Bi[col][q] = Bi[piv][q]; Br[piv][q] = tr; Bi[piv][q] = ti;
      }
    const double dr = Ar[col][col], di = Ai[col][col];
    const double den = dr * dr + di * di;
    const double ir = dr / den, ii = -di / den;  // 1 / A[col][col]
    for (int r = col + 1; r < ms; ++r) {
      const double fr = Ar[r][col] * ir - Ai[r][col] * ii;
      const double fi = Ar[r][col] * ii + Ai[r][col] * ir;
      for (int q = col; q < ms; ++q) {
        Ar[r][q] -= fr * Ar[col][q] - fi * Ai[col][q];
        Ai[r][q] -= fr * Ai[col][q] + fi * Ar[col][q];
      }
      for (int q = 0; q < ms; ++q) {
        Br[r][q] -= fr * Br[col][q] - fi * Bi[col][q];
        Bi[r][q] -= fr * Bi[col][q] + fi * Br[col][q];
      }
    }
  }
  for (int col = ms - 1; col >= 0; --col) {
    const double dr = Ar[col][col], di = Ai[col][col];
    const double den = dr * dr + di * di;
    const double ir = dr / den, ii = -di / den;
    for (int q = 0; q < ms; ++q) {
      double xr = Br[col][q], xi = Bi[col][q];
      for (int r = col + 1; r < ms; ++r) {
        xr -= Ar[col][r] * Br[r][q] - Ai[col][r] * Bi[r][q];
        xi -= Ar[col][r] * Bi[r][q] + Ai[col][r] * Br[r][q];
      }
      Br[col][q] = xr * ir - xi * ii;
      Bi[col][q] = xr * ii + xi * ir;
    }
  }
  for (int i = 0; i < ms; ++i)
    for (int j = 0; j <= i; ++j) {
      const int p = i * (i + 1) / 2 + j;
      const double q2 = g.q[i] * g.q[j];
      const double tr = ((Br[i][j] - Cr[i][j]) - g.beta * q2 * U) * sgn * g.inv_L3;
      const double ti = (Bi[i][j] - Ci[i][j]) * sgn * g.inv_L3;
      lds[(p * LINES + l) * LS + lpos(z)] = cpx<T>{T(tr), T(ti)};
    }
}

// --------------------------- 3. z c2c + chi contraction + tau + z c2c^-1
// Grid: zorder 0: x = solute (concurrent workgroups share one chi3/tau3
// tile), y = ceil(NH / LINES), z = ky row; zorder 1: x = kx tile, y = ky
// row, z = solute (concurrent workgroups stream contiguous planes of one
// solute).  Dynamic LDS:
// m * LINES * lstride_for(N2) complex.  chi3: [m(m+1)/2][KT] chi_ij - delta_ij;
// tau3: [m][KT] s_i(|k|), both on the k grid (table_index), in the working type.
template <typename T, int N2, int LINES>
__global__ void __launch_bounds__(NT)
zstar(const SoluteDesc* __restrict__ sd, GridArgs g, const cpx<T>* __restrict__ tw,
      const T* __restrict__ chi3, const T* __restrict__ tau3) {
  constexpr int LS = lstride_for(N2);
  extern __shared__ unsigned char smem[];
  cpx<T>* lds = reinterpret_cast<cpx<T>*>(smem);
  // zorder 0: grid (solute, kx tile, ky); 1: grid (kx tile, ky, solute)
  const int b = g.zorder ? blockIdx.z : blockIdx.x;
  const SoluteDesc& d = sd[b];
  if (!d.active) return;
  const int m = g.m;
  const int y = g.zorder ? blockIdx.y : blockIdx.z;
  const int kx0 = (g.zorder ? blockIdx.x : blockIdx.y) * LINES;
  const int64_t zs = (int64_t)g.N1 * g.NH;  // z stride
  const int64_t base = (int64_t)y * g.NH + kx0;
  cpx<T>* W = static_cast<cpx<T>*>(d.W) + base;
  for (int s = 0; s < m; ++s) {
    const cpx<T>* Ws = W + s * g.K;
    cpx<T>* L = lds + s * LINES * LS;
    for (int e = threadIdx.x; e < N2 * LINES; e += NT) {
      const int z = e / LINES, l = e - z * LINES;
      L[l * LS + lpos(z)] = (kx0 + l < g.NX) ? Ws[z * zs + l] : cpx<T>{T(0), T(0)};
    }
  }
  __syncthreads();
  const int nl = min(LINES, g.NX - kx0);  // valid kx columns of this tile
  if (d.mode != 4) {  // mode 4: inverse z FFTs of the loaded spectrum only
  for (int s = 0; s < m; ++s) fft_lines<T, N2, LINES, NT, false>(lds + s * LINES * LS, LS, nl, tw);
  if (d.mode == 3) {  // forward spectrum only
    for (int s = 0; s < m; ++s) {
      cpx<T>* Ws = W + s * g.K;
      const cpx<T>* L = lds + s * LINES * LS;
      for (int e = threadIdx.x; e < N2 * LINES; e += NT) {
        const int z = e / LINES, l = e - z * LINES;
        if (kx0 + l < g.NX) Ws[z * zs + l] = L[l * LS + lpos(z)];
      }
    }
    return;
  }
  const bool linear = d.mode != 0;  // chi convolution only

  const int iy = (y <= g.N1 / 2) ? y : y - g.N1;
  const double ky = iy * g.dky;
  if (g.special != 0) {
    for (int e = threadIdx.x; e < N2 * LINES; e += NT) {
      const int z = e / LINES, l = e - z * LINES;
      if (kx0 + l >= g.NX) continue;
      const int64_t kk = table_index(g, z, y, kx0 + l);
      const int iz = (z <= N2 / 2) ? z : z - N2;
      const int ix = kx0 + l;
      const double sgn = ((ix + iy + iz) & 1) ? -1.0 : 1.0;
      if (g.special == 2) {
        // Poisson: u(k) = 4 pi/eps0 h^3 rho(k) / k^2, 0 at k = 0, k^2 summed
        // z, y, x (bgy3d_poisson, bgy3d-poisson.c:103-190); / L^3 for the
        // inverse FFT
        const double kz = iz * g.dkz, kx = ix * g.dkx;
        const double k2 = (kz * kz + ky * ky) + kx * kx;
        const double fac = k2 != 0.0 ? 4 * M_PI * EPSILON0INV * g.h3 / k2 * g.inv_L3 : 0.0;
        for (int s = 0; s < m; ++s) {
          cpx<T>& v = lds[(s * LINES + l) * LS + lpos(z)];
          v = cscale(v, T(fac));
        }
        continue;
      }
      // unit long-range Coulomb as vec_kmap tabulates it: k = |k|, then
      // 4 pi/eps0 exp(-k^2/4G^2)/k^2 (bgy3d-force.c:19-36, bgy3d-force.h)
      const double kabs = sqrt(kmag2(ix * g.dkx, ky, iz * g.dkz));
      const double k2 = kabs * kabs;
      const double U = k2 == 0.0 ? 0.0
          : (4 * M_PI * EPSILON0INV) * exp(-k2 / (4 * G_COULOMB * G_COULOMB)) / k2;
      if (g.special == 3) {
        for (int s = 0; s < m; ++s)
          lds[(s * LINES + l) * LS + lpos(z)] = cpx<T>{T(U * sgn * g.inv_L3), T(0)};
        continue;
      }
      oz_pairs<T, MAX_SITES, LINES, LS>(lds, g, chi3, kk, l, z, sgn, U);
    }
  } else {
  const cpx<T>* Fs = static_cast<const cpx<T>*>(d.Fs);
  for (int e = threadIdx.x; e < N2 * LINES; e += NT) {
    const int z = e / LINES, l = e - z * LINES;
    if (kx0 + l >= g.NX) continue;
    const int64_t kk = table_index(g, z, y, kx0 + l);  // this point in the tables
    const cpx<T> fs = Fs[fs_index<T>(g, z, y, kx0 + l)];
    cpx<T> c[MAX_SITES];
    for (int s = 0; s < m; ++s) c[s] = lds[(s * LINES + l) * LS + lpos(z)];
    cpx<T> uc = {T(0), T(0)};
    if (!g.renorm && !linear) {
      // u_c(k) = 4 pi eps0^-1 exp(-k^2/4G^2)/k^2 F(k) s(k), 0 at k = 0
      // (bgy3d-force.h:140-147, bgy3d-solutes.c:767-792).
      const int iz = (z <= N2 / 2) ? z : z - N2;
      const double k2 = kmag2((kx0 + l) * g.dkx, ky, iz * g.dkz);
      const double shape = (k2 == 0.0) ? 0.0
          : (4 * M_PI * EPSILON0INV) * exp(-k2 / (4 * G_COULOMB * G_COULOMB)) / k2;
      uc = cscale(fs, T(shape));
      for (int s = 0; s < m; ++s) {
        // h^3 C_j - beta q_j u_c  (hnc3d.c:1226-1227)
        c[s] = csub(cscale(c[s], T(g.h3)), cscale(uc, T(g.beta * g.q[s])));
      }
    }
    for (int i = 0; i < m; ++i) {
      cpx<T> acc = {T(0), T(0)};
      for (int j = 0; j < m; ++j) {  // sum_j S_ij sig_j c_j / sig_i (sig = 1: one density)
        const int pi_ = (i >= j) ? i * (i + 1) / 2 + j : j * (j + 1) / 2 + i;
        const T chi = chi3[pi_ * g.KT + kk] * T(g.sig[j]);
        acc.re += chi * c[j].re;
        acc.im += chi * c[j].im;
      }
      acc = cscale(acc, T(1.0 / g.sig[i]));
      cpx<T> out;
      if (linear) {
        out = cscale(acc, T(g.a_scale));
      } else if (g.renorm) {
        // (h^3/L^3) sum_j chi_ij C_j - (beta/eps0/L^3) tau_i F s  (hnc3d.c:1245-1268)
        const T tau = tau3[i * g.KT + kk] * T(g.tau_scale);
        out = csub(cscale(acc, T(g.a_scale)), cscale(fs, tau));
      } else {
        out = cscale(csub(acc, cscale(uc, T(g.beta * g.q[i]))), T(g.inv_L3));
      }
      lds[(i * LINES + l) * LS + lpos(z)] = out;
    }
  }
  }  // g.special
  }  // d.mode != 4
  __syncthreads();
  for (int s = 0; s < m; ++s) fft_lines<T, N2, LINES, NT, true>(lds + s * LINES * LS, LS, nl, tw);
  for (int s = 0; s < m; ++s) {
    cpx<T>* Ws = W + s * g.K;
    const cpx<T>* L = lds + s * LINES * LS;
    for (int e = threadIdx.x; e < N2 * LINES; e += NT) {
      const int z = e / LINES, l = e - z * LINES;
      if (kx0 + l < g.NX) Ws[z * zs + l] = L[l * LS + lpos(z)];
    }
  }
}

// ------------------------------------------------ block reductions
__device__ __forceinline__ double warp_sum(double v) {
  for (int o = 32; o > 0; o >>= 1) v += __shfl_down(v, o, 64);
  return v;
}
__device__ __forceinline__ double warp_max(double v) {
  for (int o = 32; o > 0; o >>= 1) v = fmax(v, __shfl_down(v, o, 64));
  return v;
}

// oz_pairs for a compile-time site count MS, the MS (MS + 1) / 2 pair spectra
// of the point in registers (c, overwritten with T), w the omega of the
// off-diagonal pairs (1 on the diagonal).  Every loop unrolls and the row
// exchanges are selects, so nothing is indexed at run time.
template <int MS>
__device__ __forceinline__ void oz_point(cpx<double> (&c)[MS * (MS + 1) / 2],
                                         const double (&w)[MS * (MS + 1) / 2], const GridArgs& g,
                                         double sgn, double U) {
  auto pr = [](int i, int j) { return i >= j ? i * (i + 1) / 2 + j : j * (j + 1) / 2 + i; };
  cpx<double> A[MS][MS], B[MS][MS];
#pragma unroll
  for (int i = 0; i < MS; ++i)
#pragma unroll
    for (int j = 0; j <= i; ++j) {  // C = h^3 c s - beta q_i q_j U
      cpx<double>& v = c[pr(i, j)];
      v = cpx<double>{v.re * g.h3 * sgn - g.beta * (g.q[i] * g.q[j]) * U, v.im * g.h3 * sgn};
    }
#pragma unroll
  for (int i = 0; i < MS; ++i)
#pragma unroll
    for (int j = 0; j < MS; ++j) {  // W C, A = 1 - rho W C
      cpx<double> a = {0.0, 0.0};
#pragma unroll
      for (int q = 0; q < MS; ++q) a = cadd(a, cscale(c[pr(q, j)], w[pr(i, q)]));
      B[i][j] = a;
      A[i][j] = cpx<double>{(i == j ? 1.0 : 0.0) - g.rho * a.re, -g.rho * a.im};
    }
#pragma unroll
  for (int i = 0; i < MS; ++i) {  // B = W C W, row by row
    cpx<double> row[MS];
#pragma unroll
    for (int j = 0; j < MS; ++j) row[j] = B[i][j];
#pragma unroll
    for (int j = 0; j < MS; ++j) {
      cpx<double> b = {0.0, 0.0};
#pragma unroll
      for (int q = 0; q < MS; ++q) b = cadd(b, cscale(row[q], w[pr(q, j)]));
      B[i][j] = b;
    }
  }
  // Gaussian elimination with partial pivoting, A X = B
#pragma unroll
  for (int col = 0; col < MS; ++col) {
    int piv = col;
    double best = A[col][col].re * A[col][col].re + A[col][col].im * A[col][col].im;
#pragma unroll
    for (int r = col + 1; r < MS; ++r) {
      const double a2 = A[r][col].re * A[r][col].re + A[r][col].im * A[r][col].im;
      if (a2 > best) { best = a2; piv = r; }
    }
#pragma unroll
    for (int r = col + 1; r < MS; ++r) {
      const bool sw = piv == r;
#pragma unroll
      for (int q = 0; q < MS; ++q) {
        const cpx<double> a0 = A[col][q], a1 = A[r][q], b0 = B[col][q], b1 = B[r][q];
        A[col][q] = {sw ? a1.re : a0.re, sw ? a1.im : a0.im};
        A[r][q] = {sw ? a0.re : a1.re, sw ? a0.im : a1.im};
        B[col][q] = {sw ? b1.re : b0.re, sw ? b1.im : b0.im};
        B[r][q] = {sw ? b0.re : b1.re, sw ? b0.im : b1.im};
      }
    }
    const double den = A[col][col].re * A[col][col].re + A[col][col].im * A[col][col].im;
    const cpx<double> inv = {A[col][col].re / den, -A[col][col].im / den};
#pragma unroll
    for (int r = col + 1; r < MS; ++r) {
      const cpx<double> f = cmul(A[r][col], inv);
#pragma unroll
      for (int q = col + 1; q < MS; ++q) A[r][q] = csub(A[r][q], cmul(f, A[col][q]));
#pragma unroll
      for (int q = 0; q < MS; ++q) B[r][q] = csub(B[r][q], cmul(f, B[col][q]));
    }
    A[col][col] = inv;  // 1 / pivot, for the back substitution
  }
#pragma unroll
  for (int col = MS - 1; col >= 0; --col)
#pragma unroll
    for (int q = 0; q < MS; ++q) {
      cpx<double> x = B[col][q];
#pragma unroll
      for (int r = col + 1; r < MS; ++r) x = csub(x, cmul(A[col][r], B[r][q]));
      B[col][q] = cmul(x, A[col][col]);
    }
#pragma unroll
  for (int i = 0; i < MS; ++i)
#pragma unroll
    for (int j = 0; j <= i; ++j) {  // T = ((X - C) - beta q_i q_j U) s / L^3
      cpx<double>& v = c[pr(i, j)];
      v = cpx<double>{((B[i][j].re - v.re) - g.beta * (g.q[i] * g.q[j]) * U) * sgn * g.inv_L3,
                      (B[i][j].im - v.im) * sgn * g.inv_L3};
    }
}

// --------------------------- 3b. zstar with the spectra held in registers
// Mode 3: forward z FFTs only; mode 4: inverse z FFTs only.
// The solute residual's k-space step (modes 0-7 of zstar, special 0) for a
// compile-time site count MS: the z lines of one site at a time pass
// through LDS (LINES * N2 points, interleaved), and each thread keeps its PPT
// points of all MS sites in registers for the contraction.  LDS per
// workgroup is 1/MS of zstar's, so a 128-byte row of kx columns (16 FP32
// or 8 FP64) fits at high occupancy.  Same arithmetic as zstar, point by
// point.  1D grid: the Nyquist blocks of every solute, then the tiles (below).
// OZ > 0 (FP64, special 1): the solvent-solvent step of OZ sites instead,
// MS = OZ (OZ + 1) / 2 pairs (oz_point).  zstar's oz_pairs keeps its matrices
// in scratch (their loops run to a run-time site count) and took 60% of a
// three-site pass: 142 us at 64^3, here 25 us (43 MB of spectra and tables).
template <typename T, int N2>
constexpr int zreg_lines() {
  int L = 128 / (int)sizeof(cpx<T>);
  const int pmax = sizeof(T) == 4 ? 8 : 4;  // points per thread per site
  while (L > 2 && (N2 * L + NT - 1) / NT > pmax) L /= 2;
  return L;
}

template <typename T, int N2, int LINES, int MS, int NTZ = NT, int OZ = 0>
__global__ void __launch_bounds__(NTZ)
zstar_reg(const SoluteDesc* __restrict__ sd, GridArgs g, const cpx<T>* __restrict__ tw,
          const T* __restrict__ chi3, const T* __restrict__ tau3) {
  constexpr int PTS = N2 * LINES;
  constexpr int PPT = (PTS + NTZ - 1) / NTZ;
  __shared__ cpx<T> lds[PTS];  // interleaved: point z of line l at z * LINES + l
  __shared__ cpx<T> stw[N2];   // the twiddles
  // Block order of the 1D grid.  First the Nyquist blocks of a split launch
  // (nyq: lines are LINES rows ky of the column kx = N0/2), whose scattered
  // accesses then run beside the tiles instead of after them; a launch of
  // their own took 98 us beside 174 us at 192^3 with 5 sites and 27 beside
  // 285 us at 24 x 128^3 (FP32); the one launch 192 and 295.  Then the tiles:
  // zorder 2: consecutive blocks go to the XCDs in
  // turn, and each XCD walks all solutes of one (ky, kx tile) before the
  // next, so the tile's chi and tau stay in that XCD's L2 for every solute.
  // zorder 3: XCD x owns the row pairs ky, N1 - ky with ky = x (mod 8), which
  // share their tables (143 -> 141 us at 192^3 with 5 sites, 26 -> 25.4 at 96^3
  // in FP64, against rows in order), and walks every
  // solute of a row, the row's kx tiles back to back, so each z line's
  // columns are read by neighbouring workgroups at once (whole rows of the
  // z planes instead of one tile's 128 bytes) and the row's chi and tau
  // stay in the XCD's L2 across solutes.
  // zorder 1: kx tile fastest, then ky (in the same pairs), then the solute; zorder 0: solute
  // fastest, then the kx tile.
  int b, tile, ky;
  const int nnyq = g.nyqb * g.zB;
  const bool nyq = (int)blockIdx.x < nnyq;
  if (nyq) {
    b = blockIdx.x / g.nyqb;
    tile = 0;
    ky = (blockIdx.x - b * g.nyqb) * LINES;
  } else {
    const int lin = blockIdx.x - nnyq, xcd = lin & 7, slot = lin >> 3;
    if (g.zorder == 3) {
      tile = slot % g.ztiles;
      b = (slot / g.ztiles) % g.zB;
      const int q = slot / (g.ztiles * g.zB), p = (q >> 1) * 8 + xcd;
      ky = q & 1 ? (p ? g.N1 - p : g.N1 / 2) : p;
    } else if (g.zorder == 2) {
      const int gt = (slot / g.zB) * 8 + xcd;  // global tile, ky-major
      b = slot - (slot / g.zB) * g.zB;
      tile = gt % g.ztiles;
      ky = gt / g.ztiles;
    } else if (g.zorder == 1) {
      tile = lin % g.ztiles;
      const int q = (lin / g.ztiles) % g.N1;
      ky = q & 1 ? g.N1 - (q + 1) / 2 : q / 2;
      b = lin / (g.ztiles * g.N1);
    } else {
      b = lin % g.zB;
      tile = (lin / g.zB) % g.ztiles;
      ky = lin / (g.zB * g.ztiles);
    }
  }
  const SoluteDesc& d = sd[b];
  if (!d.active) return;
  // nyq: lines are the rows y0 + l of the Nyquist column kx = N0/2;
  // otherwise the kx columns kx0 + l of row y.
  const int y = ky;
  const int kx0 = nyq ? g.NX - 1 : tile * LINES;
  // element offsets below 2^32 bytes from per-workgroup bases (at32): the
  // tables and Fs from their starts, W from its site's
  const int zs = g.N1 * g.NH;         // z stride
  const int ls = nyq ? g.NH : 1;      // line stride
  const int base = y * g.NH + kx0;
  // W: the same index unless ylay (y-major rows, compact Nyquist column)
  int wz = zs, wl = ls;
  int64_t wsite = g.K;
  cpx<T>* W = static_cast<cpx<T>*>(d.W) + base;
  if (g.ylay) {
    if (nyq) {
      W = static_cast<cpx<T>*>(d.W) + g.m * g.K + y;
      wz = g.N1;
      wl = 1;
      wsite = (int64_t)g.N1 * g.N2;
    } else {
      W = static_cast<cpx<T>*>(d.W) + (int64_t)y * g.N2 * g.NH + kx0;
      wz = g.NH;
    }
  }
  // the tables: z-major rows, and the Nyquist column of each compact behind
  // them all, (z, ky) at z TN1 + ky, where a Nyquist block's lines are
  // contiguous (8 bytes of each 128-byte line otherwise: at B = 1 such a
  // block was the pass's last, 50 us against 33 for the rows at 96^3 in FP64)
  constexpr int NTAB = OZ > 0 ? MS : MS * (MS + 1) / 2;  // chi3's tables
  const int64_t tsite = nyq ? (int64_t)g.TN1 * g.TN2 : g.KT;
  const T* chit = nyq ? chi3 + NTAB * g.KT : chi3;
  const T* taut = nyq ? tau3 + MS * g.KT : tau3;
  const int tbase = nyq ? 0 : table_row(g, y) * g.NH + kx0, tz = nyq ? g.TN1 : g.TN1 * g.NH;
  // point (z, l) of the tile in the tables
  auto tpoint = [&](int z, int l) {
    return (uint32_t)(tbase + table_plane(g, z) * tz + (nyq ? table_row(g, y + l) : l));
  };
  const int nl = nyq ? min(LINES, g.N1 - y)  // valid lines
                     : min(LINES, (g.nyqb ? g.NX - 1 : g.NX) - kx0);
  const int tid = threadIdx.x;
  for (int i = tid; i < N2; i += NTZ) stw[i] = tw[i];
  cpx<T> c[MS][PPT];
  // every site's loads first, staged in its registers of c (its FFT result
  // lands there after its pass), so the later sites' loads overlap the
  // earlier sites' transforms; a partial tile reads only its valid lines
#pragma unroll
  for (int s = 0; s < MS; ++s) {
#pragma unroll
    for (int p = 0; p < PPT; ++p) {
      const int e = tid + p * NTZ;
      if (PPT * NTZ == PTS || e < PTS) {
        const int z = e / LINES, l = e - z * LINES;
        c[s][p] = (nl == LINES || l < nl) ? ldc(at32(W + s * wsite, (uint32_t)(z * wz + l * wl)))
                                          : cpx<T>{T(0), T(0)};
      }
    }
  }
  // RR: the z transforms keep the thread's points in registers (its PPT
  // points of line l are the inputs of one first-stage butterfly and the
  // outputs of its last-stage butterflies, fft_lines_rr); otherwise they
  // pass through LDS whole (fft_lines_il).
  constexpr bool RR = rr_ok(N2, LINES, NTZ) && PPT * NTZ == PTS;
#pragma unroll
  for (int s = 0; s < MS; ++s) {
    cpx<T>* Ws = W + s * wsite;
    if constexpr (RR) {
      if (d.mode == 4) continue;  // inverse only: the loaded spectrum goes to the inverse pass
      fft_lines_rr<T, N2, LINES, NTZ, false>(c[s], lds, nl, stw);
      if (d.mode == 3) {  // forward spectrum only
#pragma unroll
        for (int p = 0; p < PPT; ++p) {
          const int e = tid + p * NTZ;
          const int z = e / LINES, l = e - z * LINES;
          if (l < nl) stc(at32(Ws, (uint32_t)(z * wz + l * wl)), c[s][p]);
        }
      }
      continue;
    }
    {
      cpx<T>* v = c[s];
      if (d.mode == 4) continue;  // inverse only: the loaded spectrum goes to the inverse pass
#pragma unroll
      for (int p = 0; p < PPT; ++p) {
        const int e = tid + p * NTZ;
        if (PPT * NTZ == PTS || e < PTS) lds[e] = ((e & (LINES - 1)) < nl) ? v[p] : cpx<T>{T(0), T(0)};
      }
    }
    __syncthreads();
    fft_lines_il<T, N2, LINES, NTZ, false>(lds, nl, stw);
#pragma unroll
    for (int p = 0; p < PPT; ++p) {
      const int e = tid + p * NTZ;
      if (PPT * NTZ == PTS || e < PTS) {
        const int z = e / LINES, l = e - z * LINES;
        c[s][p] = lds[e];
        if (d.mode == 3 && l < nl) stc(at32(Ws, (uint32_t)(z * wz + l * wl)), c[s][p]);  // forward spectrum only
      }
    }
    __syncthreads();
  }
  if (d.mode == 3) return;
  const bool linear = d.mode != 0;  // chi convolution only
  const cpx<T>* Fs = static_cast<const cpx<T>*>(d.Fs);
  if constexpr (OZ > 0) {
    static_assert(MS == OZ * (OZ + 1) / 2 && sizeof(T) == 8, "site pairs, FP64");
#pragma unroll
    for (int p = 0; p < PPT; ++p) {
      const int e = tid + p * NTZ;
      const int z = e / LINES, l = e - z * LINES;
      if (d.mode == 4 || !(PPT * NTZ == PTS || e < PTS) || l >= nl) continue;
      const uint32_t kk = tpoint(z, l);
      const int iz = (z <= N2 / 2) ? z : z - N2, ix = nyq ? kx0 : kx0 + l;
      const int yl = nyq ? y + l : y;
      const int iy = (yl <= g.N1 / 2) ? yl : yl - g.N1;
      const double sgn = ((ix + iy + iz) & 1) ? -1.0 : 1.0;
      // the unit long-range Coulomb as zstar forms it
      const double kabs = sqrt(kmag2(ix * g.dkx, iy * g.dky, iz * g.dkz));
      const double k2 = kabs * kabs;
      const double U = k2 == 0.0 ? 0.0
          : (4 * M_PI * EPSILON0INV) * exp(-k2 / (4 * G_COULOMB * G_COULOMB)) / k2;
      double w[MS];
      cpx<double> v[MS];
#pragma unroll
      for (int i = 0; i < OZ; ++i)
#pragma unroll
        for (int j = 0; j <= i; ++j) {
          const int q = i * (i + 1) / 2 + j;
          w[q] = i == j ? 1.0 : gld(at32(chit + q * tsite, kk));
          v[q] = c[q][p];
        }
      oz_point<OZ>(v, w, g, sgn, U);
#pragma unroll
      for (int q = 0; q < MS; ++q) c[q][p] = v[q];
    }
  } else
#pragma unroll
  for (int p = 0; p < PPT; ++p) {
    const int e = tid + p * NTZ;
    if (d.mode == 4 || !(PPT * NTZ == PTS || e < PTS)) continue;
    const int z = e / LINES, l = e - z * LINES;
    if (l >= nl) continue;
    const uint32_t kk = tpoint(z, l);  // this point in the tables
    cpx<T> fs = {T(0), T(0)};
    if (!linear)
      fs = ldc(at32(Fs, nyq ? (uint32_t)(g.K + z * g.N1 + y + l)
                            : (uint32_t)fs_index<T>(g, z, y, kx0 + l)));
    cpx<T> uc = {T(0), T(0)};
    if (!g.renorm && !linear) {
      // u_c(k) = 4 pi eps0^-1 exp(-k^2/4G^2)/k^2 F(k) s(k), 0 at k = 0
      // (bgy3d-force.h:140-147, bgy3d-solutes.c:767-792).
      const int iz = (z <= N2 / 2) ? z : z - N2;
      const int yl = nyq ? y + l : y;
      const int iy = (yl <= g.N1 / 2) ? yl : yl - g.N1;
      const double k2 = kmag2((nyq ? kx0 : kx0 + l) * g.dkx, iy * g.dky, iz * g.dkz);
      const double shape = (k2 == 0.0) ? 0.0
          : (4 * M_PI * EPSILON0INV) * exp(-k2 / (4 * G_COULOMB * G_COULOMB)) / k2;
      uc = cscale(fs, T(shape));
#pragma unroll
      for (int s = 0; s < MS; ++s)  // h^3 C_j - beta q_j u_c  (hnc3d.c:1226-1227)
        c[s][p] = csub(cscale(c[s][p], T(g.h3)), cscale(uc, T(g.beta * g.q[s])));
    }
    T chi[MS * (MS + 1) / 2];
#pragma unroll
    for (int q = 0; q < MS * (MS + 1) / 2; ++q) chi[q] = gld(at32(chit + q * tsite, kk));
    cpx<T> out[MS];
#pragma unroll
    for (int i = 0; i < MS; ++i) {
      cpx<T> acc = {T(0), T(0)};
#pragma unroll
      for (int j = 0; j < MS; ++j) {  // sum_j S_ij sig_j c_j / sig_i (sig = 1: one density)
        const T x = chi[(i >= j) ? i * (i + 1) / 2 + j : j * (j + 1) / 2 + i] * T(g.sig[j]);
        acc.re += x * c[j][p].re;
        acc.im += x * c[j][p].im;
      }
      acc = cscale(acc, T(1.0 / g.sig[i]));
      if (linear) {
        out[i] = cscale(acc, T(g.a_scale));
      } else if (g.renorm) {
        // (h^3/L^3) sum_j chi_ij C_j - (beta/eps0/L^3) tau_i F s  (hnc3d.c:1245-1268)
        const T tau = gld(at32(taut + i * tsite, kk)) * T(g.tau_scale);
        out[i] = csub(cscale(acc, T(g.a_scale)), cscale(fs, tau));
      } else {
        out[i] = cscale(csub(acc, cscale(uc, T(g.beta * g.q[i]))), T(g.inv_L3));
      }
    }
#pragma unroll
    for (int i = 0; i < MS; ++i) c[i][p] = out[i];
  }
#pragma unroll
  for (int s = 0; s < MS; ++s) {
    cpx<T>* Ws = W + s * wsite;
    if constexpr (RR) {
      fft_lines_rr<T, N2, LINES, NTZ, true>(c[s], lds, nl, stw);
#pragma unroll
      for (int p = 0; p < PPT; ++p) {
        const int e = tid + p * NTZ;
        const int z = e / LINES, l = e - z * LINES;
        if (l < nl) stc(at32(Ws, (uint32_t)(z * wz + l * wl)), c[s][p]);
      }
      continue;
    }
#pragma unroll
    for (int p = 0; p < PPT; ++p) {
      const int e = tid + p * NTZ;
      if (PPT * NTZ == PTS || e < PTS) lds[e] = c[s][p];
    }
    __syncthreads();
    fft_lines_il<T, N2, LINES, NTZ, true>(lds, nl, stw);
#pragma unroll
    for (int p = 0; p < PPT; ++p) {
      const int e = tid + p * NTZ;
      if (PPT * NTZ == PTS || e < PTS) {
        const int z = e / LINES, l = e - z * LINES;
        if (l < nl) stc(at32(Ws, (uint32_t)(z * wz + l * wl)), lds[e]);
      }
    }
    __syncthreads();
  }
}

// -------------------------------------- 5. x c2r fused with the residual
// t' = c2r(...), r = t' - t, u = t + lam r, and per workgroup the partial
// max|r|, sum r^2 and dots <r, r_j> with the history (MDIIS Gram row), to
// part[q * nparts + site * gridDim.x + blockIdx.x], nparts = m gridDim.x: the
// partials of one quantity together, as reduce_resid reads them.  Grid as
// closure_r2c_x.
template <typename T, int N0, int H>
__global__ void __launch_bounds__(NT)
c2r_x_resid(const SoluteDesc* __restrict__ sd, GridArgs g,
            const cpx<T>* __restrict__ tw_half, const cpx<T>* __restrict__ tw_full) {
  constexpr int M = N0 / 2;
  constexpr int ROWS = rows_for(M);
  __shared__ cpx<T> xb[ROWS * (M + 1)];
  constexpr int LSM = lstride_for(M);
  __shared__ cpx<T> zb[ROWS * LSM];
  __shared__ double red[NPART][NT / 64];
  const SoluteDesc& d = sd[blockIdx.z];
  if (!d.active) return;
  // the twiddles in LDS: [M of the rows][M + 1 of the split]
  __shared__ cpx<T> stw[2 * M + 1];
  for (int i = threadIdx.x; i < 2 * M + 1; i += NT) stw[i] = i < M ? tw_half[i] : tw_full[i - M];
  const int site = blockIdx.y;
  const int nrows = g.N1 * g.N2;
  const int row0 = blockIdx.x * ROWS;
  const int vrows = min(ROWS, nrows - row0);
  const cpx<T>* W = static_cast<const cpx<T>*>(d.W) + site * g.K + (int64_t)row0 * g.NH;
  const int64_t off = site * g.P + (int64_t)row0 * N0;
  constexpr int VW = Vec16<T>::W;
  {
    // all loads first; rows past the last one read the last row's address
    // and are zeroed
    constexpr int PTS = ROWS * (M + 1), PT = (PTS + NT - 1) / NT;
    cpx<T> v[PT];
#pragma unroll
    for (int p = 0; p < PT; ++p) {
      const int e = threadIdx.x + p * NT;
      if (PT * NT == PTS || e < PTS) {
        const int row = e / (M + 1);
        const int k = e - row * (M + 1);
        v[p] = ldc(W + min(row, vrows - 1) * g.NH + k);
      }
    }
#pragma unroll
    for (int p = 0; p < PT; ++p) {
      const int e = threadIdx.x + p * NT;
      if (PT * NT == PTS || e < PTS) xb[e] = (e / (M + 1) < vrows) ? v[p] : cpx<T>{T(0), T(0)};
    }
  }
  __syncthreads();
  for (int e = threadIdx.x; e < ROWS * M; e += NT) {
    const int row = e / M;
    const int k = e - row * M;
    cpx<T> xk = xb[row * (M + 1) + k];
    cpx<T> xm = xb[row * (M + 1) + (M - k)];
    if (k == 0) { xk.im = T(0); xm.im = T(0); }  // c2r ignores Im at DC / Nyquist
    const cpx<T> a = cadd(xk, cconj(xm));
    const cpx<T> b = csub(xk, cconj(xm));
    const cpx<T> ib = rot90<T, true>(cmulc(b, stw[M + k]));  // i e^{+2 pi i k/N} b
    zb[row * LSM + lpos(k)] = cadd(a, ib);
  }
  __syncthreads();
  fft_lines<T, M, ROWS, NT, true>(zb, LSM, vrows, stw);
  const T* __restrict__ t = static_cast<const T*>(d.t) + off;
  T* __restrict__ r = static_cast<T*>(d.r) + off;  // (BF16 slots: addressed in e below)
  T* __restrict__ un = d.unew ? static_cast<T*>(d.unew) + off : nullptr;  // null: no u
  const bool r16 = d.r16 != 0 || d.r8 != 0;  // FP32 phase: r history in BF16 or FP8
  const int nd = d.ndot;
  const T lam = T(d.lam);
  double mx = 0.0, ss = 0.0;
  double dot[H];
#pragma unroll
  for (int j = 0; j < H; ++j) dot[j] = 0.0;
  const int mode = d.mode;
  // one vector of VW points at e: t, F(t_b) (mode 5) and the history r_j
  // (rhj(j), unpacked on use)
  auto point = [&](int e, const Vec16<T>& tv, const Vec16<T>& f, auto&& rhj) {
    Vec16<T> uo;  // u16: the u the new one replaces (loaded first, used last)
    if constexpr (sizeof(T) == 4)
      if (d.u16 && un) uo = d.plain ? tv : ld16(un + e);
    Vec16<T> z;  // t' at points e.. of row e / N0: z_n = t'_{2n} + i t'_{2n+1}
    {
      const cpx<T>* zrow = zb + (e / N0) * LSM;
      const int n0 = (e % N0) / 2;
#pragma unroll
      for (int h = 0; h < VW / 2; ++h) {
        const cpx<T> zz = zrow[lpos(n0 + h)];
        z.v[2 * h] = zz.re;
        z.v[2 * h + 1] = zz.im;
      }
    }
    Vec16<T> rv, uv;
    if (mode == 5) {  // defect correction: F(t_b) + K dc - delta
#pragma unroll
      for (int k = 0; k < VW; ++k) rv.v[k] = f.v[k] + z.v[k] - tv.v[k];
    } else {
#pragma unroll
      for (int k = 0; k < VW; ++k) {
        if (mode == 0 || mode == 6) rv.v[k] = z.v[k] - tv.v[k];                     // F(t), J v
        else if (mode == 1)                                                          // adjoint
          rv.v[k] = T(gld(d.dt + off + e + k)) * z.v[k] + T(gld(d.gv + off + e + k)) - tv.v[k];
        else rv.v[k] = z.v[k];                                                       // K t
      }
    }
#pragma unroll
    for (int k = 0; k < VW; ++k) uv.v[k] = tv.v[k] + lam * rv.v[k];
    if (un) {
      if constexpr (sizeof(T) == 4) {
        if (d.u16) {  // the difference from the u it replaces, in BF16
          Vec16<T> du;
#pragma unroll
          for (int k = 0; k < VW; ++k) du.v[k] = uv.v[k] - uo.v[k];
          stbf4(static_cast<uint16_t*>(d.dnew) + off + e, to_bf4(du));
        }
      }
      st16(un + e, uv);
    }
#pragma unroll
    for (int k = 0; k < VW; ++k) mx = fmax(mx, fabs((double)rv.v[k]));
    bool stored = false;
    if constexpr (sizeof(T) == 4) {
      if (r16) {  // store rounded, and form the Gram row from the rounded values
        rv = st_hist(d, off + e, rv);
        stored = true;
      }
    }
    if (!stored) st16(r + e, rv);
    // products of one vector in the working type, sums across vectors in FP64
    {
      T s2 = T(0);
#pragma unroll
      for (int k = 0; k < VW; ++k) s2 += rv.v[k] * rv.v[k];
      ss += (double)s2;
#pragma unroll
      for (int j = 0; j < H; ++j)
        if (j < nd) {
          const Vec16<T> x = rhj(j);
          T pj = T(0);
#pragma unroll
          for (int k = 0; k < VW; ++k) pj += rv.v[k] * x.v[k];
          dot[j] += (double)pj;
        }
    }
  };
  bool done = false;
  if constexpr (sizeof(T) == 4) {
    if (r16) {
      // the FP32 phase, bound by its 30 bytes of streams per point: two
      // vectors per step, their streams in flight together, the history
      // kept packed (88 VGPRs at 8 slots, 5 waves per SIMD).  Loading the
      // streams before the inverse FFT held 139 and, at N0 = 3 2^k, ran out
      // of threads: 377 us at 192^3 with 5 sites, this way 246 (4.3 TB/s).
      for (int e0 = threadIdx.x * VW; e0 < vrows * N0; e0 += 2 * NT * VW) {
        Vec16<T> tv[2], f[2];
        BF4 rb[2][H];
#pragma unroll
        for (int q = 0; q < 2; ++q) {
          const int e = e0 + q * NT * VW;
          if (e >= vrows * N0) continue;
          tv[q] = ld16(t + e);
          if (mode == 5) f[q] = ld16(static_cast<const T*>(d.fb) + off + e);
#pragma unroll
          for (int j = 0; j < H; ++j)
            if (j < nd) rb[q][j] = ld_hist(d, d.rh[j], off + e);
        }
#pragma unroll
        for (int q = 0; q < 2; ++q) {
          const int e = e0 + q * NT * VW;
          if (e >= vrows * N0) continue;
          point(e, tv[q], f[q], [&](int j) { return un_hist(d, j, rb[q][j]); });
        }
      }
      done = true;
    }
  }
  if (!done) {
    for (int e = threadIdx.x * VW; e < vrows * N0; e += NT * VW) {
      const Vec16<T> tv = ld16(t + e);
      Vec16<T> f;  // F(t_b), defect correction
      if (mode == 5) f = ld16(static_cast<const T*>(d.fb) + off + e);
      Vec16<T> rh[H];
#pragma unroll
      for (int j = 0; j < H; ++j)
        if (j < nd) rh[j] = ld16(static_cast<const T*>(d.rh[j]) + off + e);
      point(e, tv, f, [&](int j) { return rh[j]; });
    }
  }
  const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
  mx = warp_max(mx);
  ss = warp_sum(ss);
  if (lane == 0) { red[0][w] = mx; red[1][w] = ss; }
#pragma unroll
  for (int j = 0; j < H; ++j) {
    if (j < nd) {
      const double s = warp_sum(dot[j]);
      if (lane == 0) red[2 + j][w] = s;
    }
  }
  __syncthreads();
  if (threadIdx.x < 2 + nd) {
    const int q = threadIdx.x;
    double a = red[q][0];
    for (int i = 1; i < NT / 64; ++i) a = (q == 0) ? fmax(a, red[q][i]) : a + red[q][i];
    gst(d.part + (int64_t)q * (gridDim.x * gridDim.y) + site * gridDim.x + blockIdx.x, a);
  }
}

// ----------------------------------- 1' and 5'. the xy-plane pair
// The residual in three launches: closure_r2c_xy, zstar, c2r_xy_resid.
// A workgroup owns one z plane of one site of one solute: N1 rows of N0
// points, whose half spectrum (N1 rows of N0/2 + 1 bins, 66.5 KB in FP32
// at 128^2) stays in LDS between the x and the y transforms, so the y pass
// of the five-launch chain costs no HBM traffic.  Rows of the plane are at
// stride LS = N0/2 + 1 in LDS; the row FFTs run on the first N0/2 points of
// each row, the column FFTs on all N0/2 + 1 columns.
// Threads of a plane workgroup: two or more vectors each, so that a small
// plane's workgroup leaves room for others (24 x 48^3 in FP32 208 us per pass
// with 512 threads, 184 with 256; 24 x 32^3 84 and 61 with 128).
template <typename T, int N0, int N1>
constexpr int plane_threads() {
  constexpr int vectors = N0 * N1 * (int)sizeof(T) / 16;
  return vectors >= 1024 ? 512 : vectors >= 512 ? 256 : 128;
}

// t, c = closure(beta v, t) as closure_r2c_x over the plane, the N0-point
// r2c of every row (N0/2-point FFT of z_n = c_2n + i c_2n+1 and the split,
// in place: bins k and N0/2 - k from Z_k and Z_{N0/2-k}), then the c2c of
// every kx column along y; the plane's rows [y][kx] go to W.
// Grid: x = z plane (N2), y = site, z = solute.
template <typename T, int N0, int N1, int H>
__global__ void __launch_bounds__((plane_threads<T, N0, N1>()))
closure_r2c_xy(const SoluteDesc* __restrict__ sd, GridArgs g, const cpx<T>* __restrict__ tw_half,
               const cpx<T>* __restrict__ tw_full) {
  constexpr int NTP = plane_threads<T, N0, N1>();
  constexpr int M = N0 / 2, LS = M + 1, PLANE = N0 * N1, HP = M / 2 + 1;
  constexpr int VW = Vec16<T>::W;
  static_assert(PLANE % VW == 0, "whole vectors");
  constexpr bool WHOLE = PLANE % (2 * NTP * VW) == 0;  // batches of two vectors
  __shared__ cpx<T> lds[N1 * LS];
  const SoluteDesc& d = sd[blockIdx.z];
  if (!d.active) return;
  const int site = blockIdx.y, z = blockIdx.x;
  const int64_t off = site * g.P + (int64_t)z * PLANE;
  T* __restrict__ t = static_cast<T*>(d.t) + off;
  const T* __restrict__ bv = static_cast<const T*>(d.bv) + off;
  // the twiddles in LDS: [N0/2 of the rows][N0 of the split and the columns]
  static_assert(N0 == N1, "one table for both");
  __shared__ cpx<T> stw[M + N0];
  for (int i = threadIdx.x; i < M + N0; i += NTP) stw[i] = i < M ? tw_half[i] : tw_full[i - M];
  // two vectors per step, so that both vectors' streams are in flight together
  for (int e0 = threadIdx.x * VW; e0 < PLANE; e0 += 2 * NTP * VW) {
    Vec16<T> c[2];
#pragma unroll
    for (int q = 0; q < 2; ++q)
      if (WHOLE || e0 + q * NTP * VW < PLANE)
        c[q] = closure_vec<T, H>(d, g, off, e0 + q * NTP * VW, t, bv);
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      const int e = e0 + q * NTP * VW;
      if (!WHOLE && e >= PLANE) continue;
      cpx<T>* zrow = lds + (e / N0) * LS;
      const int n0 = (e % N0) / 2;
#pragma unroll
      for (int h = 0; h < VW / 2; ++h) zrow[n0 + h] = cpx<T>{c[q].v[2 * h], c[q].v[2 * h + 1]};
    }
  }
  __syncthreads();
  fft_lines<T, M, N1, NTP, false>(lds, LS, N1, stw);
  for (int e = threadIdx.x; e < N1 * HP; e += NTP) {
    const int row = e / HP, k = e - row * HP;
    cpx<T>* r = lds + row * LS;
    const cpx<T> a = r[k], b = r[k == 0 ? 0 : M - k];  // Z_k, Z_{M-k}
    // bin kk from Z_kk and Z_{M-kk}: (Z + conj Z') / 2 - i w_kk (Z - conj Z') / 2
    auto bin = [&](int kk, cpx<T> zk, cpx<T> zo) {
      const cpx<T> zm = cconj(zo);
      const cpx<T> sm = cadd(zk, zm);
      const cpx<T> dd = rot90<T, false>(cmul(stw[M + kk], csub(zk, zm)));
      return cpx<T>{T(0.5) * (sm.re + dd.re), T(0.5) * (sm.im + dd.im)};
    };
    if (k == 0) {
      r[0] = bin(0, a, a);
      r[M] = bin(M, a, a);
    } else {
      const cpx<T> xk = bin(k, a, b), xm = bin(M - k, b, a);
      r[k] = xk;
      r[M - k] = xm;
    }
  }
  __syncthreads();
  fft_cols<T, N1, LS, M + 1, NTP, false>(lds, stw + M);
  // y-major rows of M bins, then the Nyquist bins of the plane's rows
  cpx<T>* W = static_cast<cpx<T>*>(d.W) + site * g.K + (int64_t)z * g.NH;
  const int64_t ys = (int64_t)g.N2 * g.NH;
  for (int e = threadIdx.x; e < N1 * M; e += NTP) {
    const int y = e / M, k = e - y * M;
    stc(W + y * ys + k, lds[y * LS + k]);
  }
  cpx<T>* Q = static_cast<cpx<T>*>(d.W) + g.m * g.K + ((int64_t)site * g.N2 + z) * N1;
  for (int y = threadIdx.x; y < N1; y += NTP) stc(Q + y, lds[y * LS + M]);
}

// The inverse: the plane's rows [y][kx] from W, the inverse c2c of every
// column along y, the c2r pre-processing of every row in place (Z_k and
// Z_{N0/2-k} from bins k and N0/2 - k; Im of the DC and Nyquist bins
// dropped, as FFTW's c2r does), the inverse N0/2-point row FFTs, then
// r = t' - t (or the mode's form), u = t + lam r and the partials max|r|,
// sum r^2, <r, r_j> as c2r_x_resid, one partial per plane and quantity at
// part[q * m N2 + site * N2 + z].  Grid as closure_r2c_xy.
template <typename T, int N0, int N1, int H>
__global__ void __launch_bounds__((plane_threads<T, N0, N1>()))
c2r_xy_resid(const SoluteDesc* __restrict__ sd, GridArgs g, const cpx<T>* __restrict__ tw_half,
             const cpx<T>* __restrict__ tw_full) {
  constexpr int NTP = plane_threads<T, N0, N1>();
  constexpr int M = N0 / 2, LS = M + 1, PLANE = N0 * N1, HP = M / 2 + 1;
  constexpr int VW = Vec16<T>::W;
  static_assert(PLANE % VW == 0, "whole vectors");
  constexpr bool WHOLE = PLANE % (2 * NTP * VW) == 0;  // batches of two vectors
  __shared__ cpx<T> lds[N1 * LS];
  __shared__ double red[NPART][NTP / 64];
  const SoluteDesc& d = sd[blockIdx.z];
  if (!d.active) return;
  const int site = blockIdx.y, z = blockIdx.x;
  // the twiddles in LDS: [N0/2 of the rows][N0 of the split and the columns]
  static_assert(N0 == N1, "one table for both");
  __shared__ cpx<T> stw[M + N0];
  for (int i = threadIdx.x; i < M + N0; i += NTP) stw[i] = i < M ? tw_half[i] : tw_full[i - M];
  // the plane's y-major rows of M bins and its Nyquist bins (closure_r2c_xy)
  const cpx<T>* W = static_cast<const cpx<T>*>(d.W) + site * g.K + (int64_t)z * g.NH;
  const cpx<T>* Q = static_cast<const cpx<T>*>(d.W) + g.m * g.K + ((int64_t)site * g.N2 + z) * N1;
  const int64_t ys = (int64_t)g.N2 * g.NH;
  {
    constexpr int PTS = N1 * M, PT = (PTS + NTP - 1) / NTP;
    constexpr int QT = (N1 + NTP - 1) / NTP;
    cpx<T> v[PT], nq[QT];
#pragma unroll
    for (int p = 0; p < PT; ++p) {  // all loads first
      const int e = threadIdx.x + p * NTP;
      if (PT * NTP == PTS || e < PTS) {
        const int y = e / M, k = e - y * M;
        v[p] = ldc(W + y * ys + k);
      }
    }
#pragma unroll
    for (int p = 0; p < QT; ++p) {
      const int y = threadIdx.x + p * NTP;
      if (y < N1) nq[p] = ldc(Q + y);
    }
#pragma unroll
    for (int p = 0; p < PT; ++p) {
      const int e = threadIdx.x + p * NTP;
      if (PT * NTP == PTS || e < PTS) {
        const int y = e / M, k = e - y * M;
        lds[y * LS + k] = v[p];
      }
    }
#pragma unroll
    for (int p = 0; p < QT; ++p) {
      const int y = threadIdx.x + p * NTP;
      if (y < N1) lds[y * LS + M] = nq[p];
    }
  }
  __syncthreads();
  fft_cols<T, N1, LS, M + 1, NTP, true>(lds, stw + M);
  for (int e = threadIdx.x; e < N1 * HP; e += NTP) {
    const int row = e / HP, k = e - row * HP;
    cpx<T>* r = lds + row * LS;
    cpx<T> xk = r[k], xm = r[M - k];  // bins k and M - k (0: DC and Nyquist)
    // Z_kk = (X_kk + conj X_{M-kk}) + i e^{+2 pi i kk/N0} (X_kk - conj X_{M-kk})
    auto pre = [&](int kk, cpx<T> a0, cpx<T> b0) {
      const cpx<T> a = cadd(a0, cconj(b0));
      const cpx<T> b = csub(a0, cconj(b0));
      return cadd(a, rot90<T, true>(cmulc(b, stw[M + kk])));
    };
    if (k == 0) {
      xk.im = T(0);
      xm.im = T(0);
      r[0] = pre(0, xk, xm);
    } else {
      const cpx<T> zk = pre(k, xk, xm), zm = pre(M - k, xm, xk);
      r[k] = zk;
      r[M - k] = zm;
    }
  }
  __syncthreads();
  fft_lines<T, M, N1, NTP, true>(lds, LS, N1, stw);
  const int64_t off = site * g.P + (int64_t)z * PLANE;
  const T* __restrict__ t = static_cast<const T*>(d.t) + off;
  T* __restrict__ r = static_cast<T*>(d.r) + off;  // (BF16 slots: addressed in e below)
  T* __restrict__ un = d.unew ? static_cast<T*>(d.unew) + off : nullptr;  // null: no u
  const bool r16 = d.r16 != 0 || d.r8 != 0;  // FP32 phase: r history in BF16 or FP8
  const int nd = d.ndot;
  const int mode = d.mode;
  const T lam = T(d.lam);
  double mx = 0.0, ss = 0.0;
  double dot[H];
#pragma unroll
  for (int j = 0; j < H; ++j) dot[j] = 0.0;
  // one vector of VW points at e: t' from LDS, the streams t, F(t_b)
  // (mode 5) and the history r_j (rhj(j), unpacked on use)
  auto point = [&](int e, const Vec16<T>& tv, const Vec16<T>& f, auto&& rhj) {
    Vec16<T> uo;  // u16: the u the new one replaces (loaded first, used last)
    if constexpr (sizeof(T) == 4)
      if (d.u16 && un) uo = d.plain ? tv : ld16(un + e);
    Vec16<T> zv;  // t' at points e.. of row e / N0
    {
      const cpx<T>* zrow = lds + (e / N0) * LS;
      const int n0 = (e % N0) / 2;
#pragma unroll
      for (int h = 0; h < VW / 2; ++h) {
        const cpx<T> zz = zrow[n0 + h];
        zv.v[2 * h] = zz.re;
        zv.v[2 * h + 1] = zz.im;
      }
    }
    Vec16<T> rv, uv;
#pragma unroll
    for (int k = 0; k < VW; ++k) {
      if (mode == 5) rv.v[k] = f.v[k] + zv.v[k] - tv.v[k];  // F(t_b) + K dc - delta
      else if (mode == 0 || mode == 6) rv.v[k] = zv.v[k] - tv.v[k];
      else if (mode == 1)
        rv.v[k] = T(gld(d.dt + off + e + k)) * zv.v[k] + T(gld(d.gv + off + e + k)) - tv.v[k];
      else rv.v[k] = zv.v[k];
    }
#pragma unroll
    for (int k = 0; k < VW; ++k) uv.v[k] = tv.v[k] + lam * rv.v[k];
    if (un) {
      if constexpr (sizeof(T) == 4) {
        if (d.u16) {  // the difference from the u it replaces (uo), in BF16
          Vec16<T> du;
#pragma unroll
          for (int k = 0; k < VW; ++k) du.v[k] = uv.v[k] - uo.v[k];
          stbf4(static_cast<uint16_t*>(d.dnew) + off + e, to_bf4(du));
        }
      }
      st16(un + e, uv);
    }
#pragma unroll
    for (int k = 0; k < VW; ++k) mx = fmax(mx, fabs((double)rv.v[k]));
    bool stored = false;
    if constexpr (sizeof(T) == 4) {
      if (r16) {  // store rounded, and form the Gram row from the rounded values
        rv = st_hist(d, off + e, rv);
        stored = true;
      }
    }
    if (!stored) st16(r + e, rv);
    T s2 = T(0);
#pragma unroll
    for (int k = 0; k < VW; ++k) s2 += rv.v[k] * rv.v[k];
    ss += (double)s2;
#pragma unroll
    for (int j = 0; j < H; ++j)
      if (j < nd) {
        const Vec16<T> x = rhj(j);
        T pj = T(0);
#pragma unroll
        for (int k = 0; k < VW; ++k) pj += rv.v[k] * x.v[k];
        dot[j] += (double)pj;
      }
  };
  bool done = false;
  if constexpr (sizeof(T) == 4) {
    if (r16) {
      // BF16 history (the FP32 phase): two vectors per step, their streams
      // in flight together, the history kept packed (two VGPRs per vector)
      for (int e0 = threadIdx.x * VW; e0 < PLANE; e0 += 2 * NTP * VW) {
        Vec16<T> tv[2], f[2];
        BF4 rb[2][H];
#pragma unroll
        for (int q = 0; q < 2; ++q) {
          const int e = e0 + q * NTP * VW;
          if (!WHOLE && e >= PLANE) continue;
          tv[q] = ld16(t + e);
          if (mode == 5) f[q] = ld16(static_cast<const T*>(d.fb) + off + e);
#pragma unroll
          for (int j = 0; j < H; ++j)
            if (j < nd) rb[q][j] = ld_hist(d, d.rh[j], off + e);
        }
#pragma unroll
        for (int q = 0; q < 2; ++q) {
          const int e = e0 + q * NTP * VW;
          if (!WHOLE && e >= PLANE) continue;
          point(e, tv[q], f[q], [&](int j) { return un_hist(d, j, rb[q][j]); });
        }
      }
      done = true;
    }
  }
  if (!done) {
    for (int e = threadIdx.x * VW; e < PLANE; e += NTP * VW) {
      const Vec16<T> tv = ld16(t + e);
      Vec16<T> f;
      if (mode == 5) f = ld16(static_cast<const T*>(d.fb) + off + e);
      Vec16<T> rh[H];
#pragma unroll
      for (int j = 0; j < H; ++j)
        if (j < nd) rh[j] = ld16(static_cast<const T*>(d.rh[j]) + off + e);
      point(e, tv, f, [&](int j) { return rh[j]; });
    }
  }
  const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
  mx = warp_max(mx);
  ss = warp_sum(ss);
  if (lane == 0) { red[0][w] = mx; red[1][w] = ss; }
#pragma unroll
  for (int j = 0; j < H; ++j) {
    if (j < nd) {
      const double s2 = warp_sum(dot[j]);
      if (lane == 0) red[2 + j][w] = s2;
    }
  }
  __syncthreads();
  if (threadIdx.x < 2 + nd) {
    const int q = threadIdx.x;
    double a = red[q][0];
    for (int i = 1; i < NTP / 64; ++i) a = (q == 0) ? fmax(a, red[q][i]) : a + red[q][i];
    gst(d.part + (int64_t)q * (gridDim.x * gridDim.y) + site * gridDim.x + blockIdx.x, a);
  }
}

// The sums of v[0 .. N) over a wavefront.  Halving: at each step a lane keeps
// half of the values, adds its partner's share of them and hands the other
// half over, so N values take about N exchanges instead of 6 N.  Returns true
// in one lane per value, with the value's place in at and its sum in v[0].
template <int N, int MASK = 32>
__device__ __forceinline__ bool wave_sums(double* v, int lane, int& at) {
  static_assert(N <= 2 * MASK || N == 1, "a value per lane at most");
  if constexpr (N == 1) {
    at = 0;
    bool first = true;
#pragma unroll
    for (int k = MASK; k > 0; k >>= 1) {  // lanes that hold the same value
      v[0] += __shfl_xor(v[0], k);
      first = first && !(lane & k);
    }
    return first;
  } else {
    constexpr int H = (N + 1) / 2;
    const bool up = (lane & MASK) != 0;
#pragma unroll
    for (int k = 0; k < H; ++k) {
      const double hi = H + k < N ? v[H + k] : 0.0;
      const double keep = up ? hi : v[k], give = up ? v[k] : hi;
      v[k] = keep + __shfl_xor(give, MASK);
    }
    const bool mine = wave_sums<H, MASK / 2>(v, lane, at);
    if (up) at += H;
    return mine && at < N;
  }
}

// ------------------------------------------- Gram rows of several entries
// <rh[i], rh[j]> for i < nrow, j > i over the residual history, per workgroup
// partials gpart[(i MAX_DIIS + j) * gridDim.x + blockIdx.x].  Bound by its
// ngram streams: each thread holds one 16-byte vector of every entry at a
// time, so one reading of the history serves nrow rows (the dots inside the
// residual kernels read it once per row).  Products of one vector in the
// working type, sums across vectors in FP64, as there.  With short loops the
// sums over the workgroup count too: by halving (wave_sums) instead of one
// value after the other 32^3 took 6.0 instead of 9.8 us, 96^3 with 8 entries in
// FP64 37 instead of 50 (4.6 TB/s), 192^3 with 5 sites and 8 entries in BF16 122
// instead of 135 (4.6 TB/s).
// Grid: x = chunks, y = solute.
template <typename T, int H>
__global__ void __launch_bounds__(NT)
gram_rows(const SoluteDesc* __restrict__ sd, int64_t mP) {
  __shared__ double red[MAX_ROWS * H][NT / 64];
  const SoluteDesc& d = sd[blockIdx.y];
  const int n = d.ngram, nrow = d.nrow;
  if (!d.active || n == 0) return;
  constexpr int VW = Vec16<T>::W;
  double acc[MAX_ROWS][H];
#pragma unroll
  for (int i = 0; i < MAX_ROWS; ++i)
#pragma unroll
    for (int j = 0; j < H; ++j) acc[i][j] = 0.0;
  auto rows = [&](const Vec16<T>* v) {
#pragma unroll
    for (int i = 0; i < MAX_ROWS; ++i)
      if (i < nrow)
#pragma unroll
        for (int j = i + 1; j < H; ++j)
          if (j < n) {
            T p = T(0);
#pragma unroll
            for (int k = 0; k < VW; ++k) p += v[i].v[k] * v[j].v[k];
            acc[i][j] += (double)p;
          }
  };
  const int64_t first = (int64_t)blockIdx.x * NT + threadIdx.x, step = (int64_t)gridDim.x * NT;
  bool done = false;
  if constexpr (sizeof(T) == 4) {
    typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
    typedef __attribute__((address_space(1))) const u32x4 G4;
    if (d.r8) {  // 16 points per 16 bytes, four at a time
      for (int64_t e = first * 16; e < mP; e += step * 16) {
        u32x4 w[H];
#pragma unroll
        for (int j = 0; j < H; ++j)
          if (j < n) w[j] = *(G4*)(static_cast<const uint8_t*>(d.rh[j]) + e);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          Vec16<T> v[H];
#pragma unroll
          for (int j = 0; j < H; ++j)
            if (j < n) v[j] = from_fp8x4(w[j][q], d.rhinv[j]);
          rows(v);
        }
      }
      done = true;
    } else if (d.r16) {  // BF16: 8 points
      for (int64_t e = first * 8; e < mP; e += step * 8) {
        u32x4 w[H];
#pragma unroll
        for (int j = 0; j < H; ++j)
          if (j < n) w[j] = *(G4*)(static_cast<const uint16_t*>(d.rh[j]) + e);
#pragma unroll
        for (int q = 0; q < 2; ++q) {
          Vec16<T> v[H];
#pragma unroll
          for (int j = 0; j < H; ++j)
            if (j < n) {
              v[j].v[0] = bf16_val(w[j][2 * q] & 0xFFFFu);
              v[j].v[1] = bf16_val(w[j][2 * q] >> 16);
              v[j].v[2] = bf16_val(w[j][2 * q + 1] & 0xFFFFu);
              v[j].v[3] = bf16_val(w[j][2 * q + 1] >> 16);
            }
          rows(v);
        }
      }
      done = true;
    }
  }
  if (!done)
    for (int64_t e = first * VW; e < mP; e += step * VW) {
      Vec16<T> v[H];
#pragma unroll
      for (int j = 0; j < H; ++j)
        if (j < n) v[j] = ld16(static_cast<const T*>(d.rh[j]) + e);
      rows(v);
    }
  // the pairs j > i of all rows side by side: wave sums, then over the waves
  constexpr int NP = MAX_ROWS * H - MAX_ROWS * (MAX_ROWS + 1) / 2;
  double pair[NP];
#pragma unroll
  for (int i = 0; i < MAX_ROWS; ++i)
#pragma unroll
    for (int j = i + 1; j < H; ++j) pair[i * H - i * (i + 1) / 2 + j - i - 1] = acc[i][j];
  const int w = threadIdx.x >> 6;
  int at = 0;
  if (wave_sums<NP>(pair, threadIdx.x & 63, at)) red[at][w] = pair[0];
  __syncthreads();
  for (int q = threadIdx.x; q < MAX_ROWS * H; q += NT) {
    const int i = q / H, j = q - i * H;
    if (i >= nrow || j <= i || j >= n) continue;
    const double* r = red[i * H - i * (i + 1) / 2 + j - i - 1];
    double a = r[0];
    for (int k = 1; k < NT / 64; ++k) a += r[k];
    gst(d.gpart + (int64_t)(i * MAX_DIIS + j) * gridDim.x + blockIdx.x, a);
  }
}

}  // namespace rism

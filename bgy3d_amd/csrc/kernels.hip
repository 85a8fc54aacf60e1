// gfx950 kernels around the residual chain (chain.hpp): the norm reduction
// and the MDIIS step, setup, mu and observables, gradients, Newton-Krylov
// helpers, the 3D solvent.
#include "chain.hpp"

namespace rism {

// Chemical-potential density form(x, h, c, cl) (closures.f90:574-612).
__device__ __forceinline__ double form_mu(int method, int order, double x, double h, double c,
                                          double cl) {
  const double base = -c - h * (c + cl) / 2;
  switch (method) {
    case 0: return base + h * h / 2;
    case 1: return (h < 0) ? base + h * h / 2 : base;
    case 2: return base;
    default: {
      if (h < 0) return base + h * h / 2;
      const int m = order + 1;
      double mx = 1, xm = 1;
      for (int k = 1; k <= m; ++k) { mx *= k; xm *= x; }
      return base + (h * h / 2 - xm / mx);
    }
  }
}

// 1D table lookup (interp, bgy3d-vec.c:23-46) at |k|; the index set is
// shared by every table at one k-point.
struct Interp {
  int i, ip, im;
  double off;  // ix - i
};
__device__ __forceinline__ Interp interp_at(double k, double dk, int n) {
  const double ix = k / dk - 0.5;
  int i = (int)(ix + 0.5);
  i = i < 0 ? 0 : (i > n - 1 ? n - 1 : i);  // host guarantees range; clamp never faults
  Interp r;
  r.i = i;
  r.ip = (i < n - 2) ? i + 1 : i;
  r.im = (i > 1) ? i - 1 : i;
  r.off = ix - i;
  return r;
}
__device__ __forceinline__ double interp_eval(const Interp& a, const double* __restrict__ tab) {
  const double d = tab[a.ip] - tab[a.im];
  const double fi = (a.ip - a.im == 2) ? d * 0.5 : d;  // == d / (ip - im), exactly
  return tab[a.i] + fi * a.off;
}

// chi_ij(|k|) - delta_ij and tau_i(|k|) on the 3D k grid, once per batch
// (solute independent; solvent_kernel_rism hnc3d.c:1443-1566 tabulates
// them the same way with vec_ktab), at ky <= N1/2, kz <= N2/2 (table_index).
// Grid: x = chunks of KT.  Writes FP64 and, unless null, FP32 copies,
// [npairs][KT] and [m][KT].
__global__ void __launch_bounds__(NT)
ktab3(GridArgs g, const double* __restrict__ chi_tab, const double* __restrict__ tau_tab,
      double* __restrict__ chi3, float* __restrict__ chi3f, double* __restrict__ tau3,
      float* __restrict__ tau3f) {
  const int np = g.m * (g.m + 1) / 2;
  const int64_t stride = (int64_t)gridDim.x * NT;
  for (int64_t e = blockIdx.x * (int64_t)NT + threadIdx.x; e < g.KT; e += stride) {
    const int x = (int)(e % g.NH);
    if (x >= g.NX) continue;  // row padding
    const int y = (int)((e / g.NH) % g.TN1);
    const int z = (int)(e / ((int64_t)g.NH * g.TN1));
    const double k2 = kmag2(x * g.dkx, y * g.dky, z * g.dkz);
    const Interp ip = interp_at(sqrt(k2), g.dk_tab, g.nrad);
    for (int p = 0; p < np; ++p) {
      const double v = interp_eval(ip, chi_tab + (int64_t)p * g.nrad);
      chi3[p * g.KT + e] = v;
      if (chi3f) chi3f[p * g.KT + e] = (float)v;
    }
    for (int i = 0; i < g.m; ++i) {
      const double v = interp_eval(ip, tau_tab + (int64_t)i * g.nrad);
      tau3[i * g.KT + e] = v;
      if (tau3f) tau3f[i * g.KT + e] = (float)v;
    }
  }
}

// The Nyquist column kx = N0/2 of n tables [n][KT] once more behind them,
// [n][TN2][TN1], as the z pass's Nyquist blocks read it.  Grid: x = chunks of
// TN1 TN2, y = table.
template <typename T>
__global__ void __launch_bounds__(NT)
nyq_tables(GridArgs g, T* __restrict__ tab) {
  const int64_t n12 = (int64_t)g.TN1 * g.TN2;
  const T* src = tab + blockIdx.y * g.KT + (g.NX - 1);
  T* dst = tab + gridDim.y * g.KT + blockIdx.y * n12;
  for (int64_t j = blockIdx.x * (int64_t)NT + threadIdx.x; j < n12; j += (int64_t)gridDim.x * NT)
    dst[j] = src[j * g.NH];
}

// Fixed-order reduction of the residual-workgroup partials of each solute.
// Grid: x = quantity (2 + the history width of the pass at least, or NOUT
// where gram_rows ran, with ngparts partials), y = solute.  out[b * NOUT + q]:
// max|r|, ||r||^2, <r, r_j> or the Gram rows (NOUT); with hout instead
// the bits of the value at hout[2 (b * NOUT + q)] and those bits ^ the
// solute's key behind them, in pinned host memory, where the host polls for
// the pair (each word tells the other's arrival, so no order between the two
// stores is needed, nor the end of the kernel).  One workgroup per
// quantity, whose partials lie together: latency bound (a partial per
// thread or a few), so the quantities run side by side and each thread keeps
// four sums in flight.  One workgroup per solute over rows of NPART took
// 16.6 us at 96^3 (1728 partials) and 181 us at 192^3 with 5 sites (23040),
// 10% and 15% of a pass; this way 4.1 and 12.8 us.
constexpr int NTR = 1024;
__global__ void __launch_bounds__(NTR)
reduce_resid(const SoluteDesc* __restrict__ sd, int nparts, int ngparts, double* __restrict__ out,
             uint64_t* __restrict__ hout) {
  __shared__ double red[NTR / 64];
  const SoluteDesc& d = sd[blockIdx.y];
  const int q = blockIdx.x;
  if (!d.active) return;
  const double* p = d.part + (int64_t)q * nparts;
  if (q >= 2 && d.ngram) {
    const int i = (q - 2) / MAX_DIIS, j = (q - 2) - i * MAX_DIIS;
    if (i >= d.nrow || j <= i || j >= d.ngram) return;
    p = d.gpart + (int64_t)(q - 2) * ngparts;
    nparts = ngparts;
  } else if (q >= 2 + d.ndot) {
    return;
  }
  double acc[4] = {0.0, 0.0, 0.0, 0.0};
  for (int i = threadIdx.x; i < nparts; i += 4 * NTR) {
#pragma unroll
    for (int k = 0; k < 4; ++k)
      if (i + k * NTR < nparts) {
        const double v = gld(p + i + k * NTR);
        acc[k] = q == 0 ? fmax(acc[k], v) : acc[k] + v;
      }
  }
  // fmax drops NaNs; the sums keep them
  const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const double a = q == 0 ? warp_max(fmax(fmax(acc[0], acc[1]), fmax(acc[2], acc[3])))
                          : warp_sum((acc[0] + acc[1]) + (acc[2] + acc[3]));
  if (lane == 0) red[w] = a;
  __syncthreads();
  if (w == 0) {
    const double v = lane < NTR / 64 ? red[lane] : 0.0;
    const double r = q == 0 ? warp_max(v) : warp_sum(v);
    if (lane == 0) {
      const size_t i = (size_t)blockIdx.y * NOUT + q;
      if (hout) {
        const uint64_t bits = (uint64_t)__double_as_longlong(r);
        __hip_atomic_store(hout + 2 * i, bits, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        __hip_atomic_store(hout + 2 * i + 1, bits ^ d.key, __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_SYSTEM);
      } else {
        out[i] = r;
      }
    }
  }
}

// The descriptors of a pass from pinned host memory to the device, as the
// first kernel of the pass's graph.  Grid: x = solute.
constexpr int NTL = 128;
__global__ void __launch_bounds__(NTL)
load_sd(const SoluteDesc* __restrict__ src, SoluteDesc* __restrict__ dst) {
  constexpr int W = sizeof(SoluteDesc) / 8;
  const uint64_t* s = reinterpret_cast<const uint64_t*>(src + blockIdx.x);
  uint64_t* d = reinterpret_cast<uint64_t*>(dst + blockIdx.x);
  for (int i = threadIdx.x; i < W; i += NTL) d[i] = s[i];
}

// v from lane `lane` (the same in every lane of the wavefront) to all lanes.
__device__ __forceinline__ double lane_bcast(double v, int lane) {
  const int lo = __builtin_amdgcn_readlane(__double2loint(v), lane);
  const int hi = __builtin_amdgcn_readlane(__double2hiint(v), lane);
  return __hiloint2double(hi, lo);
}

// MDIIS step of the FP32 defect-correction phase on the device, after the
// norm reduction of a pass (out): one wavefront per solute (grid x =
// solute).  For every solute of the pass it does what the host loop does
// between two passes: the stopping and rebase tests, the new entry into
// the history and its Gram row, the restart test, the DIIS coefficients,
// and the descriptor of the next pass (the combination t = u_newest -
// sum_i (c_0 + .. + c_i) (u_{i+1} - u_i) over the BF16 differences, the
// slot of the new entry, the FP8 scales).  A solute that wants a rebase or
// failed is left inactive for the host; with hold, one whose residual fell
// 1e3 below its base's goes on and is reported ready, and one that reached
// the phase's tolerance is left inactive as parked (the host groups
// rebases).  The DIIS system is solved as
// diis_coefficients solves it on the host, to the bit: LU with partial
// pivoting (first largest pivot), one step of refinement against the
// unfactored matrix, substitutions by columns in the host's order of
// summation, no contraction into fused multiply-adds.
__global__ void __launch_bounds__(64)
mdiis_step(const double* __restrict__ out, MdiisDev* __restrict__ mst,
           SoluteDesc* __restrict__ sd, MdiisStatus* __restrict__ status) {
#pragma clang fp contract(off)
  constexpr int NM = MAX_DIIS + 1;
  constexpr int MD = MAX_DIIS;
  __shared__ MdiisDev s;
  __shared__ double o[NOUT];
  __shared__ double pcol[NM];  // |column| by row position, for the pivot scan
  __shared__ int plane[NM];    // lane holding the row at each position
  __shared__ int ctl[4];       // flag, -, -, LU ok
  const int b = blockIdx.x, l = threadIdx.x;
  SoluteDesc& d = sd[b];
  {  // every load at once: the state, the pass's norms and dots
    const int act = d.active;
    const uint64_t* src = reinterpret_cast<const uint64_t*>(mst + b);
    uint64_t* dst = reinterpret_cast<uint64_t*>(&s);
    for (int i = l; i < (int)(sizeof(MdiisDev) / 8); i += 64) dst[i] = src[i];
    if (l < NOUT) o[l] = out[(size_t)b * NOUT + l];
    if (!act) return;
  }
  __syncthreads();
  const double rinf = o[0], r2 = o[1];
  const bool fin = __builtin_isfinite(rinf) && __builtin_isfinite(r2);
  const int sn = s.slot_new, nd0 = s.ndot;
  if (fin && l < nd0) {  // the new entry after the ones it was dotted with, its Gram row
    const int q = s.dotted[l];
    s.order[l] = q;
    if (s.rows == 1) {
      s.gram[sn * MD + q] = o[2 + l];
      s.gram[q * MD + sn] = o[2 + l];
    }
  }
  if (fin && s.rows == 2 && l <= nd0) {  // or the rows of gram_rows, the newest entry first
    auto entry = [&](int k) { return k == 0 ? sn : s.dotted[nd0 - k]; };
    for (int i = 0; i <= s.pend && i < l; ++i) {
      s.gram[entry(i) * MD + entry(l)] = o[2 + i * MD + l];
      s.gram[entry(l) * MD + entry(i)] = o[2 + i * MD + l];
    }
  }
  __syncthreads();  // rows and pend are read above, written below
  if (l == 0) {
    s.iters++;
    s.iters32++;
    s.resid = rinf;
    if (rinf < s.low) s.low = rinf;
    int flag = 0;
    if (!fin) {
      flag = 2;
    } else {
      if (rinf < 0.7 * s.best32) { s.best32 = rinf; s.stall32 = 0; }
      else if (rinf <= (s.only32 ? 1e-3 : 1e-2 * s.rb_rinf)) { s.stall32++; }
      // with hold: the 1e3 drop only marks the solute ready, and one that
      // reached the phase's tolerance waits without iterating (parked)
      const bool drop = !s.only32 && rinf <= 1e-3 * s.rb_rinf, conv = rinf <= s.tol_half;
      if (s.stall32 >= stall_passes(s.period, s.low) || s.iters32 >= s.max_iter || (!s.hold && (drop || conv)) ||
          (s.only32 && conv))
        flag = 1;
      else if (conv)
        flag = 5;
      else if (drop)
        flag = 4;
      if (s.to16 && s.low <= PULAY_BELOW && (flag == 0 || flag == 4)) flag = flag == 0 ? 6 : 7;
      s.sbase[sn] = s.base;
      s.order[nd0] = sn;
      s.n = nd0 + 1;
      s.gram[sn * MD + sn] = r2;
      // restart when the residual blows up against the best one, or stalls
      if (r2 < s.best) { s.best = r2; s.since_best = 0; } else { s.since_best++; }
      const bool extrap = s.rows != 0;
      s.pend = extrap ? 0 : s.pend + 1;
      s.skipped = extrap ? 0 : s.skipped + 1;
      if (r2 > (extrap ? RESTART_EXTRAP : RESTART_PLAIN) * s.best || s.since_best > 3 * s.D) {
        s.order[0] = sn;
        s.n = 1;
        s.best = r2;
        s.since_best = 0;
        s.pend = s.skipped = 0;
        if (s.low <= PULAY_BELOW) s.period = 1;
      }
      s.picard = !extrap || s.n == 1;
    }
    ctl[0] = flag;
    ctl[3] = 0;
  }
  __syncthreads();
  const int flag = ctl[0];
  if (flag != 2 && !s.picard) {
    // bordered system [G/sc -1; -1 0] [c; l] = [0; -1], sc = max diag G
    const int nh = s.n, n = nh + 1;
    double sc = 0.0;
    for (int i = 0; i < nh; ++i) {
      const double a = fabs(s.gram[s.order[i] * MD + s.order[i]]);
      sc = sc < a ? a : sc;
    }
    if (sc > 0.0 && __builtin_isfinite(sc)) {
      // lane l < n holds row l of the matrix, a (factored in place) and a0
      // (as built); phys is the position the host's row swaps give that
      // row, so position i holds the row of lane la[i] and perm[i] = la[i]
      double a[NM], a0[NM];
      const int oi = l < nh ? s.order[l] : 0;
#pragma unroll
      for (int j = 0; j < NM; ++j) {
        double v = 0.0;
        if (l < n && j < n)
          v = (l < nh && j < nh) ? s.gram[oi * MD + s.order[j]] / sc
                                 : (l == nh && j == nh ? 0.0 : -1.0);
        a[j] = v;
        a0[j] = v;
      }
      int phys = l < n ? l : NM + l;
      bool ok = true;
#pragma unroll
      for (int col = 0; col < NM; ++col) {  // PA = LU, L unit lower
        if (!ok || col >= n) continue;
        // the host's scan over positions col..n-1: the first largest |A|
        if (l < n) {
          pcol[phys] = fabs(a[col]);
          plane[phys] = l;
        }
        __syncthreads();
        double v[NM];
        int pl[NM];
#pragma unroll
        for (int q = col; q < NM; ++q) {
          v[q] = pcol[q];
          pl[q] = plane[q];
        }
        __syncthreads();
        int piv = col, lp = pl[col];
        double pmag = v[col];
#pragma unroll
        for (int q = col + 1; q < NM; ++q)
          if (q < n && v[q] > pmag) {
            pmag = v[q];
            piv = q;
            lp = pl[q];
          }
        const int lc = pl[col];
        lp = __builtin_amdgcn_readfirstlane(lp);
        if (!(pmag > 1e-300)) { ok = false; continue; }
        if (l == lp) phys = col;  // positions col and piv swap rows
        else if (l == lc) phys = piv;
        const double inv = 1.0 / lane_bcast(a[col], lp);
        double pr[NM];
#pragma unroll
        for (int k = col + 1; k < NM; ++k) pr[k] = lane_bcast(a[k], lp);
        if (phys > col && l < n) {
          const double f = a[col] * inv;
          a[col] = f;
#pragma unroll
          for (int k = col + 1; k < NM; ++k)
            if (k < n) a[k] -= f * pr[k];
        }
      }
      if (ok) {
        int la[NM];
#pragma unroll
        for (int k = 0; k < NM; ++k) {
          const unsigned long long m = __ballot(phys == k);
          la[k] = __builtin_amdgcn_readfirstlane(m ? __ffsll(m) - 1 : 0);
        }
        // x = LU^-1 b with b_l in lane l, x_l to lane l, twice: b, then
        // the residual b - A x of one refinement step (x += A^-1 (b - A x)).
        // Row sums run by columns, in the host's order of summation.
        const double b0 = l == nh ? -1.0 : 0.0;
        double rhs = b0, xv = 0.0, c = 0.0;
#pragma unroll
        for (int it = 0; it < 2; ++it) {
          double t = rhs, y = 0.0;
#pragma unroll
          for (int k = 0; k < NM; ++k) {  // forward, L unit lower
            if (k < n) {
              const double yk = lane_bcast(t, la[k]);
              if (phys == k) y = t;
              if (phys > k && l < n) t -= a[k] * yk;
            }
          }
          t = y;
          double x = 0.0;
#pragma unroll
          for (int k = NM - 1; k >= 0; --k) {  // backward, the last column first
            if (k < n) {
              const double xk = lane_bcast(t, la[k]) / lane_bcast(a[k], la[k]);
              if (l == k) x = xk;
              if (phys < k && l < n) t -= a[k] * xk;
            }
          }
          if (it == 0) {
            xv = x;
            double r = b0;
#pragma unroll
            for (int k = 0; k < NM; ++k)
              if (k < n) {
                const double xk = lane_bcast(xv, k);
                r -= a0[k] * xk;
              }
            rhs = r;
          } else {
            c = xv + x;
          }
        }
        if (l < nh) s.coef[l] = c;
        const bool bad = __ballot(l < nh && !__builtin_isfinite(c)) != 0;
        if (l == 0) ctl[3] = bad ? 0 : 1;
      }
    }
  }
  __syncthreads();
  if (flag != 2 && !s.picard && !ctl[3] && l == 0) {  // no usable solution: restart
    s.order[0] = s.slot_new;
    s.n = 1;
    s.picard = 1;
  }
  __syncthreads();
  if (flag == 0 || flag == 4) {
    // the next pass: t = u_newest - sum_i (c_0 + .. + c_i) (u_{i+1} - u_i),
    // the new r and u in a free slot, else in the oldest one (dropped)
    const int n = s.n, D = s.D;
    bool used = l >= D;
    for (int i = 0; i < n; ++i) used |= s.order[i] == l;
    const unsigned long long busy = __ballot(used);
    const bool fresh = n < D;
    const int q = fresh ? __ffsll(~busy) - 1 : s.order[0];
    const int nd = fresh ? n : n - 1;
    // the rows of the next pass (the host's make_desc)
    const int period = s.low <= PULAY_BELOW ? s.period : 1;
    const int rows = s.skipped + 1 >= period ? (s.pend ? 2 : 1) : 0;
    if (!s.picard && l + 1 < n) {
      double cum = 0.0;
      for (int i = 0; i <= l; ++i) cum += s.coef[i];
      d.u[1 + l] = s.U + (size_t)s.order[l + 1] * s.mP;
      d.coef[1 + l] = -cum;
    }
    const float rsc = fp8_scale(rinf);
    if (l < nd) {
      const int qq = s.order[fresh ? l : l + 1];
      s.dotted[l] = qq;
      const int at = rows == 2 ? nd - l : l;  // gram_rows: the newest first
      d.rh[at] = s.R + (size_t)qq * s.mP * s.rbytes;
      d.rhinv[at] = 1.0f / s.rsc[qq];
    }
    if (l == 0) {
      if (rows == 2) {
        d.rh[0] = s.R + (size_t)q * s.mP * s.rbytes;
        d.rhinv[0] = 1.0f / rsc;
      }
      d.ngram = rows == 2 ? nd + 1 : 0;
      d.nrow = s.pend + 1;
      s.rows = rows;
      d.ncomb = s.picard ? 1 : n;
      d.plain = s.picard;
      d.u[0] = s.ucur;
      d.coef[0] = 1.0;
      s.slot_new = q;
      s.ndot = nd;
      d.ndot = rows == 1 ? nd : 0;
      s.rsc[q] = rsc;
      d.rsc = rsc;
      d.r = s.R + (size_t)q * s.mP * s.rbytes;
      d.dnew = s.U + (size_t)q * s.mP;
    }
  } else if (l == 0) {
    d.active = 0;
  }
  __syncthreads();
  if (l == 0) {
    // the iteration count last, released to the host that polls for it
    MdiisStatus& st = status[b];
    st.flag = flag;
    st.iters32 = s.iters32;
    st.hist = (flag == 0 || flag == 4) ? (d.ncomb > d.ndot ? d.ncomb : d.ndot) : 0;
    st.resid = rinf;
    st.r2 = r2;
    __threadfence_system();
    __hip_atomic_store(&st.iters, s.iters, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
  }
  {
    const uint64_t* src = reinterpret_cast<const uint64_t*>(&s);
    uint64_t* dst = reinterpret_cast<uint64_t*>(mst + b);
    for (int i = l; i < (int)(sizeof(MdiisDev) / 8); i += 64) dst[i] = src[i];
  }
}

// Host-prepared rows into the device MDIIS state and descriptors, read
// from pinned host memory: row r (grid x) is the solute index (8 bytes),
// its SoluteDesc, then its MdiisDev.
__global__ void __launch_bounds__(64)
mdiis_load(const uint64_t* __restrict__ rows, SoluteDesc* __restrict__ sd,
           MdiisDev* __restrict__ mst) {
  constexpr int WS = sizeof(SoluteDesc) / 8, WM = sizeof(MdiisDev) / 8;
  const uint64_t* row = rows + (size_t)blockIdx.x * (1 + WS + WM);
  const int b = (int)row[0];
  uint64_t* ds = reinterpret_cast<uint64_t*>(sd + b);
  uint64_t* dm = reinterpret_cast<uint64_t*>(mst + b);
  for (int i = threadIdx.x; i < WS; i += 64) ds[i] = row[1 + i];
  for (int i = threadIdx.x; i < WM; i += 64) dm[i] = row[1 + WS + i];
}

// FP8 residuals to BF16, four points a thread (once per solve, when periodic
// mixing begins).  Grid: x = chunks, y = entry.
struct HistMove {
  const uint8_t* src[MAX_DIIS];
  uint16_t* dst[MAX_DIIS];
  float inv[MAX_DIIS];  // 1 / the scale of src
};
__global__ void __launch_bounds__(NT)
hist_to_bf16(HistMove h, int64_t n) {
  const uint8_t* src = h.src[blockIdx.y];
  uint16_t* dst = h.dst[blockIdx.y];
  const float inv = h.inv[blockIdx.y];
  const int64_t stride = (int64_t)gridDim.x * NT * 4;
  for (int64_t e = (blockIdx.x * (int64_t)NT + threadIdx.x) * 4; e < n; e += stride)
    stbf4(dst + e, to_bf4(from_fp8x4(*reinterpret_cast<const uint32_t*>(src + e), inv)));
}

// FP32 <-> FP64 copies of the iterate at a precision hand-over.
// Grid: x = chunks, y = solute.
__global__ void __launch_bounds__(NT)
convert_batch(void* const* __restrict__ dst, const void* const* __restrict__ src, int to64,
              int64_t n, const int* __restrict__ active) {
  if (active && !active[blockIdx.y]) return;
  const int64_t stride = (int64_t)gridDim.x * NT;
  for (int64_t e = blockIdx.x * (int64_t)NT + threadIdx.x; e < n; e += stride) {
    if (to64)
      static_cast<double*>(dst[blockIdx.y])[e] = (double)static_cast<const float*>(src[blockIdx.y])[e];
    else
      static_cast<float*>(dst[blockIdx.y])[e] = (float)static_cast<const double*>(src[blockIdx.y])[e];
  }
}

// u = t + lam r, FP64, for one solute (first MDIIS entry of an FP64 phase).
__global__ void __launch_bounds__(NT)
seed_u(double* __restrict__ u, const double* __restrict__ t, const double* __restrict__ r,
       double lam, int64_t n) {
  const int64_t stride = (int64_t)gridDim.x * NT;
  for (int64_t e = blockIdx.x * (int64_t)NT + threadIdx.x; e < n; e += stride)
    u[e] = t[e] + lam * r[e];
}

// Defect correction, base update: t_b += delta for one solute.
__global__ void __launch_bounds__(NT)
add_delta(double* __restrict__ tb, const float* __restrict__ delta, int64_t n) {
  const int64_t stride = (int64_t)gridDim.x * NT;
  for (int64_t e = blockIdx.x * (int64_t)NT + threadIdx.x; e < n; e += stride)
    tb[e] += (double)delta[e];
}

// Defect correction, the newest u of a difference-form history moved to
// the coordinates of a new base: u -= delta (the delta folded into t_b).
__global__ void __launch_bounds__(NT)
shift_u(float* __restrict__ u, const float* __restrict__ delta, int64_t n) {
  const int64_t stride = (int64_t)gridDim.x * NT;
  for (int64_t e = blockIdx.x * (int64_t)NT + threadIdx.x; e < n; e += stride) u[e] -= delta[e];
}

// Defect correction, new base t_b with F(t_b) = f64 known: x_b = -beta v +
// t_b (PY: exp(-beta v) - 1) into xb, F(t_b) into fb; with seed (the first
// base of a solve) also delta = 0 and the first MDIIS entry r_0 = F(t_b)
// (BF16 with r16), u_0 = 0 + lam r_0.
__global__ void __launch_bounds__(NT)
rebase_prep(const double* __restrict__ tb, const double* __restrict__ bv,
            const double* __restrict__ f64, int py, int seed, float lam,
            float* __restrict__ xb, float* __restrict__ fb, float* __restrict__ delta,
            float* __restrict__ u0, void* __restrict__ r0, int r16, float r8s, int64_t n) {
  const int64_t stride = (int64_t)gridDim.x * NT;
  for (int64_t e = blockIdx.x * (int64_t)NT + threadIdx.x; e < n; e += stride) {
    const double b = bv[e];
    xb[e] = py ? (float)expm1(-b) : (float)(-b + tb[e]);
    const float f = (float)f64[e];
    fb[e] = f;
    if (seed) {
      delta[e] = 0.f;
      if (r8s > 0.f)  // FP8 e4m3 of f * r8s (clamped: the conversion does not saturate)
        static_cast<uint8_t*>(r0)[e] = (uint8_t)(__builtin_amdgcn_cvt_pk_fp8_f32(
            fminf(fmaxf(f * r8s, -448.f), 448.f), 0.f, 0, false) & 0xFF);
      else if (r16)
        static_cast<uint16_t*>(r0)[e] = (uint16_t)bf16_bits(f);
      else
        static_cast<float*>(r0)[e] = f;
      u0[e] = lam * f;
    }
  }
}

// ------------------------------------------------------ setup kernels
// Capped LJ and short-range Coulomb (bgy3d-solutes.c:45-131, 196-286).
__device__ __forceinline__ double lj0(double r) {
  const double p2 = 1.0 / (r * r);
  const double p6 = p2 * p2 * p2;
  return 4 * p6 * (p6 - 1);
}
__device__ __forceinline__ double lj1(double r) {
  const double p2 = 1.0 / (r * r);
  const double p6 = p2 * p2 * p2;
  return 4 * p6 * (6 - 12 * p6) / r;
}
__device__ __forceinline__ double ljcap0(double r) {
  const double R = 0.2;
  if (r >= R) return lj0(r);
  const double b = lj1(R) / (2 * R), a = lj0(R);
  return a + b * (r - R) * (r + R);
}
__device__ __forceinline__ double cs0(double r) { return erfc(r) / r; }
__device__ __forceinline__ double cs1(double r) {
  return -(erfc(r) + (2 / sqrt(M_PI)) * r * exp(-r * r)) / (r * r);
}
__device__ __forceinline__ double cscap0(double r) {
  const double R = 0.2;
  if (r >= R) return cs0(r);
  const double b = cs1(R) / (2 * R), a = cs0(R);
  return a + b * (r - R) * (r + R);
}
// erf(r)/r with its Taylor form below 0.02 (bgy3d-solutes.c:148-159)
__device__ __forceinline__ double cl0(double r) {
  if (r >= 0.02) return erf(r) / r;
  const double r2 = r * r;
  return (2 / sqrt(M_PI)) * (1. + r2 * (-1. / 3. + r2 * (1. / 10. + r2 * (-1. / 42.))));
}

// beta v_i(r) for every solvent site (field0, bgy3d-solutes.c:344-377).
// Grid: x = chunks of P, y = solute.  Writes FP64 and, if bv32 != NULL,
// an FP32 copy for the mixed-precision bulk iterations.  The solute sites
// pass through LDS in chunks of FB_CHUNK: position, G charge / eps0 and, per
// solvent site, sigma_ai^2 and 4 epsilon_ai of the Lorentz-Berthelot pair
// (epsilon_ai = sqrt(eps_a) sqrt(eps_i), sigma_ai = (sigma_a + sigma_i) / 2).
// Per point and site one r^2, 1 / r^2, r and the capped erfc(G r) / r (within
// G r < 6.5), then per solvent site (sigma_ai / r)^6 from 1 / r^2:
// ljcap0(r / sigma_ai) without a division or square root in the pair loop.
// Bound by FP64 arithmetic and its latencies: a thread takes FB_PTS points
// side by side in x, whose divisions overlap and which share the site's LDS
// reads and y, z terms, and one test tells whether any pair is inside its cap.
// Four waves per SIMD are worth 20 bytes of spill (218 -> 205 us).  One point
// a thread and pair parameters formed per point took 318 us for 30 sites on
// 128^3 (now 205) and 2744 us for 5 solvent sites on 192^3 (now 1282).
constexpr int FB_CHUNK = 128, FB_PTS = 2;
constexpr double FB_RC2 = (6.5 / G_COULOMB) * (6.5 / G_COULOMB);
// MS: the solvent-site arrays' size (>= g.m), so that water's three fit
// in few registers.
template <int MS>
__global__ void __launch_bounds__(NT, 4)
field_bv(const SitesDesc* __restrict__ sites, GridArgs g, const double* __restrict__ solvent_sse,
         double L0, double L1, double L2, double h0, double h1, double h2,
         double* const* __restrict__ bv64, float* const* __restrict__ bv32) {
  struct Site {
    double x, y, z, qg, top;   // top: the largest sigma_ai^2
    double sab2[MS], e4[MS];
  };
  __shared__ Site st[FB_CHUNK];
  const SitesDesc sd = sites[blockIdx.y];
  const int m = g.m;
  double sq[MS];
#pragma unroll
  for (int i = 0; i < MS; ++i) sq[i] = i < m ? solvent_sse[3 * i + 2] : 0.0;
  // ljcap0 below r = 0.2 sigma: a + b (x^2 - 0.04), x = r / sigma
  const double R = 0.2, cap_a = lj0(R), cap_b = lj1(R) / (2 * R);
  const int nch = (sd.n + FB_CHUNK - 1) / FB_CHUNK;
  auto load = [&](int c) {
    for (int k = threadIdx.x; k < FB_CHUNK; k += NT) {
      const int a = c * FB_CHUNK + k;
      if (a >= sd.n) break;
      const double* s = sd.xyz_s_e_q + 6 * a;
      Site& t = st[k];
      t.x = s[0];
      t.y = s[1];
      t.z = s[2];
      t.qg = s[5] * EPSILON0INV * G_COULOMB;
      t.top = 0.0;
      const double se = sqrt(s[4]);
#pragma unroll
      for (int i = 0; i < MS; ++i) {
        if (i >= m) continue;
        const double sab = 0.5 * (s[3] + solvent_sse[3 * i]);
        t.sab2[i] = sab * sab;
        t.e4[i] = 4 * (se * sqrt(solvent_sse[3 * i + 1]));
        t.top = fmax(t.top, t.sab2[i]);
      }
    }
  };
  if (nch == 1) {
    load(0);
    __syncthreads();
  }
  const int64_t stride = (int64_t)gridDim.x * NT, np = g.P / FB_PTS;  // N0 is even
  // rounds of NT threads, the same count in every thread (LDS reloads)
  for (int64_t e0 = blockIdx.x * (int64_t)NT; e0 < np; e0 += stride) {
    const int64_t e = (e0 + threadIdx.x) * FB_PTS;
    const bool ok = e < g.P;
    const int x = (int)(e % g.N0);
    const int y = (int)((e / g.N0) % g.N1);
    const int z = (int)(e / ((int64_t)g.N0 * g.N1));
    const double ry = y * h1 - L1 / 2, rz = z * h2 - L2 / 2;
    double rx[FB_PTS], v[MS][FB_PTS];
#pragma unroll
    for (int p = 0; p < FB_PTS; ++p) {
      rx[p] = (x + p) * h0 - L0 / 2;
#pragma unroll
      for (int i = 0; i < MS; ++i) v[i][p] = 0.0;
    }
    for (int c = 0; c < nch; ++c) {
      if (nch > 1) {
        __syncthreads();
        load(c);
        __syncthreads();
      }
      const int na = min(FB_CHUNK, sd.n - c * FB_CHUNK);
      if (!ok) continue;
      for (int k = 0; k < na; ++k) {
        const Site& s = st[k];
        const double dy = ry - s.y, dz = rz - s.z;
        const double dyz = dy * dy + dz * dz;
        double r2[FB_PTS], ir2[FB_PTS], csc[FB_PTS];
        bool capped = false;
#pragma unroll
        for (int p = 0; p < FB_PTS; ++p) {
          const double dx = rx[p] - s.x;
          r2[p] = dx * dx + dyz;
          ir2[p] = 1.0 / r2[p];
          capped |= !(s.top * ir2[p] <= 25.0);  // r = 0 gives infinity, or NaN with sigma 0
        }
        // erfc(G r) / r vanishes beyond G r = 6.5 (erfc(6.5) = 3.8e-20: the
        // term is below 2e-18 kcal/mol there, under the rounding of v)
#pragma unroll
        for (int p = 0; p < FB_PTS; ++p)
          csc[p] = r2[p] < FB_RC2 ? s.qg * cscap0(G_COULOMB * sqrt(r2[p])) : 0.0;
#pragma unroll
        for (int i = 0; i < MS; ++i) {
          if (i >= m) continue;
#pragma unroll
          for (int p = 0; p < FB_PTS; ++p) {
            const double s2 = s.sab2[i] * ir2[p];  // (sigma_ai / r)^2
            const double p6 = s2 * s2 * s2;
            double lj = s.e4[i] * (p6 * (p6 - 1));
            if (capped && !(s2 <= 25.0))
              lj = 0.25 * s.e4[i] * (cap_a + cap_b * (r2[p] / s.sab2[i] - R * R));
            v[i][p] += lj + sq[i] * csc[p];
          }
        }
      }
    }
    if (!ok) continue;
#pragma unroll
    for (int i = 0; i < MS; ++i) {
      if (i >= m) continue;
#pragma unroll
      for (int p = 0; p < FB_PTS; ++p) {
        const double b = g.beta * v[i][p];
        bv64[blockIdx.y][i * g.P + e + p] = b;
        if (bv32) bv32[blockIdx.y][i * g.P + e + p] = (float)b;
      }
    }
  }
}

// Trigonometric interpolation of one solute's spectrum from the grid
// N/2 to N in the same box: Wf(k) = Wc(k) scale at every frequency the
// coarse grid holds, zero above.  The coarse Nyquist planes of the full y
// and z axes go in halves to +N_c/2 and -N_c/2, that of the half x axis in
// half to kx = N0_c/2 (the c2r mirrors it to -N0_c/2).  scale = 1 / P_c
// with the unnormalised inverse of the fine pipeline.  Grid: x = chunks
// of Kf, y = site.
__device__ __forceinline__ int up_index(int kf, int nf, int nc, double& w) {
  const int h = nc / 2;
  w = 1.0;
  if (kf < h) return kf;
  if (kf == h || kf == nf - h) { w = 0.5; return h; }
  if (kf > nf - h) return kf - nf + nc;
  return -1;
}
__global__ void __launch_bounds__(NT)
spec_upsample(const cpx<double>* __restrict__ wc, cpx<double>* __restrict__ wf, GridArgs g,
              int N0c, int N1c, int N2c, int NHc, int64_t Kc, double scale) {
  const int s = blockIdx.y;
  const int64_t stride = (int64_t)gridDim.x * NT;
  for (int64_t e = blockIdx.x * (int64_t)NT + threadIdx.x; e < g.K; e += stride) {
    const int kx = (int)(e % g.NH);
    const int ky = (int)((e / g.NH) % g.N1);
    const int kz = (int)(e / ((int64_t)g.NH * g.N1));
    cpx<double> v = {0.0, 0.0};
    double wx = 1.0, wy, wz;
    const int hx = N0c / 2;
    const int cx = kx < hx ? kx : (kx == hx ? (wx = 0.5, hx) : -1);
    const int cy = up_index(ky, g.N1, N1c, wy);
    const int cz = up_index(kz, g.N2, N2c, wz);
    if (cx >= 0 && cy >= 0 && cz >= 0) {
      const cpx<double> c = wc[s * Kc + ((int64_t)cz * N1c + cy) * NHc + cx];
      const double w = wx * wy * wz * scale;
      v = cpx<double>{c.re * w, c.im * w};
    }
    wf[s * g.K + e] = v;
  }
}

// F(k) s(k) = s(k) sum_a Q_a exp(-i k.x_a), corner k (form_factor,
// bgy3d-solutes.c:587-600, times bgy3d_vec_fft_trans bgy3d-vec.c:619-646).
// A workgroup takes FF_X columns kx by FF_Y rows ky of one z plane; for
// FF_SITES sites at a time it puts exp(-i kx x) of the columns and
// Q exp(-i (ky y + kz z)) of the rows in LDS, so that a point costs one complex
// product per site instead of a sine and cosine (104 -> 33 us for 30 sites on
// 128^3, 21 MB to write).
// Grid: x = column tile, then row tile, then z plane; y = solute.
constexpr int FF_X = 32, FF_Y = 32, FF_SITES = 16;
__host__ __device__ inline int ff_tiles(const GridArgs& g) {
  return ((g.NX + FF_X - 1) / FF_X) * ((g.N1 + FF_Y - 1) / FF_Y) * g.N2;
}
__global__ void __launch_bounds__(NT)
form_factor(const SitesDesc* __restrict__ sites, GridArgs g, cpx<double>* const* __restrict__ fs64,
            cpx<float>* const* __restrict__ fs32) {
  constexpr int RPT = FF_X * FF_Y / NT;  // rows per thread
  __shared__ cpx<double> ex[FF_SITES][FF_X], eyz[FF_SITES][FF_Y];
  const SitesDesc sd = sites[blockIdx.y];
  const int tx = (g.NX + FF_X - 1) / FF_X, ty = (g.N1 + FF_Y - 1) / FF_Y;
  const int x0 = (int)(blockIdx.x % tx) * FF_X, y0 = (int)(blockIdx.x / tx % ty) * FF_Y;
  const int z = (int)(blockIdx.x / (tx * ty));
  const int iz = (z <= g.N2 / 2) ? z : z - g.N2;
  const int col = threadIdx.x % FF_X, row = threadIdx.x / FF_X * RPT;
  double re[RPT], im[RPT];
#pragma unroll
  for (int r = 0; r < RPT; ++r) re[r] = im[r] = 0.0;
  for (int a0 = 0; a0 < sd.n; a0 += FF_SITES) {
    const int na = min(FF_SITES, sd.n - a0);
    __syncthreads();
    for (int k = threadIdx.x; k < na * (FF_X + FF_Y); k += NT) {
      const int a = k / (FF_X + FF_Y), c = k - a * (FF_X + FF_Y);
      const double* s = sd.xyz_s_e_q + 6 * (a0 + a);
      double sn, cs;
      if (c < FF_X) {
        sincos((x0 + c) * g.dkx * s[0], &sn, &cs);
        ex[a][c] = cpx<double>{cs, -sn};
      } else {
        const int y = y0 + c - FF_X, iy = (y <= g.N1 / 2) ? y : y - g.N1;
        sincos(iy * g.dky * s[1] + iz * g.dkz * s[2], &sn, &cs);
        eyz[a][c - FF_X] = cpx<double>{s[5] * cs, -s[5] * sn};
      }
    }
    __syncthreads();
    for (int a = 0; a < na; ++a) {
      const cpx<double> u = ex[a][col];
#pragma unroll
      for (int r = 0; r < RPT; ++r) {
        const cpx<double> w = eyz[a][row + r];
        re[r] += u.re * w.re - u.im * w.im;
        im[r] += u.re * w.im + u.im * w.re;
      }
    }
  }
  const int x = x0 + col;
  if (x >= g.NX) return;
#pragma unroll
  for (int r = 0; r < RPT; ++r) {
    const int y = y0 + row + r;
    if (y >= g.N1) return;
    const int iy = (y <= g.N1 / 2) ? y : y - g.N1;
    const double sign = ((x + iy + iz) & 1) ? -1.0 : 1.0;
    const cpx<double> f = {sign * re[r], sign * im[r]};
    fs64[blockIdx.y][((int64_t)z * g.N1 + y) * g.NH + x] = f;
    if (x == g.NX - 1) fs64[blockIdx.y][g.K + (int64_t)z * g.N1 + y] = f;
    if (fs32)
      fs32[blockIdx.y][fs_index<float>(g, z, y, x)] = cpx<float>{(float)f.re, (float)f.im};
  }
}

// -------------------------------------------------- mu and observables
// Per point: c = closure(beta v, t), h = c + t, x = -beta v + t,
// cl_i = -beta q_i u_c(r) with u_c = eps0^-1 sum_a Q_a G cl0(G r)
// (coulomb_long, bgy3d-solutes.c:796-815); accumulate the chemical
// potential densities of the native closure, HNC, KH, GF and sum c
// (hnc3d.c:2172-2268), with Neumaier-compensated FP64 sums.  Writes
// g = h + 1 if gout != NULL.
// Grid: x = chunks of P, y = solute.  part[(b*gridDim.x + x)*5 + q].
__global__ void __launch_bounds__(NT)
mu_density(const SitesDesc* __restrict__ sites, GridArgs g, const double* const* __restrict__ tt,
           const double* const* __restrict__ bv64, double L0, double L1, double L2, double h0,
           double h1, double h2, double* const* __restrict__ gout, double* __restrict__ part) {
  __shared__ double red[5][NT / 64];
  const SitesDesc sd = sites[blockIdx.y];
  const double* t = tt[blockIdx.y];
  const double* bv = bv64[blockIdx.y];
  double* go = gout ? gout[blockIdx.y] : nullptr;
  double sum[5] = {0, 0, 0, 0, 0}, comp[5] = {0, 0, 0, 0, 0};
  const int64_t stride = (int64_t)gridDim.x * NT;
  for (int64_t e = blockIdx.x * (int64_t)NT + threadIdx.x; e < g.P; e += stride) {
    const int x = (int)(e % g.N0);
    const int y = (int)((e / g.N0) % g.N1);
    const int z = (int)(e / ((int64_t)g.N0 * g.N1));
    const double rx = x * h0 - L0 / 2, ry = y * h1 - L1 / 2, rz = z * h2 - L2 / 2;
    double uc = 0.0;
    for (int a = 0; a < sd.n; ++a) {
      const double* s = sd.xyz_s_e_q + 6 * a;
      const double dx = rx - s[0], dy = ry - s[1], dz = rz - s[2];
      // erf(x) rounds to 1 in FP64 beyond x = 6 (erfc(6) = 2.2e-17)
      const double xg = G_COULOMB * sqrt(dx * dx + dy * dy + dz * dz);
      uc += s[5] * G_COULOMB * (xg >= 6.0 ? 1.0 / xg : cl0(xg));
    }
    uc *= EPSILON0INV;
    double v[5] = {0, 0, 0, 0, 0};
    for (int i = 0; i < g.m; ++i) {
      const int64_t idx = i * g.P + e;
      const double ti = t[idx], bvi = bv[idx];
      const double c = closure_c<double>(g.closure, g.pse_order, bvi, ti);
      const double h = c + ti;
      const double xx = -bvi + ti;
      const double cl = -g.beta * g.q[i] * uc;
      const double w = g.rw[i];  // rho_i / rho (1: one density)
      v[0] += w * form_mu(g.closure, g.pse_order, xx, h, c, cl);
      v[1] += w * form_mu(0, 0, xx, h, c, cl);
      v[2] += w * form_mu(1, 1, xx, h, c, cl);
      v[3] += w * form_mu(2, 0, xx, h, c, cl);
      v[4] += w * c;
      if (go) go[idx] = h + 1.0;
    }
#pragma unroll
    for (int q = 0; q < 5; ++q) {  // Neumaier
      const double s = sum[q] + v[q];
      comp[q] += (fabs(sum[q]) >= fabs(v[q])) ? (sum[q] - s) + v[q] : (v[q] - s) + sum[q];
      sum[q] = s;
    }
  }
  const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
#pragma unroll
  for (int q = 0; q < 5; ++q) {
    const double s = warp_sum(sum[q] + comp[q]);
    if (lane == 0) red[q][w] = s;
  }
  __syncthreads();
  if (threadIdx.x < 5) {
    double s = red[threadIdx.x][0];
    for (int i = 1; i < NT / 64; ++i) s += red[threadIdx.x][i];
    part[((int64_t)blockIdx.y * gridDim.x + blockIdx.x) * 5 + threadIdx.x] = s;
  }
}

// ------------------------------------------------------------ gradients
// Derivatives of the capped pair functions (bgy3d-solutes.c:102-131,
// 162-190, 246-305).
__device__ __forceinline__ double ljcap1(double r) {
  const double R = 0.2;
  if (r >= R) return lj1(r);
  return 2 * (lj1(R) / (2 * R)) * r;
}
__device__ __forceinline__ double cscap1(double r) {
  const double R = 0.2;
  if (r >= R) return cs1(r);
  return 2 * (cs1(R) / (2 * R)) * r;
}
__device__ __forceinline__ double cl1(double r) {
  const double r2 = r * r;
  if (r >= 0.02) return ((2 / sqrt(M_PI)) * r * exp(-r2) - erf(r)) / r2;
  return -(4 / (3 * sqrt(M_PI))) * r * (1. + r2 * (-3. / 5. + r2 * (3. / 14. + r2 * (-1. / 18.))));
}
__device__ __forceinline__ double ccap1(double r) {
  if (r >= 0.2) return -1.0 / (r * r);
  return cscap1(r) + cl1(r);
}

// d c / d t and d c / d(beta v) of closure_c, FP64.
__device__ __forceinline__ void closure_derivs(int method, int order, double bv, double t,
                                               double* ct, double* cv) {
  const double x = -bv + t;
  switch (method) {
    case 0: *ct = expm1(x); *cv = -(*ct + 1); return;
    case 1:
      if (x <= 0) { *ct = expm1(x); *cv = -(*ct + 1); } else { *ct = 0; *cv = -1; }
      return;
    case 2: *ct = exp(-bv) - 1; *cv = -exp(-bv) * (1 + t); return;
    default: {
      *ct = (x < 0) ? expm1(x) : exps1(order - 1, x);
      *cv = -(*ct + 1);
    }
  }
}

// form1 (closures.f90:615-653): differential of the mu density.
__device__ __forceinline__ double form1_mu(int method, int order, double x, double dx, double h,
                                           double dh, double c, double dc, double cl) {
  const double base = -dc - dh * (c + cl) / 2 - h * dc / 2;
  switch (method) {
    case 0: return base + h * dh;
    case 1: return (h < 0) ? base + h * dh : base;
    case 2: return base;
    default: {
      if (h < 0) return base + h * dh;
      double nx = 1, xn = 1;
      for (int k = 1; k <= order; ++k) { nx *= k; xn *= x; }
      return base + (h * dh - xn * dx / nx);
    }
  }
}

// Per-point coefficients at the converged t (grid-stride, one solute).
// mode 0 (TPT, hnc3d.c:1666-1742): A_i = rho h^3 g_i, B = 0.
// mode 1 (adjoint, prep): D_i = dc/dt, gmu_i = dmu/dt.
// mode 2 (adjoint, final): A_i = beta (K lambda)_i dc/d(beta v) + dmu/dv_i,
//                          B = rho h^3 / 2 sum_i q_i h_i  (dmu/du_c).
// mode 4 (linear response, hnc3d.c:1969-2134): as mode 2 with the
//   reference's dc/d(beta v) = -(dc/dt + 1) (its Jacobian flag hack,
//   hnc3d.c:1310-1320) for every closure; B unused.
__global__ void __launch_bounds__(NT)
adj_coef(GridArgs g, SitesDesc sd, const double* __restrict__ t, const double* __restrict__ bv,
         const double* __restrict__ Klam, double L0, double L1, double L2, double h0, double h1,
         double h2, double rho, int mode, double* __restrict__ A, double* __restrict__ B,
         double* __restrict__ D, double* __restrict__ gmu) {
  const double fmu = rho * g.h3 / g.beta;
  const int64_t stride = (int64_t)gridDim.x * NT;
  for (int64_t e = blockIdx.x * (int64_t)NT + threadIdx.x; e < g.P; e += stride) {
    double uc = 0.0;
    if (mode != 0) {
      const int x = (int)(e % g.N0);
      const int y = (int)((e / g.N0) % g.N1);
      const int z = (int)(e / ((int64_t)g.N0 * g.N1));
      const double rx = x * h0 - L0 / 2, ry = y * h1 - L1 / 2, rz = z * h2 - L2 / 2;
      for (int a = 0; a < sd.n; ++a) {
        const double* s = sd.xyz_s_e_q + 6 * a;
        const double dx = rx - s[0], dy = ry - s[1], dz = rz - s[2];
        uc += s[5] * G_COULOMB * cl0(G_COULOMB * sqrt(dx * dx + dy * dy + dz * dz));
      }
      uc *= EPSILON0INV;
    }
    double bsum = 0.0;
    for (int i = 0; i < g.m; ++i) {
      const int64_t q = i * g.P + e;
      const double ti = t[q], bvi = bv[q];
      const double c = closure_c<double>(g.closure, g.pse_order, bvi, ti);
      const double h = c + ti;
      if (mode == 0) {
        A[q] = rho * g.h3 * (h + 1.0);
        continue;
      }
      double ct, cv;
      closure_derivs(g.closure, g.pse_order, bvi, ti, &ct, &cv);
      const double x = -bvi + ti;
      const double cl = -g.beta * g.q[i] * uc;
      if (mode == 1) {
        D[q] = ct;
        gmu[q] = fmu * form1_mu(g.closure, g.pse_order, x, 1.0, h, ct + 1, c, ct, cl);
      } else {
        const double dcv = (mode == 4 ? -(ct + 1) : cv) * g.beta;
        A[q] = Klam[q] * dcv +
               fmu * form1_mu(g.closure, g.pse_order, x, -g.beta, h, dcv, c, dcv, cl);
        bsum += g.q[i] * h;
      }
    }
    if (mode == 2) B[e] = 0.5 * rho * g.h3 * bsum;
  }
}

// sum_r sum_i A_i(r) dv_i(r)/dtheta_a (+ B(r) du_c/dtheta_a) for solute
// site a = blockIdx.y over a chunk of points blockIdx.x.  mode 0 (TPT,
// field1 bgy3d-solutes.c:381-468): full capped Coulomb, xyz only.
// mode 1 (adjoint): short-range v plus the u_c of the mu integral; x, y, z,
// q, sigma, epsilon.  Partials part[(a * gridDim.x + chunk) * 6 + p].
__global__ void __launch_bounds__(NT)
grad_field(GridArgs g, SitesDesc sd, const double* __restrict__ solvent_sse,
           const double* __restrict__ A, const double* __restrict__ B, double L0, double L1,
           double L2, double h0, double h1, double h2, int mode, double* __restrict__ part) {
  __shared__ double red[6][NT / 64];
  const int a = blockIdx.y;
  const double* s = sd.xyz_s_e_q + 6 * a;
  double acc[6] = {0, 0, 0, 0, 0, 0};
  const int64_t stride = (int64_t)gridDim.x * NT;
  const double G = G_COULOMB;
  for (int64_t e = blockIdx.x * (int64_t)NT + threadIdx.x; e < g.P; e += stride) {
    const int x = (int)(e % g.N0);
    const int y = (int)((e / g.N0) % g.N1);
    const int z = (int)(e / ((int64_t)g.N0 * g.N1));
    const double dx = x * h0 - L0 / 2 - s[0], dy = y * h1 - L1 / 2 - s[1], dz = z * h2 - L2 / 2 - s[2];
    const double r = sqrt(dx * dx + dy * dy + dz * dz);
    const double inv = r > 0 ? 1.0 / r : 0.0;
    const double gx = -dx * inv, gy = -dy * inv, gz = -dz * inv;  // dr / dx_a
    double fr = 0.0;
    for (int i = 0; i < g.m; ++i) {
      const double* sv = solvent_sse + 3 * i;
      const double eab = sqrt(sv[1] * s[4]);
      const double sab = 0.5 * (sv[0] + s[3]);
      const double qab = sv[2] * s[5] * EPSILON0INV;
      const double Ai = A[i * g.P + e];
      const double rs = r / sab;
      const double lj1v = ljcap1(rs);
      if (mode == 0) {
        fr += Ai * ((eab / sab) * lj1v + qab * G * G * ccap1(G * r));
      } else {
        fr += Ai * ((eab / sab) * lj1v + qab * G * G * cscap1(G * r));
        acc[3] += Ai * sv[2] * EPSILON0INV * G * cscap0(G * r);
        acc[4] += Ai * eab * lj1v * (-r / (sab * sab)) * 0.5;
        if (eab > 0) acc[5] += Ai * ljcap0(rs) * sv[1] / (2 * eab);
      }
    }
    if (mode != 0) {
      const double b = B[e];
      fr += b * EPSILON0INV * s[5] * G * G * cl1(G * r);
      acc[3] += b * EPSILON0INV * G * cl0(G * r);
    }
    acc[0] += fr * gx;
    acc[1] += fr * gy;
    acc[2] += fr * gz;
  }
  const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
#pragma unroll
  for (int p = 0; p < 6; ++p) {
    const double v = warp_sum(acc[p]);
    if (lane == 0) red[p][w] = v;
  }
  __syncthreads();
  if (threadIdx.x < 6) {
    double v = red[threadIdx.x][0];
    for (int i = 1; i < NT / 64; ++i) v += red[threadIdx.x][i];
    part[((int64_t)a * gridDim.x + blockIdx.x) * 6 + threadIdx.x] = v;
  }
}

// tau term of the adjoint gradient: with S(k) = w(kx) s(k) sum_i tau_i(k)
// conj(Lambda_i(k)) (Lambda = r2c(lambda), w = 1 at kx = 0 and N0/2, else
// 2), -tau_scale Re sum_k S(k) dF(k)/dtheta_a for F = sum_a Q_a e^{-ik.x_a}:
// theta = Q_a -> e^{-ik.x_a}, x_a -> -i k Q_a e^{-ik.x_a}.  Site a =
// blockIdx.y, chunk of K = blockIdx.x.  part[(a * gridDim.x + chunk) * 4 + p]
// for p = x, y, z, q.
__global__ void __launch_bounds__(NT)
grad_tau(GridArgs g, SitesDesc sd, const cpx<double>* __restrict__ Lam,
         const double* __restrict__ tau3, const double* __restrict__ chi3,
         double* __restrict__ part) {
  __shared__ double red[4][NT / 64];
  const int a = blockIdx.y;
  const double* s = sd.xyz_s_e_q + 6 * a;
  double acc[4] = {0, 0, 0, 0};
  const int64_t stride = (int64_t)gridDim.x * NT;
  for (int64_t e = blockIdx.x * (int64_t)NT + threadIdx.x; e < g.K; e += stride) {
    const int x = (int)(e % g.NH);
    if (x >= g.NX) continue;  // row padding
    const int y = (int)((e / g.NH) % g.N1);
    const int z = (int)(e / ((int64_t)g.NH * g.N1));
    const int iy = (y <= g.N1 / 2) ? y : y - g.N1;
    const int iz = (z <= g.N2 / 2) ? z : z - g.N2;
    const double kx = x * g.dkx, ky = iy * g.dky, kz = iz * g.dkz;
    // the long-range weight of site i: tau_i(k) on the tau path; on the Ng
    // path (whose residual carries -beta u_c(k) (q_i + sum_j (chi - 1)_ij q_j)
    // with u_c = eps0^-1 4 pi e^{-k^2/4G^2}/k^2 F s, 0 at k = 0) the same
    // factor without eps0^-1 F s, which tau_scale and the phase supply
    double shape = 0.0;
    if (!g.renorm) {
      const double k2 = kmag2(kx, ky, kz);
      shape = (k2 == 0.0) ? 0.0 : 4 * M_PI * exp(-k2 / (4 * G_COULOMB * G_COULOMB)) / k2;
    }
    double sre = 0.0, sim = 0.0;
    for (int i = 0; i < g.m; ++i) {
      const cpx<double> L = Lam[i * g.K + e];
      double ti;
      if (g.renorm) {
        ti = tau3[i * g.KT + table_index(g, z, y, x)];
      } else {
        double w = g.q[i];
        for (int j = 0; j < g.m; ++j)
          w += chi3[(int64_t)((i >= j) ? i * (i + 1) / 2 + j : j * (j + 1) / 2 + i) * g.KT +
                    table_index(g, z, y, x)] *
               g.q[j];
        ti = shape * w;
      }
      sre += ti * L.re;
      sim -= ti * L.im;
    }
    const double w = ((x == 0 || x == g.N0 / 2) ? 1.0 : 2.0) * (((x + iy + iz) & 1) ? -1.0 : 1.0);
    sre *= w;
    sim *= w;
    double sn, cs;
    sincos(kx * s[0] + ky * s[1] + kz * s[2], &sn, &cs);
    // S e^{-i phi} = (sre + i sim)(cs - i sn)
    const double pre = sre * cs + sim * sn;
    const double pim = sim * cs - sre * sn;
    acc[3] += pre;                       // Re S e^{-i phi}
    // Re[S e^{-i phi} (-i k Q)] = Q k Im[S e^{-i phi}]
    acc[0] += s[5] * kx * pim;
    acc[1] += s[5] * ky * pim;
    acc[2] += s[5] * kz * pim;
  }
  const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
#pragma unroll
  for (int p = 0; p < 4; ++p) {
    const double v = warp_sum(acc[p]);
    if (lane == 0) red[p][w] = v;
  }
  __syncthreads();
  if (threadIdx.x < 4) {
    double v = red[threadIdx.x][0];
    for (int i = 1; i < NT / 64; ++i) v += red[threadIdx.x][i];
    part[((int64_t)a * gridDim.x + blockIdx.x) * 4 + threadIdx.x] = -g.tau_scale * v;
  }
}

// ------------------------------------------------------ Newton-Krylov
// dc/dt at t (closure1, closures.f90:131-153) for the matrix-free Newton
// Jacobian, FP64, one solute.
__global__ void __launch_bounds__(NT)
closure_dcdt(GridArgs g, const double* __restrict__ t, const double* __restrict__ bv,
             double* __restrict__ D, int64_t n) {
  const int64_t stride = (int64_t)gridDim.x * NT;
  for (int64_t e = blockIdx.x * (int64_t)NT + threadIdx.x; e < n; e += stride) {
    double ct, cv;
    closure_derivs(g.closure, g.pse_order, bv[e], t[e], &ct, &cv);
    D[e] = ct;
  }
}

// Krylov helpers, FP64, one solute.  mdot: per workgroup partial sums of
// <w, V_i>, V_i = V + i n for i < nv, to part[block * nv + i] (the host adds
// the partials in a fixed order).  maxpy: w -= sum_i h_i V_i.  vcomb:
// y = a x + b y.
constexpr int KMAX = 32;
__global__ void __launch_bounds__(NT)
mdot(const double* __restrict__ V, int nv, const double* __restrict__ w, int64_t n,
     double* __restrict__ part) {
  __shared__ double red[KMAX][NT / 64];
  double acc[KMAX];
#pragma unroll
  for (int i = 0; i < KMAX; ++i) acc[i] = 0.0;
  const int64_t stride = (int64_t)gridDim.x * NT;
  for (int64_t e = blockIdx.x * (int64_t)NT + threadIdx.x; e < n; e += stride) {
    const double we = w[e];
#pragma unroll
    for (int i = 0; i < KMAX; ++i)
      if (i < nv) acc[i] += we * V[(int64_t)i * n + e];
  }
  const int wv = threadIdx.x >> 6, lane = threadIdx.x & 63;
#pragma unroll
  for (int i = 0; i < KMAX; ++i)
    if (i < nv) {
      const double v = warp_sum(acc[i]);
      if (lane == 0) red[i][wv] = v;
    }
  __syncthreads();
  if (threadIdx.x < nv) {
    double v = red[threadIdx.x][0];
    for (int q = 1; q < NT / 64; ++q) v += red[threadIdx.x][q];
    part[(int64_t)blockIdx.x * nv + threadIdx.x] = v;
  }
}
__global__ void __launch_bounds__(NT)
maxpy(double* __restrict__ w, const double* __restrict__ V, const double* __restrict__ h, int nv,
      int64_t n) {
  const int64_t stride = (int64_t)gridDim.x * NT;
  for (int64_t e = blockIdx.x * (int64_t)NT + threadIdx.x; e < n; e += stride) {
    double acc = w[e];
    for (int i = 0; i < nv; ++i) acc -= h[i] * V[(int64_t)i * n + e];
    w[e] = acc;
  }
}
__global__ void __launch_bounds__(NT)
vcomb(double* __restrict__ y, const double* __restrict__ x, double a, double b, int64_t n) {
  const int64_t stride = (int64_t)gridDim.x * NT;
  for (int64_t e = blockIdx.x * (int64_t)NT + threadIdx.x; e < n; e += stride)
    y[e] = a * x[e] + (b == 0.0 ? 0.0 : b * y[e]);
}

// ------------------------------------------------ 3D solvent-solvent
// beta v_short of every site pair around the grid centre
// (bgy3d_pair_potential, bgy3d-force.c:123-143): LJ with its epsilon *
// 1e8 ceiling and erfc Coulomb with its 1e3 ceiling (bgy3d-force.h:23-88),
// r^2 summed x, y, z (vec_rmap, bgy3d-vec.h:639-648).  pse: [msol][3]
// sigma, epsilon, charge.  Grid: x = chunks of P, y = pair.
__global__ void __launch_bounds__(NT)
pair_field(GridArgs g, const double* __restrict__ sse, double L0, double L1, double L2,
           double h0, double h1, double h2, double* __restrict__ bv) {
  const int p = blockIdx.y;
  int i = 0;
  while ((i + 1) * (i + 2) / 2 <= p) ++i;
  const int j = p - i * (i + 1) / 2;
  const double eps = sqrt(sse[3 * i + 1] * sse[3 * j + 1]);
  const double sig = 0.5 * (sse[3 * i] + sse[3 * j]);
  const double q2 = sse[3 * i + 2] * sse[3 * j + 2];
  const int64_t stride = (int64_t)gridDim.x * NT;
  for (int64_t e = blockIdx.x * (int64_t)NT + threadIdx.x; e < g.P; e += stride) {
    const int x = (int)(e % g.N0);
    const int y = (int)((e / g.N0) % g.N1);
    const int z = (int)(e / ((int64_t)g.N0 * g.N1));
    const double rx = x * h0 - L0 / 2, ry = y * h1 - L1 / 2, rz = z * h2 - L2 / 2;
    const double r = sqrt((rx * rx + ry * ry) + rz * rz);
    double lj;
    if ((sig == 0.0 || eps == 0.0) && r == 0.0) {
      lj = 0.0;
    } else {
      const double sr = sig / r;
      const double sr6 = (sr * sr) * (sr * sr) * (sr * sr);
      const double re = 4 * eps * sr6 * (sr6 - 1);
      lj = (fabs(re) > eps * 1.0e8) ? eps * 1.0e8 : re;
    }
    const double f = erfc(G_COULOMB * r) / r;
    const double cs = (f > 1.0e3) ? EPSILON0INV * q2 * 1.0e3 : EPSILON0INV * q2 * f;
    bv[p * g.P + e] = g.beta * (lj + cs);
  }
}

// Intramolecular omega_ij(k) = sinc(2 pi r_ij / L0 sqrt(k2)), k2 the
// integer kz^2 + ky^2 + kx^2 (omega_intra, bgy3d-pure.c:236-267), into
// w[p * K + e] for the off-diagonal pairs.  rij: [npairs].  Grid: x =
// chunks of K, y = pair.
__global__ void __launch_bounds__(NT)
omega3(GridArgs g, double L0, const double* __restrict__ rij, double* __restrict__ w) {
  const int p = blockIdx.y;
  const int64_t stride = (int64_t)gridDim.x * NT;
  for (int64_t e = blockIdx.x * (int64_t)NT + threadIdx.x; e < g.KT; e += stride) {
    const int x = (int)(e % g.NH);
    if (x >= g.NX) continue;
    const int y = (int)((e / g.NH) % g.TN1);
    const int z = (int)(e / ((int64_t)g.NH * g.TN1));
    const int k2 = z * z + y * y + x * x;
    const double kr = (2.0 * M_PI * rij[p] / L0) * sqrt((double)k2);
    w[p * g.KT + e] = (kr == 0.0) ? 1.0 : sin(kr) / kr;
  }
}

// mu densities of the solvent-solvent pairs (print_chempot m x m,
// hnc3d.c:486-623, 669-687), off-diagonal pairs counted twice: native,
// HNC, KH, GF and, with gout, g = h + 1 per pair.  uL: the unit long-range
// Coulomb in real space, cl = -beta q_i q_j uL.  Neumaier sums per thread,
// part[block * 4 + q].  Grid: x = chunks of P.
__global__ void __launch_bounds__(NT)
mu_pairs(GridArgs g, const double* __restrict__ t, const double* __restrict__ bv,
         const double* __restrict__ uL, double* __restrict__ gout, double* __restrict__ part) {
  __shared__ double red[4][NT / 64];
  double sum[4] = {0, 0, 0, 0}, comp[4] = {0, 0, 0, 0};
  const int64_t stride = (int64_t)gridDim.x * NT;
  for (int64_t e = blockIdx.x * (int64_t)NT + threadIdx.x; e < g.P; e += stride) {
    double v[4] = {0, 0, 0, 0};
    for (int i = 0; i < g.msol; ++i)
      for (int j = 0; j <= i; ++j) {
        const int p = i * (i + 1) / 2 + j;
        const int64_t idx = p * g.P + e;
        const double ti = t[idx], bvi = bv[idx];
        const double c = closure_c<double>(g.closure, g.pse_order, bvi, ti);
        const double h = c + ti;
        const double xx = -bvi + ti;
        const double cl = -g.beta * g.q[i] * g.q[j] * uL[e];
        const double mult = (i == j) ? 1.0 : 2.0;
        v[0] += mult * form_mu(g.closure, g.pse_order, xx, h, c, cl);
        v[1] += mult * form_mu(0, 0, xx, h, c, cl);
        v[2] += mult * form_mu(1, 1, xx, h, c, cl);
        v[3] += mult * form_mu(2, 0, xx, h, c, cl);
        if (gout) gout[idx] = h + 1.0;
      }
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const double s = sum[q] + v[q];
      comp[q] += (fabs(sum[q]) >= fabs(v[q])) ? (sum[q] - s) + v[q] : (v[q] - s) + sum[q];
      sum[q] = s;
    }
  }
  const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const double s = warp_sum(sum[q] + comp[q]);
    if (lane == 0) red[q][w] = s;
  }
  __syncthreads();
  if (threadIdx.x < 4) {
    double s = red[threadIdx.x][0];
    for (int i = 1; i < NT / 64; ++i) s += red[threadIdx.x][i];
    part[(int64_t)blockIdx.x * 4 + threadIdx.x] = s;
  }
}

// chi - 1 of the solvent at the corner from the spectrum W_p = FFT(rho h_p)
// (hnc3d.c:1006-1052): h^3 W s + (omega_p - 1) with omega_ii = 1; out is
// complex [npairs][N2][N1][NX] without the row padding.  Grid: x = chunks
// of K, y = pair.
__global__ void __launch_bounds__(NT)
chi_from_h(GridArgs g, const cpx<double>* __restrict__ W, const double* __restrict__ omega,
           double* __restrict__ out) {
  const int p = blockIdx.y;
  int i = 0;
  while ((i + 1) * (i + 2) / 2 <= p) ++i;
  const int j = p - i * (i + 1) / 2;
  const int64_t stride = (int64_t)gridDim.x * NT;
  const int64_t Kv = (int64_t)g.NX * g.N1 * g.N2;
  for (int64_t e = blockIdx.x * (int64_t)NT + threadIdx.x; e < g.K; e += stride) {
    const int x = (int)(e % g.NH);
    if (x >= g.NX) continue;
    const int y = (int)((e / g.NH) % g.N1);
    const int z = (int)(e / ((int64_t)g.NH * g.N1));
    const int iy = (y <= g.N1 / 2) ? y : y - g.N1;
    const int iz = (z <= g.N2 / 2) ? z : z - g.N2;
    const double sgn = ((x + iy + iz) & 1) ? -1.0 : 1.0;
    const cpx<double> wv = W[p * g.K + e];
    double re = wv.re * g.h3 * sgn, im = wv.im * g.h3 * sgn;
    if (i != j) re += omega[p * g.KT + table_index(g, z, y, x)];
    const int64_t o = p * Kv + ((int64_t)z * g.N1 + y) * g.NX + x;
    out[2 * o] = re;
    out[2 * o + 1] = im;
  }
}

// FP64 -> FP32 copy.
__global__ void __launch_bounds__(NT)
to_f32(float* __restrict__ dst, const double* __restrict__ src, int64_t n) {
  const int64_t stride = (int64_t)gridDim.x * NT;
  for (int64_t e = blockIdx.x * (int64_t)NT + threadIdx.x; e < n; e += stride)
    dst[e] = (float)src[e];
}

// ------------------------------------------------------ info observables
// Solvent charge density rho_v = sum_i (q_i rho) g_i with g_i = (c_i + t_i)
// + 1 (bgy3d_solvent_field, bgy3d-potential.c:246-262, on the g that
// hnc3d.c:2319-2325 passes).  One solute; grid-stride over P.
__global__ void __launch_bounds__(NT)
info_rho_v(GridArgs g, const double* __restrict__ t, const double* __restrict__ bv, double rho,
           double* __restrict__ rhov) {
  const int64_t stride = (int64_t)gridDim.x * NT;
  for (int64_t e = blockIdx.x * (int64_t)NT + threadIdx.x; e < g.P; e += stride) {
    double acc = 0.0;
    for (int i = 0; i < g.m; ++i) {
      const int64_t idx = i * g.P + e;
      const double c = closure_c<double>(g.closure, g.pse_order, bv[idx], t[idx]);
      acc += (g.q[i] * rho * g.rw[i]) * ((c + t[idx]) + 1.0);
    }
    rhov[e] = acc;
  }
}

// The grid sums of print_info (bgy3d-potential.c:341-443), unscaled, with
// X_a = i_a - N_a / 2 (bgy3d_moments, bgy3d-vec.c:573-593):
//   [0..9]   rho_v: 1, X, Y, Z, XX, XY, XZ, YY, YZ, ZZ
//   [10..19] rho_u, the Gaussian cores (G/sqrt(pi))^3 sum_a q_a
//            exp(-G^2 r_a^2) (bgy3d-solutes.c:555-577), same moments
//   [20] U_v rho_u   [21] U_u rho_v, U_u = eps0^-1 sum_a q_a G cl0(G r_a)
// Neumaier sums per thread, part[block * INFO_NSUM + q].  Grid: x = chunks
// of P.
__global__ void __launch_bounds__(NT)
info_sums(GridArgs g, SitesDesc sd, const double* __restrict__ rhov,
          const double* __restrict__ ve, double L0, double L1, double L2, double h0, double h1,
          double h2, double* __restrict__ part) {
  __shared__ double red[INFO_NSUM][NT / 64];
  double sum[INFO_NSUM], comp[INFO_NSUM];
#pragma unroll
  for (int q = 0; q < INFO_NSUM; ++q) { sum[q] = 0.0; comp[q] = 0.0; }
  const double gn = G_COULOMB / sqrt(M_PI);
  const double norm = gn * gn * gn;
  const int64_t stride = (int64_t)gridDim.x * NT;
  for (int64_t e = blockIdx.x * (int64_t)NT + threadIdx.x; e < g.P; e += stride) {
    const int x = (int)(e % g.N0);
    const int y = (int)((e / g.N0) % g.N1);
    const int z = (int)(e / ((int64_t)g.N0 * g.N1));
    const double rx = x * h0 - L0 / 2, ry = y * h1 - L1 / 2, rz = z * h2 - L2 / 2;
    double ru = 0.0, uc = 0.0;
    for (int a = 0; a < sd.n; ++a) {
      const double* s = sd.xyz_s_e_q + 6 * a;
      const double dx = rx - s[0], dy = ry - s[1], dz = rz - s[2];
      const double r2 = (dx * dx + dy * dy) + dz * dz;
      ru += s[5] * exp(-G_COULOMB * G_COULOMB * r2);
      uc += s[5] * G_COULOMB * cl0(G_COULOMB * sqrt(r2));
    }
    ru *= norm;
    uc *= EPSILON0INV;
    const double X = x - 0.5 * g.N0, Y = y - 0.5 * g.N1, Z = z - 0.5 * g.N2;
    const double rv = rhov[e];
    const double w[10] = {1.0, X, Y, Z, X * X, X * Y, X * Z, Y * Y, Y * Z, Z * Z};
    double v[INFO_NSUM];
#pragma unroll
    for (int q = 0; q < 10; ++q) { v[q] = rv * w[q]; v[10 + q] = ru * w[q]; }
    v[20] = ve[e] * ru;
    v[21] = uc * rv;
#pragma unroll
    for (int q = 0; q < INFO_NSUM; ++q) {
      const double s = sum[q] + v[q];
      comp[q] += (fabs(sum[q]) >= fabs(v[q])) ? (sum[q] - s) + v[q] : (v[q] - s) + sum[q];
      sum[q] = s;
    }
  }
  const int wv = threadIdx.x >> 6, lane = threadIdx.x & 63;
#pragma unroll
  for (int q = 0; q < INFO_NSUM; ++q) {
    const double s = warp_sum(sum[q] + comp[q]);
    if (lane == 0) red[q][wv] = s;
  }
  __syncthreads();
  if (threadIdx.x < INFO_NSUM) {
    double s = red[threadIdx.x][0];
    for (int i = 1; i < NT / 64; ++i) s += red[threadIdx.x][i];
    part[(int64_t)blockIdx.x * INFO_NSUM + threadIdx.x] = s;
  }
}

// The solvent potential at the solute sites by trigonometric interpolation
// (bgy3d_pot_interp, bgy3d-potential.c:125-143, and bgy3d_fft_interp,
// bgy3d-fftw3.c:504-612) straight from Y = FFT(rho_v) (spectrum of site 0
// in W, padded rows): FFT(U_v) = N0 N1 N2 Y f / L^3 with the Poisson factor
// f = 4 pi eps0^-1 h^3 / k^2 (0 at k = 0), so
//   U_v(y) = sum_k 2 Re(Y f / L^3 w_x w_y w_z) / (2 if k_x = 0 or N0/2),
// w_d = exp(2 pi i K_d y_d / N_d), cos(...) where K_d = -K_d mod N_d, and
// y_d = (x_d + L_d / 2) / h_d.  xs: [n][3].  part[(a * gridDim.x + block)].
// Grid: x = chunks of K, y = site.
__global__ void __launch_bounds__(NT)
info_interp(GridArgs g, const cpx<double>* __restrict__ W, const double* __restrict__ xs,
            double L0, double L1, double L2, double h0, double h1, double h2,
            double* __restrict__ part) {
  __shared__ double red[NT / 64];
  const int a = blockIdx.y;
  const double yx = (xs[3 * a] + L0 / 2) / h0;
  const double yy = (xs[3 * a + 1] + L1 / 2) / h1;
  const double yz = (xs[3 * a + 2] + L2 / 2) / h2;
  double sum = 0.0, comp = 0.0;
  const int64_t stride = (int64_t)gridDim.x * NT;
  for (int64_t e = blockIdx.x * (int64_t)NT + threadIdx.x; e < g.K; e += stride) {
    const int x = (int)(e % g.NH);
    if (x >= g.NX) continue;
    const int y = (int)((e / g.NH) % g.N1);
    const int z = (int)(e / ((int64_t)g.NH * g.N1));
    const int iy = (y <= g.N1 / 2) ? y : y - g.N1;
    const int iz = (z <= g.N2 / 2) ? z : z - g.N2;
    const double kx = x * g.dkx, ky = iy * g.dky, kz = iz * g.dkz;
    const double k2 = (kz * kz + ky * ky) + kx * kx;
    if (k2 == 0.0) continue;
    const double f = 4 * M_PI * EPSILON0INV * g.h3 / k2 * g.inv_L3;
    // the three one-dimensional waves
    double cx, sx, cy, sy, cz, sz;
    sincos((2 * M_PI / g.N0) * x * yx, &sx, &cx);
    sincos((2 * M_PI / g.N1) * iy * yy, &sy, &cy);
    sincos((2 * M_PI / g.N2) * iz * yz, &sz, &cz);
    if ((g.N0 - 2 * x) % g.N0 == 0) sx = 0.0;
    if ((g.N1 - 2 * y) % g.N1 == 0) sy = 0.0;
    if ((g.N2 - 2 * z) % g.N2 == 0) sz = 0.0;
    // w = wx wy wz
    const double ar = cx * cy - sx * sy, ai = cx * sy + sx * cy;
    const double wr = ar * cz - ai * sz, wi = ar * sz + ai * cz;
    const cpx<double> Yk = W[e];
    double v = 2.0 * f * (Yk.re * wr - Yk.im * wi);
    if ((g.N0 - 2 * x) % g.N0 == 0) v *= 0.5;
    const double s = sum + v;
    comp += (fabs(sum) >= fabs(v)) ? (sum - s) + v : (v - s) + sum;
    sum = s;
  }
  const int wv = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const double s = warp_sum(sum + comp);
  if (lane == 0) red[wv] = s;
  __syncthreads();
  if (threadIdx.x == 0) {
    double acc = red[0];
    for (int i = 1; i < NT / 64; ++i) acc += red[i];
    part[(int64_t)a * gridDim.x + blockIdx.x] = acc;
  }
}

}  // namespace rism

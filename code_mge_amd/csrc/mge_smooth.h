// mge_smooth.h -- implicit residual smoothing (psmoo_old.f90), templated on
// the bulk type T.
//
// psmoo_old solves, for every grid line and each direction in turn, the
// constant-coefficient tridiagonal system (1+2 eps) x_s - eps (x_(s-1) +
// x_(s+1)) = dw_s with a Thomas recurrence whose pivots e1/e2 depend only
// on the line length (psmoo.f90:134-166); blank cells are skipped (their
// value is kept and they do not feed the recurrence).
#pragma once
#include <algorithm>

#include "mge_kernels.h"

namespace mge {

template <typename T>
struct SmoothArgs {
  Dims d;
  T *dw;
  const uint8_t *flags;
  const T *e2;       // pivots of this direction (psmoo.f90:134-166)
  const double *r1;  // 1/e1, e1 rounded to T first
  const T *fa;       // x lines in FP32: -bb/e1
  T bb;
};

// The forward step's division by the pivot e1, r its reciprocal in FP64.
// FP64 multiplies by the reciprocal (one rounding more per cell, a few ulp over
// a line, and no FP64 division on the recurrence's critical path).  In FP32
// this is the quotient the division gives, bit for bit: a quotient of two
// 24-bit numbers that is no FP32 midpoint lies at least 2^-25 ulp from one, and
// the FP64 product is within 2^-28 ulp of it.
template <typename T>
__device__ __attribute__((always_inline)) inline T piv_div(T x, double r) {
  return (T)((double)x * r);
}

// sequential x lines for blocks wider than 512 cells
template <typename T>
__device__ __attribute__((always_inline)) inline void smooth_x_seq(const SmoothArgs<T> &S, int bx) {
  const Dims &d = S.d;
  long t = bx * (long)blockDim.x + threadIdx.x;
  long nl = (long)d.nj * d.nk;
  if (t >= nl * 5) return;
  int n = (int)(t / nl);
  long l = t - (long)n * nl;
  int j = 2 + (int)(l % d.nj), k = 2 + (int)(l / d.nj);
  T *D = S.dw + n * d.E;
  long b0 = ix(d, 0, j, k);
  if (S.flags[b0 + 2] & F_FLUID) D[b0 + 2] = piv_div(D[b0 + 2], S.r1[2]);
  for (int i = 3; i <= d.il; i++)
    if (S.flags[b0 + i] & F_FLUID) D[b0 + i] = piv_div(D[b0 + i] - S.bb * D[b0 + i - 1], S.r1[i]);
  for (int i = 2; i <= d.ni; i++) {
    int ir = d.il + 1 - i;
    if (S.flags[b0 + ir] & F_FLUID) D[b0 + ir] = D[b0 + ir] - S.e2[ir] * D[b0 + ir + 1];
  }
}

template <typename T>
__device__ __attribute__((always_inline)) inline void k_smooth_x_seq_body(const SmoothArgs<T> &S, int bx, int, int) {
  smooth_x_seq(S, bx);
}
MGE_ENTRY_T(k_smooth_x_seq, SmoothArgs, 256, 1)

// One line of the exact sequential recurrence of psmoo_old
// (psmoo.f90:190-237): cells s = 2..nl at stride st.  Full chunks of CH
// cells are read into registers double-buffered with unconditional loads,
// so the compiler can keep the next chunk's loads in flight (counted waits)
// while the current chunk runs its dependent divisions.  The updates are
// branch-free: blank cells hold dw = +-0 (blanked before smoothing), so
// y = m*((r - bb*y)/e1) with m = 0 on blank cells gives the reference's
// values on fluid cells and keeps the zeros.  The backward sweep starts
// at s = nl with z(nl+1) = 0 and e2(nl) = 0, which returns y(nl) there.
template <int CH, typename T>
__device__ __attribute__((always_inline)) inline void line_sweep(T *__restrict__ D, const uint8_t *__restrict__ F,
                                                                 long b0, long st, int nl,
                                                                 const double *__restrict__ r1,
                                                                 const T *__restrict__ e2, T bb) {
  const int ncell = nl - 1;
  const int nfull = ncell / CH;
  T A[CH], B[CH], MA[CH], MB[CH];
  T y = T(0);
#define LD_F(BUF, MK, c)                                              \
  _Pragma("unroll") for (int t = 0; t < CH; t++) {                    \
    long q_ = b0 + (long)(2 + (c) * CH + t) * st;                     \
    BUF[t] = D[q_];                                                   \
    MK[t] = (F[q_] & F_FLUID) ? T(1) : T(0);                          \
  }
#define PR_F(BUF, MK, c)                                              \
  _Pragma("unroll") for (int t = 0; t < CH; t++) {                    \
    int s_ = 2 + (c) * CH + t;                                        \
    y = MK[t] * piv_div(BUF[t] - bb * y, r1[s_]);                 \
    D[b0 + (long)s_ * st] = y;                                        \
  }
#define LD_B(BUF, MK, c)                                              \
  _Pragma("unroll") for (int t = 0; t < CH; t++) {                    \
    long q_ = b0 + (long)(nl - (c) * CH - t) * st;                    \
    BUF[t] = D[q_];                                                   \
    MK[t] = (F[q_] & F_FLUID) ? T(1) : T(0);                          \
  }
#define PR_B(BUF, MK, c)                                              \
  _Pragma("unroll") for (int t = 0; t < CH; t++) {                    \
    int s_ = nl - (c) * CH - t;                                       \
    y = BUF[t] - MK[t] * (e2[s_] * y);                                \
    D[b0 + (long)s_ * st] = y;                                        \
  }
  // forward
  if (nfull > 0) {
    LD_F(A, MA, 0);
    for (int c = 0; c < nfull; c += 2) {
      int c1 = c + 1 < nfull ? c + 1 : c;
      LD_F(B, MB, c1);
      PR_F(A, MA, c);
      if (c + 1 >= nfull) break;
      int c2 = c + 2 < nfull ? c + 2 : c + 1;
      LD_F(A, MA, c2);
      PR_F(B, MB, c + 1);
    }
  }
  for (int s_ = 2 + nfull * CH; s_ <= nl; s_++) {
    long q_ = b0 + (long)s_ * st;
    T m_ = (F[q_] & F_FLUID) ? T(1) : T(0);
    y = m_ * piv_div(D[q_] - bb * y, r1[s_]);
    D[q_] = y;
  }
  // backward
  y = T(0);
  if (nfull > 0) {
    LD_B(A, MA, 0);
    for (int c = 0; c < nfull; c += 2) {
      int c1 = c + 1 < nfull ? c + 1 : c;
      LD_B(B, MB, c1);
      PR_B(A, MA, c);
      if (c + 1 >= nfull) break;
      int c2 = c + 2 < nfull ? c + 2 : c + 1;
      LD_B(A, MA, c2);
      PR_B(B, MB, c + 1);
    }
  }
  for (int s_ = nl - nfull * CH; s_ >= 2; s_--) {
    long q_ = b0 + (long)s_ * st;
    T m_ = (F[q_] & F_FLUID) ? T(1) : T(0);
    y = D[q_] - m_ * (e2[s_] * y);
    D[q_] = y;
  }
#undef LD_F
#undef PR_F
#undef LD_B
#undef PR_B
}

// psmoo.f90:190-206 (y lines of more than 512 cells); thread per (i,k) and component
template <typename T>
__device__ __attribute__((always_inline)) inline void k_smooth_y_body(const SmoothArgs<T> &S, int bx, int by, int bz) {
  const Dims &d = S.d;
  int i = 2 + bx * blockDim.x + threadIdx.x;
  int k = 2 + by;
  int n = bz;
  if (i > d.il) return;
  line_sweep<8>(S.dw + n * d.E, S.flags, ix(d, i, 0, k), d.sy, d.jl, S.r1, S.e2, S.bb);
}
MGE_ENTRY_T_XCD(k_smooth_y, SmoothArgs, 64, 1)

// psmoo.f90:209-237 (z lines of more than 512 cells); thread per (i,j) and component
template <typename T>
__device__ __attribute__((always_inline)) inline void k_smooth_z_body(const SmoothArgs<T> &S, int bx, int by, int bz) {
  const Dims &d = S.d;
  int i = 2 + bx * blockDim.x + threadIdx.x;
  int j = 2 + by;
  int n = bz;
  if (i > d.il) return;
  line_sweep<8>(S.dw + n * d.E, S.flags, ix(d, i, j, 0), d.sz, d.kl, S.r1, S.e2, S.bb);
}
MGE_ENTRY_T_XCD(k_smooth_z, SmoothArgs, 64, 1)

// ---- x lines in FP32: scanned across a wave -------------------------------
//
// Lane l of a group of W lanes owns the CPL cells s0 .. s0 + CPL - 1 of each of
// K lines of n cells (ok: the cell is on the line, fl: fluid).  Both recurrences
// are composed as affine maps (forward y_i = A_i y_(i-1) + B_i, backward z_i =
// C_i z_(i+1) + y_i), scanned over the lanes, and each lane evaluates its own
// cells with the reference formula from the value that enters.  pr: 1/e1, pa:
// -bb/e1, pe2: e2 of the lane's cells.  FP32 keeps this order of operations
// where FP64 joins segments: another order rounds the entering values
// otherwise, and where a far-field face's normal velocity is next to 0 a last
// bit decides between inflow and outflow (3e-3 of a cell's value).
template <int CPL, int K>
__device__ __attribute__((always_inline)) inline void scan_lines(float (&r)[K][CPL], const bool (&fl)[K][CPL],
                                                                 const bool (&ok)[CPL], int s0, int n, int l, int W,
                                                                 const double (&pr)[CPL], const float (&pa)[CPL],
                                                                 const float (&pe2)[CPL], float bb) {
  float Al[K], Bl[K];
#pragma unroll
  for (int t = 0; t < K; t++) {
    Al[t] = 1.0f;
    Bl[t] = 0.0f;
#pragma unroll
    for (int c = 0; c < CPL; c++) {
      float A, B;
      if (!ok[c]) { A = 1.0f; B = 0.0f; }
      else if (!fl[t][c]) { A = 0.0f; B = r[t][c]; }
      else if (s0 + c == 0) { A = 0.0f; B = piv_div(r[t][c], pr[c]); }
      else { A = pa[c]; B = piv_div(r[t][c], pr[c]); }
      Bl[t] = A * Bl[t] + B;
      Al[t] = A * Al[t];
    }
  }
  for (int off = 1; off < W; off <<= 1) {
#pragma unroll
    for (int t = 0; t < K; t++) {
      const float Ap = __shfl_up(Al[t], off, W), Bp = __shfl_up(Bl[t], off, W);
      if (l >= off) {
        Bl[t] = Al[t] * Bp + Bl[t];
        Al[t] = Al[t] * Ap;
      }
    }
  }
#pragma unroll
  for (int t = 0; t < K; t++) {
    float yp = __shfl_up(Bl[t], 1, W);
    if (l == 0) yp = 0.0f;
#pragma unroll
    for (int c = 0; c < CPL; c++) {
      float v = r[t][c];
      if (fl[t][c]) v = piv_div(s0 + c == 0 ? r[t][c] : r[t][c] - bb * yp, pr[c]);
      r[t][c] = v;
      yp = v;
    }
  }
  // backward: C_i = -e2_i on fluid cells but the line's last
#pragma unroll
  for (int t = 0; t < K; t++) {
    Al[t] = 1.0f;
    Bl[t] = 0.0f;
#pragma unroll
    for (int c = CPL - 1; c >= 0; c--) {
      float C, D;
      if (!ok[c]) { C = 1.0f; D = 0.0f; }
      else if (fl[t][c] && s0 + c < n - 1) { C = -pe2[c]; D = r[t][c]; }
      else { C = 0.0f; D = r[t][c]; }
      Bl[t] = C * Bl[t] + D;
      Al[t] = C * Al[t];
    }
  }
  for (int off = 1; off < W; off <<= 1) {
#pragma unroll
    for (int t = 0; t < K; t++) {
      const float Cn = __shfl_down(Al[t], off, W), Dn = __shfl_down(Bl[t], off, W);
      if (l + off < W) {
        Bl[t] = Al[t] * Dn + Bl[t];
        Al[t] = Al[t] * Cn;
      }
    }
  }
#pragma unroll
  for (int t = 0; t < K; t++) {
    float zn = __shfl_down(Bl[t], 1, W);
    if (l == W - 1) zn = 0.0f;
#pragma unroll
    for (int c = CPL - 1; c >= 0; c--) {
      if (!ok[c]) continue;
      if (fl[t][c] && s0 + c < n - 1) r[t][c] = r[t][c] - pe2[c] * zn;
      zn = r[t][c];
    }
  }
}

// a lane moves its CPL cells as pairs when CPL is even, the line's first
// cell (i = 2) sits on a pair boundary (so does every lane's first cell,
// i0 - 2 being a multiple of CPL) and all its cells are inside the line
template <int CPL>
__device__ __attribute__((always_inline)) inline bool xscan_pairs(const float *row, int i0, int il) {
  if constexpr (CPL % 2 != 0) return false;
  else return ((reinterpret_cast<uintptr_t>(row + 2) & (2 * sizeof(float) - 1)) == 0) && i0 + CPL - 1 <= il;
}

// x lines of levels whose planes do not fit k_smooth_xy: a wave takes K
// consecutive (j,k) lines of a component; the lines' loads are in flight
// together and their shuffles interleave.  Four lines of up to 256 cells
// share a wave, 512-cell lines take one (256^3: one, two and four lines 409,
// 339 and 324 us with single loads; with pairs, four lines 304 us; with the
// quotients by reciprocal pivots 250 us).
template <int CPL>
constexpr int xscan_lines() { return CPL >= 8 ? 1 : 4; }
template <int CPL>
__device__ __attribute__((always_inline)) inline void smooth_x_scan(const SmoothArgs<float> &S, int bx) {
  constexpr int K = xscan_lines<CPL>();
  const Dims &d = S.d;
  const int lane = threadIdx.x & 63;
  // the wave index is uniform: keep the line arithmetic scalar
  const int wave = __builtin_amdgcn_readfirstlane((int)((bx * (long)blockDim.x + threadIdx.x) >> 6));
  const int nl = d.nj * d.nk, nlines = nl * 5, l0 = wave * K;
  if (l0 >= nlines) return;  // uniform per wave
  const int il = d.il, i0 = 2 + lane * CPL;
  double pr[CPL];
  float pa[CPL], pe2[CPL];
  bool ok[CPL];
#pragma unroll
  for (int c = 0; c < CPL; c++) {
    ok[c] = i0 + c <= il;
    const int ic = ok[c] ? i0 + c : 2;
    pr[c] = S.r1[ic];
    pa[c] = S.fa[ic];
    pe2[c] = S.e2[ic];
  }
  float r[K][CPL];
  bool fl[K][CPL];
  long base[K];
#pragma unroll
  for (int t = 0; t < K; t++) {
    const int lc = l0 + t < nlines ? l0 + t : l0;  // a missing line repeats the first; it is never stored
    const int n = lc / nl, l = lc - n * nl;
    const long f = ix(d, 0, 2 + l % d.nj, 2 + l / d.nj);
    base[t] = (long)n * d.E + f;
    if (xscan_pairs<CPL>(S.dw + base[t], i0, il)) {
      const float2 *pp = reinterpret_cast<const float2 *>(S.dw + base[t] + i0);
#pragma unroll
      for (int h = 0; h < CPL / 2; h++) {
        const float2 v = pp[h];
        r[t][2 * h] = v.x;
        r[t][2 * h + 1] = v.y;
      }
    } else {
#pragma unroll
      for (int c = 0; c < CPL; c++) r[t][c] = ok[c] ? S.dw[base[t] + i0 + c] : 0.0f;
    }
#pragma unroll
    for (int c = 0; c < CPL; c++) fl[t][c] = ok[c] && (S.flags[f + i0 + c] & F_FLUID);
  }
  scan_lines<CPL, K>(r, fl, ok, i0 - 2, d.ni, lane, 64, pr, pa, pe2, S.bb);
#pragma unroll
  for (int t = 0; t < K; t++) {
    if (l0 + t >= nlines) continue;
    if (xscan_pairs<CPL>(S.dw + base[t], i0, il)) {
      // blank cells are written back with the value they were read with
      float2 *pp = reinterpret_cast<float2 *>(S.dw + base[t] + i0);
#pragma unroll
      for (int h = 0; h < CPL / 2; h++) pp[h] = float2{r[t][2 * h], r[t][2 * h + 1]};
    } else {
#pragma unroll
      for (int c = 0; c < CPL; c++)
        if (fl[t][c]) S.dw[base[t] + i0 + c] = r[t][c];
    }
  }
}
// one pair of entry points per scan width; a batch launches each width once
// over the cases that use it
template <int CPL>
__global__ void __launch_bounds__(256) k_smooth_x_scan(SmoothArgs<float> S) {
  smooth_x_scan<CPL>(S, (int)blockIdx.x);
}
template <int CPL>
__global__ void __launch_bounds__(256) k_smooth_x_scan_b(const SmoothArgs<float> *As, const int4 *cg, int nc,
                                                         const int *act) {
  const int b = (int)blockIdx.x;
  const int c = batch_case(cg, nc, b);
  const int4 g = cg[c];
  if (!act[g.w]) return;
  smooth_x_scan<CPL>(As[c], b - g.x);
}

// ---- lines in segments ---------------------------------------------------
//
// A line split into segments of L cells, one thread each, all of its cells in
// registers; the segments are joined through LDS.
//
// FP64: both recurrences are evaluated within the segment from zero, giving
// the segment's map from the value entering it to the value leaving it; every
// thread then runs through the maps before (backward: after) it and
// re-evaluates its cells with the reference formula from the value entering.
// The entering values are a few ulp from the sequential ones.
//
// FP32: the bits of the sequential recurrence.  Every segment evaluates its
// cells from the value its neighbour leaves, and again as long as that value
// changes, up to the cell from which nothing changes any more.  Segment g is
// final after g rounds at the latest; as a change shrinks by bb/e1 a cell (0.3
// at the default coefficient, 4e-9 over 16 cells), the third round mostly ends
// it.  Thread per line -> this -> joined by maps as FP64 (other last bits), y
// lines: 96^3 31 -> 20 -> 15.5 us, 256^3 243 -> 199 -> 185 us.
//
// Branch-free: a cell's fluid bit selects its pivots or zeros (blank cells
// hold dw = +-0, see line_sweep, and come out as 0), and the places past the
// line's end count as blank; a branch per cell would wait for every LDS read
// by itself (64^3 in k_smooth_xy: 25 us with branches, 13 without).
// Called by all threads of the workgroup (barriers); sa, sb, sc, sd: LDS of
// G x nline values each (FP32: sa and sc alone); `act` threads hold segment g
// of line `line`.
template <typename T>
struct SegPiv {   // a line's pivots, in LDS, indexed by cell from 0
  const double *r1;
  const T *e2;
};
template <int L>
__device__ __attribute__((always_inline)) inline void seg_solve(bool act, float (&r)[L], unsigned fl, int s0, int g,
                                                                int G, int line, int nline, const SegPiv<float> &P,
                                                                float bb, float *sa, float *, float *sc, float *) {
  auto rm = [&](int c) { return (fl >> c) & 1u ? P.r1[s0 + c] : 0.0; };
  auto qm = [&](int c) { return (fl >> c) & 1u ? P.e2[s0 + c] : 0.0f; };
  float v[L], in = 0.0f;
  bool again;
  // takes `in` from segment nb's place (none: zero); whether any thread's changed
  auto join = [&](const float *s, int nb, bool none) {
    __syncthreads();
    const float x = act && !none ? s[nb * nline + line] : 0.0f;
    again = __float_as_uint(x) != __float_as_uint(in);
    in = x;
    return __syncthreads_or(again) != 0;
  };
  // cell c's new value; true every fourth cell if no thread's value there changed
  auto put = [&](float &o, float x, int c, bool first) {
    const bool diff = __float_as_uint(x) != __float_as_uint(o);
    o = x;
    return !first && c % 4 == 3 && !__any(diff);
  };
  auto forward = [&](bool first) {
    float y = in;
#pragma unroll
    for (int c = 0; c < L; c++) {
      y = piv_div(r[c] - bb * y, rm(c));
      if (put(v[c], y, c, first)) return;
    }
    if (act) sa[g * nline + line] = y;
  };
  forward(true);
  for (int it = 1; it < G && join(sa, g - 1, g == 0); it++)   // uniform
    if (again) forward(false);
  // backward: z = y - e2 z', e2 = 0 on the line's last cell
  in = 0.0f;
  auto backward = [&](bool first) {
    float z = in;
#pragma unroll
    for (int c = 0; c < L; c++) {
      const int b = L - 1 - c;
      z = v[b] - qm(b) * z;
      if (put(r[b], z, c, first)) return;
    }
    if (act) sc[g * nline + line] = z;
  };
  backward(true);
  for (int it = 1; it < G && join(sc, g + 1, g == G - 1); it++)
    if (again) backward(false);
}
template <int L>
__device__ __attribute__((always_inline)) inline void seg_solve(bool act, double (&r)[L], unsigned fl, int s0, int g,
                                                                int G, int line, int nline, const SegPiv<double> &P,
                                                                double bb, double *sa, double *sb, double *sc,
                                                                double *sd) {
  auto rm = [&](int c) { return (fl >> c) & 1u ? P.r1[s0 + c] : 0.0; };
  auto qm = [&](int c) { return (fl >> c) & 1u ? P.e2[s0 + c] : 0.0; };
  double A = 1.0, B = 0.0;
#pragma unroll
  for (int c = 0; c < L; c++) {
    const double m = rm(c);
    B = piv_div(r[c] - bb * B, m);
    A = A * (-bb * m);
  }
  if (act) {
    sa[g * nline + line] = A;
    sb[g * nline + line] = B;
  }
  __syncthreads();
  double y = 0.0;
  for (int q = 0; q < G - 1; q++) {   // uniform; the maps before this segment
    const double ny = sa[q * nline + line] * y + sb[q * nline + line];
    y = q < g ? ny : y;
  }
  double C = 1.0, D = 0.0;
#pragma unroll
  for (int c = 0; c < L; c++) {
    y = piv_div(r[c] - bb * y, rm(c));
    r[c] = y;
  }
  // backward: z = y - e2 z', e2 = 0 on the line's last cell
#pragma unroll
  for (int c = L - 1; c >= 0; c--) {
    const double m = qm(c);
    D = r[c] - m * D;
    C = -(m * C);
  }
  if (act) {
    sc[g * nline + line] = C;
    sd[g * nline + line] = D;
  }
  __syncthreads();
  double z = 0.0;
  for (int q = G - 1; q > 0; q--) {
    const double nz = sc[q * nline + line] * z + sd[q * nline + line];
    z = q > g ? nz : z;
  }
#pragma unroll
  for (int c = L - 1; c >= 0; c--) {
    z = r[c] - qm(c) * z;
    r[c] = z;
  }
}

// x and y lines of a level whose k planes fit the LDS: a workgroup holds one
// plane of one component, solves its x lines, then its y lines, and writes it
// once.  In x a wave's lanes take neighbouring rows (the row length is odd in
// LDS, so they fall on different banks), in y neighbouring columns.  The
// separate launches read and write the field twice and, on small levels, wait
// for one thread's walk along a whole line.  The plane's memory also carries
// the segments' maps while its cells are in registers.  FP64, x and y sweeps
// as they were -> this: 32^3 13.7 -> 6 us, 48^3 19 -> 8 us, 64^3 31 -> 13 us.
template <typename T>
struct SmoothXYArgs {
  Dims d;
  T *dw;
  const uint8_t *flags;
  const T *e2x, *e2y;
  const double *r1x, *r1y;
  const T *fax;
  T bb;
};
// FP32 scans its x lines while it reads them (scan_lines; rows of up to 64
// cells, one cell a lane): x and y of 48^3 24 us in two launches, 16 in this.
// plane classes: cells of LDS (rows of nx | 1), mask words, pivots per
// direction, threads, segment length.  Planes of more than 64 x 65 cells leave
// too few workgroups a CU: 128 x 128 x 4 took 21 us in one launch, 11 in two.
struct XYClass {
  int cells, words, piv, threads, seg;
};
constexpr XYClass kXY[2] = {{2560, 128, 264, 512, 8}, {4416, 256, 264, 512, 8}};
// the class that holds an nx x ny plane (-1: none)
template <typename T>
int xy_class(int nx, int ny) {
  if (kDelta<T> && nx > 64) return -1;
  for (int c = 0; c < 2; c++) {
    const XYClass &K = kXY[c];
    const int gx = (nx + K.seg - 1) / K.seg, gy = (ny + K.seg - 1) / K.seg;
    const long lx = (long)ny * gx, ly = (long)nx * gy;
    if ((long)(nx | 1) * ny <= K.cells && (long)ny * ((nx + 63) / 64) <= K.words && lx <= K.threads &&
        ly <= K.threads && 4 * std::max(lx, ly) <= K.cells && std::max(gx, gy) * K.seg <= K.piv)
      return c;
  }
  return -1;
}

template <typename T, int CLS>
__device__ __attribute__((always_inline)) inline void k_smooth_xy_body(const SmoothXYArgs<T> &S, int bx, int by) {
  constexpr XYClass K = kXY[CLS];
  constexpr int L = K.seg;
  constexpr bool SCAN = kDelta<T>;
  __shared__ T pl[K.cells];
  __shared__ double pr[SCAN ? 1 : 2][K.piv];   // y, x: 1/e1
  __shared__ T pe[SCAN ? 1 : 2][K.piv];        // y, x: e2
  __shared__ unsigned long long mk[K.words];
  const Dims &d = S.d;
  const int nx = d.ni, ny = d.nj, P = nx | 1, nch = (nx + 63) >> 6;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  for (int t = tid; t < K.piv; t += K.threads) {
    const int ix2 = 2 + min(t, nx - 1), iy2 = 2 + min(t, ny - 1);
    pr[0][t] = S.r1y[iy2];
    pe[0][t] = S.e2y[iy2];
    if constexpr (!SCAN) {
      pr[1][t] = S.r1x[ix2];
      pe[1][t] = S.e2x[ix2];
    }
  }
  // rows by groups of lp lanes (a power of two), RW rows a wave
  const int lp = nx > 32 ? 64 : (nx > 16 ? 32 : (nx > 8 ? 16 : 8));
  const int sub = lane / lp, l = lane & (lp - 1), RW = 64 / lp;
  const long base = ix(d, 2, 2, 2 + bx);
  T *D = S.dw + by * d.E + base;
  const uint8_t *F = S.flags + base;
  constexpr int NW = K.threads / 64, U = 8;
  double xr[1];   // FP32: the pivots of the lane's cell
  T xa[1], xe2[1];
  if constexpr (SCAN) {
    const int ic = 2 + min(l, nx - 1);
    xr[0] = S.r1x[ic];
    xa[0] = S.fax[ic];
    xe2[0] = S.e2x[ic];
  }
  for (int ch = 0; ch < nch; ch++) {
    const int i = (ch << 6) + l, ic = min(i, nx - 1);
    for (int t0 = wave * RW + sub; t0 - sub < ny; t0 += NW * RW * U) {
      T v[U];
      uint8_t f[U];
#pragma unroll
      for (int u = 0; u < U; u++) {
        const long q = (long)min(t0 + u * NW * RW, ny - 1) * d.sy + ic;
        v[u] = D[q];
        f[u] = F[q];
      }
      if constexpr (SCAN) {
        const bool ok[1] = {i < nx};
        constexpr int KR = 2;   // rows scanned together (planes of 12^2 to 48^2 in a batch: 25 us; all eight 35 us)
#pragma unroll
        for (int g = 0; g < U; g += KR) {
          if (t0 - sub + g * NW * RW >= ny) break;   // rows past the plane (uniform in the wave)
          T x[KR][1];
          bool xf[KR][1];
#pragma unroll
          for (int u = 0; u < KR; u++) {
            x[u][0] = v[g + u];
            xf[u][0] = ok[0] && (f[g + u] & F_FLUID);
          }
          scan_lines<1, KR>(x, xf, ok, i, nx, l, lp, xr, xa, xe2, S.bb);
#pragma unroll
          for (int u = 0; u < KR; u++) v[g + u] = x[u][0];
        }
      }
#pragma unroll
      for (int u = 0; u < U; u++) {
        const int row = t0 + u * NW * RW;
        const unsigned long long b = __ballot(i < nx && (f[u] & F_FLUID));
        if (row < ny) {
          if (i < nx) pl[row * P + i] = v[u];
          if (l == 0) mk[ch * ny + row] = lp == 64 ? b : (b >> (sub * lp)) & ((1ull << lp) - 1ull);
        }
      }
    }
  }
  __syncthreads();
  T r[L];
  if constexpr (!SCAN) {  // x lines
    const int G = (nx + L - 1) / L, line = tid % ny, g = tid / ny;
    const bool act = g < G;
    const int i0 = act ? g * L : 0, m = act ? min(L, nx - i0) : 0;
    const int c0 = i0 >> 6, sh = i0 & 63;
    unsigned fl = (unsigned)(mk[c0 * ny + line] >> sh);
    if (sh + L > 64) fl |= c0 + 1 < nch ? (unsigned)(mk[(c0 + 1) * ny + line] << (64 - sh)) : 0u;
    const T *row = pl + line * P;
#pragma unroll
    for (int c = 0; c < L; c++) r[c] = row[min(i0 + c, nx - 1)];
    __syncthreads();
    const int n = G * ny;
    seg_solve<L>(act, r, fl, i0, g, G, line, ny, SegPiv<T>{pr[1], pe[1]}, S.bb, pl, pl + n,
                 pl + 2 * n, pl + 3 * n);
    __syncthreads();
#pragma unroll
    for (int c = 0; c < L; c++)
      if (c < m) pl[line * P + i0 + c] = r[c];
  }
  __syncthreads();
  {  // y lines
    const int G = (ny + L - 1) / L, line = tid % nx, g = tid / nx;
    const bool act = g < G;
    const int j0 = act ? g * L : 0, m = act ? min(L, ny - j0) : 0;
    unsigned fl = 0;
    const unsigned long long *mc = mk + (line >> 6) * ny;
#pragma unroll
    for (int c = 0; c < L; c++) {
      const int j = min(j0 + c, ny - 1);
      r[c] = pl[j * P + line];
      fl |= ((unsigned)(mc[j] >> (line & 63)) & (j0 + c < ny ? 1u : 0u)) << c;
    }
    __syncthreads();
    const int n = G * nx;
    seg_solve<L>(act, r, fl, j0, g, G, line, nx, SegPiv<T>{pr[0], pe[0]}, S.bb, pl, pl + n,
                 pl + 2 * n, pl + 3 * n);
    __syncthreads();
#pragma unroll
    for (int c = 0; c < L; c++)
      if (c < m) pl[(j0 + c) * P + line] = r[c];
  }
  __syncthreads();
  for (int ch = 0; ch < nch; ch++) {
    const int i = (ch << 6) + l;
    if (i >= nx) continue;
#pragma unroll 4
    for (int row = wave * RW + sub; row < ny; row += NW * RW) D[(long)row * d.sy + i] = pl[row * P + i];
  }
}
template <typename T, int CLS>
__global__ void __launch_bounds__(kXY[CLS].threads) k_smooth_xy(SmoothXYArgs<T> S) {
  k_smooth_xy_body<T, CLS>(S, (int)blockIdx.x, (int)blockIdx.y);
}
template <typename T, int CLS>
__global__ void __launch_bounds__(kXY[CLS].threads)
    k_smooth_xy_b(const SmoothXYArgs<T> *As, const int4 *cg, int nc, const int *act) {
  const int b = (int)blockIdx.x;
  const int c = batch_case(cg, nc, b);
  const int4 g = cg[c];
  if (!act[g.w]) return;
  const int l = b - g.x;
  k_smooth_xy_body<T, CLS>(As[c], l % g.y, l / g.y);
}

// y (DIR 1) or z (DIR 2) lines in segments: a workgroup takes SX lines that
// lie side by side in x, one thread a segment of L cells, so the field is read
// once and written once and no thread walks a whole line.  Lines of up to 16
// cells are one segment (64 lines a wave), up to 256 cells 32 lines in 16
// segments of 8 or 16, up to 512 cells 16 lines in 32.  Bound by the field's
// one read and write where the level is large.  Thread per line before ->
// this, FP64 y lines: 256^3 421 -> 296 us (4.6 TB/s); 128^3 46 -> 32 us; 512 x
// 512 x 4 105 -> 26 us.  FP32 takes 16 cells beyond 16: the fewer rounds (96^3
// 25 us with 8).
struct SegShape {
  int sx, len;   // lines side by side, cells per segment (0: too long)
};
template <typename T>
SegShape seg_shape(int n) {
  if (n <= 16) return SegShape{64, n <= 4 ? 4 : (n <= 8 ? 8 : 16)};
  if (n <= 256) return SegShape{32, n <= 128 && !kDelta<T> ? 8 : 16};
  return n <= 512 ? SegShape{16, 16} : SegShape{0, 0};
}
template <typename T, int SX, int L, int DIR>
__device__ __attribute__((always_inline)) inline void k_smooth_seg_body(const SmoothArgs<T> &S, int bx, int by,
                                                                        int bz) {
  constexpr int GM = SX == 64 ? 1 : 512 / SX;
  __shared__ T sh[4][GM * SX], pe[L * GM];
  __shared__ double pr[L * GM];
  const Dims &d = S.d;
  const int n = DIR == 1 ? d.nj : d.nk, G = (n + L - 1) / L;
  const long st = DIR == 1 ? d.sy : d.sz;
  const int line = threadIdx.x & (SX - 1), g = threadIdx.x / SX;
  const int i = 2 + bx * SX + line;
  const bool act = g < G && i <= d.il;
  const int s0 = g < G ? g * L : 0, m = act ? min(L, n - s0) : 0;
  const long q0 = DIR == 1 ? ix(d, min(i, d.il), 2, 2 + by) : ix(d, min(i, d.il), 2 + by, 2);
  T *D = S.dw + bz * d.E + q0;
  const uint8_t *F = S.flags + q0;
  T r[L];
  unsigned fl = 0;
#pragma unroll
  for (int c = 0; c < L; c++) {
    const long o = (long)min(s0 + c, n - 1) * st;
    r[c] = D[o];
    fl |= (F[o] & F_FLUID && s0 + c < n ? 1u : 0u) << c;
  }
  for (int t = threadIdx.x; t < G * L; t += blockDim.x) {
    const int s = 2 + min(t, n - 1);
    pr[t] = S.r1[s];
    pe[t] = S.e2[s];
  }
  __syncthreads();
  seg_solve<L>(act, r, fl, s0, g, G, line, SX, SegPiv<T>{pr, pe}, S.bb, sh[0], sh[1], sh[2], sh[3]);
#pragma unroll
  for (int c = 0; c < L; c++)
    if (c < m) D[(long)(s0 + c) * st] = r[c];
}
template <typename T, int SX, int L, int DIR>
__global__ void __launch_bounds__(SX == 64 ? 64 : 512) k_smooth_seg(SmoothArgs<T> S) {
  int bx, by, bz;
  xcd_block(bx, by, bz);
  k_smooth_seg_body<T, SX, L, DIR>(S, bx, by, bz);
}
template <typename T, int SX, int L, int DIR>
__global__ void __launch_bounds__(SX == 64 ? 64 : 512)
    k_smooth_seg_b(const SmoothArgs<T> *As, const int4 *cg, int nc, const int *act) {
  const int b = (int)blockIdx.x;
  const int c = batch_case(cg, nc, b);
  const int4 g = cg[c];
  if (!act[g.w]) return;
  const int l = b - g.x;
  k_smooth_seg_body<T, SX, L, DIR>(As[c], l % g.y, (l / g.y) % g.z, l / (g.y * g.z));
}

// FP64 x lines in segments of 16 cells, where the planes do not fit k_smooth_xy:
// a workgroup stages 16 (N = 128: 32) rows of up to N cells in LDS (whole rows,
// so loads and stores are coalesced), each thread takes a segment.  With lines
// scanned across a wave's lanes by shuffles -> this: 256^3 FP64 399 -> 286 us
// (4.7 TB/s); 128^3 54 -> 48 us; 96^3 33 -> 24 us.
template <int N>
constexpr int xseg_rows() { return N == 128 ? 32 : 16; }
template <int N>
__device__ __attribute__((always_inline)) inline void k_smooth_xseg_body(const SmoothArgs<double> &S, int bx, int by) {
  constexpr int L = 16, kXR = xseg_rows<N>(), NT = kXR * N / L, NW = NT / 64;
  __shared__ double pl[kXR * (N + 1)], pr[N], pe[N];
  __shared__ unsigned long long mk[kXR * N / 64];
  const Dims &d = S.d;
  const int nx = d.ni, P = nx | 1, nch = (nx + 63) >> 6, G = (nx + L - 1) / L;
  const int nl = d.nj * d.nk, l0 = bx * kXR, rows = min(kXR, nl - l0);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  double *D = S.dw + by * d.E;
  auto at = [&](int row) {   // the first cell of the workgroup's row
    const int l = l0 + min(row, rows - 1), k = l / d.nj;
    return ix(d, 2, 2 + l - k * d.nj, 2 + k);
  };
  for (int t = tid; t < G * L; t += NT) {
    const int s = 2 + min(t, nx - 1);
    pr[t] = S.r1[s];
    pe[t] = S.e2[s];
  }
  constexpr int RW = kXR / NW;                      // rows of a wave
  constexpr int U = N / 64;                         // chunks of a row
#pragma unroll 2
  for (int u = 0; u < RW; u++) {
    const int row = wave * RW + u;
    const long q = at(row);
    double v[U];
    uint8_t f[U];
#pragma unroll
    for (int c = 0; c < U; c++) {
      const int i = min(c * 64 + lane, nx - 1);
      v[c] = D[q + i];
      f[c] = S.flags[q + i];
    }
#pragma unroll
    for (int c = 0; c < U; c++) {
      const int i = c * 64 + lane;
      const unsigned long long b = __ballot(i < nx && (f[c] & F_FLUID));
      if (i < nx) pl[row * P + i] = v[c];
      if (lane == 0) mk[c * kXR + row] = b;
    }
  }
  __syncthreads();
  const int line = tid & (kXR - 1), g = tid / kXR;
  const bool act = g < G;
  const int i0 = act ? g * L : 0, m = act ? min(L, nx - i0) : 0;
  const unsigned fl = (unsigned)(mk[(i0 >> 6) * kXR + line] >> (i0 & 63)) & 0xffffu;
  double r[L];
#pragma unroll
  for (int c = 0; c < L; c++) r[c] = pl[line * P + min(i0 + c, nx - 1)];
  __syncthreads();
  const int n = G * kXR;
  seg_solve<L>(act, r, fl, i0, g, G, line, kXR, SegPiv<double>{pr, pe}, S.bb, pl, pl + n, pl + 2 * n,
               pl + 3 * n);
  __syncthreads();
#pragma unroll
  for (int c = 0; c < L; c++)
    if (c < m) pl[line * P + i0 + c] = r[c];
  __syncthreads();
#pragma unroll 2
  for (int u = 0; u < RW; u++) {
    const int row = wave * RW + u;
    if (row >= rows) break;
    const long q = at(row);
#pragma unroll
    for (int c = 0; c < U; c++) {
      const int i = c * 64 + lane;
      if (i < nx) D[q + i] = pl[row * P + i];   // blank cells: 0
    }
  }
}
template <int N>
__global__ void __launch_bounds__(xseg_rows<N>() * N / 16) k_smooth_xseg(SmoothArgs<double> S) {
  int bx, by, bz;
  xcd_block(bx, by, bz);
  k_smooth_xseg_body<N>(S, bx, by);
}
template <int N>
__global__ void __launch_bounds__(xseg_rows<N>() * N / 16)
    k_smooth_xseg_b(const SmoothArgs<double> *As, const int4 *cg, int nc, const int *act) {
  const int b = (int)blockIdx.x;
  const int c = batch_case(cg, nc, b);
  const int4 g = cg[c];
  if (!act[g.w]) return;
  const int l = b - g.x;
  k_smooth_xseg_body<N>(As[c], l % g.y, l / g.y);
}

// ---- psmoo (psmoo.f90:1-95) with progon3's sweep (progon3.f90:1-62) ------
// Rows (1+2e_r) x_r - e_r x_{r-1} - e_r x_{r+1} = d_r along each line of
// direction DIR with the per-cell coefficients e of timestep (the end
// couplings removed, as psmoo passes them, so progon3's sweep is the Thomas
// recurrence).  One thread per line carries all five components: the
// forward sweep leaves u_{r+1} in dw and v_{r+1} in vb, the backward sweep
// forms x_r = v_{r+1} x_{r+1} + u_{r+1} in place.  Lines are numbered with
// the fastest index of the other two first, so neighbouring threads touch
// neighbouring cells on y and z lines.
template <typename T>
struct PsmooArgs {
  Dims d;
  T *dw;
  const T *eps;  // this direction's coefficients
  T *vb;         // per-cell scratch of the forward sweep (E)
};

template <int DIR, typename T>
__device__ __attribute__((always_inline)) inline void k_psmoo_line_body(const PsmooArgs<T> &A, int bx, int, int) {
  const Dims &d = A.d;
  const int t = bx * blockDim.x + threadIdx.x;
  int n, na, nb;
  long st;
  if (DIR == 0) { n = d.ni; na = d.nj; nb = d.nk; st = 1; }
  else if (DIR == 1) { n = d.nj; na = d.ni; nb = d.nk; st = d.sy; }
  else { n = d.nk; na = d.ni; nb = d.nj; st = d.sz; }
  if (t >= na * nb) return;
  const int a = 2 + t % na, b = 2 + t / na;
  long q;
  if (DIR == 0) q = ix(d, 2, a, b);
  else if (DIR == 1) q = ix(d, a, 2, b);
  else q = ix(d, a, b, 2);
  const long E = d.E;
  T v = T(0), u[5] = {T(0), T(0), T(0), T(0), T(0)};
  for (int r = 1; r <= n; r++, q += st) {
    const T e = A.eps[q];
    const T aa = T(1) + T(2) * e;
    const T bb = r == n ? T(0) : -e;
    const T cc = r == 1 ? T(0) : -e;
    const T z = T(1) / (aa + cc * v);
    v = -bb * z;
    A.vb[q] = v;
#pragma unroll
    for (int m = 0; m < 5; m++) {
      u[m] = (-cc * u[m] + A.dw[m * E + q]) * z;
      A.dw[m * E + q] = u[m];
    }
  }
  q -= st;  // last cell: x_n = u_{n+1}, already in place
  for (int r = n - 1; r >= 1; r--) {
    const T vn = A.vb[q - st];
#pragma unroll
    for (int m = 0; m < 5; m++) {
      u[m] = vn * u[m] + A.dw[m * E + q - st];
      A.dw[m * E + q - st] = u[m];
    }
    q -= st;
  }
}
template <typename T>
__device__ __attribute__((always_inline)) inline void k_psmoo_x_body(const PsmooArgs<T> &A, int bx, int by, int bz) {
  k_psmoo_line_body<0, T>(A, bx, by, bz);
}
template <typename T>
__device__ __attribute__((always_inline)) inline void k_psmoo_y_body(const PsmooArgs<T> &A, int bx, int by, int bz) {
  k_psmoo_line_body<1, T>(A, bx, by, bz);
}
template <typename T>
__device__ __attribute__((always_inline)) inline void k_psmoo_z_body(const PsmooArgs<T> &A, int bx, int by, int bz) {
  k_psmoo_line_body<2, T>(A, bx, by, bz);
}
MGE_ENTRY_T(k_psmoo_x, PsmooArgs, 64, 1)
MGE_ENTRY_T(k_psmoo_y, PsmooArgs, 64, 1)
MGE_ENTRY_T(k_psmoo_z, PsmooArgs, 64, 1)

}  // namespace mge

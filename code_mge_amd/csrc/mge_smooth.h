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
  const T *e1, *e2;  // pivots of this direction (psmoo.f90:134-166)
  const T *r1;       // 1/e1, rounded once from the FP64 pivots
  T bb;
};

// The forward step's division by the pivot e1_s.  FP64 multiplies by the
// reciprocal pivot instead (one rounding more per cell, a few ulp over a
// line, and no FP64 division on the recurrence's critical path); FP32
// divides, as the reference does.
template <typename T>
__device__ __attribute__((always_inline)) inline T piv_div(T x, const T *__restrict__ e1,
                                                           const T *__restrict__ r1, int s) {
  if constexpr (kDelta<T>) return x / e1[s];
  else return x * r1[s];
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
  if (S.flags[b0 + 2] & F_FLUID) D[b0 + 2] = piv_div(D[b0 + 2], S.e1, S.r1, 2);
  for (int i = 3; i <= d.il; i++)
    if (S.flags[b0 + i] & F_FLUID) D[b0 + i] = piv_div(D[b0 + i] - S.bb * D[b0 + i - 1], S.e1, S.r1, i);
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
                                                                 long b0, long st, int nl, const T *__restrict__ e1,
                                                                 const T *__restrict__ r1, const T *__restrict__ e2,
                                                                 T bb) {
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
    y = MK[t] * piv_div(BUF[t] - bb * y, e1, r1, s_);                 \
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
    y = m_ * piv_div(D[q_] - bb * y, e1, r1, s_);
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
  line_sweep<8>(S.dw + n * d.E, S.flags, ix(d, i, 0, k), d.sy, d.jl, S.e1, S.r1, S.e2, S.bb);
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
  line_sweep<8>(S.dw + n * d.E, S.flags, ix(d, i, j, 0), d.sz, d.kl, S.e1, S.r1, S.e2, S.bb);
}
MGE_ENTRY_T_XCD(k_smooth_z, SmoothArgs, 64, 1)

// ---- lines in segments ---------------------------------------------------
//
// A line split into segments of L cells, one thread each, all of its cells in
// registers and the segments joined through LDS.  Both
// recurrences are evaluated within the segment from zero, giving the
// segment's map from the value entering it to the value leaving it; every
// thread then runs through the maps before (backward: after) it and
// re-evaluates its cells with the reference formula from the value entering.
// Branch-free: a cell's fluid bit selects its pivots or zeros (blank cells
// hold dw = +-0, see line_sweep, and come out as 0), and the places past the
// line's end count as blank; a branch per cell would wait for every LDS read
// by itself (64^3 in k_smooth_xy: 25 us with branches, 13 without).
// Called by all threads of the workgroup (barriers); sa, sb, sc, sd: LDS of
// G x nline values each; `act` threads hold segment g of line `line`.
template <typename T>
struct SegPiv {   // a line's pivots, in LDS, indexed by cell from 0
  const T *e1, *r1, *e2;
};
// x / e1 on a fluid cell, 0 on a blank one (rm: r1 or 0).  FP64 multiplies by
// the reciprocal pivot; FP32 corrects the product by its remainder, which
// gives the quotient the reference's division gives
template <typename T>
__device__ inline T seg_div(T x, T e1, T rm) {
  const T q = x * rm;
  if constexpr (kDelta<T>) return __builtin_fmaf(__builtin_fmaf(-e1, q, x), rm, q);
  else return q;
}
template <int L, typename T>
__device__ __attribute__((always_inline)) inline void seg_solve(bool act, T (&r)[L], unsigned fl, int s0, int g, int G,
                                                                int line, int nline, const SegPiv<T> &P, T bb, T *sa,
                                                                T *sb, T *sc, T *sd) {
  auto rm = [&](int c) { return (fl >> c) & 1u ? P.r1[s0 + c] : T(0); };
  auto e1 = [&](int c) { if constexpr (kDelta<T>) return P.e1[s0 + c]; else return T(0); };
  auto qm = [&](int c) { return (fl >> c) & 1u ? P.e2[s0 + c] : T(0); };
  T A = T(1), B = T(0);
#pragma unroll
  for (int c = 0; c < L; c++) {
    const T m = rm(c);
    B = seg_div(r[c] - bb * B, e1(c), m);
    A = A * (-bb * m);
  }
  if (act) {
    sa[g * nline + line] = A;
    sb[g * nline + line] = B;
  }
  __syncthreads();
  T y = T(0);
  for (int q = 0; q < G - 1; q++) {   // uniform; the maps before this segment
    const T ny = sa[q * nline + line] * y + sb[q * nline + line];
    y = q < g ? ny : y;
  }
  T C = T(1), D = T(0);
#pragma unroll
  for (int c = 0; c < L; c++) {
    y = seg_div(r[c] - bb * y, e1(c), rm(c));
    r[c] = y;
  }
  // backward: z = y - e2 z', e2 = 0 on the line's last cell
#pragma unroll
  for (int c = L - 1; c >= 0; c--) {
    const T m = qm(c);
    D = r[c] - m * D;
    C = -(m * C);
  }
  if (act) {
    sc[g * nline + line] = C;
    sd[g * nline + line] = D;
  }
  __syncthreads();
  T z = T(0);
  for (int q = G - 1; q > 0; q--) {
    const T nz = sc[q * nline + line] * z + sd[q * nline + line];
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
  const T *e1x, *e2x, *r1x, *e1y, *e2y, *r1y;
  T bb;
};
// plane classes: cells of LDS (rows of nx | 1), mask words, pivots per
// direction, threads, segment length.  Planes of more than 64 x 65 cells leave
// too few workgroups a CU: 128 x 128 x 4 took 21 us in one launch, 11 in two.
struct XYClass {
  int cells, words, piv, threads, seg;
};
constexpr XYClass kXY[2] = {{2560, 128, 264, 512, 8}, {4416, 256, 264, 512, 8}};
// the class that holds an nx x ny plane (-1: none)
inline int xy_class(int nx, int ny) {
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
  constexpr int L = K.seg, NP = kDelta<T> ? 3 : 2;
  __shared__ T pl[K.cells];
  __shared__ T pv[2][NP][K.piv];   // x, y: 1/e1, e2 (and e1 in FP32)
  __shared__ unsigned long long mk[K.words];
  const Dims &d = S.d;
  const int nx = d.ni, ny = d.nj, P = nx | 1, nch = (nx + 63) >> 6;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  for (int t = tid; t < K.piv; t += K.threads) {
    const int ix2 = 2 + min(t, nx - 1), iy2 = 2 + min(t, ny - 1);
    pv[0][0][t] = S.r1x[ix2];
    pv[0][1][t] = S.e2x[ix2];
    pv[1][0][t] = S.r1y[iy2];
    pv[1][1][t] = S.e2y[iy2];
    if constexpr (kDelta<T>) {
      pv[0][NP - 1][t] = S.e1x[ix2];
      pv[1][NP - 1][t] = S.e1y[iy2];
    }
  }
  // rows by groups of lp lanes (a power of two), RW rows a wave
  const int lp = nx > 32 ? 64 : (nx > 16 ? 32 : (nx > 8 ? 16 : 8));
  const int sub = lane / lp, l = lane & (lp - 1), RW = 64 / lp;
  const long base = ix(d, 2, 2, 2 + bx);
  T *D = S.dw + by * d.E + base;
  const uint8_t *F = S.flags + base;
  constexpr int NW = K.threads / 64, U = 8;
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
  {  // x lines
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
    seg_solve<L>(act, r, fl, i0, g, G, line, ny, SegPiv<T>{pv[0][NP - 1], pv[0][0], pv[0][1]}, S.bb, pl, pl + n,
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
    seg_solve<L>(act, r, fl, j0, g, G, line, nx, SegPiv<T>{pv[1][NP - 1], pv[1][0], pv[1][1]}, S.bb, pl, pl + n,
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
// this, y lines: 256^3 FP64 421 -> 296 us (4.6 TB/s), FP32 243 -> 183 us;
// 128^3 46 -> 32 us; 512 x 512 x 4 105 -> 26 us.
struct SegShape {
  int sx, len;   // lines side by side, cells per segment (0: too long)
};
inline SegShape seg_shape(int n) {
  if (n <= 16) return SegShape{64, n <= 4 ? 4 : (n <= 8 ? 8 : 16)};
  if (n <= 256) return SegShape{32, n <= 128 ? 8 : 16};
  return n <= 512 ? SegShape{16, 16} : SegShape{0, 0};
}
template <typename T, int SX, int L, int DIR>
__device__ __attribute__((always_inline)) inline void k_smooth_seg_body(const SmoothArgs<T> &S, int bx, int by,
                                                                        int bz) {
  constexpr int NP = kDelta<T> ? 3 : 2, GM = SX == 64 ? 1 : 512 / SX;
  __shared__ T sh[4][GM * SX], pv[NP][L * GM];
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
    pv[0][t] = S.r1[s];
    pv[1][t] = S.e2[s];
    if constexpr (kDelta<T>) pv[NP - 1][t] = S.e1[s];
  }
  __syncthreads();
  seg_solve<L>(act, r, fl, s0, g, G, line, SX, SegPiv<T>{pv[NP - 1], pv[0], pv[1]}, S.bb, sh[0], sh[1], sh[2], sh[3]);
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

// x lines in segments of 16 cells, where the planes do not fit k_smooth_xy:
// a workgroup stages 16 (N = 128: 32) rows of up to N cells in LDS (whole rows,
// so loads and stores are coalesced), each thread takes a segment.  With lines
// scanned across a wave's lanes by shuffles -> this: 256^3 FP64 399 -> 286 us
// (4.7 TB/s), FP32 291 -> 201 us; 128^3 54 -> 48 us; 96^3 33 -> 24 us.
template <int N>
constexpr int xseg_rows() { return N == 128 ? 32 : 16; }
template <typename T, int N>
__device__ __attribute__((always_inline)) inline void k_smooth_xseg_body(const SmoothArgs<T> &S, int bx, int by) {
  constexpr int NP = kDelta<T> ? 3 : 2, L = 16, kXR = xseg_rows<N>(), NT = kXR * N / L, NW = NT / 64;
  __shared__ T pl[kXR * (N + 1)], pv[NP][N];
  __shared__ unsigned long long mk[kXR * N / 64];
  const Dims &d = S.d;
  const int nx = d.ni, P = nx | 1, nch = (nx + 63) >> 6, G = (nx + L - 1) / L;
  const int nl = d.nj * d.nk, l0 = bx * kXR, rows = min(kXR, nl - l0);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  T *D = S.dw + by * d.E;
  auto at = [&](int row) {   // the first cell of the workgroup's row
    const int l = l0 + min(row, rows - 1), k = l / d.nj;
    return ix(d, 2, 2 + l - k * d.nj, 2 + k);
  };
  for (int t = tid; t < G * L; t += NT) {
    const int s = 2 + min(t, nx - 1);
    pv[0][t] = S.r1[s];
    pv[1][t] = S.e2[s];
    if constexpr (kDelta<T>) pv[NP - 1][t] = S.e1[s];
  }
  constexpr int RW = kXR / NW;                      // rows of a wave
  constexpr int U = N / 64;                         // chunks of a row
#pragma unroll 2
  for (int u = 0; u < RW; u++) {
    const int row = wave * RW + u;
    const long q = at(row);
    T v[U];
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
  T r[L];
#pragma unroll
  for (int c = 0; c < L; c++) r[c] = pl[line * P + min(i0 + c, nx - 1)];
  __syncthreads();
  const int n = G * kXR;
  seg_solve<L>(act, r, fl, i0, g, G, line, kXR, SegPiv<T>{pv[NP - 1], pv[0], pv[1]}, S.bb, pl, pl + n, pl + 2 * n,
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
      if (i < nx) D[q + i] = pl[row * P + i];   // blank cells: as they were read
    }
  }
}
template <typename T, int N>
__global__ void __launch_bounds__(xseg_rows<N>() * N / 16) k_smooth_xseg(SmoothArgs<T> S) {
  int bx, by, bz;
  xcd_block(bx, by, bz);
  k_smooth_xseg_body<T, N>(S, bx, by);
}
template <typename T, int N>
__global__ void __launch_bounds__(xseg_rows<N>() * N / 16)
    k_smooth_xseg_b(const SmoothArgs<T> *As, const int4 *cg, int nc, const int *act) {
  const int b = (int)blockIdx.x;
  const int c = batch_case(cg, nc, b);
  const int4 g = cg[c];
  if (!act[g.w]) return;
  const int l = b - g.x;
  k_smooth_xseg_body<T, N>(As[c], l % g.y, l / g.y);
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

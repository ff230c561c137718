// mge_visc.h -- laminar viscous fluxes (the role of viscpak's fgradi/j/k
// and vflux, called from euler.f90:137-181 when cdis(m) > 0).
//
// viscpak has no source in the reference tree; the flux is this build's
// own and the CPU restatement evaluates the same expressions:
//  - velocity and temperature per cell (euler.f90:140-150: vel = m/rho,
//    tem = p/(rho R)); the FP32 path keeps their deviations from the
//    freestream so that differences of neighbouring cells keep their digits;
//  - face gradient: normal derivative (phi_a - phi_(a-1))/hn with hn the
//    centre distance; tangential derivatives the mean of the two cells'
//    centred differences, one-sided next to a blank cell, zero between two;
//  - tau = mu (G + G^T) - 2/3 mu div(u) I, q = -kappa dT/dn,
//    kappa = mu gamma R / ((gamma-1) Pr); flux (0, tau_n, u_f . tau_n - q_n)
//    times the face vector S, u_f the mean of the two cells;
//  - no bulk flux through a face with a blank side; the wall records add the
//    flux of the face between each cut cell and its no-slip mirror state
//    (normal derivatives only), in FP64 and in record order;
//  - per cell fw = blend fw + cdis ((gx_hi - gx_lo) + (gy_hi - gy_lo) +
//    (gz_hi - gz_lo)) before the dissipation of the stage is added.
#pragma once
#include "mge_stage.h"

namespace mge {

// a wall record as the flux kernel reads it: records of one tile are
// contiguous, a cell's records contiguous in record order
struct ViscRec {
  int m, cell, dir, hi;  // record, cell of the tile, face direction and side
  int c[3], s[3];        // cut cell and solid cell
};

// The kernel's tile of cells and its threads; its brick of states has one
// cell more on each side.  17 x 4 x 4 i faces, 16 x 5 x 4 j faces and
// 16 x 4 x 5 k faces each fit one round of 320 threads, and the brick
// without its 8 corners, which no stencil reads, is two loads per thread.
constexpr int kVX = 16, kVY = 4, kVZ = 4, kVNT = 320;
constexpr int kVSY = kVX + 2, kVSZ = kVSY * (kVY + 2), kVBrick = kVSZ * (kVZ + 2);
constexpr int kVEnd = kVSZ - 4, kVMid = kVZ * kVSZ;  // cells of an end layer without corners, of the middle layers
static_assert(2 * kVEnd + kVMid == 2 * kVNT, "two brick cells per thread");
static_assert(kVX * (kVY + 1) * kVZ == kVNT && kVX * kVY * (kVZ + 1) == kVNT && (kVX + 1) * kVY * kVZ <= kVNT,
              "one face per thread and direction");

template <typename T>
struct ViscArgs {
  Dims d;
  StateC<T> s;
  const uint8_t *flags;
  Geo<T> g;
  T *fw;
  Inf<T> inf;
  T uinf[3];     // freestream velocity (FP32 work term)
  T tinf;        // freestream temperature
  T rgas, mu, kap, cdis, blend;
  int m;         // stage; fw is blended in only for m > 1
  const int *vtile;      // wall records of tile t: vrec[vtile[t] .. vtile[t + 1]); null: none on this level
  const ViscRec *vrec;
  const double *wsol, *psol;  // mirror states by record
  int nmir;
};

// euler.f90:140-150: velocity and temperature of a cell (FP32: deviations
// from the freestream), zero on a blank one
template <typename T>
__device__ inline void visc_prim(const ViscArgs<T> &A, bool fluid, const T *w, T p, T *o) {
  if constexpr (kDelta<T>) {
    const T rho = A.inf.w[0] + w[0];
#pragma unroll
    for (int a = 0; a < 3; a++) o[a] = (w[a + 1] - A.uinf[a] * w[0]) / rho;
    o[3] = (p - (A.tinf * A.rgas) * w[0]) / (rho * A.rgas);
  } else {
#pragma unroll
    for (int a = 0; a < 3; a++) o[a] = w[a + 1] / w[0];
    o[3] = p / (w[0] * A.rgas);
  }
#pragma unroll
  for (int a = 0; a < 4; a++) o[a] = fluid ? o[a] : T(0);
}

// one face: pL/pR velocity + temperature of the two cells (FP32: deviations,
// u0 the freestream velocity), dn their normal derivatives, t1*/t2* the
// tangential velocity derivatives of the two cells; momentum and energy flux
template <int DIR, typename T>
__device__ inline void visc_face(const ViscArgs<T> &A, const T *pL, const T *pR, const T *dn, const T *t1L,
                                 const T *t1R, const T *t2L, const T *t2R, T S, T *g) {
  constexpr int t1 = DIR == 0 ? 1 : 0, t2 = DIR == 2 ? 1 : 2;
  T G[3][3];
#pragma unroll
  for (int a = 0; a < 3; a++) {
    G[a][DIR] = dn[a];
    G[a][t1] = T(0.5) * (t1L[a] + t1R[a]);
    G[a][t2] = T(0.5) * (t2L[a] + t2R[a]);
  }
  const T div = (G[0][0] + G[1][1]) + G[2][2];
  T tau[3], uf[3];
#pragma unroll
  for (int a = 0; a < 3; a++) tau[a] = A.mu * (G[a][DIR] + G[DIR][a]);
  tau[DIR] = A.mu * (T(2) * G[DIR][DIR] - T(2.0 / 3.0) * div);
#pragma unroll
  for (int a = 0; a < 3; a++)
    uf[a] = kDelta<T> ? A.uinf[a] + T(0.5) * (pL[a] + pR[a]) : T(0.5) * (pL[a] + pR[a]);
  const T qn = -A.kap * dn[3];
  g[0] = tau[0] * S;
  g[1] = tau[1] * S;
  g[2] = tau[2] * S;
  g[3] = (((uf[0] * tau[0] + uf[1] * tau[1]) + uf[2] * tau[2]) - qn) * S;
}

// an axis' widths over the tile: h, the centre distance to the lower cell
// (hm) and between the two neighbours (hc), and their reciprocals
template <typename T, int N>
struct ViscAxis {
  T h[N + 1], hm[N + 1], rm[N + 1], hc[N + 1], rc[N + 1];
};
template <typename T, int N>
__device__ inline void visc_axis(ViscAxis<T, N> &X, const T *h, int base, int last, int e) {
  const int c = base + e < last ? base + e : last;  // last: the high ghost layer
  const T h0 = h[c - 1], h1 = h[c], h2 = h[c + 1 <= last ? c + 1 : last];
  const T hm = T(0.5) * (h0 + h1), hc = hm + T(0.5) * (h1 + h2);
  X.h[e] = h1;
  X.hm[e] = hm;
  X.rm[e] = T(1) / hm;
  X.hc[e] = hc;
  X.rc[e] = T(1) / hc;
}

template <typename T>
struct ViscLds {
  T pr[4][kVBrick];
  double buf[4 * kVNT];  // a direction's fluxes (T), or the wall records' fluxes
  ViscAxis<T, kVX> x;
  ViscAxis<T, kVY> y;
  ViscAxis<T, kVZ> z;
  short start[kVX * kVY * kVZ], cell[kVNT];
  uint8_t fl[kVBrick];
};

// centred velocity difference of brick cell o along an axis with stride st,
// one-sided next to a blank cell and zero between two; c the cell's index on
// the tile's axis
template <int N, typename T>
__device__ inline void visc_dt(const ViscLds<T> &L, const ViscAxis<T, N> &X, int o, int st, int c, T *out) {
  const bool fp = L.fl[o + st] != 0, fm = L.fl[o - st] != 0;
  const int oh = fp ? o + st : o, ol = fm ? o - st : o;
  const T h1 = fp ? X.hm[c + 1] : X.hm[c], r1 = fp ? X.rm[c + 1] : X.rm[c];
  const T h = fp && fm ? X.hc[c] : h1, r = fp && fm ? X.rc[c] : r1;
#pragma unroll
  for (int a = 0; a < 3; a++) out[a] = quot(L.pr[a][oh] - L.pr[a][ol], h, r);
}

// thread t's face of direction DIR: its flux into the buffer
template <int DIR, typename T>
__device__ inline void visc_bulk_face(const ViscArgs<T> &A, const ViscLds<T> &L, int t, T *buf) {
  constexpr int NX = kVX + (DIR == 0), NY = kVY + (DIR == 1);
  const int x = t % NX, y = (t / NX) % NY, z = t / (NX * NY);
  if (DIR == 0 && z >= kVZ) return;
  constexpr int sd = DIR == 0 ? 1 : (DIR == 1 ? kVSY : kVSZ);
  const int oR = (z + 1) * kVSZ + (y + 1) * kVSY + x + 1, oL = oR - sd;
  T g[4] = {T(0), T(0), T(0), T(0)};
  if (L.fl[oR] && L.fl[oL]) {
    T pL[4], pR[4], dn[4], t1L[3], t1R[3], t2L[3], t2R[3];
    const T hn = DIR == 0 ? L.x.hm[x] : (DIR == 1 ? L.y.hm[y] : L.z.hm[z]);
    const T rn = DIR == 0 ? L.x.rm[x] : (DIR == 1 ? L.y.rm[y] : L.z.rm[z]);
#pragma unroll
    for (int a = 0; a < 4; a++) {
      pL[a] = L.pr[a][oL];
      pR[a] = L.pr[a][oR];
      dn[a] = quot(pR[a] - pL[a], hn, rn);
    }
    if constexpr (DIR == 0) {
      visc_dt(L, L.y, oL, kVSY, y, t1L);
      visc_dt(L, L.y, oR, kVSY, y, t1R);
    } else {
      visc_dt(L, L.x, oL, 1, x, t1L);
      visc_dt(L, L.x, oR, 1, x, t1R);
    }
    if constexpr (DIR == 2) {
      visc_dt(L, L.y, oL, kVSY, y, t2L);
      visc_dt(L, L.y, oR, kVSY, y, t2R);
    } else {
      visc_dt(L, L.z, oL, kVSZ, z, t2L);
      visc_dt(L, L.z, oR, kVSZ, z, t2R);
    }
    const T S = DIR == 0 ? -(L.y.h[y] * L.z.h[z]) : (DIR == 1 ? -(L.x.h[x] * L.z.h[z]) : -(L.x.h[x] * L.y.h[y]));
    visc_face<DIR>(A, pL, pR, dn, t1L, t1R, t2L, t2R, S, g);
  }
#pragma unroll
  for (int n = 0; n < 4; n++) buf[n * kVNT + t] = g[n];
}

template <int DIR, typename T>
__device__ inline void visc_dir(const ViscArgs<T> &A, ViscLds<T> &L, int t, int x, int y, int z, T *acc) {
  T *buf = reinterpret_cast<T *>(L.buf);
  visc_bulk_face<DIR>(A, L, t, buf);
  __syncthreads();
  constexpr int NX = kVX + (DIR == 0), NY = kVY + (DIR == 1);
  constexpr int st = DIR == 0 ? 1 : (DIR == 1 ? NX : NX * NY);
  const int lo = (z * NY + y) * NX + x;
  if (t < kVX * kVY * kVZ) {
#pragma unroll
    for (int n = 0; n < 4; n++) acc[n] = acc[n] + (buf[n * kVNT + lo + st] - buf[n * kVNT + lo]);
  }
  __syncthreads();
}

// the wall-face viscous flux between cut cell c and mirror state ws, ps
// (FP64; normal derivatives only)
template <typename T>
__device__ inline void visc_wall_flux(const ViscArgs<T> &A, int dir, bool hi, const int *c, const int *s,
                                      const double *ws, double ps, double *g) {
  const Dims &d = A.d;
  const long E = d.E;
  const long qc = ix(d, c[0], c[1], c[2]);
  const double rc = full(A.inf, 0, A.s.w[qc]);
  double pc[4], pg[4], h[3];
  for (int a = 0; a < 3; a++) pc[a] = full(A.inf, a + 1, A.s.w[(a + 1) * E + qc]) / rc;
  pc[3] = full(A.inf, 5, A.s.p[qc]) / (rc * (double)A.rgas);
  const int up = hi ? 1 : 0;
  h[0] = (double)A.g.dx[c[0] - 1 + up] + (double)A.g.dx[c[0] + up];
  h[1] = (double)A.g.dy[c[1] - 1 + up] + (double)A.g.dy[c[1] + up];
  h[2] = (double)A.g.dz[c[2] - 1 + up] + (double)A.g.dz[c[2] + up];
  const double hn = 0.5 * (dir == 0 ? h[0] : (dir == 1 ? h[1] : h[2]));
  const double S = face_s_any(A.g, dir + 1, hi ? s[0] : c[0], hi ? s[1] : c[1], hi ? s[2] : c[2]);
  for (int a = 0; a < 3; a++) pg[a] = ws[a + 1] / ws[0];
  pg[3] = ps / (ws[0] * (double)A.rgas);
  double dn[4], tau[3], uf[3];
  for (int a = 0; a < 4; a++) dn[a] = (hi ? pg[a] - pc[a] : pc[a] - pg[a]) / hn;
  const double mu = (double)A.mu, kap = (double)A.kap;
  for (int a = 0; a < 3; a++) {
    tau[a] = a == dir ? mu * (2.0 * dn[a] - (2.0 / 3.0) * dn[a]) : mu * dn[a];
    uf[a] = 0.5 * (pc[a] + pg[a]);
  }
  const double qn = -kap * dn[3];
  g[0] = tau[0] * S;
  g[1] = tau[1] * S;
  g[2] = tau[2] * S;
  g[3] = (((uf[0] * tau[0] + uf[1] * tau[1]) + uf[2] * tau[2]) - qn) * S;
}

// record e's flux, signed by its side of the cell
template <typename T>
__device__ inline void visc_rec_flux(const ViscArgs<T> &A, const ViscRec &r, double *g) {
  double ws[4];
  for (int n = 0; n < 4; n++) ws[n] = A.wsol[n * (long)A.nmir + r.m];
  visc_wall_flux(A, r.dir, r.hi != 0, r.c, r.s, ws, A.psol[r.m], g);
  for (int n = 0; n < 4; n++) g[n] = r.hi ? g[n] : -g[n];
}

// fw = blend fw + cdis * (viscous balance + wall records), every interior
// cell.  A tile's states are read once into LDS as velocity and temperature;
// each face is formed once by one thread from differences in LDS and summed
// by its two cells; divisions by widths are products with reciprocals formed
// once per tile; the tile's wall records are evaluated by one thread each
// while the states arrive, and their cells add them in record order.
// Bound by FP64 issue and LDS reads (24 per face) on large levels and by one
// chain of load, face and sum on small ones.  Against a launch for the
// velocities, one thread per cell forming its six faces from global memory
// with a division per difference and a launch for the wall records: 512 x 512
// x 4 FP64 205 -> 59 us, 128 x 128 x 4 39 -> 9 us, 48 x 48 x 2 27 -> 8.4 us,
// 96^3 FP32 130 -> 33 us.
template <typename T>
__device__ __attribute__((always_inline)) inline void k_visc_body(const ViscArgs<T> &A, int bx, int by, int bz) {
  __shared__ ViscLds<T> L;
  const Dims &d = A.d;
  const long E = d.E;
  const int t = threadIdx.x;
  const int i0 = 2 + bx * kVX, j0 = 2 + by * kVY, k0 = 2 + bz * kVZ;
  // the brick; cells beyond the high ghost layer repeat it and are not used
  T w[2][5], p[2];
  int pos[2];
  bool fluid[2];
#pragma unroll
  for (int r = 0; r < 2; r++) {
    const int c = t + r * kVNT;
    const int top = c >= kVEnd + kVMid, u = top ? c - (kVEnd + kVMid) : c;
    const int corner = u + 1 + (u >= kVX) + (u >= kVX + kVY * kVSY);
    pos[r] = c >= kVEnd && !top ? c + 4 : (top ? kVSZ + kVMid + corner : corner);
    const int z = pos[r] / kVSZ, y = (pos[r] % kVSZ) / kVSY, x = pos[r] % kVSY;
    const int i = i0 - 1 + x, j = j0 - 1 + y, k = k0 - 1 + z;
    const long q = ix(d, i <= d.il + 1 ? i : d.il + 1, j <= d.jl + 1 ? j : d.jl + 1, k <= d.kl + 1 ? k : d.kl + 1);
    fluid[r] = (A.flags[q] & F_FLUID) != 0;
#pragma unroll
    for (int n = 0; n < 4; n++) w[r][n] = A.s.w[n * E + q];
    p[r] = A.s.p[q];
  }
  const int x = t % kVX, y = (t / kVX) % kVY, z = t / (kVX * kVY);
  const bool in = z < kVZ && i0 + x <= d.il && j0 + y <= d.jl && k0 + z <= d.kl;
  const long q = in ? ix(d, i0 + x, j0 + y, k0 + z) : 0;
  T f[5];
#pragma unroll
  for (int n = 0; n < 5; n++) f[n] = in && A.m > 1 ? A.fw[n * E + q] : T(0);
  int e0 = 0, ne = 0;
  if (A.vtile) {
    const int tile = (bz * ((d.nj + kVY - 1) / kVY) + by) * ((d.ni + kVX - 1) / kVX) + bx;
    e0 = A.vtile[tile];
    ne = A.vtile[tile + 1] - e0;
  }
  if (t <= kVX) visc_axis(L.x, A.g.dx, i0, d.il + 1, t);
  else if (t >= 64 && t <= 64 + kVY) visc_axis(L.y, A.g.dy, j0, d.jl + 1, t - 64);
  else if (t >= 128 && t <= 128 + kVZ) visc_axis(L.z, A.g.dz, k0, d.kl + 1, t - 128);
  if (t < kVX * kVY * kVZ) L.start[t] = -1;
#pragma unroll
  for (int r = 0; r < 2; r++) {
    T o[4];
    visc_prim(A, fluid[r], w[r], p[r], o);
#pragma unroll
    for (int a = 0; a < 4; a++) L.pr[a][pos[r]] = o[a];
    L.fl[pos[r]] = fluid[r];
  }
  double wg[4] = {0.0, 0.0, 0.0, 0.0};
  if (t < ne) visc_rec_flux(A, A.vrec[e0 + t], wg);
  __syncthreads();
  T acc[4] = {T(0), T(0), T(0), T(0)};
  visc_dir<0>(A, L, t, x, y, z, acc);
  visc_dir<1>(A, L, t, x, y, z, acc);
  visc_dir<2>(A, L, t, x, y, z, acc);
  if (A.m > 1) {
#pragma unroll
    for (int n = 0; n < 5; n++) f[n] = f[n] * A.blend;
  }
#pragma unroll
  for (int n = 0; n < 4; n++) f[n + 1] = f[n + 1] + A.cdis * acc[n];
  if (ne > 0) {  // one value per block
    double fd[4];
    for (int n = 0; n < 4; n++) fd[n] = (double)f[n + 1];
    for (int b = 0; b < ne; b += kVNT) {
      const int nb = ne - b < kVNT ? ne - b : kVNT;
      if (b > 0) {
        if (t < kVX * kVY * kVZ) L.start[t] = -1;
        if (t < nb) visc_rec_flux(A, A.vrec[e0 + b + t], wg);
        __syncthreads();
      }
      if (t < nb) {
        const int c = A.vrec[e0 + b + t].cell;
        if (t == 0 || A.vrec[e0 + b + t - 1].cell != c) L.start[c] = (short)t;
        L.cell[t] = (short)c;
        for (int n = 0; n < 4; n++) L.buf[n * kVNT + t] = wg[n];
      }
      __syncthreads();
      if (t < kVX * kVY * kVZ && L.start[t] >= 0) {
        for (int o = L.start[t]; o < nb && L.cell[o] == t; o++)
          for (int n = 0; n < 4; n++) fd[n] = fd[n] + (double)A.cdis * L.buf[n * kVNT + o];
      }
      __syncthreads();
    }
    for (int n = 0; n < 4; n++) f[n + 1] = (T)fd[n];
  }
  if (in) {
#pragma unroll
    for (int n = 0; n < 5; n++) A.fw[n * E + q] = f[n];
  }
}
MGE_ENTRY_T_XCD(k_visc, ViscArgs, kVNT, 1)

// wall force: adds each record's viscous part (minus the viscous momentum
// flux leaving the fluid through its wall face) to the record's term
template <typename T>
__global__ void k_wall_visc_terms(ViscArgs<T> A, const DevRec *recs, const double *wsol, const double *psol,
                                  int nmir, double *terms) {
  const int m = blockIdx.x * blockDim.x + threadIdx.x;
  if (m >= nmir) return;
  const DevRec &r = recs[m];
  const bool hi = r.faceid >= 4;
  double ws[4], g[4];
  for (int n = 0; n < 4; n++) ws[n] = wsol[n * nmir + m];
  visc_wall_flux(A, r.zz - 1, hi, r.c, r.s, ws, psol[m], g);
  for (int dd = 0; dd < 3; dd++) terms[3 * m + dd] = terms[3 * m + dd] + (hi ? g[dd] : -g[dd]);
}

}  // namespace mge

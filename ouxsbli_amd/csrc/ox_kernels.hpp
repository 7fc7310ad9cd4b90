// ox_kernels.hpp -- gfx950 kernels of one RK stage (templated; instantiated
// by ox_fp64.hip / ox_fp32.hip).
//
// Data layout in HBM (all on one GPU, ghosts included):
//   state  QJ(nx,5,ny,nz) FP64, the reference layout (x fastest, then the
//          variable, then y, z): drop-in for set_state/get_state/checkpoints.
//   prims  rho,u,v,w,p,sensor as separate (nx,ny,nz) arrays of type S
//          (FP64 plain form, FP32 in the FP32-bulk form); T and mu are
//          formed from rho and p where a sweep reads a cell.
//   Racc   residual accumulator in the state layout, type S.
//
// One stage = k_sweep_x (runs of faces in LDS rows; Ducros sensor; writes
// R = c_x*dE; on periodic rows of 64, 128 or 256 cells k_sweep_xrow, whole rows
// in LDS) -> k_sweep_line<DIR=1>
// (register sliding window along y; R += c_y*dF) -> k_sweep_line<DIR=2>
// (sliding window along z; R += c_z*dG, then the RK combination, and the
// primitives of the new state for the next stage).  k_prim (QJ -> primitives)
// runs only after the state is uploaded, k_ghost_fill at the end of a call.  Face fluxes (convective minus viscous) live only in
// registers: E, F and G are never written to memory.  The summation order
// x, then y, then z is the order of calc_R (3D_solver/src/calc_steps.f90:8-38).
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>

#include "ox_physics.hpp"
#include "ox_types.hpp"
#include "ox_xcd.hpp"

namespace ox {

template <class S> struct Prim {
  S *rho, *u, *v, *w, *p, *s, *mut, *qc2;
};
constexpr int kPrimArrays = 8;

// The pointer seen as one into global memory.  Pointers a kernel receives as
// arguments are known global; those the batched kernels read from their
// descriptor arrays are not, and accesses through them would compile to flat
// loads and stores (addresses in VGPRs only, and counted on the LDS wait
// counter as well).  Every access to primitives, residual and state goes
// through G.
template <class T> __device__ __forceinline__ __attribute__((address_space(1))) T* G(T* p) {
  return (__attribute__((address_space(1))) T*)p;
}

constexpr int KEEP = OX_SCHEME_KEEP;
constexpr int SLAU = OX_SCHEME_SLAU;
constexpr int ROE = OX_SCHEME_ROE;
constexpr int HYBRID = OX_SCHEME_HYBRID;
// schemes that read the Ducros sensor (calc_flux_base.f90.fypp:56-58)
// (MUSCL reads it at ORDER 4/6; the hybrid switch at every order)
template <int SCHEME, int ORDER> constexpr bool kUsesSensor = SCHEME == HYBRID || (SCHEME != KEEP && ORDER > 2);
// schemes whose face flux reads T (KEEP's internal-energy term)
template <int SCHEME> constexpr bool kUsesT = SCHEME == KEEP || SCHEME == HYBRID;

// Viscous stencil codes VO: 4 and 6 are the central stencils of that order
// (calc_visc_cent.f90.fypp); 5 is ME4Base (calc_visc_me4_base.f90): a 6-cell
// face window with 4th-order cross derivatives.
template <int VO> constexpr int vwin() { return VO == 5 ? 6 : VO; }    // face window (cells)
template <int VO> constexpr int vcross() { return VO == 5 ? 4 : VO; }  // cross-derivative order

// Stencil width of a face: the convective stencil (ORDER cells) and the
// viscous one (vwin cells) are both centred on the face.
template <int ORDER, int VISC, int VO> struct Sten {
  static constexpr int SW = (VISC && vwin<VO>() > ORDER) ? vwin<VO>() : ORDER;
  static constexpr int HW = SW / 2;
  static constexpr int CO = HW - ORDER / 2;  // first convective cell in the window
  static constexpr int VOFF = VISC ? HW - vwin<VO>() / 2 : 0;
  static constexpr int VH = vcross<VO>() / 2;  // half width of the cross-derivative stencil
};

// state index of (i,l,j,k), 0-based: 64-bit, since the state holds five
// values per cell and a grid of up to 2^31 cells fits one GPU's HBM (the
// bracket, 5 * (j + ny * k) + l, stays below 5 * ny * nz)
__device__ __forceinline__ long long qidx(const Geom& g, int i, int l, int j, int k) {
  return i + (long long)g.nx * (l + 5 * (j + g.ny * k));
}
__device__ __forceinline__ int cidx(const Geom& g, int i, int j, int k) { return i + g.nx * (j + g.ny * k); }

// ---------------------------------------------------------------------------
// Primitive recovery.  calc_quantities_T_3D / calc_quantities_3D
// (src/calc_physical_quantities.f90:60-116), always in FP64.
// ---------------------------------------------------------------------------
// Primitives of one cell from its conserved values (J * Q = physical).
struct PrimVals {
  double rho, u, v, w, p;
};
__device__ __forceinline__ PrimVals prim_of(double q1, double q2, double q3, double q4, double q5, double J,
                                            const PhysC<double>& c) {
  PrimVals r;
  const double over_Q1 = 1.0 / q1;
  r.rho = J * q1;
  r.u = q2 * over_Q1;
  r.v = q3 * over_Q1;
  r.w = q4 * over_Q1;
  r.p = c.gamma_1 * (J * q5 - 0.5 * r.rho * (r.u * r.u + r.v * r.v + r.w * r.w));
  return r;
}
// T and mu are not stored: the sweeps form them from the stored rho and p
// where they read a cell (finish_cell), with the reference's expressions
// (calc_quantities_T_3D, src/calc_physical_quantities.f90:60-116), the same
// values bit for bit as forming them here in FP64.  That takes two arrays off
// the z sweep's writes and off every sweep's reads, for one division, one
// square root and one more division per window cell.
template <class S>
__device__ __forceinline__ void store_prim(const Prim<S>& P, int m, const PrimVals& r) {
  G(P.rho)[m] = (S)r.rho;
  G(P.u)[m] = (S)r.u;
  G(P.v)[m] = (S)r.v;
  G(P.w)[m] = (S)r.w;
  G(P.p)[m] = (S)r.p;
}

template <class S>
__global__ __launch_bounds__(256) void k_prim(const double* __restrict__ QJ, Prim<S> P, Geom g, PhysC<double> c) {
  const int i = blockIdx.x * 64 + threadIdx.x;
  const int j = blockIdx.y * 4 + threadIdx.y;
  const int k = blockIdx.z;
  if (i >= g.nx || j >= g.ny) return;
  const long long q = qidx(g, i, 0, j, k);
  const int st = g.nx;
  const PrimVals r = prim_of(QJ[q], QJ[q + st], QJ[q + 2 * st], QJ[q + 3 * st], QJ[q + 4 * st], g.jac, c);
  store_prim<S>(P, cidx(g, i, j, k), r);
}

// ---------------------------------------------------------------------------
// Selective mixed-scale SGS viscosity (calc_mut, 3D_solver/src/calc_les.f90:
// 12-125) over the cells the reference computes (Fortran 2..n-1), exponents 1/4
// as sqrt(sqrt(.)), and its ghost cells (set_bc_mut_common,
// 3D_solver/src/set_bc_common.f90:296-335).
//
// A cell reads the test-filtered velocity at itself and its six face neighbours,
// each a seven-point stencil.  A workgroup takes LES_X x LES_Y columns and walks
// les_seg planes: every plane is filtered once, tile and rim, into LDS, and the
// cells of the plane before read the three planes around theirs (four slots, so
// one barrier per plane).  Each thread keeps its column's last planes, and their
// in-plane neighbours, in registers.  That is 1.3 filter evaluations per cell and
// velocity component instead of seven, and 24 loads per cell instead of 168.
// Bound by latency and the vector units.  Each cell filtering its seven points by
// itself, and two launches for the ghost cells, took at 192^3 484 us in FP64 and
// 232 us in FP32; this takes 237 and 148 us (96^3: 70 -> 45 and 37 -> 26 us).
// ---------------------------------------------------------------------------
constexpr int LES_X = 32, LES_Y = 8;
// Planes per workgroup: eight, or four where eight leave less than two
// workgroups per CU (at 64^3, FP64: eight 28 us, four 23 us; at 192^3 246 and 270).
__host__ __device__ inline int les_seg(const Geom& g) {
  const long long n = (long long)((g.nx - 2 + LES_X - 1) / LES_X) * ((g.ny - 2 + LES_Y - 1) / LES_Y) * ((g.nz - 2 + 7) / 8);
  return n < 512 ? 4 : 8;
}
// workgroups along x, y, z over the computed cells
inline void les_tiles(const Geom& g, int& bx, int& by, int& bz) {
  bx = (g.nx - 2 + LES_X - 1) / LES_X;
  by = (g.ny - 2 + LES_Y - 1) / LES_Y;
  bz = (g.nz - 2 + les_seg(g) - 1) / les_seg(g);
}

// The test filter at one point from its centre and its neighbours in the order
// -x, +x, -y, +y, -z, +z.
template <class R>
__device__ __forceinline__ R tfilt(R c0, R xm, R xp, R ym, R yp, R zm, R zp) {
  return c0 + R(0.25) * (xm - R(2) * c0 + xp + ym - R(2) * c0 + yp + zm - R(2) * c0 + zp);
}

template <class R>
__device__ __forceinline__ void grad9(R um, R up, R vm, R vp, R wm, R wp, R dx, R dy, R dz, const R* uy, const R* vy,
                                      const R* wy, const R* uz, const R* vz, const R* wz, R* g) {
  g[0] = R(0.5) * (-um + up) * dx;        // dudx
  g[1] = R(0.5) * (-uy[0] + uy[1]) * dy;  // dudy
  g[2] = R(0.5) * (-uz[0] + uz[1]) * dz;  // dudz
  g[3] = R(0.5) * (-vm + vp) * dx;
  g[4] = R(0.5) * (-vy[0] + vy[1]) * dy;
  g[5] = R(0.5) * (-vz[0] + vz[1]) * dz;
  g[6] = R(0.5) * (-wm + wp) * dx;
  g[7] = R(0.5) * (-wy[0] + wy[1]) * dy;
  g[8] = R(0.5) * (-wz[0] + wz[1]) * dz;
}

// The filtered velocity of LES_Y x LES_X columns and a rim of one, four planes.
template <class R> using LesPlanes = R[4][3][LES_Y + 2][LES_X + 2];

// nu_t and qc2 of cell (i, j, k), 1 <= i <= nx-2, 1 <= j <= ny-2, 1 <= k <= nz-2,
// and of the ghost cells that copy it, from the velocities at the cell and its
// neighbours (centre, -x, +x, -y, +y, -z, +z) and the filtered planes (the cell at
// (px, py), plane k in slot k % 4).
template <class S, class R>
__device__ __forceinline__ void les_mut_cell(const Prim<S>& P, const Geom& g, const PhysC<R>& c, int i, int j,
                                             int k, const R (&raw)[3][7], int px, int py,
                                             const LesPlanes<R>& pl) {
  const int m = cidx(g, i, j, k);
  // cells next to the outermost layer are not filtered
  const bool filt = (i >= 2 && i <= g.nx - 3 && j >= 2 && j <= g.ny - 3 && k >= 2 && k <= g.nz - 3);
  R fil[3][7];
#pragma unroll
  for (int f = 0; f < 3; ++f) {
    const auto& pm = pl[(k - 1) & 3][f];
    const auto& pc = pl[k & 3][f];
    const auto& pp = pl[(k + 1) & 3][f];
    const R ft[7] = {pc[py][px], pc[py][px - 1], pc[py][px + 1], pc[py - 1][px], pc[py + 1][px], pm[py][px], pp[py][px]};
#pragma unroll
    for (int t = 0; t < 7; ++t) fil[f][t] = filt ? ft[t] : raw[f][t];
  }
  const R dx = R(g.inv_dx), dy = R(g.inv_dy), dz = R(g.inv_dz);
  R gr[9], gh[9];
  {
    const R uy[2] = {raw[0][3], raw[0][4]}, vy[2] = {raw[1][3], raw[1][4]}, wy[2] = {raw[2][3], raw[2][4]};
    const R uz[2] = {raw[0][5], raw[0][6]}, vz[2] = {raw[1][5], raw[1][6]}, wz[2] = {raw[2][5], raw[2][6]};
    grad9<R>(raw[0][1], raw[0][2], raw[1][1], raw[1][2], raw[2][1], raw[2][2], dx, dy, dz, uy, vy, wy, uz, vz, wz,
             gr);
  }
  {
    const R uy[2] = {fil[0][3], fil[0][4]}, vy[2] = {fil[1][3], fil[1][4]}, wy[2] = {fil[2][3], fil[2][4]};
    const R uz[2] = {fil[0][5], fil[0][6]}, vz[2] = {fil[1][5], fil[1][6]}, wz[2] = {fil[2][5], fil[2][6]};
    grad9<R>(fil[0][1], fil[0][2], fil[1][1], fil[1][2], fil[2][1], fil[2][2], dx, dy, dz, uy, vy, wy, uz, vz, wz,
             gh);
  }
  const R du = raw[0][0] - fil[0][0], dv = raw[1][0] - fil[1][0], dw = raw[2][0] - fil[2][0];
  const R q2 = R(0.5) * (du * du + dv * dv + dw * dw);
  // SMS (calc_les.f90:30-86)
  const R vor1 = gr[7] - gr[5], vor2_ = gr[2] - gr[6], vor3 = gr[3] - gr[1];
  const R vh1 = gh[7] - gh[5], vh2 = gh[2] - gh[6], vh3 = gh[3] - gh[1];
  const R d1 = vor1 - vh1, d2 = vor2_ - vh2, d3 = vor3 - vh3;
  const R vor2 = vor1 * vor1 + vor2_ * vor2_ + vor3 * vor3;
  const R vorh2 = vh1 * vh1 + vh2 * vh2 + vh3 * vh3;
  const R vdiff2 = d1 * d1 + d2 * d2 + d3 * d3;
  const R svor2 = R(2) * fsqrt(vor2) * fsqrt(vorh2) + vorh2 + vor2 - vdiff2;
  R tan2;
  if (fabs_(svor2) < R(1.0e-30)) tan2 = R(0);
  else tan2 = (R(2) * fsqrt(vorh2) * fsqrt(vor2) - vorh2 - vor2 + vdiff2) / svor2;
  const R rtheta = tan2 / c.tan10deg2;
  const R ftheta = fmin2(R(1), rtheta * rtheta);
  const R S2 = R(2) * (gr[0] * gr[0] + gr[4] * gr[4] + gr[8] * gr[8]) +
               ((gr[3] + gr[1]) * (gr[3] + gr[1]) + (gr[7] + gr[5]) * (gr[7] + gr[5]) +
                (gr[2] + gr[6]) * (gr[2] + gr[6]));
  const R nut = ftheta * R(0.06) * fsqrt(fsqrt(S2)) * fsqrt(fsqrt(q2)) * c.les_delta15;
  const S qv = (S)q2, mv = (S)(R(G(P.rho)[m]) * nut);
  G(P.qc2)[m] = qv;
  G(P.mut)[m] = mv;
  // the outermost layer along each direction copies the cell one layer inside
  // the opposite end: up to seven copies of this cell
  const int ai = i == 1 ? g.nx - 1 : (i == g.nx - 2 ? 0 : -1);
  const int aj = j == 1 ? g.ny - 1 : (j == g.ny - 2 ? 0 : -1);
  const int ak = k == 1 ? g.nz - 1 : (k == g.nz - 2 ? 0 : -1);
  if (ai >= 0 || aj >= 0 || ak >= 0) {
    const int xs[2] = {i, ai}, ys[2] = {j, aj}, zs[2] = {k, ak};
    for (int c3 = 1; c3 < 8; ++c3) {
      const int x = xs[c3 & 1], y = ys[(c3 >> 1) & 1], z = zs[(c3 >> 2) & 1];
      if (x >= 0 && y >= 0 && z >= 0) {
        G(P.qc2)[cidx(g, x, y, z)] = qv;
        G(P.mut)[cidx(g, x, y, z)] = mv;
      }
    }
  }
}

// One workgroup's columns and planes (blocks of 256 threads).
template <class S, class R>
__device__ __forceinline__ void les_mut_tile(const Prim<S>& P, const Geom& g, const PhysC<R>& c, int bx, int by, int bz,
                                             LesPlanes<R>& pl) {
  const int sy = g.nx, sz = g.nx * g.ny;
  const int i0 = 1 + bx * LES_X, j0 = 1 + by * LES_Y, k0 = 1 + bz * les_seg(g);
  const int k1 = min(k0 + les_seg(g), g.nz - 1);  // cells of planes k0 .. k1 - 1
  const int tid = threadIdx.x, tx = tid % LES_X, ty = tid / LES_X;
  const int i = i0 + tx, j = j0 + ty;
  const bool inside = i <= g.nx - 2 && j <= g.ny - 2;
  const S* U[3] = {P.u, P.v, P.w};
  // the rim's points (its corners are not read): the rows below and above the
  // tile, then the columns left and right of it, one per thread
  constexpr int RIM = 2 * LES_X + 2 * LES_Y;
  static_assert(RIM <= 256, "one rim point per thread");
  int rx = 0, ry = 0;
  if (tid < 2 * LES_X) rx = 1 + tid % LES_X, ry = tid < LES_X ? 0 : LES_Y + 1;
  else rx = tid < 2 * LES_X + LES_Y ? 0 : LES_X + 1, ry = 1 + tid % LES_Y;
  const int ri = i0 - 1 + rx, rj = j0 - 1 + ry;
  const bool rim = tid < RIM && ri >= 1 && ri <= g.nx - 2 && rj >= 1 && rj <= g.ny - 2;
  // this thread's column (a corner's where it has none): the velocities of planes
  // kk - 2 .. kk + 1 and the in-plane neighbours of planes kk - 1 .. kk + 1, the
  // last loaded a plane ahead of their use
  const int col = inside ? cidx(g, i, j, 0) : cidx(g, 1, 1, 0), rcol = rim ? cidx(g, ri, rj, 0) : 0;
  R z2[3], z1[3], z0[3], zp[3], n1[3][4], n0[3][4], np[3][4];
  auto neighbours = [&](int m) {
#pragma unroll
    for (int f = 0; f < 3; ++f) {
      np[f][0] = R(G(U[f])[m - 1]);
      np[f][1] = R(G(U[f])[m + 1]);
      np[f][2] = R(G(U[f])[m - sy]);
      np[f][3] = R(G(U[f])[m + sy]);
    }
  };
  neighbours(col + (k0 - 1) * sz);
#pragma unroll
  for (int f = 0; f < 3; ++f) {
    z2[f] = z1[f] = R(0);
    z0[f] = R(G(U[f])[col + max(k0 - 2, 0) * sz]);
    zp[f] = R(G(U[f])[col + (k0 - 1) * sz]);
  }
  for (int kk = k0 - 1; kk <= k1; ++kk) {
#pragma unroll
    for (int f = 0; f < 3; ++f) {
      z2[f] = z1[f];
      z1[f] = z0[f];
      z0[f] = zp[f];
#pragma unroll
      for (int t = 0; t < 4; ++t) n1[f][t] = n0[f][t], n0[f][t] = np[f][t];
    }
    const int next = col + min(kk + 1, g.nz - 1) * sz;
#pragma unroll
    for (int f = 0; f < 3; ++f) zp[f] = R(G(U[f])[next]);
    neighbours(next);
    // filtered plane kk where the filter's stencil exists
    if (kk >= 1 && kk <= g.nz - 2) {
      if (inside) {
#pragma unroll
        for (int f = 0; f < 3; ++f)
          pl[kk & 3][f][ty + 1][tx + 1] = tfilt<R>(z0[f], n0[f][0], n0[f][1], n0[f][2], n0[f][3], z1[f], zp[f]);
      }
      if (rim) {
        const int m = rcol + kk * sz;
#pragma unroll
        for (int f = 0; f < 3; ++f)
          pl[kk & 3][f][ry][rx] =
              tfilt<R>(R(G(U[f])[m]), R(G(U[f])[m - 1]), R(G(U[f])[m + 1]), R(G(U[f])[m - sy]), R(G(U[f])[m + sy]),
                       R(G(U[f])[m - sz]), R(G(U[f])[m + sz]));
      }
    }
    __syncthreads();
    if (kk > k0 && inside) {
      R raw[3][7];
#pragma unroll
      for (int f = 0; f < 3; ++f) {
        raw[f][0] = z1[f];
        raw[f][1] = n1[f][0]; raw[f][2] = n1[f][1]; raw[f][3] = n1[f][2]; raw[f][4] = n1[f][3];
        raw[f][5] = z2[f]; raw[f][6] = z0[f];
      }
      les_mut_cell<S, R>(P, g, c, i, j, kk - 1, raw, tx + 1, ty + 1, pl);
    }
  }
}

template <class S, class R>
__global__ __launch_bounds__(256) void k_les_mut(Prim<S> P, Geom g, PhysC<R> c, int nbx, int nby) {
  __shared__ LesPlanes<R> pl;
  const int t = xcd_tile(blockIdx.x, gridDim.x);
  les_mut_tile<S, R>(P, g, c, t % nbx, (t / nbx) % nby, t / (nbx * nby), pl);
}

// ---------------------------------------------------------------------------
// One cell's worth of window data.
// ---------------------------------------------------------------------------
template <class R, int DIR, int ORDER, int SCHEME, int VISC, int VO> struct CellData {
  R rho, u, v, w, p, T, mu, s, d1, d2, d3, d4, mt, H;  // mt, H: LES only
};

// The values one window cell is built from, as they sit in memory: its
// primitives and, for viscous runs, the transverse stencil values of the four
// cross derivatives a face in direction DIR needs (centre excluded).  Kept
// separate from CellData so that a sweep can issue the loads of the next cell
// one face ahead of their use.
template <class S, int VISC, int VO> struct RawCell {
  static constexpr int NX = VISC ? vcross<VO>() : 1;
  S rho, u, v, w, p, s, mt, qc2;
  S x[4][NX];
};

// The four cross derivatives by face direction:
//   DIR 0: uy, vy, uz, wz   DIR 1: ux, vx, vz, wz   DIR 2: ux, wx, vy, wy
template <class S, int DIR>
__device__ __forceinline__ void cross_fields(const Prim<S>& P, const Geom& g, const S* (&f)[4], int (&st)[4]) {
  const int sx = 1, sy = g.nx, sz = g.nx * g.ny;
  if constexpr (DIR == 0) {
    f[0] = P.u; st[0] = sy; f[1] = P.v; st[1] = sy; f[2] = P.u; st[2] = sz; f[3] = P.w; st[3] = sz;
  } else if constexpr (DIR == 1) {
    f[0] = P.u; st[0] = sx; f[1] = P.v; st[1] = sx; f[2] = P.v; st[2] = sz; f[3] = P.w; st[3] = sz;
  } else {
    f[0] = P.u; st[0] = sx; f[1] = P.w; st[1] = sx; f[2] = P.v; st[2] = sy; f[3] = P.w; st[3] = sy;
  }
}

// A cell by its index (the line sweeps), or as the x sweep's waves address it: an
// index that is the same for all lanes, kept in scalar registers, and this lane's
// distance from it in bytes.  The second form leaves a load's address to the
// scalar unit: 115 vector instructions less in the FP64 SLAU6 NS run, and 437 ->
// 415 us for Hybrid6 LES 192^3.  In the line sweeps' loops it spilled scalar
// registers.
struct CellAt {
  long long u;
  unsigned lane;
};
template <class S> __device__ __forceinline__ S at(const S* f, const CellAt& c, long long off = 0) {
  using GC = __attribute__((address_space(1))) const char;
  using GS = __attribute__((address_space(1))) const S;
  return *(GS*)((GC*)G(f + (c.u + off)) + c.lane);
}
template <class S> __device__ __forceinline__ S at(const S* f, int m, int off = 0) { return G(f)[m + off]; }

// Issues the loads of cell m (sensor read at ms, its periodic image): its own
// values, and the transverse stencil values of a viscous run.
template <class S, int DIR, int ORDER, int SCHEME, int VISC, int VO, bool LOAD_S = true, class C>
__device__ __forceinline__ void fetch_values(const Prim<S>& P, const C& m, const C& ms,
                                             RawCell<S, VISC, VO>& r) {
  r.rho = at(P.rho, m);
  r.u = at(P.u, m);
  r.v = at(P.v, m);
  r.w = at(P.w, m);
  r.p = at(P.p, m);
  if constexpr (LOAD_S && kUsesSensor<SCHEME, ORDER>) r.s = at(P.s, ms);
  if constexpr (VISC == 2) {
    r.mt = at(P.mut, m);
    r.qc2 = at(P.qc2, m);
  }
}
template <class S, int DIR, int VISC, int VO, class C>
__device__ __forceinline__ void fetch_cross(const Prim<S>& P, const Geom& g, const C& m, RawCell<S, VISC, VO>& r) {
  if constexpr (VISC) {
    const S* f[4];
    int st[4];
    cross_fields<S, DIR>(P, g, f, st);
    constexpr int VC = vcross<VO>();
#pragma unroll
    for (int q = 0; q < 4; ++q) {
#pragma unroll
      for (int t = 0; t < VC; ++t) {
        const int off = t < VC / 2 ? t - VC / 2 : t - VC / 2 + 1;
        r.x[q][t] = at(f[q], m, off * st[q]);
      }
    }
  }
}
template <class S, int DIR, int ORDER, int SCHEME, int VISC, int VO, bool LOAD_S = true, class C>
__device__ __forceinline__ void fetch_cell(const Prim<S>& P, const Geom& g, const C& m, const C& ms,
                                           RawCell<S, VISC, VO>& r) {
  fetch_values<S, DIR, ORDER, SCHEME, VISC, VO, LOAD_S>(P, m, ms, r);
  fetch_cross<S, DIR, VISC, VO>(P, g, m, r);
}

// cross_d over the raw stencil values (centre entry zero, never read)
template <class R, class S, int VO>
__device__ __forceinline__ R cross_raw(const PhysC<R>& c, const S* x, R inv) {
  constexpr int VC = vcross<VO>();
  R a[VC + 1];
#pragma unroll
  for (int t = 0; t <= VC; ++t) a[t] = (t == VC / 2) ? R(0) : R(x[t < VC / 2 ? t : t - 1]);
  return cross_d<R, VC>(c, inv, a);
}

// Turns the loaded values into the window cell (conversions, cross
// derivatives, LES total enthalpy).
template <class R, class S, int DIR, int ORDER, int SCHEME, int VISC, int VO, bool LOAD_S = true>
__device__ __forceinline__ void finish_cell(const Geom& g, const PhysC<R>& c, const RawCell<S, VISC, VO>& r,
                                            CellData<R, DIR, ORDER, SCHEME, VISC, VO>& d) {
  d.rho = R(r.rho);
  d.u = R(r.u);
  d.v = R(r.v);
  d.w = R(r.w);
  d.p = R(r.p);
  // T = p / (R rho) and Sutherland's law (calc_quantities_T_3D,
  // src/calc_physical_quantities.f90:60-116)
  if constexpr (kUsesT<SCHEME> || VISC) d.T = d.p / (c.Rgas * d.rho);
  if constexpr (VISC) d.mu = c.mu0c / (d.T + R(111.0)) * (d.T * fsqrt(d.T));
  if constexpr (LOAD_S && kUsesSensor<SCHEME, ORDER>) d.s = R(r.s);
  if constexpr (VISC) {
    if constexpr (VISC == 2) {
      d.mt = R(r.mt);
      d.H = c.Cp * d.T + R(0.5) * (d.u * d.u + d.v * d.v + d.w * d.w) + R(r.qc2);
    }
    const R ix = R(g.inv_dx), iy = R(g.inv_dy), iz = R(g.inv_dz);
    const R i0 = DIR == 0 ? iy : ix, i1 = DIR == 0 ? iy : ix;
    const R i2 = DIR == 2 ? iy : iz, i3 = DIR == 2 ? iy : iz;
    d.d1 = cross_raw<R, S, VO>(c, r.x[0], i0);
    d.d2 = cross_raw<R, S, VO>(c, r.x[1], i1);
    d.d3 = cross_raw<R, S, VO>(c, r.x[2], i2);
    d.d4 = cross_raw<R, S, VO>(c, r.x[3], i3);
  }
}

// Loads the primitive values (and, for viscous runs, the cross derivatives a
// face in direction DIR needs) of cell (i,j,k) = linear m.
template <class R, class S, int DIR, int ORDER, int SCHEME, int VISC, int VO, bool LOAD_S = true>
__device__ __forceinline__ void load_cell(const Prim<S>& P, const Geom& g, const PhysC<R>& c, int m, int ms,
                                          CellData<R, DIR, ORDER, SCHEME, VISC, VO>& d) {
  RawCell<S, VISC, VO> r;
  fetch_cell<S, DIR, ORDER, SCHEME, VISC, VO, LOAD_S>(P, g, m, ms, r);
  finish_cell<R, S, DIR, ORDER, SCHEME, VISC, VO, LOAD_S>(g, c, r, d);
}

// Convective face flux from SW window cells w[0..SW-1]; the face lies
// between w[HW-1] and w[HW].
template <class R, int DIR, int ORDER, int SCHEME, int VISC, int VO>
__device__ __forceinline__ void face_conv(const PhysC<R>& c, int tvd, int variant,
                                          const CellData<R, DIR, ORDER, SCHEME, VISC, VO>* w, R* F) {
  using St = Sten<ORDER, VISC, VO>;
  constexpr int N = ORDER;
  R rho[N], u[N], v[N], wv[N], p[N], T[N];
#pragma unroll
  for (int m = 0; m < N; ++m) {
    rho[m] = w[St::CO + m].rho;
    u[m] = w[St::CO + m].u;
    v[m] = w[St::CO + m].v;
    wv[m] = w[St::CO + m].w;
    p[m] = w[St::CO + m].p;
    if constexpr (kUsesT<SCHEME>) T[m] = w[St::CO + m].T;
  }
  R fs = R(0);
  if constexpr (kUsesSensor<SCHEME, ORDER>) fs = R(0.5) * (w[St::HW - 1].s + w[St::HW].s);
  if constexpr (SCHEME == KEEP) {
    keep_face<R, DIR, N>(c, rho, u, v, wv, p, T, F);
  } else if constexpr (SCHEME == SLAU) {
    slau_face<R, DIR, N>(c, tvd, variant, rho, u, v, wv, p, fs, F);
  } else if constexpr (SCHEME == ROE) {
    roe_face<R, DIR, N>(c, tvd, rho, u, v, wv, p, fs, F);
  } else {
    // calc_hybrid_{x,y,z}_in (calc_hybrid_kernel_internal.f90.fypp:96-121)
    if (fs <= c.threshold) {
      keep_face<R, DIR, N>(c, rho, u, v, wv, p, T, F);
    } else {
      R L[5], Rr[5];
      reconstruct<R, N>(c, tvd, fs, rho, u, v, wv, p, L, Rr);
      slau<R, DIR>(c, variant, L[0], Rr[0], L[1], Rr[1], L[2], Rr[2], L[3], Rr[3], L[4], Rr[4], R(1), F);
    }
  }
}

// Subtracts the viscous face flux from F (convective in, total out).
template <class R, int DIR, int ORDER, int SCHEME, int VISC, int VO>
__device__ __forceinline__ void face_visc(const PhysC<R>& c, R inv_d,
                                          const CellData<R, DIR, ORDER, SCHEME, VISC, VO>* w, R* F) {
  using St = Sten<ORDER, VISC, VO>;
  if constexpr (VISC) {
    constexpr int M = vwin<VO>();
    R mu_[M], T_[M], u_[M], v_[M], w_[M], a1[M], a2[M], a3[M], a4[M], mt_[M], H_[M];
#pragma unroll
    for (int m = 0; m < M; ++m) {
      const auto& x = w[St::VOFF + m];
      mu_[m] = x.mu; T_[m] = x.T; u_[m] = x.u; v_[m] = x.v; w_[m] = x.w;
      a1[m] = x.d1; a2[m] = x.d2; a3[m] = x.d3; a4[m] = x.d4;
      if constexpr (VISC == 2) { mt_[m] = x.mt; H_[m] = x.H; }
    }
    R tau[3], en;
    if constexpr (VO == 5) visc_face_me4<R, DIR, (VISC == 2)>(c, inv_d, mu_, T_, u_, v_, w_, a1, a2, a3, a4, tau, en, mt_, H_);
    else visc_face<R, DIR, M, (VISC == 2)>(c, inv_d, mu_, T_, u_, v_, w_, a1, a2, a3, a4, tau, en, mt_, H_);
    F[1] = F[1] - tau[0];
    F[2] = F[2] - tau[1];
    F[3] = F[3] - tau[2];
    F[4] = F[4] - en;
  }
}

// Face flux (convective minus viscous) from SW window cells w[0..SW-1].
template <class R, int DIR, int ORDER, int SCHEME, int VISC, int VO>
__device__ __forceinline__ void face_flux(const PhysC<R>& c, int tvd, int variant, R inv_d,
                                          const CellData<R, DIR, ORDER, SCHEME, VISC, VO>* w, R* F) {
  face_conv<R, DIR, ORDER, SCHEME, VISC, VO>(c, tvd, variant, w, F);
  face_visc<R, DIR, ORDER, SCHEME, VISC, VO>(c, inv_d, w, F);
}

// ---------------------------------------------------------------------------
// Launch descriptors.  SweepArgs carries everything one sweep of one case
// needs; the single-case kernels take it by value, the batched kernels read
// an array of them (one per case) and map their blocks onto the cases' tiles
// through a TileMap (first global tile index and tile counts per case).
// ---------------------------------------------------------------------------
template <class R, class S> struct SweepArgs {
  Prim<S> P;        // primitives read by the stage
  Prim<S> Pn;       // primitives of the new state (written by the z epilogue)
  S* Racc;          // residual accumulator
  Geom g;
  PhysC<R> c;
  PhysC<double> c64;
  StageArgs sa;
  double cd;        // c_x, c_y or c_z of calc_R (stage coefficient * dt * face area)
  int tvd, variant;
  int lseg;         // cells per thread segment in the y / z sweeps
  int xrows, xwgs;  // x sweep: rows of a band, workgroups per band and plane
};

struct TileMap {
  int start;     // first global tile of the case
  int nbx, nby;  // tiles along the three launch dimensions
  int nbz;
};

// Case owning global tile t (map[].start ascending, map[0].start == 0).
__device__ __forceinline__ int find_case(const TileMap* __restrict__ map, int ncase, int t) {
  int lo = 0, hi = ncase - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (map[mid].start <= t) lo = mid;
    else hi = mid - 1;
  }
  return lo;
}

#ifndef OX_SPLIT_FENCE
#define OX_SPLIT_FENCE() asm volatile("" ::: "memory")
#endif

// Ducros sensor of one cell (calc_Ducros, 3D_solver/src/calc_hybrid.f90:11-72)
// from its six face neighbours' velocities.
template <class R>
__device__ __forceinline__ R ducros(const Geom& g, R uxm, R uxp, R vxm, R vxp, R wxm, R wxp, R uym, R uyp, R vym,
                                    R vyp, R wym, R wyp, R uzm, R uzp, R vzm, R vzp, R wzm, R wzp) {
  const R dxt = R(0.25) * (R(g.inv_dx) + R(g.inv_dx));
  const R dyt = R(0.25) * (R(g.inv_dy) + R(g.inv_dy));
  const R dzt = R(0.25) * (R(g.inv_dz) + R(g.inv_dz));
  const R dudx = (-uxm + uxp) * dxt;
  const R dvdx = (-vxm + vxp) * dxt;
  const R dwdx = (-wxm + wxp) * dxt;
  const R dudy = (-uym + uyp) * dyt;
  const R dvdy = (-vym + vyp) * dyt;
  const R dwdy = (-wym + wyp) * dyt;
  const R dudz = (-uzm + uzp) * dzt;
  const R dvdz = (-vzm + vzp) * dzt;
  const R dwdz = (-wzm + wzp) * dzt;
  const R div = dudx + dvdy + dwdz;
  const R r1 = dwdy - dvdz;
  const R r2 = dudz - dwdx;
  const R r3 = dvdx - dudy;
  R fd = (div * div) / (div * div + (r1 * r1 + r2 * r2 + r3 * r3) + R(1.0e-12));
  return fmin2(R(1), fd);
}

// The same sensor in two parts: the y/z-derivative terms (from loads the
// cell's own thread issues) and the completion with the x derivatives (from
// the LDS row).  Same operations in the same order as ducros().
template <class R> struct DucrosPart {
  R dudy, dvdy, dwdz, dudz, r1;
};
template <class R>
__device__ __forceinline__ DucrosPart<R> ducros_yz(const Geom& g, R uym, R uyp, R vym, R vyp, R wym, R wyp, R uzm,
                                                   R uzp, R vzm, R vzp, R wzm, R wzp) {
  const R dyt = R(0.25) * (R(g.inv_dy) + R(g.inv_dy));
  const R dzt = R(0.25) * (R(g.inv_dz) + R(g.inv_dz));
  DucrosPart<R> d;
  d.dudy = (-uym + uyp) * dyt;
  d.dvdy = (-vym + vyp) * dyt;
  const R dwdy = (-wym + wyp) * dyt;
  d.dudz = (-uzm + uzp) * dzt;
  const R dvdz = (-vzm + vzp) * dzt;
  d.dwdz = (-wzm + wzp) * dzt;
  d.r1 = dwdy - dvdz;
  return d;
}
template <class R>
__device__ __forceinline__ R ducros_x(const Geom& g, const DucrosPart<R>& d, R uxm, R uxp, R vxm, R vxp, R wxm,
                                      R wxp) {
  const R dxt = R(0.25) * (R(g.inv_dx) + R(g.inv_dx));
  const R dudx = (-uxm + uxp) * dxt;
  const R dvdx = (-vxm + vxp) * dxt;
  const R dwdx = (-wxm + wxp) * dxt;
  const R div = dudx + d.dvdy + d.dwdz;
  const R r2 = d.dudz - dwdx;
  const R r3 = dvdx - d.dudy;
  R fd = (div * div) / (div * div + (d.r1 * d.r1 + r2 * r2 + r3 * r3) + R(1.0e-12));
  return fmin2(R(1), fd);
}

// ---------------------------------------------------------------------------
// x sweep: runs of faces.  A row of ix cells has ix + 1 faces; the faces of a
// band of rows of one plane, row after row, are dealt to waves, one face per
// lane, each starting at the last face of the wave before (its first cell needs
// that face too); the four waves of a workgroup share the LDS rows.  A lane
// loads the cell right of its face; the SW - 1 other cells that the faces of a
// row piece read, left and right of it, are loaded by the first lanes.  The LDS
// rows are structure-of-arrays so that lane-consecutive reads are bank-conflict
// free.  The flux of a cell's right face comes from the next lane.
//
// Writes Racc = c_x * (E_right - E_left) (the first term of calc_R).  For
// the schemes that read the Ducros sensor the sweep also computes it for its
// cells and stores it for the y and z sweeps.
//
// Bound by the vector units and, on large grids, by memory as well (FP64 SLAU6 NS
// 256^3: units busy 0.58 to 0.61 of the time, 4.4 TB/s), so by the lanes that hold
// no face.  Row tiles of one wave, 64 less the halo's SW - 1, spent 192 lanes on a
// row of 124 cells and 128 on one of 80; runs lose one lane in 64, the halo cells'
// loads and the end of a band.  Measured (us), tiles -> runs: FP64 SLAU6 NS 80 x
// 112 x 48 38 -> 29, 124^3 122 -> 101, 192^3 417 -> 366; Hybrid6 LES 64^3 35 -> 26,
// 192^3 494 -> 415, 256^3 1088 -> 958; KEEP4 NS 192^3 241 -> 226, 96^3 23.1 -> 24.8
// (rows of 97 faces fit two tiles as well, and memory bounds it); FP32 Roe4 NS
// 124^3 52 -> 44, SLAU6 Euler 124^3 49 -> 41, KEEP4 Euler 144^3 34 -> 30.
// ---------------------------------------------------------------------------
// The fields of an LDS row: rho,u,v,w,p, then those that the scheme reads.
template <int ORDER, int SCHEME, int VISC> struct XFields {
  static constexpr int T = 5;
  static constexpr int s = T + (kUsesT<SCHEME> || VISC ? 1 : 0);
  static constexpr int mu = s + (kUsesSensor<SCHEME, ORDER> ? 1 : 0);
  static constexpr int d = mu + 1;  // d1..d4
  static constexpr int mt = d + 4, H = mt + 1;
  static constexpr int N = VISC == 0 ? mu : VISC == 1 ? mt : H + 1;
};
constexpr int XRUN = 4 * 63;  // cells of a run: 64 faces per wave, one shared with the next wave
// row pieces of a run at most: rows have at least 2 ORDER + 1 faces
template <int ORDER> constexpr int xrun_pieces() { return XRUN / (2 * ORDER + 1) + 2; }
template <int ORDER, int VISC, int VO> constexpr int xrun_len() {
  return XRUN + 1 + (Sten<ORDER, VISC, VO>::SW - 1) * xrun_pieces<ORDER>();
}
template <class R, int ORDER, int SCHEME, int VISC, int VO> struct XRunTile {
  R f[XFields<ORDER, SCHEME, VISC>::N][xrun_len<ORDER, VISC, VO>()];
};

// Rows per band and workgroups per band and plane: the workgroups of a band walk
// its planes, so that the y neighbours of the cross-derivative and sensor stencils
// are read once per band from L2; 8 to 32 rows, the number that leaves the
// fewest lanes idle, near 16 where several do.
inline void xrun_shape(const Geom& g, int& rows, int& wgs) {
  long long best = -1;
  rows = wgs = 1;
  for (int d = 0; d <= 24; ++d) {
    const int n = 16 + ((d & 1) ? (d + 1) / 2 : -(d / 2));  // 16, 17, 15, 18, 14, ...
    if (n < 8 || n > 32) continue;
    const int m = n < g.iy ? n : g.iy;
    const long long per = ((long long)m * (g.ix + 1) - 1 + XRUN - 1) / XRUN;
    const long long total = per * ((g.iy + m - 1) / m);
    if (best < 0 || total < best) best = total, rows = m, wgs = (int)per;
  }
}
inline long long xrun_blocks(const Geom& g) {
  int rows, wgs;
  xrun_shape(g, rows, wgs);
  return (long long)wgs * g.iz * ((g.iy + rows - 1) / rows);
}

template <class R, class S, int ORDER, int SCHEME, int VISC, int VO>
__device__ __forceinline__ void sweep_x_run(const SweepArgs<R, S>& a, int t, XRunTile<R, ORDER, SCHEME, VISC, VO>& lds) {
  using St = Sten<ORDER, VISC, VO>;
  using CD = CellData<R, 0, ORDER, SCHEME, VISC, VO>;
  using RC = RawCell<S, VISC, VO>;
  constexpr bool SENS = kUsesSensor<SCHEME, ORDER>;
  // With one ghost layer (ORDER 2) a ghost cell's sensor is the boundary copy
  // of its interior neighbour (calc_hybrid.f90:54-71), taken from a clamped
  // index; with more layers every sensor the faces read belongs to a cell in
  // 1..nx-2 whose x neighbours are in the LDS row.
  constexpr bool SPLIT_SENS = SENS && ORDER > 2;
  // With few fields and little arithmetic the loads' latency shows: the halo's go
  // first (FP32 KEEP Euler 144^3 33 -> 30 us; SLAU6 Euler lost 3%).
  constexpr bool EARLY = SCHEME == KEEP && !VISC;
  using XF = XFields<ORDER, SCHEME, VISC>;
  constexpr int HW = St::HW, SW = St::SW;
  static_assert((SW - 1) * xrun_pieces<ORDER>() <= 256, "one halo cell per lane");
  auto& tile = lds.f;
  const Prim<S>& P = a.P;
  const Geom& g = a.g;
  const PhysC<R>& c = a.c;
  const int tid = threadIdx.x, lane = tid & 63;
  const int sy = g.nx, sz = g.nx * g.ny;
  // run w of plane k and band of rows j0 ..: faces c0 .. last of the band's rows
  const int n1 = g.ix + 1;  // faces of a row
  const int w = t % a.xwgs, kb = t / a.xwgs;
  const int k = g.h + kb % g.iz, j0 = kb / g.iz * a.xrows;
  const int total = min(a.xrows, g.iy - j0) * n1;
  const int c0 = w * XRUN, last = min(XRUN, total - 1 - c0);
  if (last < 1) return;  // (the whole workgroup) a shorter last band
  const int p0 = c0 / n1, f0 = c0 - p0 * n1;  // the run's first row and face
  // piece of lane (or face offset) x: rows shorter than a run by an exact float
  // quotient (x + f0 < 512), longer ones have two pieces at most
  const float inv = 1.0f / (float)n1;
  auto piece = [&](int x) { return n1 > 256 ? (int)(x + f0 >= n1) : (int)((x + f0 + 0.5f) * inv); };
  const int x = (tid >> 6) * 63 + lane;  // this lane's face of the run
  const int q = piece(x), f = x + f0 - q * n1;
  const bool ok = x <= last;
  const int i = g.h + f, j = g.h + j0 + p0 + q;
  const int pos = x + (SW - 1) * q + HW;  // this lane's cell in the LDS row
  const bool own = ok && lane < 63 && f < g.ix;  // the cell this lane completes
  // halo cell tid: cell he of piece hq, left (e < HW) or right of it
  const int hq = tid / (SW - 1), e = tid % (SW - 1);
  const bool halo = hq <= piece(last);
  const int l0 = hq == 0 ? 0 : hq * n1 - f0, l1 = min(last, (hq + 1) * n1 - 1 - f0);  // the piece's lanes
  const int hx = e < HW ? l0 - HW + e : l1 + 1 + e - HW;  // as a lane
  const int hat = hx + (SW - 1) * hq + HW;
  const int hi = g.h + hx + f0 - hq * n1, hj = g.h + j0 + p0 + hq;
  const bool hsens = SENS && halo && e == HW - 1;  // left of the piece's first face

  auto part = [&](const CellAt& m, const RC& r) {
    constexpr int H = vcross<VO>() / 2;  // r.x[.][H-1], r.x[.][H]: the -1 and +1 neighbours
    R uym, uyp, vym, vyp, uzm, uzp, wzm, wzp;
    if constexpr (VISC) {  // DIR 0 cross stencils: u,v along y; u,w along z
      uym = R(r.x[0][H - 1]); uyp = R(r.x[0][H]);
      vym = R(r.x[1][H - 1]); vyp = R(r.x[1][H]);
      uzm = R(r.x[2][H - 1]); uzp = R(r.x[2][H]);
      wzm = R(r.x[3][H - 1]); wzp = R(r.x[3][H]);
    } else {
      uym = R(at(P.u, m, -sy)); uyp = R(at(P.u, m, sy));
      vym = R(at(P.v, m, -sy)); vyp = R(at(P.v, m, sy));
      uzm = R(at(P.u, m, -sz)); uzp = R(at(P.u, m, sz));
      wzm = R(at(P.w, m, -sz)); wzp = R(at(P.w, m, sz));
    }
    return ducros_yz<R>(g, uym, uyp, vym, vyp, R(at(P.w, m, -sy)), R(at(P.w, m, sy)), uzm, uzp, R(at(P.v, m, -sz)),
                        R(at(P.v, m, sz)), wzm, wzp);
  };
  auto put = [&](int x, const CD& d) {
    tile[0][x] = d.rho; tile[1][x] = d.u; tile[2][x] = d.v; tile[3][x] = d.w; tile[4][x] = d.p;
    if constexpr (kUsesT<SCHEME> || VISC) tile[XF::T][x] = d.T;
    if constexpr (VISC) {
      tile[XF::mu][x] = d.mu;
      tile[XF::d][x] = d.d1; tile[XF::d + 1][x] = d.d2; tile[XF::d + 2][x] = d.d3; tile[XF::d + 3][x] = d.d4;
      if constexpr (VISC == 2) { tile[XF::mt][x] = d.mt; tile[XF::H][x] = d.H; }
    }
  };
  DucrosPart<R> dp{}, hdp{};
  // cells from the start of the run's first row
  const int row0 = cidx(g, 0, g.h + j0 + p0, k);
  const CellAt m{row0, (unsigned)(i + q * sy) * (unsigned)sizeof(S)};
  const CellAt hm{row0, (unsigned)(hi + hq * sy) * (unsigned)sizeof(S)};
  RC r, hr;
  auto take = [&](const CellAt& m, RC& r) { fetch_cell<S, 0, ORDER, SCHEME, VISC, VO, false>(P, g, m, m, r); };
  auto fill = [&](int x, const RC& r) {
    CD d;
    finish_cell<R, S, 0, ORDER, SCHEME, VISC, VO, false>(g, c, r, d);
    put(x, d);
  };
  if constexpr (EARLY) {
    if (halo) take(hm, hr);
  }
  if (ok) {
    take(m, r);
    if constexpr (SPLIT_SENS) dp = part(m, r);
    fill(pos, r);
  }
  if (halo) {
    if constexpr (!EARLY) take(hm, hr);
    if constexpr (SPLIT_SENS) {
      if (hsens) hdp = part(hm, hr);
    }
    fill(hat, hr);
  }
  __syncthreads();
  if constexpr (SENS) {
    auto sensor = [&](int x, int ci, int cj, const DucrosPart<R>& part_yz) {
      if constexpr (SPLIT_SENS) {
        return ducros_x<R>(g, part_yz, tile[1][x - 1], tile[1][x + 1], tile[2][x - 1], tile[2][x + 1], tile[3][x - 1],
                           tile[3][x + 1]);
      } else {
        const int n = cidx(g, min(max(ci, 1), g.nx - 2), cj, k);
        return ducros<R>(g, R(G(P.u)[n - 1]), R(G(P.u)[n + 1]), R(G(P.v)[n - 1]), R(G(P.v)[n + 1]), R(G(P.w)[n - 1]),
                         R(G(P.w)[n + 1]), R(G(P.u)[n - sy]), R(G(P.u)[n + sy]), R(G(P.v)[n - sy]), R(G(P.v)[n + sy]),
                         R(G(P.w)[n - sy]), R(G(P.w)[n + sy]), R(G(P.u)[n - sz]), R(G(P.u)[n + sz]), R(G(P.v)[n - sz]),
                         R(G(P.v)[n + sz]), R(G(P.w)[n - sz]), R(G(P.w)[n + sz]));
      }
    };
    if (ok) {
      const R fd = sensor(pos, i, j, dp);
      tile[XF::s][pos] = fd;
      if (own) G(P.s)[cidx(g, i, j, k)] = (S)fd;  // one run stores a cell
    }
    if (hsens) tile[XF::s][hat] = sensor(hat, hi, hj, hdp);
    __syncthreads();
  }
  // face f: window cells f - HW .. f + HW - 1
  R F[5] = {R(0), R(0), R(0), R(0), R(0)};
  if (ok) {
    const int w0 = pos - HW;
    // The convective and the viscous halves each read their window from the
    // LDS row just before use, which keeps the two halves' inputs out of
    // registers at the same time.
    {
      CD win[SW];
#pragma unroll
      for (int n = 0; n < SW; ++n) {
        win[n].rho = tile[0][w0 + n]; win[n].u = tile[1][w0 + n]; win[n].v = tile[2][w0 + n];
        win[n].w = tile[3][w0 + n]; win[n].p = tile[4][w0 + n];
        if constexpr (kUsesT<SCHEME>) win[n].T = tile[XF::T][w0 + n];
        if constexpr (SENS) {
          if (n == HW - 1 || n == HW) win[n].s = tile[XF::s][w0 + n];
        }
      }
      face_conv<R, 0, ORDER, SCHEME, VISC, VO>(c, a.tvd, a.variant, win, F);
    }
    if constexpr (VISC) {
      OX_SPLIT_FENCE();
      CD win[SW];
#pragma unroll
      for (int n = 0; n < SW; ++n) {
        win[n].u = tile[1][w0 + n]; win[n].v = tile[2][w0 + n]; win[n].w = tile[3][w0 + n];
        win[n].T = tile[XF::T][w0 + n];
        win[n].mu = tile[XF::mu][w0 + n];
        win[n].d1 = tile[XF::d][w0 + n]; win[n].d2 = tile[XF::d + 1][w0 + n];
        win[n].d3 = tile[XF::d + 2][w0 + n]; win[n].d4 = tile[XF::d + 3][w0 + n];
        if constexpr (VISC == 2) { win[n].mt = tile[XF::mt][w0 + n]; win[n].H = tile[XF::H][w0 + n]; }
      }
      face_visc<R, 0, ORDER, SCHEME, VISC, VO>(c, R(g.inv_dx), win, F);
    }
  }
  // the right face is the next lane's
  double Fr[5];
#pragma unroll
  for (int l = 0; l < 5; ++l) Fr[l] = __shfl_down((double)F[l], 1, 64);
  if (own) {
    const double cx = a.cd;
#pragma unroll
    for (int l = 0; l < 5; ++l) G(a.Racc)[qidx(g, i, l, j, k)] = (S)(cx * (-(double)F[l] + Fr[l]));
  }
}

template <class R, class S, int ORDER, int SCHEME, int VISC, int VO>
__global__ __launch_bounds__(256) void k_sweep_x(SweepArgs<R, S> a) {
  __shared__ XRunTile<R, ORDER, SCHEME, VISC, VO> lds;
  sweep_x_run<R, S, ORDER, SCHEME, VISC, VO>(a, xcd_tile(blockIdx.x, gridDim.x), lds);
}

// ---------------------------------------------------------------------------
// x sweep over whole rows of a periodic grid whose interior width ix is 64,
// 128 or 256.  The runs above load a second cell in the lanes of a halo and one
// face in 64 twice; here a workgroup of 256 lanes holds 256 / ix whole rows, one lane per cell
// and one face per lane (its cell's left face), and the halo positions of the
// LDS row hold the periodic images of the row's other end.  The face left of
// the first cell is then the face right of the last: its window cells are the
// periodic images of that face's window cells.  The run computes the same face
// from the ghost cells, which hold exact copies of those images once a z-sweep
// epilogue has written the primitive set, so both give the same bits.  Used for
// such primitive sets only (k_prim takes the ghost layers of an uploaded state as
// they are), on fully periodic grids, without LES (the ghost SGS fields are copies
// of the layer next to the boundary), and not for ORDER 2 with the sensor, whose
// ghost cells copy the adjacent interior sensor
// (calc_hybrid.f90:54-71) instead of the image's.
// ---------------------------------------------------------------------------
template <int ORDER, int SCHEME, int VISC>
constexpr bool kXRowSweep = VISC != 2 && !(kUsesSensor<SCHEME, ORDER> && ORDER == 2);
__host__ __device__ constexpr bool xrow_width(int ix) { return ix == 64 || ix == 128 || ix == 256; }
// Consecutive workgroups take the rows of a band of XROW_BAND rows in one
// plane, then the next plane: the y neighbours that the cross-derivative and
// sensor stencils read are shared by workgroups resident together in one L2,
// and the z neighbours by the bands of the next planes.  (Whole rows one after
// another through the planes re-read the y neighbours of every row from HBM.)
constexpr int XROW_BAND = 16;

template <class R, class S, int ORDER, int SCHEME, int VISC, int VO>
__global__ __launch_bounds__(256) void k_sweep_xrow(SweepArgs<R, S> a) {
  using St = Sten<ORDER, VISC, VO>;
  using CD = CellData<R, 0, ORDER, SCHEME, VISC, VO>;
  using RC = RawCell<S, VISC, VO>;
  constexpr bool SENS = kUsesSensor<SCHEME, ORDER>;
  using XF = XFields<ORDER, SCHEME, VISC>;
  constexpr int HW = St::HW, SW = St::SW;
  static_assert(kXRowSweep<ORDER, SCHEME, VISC>, "row sweep for image-ghost schemes only");
  // rows of L + SW - 1 positions: 4 * (63 + SW) covers L = 64 (four rows) to 256 (one)
  __shared__ R tile[XF::N][4 * (63 + SW)];
  __shared__ double edge[4][5];  // each wave's lane-0 face flux
  const Prim<S>& P = a.P;
  const Geom& g = a.g;
  const PhysC<R>& c = a.c;
  const int L = g.ix, rw = 256 / L;  // row length, rows per workgroup
  const int tid = threadIdx.x, lane = tid & 63;
  const int r = tid / L, p = tid - r * L;  // row in the workgroup, cell in the row
  const int nbb = XROW_BAND / rw;  // workgroups per band
  const int t = xcd_tile(blockIdx.x, gridDim.x);
  const int j = g.h + (t / (nbb * g.iz)) * XROW_BAND + (t % nbb) * rw + r, k = g.h + (t / nbb) % g.iz;
  const bool rowok = j < g.h + g.iy;
  const int i = g.h + p;
  const int rb = r * (L + SW - 1);  // the row's first position, cell h - HW
  const int m = p + HW;             // this lane's position
  const int q = cidx(g, i, j, k);
  DucrosPart<R> dp{};
  if (rowok) {
    RC rc;
    // Scalar addresses where the registers that they cost lower no occupancy: FP64
    // KEEP4 NS 256^3 421 -> 391 us, 128^3 60.6 -> 56.1; SLAU6 NS 128^3 99 -> 108.
    const auto qa = [&] {
      if constexpr (SCHEME == KEEP && VISC && sizeof(R) == 8)
        return CellAt{cidx(g, 0, j - r, k), (unsigned)(i + r * g.nx) * (unsigned)sizeof(S)};
      else
        return q;
    }();
    fetch_cell<S, 0, ORDER, SCHEME, VISC, VO, false>(P, g, qa, qa, rc);
    if constexpr (SENS) {
      const int sy = g.nx, sz = g.nx * g.ny;
      constexpr int H = vcross<VO>() / 2;
      R uym, uyp, vym, vyp, uzm, uzp, wzm, wzp;
      if constexpr (VISC) {
        uym = R(rc.x[0][H - 1]); uyp = R(rc.x[0][H]);
        vym = R(rc.x[1][H - 1]); vyp = R(rc.x[1][H]);
        uzm = R(rc.x[2][H - 1]); uzp = R(rc.x[2][H]);
        wzm = R(rc.x[3][H - 1]); wzp = R(rc.x[3][H]);
      } else {
        uym = R(at(P.u, qa, -sy)); uyp = R(at(P.u, qa, sy));
        vym = R(at(P.v, qa, -sy)); vyp = R(at(P.v, qa, sy));
        uzm = R(at(P.u, qa, -sz)); uzp = R(at(P.u, qa, sz));
        wzm = R(at(P.w, qa, -sz)); wzp = R(at(P.w, qa, sz));
      }
      dp = ducros_yz<R>(g, uym, uyp, vym, vyp, R(at(P.w, qa, -sy)), R(at(P.w, qa, sy)), uzm, uzp, R(at(P.v, qa, -sz)),
                        R(at(P.v, qa, sz)), wzm, wzp);
    }
    CD d;
    finish_cell<R, S, 0, ORDER, SCHEME, VISC, VO, false>(g, c, rc, d);
    auto put = [&](int x) {
      x += rb;
      tile[0][x] = d.rho; tile[1][x] = d.u; tile[2][x] = d.v; tile[3][x] = d.w; tile[4][x] = d.p;
      if constexpr (kUsesT<SCHEME> || VISC) tile[XF::T][x] = d.T;
      if constexpr (VISC) {
        tile[XF::mu][x] = d.mu;
        tile[XF::d][x] = d.d1; tile[XF::d + 1][x] = d.d2; tile[XF::d + 2][x] = d.d3; tile[XF::d + 3][x] = d.d4;
      }
    };
    put(m);
    if (p >= L - HW) put(m - L);      // left halo: images of the row's last HW cells
    if (p < SW - HW - 1) put(m + L);  // right halo: images of its first SW - HW - 1
  }
  __syncthreads();
  if constexpr (SENS) {
    if (rowok) {
      const int x = rb + m;
      const R fd = ducros_x<R>(g, dp, tile[1][x - 1], tile[1][x + 1], tile[2][x - 1], tile[2][x + 1],
                               tile[3][x - 1], tile[3][x + 1]);
      tile[XF::s][x] = fd;
      if (p == L - 1) tile[XF::s][rb + HW - 1] = fd;  // the image left of the row
      G(P.s)[q] = (S)fd;
    }
    __syncthreads();
  }
  R F[5] = {R(0), R(0), R(0), R(0), R(0)};
  if (rowok) {
    const int w0 = rb + p;  // window cells h + p - HW .. h + p + HW - 1
    {
      CD win[SW];
#pragma unroll
      for (int n = 0; n < SW; ++n) {
        win[n].rho = tile[0][w0 + n]; win[n].u = tile[1][w0 + n]; win[n].v = tile[2][w0 + n];
        win[n].w = tile[3][w0 + n]; win[n].p = tile[4][w0 + n];
        if constexpr (kUsesT<SCHEME>) win[n].T = tile[XF::T][w0 + n];
        if constexpr (SENS) {
          if (n == HW - 1 || n == HW) win[n].s = tile[XF::s][w0 + n];
        }
      }
      face_conv<R, 0, ORDER, SCHEME, VISC, VO>(c, a.tvd, a.variant, win, F);
    }
    if constexpr (VISC) {
      OX_SPLIT_FENCE();
      CD win[SW];
#pragma unroll
      for (int n = 0; n < SW; ++n) {
        win[n].u = tile[1][w0 + n]; win[n].v = tile[2][w0 + n]; win[n].w = tile[3][w0 + n];
        win[n].T = tile[XF::T][w0 + n];
        win[n].mu = tile[XF::mu][w0 + n];
        win[n].d1 = tile[XF::d][w0 + n]; win[n].d2 = tile[XF::d + 1][w0 + n];
        win[n].d3 = tile[XF::d + 2][w0 + n]; win[n].d4 = tile[XF::d + 3][w0 + n];
      }
      face_visc<R, 0, ORDER, SCHEME, VISC, VO>(c, R(g.inv_dx), win, F);
    }
  }
  // the right face is the next cell's left face: the next lane's, across a
  // wave boundary the next wave's lane 0, and after the row's last cell the
  // row's first (with L = 64 the row is the wave, and the rotation covers it)
  double Fr[5];
#pragma unroll
  for (int l = 0; l < 5; ++l) Fr[l] = __shfl((double)F[l], (lane + 1) & 63, 64);
  if (L > 64) {
    if (lane == 0) {
#pragma unroll
      for (int l = 0; l < 5; ++l) edge[tid >> 6][l] = (double)F[l];
    }
    __syncthreads();
    if (lane == 63) {
      const int wn = (r * L + ((p + 1) & (L - 1))) >> 6;
#pragma unroll
      for (int l = 0; l < 5; ++l) Fr[l] = edge[wn][l];
    }
  }
  if (rowok) {
    const double cx = a.cd;
#pragma unroll
    for (int l = 0; l < 5; ++l) G(a.Racc)[qidx(g, i, l, j, k)] = (S)(cx * (-(double)F[l] + Fr[l]));
  }
}

// Batched sweeps over the tiles of several cases, one workgroup per tile, as in a
// lone case's launch: the hardware gives a free slot the next tile.  1024
// workgroups that each walked every 1024th tile left the compute units at half
// their waves and finished unevenly: six FP32 requests of 64^3 to 160^3, 60 steps,
// 156 -> 150 ms for the x sweep and 139 with the y and z sweeps.
template <class R, class S, int ORDER, int SCHEME, int VISC, int VO>
__global__ __launch_bounds__(256) void k_sweep_x_batch(const SweepArgs<R, S>* __restrict__ cases,
                                                       const TileMap* __restrict__ map, int ncase, int ntiles) {
  __shared__ XRunTile<R, ORDER, SCHEME, VISC, VO> lds;
  const unsigned b = launch_block();
  if (b >= (unsigned)ntiles) return;
  const int t = xcd_tile(b, ntiles), ci = find_case(map, ncase, t);
  sweep_x_run<R, S, ORDER, SCHEME, VISC, VO>(cases[ci], t - map[ci].start, lds);
}

// The residual of one cell and, for the z sweep, the state values its RK
// epilogue reads (A = Qin, B = Qout, C = Rs), per conserved variable.
template <int DIR, int EP> struct CellState {
  double R[5], A[5], B[5], C[5];
};
template <int DIR, int EP, class S>
__device__ __forceinline__ void fetch_state(const S* __restrict__ Racc, const StageArgs& sa, int q, int st,
                                            CellState<DIR, EP>& cs) {
#pragma unroll
  for (int l = 0; l < 5; ++l) cs.R[l] = (double)G(Racc)[q + l * st];
  if constexpr (DIR == 2) {
    if constexpr (EP == EP_RK3_S1 || EP == EP_RK3_S23 || EP == EP_RK4_S) {
#pragma unroll
      for (int l = 0; l < 5; ++l) cs.A[l] = G(sa.Qin)[q + l * st];
    }
    if constexpr (EP == EP_RK3_S23 || EP == EP_RK4_S4) {
#pragma unroll
      for (int l = 0; l < 5; ++l) cs.B[l] = G(sa.Qout)[q + l * st];
    }
    if constexpr (EP == EP_RK4_S || EP == EP_RK4_S4) {
#pragma unroll
      for (int l = 0; l < 5; ++l) cs.C[l] = G(sa.Rs)[q + l * st];
    }
  }
}

// ---------------------------------------------------------------------------
// y / z sweeps: each thread owns one (x, transverse) column and marches a
// segment of LSEG cells along DIR with a register window of SW cells; loads
// are coalesced along x across the wavefront.  DIR=1 accumulates
// R += c_y*(F_right - F_left); DIR=2 adds c_z*(G_right - G_left) and applies
// the stage epilogue.
// ---------------------------------------------------------------------------
// Line-sweep workgroup: LINE_X consecutive x cells by LINE_Y rows (y rows for
// the z sweep, z rows for the y sweep), 256 threads.  The y sweep takes the
// rows in groups of LINE_Y and runs through the cells of group after group, so
// a workgroup whose x run reaches the end of the rows goes on in the next group
// and only the last workgroup has idle lanes; with whole tiles 64 - ix % 64
// lanes of every row's last tile idle (y sweep of the LES scheme at 96^3, FP64:
// tiles 72 us, this 62 us; ME4 at 150 x 77 x 53: 60 and 57 us).  The z sweep, bound
// by memory, keeps whole tiles: runs across rows slowed it (SLAU6 Euler at 124^3,
// FP64: tiles 105 us, runs 111 us).
#ifndef OX_LINE_X
#define OX_LINE_X 64
#endif
constexpr int LINE_X = OX_LINE_X;
constexpr int LINE_Y = 256 / LINE_X;
static_assert(LINE_X % 64 == 0 && LINE_X * LINE_Y == 256, "line-sweep workgroup of whole wavefronts");
// workgroups of one segment layer of the line sweep along dir
__host__ __device__ inline unsigned line_tiles(const Geom& g, int dir) {
  const long long groups = ((dir == 1 ? g.iz : g.iy) + LINE_Y - 1) / LINE_Y;
  if (dir == 1) return (unsigned)((groups * g.ix + LINE_X - 1) / LINE_X);
  return (unsigned)(groups * ((g.ix + LINE_X - 1) / LINE_X));
}

// Longest segment of the y (dir 1) or z (dir 2) sweep whose state offsets
// from a thread's column pointer (the cell before the segment) stay below
// 2^31: a thread reaches lseg + 1 cells along dir past it, plus the five
// variables of a cell, so (lseg + 2) cells of 5 nx (y) or 5 nx ny (z) values.
// At least 1 for any grid ox_create accepts (15 nx ny < 2^31).
inline int lseg_limit(const Geom& g, int dir) {
  const long long step = dir == 1 ? 5LL * g.nx : 5LL * g.nx * g.ny;
  const long long n = 2147483647LL / step - 2;
  return (int)std::max(1LL, std::min(n, 4096LL));
}
inline int clamp_lseg(const Geom& g, int dir, int lseg) { return std::min(lseg, lseg_limit(g, dir)); }

// One line sweep to be cut into segments: workgroups per segment layer and
// cells along the sweep.
struct LineWork {
  int tiles, cells;
};
inline LineWork line_work(const Geom& g, int dir) {
  return {(int)line_tiles(g, dir), dir == 1 ? g.iy : g.iz};
}
// Segment length of `cells` cells cut into the fewest segments of at most
// `lseg`, made equally long.
inline int even_lseg(int cells, int lseg) {
  const int n = (cells + lseg - 1) / lseg;
  return (cells + n - 1) / n;
}
// Longest segment of a launch over n line sweeps on `cus` compute units that
// hold `occ` workgroups each: the length L whose modelled time is least.  A
// segment costs L cells and about 5 more (the window's first cells, one extra
// face).  With k workgroups per compute unit the launch lasts
//   (L + 5) * (max(ceil(k / occ), 0.8 k) + 0.5)
// cell times of a lone workgroup: k / occ rounds while latency bounds a wave,
// 0.8 of a cell time per workgroup once the vector units or the memory do, and
// half a segment of uneven finish.  Short segments fill the chip on small
// grids, longer ones save the restarts on large ones.  Measured over grids of
// 32^3 to 256^3, KEEP4 and SLAU6, Euler and NS, both precisions: on average
// 3%, at most 19%, above the best length found by trying all; always 64 cells
// took 100 us for a KEEP4 NS y sweep at 64^3 (16 workgroups), this rule's 4
// cells 16 us.  At 256^3, where it gives 43 cells, both lie within 6%: FP64 SLAU6
// NS y 658 us and 666, z 1025 and 1043; KEEP4 NS y 488 and 518, z 955 and 947; FP32
// SLAU6 NS y 343 and 358, z 728 and 742.  The y and the z sweep share the two
// constants although their best lengths differ: KEEP4 NS z takes 838 us in segments
// of 256.
inline int pick_lseg(const LineWork* p, int n, int occ, int cus) {
  int longest = 1;
  for (int m = 0; m < n; ++m) longest = std::max(longest, p[m].cells);
  int best = longest;
  double cost = 0.0;
  for (int parts = 1, last = 0; parts <= longest; ++parts) {
    const int L = (longest + parts - 1) / parts;
    if (L == last) continue;
    last = L;
    long long blocks = 0;
    int len = 1;
    for (int m = 0; m < n; ++m) {
      const int l = even_lseg(p[m].cells, L);
      blocks += (long long)p[m].tiles * ((p[m].cells + l - 1) / l);
      len = std::max(len, l);
    }
    const long long k = (blocks + cus - 1) / cus;
    const double t = (len + 5) * (std::max((double)((k + occ - 1) / occ), 0.8 * (double)k) + 0.5);
    if (parts == 1 || t < cost) cost = t, best = L;
  }
  return best;
}

// The viscous part of a line sweep's window in LDS, a ring of SW cells per
// thread (FP64 NS): the cross derivatives, mu and (unless the convective flux
// reads it) T.  Only the viscous half of a face reads these values, so they need
// not sit in registers through the convective half nor be moved from face to
// face.  That and loading a face's operands after its convective half (below)
// let the SLAU6 NS sweeps run two waves per SIMD (254 and 256 registers; with
// the whole window in registers 368 and 416, one wave) on 74 KB of LDS per
// workgroup, with 13% fewer vector instructions.  At 256^3 y is bound by the vector
// units and latency (units busy 0.56 to 0.60 of the time), z by memory.  Best segment length on either
// side: at 256^3 y 764 -> 700, z 1091 -> 1036 us; at 192^3 y 425 -> 355, z 538 ->
// 461 us; KEEP4 NS at 64^3 y 18 -> 16, z 23 -> 21 us.  FP32 windows fit two to
// four waves as they are, and their ring was slower (SLAU6 NS at 128^3: y 58 ->
// 62, z 87 -> 88 us).  LES stays in registers at one wave: with its ring (mt and H
// as well) the FP64 z sweep spilled and took 780 us where it takes 691 (Hybrid6
// at 192^3).  Built without the memory-clause scheduler that the FP64 units use, that
// LES ring ended in an illegal memory access (Hybrid6 LES, FP64, 192^3).  Its cause is
// not known: neither ring's indices leave their arrays, nor is a slot read before it
// is written, in a host build with every array checked.  So the form is closed.
template <class R, int SCHEME, int VISC> constexpr int ring_fields() {
  return VISC != 1 || sizeof(R) != 8 ? 0 : kUsesT<SCHEME> ? 5 : 6;  // d1..d4, mu[, T]
}
template <class R, int ORDER, int SCHEME, int VISC, int VO> constexpr int ring_values() {
  return ring_fields<R, SCHEME, VISC>() * Sten<ORDER, VISC, VO>::SW * 256;
}
template <int ORDER, int SCHEME, int VISC, int VO, class R, class CD>
__device__ __forceinline__ void ring_put(R* p, const CD& d) {
  constexpr int st = Sten<ORDER, VISC, VO>::SW * 256;  // one field
  p[0] = d.d1; p[st] = d.d2; p[2 * st] = d.d3; p[3 * st] = d.d4; p[4 * st] = d.mu;
  if constexpr (!kUsesT<SCHEME>) p[5 * st] = d.T;
}
template <int ORDER, int SCHEME, int VISC, int VO, class R, class CD>
__device__ __forceinline__ void ring_get(const R* p, CD& d) {
  constexpr int st = Sten<ORDER, VISC, VO>::SW * 256;
  d.d1 = p[0]; d.d2 = p[st]; d.d3 = p[2 * st]; d.d4 = p[3 * st]; d.mu = p[4 * st];
  if constexpr (!kUsesT<SCHEME>) d.T = p[5 * st];
}
// waves per SIMD a line sweep's registers are held to
template <int VISC> constexpr int line_waves() { return VISC == 2 ? 1 : 2; }

template <class R, class S, int ORDER, int SCHEME, int VISC, int VO, int DIR, int EP>
__device__ __forceinline__ void sweep_line_tile(const SweepArgs<R, S>& a, int bx, int bz, R* ring) {
  const Prim<S>& P = a.P;
  const Prim<S>& Pn = a.Pn;
  const Geom& g = a.g;
  const PhysC<R>& c = a.c;
  const PhysC<double>& c64 = a.c64;
  const int tvd = a.tvd, variant = a.variant;
  const double cd = a.cd;
  using St = Sten<ORDER, VISC, VO>;
  using CD = CellData<R, DIR, ORDER, SCHEME, VISC, VO>;
  const int nbx = (g.ix + LINE_X - 1) / LINE_X;
  const int pos = bx * LINE_X + threadIdx.x;
  const int group = DIR == 1 ? pos / g.ix : bx / nbx;
  const int i = g.h + pos - group * (DIR == 1 ? g.ix : nbx * LINE_X);
  const int t = g.h + group * LINE_Y + threadIdx.y;  // k for DIR 1, j for DIR 2
  const int s0 = g.h + bz * a.lseg;
  const int nt = DIR == 1 ? g.iz : g.iy;
  const int nd = DIR == 1 ? g.iy : g.iz;
  if (i >= g.h + g.ix || t >= g.h + nt) return;
  const int s_end = min(s0 + a.lseg, g.h + nd);
  const int stride = DIR == 1 ? g.nx : g.nx * g.ny;
  const int mbase = DIR == 1 ? cidx(g, i, 0, t) : cidx(g, i, t, 0);
  // State, residual and RK operands: each thread's pointers to its column
  // at the cell before the segment (64-bit: the state of a large grid spans
  // more than 2^31 values), and offsets along DIR that are the same for the
  // whole workgroup (scalar registers, 32-bit: below 2^31 by the
  // segment-length limit, lseg_limit).
  const long long qcol = DIR == 1 ? qidx(g, i, 0, s0 - 1, t) : qidx(g, i, 0, t, s0 - 1);
  S* __restrict__ Racc = a.Racc + qcol;
  StageArgs sa = a.sa;
  if constexpr (DIR == 2) {
    // only the operands this epilogue touches (the others may be null)
    if constexpr (EP == EP_RK3_S1 || EP == EP_RK3_S23 || EP == EP_RK4_S) sa.Qin += qcol;
    sa.Qout += qcol;
    if constexpr (EP == EP_RK4_S || EP == EP_RK4_S4) sa.Rs += qcol;
  }
  const int qstride = DIR == 1 ? 5 * g.nx : 5 * g.nx * g.ny;
  const R inv_d = DIR == 1 ? R(g.inv_dy) : R(g.inv_dz);
  // the sensor is stored for interior cells only; a ghost cell's sensor is
  // bitwise that of its periodic image (its inputs are exact copies), except
  // with one ghost layer (ORDER 2), where the reference copies the adjacent
  // interior value into the ghost cell (calc_hybrid.f90:54-71), and along a
  // non-periodic direction, where the inner ghost layer holds its own sensor
  // (the shift is a select, not a branch: a branch in the loop would make the
  // compiler wait for every load in flight at its merge point)
  const int period = g.bc[DIR] == OX_BC_PERIODIC ? nd : 0;
  auto wrap = [&](int sp) {
    if constexpr (ORDER == 2) return sp < g.h ? g.h : (sp >= g.h + nd ? g.h + nd - 1 : sp);
    return sp < g.h ? sp + period : (sp >= g.h + nd ? sp - period : sp);
  };
  using RC = RawCell<S, VISC, VO>;
  constexpr bool RING = ring_fields<R, SCHEME, VISC>() > 0;
  static_assert(!(RING && VISC == 2), "no LES ring before the cause of its memory access fault is known");
  R* mine = ring + threadIdx.x + LINE_X * threadIdx.y;
  CD win[St::SW];
#pragma unroll
  for (int m = 0; m < St::SW - 1; ++m) {
    const int sp = s0 - St::HW + m;
    load_cell<R, S, DIR, ORDER, SCHEME, VISC, VO>(P, g, c, mbase + sp * stride, mbase + wrap(sp) * stride, win[m]);
    if constexpr (RING) ring_put<ORDER, SCHEME, VISC, VO>(mine + m * 256, win[m]);
  }
  int head = 0;  // ring slot of the window's first cell
  RC nxt;  // the raw values of the cell that enters the window next
  {
    const int sp = s0 - 1 + St::HW;
    fetch_cell<S, DIR, ORDER, SCHEME, VISC, VO>(P, g, mbase + sp * stride, mbase + wrap(sp) * stride, nxt);
  }
  R Fp[5];
  CellState<DIR, EP> cs;
  // Software pipeline: the values of the cell that enters the window at face
  // f+1 are loaded while face f is computed, so that one face's arithmetic covers
  // the memory latency of the next.  Windows held in registers through a viscous
  // face issue its transverse stencils, and the state of the cell that face f+1
  // completes, a whole face ahead.  With the ring the state of cell f,
  // which face f completes, and the next cell's stencils are issued between the
  // two halves of face f, so that those registers are free during the convective
  // half; Euler sweeps load the state of cell f at the top of the iteration.
  // The loads are issued on every iteration, the last one included (its
  // values are never used): a load behind a branch makes the compiler wait
  // for every outstanding memory operation, the residual stores of the
  // iteration included, at the loop's merge points.  On the last iteration
  // the cell entering the window is clamped to the array's last layer along
  // DIR, and cell f+1 = s_end is at most that layer as well; on the first, cell
  // f = s0 - 1 is at least layer 0.
  constexpr bool AHEAD = VISC && !RING;
  const int n_along = DIR == 1 ? g.ny : g.nz;
  for (int f = s0 - 1; f < s_end; ++f) {
    finish_cell<R, S, DIR, ORDER, SCHEME, VISC, VO>(g, c, nxt, win[St::SW - 1]);
    if constexpr (RING)
      ring_put<ORDER, SCHEME, VISC, VO>(mine + (head == 0 ? St::SW - 1 : head - 1) * 256, win[St::SW - 1]);
    const int sp = min(f + 1 + St::HW, n_along - 1);
    fetch_values<S, DIR, ORDER, SCHEME, VISC, VO>(P, mbase + sp * stride, mbase + wrap(sp) * stride, nxt);
    if constexpr (AHEAD) fetch_cross<S, DIR, VISC, VO>(P, g, mbase + sp * stride, nxt);
    const int q = (f - s0 + 1) * qstride;  // cell f, from the column pointers
    CellState<DIR, EP> ncs;
    if constexpr (AHEAD) fetch_state<DIR, EP>(Racc, sa, q + qstride, g.nx, ncs);
    if constexpr (!VISC) fetch_state<DIR, EP>(Racc, sa, q, g.nx, cs);
    R F[5];
    face_conv<R, DIR, ORDER, SCHEME, VISC, VO>(c, tvd, variant, win, F);
    if constexpr (RING) {
      OX_SPLIT_FENCE();
      fetch_state<DIR, EP>(Racc, sa, q, g.nx, cs);
      fetch_cross<S, DIR, VISC, VO>(P, g, mbase + sp * stride, nxt);
      CD vw[St::SW];
#pragma unroll
      for (int m = 0; m < St::SW; ++m) {
        vw[m] = win[m];
        ring_get<ORDER, SCHEME, VISC, VO>(mine + (head + m >= St::SW ? head + m - St::SW : head + m) * 256, vw[m]);
      }
      face_visc<R, DIR, ORDER, SCHEME, VISC, VO>(c, inv_d, vw, F);
      head = head + 1 == St::SW ? 0 : head + 1;
    } else {
      face_visc<R, DIR, ORDER, SCHEME, VISC, VO>(c, inv_d, win, F);
    }
    if (f >= s0) {
      const double *Ra = cs.R, *Qa = cs.A, *Qb = cs.B, *Qc = cs.C;
      double Rl[5];
#pragma unroll
      for (int l = 0; l < 5; ++l) Rl[l] = Ra[l] + cd * (-(double)Fp[l] + (double)F[l]);
      if constexpr (DIR == 1) {
#pragma unroll
        for (int l = 0; l < 5; ++l) G(Racc)[q + l * g.nx] = (S)Rl[l];
      } else {
        // stage epilogue (3D_solver/src/calc_steps.f90:60-69, :98-106, :137-145, :173-183)
        double Qn[5];
        if constexpr (EP == EP_RK3_S1) {
#pragma unroll
          for (int l = 0; l < 5; ++l) Qn[l] = Qa[l] - Rl[l];
        } else if constexpr (EP == EP_RK3_S23) {
#pragma unroll
          for (int l = 0; l < 5; ++l) Qn[l] = (sa.c1 * Qa[l] + sa.c2 * Qb[l] - Rl[l]) * sa.c4inv;
        } else if constexpr (EP == EP_RK4_S) {
#pragma unroll
          for (int l = 0; l < 5; ++l) {
            Qn[l] = Qa[l] - sa.c1 * Rl[l];
            G(sa.Rs)[q + l * g.nx] = Qc[l] + sa.c2 * Rl[l];
          }
        } else if constexpr (EP == EP_RK4_S4) {
#pragma unroll
          for (int l = 0; l < 5; ++l) {
            const double r = Qc[l] + Rl[l];
            Qn[l] = Qb[l] - r * sa.c1;  // c1 = one_sixth
            G(sa.Rs)[q + l * g.nx] = 0.0;
          }
        } else {
#pragma unroll
          for (int l = 0; l < 5; ++l) Qn[l] = Rl[l];
        }
#pragma unroll
        for (int l = 0; l < 5; ++l) G(sa.Qout)[q + l * g.nx] = Qn[l];
        if constexpr (EP != EP_RHS) {
          // primitives of the new state for the next stage (what k_prim
          // would compute from it), into the other primitive set, at the
          // cell and at every ghost cell that is its periodic image (the
          // ghost fill of set_bc_cyclic applied to the primitives)
          const PrimVals pv = prim_of(Qn[0], Qn[1], Qn[2], Qn[3], Qn[4], g.jac, c64);
          const int jj = t, kk = f;
          store_prim<S>(Pn, cidx(g, i, jj, kk), pv);
          const int ai = i < 2 * g.h ? i + g.ix : (i >= g.ix ? i - g.ix : -1);
          const int aj = jj < 2 * g.h ? jj + g.iy : (jj >= g.iy ? jj - g.iy : -1);
          const int ak = kk < 2 * g.h ? kk + g.iz : (kk >= g.iz ? kk - g.iz : -1);
          if (ai >= 0 || aj >= 0 || ak >= 0) {
            const int xs[2] = {i, ai}, ys[2] = {jj, aj}, zs[2] = {kk, ak};
            for (int c3 = 1; c3 < 8; ++c3) {
              const int x = xs[c3 & 1], y = ys[(c3 >> 1) & 1], z = zs[(c3 >> 2) & 1];
              if (x >= 0 && y >= 0 && z >= 0) store_prim<S>(Pn, cidx(g, x, y, z), pv);
            }
          }
        }
      }
    }
#pragma unroll
    for (int l = 0; l < 5; ++l) Fp[l] = F[l];
#pragma unroll
    for (int m = 0; m < St::SW - 1; ++m) win[m] = win[m + 1];
    if constexpr (AHEAD) cs = ncs;
  }
}

template <class R, class S, int ORDER, int SCHEME, int VISC, int VO, int DIR, int EP>
__global__ __launch_bounds__(256, line_waves<VISC>()) void k_sweep_line(SweepArgs<R, S> a) {
  __shared__ R ring[std::max(1, ring_values<R, ORDER, SCHEME, VISC, VO>())];
  const int gx = line_tiles(a.g, DIR);
  const int t = xcd_tile(blockIdx.x, gridDim.x, true);
  sweep_line_tile<R, S, ORDER, SCHEME, VISC, VO, DIR, EP>(a, t % gx, t / gx, ring);
}

template <class R, class S, int ORDER, int SCHEME, int VISC, int VO, int DIR, int EP>
__global__ __launch_bounds__(256, line_waves<VISC>()) void k_sweep_line_batch(
    const SweepArgs<R, S>* __restrict__ cases, const TileMap* __restrict__ map, int ncase, int ntiles) {
  __shared__ R ring[std::max(1, ring_values<R, ORDER, SCHEME, VISC, VO>())];
  const int t = xcd_tile(blockIdx.x, ntiles), ci = find_case(map, ncase, t);
  const int local = t - map[ci].start, nbx = map[ci].nbx;
  sweep_line_tile<R, S, ORDER, SCHEME, VISC, VO, DIR, EP>(cases[ci], local % nbx, local / nbx, ring);
}

// Batched SGS viscosity of LES cases over the tiles of several cases, reading
// each case's x-sweep descriptor: the primitive set the stage reads, the
// geometry and the constants.
template <class R, class S>
__global__ __launch_bounds__(256) void k_les_mut_batch(const SweepArgs<R, S>* __restrict__ cases,
                                                       const TileMap* __restrict__ map, int ncase, int ntiles) {
  __shared__ LesPlanes<R> pl;
  const int t = xcd_tile(blockIdx.x, ntiles), ci = find_case(map, ncase, t);
  const int local = t - map[ci].start, nbx = map[ci].nbx, nby = map[ci].nby;
  const SweepArgs<R, S>& a = cases[ci];
  les_mut_tile<S, R>(a.P, a.g, a.c, local % nbx, (local / nbx) % nby, local / (nbx * nby), pl);
}

}  // namespace ox

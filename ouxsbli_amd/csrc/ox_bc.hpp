// ox_bc.hpp -- ghost fills of non-periodic directions (OX_BC_EXTRAPOLATE,
// OX_BC_SLIP) for the state, the primitives and the Ducros sensor.
//
// The reference fills the ghost layers of the state after every RK stage
// with the case's set_bc (3D_solver/STZ/set.f90:77-138: slip walls mirror
// the state about the boundary face and negate the normal momentum,
// zero-gradient ends copy the adjacent interior cell), then recomputes the
// primitives of every cell.  Here the stage epilogue writes the primitives of
// interior cells, and the fills below write those of the ghost cells: a
// copied or mirrored state gives the same primitives bit for bit as the
// interior cell it came from (the normal velocity negated, an exact
// operation), so the primitives are filled directly.  set_bc fills x, then y,
// then z over the whole extent of the other two directions; the fills of different
// directions commute, so a ghost cell is the interior cell that the source
// indices of its three directions name, and one launch fills them all.
#pragma once

#include "ox_kernels.hpp"

namespace ox {

// Source index along one direction of extent h + m + h (h ghost layers, m
// interior cells) for index p, and whether the normal component changes sign.
__device__ __forceinline__ int bc_source(int kind, int p, int h, int m, bool& flip) {
  flip = false;
  if (p >= h && p < h + m) return p;
  if (kind == OX_BC_PERIODIC) return p < h ? p + m : p - m;
  if (kind == OX_BC_EXTRAPOLATE) return p < h ? h : h + m - 1;
  flip = true;  // OX_BC_SLIP: ghost h-1-n mirrors interior h+n
  return p < h ? 2 * h - 1 - p : 2 * (h + m) - 1 - p;
}

// Cell (i, j, k) of the 2h ghost layers of direction d for linear index t
// over (2h) x (extent of the other two directions); false past the end.
__device__ __forceinline__ bool bc_cell(const Geom& g, int d, long long t, int& i, int& j, int& k) {
  const int h = g.h;
  if (d == 0) {
    if (t >= 2LL * h * g.ny * g.nz) return false;
    const int s = (int)(t % (2 * h));
    const long long r = t / (2 * h);
    i = s < h ? s : g.nx - 2 * h + s;
    j = (int)(r % g.ny);
    k = (int)(r / g.ny);
  } else if (d == 1) {
    if (t >= 2LL * h * g.nx * g.nz) return false;
    i = (int)(t % g.nx);
    const long long r = t / g.nx;
    const int s = (int)(r % (2 * h));
    j = s < h ? s : g.ny - 2 * h + s;
    k = (int)(r / (2 * h));
  } else {
    if (t >= 2LL * h * g.nx * g.ny) return false;
    i = (int)(t % g.nx);
    const long long r = t / g.nx;
    j = (int)(r % g.ny);
    const int s = (int)(r / g.ny);
    k = s < h ? s : g.nz - 2 * h + s;
  }
  return true;
}

inline long long bc_cells(const Geom& g, int d) {
  return 2LL * g.h * (d == 0 ? (long long)g.ny * g.nz : d == 1 ? (long long)g.nx * g.nz : (long long)g.nx * g.ny);
}

// The interior cell that cell (i, j, k) copies or mirrors, and the signs.
struct BcSource {
  int m;
  bool fu, fv, fw;
};
__device__ __forceinline__ BcSource bc_interior(const Geom& g, int i, int j, int k) {
  BcSource s;
  const int si = bc_source(g.bc[0], i, g.h, g.ix, s.fu), sj = bc_source(g.bc[1], j, g.h, g.iy, s.fv);
  s.m = cidx(g, si, sj, bc_source(g.bc[2], k, g.h, g.iz, s.fw));
  return s;
}

// Cell t of the ghost layers next to the interior along the non-periodic
// direction d (1: y, 2: z) over the interior of the other two: the cells whose
// sensor the faces of interior cells read (calc_Ducros,
// 3D_solver/src/calc_hybrid.f90:11-72, computes it at every cell 2..n-1 from
// the filled primitives).  The x sweep forms the sensors of its own ghost
// cells from its row.
__device__ __forceinline__ bool sensor_cell(const Geom& g, int d, long long t, int& i, int& j, int& k) {
  if (t >= 2LL * g.ix * (d == 1 ? g.iz : g.iy)) return false;
  i = g.h + (int)(t % g.ix);
  const long long r = t / g.ix;
  const int side = (int)(r & 1);
  const int o = g.h + (int)(r >> 1);  // k for d 1, j for d 2
  j = d == 1 ? (side ? g.h + g.iy : g.h - 1) : o;
  k = d == 1 ? o : (side ? g.h + g.iz : g.h - 1);
  return true;
}
inline long long sensor_cells(const Geom& g, int d) { return 2LL * g.ix * (d == 1 ? g.iz : g.iy); }

// The sensor of cell (i, j, k) from its six neighbours' velocities: as they
// are (FILLED), or those that the ghost cells among them are being filled with.
template <class S, class R, bool FILLED>
__device__ __forceinline__ void bc_sensor(const Prim<S>& P, const Geom& g, int i, int j, int k) {
  R u[6], v[6], w[6];
#pragma unroll
  for (int n = 0; n < 6; ++n) {
    const int o = (n & 1) ? 1 : -1;
    const int ni = n < 2 ? i + o : i, nj = n / 2 == 1 ? j + o : j, nk = n > 3 ? k + o : k;
    BcSource s{cidx(g, ni, nj, nk), false, false, false};
    if constexpr (!FILLED) s = bc_interior(g, ni, nj, nk);
    u[n] = R(G(P.u)[s.m]); v[n] = R(G(P.v)[s.m]); w[n] = R(G(P.w)[s.m]);
    u[n] = s.fu ? -u[n] : u[n]; v[n] = s.fv ? -v[n] : v[n]; w[n] = s.fw ? -w[n] : w[n];
  }
  const R fd = ducros<R>(g, u[0], u[1], v[0], v[1], w[0], w[1], u[2], u[3], v[2], v[3], w[2], w[3], u[4], u[5], v[4],
                         v[5], w[4], w[5]);
  G(P.s)[cidx(g, i, j, k)] = (S)fd;
}

// The sensors of a primitive set whose ghost cells are filled.
template <class S, class R>
__global__ __launch_bounds__(256) void k_bc_sensor(Prim<S> P, Geom g, int d) {
  int i, j, k;
  if (sensor_cell(g, d, (long long)blockIdx.x * 256 + threadIdx.x, i, j, k)) bc_sensor<S, R, true>(P, g, i, j, k);
}

// The ghost primitives of all non-periodic directions and the sensors of their
// inner ghost layers, both from interior cells, in one launch: blocks 0 ..
// nb[0] - 1 take the x layers, then y, z, then the sensors along y and z.  Bound
// by the launch: five of them (three without a sensor), each waiting for the one
// before, took 12.4 us of a stage of a 4 x 4 x 256 tube, one takes 6.9 (100 steps 7.75
// -> 6.0 ms); 150 x 77 x 53 between walls with sensors 10 -> 7.2.
struct BcBlocks {
  unsigned nb[5];
};
template <class S, class R>
__global__ __launch_bounds__(256) void k_bc_fill(Prim<S> P, Geom g, BcBlocks b) {
  unsigned x = blockIdx.x;
  int d = 0;
  while (d < 4 && x >= b.nb[d]) x -= b.nb[d++];
  const long long t = (long long)x * 256 + threadIdx.x;
  int i, j, k;
  if (d > 2) {
    if (sensor_cell(g, d - 2, t, i, j, k)) bc_sensor<S, R, false>(P, g, i, j, k);
    return;
  }
  if (!bc_cell(g, d, t, i, j, k)) return;
  // a cell in the layers of several directions is the first one's
  if (d > 0 && g.bc[0] && (i < g.h || i >= g.h + g.ix)) return;
  if (d > 1 && g.bc[1] && (j < g.h || j >= g.h + g.iy)) return;
  const BcSource s = bc_interior(g, i, j, k);
  const int m = cidx(g, i, j, k);
  const S u = G(P.u)[s.m], v = G(P.v)[s.m], w = G(P.w)[s.m];
  G(P.rho)[m] = G(P.rho)[s.m];
  G(P.u)[m] = s.fu ? -u : u;
  G(P.v)[m] = s.fv ? -v : v;
  G(P.w)[m] = s.fw ? -w : w;
  G(P.p)[m] = G(P.p)[s.m];
}

inline bool any_bc(const Geom& g) { return g.bc[0] || g.bc[1] || g.bc[2]; }

// After a stage whose epilogue wrote the interior primitives of its new state
// and their images along periodic directions into Pn: the ghost primitives of
// the non-periodic directions and the sensors of their inner ghost layers.
template <class R, class S, int ORDER, int SCHEME>
void launch_bc_fill(const Geom& g, const Prim<S>& Pn, hipStream_t st) {
  auto blocks = [](long long n) { return (unsigned)((n + 255) / 256); };
  BcBlocks b{};
  for (int d = 0; d < 3; ++d)
    if (g.bc[d]) b.nb[d] = blocks(bc_cells(g, d));
  if constexpr (kUsesSensor<SCHEME, ORDER> && ORDER > 2) {
    for (int d = 1; d < 3; ++d)
      if (g.bc[d]) b.nb[2 + d] = blocks(sensor_cells(g, d));
  }
  unsigned n = 0;
  for (unsigned x : b.nb) n += x;
  if (n) k_bc_fill<S, R><<<n, 256, 0, st>>>(Pn, g, b);
}
// The sensors alone, of primitives whose ghost cells came with the state.
template <class R, class S, int ORDER, int SCHEME>
void launch_bc_sensors(const Geom& g, const Prim<S>& P, hipStream_t st) {
  if constexpr (kUsesSensor<SCHEME, ORDER> && ORDER > 2) {
    for (int d = 1; d < 3; ++d)
      if (g.bc[d]) k_bc_sensor<S, R><<<(unsigned)((sensor_cells(g, d) + 255) / 256), 256, 0, st>>>(P, g, d);
  }
}

}  // namespace ox

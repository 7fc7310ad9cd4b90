// sweep_bounds.cpp -- the kernels' bodies on the host, every array of its exact
// size and checked (-fsanitize=address): the y and z sweeps, the x sweep's runs and
// rows and the SGS viscosity, over ragged grids and segment lengths.  Lanes of a
// workgroup are coroutines that meet at its barriers and shuffles; the LDS arrays are
// heap arrays of their own, and hold NaN at first, so that a value that is read before
// it is written shows in the result.
// Build: g++ -std=c++17 -O0 -w -fsanitize=address,undefined -I/opt/rocm/include
//        -D__HIP_PLATFORM_AMD__ -x c++ sweep_bounds.cpp (an argument: fewer grids)
#include <hip/hip_runtime.h>
#include <ucontext.h>

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <limits>
#include <memory>
#include <type_traits>
#include <vector>

// ---------------------------------------------------------------------------
// A workgroup: lanes run one after another, each up to its next meeting point.
// ---------------------------------------------------------------------------
using std::max;
using std::min;
static uint3 blockIdx, threadIdx;
static dim3 gridDim, blockDim;

struct Workgroup {
  static constexpr size_t STACK = 1 << 18;
  static constexpr int MAX = 512;
  std::vector<std::unique_ptr<char[]>> stacks;
  ucontext_t home, ctx[MAX];
  bool over[MAX];
  int met[MAX];        // meeting points a lane has reached
  double passed[MAX];  // shuffled values
  int lane = 0, lanes = 0;
  std::function<void()> body;

  static Workgroup& get() {
    static Workgroup w;
    return w;
  }
  static void entry() {
    Workgroup& w = get();
    w.body();
    w.over[w.lane] = true;
    swapcontext(&w.ctx[w.lane], &w.home);
  }
  void meet() {
    ++met[lane];
    swapcontext(&ctx[lane], &home);
  }
  void run(int bx, int by, std::function<void()> f) {
    lanes = bx * by;
    body = std::move(f);
    while ((int)stacks.size() < lanes) stacks.emplace_back(new char[STACK]);
    for (int l = 0; l < lanes; ++l) {
      over[l] = false;
      met[l] = 0;
      getcontext(&ctx[l]);
      ctx[l].uc_stack.ss_sp = stacks[l].get();
      ctx[l].uc_stack.ss_size = STACK;
      ctx[l].uc_link = nullptr;
      makecontext(&ctx[l], entry, 0);
    }
    for (bool any = true; any;) {
      any = false;
      for (lane = 0; lane < lanes; ++lane) {
        if (over[lane]) continue;
        threadIdx.x = lane % bx;
        threadIdx.y = lane / bx;
        swapcontext(&home, &ctx[lane]);
        any = any || !over[lane];
      }
      // lanes that are still under way have met the same number of times
      int m = -1;
      for (int l = 0; l < lanes; ++l)
        if (!over[l]) {
          if (m >= 0 && met[l] != m) std::printf("lanes of a workgroup part at a barrier\n"), std::exit(1);
          m = met[l];
        }
    }
  }
};
static void __syncthreads() { Workgroup::get().meet(); }
static double __shfl_down(double v, int d, int width) {
  Workgroup& w = Workgroup::get();
  const int me = w.lane;
  w.passed[me] = v;
  w.meet();
  const double r = me % width + d < width ? w.passed[me + d] : v;
  w.meet();
  return r;
}
static double __shfl(double v, int src, int width) {
  Workgroup& w = Workgroup::get();
  const int me = w.lane;
  w.passed[me] = v;
  w.meet();
  const double r = w.passed[me / width * width + src];
  w.meet();
  return r;
}

#undef __launch_bounds__
#define __launch_bounds__(...)
#undef __shared__
#define __shared__ static
#include "ox_kernels.hpp"

using namespace ox;

static int g_bad = 0, g_runs = 0;

// An array of exactly n values on the heap.
template <class T> struct Arr {
  std::unique_ptr<T[]> p;
  size_t n;
  explicit Arr(size_t n, T v = T(0)) : p(new T[n]), n(n) {
    for (size_t k = 0; k < n; ++k) p[k] = v;
  }
};

template <class S> struct PrimSet {
  std::vector<Arr<S>> a;
  explicit PrimSet(size_t cells) {
    for (int m = 0; m < kPrimArrays; ++m) a.emplace_back(cells);
  }
  Prim<S> get(bool les) {
    return {a[0].p.get(), a[1].p.get(), a[2].p.get(), a[3].p.get(), a[4].p.get(), a[5].p.get(),
            les ? a[6].p.get() : nullptr, les ? a[7].p.get() : nullptr};
  }
};

struct Case {
  ox_config cfg{};
  Geom g{};
  HostConsts hc{};
  Case(int order, int scheme, int visc, int ix, int iy, int iz, int bx = 0, int by = 0, int bz = 0) {
    const int h = order / 2;
    cfg.order = order; cfg.scheme = scheme; cfg.visc = visc;
    cfg.nx = ix + 2 * h; cfg.ny = iy + 2 * h; cfg.nz = iz + 2 * h;
    cfg.gamma = 1.4; cfg.R = 287.03; cfg.Pr = 0.71; cfg.Prt = 0.9; cfg.threshold = 0.4;
    cfg.Lx = cfg.Ly = cfg.Lz = 1.0;
    cfg.dt = 1e-6;
    hc.init(cfg);
    hc.les_delta15 = 1e-3;
    g.nx = cfg.nx; g.ny = cfg.ny; g.nz = cfg.nz; g.h = h;
    g.ix = ix; g.iy = iy; g.iz = iz;
    g.jac = 1.0;
    g.inv_dx = ix; g.inv_dy = iy; g.inv_dz = iz;
    g.a_xy = g.a_yz = g.a_zx = 1e-6;
    g.bc[0] = bx; g.bc[1] = by; g.bc[2] = bz;
  }
  size_t cells() const { return (size_t)g.nx * g.ny * g.nz; }
};

static double noise() { return 0.1 * (std::rand() / (double)RAND_MAX - 0.5); }

// The arrays of one case, filled as a stage finds them.
template <class R, class S> struct Arrays {
  PrimSet<S> P, Pn;
  Arr<S> Racc;
  Arr<double> Qin, Qout, Rs;
  SweepArgs<R, S> a{};
  Arrays(const Case& c, int ep)
      : P(c.cells()), Pn(c.cells()), Racc(5 * c.cells()), Qin(5 * c.cells()), Qout(5 * c.cells()),
        Rs(ep == EP_RK4_S || ep == EP_RK4_S4 ? 5 * c.cells() : 0) {
    for (size_t m = 0; m < c.cells(); ++m) {
      P.a[0].p[m] = S(1.2 + noise());
      for (int k = 1; k < 4; ++k) P.a[k].p[m] = S(100.0 * noise());
      P.a[4].p[m] = S(1e5 * (1.0 + noise()));
      P.a[5].p[m] = S(0.5);
      P.a[6].p[m] = P.a[7].p[m] = S(1e-5);
    }
    for (size_t k = 0; k < 5 * c.cells(); ++k) Qin.p[k] = Qout.p[k] = 1.0;
    for (int k = 0; k < c.g.nz * c.g.ny; ++k)
      for (int i = 0; i < c.g.nx; ++i) Qin.p[i + (size_t)c.g.nx * (4 + 5 * k)] = Qout.p[i + (size_t)c.g.nx * (4 + 5 * k)] = 2.5e5;
    const bool les = c.cfg.visc == OX_VISC_LES;
    a.P = P.get(les);
    a.Pn = Pn.get(les);
    a.Racc = Racc.p.get();
    a.g = c.g;
    a.c = make_physc<R>(c.hc);
    a.c64 = make_physc<double>(c.hc);
    a.sa = {Qin.p.get(), Qout.p.get(), Rs.n ? Rs.p.get() : nullptr, 0.75, 0.25, 1.0, ep};
    a.cd = 1e-6;
    a.tvd = OX_TVD_HYBRID;
    a.variant = 1;
    xrun_shape(c.g, a.xrows, a.xwgs);
  }
  // every interior value of the residual (or the new state) is a number
  void check(const Case& c, bool state, const char* what) {
    ++g_runs;
    const Geom& g = c.g;
    long long bad = 0;
    for (int k = g.h; k < g.h + g.iz; ++k)
      for (int j = g.h; j < g.h + g.iy; ++j)
        for (int l = 0; l < 5; ++l)
          for (int i = g.h; i < g.h + g.ix; ++i) {
            const size_t q = i + (size_t)g.nx * (l + 5 * (j + (size_t)g.ny * k));
            if (!std::isfinite(state ? Qout.p[q] : (double)Racc.p[q])) ++bad;
          }
    if (bad) {
      std::printf("%s order %d scheme %d visc %d grid %d x %d x %d: %lld values are no numbers\n", what, c.cfg.order,
                  c.cfg.scheme, c.cfg.visc, g.ix, g.iy, g.iz, bad);
      ++g_bad;
    }
  }
};

template <class R, class S, int ORDER, int SCHEME, int VISC, int VO, int DIR, int EP>
void line(const Case& c, int lseg) {
  Arrays<R, S> A(c, EP);
  A.a.lseg = lseg;
  const int gx = line_tiles(c.g, DIR), nd = DIR == 1 ? c.g.iy : c.g.iz, nb = gx * ((nd + lseg - 1) / lseg);
  for (int t = 0; t < nb; ++t) {
    Arr<R> ring(std::max(1, ring_values<R, ORDER, SCHEME, VISC, VO>()), std::numeric_limits<R>::quiet_NaN());
    for (int y = 0; y < LINE_Y; ++y)  // (no lane waits for another)
      for (int x = 0; x < LINE_X; ++x) {
        threadIdx.x = x;
        threadIdx.y = y;
        sweep_line_tile<R, S, ORDER, SCHEME, VISC, VO, DIR, EP>(A.a, t % gx, t / gx, ring.p.get());
      }
  }
  A.check(c, DIR == 2, DIR == 1 ? "y sweep" : "z sweep");
}

template <class R, class S, int ORDER, int SCHEME, int VISC, int VO> void lines(const Case& c, int lseg) {
  line<R, S, ORDER, SCHEME, VISC, VO, 1, EP_RHS>(c, lseg);
  line<R, S, ORDER, SCHEME, VISC, VO, 2, EP_RK3_S1>(c, lseg);
  line<R, S, ORDER, SCHEME, VISC, VO, 2, EP_RK3_S23>(c, lseg);
  line<R, S, ORDER, SCHEME, VISC, VO, 2, EP_RK4_S>(c, lseg);
  line<R, S, ORDER, SCHEME, VISC, VO, 2, EP_RK4_S4>(c, lseg);
  line<R, S, ORDER, SCHEME, VISC, VO, 2, EP_RHS>(c, lseg);
}

// A block of LDS of type T, of its exact size and full of NaN.
template <class T, class R> std::unique_ptr<T> lds_block() {
  std::unique_ptr<T> p(new T);
  R* v = reinterpret_cast<R*>(p.get());
  for (size_t k = 0; k < sizeof(T) / sizeof(R); ++k) v[k] = std::numeric_limits<R>::quiet_NaN();
  return p;
}

template <class R, class S, int ORDER, int SCHEME, int VISC, int VO> void xruns(const Case& c) {
  Arrays<R, S> A(c, EP_RHS);
  const long long nb = xrun_blocks(c.g);
  for (int t = 0; t < nb; ++t) {
    auto lds = lds_block<XRunTile<R, ORDER, SCHEME, VISC, VO>, R>();
    Workgroup::get().run(256, 1, [&] { sweep_x_run<R, S, ORDER, SCHEME, VISC, VO>(A.a, t, *lds); });
  }
  A.check(c, false, "x runs");
}

template <class R, class S> void les(const Case& c) {
  Arrays<R, S> A(c, EP_RHS);
  for (size_t m = 0; m < c.cells(); ++m) A.P.a[6].p[m] = A.P.a[7].p[m] = std::numeric_limits<S>::quiet_NaN();
  int bx, by, bz;
  les_tiles(c.g, bx, by, bz);
  for (int t = 0; t < bx * by * bz; ++t) {
    struct Planes { LesPlanes<R> v; };
    auto lds = lds_block<Planes, R>();
    Workgroup::get().run(256, 1,
                         [&] { les_mut_tile<S, R>(A.a.P, c.g, A.a.c, t % bx, (t / bx) % by, t / (bx * by), lds->v); });
  }
  ++g_runs;
  // every cell has its viscosity, the outermost layer the copy of the opposite end's
  long long bad = 0;
  auto src = [](int i, int n) { return i == 0 ? n - 2 : i == n - 1 ? 1 : i; };
  for (int k = 0; k < c.g.nz; ++k)
    for (int j = 0; j < c.g.ny; ++j)
      for (int i = 0; i < c.g.nx; ++i)
        for (int f = 6; f < 8; ++f) {
          const S v = A.P.a[f].p[cidx(c.g, i, j, k)];
          const S w = A.P.a[f].p[cidx(c.g, src(i, c.g.nx), src(j, c.g.ny), src(k, c.g.nz))];
          if (!std::isfinite((double)v) || v != w) ++bad;
        }
  if (bad) std::printf("SGS viscosity %d x %d x %d: %lld cells are wrong\n", c.g.ix, c.g.iy, c.g.iz, bad), ++g_bad;
}

template <class R, class S, int ORDER, int SCHEME, int VISC, int VO> void xrows(const Case& c) {
  Arrays<R, S> A(c, EP_RHS);
  const int nb = (c.g.iy + XROW_BAND - 1) / XROW_BAND * c.g.iz * (XROW_BAND / (256 / c.g.ix));
  gridDim = dim3(nb);
  for (int t = 0; t < nb; ++t) {
    blockIdx.x = t;
    Workgroup::get().run(256, 1, [&] { k_sweep_xrow<R, S, ORDER, SCHEME, VISC, VO>(A.a); });
  }
  A.check(c, false, "x rows");
}

template <class R, class S> void all(bool quick) {
  struct N { int x, y, z; };
  // widths around a workgroup's 64 cells and 253 faces, rows around groups of four,
  // and segments that divide the line, leave one cell, leave all but one, or are longer
  for (N n : quick ? std::vector<N>{{65, 13, 14}} : std::vector<N>{{12, 12, 12}, {63, 13, 14}, {65, 17, 15}}) {
    for (int lseg : quick ? std::vector<int>{5} : std::vector<int>{1, 4, 11, 64}) {
      lines<R, S, 6, SLAU, 1, 6>(Case(6, SLAU, 1, n.x, n.y, n.z), lseg);
      lines<R, S, 4, KEEP, 1, 4>(Case(4, KEEP, 1, n.x, n.y, n.z), lseg);
      lines<R, S, 6, HYBRID, 1, 5>(Case(6, HYBRID, 1, n.x, n.y, n.z, 0, OX_BC_SLIP, OX_BC_EXTRAPOLATE), lseg);
      lines<R, S, 6, SLAU, 1, 4>(Case(6, SLAU, 1, n.x, n.y, n.z, OX_BC_SLIP, OX_BC_SLIP, OX_BC_SLIP), lseg);
      lines<R, S, 6, HYBRID, 2, 6>(Case(6, HYBRID, 2, n.x, n.y, n.z), lseg);
      lines<R, S, 2, HYBRID, 0, 0>(Case(2, HYBRID, 0, n.x, n.y, n.z), lseg);
      lines<R, S, 6, SLAU, 0, 0>(Case(6, SLAU, 0, n.x, n.y, n.z), lseg);
    }
  }
  for (N n : quick ? std::vector<N>{{12, 40, 4}, {126, 9, 4}} : std::vector<N>{{12, 40, 4}, {62, 33, 4}, {126, 9, 4}, {252, 5, 4}, {254, 9, 4}, {505, 4, 4}}) {
    const N m{n.x, std::max(n.y, 12), 12};
    xruns<R, S, 6, SLAU, 1, 6>(Case(6, SLAU, 1, m.x, m.y, m.z));
    xruns<R, S, 6, HYBRID, 2, 6>(Case(6, HYBRID, 2, m.x, m.y, m.z, 0, 0, 0));
    xruns<R, S, 2, SLAU, 0, 0>(Case(2, SLAU, 0, std::max(4, n.x - 8), n.y, n.z, OX_BC_SLIP, 0, 0));
    xruns<R, S, 2, HYBRID, 0, 0>(Case(2, HYBRID, 0, n.x, n.y, n.z));
    xruns<R, S, 4, KEEP, 0, 0>(Case(4, KEEP, 0, n.x, std::max(n.y, 8), 8));
  }
  for (N n : quick ? std::vector<N>{{29, 13, 13}} : std::vector<N>{{28, 12, 12}, {29, 13, 13}, {31, 14, 14}, {13, 30, 15}})
    les<R, S>(Case(6, HYBRID, 2, n.x, n.y, n.z));
  for (int w : quick ? std::vector<int>{128} : std::vector<int>{64, 128, 256}) {
    xrows<R, S, 6, SLAU, 1, 6>(Case(6, SLAU, 1, w, 17, 12));
    xrows<R, S, 4, KEEP, 1, 4>(Case(4, KEEP, 1, w, 17, 8));
    xrows<R, S, 2, SLAU, 0, 0>(Case(2, SLAU, 0, w, 15, 4));
  }
}

int main(int argc, char** argv) {
  all<double, double>(argc > 1);
  all<float, float>(true);
  std::printf("%d runs, bad=%d\n", g_runs, g_bad);
  return g_bad ? 1 : 0;
}

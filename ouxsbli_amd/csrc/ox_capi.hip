// ox_capi.hip -- the C ABI of include/ouxsbli.h: handle lifecycle, state
// transfer, the RK driver, diagnostics.
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdio>
#include <cstring>
#include <mutex>
#include <new>
#include <string>
#include <vector>

#include "ox_bc.hpp"
#include "ox_core.hpp"
#include "ox_diag.hpp"
#include "ox_kernels.hpp"
#include "ox_solver.hpp"

namespace ox {

// The state's ghost layers of a non-periodic direction d (the case's set_bc,
// 3D_solver/STZ/set.f90:77-138, at the end of a step).
__global__ __launch_bounds__(256) void k_bc_state(double* __restrict__ Q, Geom g, int d) {
  int i, j, k;
  if (!bc_cell(g, d, (long long)blockIdx.x * 256 + threadIdx.x, i, j, k)) return;
  bool flip;
  int si = i, sj = j, sk = k;
  if (d == 0) si = bc_source(g.bc[0], i, g.h, g.ix, flip);
  else if (d == 1) sj = bc_source(g.bc[1], j, g.h, g.iy, flip);
  else sk = bc_source(g.bc[2], k, g.h, g.iz, flip);
#pragma unroll
  for (int l = 0; l < 5; ++l) {
    const double v = Q[qidx(g, si, l, sj, sk)];
    Q[qidx(g, i, l, j, k)] = (flip && l == 1 + d) ? -v : v;
  }
}

// ---------------------------------------------------------------------------
// Periodic ghost fill: every ghost cell takes its periodic image (the net
// effect of set_bc_cyclic{2,4,6}, 3D_solver/src/set_bc_common.f90:101-273).
// Sources are interior cells only, so one pass has no ordering hazard.
// Thread mapping: linear index over the ghost shell:
//   [0, A)        z slabs  (2h planes of nx*ny)
//   [A, A+B)      y slabs  (iz rows-planes of 2h*nx)
//   [A+B, A+B+C)  x slabs  (iz*iy rows of 2h)
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_ghost_fill(double* __restrict__ Q, Geom g) {
  const long long t = (long long)blockIdx.x * 256 + threadIdx.x;
  const int h = g.h, nx = g.nx, ny = g.ny;
  const long long A = 2LL * h * nx * ny;
  const long long B = (long long)g.iz * 2 * h * nx;
  const long long C = (long long)g.iz * g.iy * 2 * h;
  int i, j, k;
  if (t < A) {
    const int pl = (int)(t / ((long long)nx * ny));
    const int r = (int)(t % ((long long)nx * ny));
    i = r % nx;
    j = r / nx;
    k = pl < h ? pl : g.nz - 2 * h + pl;
  } else if (t < A + B) {
    const long long u = t - A;
    const int row = (int)(u / nx);
    i = (int)(u % nx);
    k = h + row / (2 * h);
    const int s = row % (2 * h);
    j = s < h ? s : g.ny - 2 * h + s;
  } else if (t < A + B + C) {
    const long long u = t - A - B;
    const int s = (int)(u % (2 * h));
    const long long row = u / (2 * h);
    j = h + (int)(row % g.iy);
    k = h + (int)(row / g.iy);
    i = s < h ? s : nx - 2 * h + s;
  } else {
    return;
  }
  // periodic image inside the interior [h, h+n)
  const int si = i < h ? i + g.ix : (i >= h + g.ix ? i - g.ix : i);
  const int sj = j < h ? j + g.iy : (j >= h + g.iy ? j - g.iy : j);
  const int sk = k < h ? k + g.iz : (k >= h + g.iz ? k - g.iz : k);
#pragma unroll
  for (int l = 0; l < 5; ++l) Q[qidx(g, i, l, j, k)] = Q[qidx(g, si, l, sj, sk)];
}

// QJ = Q / J (pre_calc, 3D_solver/src/preprocess.f90.fypp:65-71) and back.
__global__ __launch_bounds__(256) void k_scale(double* __restrict__ Q, long long n, double J, int divide) {
  const long long t = (long long)blockIdx.x * 256 + threadIdx.x;
  if (t >= n) return;
  Q[t] = divide ? Q[t] / J : J * Q[t];
}

// dst = J * src (the physical state of ox_get_state, written to scratch).
__global__ __launch_bounds__(256) void k_scale_to(const double* __restrict__ src, double* __restrict__ dst, long long n,
                                                  double J) {
  const long long t = (long long)blockIdx.x * 256 + threadIdx.x;
  if (t >= n) return;
  dst[t] = J * src[t];
}

}  // namespace ox

namespace {
thread_local std::string g_err;
}  // namespace

// ---------------------------------------------------------------------------
// Allocation-free diagnostics (ox_diagnostics_noalloc).  The per-block
// partials of k_diag and the merged result live in one file-scope device
// array instead of the handle's scratch buffer, and the final merge over the
// partials runs on the device, so a call makes no device or host allocation.
// Each GPU holds its own copy of the array (`noalloc_scratch`, 352 KiB) until
// the process ends; its device address is looked up once per device.
// ---------------------------------------------------------------------------
namespace {
constexpr int kNoAllocMaxBlocks = 4096;  // k_diag never launches more (the same cap as ox_diagnostics)
constexpr int kDiagStride = 2 * ox::DIAG_NQ + 1;
constexpr size_t kNoAllocDoubles = (size_t)kNoAllocMaxBlocks * kDiagStride + 8;
static __device__ __align__(256) double noalloc_scratch[kNoAllocDoubles];
constexpr int kMaxDevices = 64;
std::mutex g_noalloc_mu;
double* g_noalloc_ptr[kMaxDevices] = {};

// Device address of this device's noalloc_scratch (the device must be
// current).  Host code uses only this address, never the array's name.
int noalloc_scratch_ptr(int dev, double** out) {
  if (dev < 0 || dev >= kMaxDevices) return ox_fail(OX_EINVAL, "device ordinal out of range for the static scratch");
  std::lock_guard<std::mutex> lk(g_noalloc_mu);
  if (!g_noalloc_ptr[dev]) {
    void* p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(noalloc_scratch));
    if (e != hipSuccess || !p)
      return ox_fail(OX_EDEVICE, std::string("hipGetSymbolAddress(noalloc_scratch): ") + hipGetErrorString(e));
    g_noalloc_ptr[dev] = static_cast<double*>(p);
  }
  *out = g_noalloc_ptr[dev];
  return OX_OK;
}
}  // namespace

namespace ox {
// Merges the k_diag partials of nb blocks in block order, one thread per
// quantity (and one for the wave speed), with exactly the operations of the
// host merge in ox_diagnostics, into out[0..DIAG_NQ] (sums) and
// out[DIAG_NQ] (max wave speed).
__global__ void k_diag_merge(const double* __restrict__ part, int nb, double* __restrict__ out) {
  const int q = threadIdx.x;
  if (q < DIAG_NQ) {
    double sum = 0.0, comp = 0.0;
    for (int b = 0; b < nb; ++b) {
      const double* p = part + (size_t)b * (2 * DIAG_NQ + 1);
      const double x = p[2 * q];
      const double t = sum + x;
      if (__builtin_fabs(sum) >= __builtin_fabs(x)) comp += (sum - t) + x;
      else comp += (x - t) + sum;
      sum = t;
      comp += p[2 * q + 1];
    }
    out[q] = sum + comp;
  } else if (q == DIAG_NQ) {
    double wmax = 0.0;
    for (int b = 0; b < nb; ++b) wmax = nan_max(wmax, part[(size_t)b * (2 * DIAG_NQ + 1) + 2 * DIAG_NQ]);
    out[DIAG_NQ] = wmax;
  }
}
}  // namespace ox

int ox_fail(int code, const std::string& msg) {
  g_err = msg;
  // HIP keeps an error until it is asked for: one that is reported here must not
  // come back from the launch check of a later call, which may be on another,
  // healthy handle (a result that cannot be page-locked is an ordinary array, and
  // an admission that runs out of memory is tried again)
  if (code == OX_EDEVICE || code == OX_ENOMEM) (void)hipGetLastError();
  return code;
}

void prof_record(ox::Core* C, const char* name) {
  ProfState* P = static_cast<ProfState*>(C->prof_state);
  if (P->used == P->pool.size()) {
    hipEvent_t e;
    if (hipEventCreate(&e) != hipSuccess) return;
    P->pool.push_back(e);
    P->names.push_back(nullptr);
  }
  hipEventRecord(P->pool[P->used], C->stream);
  P->names[P->used] = name;
  ++P->used;
}

// Stage `st` (0-based) of one RK step: its source state, epilogue and the
// factor on dt * face area (calc_time_dev.f90.fypp:86-100, :268-285).
void rk_stage(ox_solver* s, int st, const double** Qsrc, ox::StageArgs* sa, double* coef) {
  const ox::Core& C = s->C;
  if (C.cfg.rk == 3) {
    if (st == 0) {
      *sa = {s->QJ, s->QJ2, s->Rs, 0, 0, 0, ox::EP_RK3_S1};
      *Qsrc = s->QJ;
      *coef = 1.0;
    } else if (st == 1) {
      *sa = {s->QJ, s->QJ2, s->Rs, 0.75, 0.25, 1.0, ox::EP_RK3_S23};
      *Qsrc = s->QJ2;
      *coef = 0.25;
    } else {
      *sa = {s->QJ2, s->QJ, s->Rs, 2.0, 1.0, C.hc.one_third, ox::EP_RK3_S23};
      *Qsrc = s->QJ2;
      *coef = 2.0;
    }
  } else {
    static const double w[3][2] = {{0.5, 1.0}, {0.5, 2.0}, {1.0, 2.0}};
    if (st < 3) *sa = {s->QJ, s->QJ2, s->Rs, w[st][0], w[st][1], 0, ox::EP_RK4_S};
    else *sa = {s->QJ, s->QJ, s->Rs, C.hc.one_sixth, 0, 0, ox::EP_RK4_S4};
    *Qsrc = st == 0 ? s->QJ : s->QJ2;
    *coef = 1.0;
  }
}

namespace {

// Where the arrays of a handle lie in its one allocation, each from a multiple of
// 256 bytes on.
struct Layout {
  size_t qj, qj2, racc, rs, prim[2][ox::kPrimArrays], scratch;
  int nprim;
  size_t cleared;  // everything before the reduction partials starts as zero
  size_t scratch_bytes, bytes;

  explicit Layout(const ox_config& c) {
    const size_t nc = (size_t)c.nx * c.ny * c.nz, ns = 5 * nc;
    const size_t pe = c.precision == OX_PREC_FP64 ? sizeof(double) : sizeof(float);
    bytes = 0;
    qj = place(ns * sizeof(double));
    qj2 = place(ns * sizeof(double));
    racc = place(ns * pe);
    rs = place(c.rk == 4 ? ns * sizeof(double) : 0);
    // rho,u,v,w,p,sensor (+mut,qc2 for LES); the sweeps form T and mu
    nprim = c.visc == OX_VISC_LES ? 8 : 6;
    for (int set = 0; set < 2; ++set)
      for (int m = 0; m < nprim; ++m) prim[set][m] = place(nc * pe);
    cleared = bytes;
    scratch_bytes = 4096 * (2 * ox::DIAG_NQ + 1) * sizeof(double);
    scratch = place(scratch_bytes);
  }

 private:
  size_t place(size_t n) {
    const size_t at = bytes;
    bytes += (n + 255) & ~(size_t)255;
    return at;
  }
};

}  // namespace

size_t solver_footprint(const ox_config& c) { return Layout(c).bytes; }

namespace {

int validate(const ox_config& c) {
  if (c.abi_version != OX_ABI_VERSION) return ox_fail(OX_EINVAL, "abi_version mismatch");
  if (c.order != 2 && c.order != 4 && c.order != 6) return ox_fail(OX_EINVAL, "order must be 2, 4 or 6");
  if (c.rk != 3 && c.rk != 4) return ox_fail(OX_EINVAL, "rk must be 3 or 4");
  for (int b : {c.bc_x, c.bc_y, c.bc_z})
    if (b != OX_BC_PERIODIC && b != OX_BC_EXTRAPOLATE && b != OX_BC_SLIP) return ox_fail(OX_EINVAL, "unknown boundary kind");
  if ((c.bc_x || c.bc_y || c.bc_z) && (c.visc == OX_VISC_LES || c.scheme == OX_SCHEME_ROE))
    // an LES case's ghost fill of nu_t and qc2 next to walls is its own
    // set_bc_mut (3D_solver/TBL/set.f90:142-185), not built; the reference's
    // non-periodic Roe kernels compare the half-order io (0..2) with 4 and 6,
    // so they are first order on every face, and take an id_accuracy argument
    // their call site does not pass (3D_solver/src/calc_roe_kernel.f90.fypp:
    // 31-92, calc_flux_base.f90.fypp:60): that path does not build
    return ox_fail(OX_EUNSUPPORTED, "non-periodic boundaries are built for Euler and NS with KEEP, SLAU and Hybrid");
  if (c.visc_stencil != OX_STENCIL_CENTRAL && c.visc_stencil != OX_STENCIL_ME4BASE)
    return ox_fail(OX_EINVAL, "unknown viscous stencil");
  if (c.scheme < OX_SCHEME_KEEP || c.scheme > OX_SCHEME_HYBRID) return ox_fail(OX_EINVAL, "unknown scheme");
  if (c.tvd < 0 || c.tvd > 2) return ox_fail(OX_EINVAL, "tvd must be 0, 1 or 2");
  if (c.slau_variant < 0 || c.slau_variant > 1) return ox_fail(OX_EINVAL, "slau_variant must be 0 or 1");
  if (c.precision != OX_PREC_FP64 && c.precision != OX_PREC_FP32_BULK) return ox_fail(OX_EINVAL, "bad precision");
  const int h = c.order / 2;
  if (c.nx < 2 * h + 2 * c.order || c.ny < 2 * h + 2 * c.order || c.nz < 2 * h + 2 * c.order)
    return ox_fail(OX_EINVAL, "grid too small for the stencil");
  // cell indices are 32-bit (state indices, five values per cell, 64-bit)
  if ((double)c.nx * c.ny * c.nz >= 2147483647.0) return ox_fail(OX_EINVAL, "grid over 2^31 cells");
  // the z sweep's 32-bit state offsets span at least three xy planes
  if (15.0 * c.nx * c.ny >= 2147483647.0) return ox_fail(OX_EINVAL, "xy plane over 2^31 / 15 cells");
  if (c.nz > 65535 || c.ny > 65535 * 4) return ox_fail(OX_EINVAL, "grid extent exceeds launch limits");
  if (!(c.dt > 0.0) || !(c.Lx > 0.0) || !(c.Ly > 0.0) || !(c.Lz > 0.0) || !(c.gamma > 1.0) || !(c.R > 0.0))
    return ox_fail(OX_EINVAL, "non-positive dt, box length, gamma-1 or R");
  return OX_OK;
}

// set_grid_cyclic / set_Jacobian_xy3 / pre_calc metric scalars for a uniform
// periodic grid (src/set_coordinate.f90:99-339, preprocess.f90.fypp:72-87).
ox::Geom make_geom(const ox_config& c) {
  ox::Geom g;
  g.nx = c.nx; g.ny = c.ny; g.nz = c.nz;
  g.h = c.order / 2;
  g.ix = c.nx - 2 * g.h; g.iy = c.ny - 2 * g.h; g.iz = c.nz - 2 * g.h;
  const double dx = c.Lx / (double)(c.nx - c.order);
  const double dy = c.Ly / (double)(c.ny - c.order);
  const double dz = c.Lz / (double)(c.nz - c.order);
  g.jac = 8.0 / ((dx + dx) * (dy + dy) * 2.0 * dz);
  g.inv_dx = 1.0 / dx;
  g.inv_dy = 1.0 / dy;
  g.inv_dz = 1.0 / dz;
  g.a_xy = 0.25 * c.dt * (dx + dx) * (dy + dy);
  g.a_yz = 0.25 * c.dt * (dy + dy) * (dz + dz);
  g.a_zx = 0.25 * c.dt * (dz + dz) * (dx + dx);
  g.bc[0] = c.bc_x;
  g.bc[1] = c.bc_y;
  g.bc[2] = c.bc_z;
  return g;
}

void destroy(ox_solver* s) {
  if (!s) return;
  hipFree(s->slab);
  for (hipEvent_t e : s->prof.pool) hipEventDestroy(e);
  if (s->ev0) hipEventDestroy(s->ev0);
  if (s->ev1) hipEventDestroy(s->ev1);
  if (s->own_stream) hipStreamDestroy(s->own_stream);
  delete s;
}

int run_rk_step(ox_solver* s) {
  ox::Core& C = s->C;
  const ox::Geom& g = C.g;
  for (int st = 0; st < C.cfg.rk; ++st) {
    const double* Qsrc;
    ox::StageArgs sa;
    double coef;
    rk_stage(s, st, &Qsrc, &sa, &coef);
    s->stage(C, Qsrc, sa, coef * g.a_yz, coef * g.a_zx, coef * g.a_xy);
  }
  return OX_OK;
}

}  // namespace

namespace ox {
int device_cus() {
  int dev = 0, cus = 0;
  if (hipGetDevice(&dev) != hipSuccess ||
      hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
    cus = 256;
  return std::max(cus, 1);
}

void solo_segments(const Geom& g, const BatchOps& ops, int* lseg) {
  for (int d = 1; d <= 2; ++d) {
    const LineWork w = line_work(g, d);
    lseg[d - 1] = clamp_lseg(g, d, even_lseg(w.cells, pick_lseg(&w, 1, ops.line_occ(d), device_cus())));
  }
}

void launch_ghost_fill(Core& C, double* Q) {
  const Geom& g = C.g;
  const long long total = 2LL * g.h * g.nx * g.ny + (long long)g.iz * 2 * g.h * g.nx + (long long)g.iz * g.iy * 2 * g.h;
  k_ghost_fill<<<(unsigned)((total + 255) / 256), 256, 0, C.stream>>>(Q, g);
  // non-periodic directions: the case's ghost fill overwrites those layers
  // (including the periodic images just written there)
  for (int d = 0; d < 3; ++d)
    if (g.bc[d]) k_bc_state<<<(unsigned)((bc_cells(g, d) + 255) / 256), 256, 0, C.stream>>>(Q, g, d);
}
}  // namespace ox

int solver_create(const ox_config* cfg, hipStream_t shared, ox_solver** out) {
  if (!cfg || !out) return ox_fail(OX_EINVAL, "null argument");
  *out = nullptr;
  int rc = validate(*cfg);
  if (rc != OX_OK) return rc;
  ox_solver* s = new (std::nothrow) ox_solver();
  if (!s) return ox_fail(OX_ENOMEM, "host allocation failed");
  ox::Core& C = s->C;
  C.cfg = *cfg;
  C.g = make_geom(*cfg);
  C.hc.init(*cfg);
  C.hc.les_delta15 = ox::sms_delta15(C.g.inv_dx, C.g.inv_dy, C.g.inv_dz);
  C.vorder = cfg->visc == OX_VISC_EULER ? 0 : (cfg->visc_order ? cfg->visc_order : cfg->order);
  // ME4Base replaces the central-6 stencil only (calc_visc_high_internal.f90.fypp:17-23):
  // internal stencil code 5
  const bool me4 = C.vorder == 6 && cfg->visc_stencil == OX_STENCIL_ME4BASE;
  C.tvd = cfg->tvd;
  C.variant = cfg->slau_variant;
  C.Racc = nullptr;
  for (int set = 0; set < 2; ++set)
    for (int m = 0; m < ox::kPrimArrays; ++m) C.prim[set][m] = nullptr;
  C.cur = 0;
  C.prim_for = nullptr;
  C.prim_images[0] = C.prim_images[1] = false;
  C.stream = nullptr;
  C.lseg[0] = C.lseg[1] = 1;  // set below, once the device is known
  C.prof = false;
  C.mark = &prof_record;
  C.prof_state = &s->prof;
  if (C.vorder != 0 && C.vorder != 4 && C.vorder != 6) {
    delete s;
    return ox_fail(OX_EINVAL, "visc_order must be 4 or 6");
  }
  if (C.vorder == 6 && cfg->order != 6) {
    delete s;
    return ox_fail(OX_EINVAL, "visc_order 6 needs order 6 (three ghost layers)");
  }
  if (me4) C.vorder = 5;
  s->stage = cfg->precision == OX_PREC_FP64 ? ox::find_stage_fp64(cfg->order, cfg->scheme, cfg->visc, C.vorder)
                                            : ox::find_stage_fp32(cfg->order, cfg->scheme, cfg->visc, C.vorder);
  ox::BatchOps ops;
  const bool known = cfg->precision == OX_PREC_FP64
                         ? ox::find_batch_fp64(cfg->order, cfg->scheme, cfg->visc, C.vorder, &ops)
                         : ox::find_batch_fp32(cfg->order, cfg->scheme, cfg->visc, C.vorder, &ops);
  if (!s->stage || !known) {
    delete s;
    return ox_fail(OX_EUNSUPPORTED, "no kernel specialisation for this (order, scheme, visc, visc_order)");
  }
  hipError_t e = hipSetDevice(cfg->device);
  if (e != hipSuccess) {
    delete s;
    return ox_fail(OX_EDEVICE, std::string("hipSetDevice: ") + hipGetErrorString(e));
  }
  ox::solo_segments(C.g, ops, C.lseg);
  bool ok = shared || hipStreamCreateWithFlags(&s->own_stream, hipStreamNonBlocking) == hipSuccess;
  C.stream = shared ? shared : s->own_stream;
  // every array of the handle in one allocation: a hipFree of more than a few
  // MB costs about 0.1 ms, whatever its size
  const Layout at(*cfg);
  ok = ok && hipMalloc(&s->slab, at.bytes) == hipSuccess;
  ok = ok && hipEventCreate(&s->ev0) == hipSuccess && hipEventCreate(&s->ev1) == hipSuccess;
  if (!ok) {
    destroy(s);
    return ox_fail(OX_ENOMEM, "device allocation failed");
  }
  s->QJ = (double*)(s->slab + at.qj);
  s->QJ2 = (double*)(s->slab + at.qj2);
  C.Racc = s->slab + at.racc;
  if (cfg->rk == 4) s->Rs = (double*)(s->slab + at.rs);
  for (int set = 0; set < 2; ++set)
    for (int m = 0; m < at.nprim; ++m) C.prim[set][m] = s->slab + at.prim[set][m];
  s->scratch = (double*)(s->slab + at.scratch);
  s->scratch_bytes = at.scratch_bytes;
  // Zero everything once: ghost layers of QJ2 and the accumulators start defined.
  ok = hipMemsetAsync(s->slab, 0, at.cleared, C.stream) == hipSuccess;
  ok = ok && hipStreamSynchronize(C.stream) == hipSuccess;
  if (!ok) {
    destroy(s);
    return ox_fail(OX_EDEVICE, "device initialisation failed");
  }
  *out = s;
  return OX_OK;
}

extern "C" {

const char* ox_last_error(void) { return g_err.c_str(); }

int ox_host_alloc(uint64_t bytes, void** ptr) {
  if (!ptr || bytes == 0) return ox_fail(OX_EINVAL, "null pointer or zero size");
  *ptr = nullptr;
  OX_HIP(hipHostMalloc(ptr, (size_t)bytes, hipHostMallocDefault));
  return OX_OK;
}

int ox_host_free(void* ptr) {
  if (!ptr) return OX_OK;
  OX_HIP(hipHostFree(ptr));
  return OX_OK;
}

const char* ox_version(void) { return "ouxsbli-mi355x 1 gfx950"; }

int ox_real4_sum(const double* terms, int64_t n, float* out) {
  if (!out || (n > 0 && !terms) || n < 0) return ox_fail(OX_EINVAL, "null argument or negative count");
  // a REAL(4) accumulator: each REAL(8) term is added in double precision and
  // the sum rounded back to single, in order
  float acc = 0.0f;
  for (int64_t m = 0; m < n; ++m) acc = (float)((double)acc + terms[m]);
  *out = acc;
  return OX_OK;
}

int ox_create(const ox_config* cfg, ox_solver** out) { return solver_create(cfg, nullptr, out); }

void ox_destroy(ox_solver* s) {
  if (!s) return;
  hipSetDevice(s->C.cfg.device);
  if (s->C.stream) hipStreamSynchronize(s->C.stream);
  destroy(s);
}

int ox_set_qj(ox_solver* s, const double* QJ) {
  if (!s || !QJ) return ox_fail(OX_EINVAL, "null argument");
  OX_HIP(hipSetDevice(s->C.cfg.device));
  const size_t n = state_elems(s->C.g);
  OX_HIP(hipMemcpyAsync(s->QJ, QJ, n * sizeof(double), hipMemcpyHostToDevice, s->C.stream));
  if (s->Rs) OX_HIP(hipMemsetAsync(s->Rs, 0, n * sizeof(double), s->C.stream));
  s->C.prim_for = nullptr;  // the primitives no longer describe the state
  OX_HIP(hipStreamSynchronize(s->C.stream));
  return OX_OK;
}

int ox_get_qj(ox_solver* s, double* QJ) {
  if (!s || !QJ) return ox_fail(OX_EINVAL, "null argument");
  OX_HIP(hipSetDevice(s->C.cfg.device));
  const size_t n = state_elems(s->C.g);
  return copy_to_host(s->C.cfg.device, QJ, s->QJ, n * sizeof(double), s->C.stream);
}

int ox_set_state(ox_solver* s, const double* Q) {
  if (!s || !Q) return ox_fail(OX_EINVAL, "null argument");
  int rc = ox_set_qj(s, Q);
  if (rc != OX_OK) return rc;
  const long long n = (long long)state_elems(s->C.g);
  ox::k_scale<<<(unsigned)((n + 255) / 256), 256, 0, s->C.stream>>>(s->QJ, n, s->C.g.jac, 1);
  OX_HIP(hipGetLastError());
  OX_HIP(hipStreamSynchronize(s->C.stream));
  return OX_OK;
}

int ox_get_state(ox_solver* s, double* Q) {
  if (!s || !Q) return ox_fail(OX_EINVAL, "null argument");
  OX_HIP(hipSetDevice(s->C.cfg.device));
  const long long n = (long long)state_elems(s->C.g);
  // J * QJ into the second state buffer, which holds no live data between
  // calls (every RK step rewrites it from QJ before reading it), then one copy
  OX_HIP(hipStreamSynchronize(s->C.stream));
  ox::k_scale_to<<<(unsigned)((n + 255) / 256), 256, 0, s->C.stream>>>(s->QJ, s->QJ2, n, s->C.g.jac);
  OX_HIP(hipGetLastError());
  if (s->C.prim_for == s->QJ2) s->C.prim_for = nullptr;
  return copy_to_host(s->C.cfg.device, Q, s->QJ2, n * sizeof(double), s->C.stream);
}

int ox_step(ox_solver* s, int32_t nsteps) {
  if (!s) return ox_fail(OX_EINVAL, "null handle");
  if (nsteps < 0) return ox_fail(OX_EINVAL, "nsteps < 0");
  OX_HIP(hipSetDevice(s->C.cfg.device));
  OX_HIP(hipEventRecord(s->ev0, s->C.stream));
  if (s->C.prof) {
    s->prof.used = 0;
    prof_record(&s->C, "start");
  }
  for (int t = 0; t < nsteps; ++t) run_rk_step(s);
  if (nsteps > 0) {
    // the stages keep the primitives of ghost cells current themselves; the
    // state's own ghost layers are filled once, for its readers (get_state,
    // diagnostics, the RHS hook)
    ox::launch_ghost_fill(s->C, s->QJ);
    ox::prof_mark(s->C, "ghost_fill");
  }
  OX_HIP(hipGetLastError());
  OX_HIP(hipEventRecord(s->ev1, s->C.stream));
  OX_HIP(hipEventSynchronize(s->ev1));
  float ms = 0.f;
  OX_HIP(hipEventElapsedTime(&ms, s->ev0, s->ev1));
  s->last_ms = ms;
  if (s->C.prof) {
    ProfState& P = s->prof;
    for (size_t m = 1; m < P.used; ++m) {
      float d = 0.f;
      OX_HIP(hipEventElapsedTime(&d, P.pool[m - 1], P.pool[m]));
      size_t a = 0;
      while (a < P.acc_names.size() && P.acc_names[a] != P.names[m]) ++a;
      if (a == P.acc_names.size()) {
        P.acc_names.emplace_back(P.names[m]);
        P.acc_ms.push_back(0.0);
        P.acc_n.push_back(0);
      }
      P.acc_ms[a] += d;
      P.acc_n[a] += 1;
    }
    P.used = 0;
  }
  return OX_OK;
}

int ox_rhs(ox_solver* s, double* R) {
  if (!s || !R) return ox_fail(OX_EINVAL, "null argument");
  OX_HIP(hipSetDevice(s->C.cfg.device));
  const ox::Geom& g = s->C.g;
  const size_t n = state_elems(g);
  // the result goes to the second state buffer, which is then restored from
  // Q^n semantics: QJ2 is scratch between steps.
  OX_HIP(hipMemsetAsync(s->QJ2, 0, n * sizeof(double), s->C.stream));
  if (s->C.prim_for == s->QJ2) s->C.prim_for = nullptr;
  ox::StageArgs sa{s->QJ, s->QJ2, s->Rs, 0, 0, 0, ox::EP_RHS};
  s->stage(s->C, s->QJ, sa, g.a_yz, g.a_zx, g.a_xy);
  OX_HIP(hipGetLastError());
  return copy_to_host(s->C.cfg.device, R, s->QJ2, n * sizeof(double), s->C.stream);
}

int ox_diagnostics(ox_solver* s, ox_diag* out) {
  if (!s || !out) return ox_fail(OX_EINVAL, "null argument");
  OX_HIP(hipSetDevice(s->C.cfg.device));
  const ox::Geom& g = s->C.g;
  const long long n = (long long)g.ix * g.iy * g.iz;
  int nb = (int)std::min<long long>(4096, (n + ox::DIAG_BLOCK - 1) / ox::DIAG_BLOCK);
  if (nb < 1) nb = 1;
  ox::k_diag<<<nb, ox::DIAG_BLOCK, 0, s->C.stream>>>(s->QJ, g, s->C.cfg.gamma, s->scratch);
  OX_HIP(hipGetLastError());
  std::vector<double> part((size_t)nb * (2 * ox::DIAG_NQ + 1));
  OX_HIP(hipMemcpyAsync(part.data(), s->scratch, part.size() * sizeof(double), hipMemcpyDeviceToHost, s->C.stream));
  OX_HIP(hipStreamSynchronize(s->C.stream));
  double sum[ox::DIAG_NQ], comp[ox::DIAG_NQ];
  for (int q = 0; q < ox::DIAG_NQ; ++q) sum[q] = comp[q] = 0.0;
  double wmax = 0.0;
  for (int b = 0; b < nb; ++b) {
    const double* p = part.data() + (size_t)b * (2 * ox::DIAG_NQ + 1);
    for (int q = 0; q < ox::DIAG_NQ; ++q) {
      const double x = p[2 * q];
      const double t = sum[q] + x;
      if (std::fabs(sum[q]) >= std::fabs(x)) comp[q] += (sum[q] - t) + x;
      else comp[q] += (x - t) + sum[q];
      sum[q] = t;
      comp[q] += p[2 * q + 1];
    }
    wmax = ox::nan_max(wmax, p[2 * ox::DIAG_NQ]);
  }
  const double ncell = (double)g.ix * (double)g.iy * (double)g.iz;
  out->ke = (sum[0] + comp[0]) / ncell;
  out->entropy = (sum[1] + comp[1]) / ncell;
  out->enstrophy = (sum[2] + comp[2]) / ncell;
  out->max_wave_speed = wmax;
  out->mass = sum[3] + comp[3];
  out->energy = sum[4] + comp[4];
  return OX_OK;
}

int ox_diagnostics_noalloc(ox_solver* s, ox_diag* out) {
  if (!s || !out) return ox_fail(OX_EINVAL, "null argument");
  OX_HIP(hipSetDevice(s->C.cfg.device));
  double* scratch = nullptr;
  int rc = noalloc_scratch_ptr(s->C.cfg.device, &scratch);
  if (rc != OX_OK) return rc;
  const ox::Geom& g = s->C.g;
  const long long n = (long long)g.ix * g.iy * g.iz;
  int nb = (int)std::min<long long>(kNoAllocMaxBlocks, (n + ox::DIAG_BLOCK - 1) / ox::DIAG_BLOCK);
  if (nb < 1) nb = 1;
  if ((size_t)nb * kDiagStride + ox::DIAG_NQ + 1 > kNoAllocDoubles)
    return ox_fail(OX_EINVAL, "diagnostics need " + std::to_string(nb) + " partials, beyond the static scratch of " +
                                  std::to_string(kNoAllocMaxBlocks));
  double* result = scratch + (size_t)kNoAllocMaxBlocks * kDiagStride;
  ox::k_diag<<<nb, ox::DIAG_BLOCK, 0, s->C.stream>>>(s->QJ, g, s->C.cfg.gamma, scratch);
  OX_HIP(hipGetLastError());
  ox::k_diag_merge<<<1, 64, 0, s->C.stream>>>(scratch, nb, result);
  OX_HIP(hipGetLastError());
  double r[ox::DIAG_NQ + 1];
  OX_HIP(hipMemcpyAsync(r, result, sizeof(r), hipMemcpyDeviceToHost, s->C.stream));
  OX_HIP(hipStreamSynchronize(s->C.stream));
  const double ncell = (double)g.ix * (double)g.iy * (double)g.iz;
  out->ke = r[0] / ncell;
  out->entropy = r[1] / ncell;
  out->enstrophy = r[2] / ncell;
  out->max_wave_speed = r[ox::DIAG_NQ];
  out->mass = r[3];
  out->energy = r[4];
  return OX_OK;
}

int ox_check_state(ox_solver* s, int64_t* bad_index, int64_t* count) {
  if (!s) return ox_fail(OX_EINVAL, "null handle");
  OX_HIP(hipSetDevice(s->C.cfg.device));
  const ox::Geom& g = s->C.g;
  const long long n = (long long)g.ix * g.iy * g.iz;
  int nb = (int)std::min<long long>(4096, (n + ox::DIAG_BLOCK - 1) / ox::DIAG_BLOCK);
  if (nb < 1) nb = 1;
  long long* part = reinterpret_cast<long long*>(s->scratch);
  ox::k_check<<<nb, ox::DIAG_BLOCK, 0, s->C.stream>>>(s->QJ, g, s->C.cfg.gamma, part);
  OX_HIP(hipGetLastError());
  std::vector<long long> h((size_t)2 * nb);
  OX_HIP(hipMemcpyAsync(h.data(), part, h.size() * sizeof(long long), hipMemcpyDeviceToHost, s->C.stream));
  OX_HIP(hipStreamSynchronize(s->C.stream));
  long long cnt = 0, first = -1;
  for (int b = 0; b < nb; ++b) {
    cnt += h[2 * b];
    const long long f = h[2 * b + 1];
    if (f >= 0 && (first < 0 || f < first)) first = f;
  }
  if (bad_index) *bad_index = first;
  if (count) *count = cnt;
  if (cnt > 0) return ox_fail(OX_ESTATE, "non-physical state: " + std::to_string(cnt) + " bad cells, first at linear index " +
                                          std::to_string(first));
  return OX_OK;
}

int ox_synchronize(ox_solver* s) {
  if (!s) return ox_fail(OX_EINVAL, "null handle");
  OX_HIP(hipSetDevice(s->C.cfg.device));
  OX_HIP(hipStreamSynchronize(s->C.stream));
  return OX_OK;
}

int ox_set_profiling(ox_solver* s, int32_t enable) {
  if (!s) return ox_fail(OX_EINVAL, "null handle");
  s->C.prof = enable != 0;
  s->prof.acc_names.clear();
  s->prof.acc_ms.clear();
  s->prof.acc_n.clear();
  s->prof.used = 0;
  return OX_OK;
}

int ox_kernel_times(ox_solver* s, ox_kernel_time* out, int32_t cap, int32_t* n) {
  if (!s || !n) return ox_fail(OX_EINVAL, "null argument");
  const ProfState& P = s->prof;
  *n = (int32_t)P.acc_names.size();
  for (int32_t a = 0; a < *n && a < cap && out; ++a) {
    std::memset(out[a].name, 0, sizeof(out[a].name));
    std::strncpy(out[a].name, P.acc_names[a].c_str(), sizeof(out[a].name) - 1);
    out[a].total_ms = P.acc_ms[a];
    out[a].launches = P.acc_n[a];
  }
  return OX_OK;
}

int ox_last_step_ms(ox_solver* s, double* ms) {
  if (!s || !ms) return ox_fail(OX_EINVAL, "null argument");
  *ms = s->last_ms;
  return OX_OK;
}

}  // extern "C"

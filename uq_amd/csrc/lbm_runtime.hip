// lbm_runtime.hip — host runtime and C ABI (include/uqlbm.h) of the MI355X
// D2Q13 thermal FD-LBM: deck refinement, device state, work lists, batched
// stepping, geometry validation.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <chrono>
#include <climits>
#include <cmath>
#include <cstdarg>
#include <cstdio>
#include <cstring>
#include <map>
#include <memory>
#include <mutex>
#include <string>
#include <utility>
#include <vector>

#include "../../include/uqlbm.h"
#include "lbm_common.hpp"
#include "lbm_device.hpp"
#include "lbm_launch.hpp"
#include "lbm_point.hpp"
#include "lbm_runtime.hpp"

namespace uqlbm {

// ---------------------------------------------------------------------------
// errors
// ---------------------------------------------------------------------------
static thread_local std::string g_error;

int fail_with(int status, const char* fmt, ...) {
  char buf[512];
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(buf, sizeof(buf), fmt, ap);
  va_end(ap);
  g_error = buf;
  return status;
}

#define HIP_TRY(expr)                                                                          \
  do {                                                                                         \
    hipError_t e_ = (expr);                                                                    \
    if (e_ != hipSuccess) return fail_with(LBM_ERR_HIP, "%s: %s", #expr, hipGetErrorString(e_)); \
  } while (0)

static thread_local KernelTimer* g_timer = nullptr;
static bool g_timing_enabled = false;
static thread_local lbm_timing g_last_timing = {};

// ---------------------------------------------------------------------------
// deck refinement (reference refineInput / setupVars, cpuLBM.cpp:283-450)
// ---------------------------------------------------------------------------
static void steps_from_dt(Solver& s);

static void refine_deck(Solver& s) {
  lbm_params& p = s.p;
  if (p.dx == 0) p.dx = p.Lx / ((double)s.nx - 1);
  else p.Lx = p.dx * (s.nx - 1);
  if (p.dy == 0 && p.Ly != 0) p.dy = p.Ly / ((double)s.ny - 1);
  else if (p.dy == 0 && p.Ly == 0) { p.dy = p.dx; p.Ly = p.dy * (s.ny - 1); }
  else p.Ly = p.dy * (s.ny - 1);
  if (p.rho_ref == 0) p.rho_ref = p.p_ref / (p.R * p.T_ref);
  else if (p.p_ref == 0) p.p_ref = p.rho_ref * p.R * p.T_ref;
  else if (p.T_ref == 0) p.T_ref = p.p_ref / (p.rho_ref * p.R);
  for (auto& r : s.props) {
    if (r.rho == 0) r.rho = r.p / (p.R * r.T);
    else if (r.p == 0) r.p = r.rho * p.R * r.T;
    else if (r.T == 0) r.T = r.p / (r.rho * p.R);
  }
  s.b = 2 / (p.gamma - 1);
  s.K = s.b - 2;
  s.Tc = p.Tc_Tref * p.T_ref;
  const double tau_ref = p.mu / p.p_ref;
  s.c = std::sqrt(p.R * s.Tc);
  const double e9 = 2 * s.c;
  s.dt = p.dtau == 0 ? (p.cfl * std::min(p.dx, p.dy)) / e9 : p.dtau * tau_ref;
  steps_from_dt(s);
}

// nsteps from tt_tref, tt_time or steps (cpuLBM.cpp:423-448)
static void steps_from_dt(Solver& s) {
  const lbm_params& p = s.p;
  const double t_ref = std::max(p.Lx, p.Ly) / std::sqrt(p.R * p.T_ref);
  double total = 0;
  bool need = false;
  s.nsteps = 0;
  if (p.tt_tref > 0) { total = p.tt_tref * t_ref; need = true; }
  else if (p.tt_time > 0) { total = p.tt_time; need = true; }
  else if (p.steps > 0) s.nsteps = p.steps;
  if (need) s.nsteps = (int)std::ceil(total / s.dt);
}

// ---------------------------------------------------------------------------
// Stencil addressing per cell: the tile kernels resolve a stencil point from
// its logical position (cell + offset mapped once through the boundary
// rules, direction remapped at mirrors) and take an upwind face flux across
// a clamped edge from the cell itself. The reference instead maps the
// physical neighbour of a physical point (extrapolation points, upwind
// owners). The two agree except next to solid features one cell thick or
// solids near a mirror edge; this check compares them cell by cell and
// marks the cells where they differ, whose tiles then form every net flux
// with the reference's addressing (phys_net in the flux kernels).
// ---------------------------------------------------------------------------
struct Pt {
  int x, y, d;
  bool operator==(const Pt& o) const { return x == o.x && y == o.y && d == o.d; }
};

static int ref_map(const Solver& s, int i, int axis, int& mir, bool& clamped) {
  const int n = axis == 0 ? s.nx : s.ny;
  const bool per = axis == 0 ? s.p.periodic_x > 0 : s.p.periodic_y > 0;
  const bool mlo = axis == 0 ? s.p.mirror_west > 0 : s.p.mirror_south > 0;
  const bool mhi = axis == 0 ? s.p.mirror_east > 0 : s.p.mirror_north > 0;
  mir = 0;
  clamped = false;
  if (i < 0) {
    if (per) i = n + i;
    else if (mlo) { i = -i - 1; mir = 1; }
    else { i = 0; clamped = true; }
  } else if (i > n - 1) {
    if (per) i = i - n;
    else if (mhi) { i = 2 * n - i - 1; mir = 1; }
    else { i = n - 1; clamped = true; }
  }
  return std::min(std::max(i, 0), n - 1);
}

static int type_at(const Solver& s, int x, int y) { return s.ctype_host[(size_t)y * s.nx + x]; }

struct LineReads {
  int L = 0;
  Pt pts[5];
  int sld[5] = {0, 0, 0, 0, 0};
  bool any = false;
  int jj = 0, diff = 0;
  Pt e1{}, e2{};
  bool wall_owner = false;
  Pt wall_src{};
};

// Reference: out-face stencil of physical cell (cx, cy), direction i, axis.
static void ref_line(const Solver& s, int cx, int cy, int i, int axis, LineReads& r) {
  const int e = axis == 0 ? lat_x(i) : lat_y(i), sg = sgn_i(e);
  r = LineReads();
  if (type_at(s, cx, cy) == 2) {
    r.wall_owner = true;
    r.wall_src = {cx, cy, i};
    return;
  }
  r.L = s.p.flux_method == 1 ? 5 : 3;
  const int low = (r.L - 1) / 2;
  const int start = (axis == 0 ? cx : cy) - sg * low;
  for (int j = 0; j < r.L; j++) {
    int mir;
    bool cl;
    const int p = ref_map(s, start + sg * j, axis, mir, cl);
    const int d = mir ? (axis == 0 ? mirror_ew(i) : mirror_ns(i)) : i;
    r.pts[j] = axis == 0 ? Pt{p, cy, d} : Pt{cx, p, d};
    r.sld[j] = (axis == 0 ? type_at(s, p, cy) : type_at(s, cx, p)) == 2;
    r.any |= r.sld[j] != 0;
  }
  if (!r.any) return;
  int pos = 0;
  for (int j = 0; j < r.L - 1; j++) {
    const int d = r.sld[j] - r.sld[j + 1];
    int mir;
    bool cl;
    if (d > 0) { r.diff = d; r.jj = j; pos = ref_map(s, start + sg * j, axis, mir, cl); break; }
    if (d < 0) { r.diff = d; r.jj = j + 1; pos = ref_map(s, start + sg * (j + 1), axis, mir, cl); break; }
  }
  int mir;
  bool cl;
  const int m1 = ref_map(s, pos + sg * r.diff, axis, mir, cl);
  const int m2 = ref_map(s, pos + sg * 2 * r.diff, axis, mir, cl);
  r.e1 = axis == 0 ? Pt{m1, cy, i} : Pt{cx, m1, i};
  r.e2 = axis == 0 ? Pt{m2, cy, i} : Pt{cx, m2, i};
}

// Kernel: out-face stencil of the owner at logical position (lx, ly) (one
// coordinate may lie outside the grid), direction i, axis.
static Pt ker_point(const Solver& s, int lx, int ly, int i) {
  int mx, my;
  bool cx, cy;
  const int X = ref_map(s, lx, 0, mx, cx);
  const int Y = ref_map(s, ly, 1, my, cy);
  int d = i;
  if (mx) d = mirror_ew(d);
  if (my) d = mirror_ns(d);
  return {X, Y, d};
}

static void ker_line(const Solver& s, int lx, int ly, int i, int axis, LineReads& r) {
  const int e = axis == 0 ? lat_x(i) : lat_y(i), sg = sgn_i(e);
  r = LineReads();
  const Pt own = ker_point(s, lx, ly, i);
  if (type_at(s, own.x, own.y) == 2) {
    r.wall_owner = true;
    r.wall_src = own;
    return;
  }
  r.L = s.p.flux_method == 1 ? 5 : 3;
  const int low = (r.L - 1) / 2;
  for (int k = 0; k < r.L; k++) {
    const int px = axis == 0 ? lx + (k - low) * sg : lx;
    const int py = axis == 0 ? ly : ly + (k - low) * sg;
    r.pts[k] = ker_point(s, px, py, i);
    r.sld[k] = type_at(s, r.pts[k].x, r.pts[k].y) == 2;
    r.any |= r.sld[k] != 0;
  }
  if (!r.any) return;
  for (int j = 0; j < r.L - 1; j++) {
    const int d = r.sld[j] - r.sld[j + 1];
    if (d != 0) { r.diff = d; r.jj = d > 0 ? j : j + 1; break; }
  }
  const int k1 = std::min(std::max(r.jj + r.diff, 0), r.L - 1);
  const int k2 = std::min(std::max(r.jj + 2 * r.diff, 0), r.L - 1);
  r.e1 = r.pts[k1];
  r.e2 = r.pts[k2];
}

static bool same(const LineReads& a, const LineReads& b) {
  if (a.wall_owner != b.wall_owner) return false;
  if (a.wall_owner) return a.wall_src == b.wall_src;
  if (a.L != b.L || a.any != b.any) return false;
  for (int k = 0; k < a.L; k++)
    if (!(a.pts[k] == b.pts[k]) || a.sld[k] != b.sld[k]) return false;
  if (!a.any) return true;
  return a.jj == b.jj && a.diff == b.diff && a.e1 == b.e1 && a.e2 == b.e2;
}

// Marks in s.phys_cells ([y][x]) every fluid or permanent cell one of whose
// faces the logical addressing would form differently from the reference.
static void mark_physical_cells(Solver& s) {
  const int R = 5;  // reach of owner (1) + stencil (2) + extrapolation (2)
  s.phys_cells.assign((size_t)s.nx * s.ny, 0);
  s.any_phys = false;
  for (int axis = 0; axis < 2; axis++) {
    const int n = axis == 0 ? s.nx : s.ny, m = axis == 0 ? s.ny : s.nx;
    std::vector<char> near(n);
    for (int line = 0; line < m; line++) {
      std::fill(near.begin(), near.end(), 0);
      for (int k = 0; k < n; k++) {
        const bool edge = k < R || k >= n - R;
        const int t = axis == 0 ? type_at(s, k, line) : type_at(s, line, k);
        if (edge) near[k] = 1;
        if (t == 2)
          for (int q = std::max(0, k - R); q <= std::min(n - 1, k + R); q++) near[q] = 1;
      }
      for (int k = 0; k < n; k++) {
        if (!near[k]) continue;
        const int cx = axis == 0 ? k : line, cy = axis == 0 ? line : k;
        if (type_at(s, cx, cy) == 2) continue;
        bool differs = false;
        for (int i = 1; i < kQ && !differs; i++) {
          const int e = axis == 0 ? lat_x(i) : lat_y(i);
          if (e == 0) continue;
          const int sg = sgn_i(e);
          LineReads a, b;
          // own out-face
          ref_line(s, cx, cy, i, axis, a);
          ker_line(s, cx, cy, i, axis, b);
          if (!same(a, b)) {
            differs = true;
            break;
          }
          // upwind owner (reference cFLUX: index(x,-s) with mirror remap);
          // across a clamped edge both take the cell's own out-face
          int mir;
          bool cl;
          const int up = ref_map(s, (axis == 0 ? cx : cy) - sg, axis, mir, cl);
          const int iu = mir ? (axis == 0 ? mirror_ew(i) : mirror_ns(i)) : i;
          if (cl) {
            differs = up != (axis == 0 ? cx : cy);
            continue;
          }
          ref_line(s, axis == 0 ? up : cx, axis == 0 ? cy : up, iu, axis, a);
          ker_line(s, axis == 0 ? cx - sg : cx, axis == 0 ? cy : cy - sg, i, axis, b);
          differs = !same(a, b);
        }
        if (differs) {
          s.phys_cells[(size_t)cy * s.nx + cx] = 1;
          s.any_phys = true;
        }
      }
    }
  }
}

// ---------------------------------------------------------------------------
// solver lifetime
// ---------------------------------------------------------------------------
static size_t elem_size(int precision) { return precision == LBM_PREC_FP64 ? sizeof(double) : sizeof(float); }

// Device bytes of one solver: 4 x 26 distribution planes (two state buffers,
// f2, f3), the dF planes, cell types, wall factor, property ids and the
// macroscopic output planes.
size_t uqlbm::solver_footprint(int nx, int ny, int precision) {
  const size_t pitch = (size_t)((nx + 63) / 64 * 64);
  const size_t plane = pitch * ny;
  const size_t es = elem_size(precision);
  const size_t mom = precision == LBM_PREC_FP64 ? 0 : 2 * 4 * sizeof(double);  // moment planes of FP32 storage
  return plane * (kPlanes * 4 + dflux_planes()) * es +
         plane * (1 + sizeof(double) + sizeof(int) + 5 * sizeof(double) + mom);
}

// Reference equilibrium of FP32 storage: the equilibrium at rest at the mean
// density and temperature of the deck's fluid cells. Stored values are the
// distributions' deviations from it; being at rest it depends on |e| only,
// so a direction and its mirror images share it.
template <int... Is>
static void eq_all(const EqIn<double>& q, double* f, double* h, std::integer_sequence<int, Is...>) {
  ((eq_dir<Is>(q, f[Is], h[Is])), ...);
}

// FP32 storage: whether every fluid or permanent cell starts near the
// reference equilibrium (density and temperature within 25 % of the
// reference's, speed within half of sqrt(R Tc)). Launch groups made of such
// instances evaluate their equilibria in FP32 in the deviation form, whose
// terms are then small; others in FP64.
static bool near_reference(const Solver& s) {
  std::vector<char> used(s.props.size(), 0);
  for (int id : s.ids_host) used[id] = 1;
  const double sc = std::sqrt(s.p.R * s.Tc);
  for (size_t r = 0; r < s.props.size(); r++) {
    const PropRow& p = s.props[r];
    if (!used[r] || p.type == 2) continue;
    if (std::fabs(p.rho - s.ref_rho) > 0.25 * s.ref_rho) return false;
    if (std::fabs(p.T / s.Tc - s.ref_t) > 0.25 * s.ref_t) return false;
    if (std::hypot(p.ux, p.uy) > 0.5 * sc) return false;
  }
  return true;
}

static void set_reference(Solver& s) {
  double rho = 0, T = 0;
  long long n = 0;
  for (int pass = 0; pass < 2 && n == 0; pass++)
    for (size_t k = 0; k < s.ids_host.size(); k++) {
      const PropRow& r = s.props[s.ids_host[k]];
      if (pass == 0 && r.type != 0) continue;
      rho += r.rho;
      T += r.T;
      n++;
    }
  rho /= (double)n;
  T /= (double)n;
  EqIn<double> q;
  q.rho = rho;
  q.u = 0;
  q.v = 0;
  q.t = T / s.Tc;
  q.K = s.K;
  q.scale = rho * s.p.R * s.Tc;
  double f[kQ], h[kQ];
  eq_all(q, f, h, std::make_integer_sequence<int, kQ>{});
  for (int i = 0; i < kQ; i++) {
    s.ref[i] = f[i];
    s.ref[kQ + i] = h[i];
  }
  s.ref_rho = rho;
  s.ref_t = q.t;
}

// Device buffers of destroyed solvers, kept per device and size for the
// next solver that needs the same (a served request stream creates and
// destroys solvers of recurring sizes; hipMalloc and hipFree, which waits
// for the whole device, leave the serving loop). At most kCacheMax bytes
// are kept; a hipMalloc that finds the device full returns the device's
// kept buffers first (lbm_release_cached returns them on request).
namespace {
constexpr size_t kCacheMax = size_t(32) << 30;
struct BufferCache {
  std::mutex mu;
  std::map<std::pair<int, size_t>, std::vector<void*>> free;
  size_t bytes = 0;
  void drop(int dev) {  // with mu held
    for (auto it = free.begin(); it != free.end();) {
      if (dev >= 0 && it->first.first != dev) {
        ++it;
        continue;
      }
      for (void* p : it->second) (void)hipFree(p);
      bytes -= it->first.second * it->second.size();
      it = free.erase(it);
    }
  }
};
BufferCache& buffer_cache() {
  static BufferCache* c = new BufferCache();  // never destroyed: outlives every solver
  return *c;
}
}  // namespace

hipError_t uqlbm::solver_alloc(Solver& s, void** p, size_t bytes) {
  *p = nullptr;
  int dev = 0;
  (void)hipGetDevice(&dev);
  BufferCache& c = buffer_cache();
  {
    std::lock_guard<std::mutex> lock(c.mu);
    auto it = c.free.find({dev, bytes});
    if (it != c.free.end() && !it->second.empty()) {
      *p = it->second.back();
      it->second.pop_back();
      c.bytes -= bytes;
    }
  }
  if (!*p) {
    hipError_t e = hipMalloc(p, bytes);
    if (e == hipErrorOutOfMemory) {
      (void)hipGetLastError();
      {
        std::lock_guard<std::mutex> lock(c.mu);
        c.drop(dev);
      }
      e = hipMalloc(p, bytes);
    }
    if (e != hipSuccess) return e;
  }
  s.owned.push_back({*p, bytes});
  return hipSuccess;
}

Solver::~Solver() {
  if (graphs) graphs->clear();
  // no work of this solver may still use a buffer that the next solver gets
  if (stream) (void)hipStreamSynchronize(stream);
  int dev = 0;
  (void)hipGetDevice(&dev);
  BufferCache& c = buffer_cache();
  {
    std::lock_guard<std::mutex> lock(c.mu);
    for (auto& ob : owned) {
      if (c.bytes + ob.second <= kCacheMax) {
        c.free[{dev, ob.second}].push_back(ob.first);
        c.bytes += ob.second;
      } else {
        (void)hipFree(ob.first);
      }
    }
  }
  if (stream) (void)hipStreamDestroy(stream);
  if (result) (void)hipHostFree(result);
}

extern "C" void lbm_release_cached(void) {
  release_slots();
  BufferCache& c = buffer_cache();
  std::lock_guard<std::mutex> lock(c.mu);
  c.drop(-1);
}

static void fill_inst(const Solver& s, InstDev& d) {
  d = InstDev{};
  d.nx = s.nx;
  d.ny = s.ny;
  d.pitch = s.pitch;
  d.flags = (s.p.periodic_x > 0 ? kPeriodicX : 0) | (s.p.periodic_y > 0 ? kPeriodicY : 0) |
            (s.p.mirror_north > 0 ? kMirrorN : 0) | (s.p.mirror_south > 0 ? kMirrorS : 0) |
            (s.p.mirror_east > 0 ? kMirrorE : 0) | (s.p.mirror_west > 0 ? kMirrorW : 0);
  d.flux_method = s.p.flux_method;
  d.parity0 = s.cur;
  d.step_base = s.step;
  d.plane = (long long)s.pitch * s.ny;
  d.state[0] = s.state[0];
  d.state[1] = s.state[1];
  d.f2 = s.f2;
  d.f3 = s.f3;
  d.dflux = s.dflux;
  d.ctype = s.ctype;
  d.alpha = s.alpha;
  d.fail = s.fail;
  d.mom[0] = s.mom[0];
  d.mom[1] = s.mom[1];
  for (int k = 0; k < kPlanes; k++) d.ref[k] = s.precision == LBM_PREC_FP64 ? 0.0 : s.ref[k];
  for (int k = 0; k < 4; k++) d.refsum[k] = 0.0;
  if (s.precision != LBM_PREC_FP64)
    for (int i = 0; i < kQ; i++) {
      d.refsum[0] += s.ref[i];
      d.refsum[1] += s.ref[i] * (lat_x(i) * s.c);
      d.refsum[2] += s.ref[i] * (lat_y(i) * s.c);
      d.refsum[3] += s.ref[kQ + i];
    }
  d.i2c = 0.5 / s.c;
  d.eq32 = s.eq32 ? 1 : 0;
  if (s.precision != LBM_PREC_FP64) {
    // base polynomials of the reference: f per unit density, h per unit rho R Tc
    static constexpr int kBase[4] = {0, 1, 5, 9};
    d.rho0 = s.ref_rho;
    d.t0 = s.ref_t;
    for (int j = 0; j < 4; j++) {
      d.eqref[j] = float(s.ref[kBase[j]] / s.ref_rho);
      d.eqref[4 + j] = float(s.ref[kQ + kBase[j]] / (s.ref_rho * s.p.R * s.Tc));
    }
  }
  d.dt = s.dt;
  d.dx = s.p.dx;
  d.dy = s.p.dy;
  d.rdx = s.dt / s.p.dx;
  d.rdy = s.dt / s.p.dy;
  d.rdxs = s.spacing_dev;
  d.rdys = s.spacing_dev ? s.spacing_dev + s.nx : nullptr;
  d.dxs = s.spacing_dev ? s.spacing_dev + s.nx + s.ny : nullptr;
  d.dys = s.spacing_dev ? s.spacing_dev + 2 * s.nx + s.ny : nullptr;
  d.c = s.c;
  d.sRTc = std::sqrt(s.p.R * s.Tc);
  d.Tc = s.Tc;
  d.R = s.p.R;
  d.b = s.b;
  d.K = s.K;
  d.bR = s.b * s.p.R;
  d.RTc = s.p.R * s.Tc;
  d.mu = s.p.mu;
  d.Pr = s.p.Pr;
  d.isRTc = 1.0 / d.sRTc;
  d.iTc = 1.0 / d.Tc;
  d.ibR = 1.0 / d.bR;
  d.iRTc = 1.0 / d.RTc;
  d.imu = 1.0 / d.mu;
  d.Pr_m1 = d.Pr - 1.0;
  point_consts(s.K, d.kq);
  d.visc_model = s.visc_model;
  d.mu_ref = s.mu_ref;
  d.T_ref_v = s.T_ref_v;
  d.iT_ref_v = s.T_ref_v > 0 ? 1.0 / s.T_ref_v : 0.0;
  d.vexp = 0.5 + s.visc_param;
  d.vS = s.visc_param;
  d.res_hist = nullptr;  // set per launch group (run_group)
  d.res_last = 0;
  d.ptile0 = 0;
  d.nptiles = s.nptiles;
  d.strips = 0;  // set per launch group (run_group)
}

// Flux tiles of one shape with the per-tile solid flag (the tile's region
// holds a solid cell), instance index 0.
static std::vector<TileRef> build_flux_tiles(const Solver& s, int shape) {
  std::vector<TileRef> tiles;
  int TW = 0, TH = 0;
  flux_tile_dims(shape, &TW, &TH);
  const int H = tile_halo();
  const int tx_n = (s.nx + TW - 1) / TW, ty_n = (s.ny + TH - 1) / TH;
  // prefix count of solid cells for the per-tile solid flag
  std::vector<int> pre((size_t)(s.nx + 1) * (s.ny + 1), 0);
  auto P = [&](int x, int y) -> int& { return pre[(size_t)y * (s.nx + 1) + x]; };
  for (int y = 0; y < s.ny; y++)
    for (int x = 0; x < s.nx; x++)
      P(x + 1, y + 1) = P(x, y + 1) + P(x + 1, y) - P(x, y) + (type_at(s, x, y) == 2);
  auto count = [&](int x0, int y0, int x1, int y1) {
    x0 = std::max(x0, 0); y0 = std::max(y0, 0);
    x1 = std::min(x1, s.nx); y1 = std::min(y1, s.ny);
    if (x0 >= x1 || y0 >= y1) return 0;
    return P(x1, y1) - P(x0, y1) - P(x1, y0) + P(x0, y0);
  };
  const bool any_edge_solid = count(0, 0, s.nx, H + 1) || count(0, s.ny - H - 1, s.nx, s.ny) ||
                              count(0, 0, H + 1, s.ny) || count(s.nx - H - 1, 0, s.nx, s.ny);
  for (int ty = 0; ty < ty_n; ty++)
    for (int tx = 0; tx < tx_n; tx++) {
      const int x0 = tx * TW, y0 = ty * TH;
      bool solid = count(x0 - H, y0 - H, x0 + TW + H, y0 + TH + H) > 0;
      // halo positions wrapped or mirrored across an edge may reach solids
      // on the far side: be conservative on edge tiles
      const bool edge = x0 - H < 0 || y0 - H < 0 || x0 + TW + H > s.nx || y0 + TH + H > s.ny;
      if (edge && any_edge_solid) solid = true;
      bool phys = false;
      if (s.any_phys)
        for (int y = y0; y < std::min(y0 + TH, s.ny) && !phys; y++)
          for (int x = x0; x < std::min(x0 + TW, s.nx) && !phys; x++) phys = s.phys_cells[(size_t)y * s.nx + x];
      tiles.push_back(TileRef{0, tx, ty, (solid ? kTileSolid : 0) | (phys ? kTilePhysical : 0)});
    }
  return tiles;
}

// Strip work items of up to `rows` rows (`most_solid` of them near solids) of
// an instance (instance index `inst`), appended to out. Consecutive rows of the same kind (solid or not)
// form an item, so that only the rows near a solid take the solid path.
// TileRef: tx = strip index, ty = first row, flags = kTileSolid (solid rows)
// | kStripDesc (every second item of a column) | row count << kStripRowsBit.
static void strip_items(const Solver& s, int rows, int most_solid, int inst, std::vector<TileRef>& out) {
  const size_t first = out.size();
  for (int sx = 0; sx < s.strip_cols; sx++) {
    const char* solid = s.strip_solid.data() + (size_t)sx * s.ny;
    // the items of a strip column alternate between ascending and
    // descending row order (kStripDesc), so that neighbours one above the
    // other read the rows they share at about the same time
    for (int y = 0, k = 0; y < s.ny; k++) {
      int n = 1;
      const int most = solid[y] ? most_solid : rows;
      while (y + n < s.ny && n < most && solid[y + n] == solid[y]) n++;
      out.push_back(TileRef{inst, sx, y, (solid[y] ? kTileSolid : 0) | ((k & 1) ? kStripDesc : 0) | (n << kStripRowsBit)});
      y += n;
    }
  }
  // row-major order (first row, then strip): the waves of a workgroup take
  // consecutive items, side by side strips of the same rows, whose halo
  // columns they then share in L2 (4096^2 Riemann stage-2 and stage-3 flux
  // 1.75 and 2.17 ms in this order, 2.18 and 2.74 ms strip by strip)
  std::stable_sort(out.begin() + first, out.end(),
                   [](const TileRef& a, const TileRef& b) { return a.ty != b.ty ? a.ty < b.ty : a.tx < b.tx; });
}

// Rows of the items that count towards the size of a launch group (far_fp64).
static constexpr int kStripBlock = 32;

// Strip columns of an instance whose cells all take the logical stencil
// addressing (none otherwise). Strip sx covers columns 58 sx .. 58 sx + 57.
// A row of a strip is solid when the region its cells' stencils read (the
// strip's 64 columns x0 - 3 .. x0 + 60 by rows y - 3 .. y + 3, each position
// mapped as the kernels map it: periodic, mirrored or clamped) holds a solid
// cell.
static void mark_strips(Solver& s) {
  s.strip_solid.clear();
  s.strip_runs.clear();
  s.strip_cols = s.strip_blocks = 0;
  if (s.any_phys) return;
  const int H = tile_halo();
  bool any_solid = false;
  for (size_t k = 0; k < s.ctype_host.size() && !any_solid; k++) any_solid = s.ctype_host[k] == 2;
  s.strip_cols = (s.nx + kStripW - 1) / kStripW;
  s.strip_solid.assign((size_t)s.strip_cols * s.ny, 0);
  if (any_solid) {
    int m;
    bool cl;
    std::vector<int> xs(64), ys(s.ny + 2 * H);
    for (int j = 0; j < s.ny + 2 * H; j++) ys[j] = ref_map(s, j - H, 1, m, cl);
    std::vector<char> rs(s.ny + 2 * H, 0);
    for (int sx = 0; sx < s.strip_cols; sx++) {
      for (int l = 0; l < 64; l++) xs[l] = ref_map(s, sx * kStripW - H + l, 0, m, cl);
      for (int j = 0; j < s.ny + 2 * H; j++) {  // mapped row j - H across the strip's columns
        bool any = false;
        for (int l = 0; l < 64 && !any; l++) any = type_at(s, xs[l], ys[j]) == 2;
        rs[j] = any;
      }
      for (int y = 0; y < s.ny; y++) {
        bool any = false;
        for (int k = 0; k <= 2 * H && !any; k++) any = rs[y + k];  // rows y - H .. y + H
        s.strip_solid[(size_t)sx * s.ny + y] = any;
      }
    }
  }
  std::vector<TileRef> items;
  strip_items(s, kStripBlock, kStripBlock, 0, items);
  s.strip_blocks = (int)items.size();
  for (int sx = 0; sx < s.strip_cols; sx++)
    for (int y = 0, n; y < s.ny; y += n) {
      const char* solid = s.strip_solid.data() + (size_t)sx * s.ny + y;
      for (n = 1; y + n < s.ny && solid[n] == solid[0]; n++) {
      }
      s.strip_runs.push_back(solid[0] ? -n : n);
    }
}

static int g_strips = 1;  // lbm_set_strips mode
bool uqlbm::strips_enabled() { return g_strips != 0; }

// FP32 storage far from its reference equilibrium: FP64 stencils in groups
// of at least 2048 items of 32 rows (3.6 million cells), where the shock
// decks run their long solves; FP32 below.
static constexpr int kFarMinBlocks = 2048;
bool uqlbm::far_fp64(int blocks) { return g_strips == 2 || blocks >= kFarMinBlocks; }

// Rows per strip item of a launch group, 1 to kStripRows: those of the least
// (n + 1) * (rows + 2), with n the workgroups of the busiest CU, `blocks` of
// them per item (three of k_strip's directions, one of four wavefronts). A
// row of the march takes the longer the more workgroups share the CU, but a
// lone one cannot fill it (stage23, items of 32 rows: 3.9, 6.3, 8.3 and 10.9 us
// per row with one to four), and the window that an item fills costs about two
// rows. Whole numbers of workgroups per CU matter as much as the length: 512^2 at
// 6 rows has 774 items, four on some CUs, at 7 rows 666, three: 110 and 99 us.
// us per step (FP64; its share of the launch that begins a sequence included) or
// launch at 1 / 2 / 4 / 8 / 16 / 32 rows, and at the rule's:
//   64^2 Couette, step           29 / 31 / 42 / 63 / 103 / 189       1: 29
//   256^2 shear, step            39 / 39 / 48 / 56 / 97 / 182        3: 40
//   512^2 shear, step            112 / 95 / 97 / 108 / 147 / 185     5: 98
//   ensemble of 48, step         2305 / 1930 / 1678 / 1555 / 1554 / 1639   12: 1550
//   3072^2 Riemann, step         4869 / 4084 / 3438 / 3174 / 3107 / 3165   32: 3165
//   512^2, FP32 k_strip          62 / 44 / 36 / 33 / 35 / 49         8: 33
//   1100^2, FP32 k_strip_mom     266 / 199 / 164 / 147 / 150 / 150   12: 141
// so the rule is within 3 % of the best of these everywhere; where it is not the
// best itself (512^2 at 2 rows, 3072^2 at 16) fewer rows do slightly better than
// the cost of a window suggests.
// Items near solids have half as many: their rows take about twice as long,
// and the launch waits for the last of them (301^2 with a block, FP64 step 79
// us with all rows, 64 with half, 64 with a third; FP32 storage 110, 91, 93).
// kCus: the compute units of an MI355X.
static constexpr int kStripRows = 32, kCus = 256;
static int solid_rows(int rows) { return (rows + 1) / 2; }
static int strip_rows(const std::vector<Solver*>& members, int blocks) {
  long long least = LLONG_MAX;
  int best = 1;
  for (int h = 1; h <= kStripRows; h++) {
    long long items = 0;
    for (const Solver* s : members)
      for (const int run : s->strip_runs)
        items += run > 0 ? (run + h - 1) / h : (solid_rows(h) - run - 1) / solid_rows(h);
    const long long cost = ((items * blocks + kCus - 1) / kCus + 1) * (h + 2);
    if (cost < least) {
      least = cost;
      best = h;
    }
  }
  return best;
}

// The fused step takes FP64 RK3 groups whose members all have strips and
// arrays within the 32-bit offsets of its buffer accesses (19 million cells);
// the others keep four launches a step. Not a matter of size otherwise: it is
// the faster one from 64^2 (29 against 41 us per step) over an ensemble of 48
// (1550, 1855) to 3072^2 (3165, 3865).
static constexpr unsigned long long kFusedMaxBytes = 0xF0000000ull;
static bool fused_instance(const Solver& s) {
  return s.precision == LBM_PREC_FP64 && s.p.rk_method == 1 && s.strip_cols > 0 &&
         (unsigned long long)s.pitch * s.ny * kPlanes * sizeof(double) <= kFusedMaxBytes;
}

uqlbm::StripLists::StripLists(const std::vector<Solver*>& members, int shape) {
  const int rows = strip_rows(members, 3);
  for (size_t k = 0; k < members.size(); k++) {
    strip_items(*members[k], rows, solid_rows(rows), (int)k, items);
    blocks += members[k]->strip_blocks;
    if (members[k]->strip_cols == 0) tiles_rest += (int)solver_tiles(*members[k], shape).size();
  }
  n = (int)items.size();
  // items of k_strip_mom, or of the fused step: four wavefronts each
  const int mrows = strip_rows(members, 1);
  fused = !members.empty();
  for (size_t k = 0; k < members.size(); k++) {
    strip_items(*members[k], mrows, solid_rows(mrows), (int)k, items);
    fused = fused && fused_instance(*members[k]);
  }
  nmom = (int)items.size() - n;
}

void uqlbm::launch_strips_of(StepLaunch& L, const TileRef* items_dev, int n, int nmom, bool fused, int blocks,
                             int tiles_rest, int ntiles) {
  if (!strips_enabled() || n == 0) {
    L.tiles_rest = ntiles;
    return;
  }
  L.strips = items_dev;
  L.nstrips = n;
  L.mstrips = items_dev + n;
  L.nmstrips = nmom;
  L.fused = fused;
  L.far64 = far_fp64(blocks);
  L.tiles_rest = tiles_rest;
}

const std::vector<TileRef>& uqlbm::solver_tiles(Solver& s, int shape) {
  if (shape < 0 || shape >= kFluxShapes) shape = 0;
  if (s.tiles_shape[shape].empty()) s.tiles_shape[shape] = build_flux_tiles(s, shape);
  return s.tiles_shape[shape];
}

// Pointwise tiles and wall cells (instance index `inst`).
static void build_lists(const Solver& s, std::vector<WallRef>& walls, std::vector<TileRef>& ptiles, int inst) {
  for (int ty = 0; ty < (s.ny + kPointH - 1) / kPointH; ty++)
    for (int tx = 0; tx < (s.nx + kPointW - 1) / kPointW; tx++) ptiles.push_back(TileRef{inst, tx, ty, 0});
  for (int y = 0; y < s.ny; y++)
    for (int x = 0; x < s.nx; x++) {
      if (type_at(s, x, y) != 2) continue;
      static const int dxs[4] = {-1, 1, 0, 0}, dys[4] = {0, 0, -1, 1};
      bool need = false;
      for (int j = 0; j < 4 && !need; j++) {
        int m;
        bool cl;
        const int xn = ref_map(s, x + dxs[j], 0, m, cl);
        const int yn = ref_map(s, y + dys[j], 1, m, cl);
        need = type_at(s, xn, yn) < 2;
      }
      if (need) walls.push_back(WallRef{inst, x, y});
    }
}

}  // namespace uqlbm

using namespace uqlbm;

extern "C" const char* lbm_last_error(void) { return g_error.c_str(); }

extern "C" int32_t lbm_device_count(void) {
  int n = 0;
  if (hipGetDeviceCount(&n) != hipSuccess) return 0;
  int usable = 0;
  for (int d = 0; d < n; d++) {
    hipDeviceProp_t p;
    if (hipGetDeviceProperties(&p, d) == hipSuccess && std::strncmp(p.gcnArchName, "gfx950", 6) == 0) usable++;
  }
  return usable;
}

extern "C" int lbm_create(const lbm_params* params, int32_t nx, int32_t ny, const int32_t* bnd, const lbm_props* props,
               int32_t precision, lbm_solver** out) {
  if (!params || !bnd || !props || !out) return fail_with(LBM_ERR_ARG, "null argument");
  *out = nullptr;
  if (nx < 4 || ny < 4) return fail_with(LBM_ERR_ARG, "grid %dx%d too small (need at least 4x4)", nx, ny);
  if (precision != LBM_PREC_FP64 && precision != LBM_PREC_MIXED)
    return fail_with(LBM_ERR_ARG, "unknown precision %d", precision);
  if (params->rk_method < 0 || params->rk_method > 3)
    return fail_with(LBM_ERR_ARG, "RKMETHOD %d unknown (0 RK1, 1 RK3, 2 EULER, 3 EULER_EQ)", params->rk_method);
  if (params->flux_method != 0 && params->flux_method != 1)
    return fail_with(LBM_ERR_ARG, "FMETHOD %d unknown", params->flux_method);
  // the relaxation times tf = mu/p and th = tf/Pr need a positive viscosity
  // and Prandtl number (the reference would divide by zero further on)
  if (!(params->mu > 0) || !(params->Pr > 0) || !std::isfinite(params->mu) || !std::isfinite(params->Pr))
    return fail_with(LBM_ERR_ARG, "mu = %g and Pr = %g must be positive", params->mu, params->Pr);
  if (props->num_props < 1 || !props->density || !props->pressure || !props->temp || !props->velocity_x ||
      !props->velocity_y || !props->cell_type)
    return fail_with(LBM_ERR_ARG, "incomplete property table");
  std::unique_ptr<Solver> s(new Solver());
  s->p = *params;
  s->nx = nx;
  s->ny = ny;
  s->precision = precision;
  s->props.resize(props->num_props);
  for (int r = 0; r < props->num_props; r++) {
    s->props[r] = {props->density[r], props->pressure[r], props->temp[r], props->velocity_x[r],
                   props->velocity_y[r], props->cell_type[r]};
    if (props->cell_type[r] < 0 || props->cell_type[r] > 2)
      return fail_with(LBM_ERR_ARG, "cellType %d of property %d out of range", props->cell_type[r], r);
  }
  refine_deck(*s);
  if (!(s->dt > 0) || !std::isfinite(s->dt)) return fail_with(LBM_ERR_ARG, "derived time step is not positive");

  // host maps in [y][x]
  s->ids_host.assign((size_t)nx * ny, 0);
  s->ctype_host.assign((size_t)nx * ny, 0);
  for (int x = 0; x < nx; x++)
    for (int y = 0; y < ny; y++) {
      const int id = bnd[(size_t)x * ny + y];
      if (id < 0 || id >= props->num_props)
        return fail_with(LBM_ERR_ARG, "bndArray(%d,%d) = %d is not a property id", x, y, id);
      s->ids_host[(size_t)y * nx + x] = id;
      s->ctype_host[(size_t)y * nx + x] = (uint8_t)s->props[id].type;
    }
  mark_physical_cells(*s);
  if (lbm_device_count() < 1) return fail_with(LBM_ERR_NOGPU, "no gfx950 device visible");

  const int align = 64;
  s->pitch = (nx + align - 1) / align * align;
  const size_t plane = (size_t)s->pitch * ny;
  const size_t es = elem_size(precision);
  HIP_TRY(hipStreamCreateWithFlags(&s->stream, hipStreamNonBlocking));
  for (void** b : {&s->state[0], &s->state[1], &s->f2, &s->f3}) HIP_TRY(solver_alloc(*s, b, plane * kPlanes * es));
  HIP_TRY(solver_alloc(*s, &s->dflux, plane * dflux_planes() * es));
  if (precision != LBM_PREC_FP64) {
    for (double** m : {&s->mom[0], &s->mom[1]}) {
      HIP_TRY(solver_alloc(*s, (void**)m, plane * 4 * sizeof(double)));
      HIP_TRY(hipMemset(*m, 0, plane * 4 * sizeof(double)));
    }
    set_reference(*s);
    s->eq32 = near_reference(*s);
  }
  HIP_TRY(solver_alloc(*s, (void**)&s->ctype, plane));
  HIP_TRY(solver_alloc(*s, (void**)&s->alpha, plane * sizeof(double)));
  HIP_TRY(solver_alloc(*s, (void**)&s->fail, sizeof(int)));
  HIP_TRY(solver_alloc(*s, (void**)&s->ids, plane * sizeof(int)));
  HIP_TRY(solver_alloc(*s, (void**)&s->props_dev, s->props.size() * 4 * sizeof(double)));
  HIP_TRY(solver_alloc(*s, (void**)&s->inst_dev, sizeof(InstDev)));
  HIP_TRY(solver_alloc(*s, (void**)&s->macro_dev, plane * 5 * sizeof(double)));
  HIP_TRY(solver_alloc(*s, (void**)&s->step_ctr, 2 * sizeof(int)));
  HIP_TRY(solver_alloc(*s, (void**)&s->fails_dev, sizeof(int)));
  s->device_bytes = solver_footprint(nx, ny, precision);

  std::vector<uint8_t> ct(plane, 2);
  std::vector<int> ids(plane, 0);
  for (int y = 0; y < ny; y++)
    for (int x = 0; x < nx; x++) {
      ct[(size_t)y * s->pitch + x] = s->ctype_host[(size_t)y * nx + x];
      ids[(size_t)y * s->pitch + x] = s->ids_host[(size_t)y * nx + x];
    }
  HIP_TRY(hipMemcpy(s->ctype, ct.data(), plane, hipMemcpyHostToDevice));
  HIP_TRY(hipMemcpy(s->ids, ids.data(), plane * sizeof(int), hipMemcpyHostToDevice));
  std::vector<double> pr(s->props.size() * 4);
  for (size_t r = 0; r < s->props.size(); r++) {
    pr[4 * r + 0] = s->props[r].rho;
    pr[4 * r + 1] = s->props[r].ux;
    pr[4 * r + 2] = s->props[r].uy;
    pr[4 * r + 3] = s->props[r].T;
  }
  HIP_TRY(hipMemcpy(s->props_dev, pr.data(), pr.size() * sizeof(double), hipMemcpyHostToDevice));
  HIP_TRY(hipMemset(s->alpha, 0, plane * sizeof(double)));
  for (void* b : {s->state[0], s->state[1], s->f2, s->f3}) HIP_TRY(hipMemset(b, 0, plane * kPlanes * es));
  HIP_TRY(hipMemset(s->dflux, 0, plane * dflux_planes() * es));

  std::vector<WallRef> walls;
  std::vector<TileRef> ptiles;
  build_lists(*s, walls, ptiles, 0);
  s->flux_shape = default_flux_shape(precision);
  const std::vector<TileRef>& tiles = solver_tiles(*s, s->flux_shape);
  s->ntiles = (int)tiles.size();
  s->nphys = count_physical(tiles);
  s->nwalls = (int)walls.size();
  s->nptiles = (int)ptiles.size();
  HIP_TRY(solver_alloc(*s, (void**)&s->ptiles_dev, ptiles.size() * sizeof(TileRef)));
  HIP_TRY(hipMemcpy(s->ptiles_dev, ptiles.data(), ptiles.size() * sizeof(TileRef), hipMemcpyHostToDevice));
  HIP_TRY(solver_alloc(*s, (void**)&s->tiles_dev, tiles.size() * sizeof(TileRef)));
  HIP_TRY(hipMemcpy(s->tiles_dev, tiles.data(), tiles.size() * sizeof(TileRef), hipMemcpyHostToDevice));
  if (!walls.empty()) {
    HIP_TRY(solver_alloc(*s, (void**)&s->walls_dev, walls.size() * sizeof(WallRef)));
    HIP_TRY(hipMemcpy(s->walls_dev, walls.data(), walls.size() * sizeof(WallRef), hipMemcpyHostToDevice));
  }
  s->walls_host = std::move(walls);
  s->ptiles_host = std::move(ptiles);
  mark_strips(*s);
  const StripLists strips({s.get()}, s->flux_shape);
  s->nstrips = strips.n;
  s->nmstrips = strips.nmom;
  s->fused = strips.fused;
  if (s->nstrips) {
    HIP_TRY(solver_alloc(*s, (void**)&s->strips_dev, strips.items.size() * sizeof(TileRef)));
    HIP_TRY(hipMemcpy(s->strips_dev, strips.items.data(), strips.items.size() * sizeof(TileRef), hipMemcpyHostToDevice));
  }
  const int st = upload_inst(*s);
  if (st != LBM_OK) return st;
  *out = reinterpret_cast<lbm_solver*>(s.release());
  return LBM_OK;
}

extern "C" int lbm_init(lbm_solver* h) {
  if (!h) return fail_with(LBM_ERR_ARG, "null solver");
  Solver& s = *reinterpret_cast<Solver*>(h);
  s.cur = 0;
  s.step = 0;
  int st = upload_inst(s);
  if (st != LBM_OK) return st;
  const int none = INT_MAX;
  HIP_TRY(hipMemcpyAsync(s.fail, &none, sizeof(int), hipMemcpyHostToDevice, s.stream));
  const long long cells = (long long)s.pitch * s.ny;
  if (s.precision == LBM_PREC_FP64) launch_init<double>(s.inst_dev, 0, s.ids, s.props_dev, cells, s.stream);
  else launch_init<float>(s.inst_dev, 0, s.ids, s.props_dev, cells, s.stream);
  HIP_TRY(hipGetLastError());
  HIP_TRY(hipStreamSynchronize(s.stream));
  s.inited = true;
  return LBM_OK;
}

// Refresh the solver's own instance record (current buffer, step base) on
// its stream; later work on that stream sees it in order.
int uqlbm::upload_inst(Solver& s) {
  fill_inst(s, s.inst_host);
  launch_put_inst(s.inst_host, s.inst_dev, nullptr, nullptr, s.stream);
  HIP_TRY(hipGetLastError());
  return LBM_OK;
}

// Steps of a captured fused graph.
static constexpr int kFusedGraph = 8;

static void launch_steps(const StepLaunch& L, int precision, hipStream_t stream, int nsteps,
                         KernelTimer* tm) {
  for (int k = 0; k < nsteps; k++) {
    const int par = k & 1;
    if (precision == LBM_PREC_FP64) launch_step<double, double>(L, stream, par, tm);
    else launch_step<float, float>(L, stream, par, tm);
  }
}

// HIP graph replay of the step sequence (on unless lbm_set_graphs(0)).
static bool g_graphs_enabled = true;

// Flux tile shape used by solvers, batches and servers created from now on,
// per precision: set by lbm_set_flux_shape or by the autotuner.
static int g_flux_shape[2] = {0, 0};

int uqlbm::default_flux_shape(int precision) { return g_flux_shape[precision == LBM_PREC_FP64 ? 0 : 1]; }

static int capture_steps(const StepLaunch& L, int precision, hipStream_t stream, int nsteps,
                         hipGraphExec_t* out) {
  hipGraph_t g = nullptr;
  HIP_TRY(hipStreamBeginCapture(stream, hipStreamCaptureModeThreadLocal));
  launch_steps(L, precision, stream, nsteps, nullptr);
  const hipError_t e = hipStreamEndCapture(stream, &g);
  if (e != hipSuccess) return fail_with(LBM_ERR_HIP, "stream capture: %s", hipGetErrorString(e));
  const hipError_t e2 = hipGraphInstantiate(out, g, nullptr, nullptr, 0);
  (void)hipGraphDestroy(g);
  if (e2 != hipSuccess) return fail_with(LBM_ERR_HIP, "graph instantiate: %s", hipGetErrorString(e2));
  return LBM_OK;
}

// n steps of the fused step: the first step's f2 from the state, then steps
// that keep the state in f2 (through a cached graph of kFusedGraph of them
// where `gc` is given and the sequence is long enough), and the last two,
// which write the state.
static int fused_steps(GraphCache* gc, const StepLaunch& L, hipStream_t stream, int n, KernelTimer* tm) {
  launch_fused_begin(L, stream, tm);
  int left = n - 2;
  if (gc && left >= kFusedGraph) {
    if (gc->precision != LBM_PREC_FP64 || !same_launch(gc->key, L)) {
      gc->clear();
      hipGraph_t g = nullptr;
      HIP_TRY(hipStreamBeginCapture(stream, hipStreamCaptureModeThreadLocal));
      for (int k = 0; k < kFusedGraph; k++) launch_fused_step(L, stream, false, true, nullptr);
      const hipError_t e = hipStreamEndCapture(stream, &g);
      if (e != hipSuccess) return fail_with(LBM_ERR_HIP, "stream capture: %s", hipGetErrorString(e));
      const hipError_t e2 = hipGraphInstantiate(&gc->two, g, nullptr, nullptr, 0);
      (void)hipGraphDestroy(g);
      if (e2 != hipSuccess) {
        gc->clear();
        return fail_with(LBM_ERR_HIP, "graph instantiate: %s", hipGetErrorString(e2));
      }
      gc->key = L;
      gc->precision = LBM_PREC_FP64;
    }
    for (; left >= kFusedGraph; left -= kFusedGraph) HIP_TRY(hipGraphLaunch(gc->two, stream));
  }
  for (; left > 0; left--) launch_fused_step(L, stream, false, true, tm);
  if (n > 1) launch_fused_step(L, stream, true, true, tm);
  launch_fused_step(L, stream, true, false, tm);
  return LBM_OK;
}

// n steps of L through the cached graphs (captured on first use or when L
// changed): the two-step graph n/2 times, then the one-step graph.
static int replay_steps(GraphCache& gc, const StepLaunch& L, int precision, hipStream_t stream, int n) {
  if (gc.precision != precision || !same_launch(gc.key, L)) {
    gc.clear();
    prepare_launch(precision == LBM_PREC_FP64);
    int st = capture_steps(L, precision, stream, 2, &gc.two);
    if (st == LBM_OK) st = capture_steps(L, precision, stream, 1, &gc.one);
    if (st != LBM_OK) {
      gc.clear();
      return st;
    }
    gc.key = L;
    gc.precision = precision;
  }
  for (int k = 0; k + 1 < n; k += 2) HIP_TRY(hipGraphLaunch(gc.two, stream));
  if (n & 1) HIP_TRY(hipGraphLaunch(gc.one, stream));
  return LBM_OK;
}

static KernelTimer* active_timer() {
  if (!g_timing_enabled) return nullptr;
  if (!g_timer) {
    g_timer = new KernelTimer();
    g_timer->set_names({"s12", "alpha", "flux2", "s3", "flux3"});
  }
  return g_timer;
}

static void record_timing(double total_ms, KernelTimer* tm) {
  g_last_timing = lbm_timing{};
  g_last_timing.total_ms = total_ms;
  if (tm) {
    tm->collect();
    const auto& names = tm->names();
    g_last_timing.n_kernels = (int)names.size();
    for (size_t k = 0; k < names.size() && k < 8; k++) {
      std::snprintf(g_last_timing.names[k], 32, "%s", names[k].c_str());
      g_last_timing.avg_ms[k] = tm->avg_ms((int)k);
      g_last_timing.launches[k] = tm->count((int)k);
    }
    tm->reset();
  }
}

// Advance every member of a group by n steps with batched launches: upload
// the instance table (current buffer, step base), launch, gather every
// member's failure step into fails_dev and read them with one copy, then
// account each member's steps, stopping a member at its failing step
// (reference main loop stop on runOne failure, main.cpp:21,56,73). With
// `graphs` null the kernels are launched directly; with `timed` the call's
// device time is recorded (lbm_get_timing). A lone solver with `result` gets
// its failure step and, where `resid_rows` is given (ny doubles), its residual
// there instead: one wait and no copies for the whole call.
int uqlbm::run_group(const std::vector<Solver*>& members, InstDev* table_dev, const StepLaunch& L, int precision,
                     hipStream_t stream, int n, GraphCache* graphs, int* fails_dev, bool timed, StepResult* result,
                     double* resid_rows) {
  static const int kFirstStep = 1;
  std::vector<InstDev> table(members.size());
  int ptile0 = 0;
  for (size_t k = 0; k < members.size(); k++) {
    fill_inst(*members[k], table[k]);
    table[k].res_hist = members[k]->res_hist;
    table[k].res_last = members[k]->step + n;
    table[k].ptile0 = ptile0;
    table[k].nptiles = members[k]->nptiles;
    table[k].strips = L.nstrips > 0 && members[k]->strip_cols > 0 ? 1 : 0;
    ptile0 += members[k]->nptiles;
  }
  if (table.size() == 1) {
    launch_put_inst(table[0], table_dev, L.step_ctr, result ? &result->begin : nullptr, stream);
  } else {
    HIP_TRY(hipMemcpyAsync(table_dev, table.data(), table.size() * sizeof(InstDev), hipMemcpyHostToDevice, stream));
    HIP_TRY(hipMemcpyAsync(L.step_ctr, &kFirstStep, sizeof(int), hipMemcpyHostToDevice, stream));
  }
  KernelTimer* tm = timed ? active_timer() : nullptr;
  hipEvent_t e0 = nullptr, e1 = nullptr;
  const bool events = timed && !result;  // a lone solver's first and last launch read the clock
  if (events) {
    HIP_TRY(hipEventCreate(&e0));
    HIP_TRY(hipEventCreate(&e1));
    HIP_TRY(hipEventRecord(e0, stream));
  }
  // per-step residuals need every step's state: four launches per step then
  const bool fused = L.fused && !L.res_partial;
  const bool replay = graphs && g_graphs_enabled && !tm;
  if (fused || replay) {
    const int st = fused ? fused_steps(replay ? graphs : nullptr, L, stream, n, tm)
                         : replay_steps(*graphs, L, precision, stream, n);
    if (st != LBM_OK) {
      (void)hipStreamSynchronize(stream);
      return st;
    }
  } else {
    launch_steps(L, precision, stream, n, tm);
  }
  if (events) HIP_TRY(hipEventRecord(e1, stream));
  std::vector<int> fail_step(members.size(), INT_MAX);
  if (result) {
    Solver& s = *members[0];
    launch_gather_fail(table_dev, 1, &result->fail, &result->end, stream);
    if (resid_rows) {  // the previous state is still in the other state buffer
      if (precision == LBM_PREC_FP64)
        launch_residual<double>(table_dev, 0, n, resid_rows, &result->residual, s.nx, s.ny, stream);
      else
        launch_residual<float>(table_dev, 0, n, resid_rows, &result->residual, s.nx, s.ny, stream);
    }
  } else {
    launch_gather_fail(table_dev, (int)members.size(), fails_dev, nullptr, stream);
    HIP_TRY(hipMemcpyAsync(fail_step.data(), fails_dev, fail_step.size() * sizeof(int), hipMemcpyDeviceToHost,
                           stream));
  }
  HIP_TRY(hipGetLastError());
  HIP_TRY(hipStreamSynchronize(stream));
  if (result) fail_step[0] = result->fail;
  if (events) {
    float ms = 0;
    HIP_TRY(hipEventElapsedTime(&ms, e0, e1));
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    record_timing(ms, tm);
  } else if (timed) {
    int dev = 0, khz = 0;
    HIP_TRY(hipGetDevice(&dev));
    HIP_TRY(hipDeviceGetAttribute(&khz, hipDeviceAttributeWallClockRate, dev));
    record_timing((double)(result->end - result->begin) / khz, tm);
  }
  int status = LBM_OK;
  for (size_t k = 0; k < members.size(); k++) {
    Solver* s = members[k];
    if (fail_step[k] != INT_MAX) {
      const int taken = std::max(0, fail_step[k] - s->step);
      // the fused step leaves the state of a failing inner step beside the sequence's first state
      s->cur ^= fused && taken < n ? taken > 0 : taken & 1;
      s->step += taken;
      s->failed = true;
      status = LBM_FAILED;
    } else {
      s->cur ^= n & 1;
      s->step += n;
    }
  }
  return status;
}

// n steps of a lone solver, as run_group. A residual compares the states of the
// last two steps taken; where the fused step fails at an inner step of the
// sequence, the state before that step was never written, and the sequence,
// whose first state is still there, is taken again with its end there: up to
// the step before (which the last steps of a sequence write), then the failing
// step alone. The same values either way, so only a failing call pays for it.
static int lone_step(Solver& s, const StepLaunch& L, int n, GraphCache* graphs, bool timed, bool resid,
                     StepResult* result, double* rows) {
  const std::vector<Solver*> one{&s};
  const int cur = s.cur, step = s.step;
  if (!resid) rows = nullptr;
  const int st = run_group(one, s.inst_dev, L, s.precision, s.stream, n, graphs, s.fails_dev, timed, result, rows);
  const int taken = s.step - step;
  if (st != LBM_FAILED || !resid || !L.fused || taken <= 1 || taken >= n) return st;
  static const int none = INT_MAX;
  HIP_TRY(hipMemcpyAsync(s.fail, &none, sizeof(int), hipMemcpyHostToDevice, s.stream));
  s.cur = cur;
  s.step = step;
  s.failed = false;
  const int before = run_group(one, s.inst_dev, L, s.precision, s.stream, taken - 1, graphs, s.fails_dev, false, result);
  if (before != LBM_OK) return before;
  return run_group(one, s.inst_dev, L, s.precision, s.stream, 1, graphs, s.fails_dev, false, result, rows);
}

// Residual of the solver's last step on the device (cpuLBM.cpp:2322-2331),
// after the call's steps: `rows` holds ny + 1 doubles; the result is copied to
// *out.
static int device_residual(Solver& s, double* rows, double* out) {
  if (s.precision == LBM_PREC_FP64) launch_residual<double>(s.inst_dev, 0, 0, rows, rows + s.ny, s.nx, s.ny, s.stream);
  else launch_residual<float>(s.inst_dev, 0, 0, rows, rows + s.ny, s.nx, s.ny, s.stream);
  HIP_TRY(hipGetLastError());
  HIP_TRY(hipMemcpyAsync(out, rows + s.ny, sizeof(double), hipMemcpyDeviceToHost, s.stream));
  HIP_TRY(hipStreamSynchronize(s.stream));
  return LBM_OK;
}

extern "C" int lbm_step(lbm_solver* h, int32_t nsteps, int32_t want_residual, double* residual_out) {
  if (!h) return fail_with(LBM_ERR_ARG, "null solver");
  Solver& s = *reinterpret_cast<Solver*>(h);
  if (!s.inited) return fail_with(LBM_ERR_STATE, "lbm_step before lbm_init");
  if (nsteps < 0) return fail_with(LBM_ERR_ARG, "negative step count");
  if (s.failed) return LBM_FAILED;
  if (nsteps == 0) return LBM_OK;
  StepLaunch L{s.inst_dev,    s.tiles_dev, s.ntiles,      s.walls_dev, s.nwalls,
               s.ptiles_dev, s.nptiles,   s.p.rk_method, s.step_ctr,  s.flux_shape};
  L.nphys = s.nphys;
  launch_strips_of(L, s.strips_dev, s.nstrips, s.nmstrips, s.fused, s.strip_blocks, 0, s.ntiles);
  L.eq_kinds = s.precision == LBM_PREC_FP64 ? 1 : (s.eq32 ? 2 : 1);
  const bool resid = want_residual && residual_out;
  if (!s.result && hipHostMalloc((void**)&s.result, sizeof(StepResult), hipHostMallocDefault) != hipSuccess) {
    s.result = nullptr;  // no pinned memory to be had: the results are copied
    (void)hipGetLastError();
  }
  if (resid && !s.resid_dev) HIP_TRY(solver_alloc(s, (void**)&s.resid_dev, ((size_t)s.ny + 1) * sizeof(double)));
  const int st = lone_step(s, L, nsteps, s.graphs.get(), true, resid, s.result, s.resid_dev);
  const int st2 = upload_inst(s);
  if (st < 0) return st;
  if (st2 != LBM_OK) return st2;
  if (resid && s.result) *residual_out = s.result->residual;
  if (resid && !s.result) {
    const int st3 = device_residual(s, s.resid_dev, residual_out);
    if (st3 != LBM_OK) return st3;
  }
  return st;
}

// ---------------------------------------------------------------------------
// Stepping without allocation (lbm_step_noalloc): the residual's row sums
// live in a file-scope device array instead of the solver's lazily
// allocated buffer, the kernels are launched directly (no graph capture or
// instantiation) and no events are created. Host code never passes the
// array's name to a kernel: its device address is looked up once per device
// (hipGetSymbolAddress, with that device current) and that pointer is used.
// Every call on one GPU shares that GPU's array; calls that overlap on one
// GPU race for it. Nothing in it needs clearing: every call writes each row
// sum it later reads.
// ---------------------------------------------------------------------------
constexpr int kNoAllocMaxRows = 32768;  // grid rows (ny) the array serves: 256 KiB of doubles
static __device__ __align__(256) double scratch[kNoAllocMaxRows + 1];

constexpr int kMaxDevices = 64;
static std::mutex g_scratch_mu;
static double* g_scratch_ptr[kMaxDevices] = {};

static int scratch_on_current_device(double** out) {
  int dev = 0;
  HIP_TRY(hipGetDevice(&dev));
  if (dev < 0 || dev >= kMaxDevices) return fail_with(LBM_ERR_ARG, "device %d beyond the supported %d", dev, kMaxDevices);
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (!g_scratch_ptr[dev]) {
    void* ptr = nullptr;
    const hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !ptr)
      return fail_with(LBM_ERR_HIP, "hipGetSymbolAddress(scratch) on device %d: %s", dev, hipGetErrorString(e));
    g_scratch_ptr[dev] = reinterpret_cast<double*>(ptr);
  }
  *out = g_scratch_ptr[dev];
  return LBM_OK;
}

extern "C" int lbm_step_noalloc(lbm_solver* h, int32_t nsteps, int32_t want_residual, double* residual_out) {
  if (!h) return fail_with(LBM_ERR_ARG, "null solver");
  Solver& s = *reinterpret_cast<Solver*>(h);
  if (!s.inited) return fail_with(LBM_ERR_STATE, "lbm_step_noalloc before lbm_init");
  if (nsteps < 0) return fail_with(LBM_ERR_ARG, "negative step count");
  if (want_residual && s.ny > kNoAllocMaxRows)
    return fail_with(LBM_ERR_ARG, "lbm_step_noalloc: the residual serves grids of at most %d rows, this one has %d",
                     kNoAllocMaxRows, s.ny);
  double* rows = nullptr;
  if (want_residual) {
    const int st = scratch_on_current_device(&rows);
    if (st != LBM_OK) return st;
  }
  if (s.failed) return LBM_FAILED;
  if (nsteps == 0) return LBM_OK;
  StepLaunch L{s.inst_dev,    s.tiles_dev, s.ntiles,      s.walls_dev, s.nwalls,
               s.ptiles_dev, s.nptiles,   s.p.rk_method, s.step_ctr,  s.flux_shape};
  L.nphys = s.nphys;
  launch_strips_of(L, s.strips_dev, s.nstrips, s.nmstrips, s.fused, s.strip_blocks, 0, s.ntiles);
  L.eq_kinds = s.precision == LBM_PREC_FP64 ? 1 : (s.eq32 ? 2 : 1);
  prepare_launch(s.precision == LBM_PREC_FP64);
  const int st = lone_step(s, L, nsteps, nullptr, false, want_residual && residual_out, nullptr, nullptr);
  const int st2 = upload_inst(s);
  if (st < 0) return st;
  if (st2 != LBM_OK) return st2;
  if (want_residual && residual_out) {
    const int st3 = device_residual(s, rows, residual_out);
    if (st3 != LBM_OK) return st3;
  }
  return st;
}

extern "C" int lbm_get_macro(lbm_solver* h, double* rho, double* ux, double* uy, double* p, double* T) {
  if (!h) return fail_with(LBM_ERR_ARG, "null solver");
  Solver& s = *reinterpret_cast<Solver*>(h);
  if (!s.inited) return fail_with(LBM_ERR_STATE, "lbm_get_macro before lbm_init");
  if (s.precision == LBM_PREC_FP64) launch_macro<double>(s.inst_dev, 0, 0, s.macro_dev, s.nx, s.ny, s.stream);
  else launch_macro<float>(s.inst_dev, 0, 0, s.macro_dev, s.nx, s.ny, s.stream);
  HIP_TRY(hipGetLastError());
  const size_t field = (size_t)s.nx * s.ny * sizeof(double);
  HIP_TRY(staged_copy((char*)s.macro_dev, {{rho, field}, {ux, field}, {uy, field}, {p, field}, {T, field}}, true,
                      s.stream));
  return LBM_OK;
}

extern "C" int lbm_get_totals(lbm_solver* h, double* out) {
  if (!h || !out) return fail_with(LBM_ERR_ARG, "null argument");
  Solver& s = *reinterpret_cast<Solver*>(h);
  if (!s.inited) return fail_with(LBM_ERR_STATE, "lbm_get_totals before lbm_init");
  if (!s.totals_dev) HIP_TRY(solver_alloc(s, (void**)&s.totals_dev, totals_scratch_doubles() * sizeof(double)));
  const long long cells = (long long)s.pitch * s.ny;
  if (s.precision == LBM_PREC_FP64) launch_totals<double>(s.inst_dev, 0, 0, s.totals_dev, cells, s.stream);
  else launch_totals<float>(s.inst_dev, 0, 0, s.totals_dev, cells, s.stream);
  HIP_TRY(hipGetLastError());
  HIP_TRY(hipMemcpyAsync(out, s.totals_dev + totals_scratch_doubles() - 4, 4 * sizeof(double),
                         hipMemcpyDeviceToHost, s.stream));
  HIP_TRY(hipStreamSynchronize(s.stream));
  return LBM_OK;
}

// Distributions at the boundary: transposed on the device into (out of) the
// stage buffers f2 and f3, which hold nothing between step calls (each has
// 13 doubles per cell in both storage types), and copied from (to) there.
static int get_dist(Solver& s, double* f, double* h) {
  double *df = (double*)s.f2, *dh = (double*)s.f3;
  launch_dist_out(s, f ? df : nullptr, h ? dh : nullptr);
  HIP_TRY(hipGetLastError());
  const size_t bytes = (size_t)s.nx * s.ny * kQ * sizeof(double);
  if (f) HIP_TRY(staged_copy((char*)df, {{f, bytes}}, true, s.stream));
  if (h) HIP_TRY(staged_copy((char*)dh, {{h, bytes}}, true, s.stream));
  HIP_TRY(hipStreamSynchronize(s.stream));
  return LBM_OK;
}

static int set_dist(Solver& s, const double* f, const double* h) {
  double *df = (double*)s.f2, *dh = (double*)s.f3;
  const size_t bytes = (size_t)s.nx * s.ny * kQ * sizeof(double);
  if (f) HIP_TRY(staged_copy((char*)df, {{const_cast<double*>(f), bytes}}, false, s.stream));
  if (h) HIP_TRY(staged_copy((char*)dh, {{const_cast<double*>(h), bytes}}, false, s.stream));
  launch_dist_in(s, f ? df : nullptr, h ? dh : nullptr);
  HIP_TRY(hipGetLastError());
  HIP_TRY(hipStreamSynchronize(s.stream));
  return LBM_OK;
}

extern "C" int lbm_get_dist(lbm_solver* h, double* f, double* hh) {
  if (!h) return fail_with(LBM_ERR_ARG, "null solver");
  Solver& s = *reinterpret_cast<Solver*>(h);
  if (!s.inited) return fail_with(LBM_ERR_STATE, "lbm_get_dist before lbm_init");
  return get_dist(s, f, hh);
}

extern "C" int lbm_set_dist(lbm_solver* h, const double* f, const double* hh) {
  if (!h) return fail_with(LBM_ERR_ARG, "null solver");
  Solver& s = *reinterpret_cast<Solver*>(h);
  if (!s.inited) return fail_with(LBM_ERR_STATE, "lbm_set_dist before lbm_init");
  return set_dist(s, f, hh);
}

extern "C" int lbm_get_info(const lbm_solver* h, lbm_info* out) {
  if (!h || !out) return fail_with(LBM_ERR_ARG, "null argument");
  const Solver& s = *reinterpret_cast<const Solver*>(h);
  *out = lbm_info{};
  out->nx = s.nx;
  out->ny = s.ny;
  out->nsteps = s.nsteps;
  out->step = s.step;
  out->dt = s.dt;
  out->c = s.c;
  out->Tc = s.Tc;
  out->b = s.b;
  out->K = s.K;
  out->dx = s.p.dx;
  out->dy = s.p.dy;
  out->tstep = s.step * s.dt;
  out->precision = s.precision;
  out->halo = tile_halo();
  out->device_bytes = s.device_bytes;
  return LBM_OK;
}

// A solver still held by a batch is freed when its last batch is destroyed
// (the batch keeps stepping it meanwhile); otherwise at once.
extern "C" void lbm_destroy(lbm_solver* h) {
  Solver* s = reinterpret_cast<Solver*>(h);
  if (!s) return;
  if (s->batch_refs > 0) s->destroy_pending = true;
  else delete s;
}

extern "C" int lbm_set_viscosity(lbm_solver* h, int32_t model, double mu_ref, double T_ref, double param) {
  if (!h) return fail_with(LBM_ERR_ARG, "null solver");
  if (model < 0 || model > 2) return fail_with(LBM_ERR_ARG, "unknown viscosity law %d", model);
  if (model > 0 && !(mu_ref > 0 && T_ref > 0 && std::isfinite(mu_ref) && std::isfinite(T_ref) && std::isfinite(param)))
    return fail_with(LBM_ERR_ARG, "viscosity law needs positive mu_ref and T_ref");
  if (model == 2 && !(param >= 0)) return fail_with(LBM_ERR_ARG, "Sutherland constant must be >= 0");
  Solver& s = *reinterpret_cast<Solver*>(h);
  s.visc_model = model;
  s.mu_ref = mu_ref;
  s.T_ref_v = T_ref;
  s.visc_param = param;
  return upload_inst(s);
}

// Non-uniform grid spacing after the OpenCL front end (PY/codeCL.py:611-618,
// 676-679): face fluxes weighted by their face length and the net divided by
// the cell area, i.e. cFLUX with the cell's own dt/dx[x] and dt/dy[y] (the
// two cells of a face share its length); dt from the smallest spacing
// (PY/LBM.py:216), nsteps recomputed. Walls keep the C++ closure
// (cpuLBM.cpp:1502-1590) with the front end's face-length weights, which is
// the C++ balance with the wall cell's own dx, dy. Before the first step.
extern "C" int lbm_set_spacing(lbm_solver* h, const double* dx, const double* dy) {
  if (!h || !dx || !dy) return fail_with(LBM_ERR_ARG, "null argument");
  Solver& s = *reinterpret_cast<Solver*>(h);
  if (s.step != 0) return fail_with(LBM_ERR_STATE, "spacing must be set before the first step");
  for (int x = 0; x < s.nx; x++)
    if (!(dx[x] > 0) || !std::isfinite(dx[x])) return fail_with(LBM_ERR_ARG, "dx[%d] is not positive", x);
  for (int y = 0; y < s.ny; y++)
    if (!(dy[y] > 0) || !std::isfinite(dy[y])) return fail_with(LBM_ERR_ARG, "dy[%d] is not positive", y);
  s.dxs.assign(dx, dx + s.nx);
  s.dys.assign(dy, dy + s.ny);
  const double mn = std::min(*std::min_element(s.dxs.begin(), s.dxs.end()),
                             *std::min_element(s.dys.begin(), s.dys.end()));
  if (s.p.dtau == 0) {
    s.dt = (s.p.cfl * mn) / (2 * s.c);
    steps_from_dt(s);
  }
  // [dt/dx (nx) | dt/dy (ny) | dx (nx) | dy (ny)]
  std::vector<double> r(2 * (s.nx + s.ny));
  for (int x = 0; x < s.nx; x++) r[x] = s.dt / s.dxs[x];
  for (int y = 0; y < s.ny; y++) r[s.nx + y] = s.dt / s.dys[y];
  for (int x = 0; x < s.nx; x++) r[s.nx + s.ny + x] = s.dxs[x];
  for (int y = 0; y < s.ny; y++) r[2 * s.nx + s.ny + y] = s.dys[y];
  if (!s.spacing_dev) HIP_TRY(solver_alloc(s, (void**)&s.spacing_dev, r.size() * sizeof(double)));
  HIP_TRY(hipMemcpy(s.spacing_dev, r.data(), r.size() * sizeof(double), hipMemcpyHostToDevice));
  return upload_inst(s);
}

extern "C" int lbm_set_kernel_timing(int32_t enable) {
  g_timing_enabled = enable != 0;
  return LBM_OK;
}

extern "C" int lbm_set_strips(int32_t mode) {
  if (mode < 0 || mode > 2) return fail_with(LBM_ERR_ARG, "strip mode must be 0, 1 or 2");
  g_strips = mode;
  return LBM_OK;
}

extern "C" int lbm_set_graphs(int32_t enable) {
  g_graphs_enabled = enable != 0;
  return LBM_OK;
}

extern "C" int lbm_get_timing(lbm_timing* out) {
  if (!out) return fail_with(LBM_ERR_ARG, "null argument");
  *out = g_last_timing;
  return LBM_OK;
}

extern "C" double lbm_clock_s(void) {
  using namespace std::chrono;
  return duration<double>(steady_clock::now().time_since_epoch()).count();
}

// ---------------------------------------------------------------------------
// batches
// ---------------------------------------------------------------------------
extern "C" int lbm_batch_create(lbm_solver* const* members, int32_t n, lbm_batch** out) {
  if (!members || n < 1 || !out) return fail_with(LBM_ERR_ARG, "bad batch arguments");
  *out = nullptr;
  std::unique_ptr<Batch> b(new Batch());
  for (int k = 0; k < n; k++) {
    Solver* s = reinterpret_cast<Solver*>(members[k]);
    if (!s || !s->inited) return fail_with(LBM_ERR_STATE, "batch member %d not initialised", k);
    if (k && (s->precision != b->precision || s->p.rk_method != b->rk_method))
      return fail_with(LBM_ERR_ARG, "batch members differ in precision or RK method");
    b->precision = s->precision;
    b->rk_method = s->p.rk_method;
    b->members.push_back(s);
    s->batch_refs++;  // released by ~Batch, also when creation fails below
  }
  return batch_finish(*b, out);
}

// Uploads the batch's flux tile list for `shape` (members' tiles with their
// batch index).
int uqlbm::batch_set_shape(Batch& b, int shape) {
  std::vector<TileRef> tiles;
  for (size_t k = 0; k < b.members.size(); k++)
    for (TileRef t : solver_tiles(*b.members[k], shape)) {
      t.inst = (int)k;
      tiles.push_back(t);
    }
  if (b.tiles_dev) HIP_TRY(hipFree(b.tiles_dev));
  b.tiles_dev = nullptr;
  HIP_TRY(hipMalloc((void**)&b.tiles_dev, tiles.size() * sizeof(TileRef)));
  HIP_TRY(hipMemcpy(b.tiles_dev, tiles.data(), tiles.size() * sizeof(TileRef), hipMemcpyHostToDevice));
  b.ntiles = (int)tiles.size();
  b.nphys = count_physical(tiles);
  b.tiles_rest = 0;
  for (Solver* m : b.members)
    if (m->strip_cols == 0) b.tiles_rest += (int)solver_tiles(*m, shape).size();
  b.eq_kinds = eq_kinds_of(b.precision == LBM_PREC_FP64, b.members.begin(), b.members.end(),
                           [](const Solver* m) { return m->eq32; });
  b.flux_shape = shape;
  return LBM_OK;
}

int uqlbm::batch_finish(Batch& b, lbm_batch** out) {
  std::vector<WallRef> walls;
  std::vector<TileRef> ptiles;
  for (size_t k = 0; k < b.members.size(); k++) {
    for (TileRef t : b.members[k]->ptiles_host) {
      t.inst = (int)k;
      ptiles.push_back(t);
    }
    for (WallRef w : b.members[k]->walls_host) {
      w.inst = (int)k;
      walls.push_back(w);
    }
  }
  b.nwalls = (int)walls.size();
  b.nptiles = (int)ptiles.size();
  HIP_TRY(hipStreamCreateWithFlags(&b.stream, hipStreamNonBlocking));
  HIP_TRY(hipMalloc((void**)&b.inst_dev, b.members.size() * sizeof(InstDev)));
  HIP_TRY(hipMalloc((void**)&b.step_ctr, 2 * sizeof(int)));
  HIP_TRY(hipMalloc((void**)&b.fails_dev, b.members.size() * sizeof(int)));
  int st = batch_set_shape(b, default_flux_shape(b.precision));
  if (st != LBM_OK) return st;
  if (!walls.empty()) {
    HIP_TRY(hipMalloc((void**)&b.walls_dev, walls.size() * sizeof(WallRef)));
    HIP_TRY(hipMemcpy(b.walls_dev, walls.data(), walls.size() * sizeof(WallRef), hipMemcpyHostToDevice));
  }
  HIP_TRY(hipMalloc((void**)&b.ptiles_dev, ptiles.size() * sizeof(TileRef)));
  HIP_TRY(hipMemcpy(b.ptiles_dev, ptiles.data(), ptiles.size() * sizeof(TileRef), hipMemcpyHostToDevice));
  const StripLists strips(b.members, b.flux_shape);
  b.nstrips = strips.n;
  b.nmstrips = strips.nmom;
  b.fused = strips.fused;
  b.strip_blocks = strips.blocks;
  b.tiles_rest = strips.tiles_rest;
  if (b.nstrips) {
    HIP_TRY(hipMalloc((void**)&b.strips_dev, strips.items.size() * sizeof(TileRef)));
    HIP_TRY(hipMemcpy(b.strips_dev, strips.items.data(), strips.items.size() * sizeof(TileRef), hipMemcpyHostToDevice));
  }
  *out = reinterpret_cast<lbm_batch*>(new Batch(std::move(b)));
  return LBM_OK;
}

uqlbm::Batch::~Batch() {
  if (graphs) graphs->clear();
  for (Solver* s : members)
    if (--s->batch_refs == 0 && s->destroy_pending) delete s;
  for (void* p : {(void*)inst_dev, (void*)tiles_dev, (void*)walls_dev, (void*)ptiles_dev, (void*)step_ctr,
                  (void*)fails_dev, (void*)strips_dev})
    if (p) (void)hipFree(p);
  if (stream) (void)hipStreamDestroy(stream);
}

int uqlbm::batch_step(Batch& b, int nsteps) {
  StepLaunch L{b.inst_dev,    b.tiles_dev, b.ntiles,    b.walls_dev, b.nwalls,
               b.ptiles_dev, b.nptiles,   b.rk_method, b.step_ctr,  b.flux_shape};
  L.nphys = b.nphys;
  L.eq_kinds = b.eq_kinds;
  launch_strips_of(L, b.strips_dev, b.nstrips, b.nmstrips, b.fused, b.strip_blocks, b.tiles_rest, b.ntiles);
  int st = run_group(b.members, b.inst_dev, L, b.precision, b.stream, nsteps, b.graphs.get(), b.fails_dev, true);
  for (Solver* s : b.members) {
    int st2 = upload_inst(*s);
    if (st2 != LBM_OK) return st2;
  }
  return st;
}

extern "C" int lbm_batch_step(lbm_batch* hb, int32_t nsteps) {
  if (!hb) return fail_with(LBM_ERR_ARG, "null batch");
  if (nsteps < 0) return fail_with(LBM_ERR_ARG, "negative step count");
  if (nsteps == 0) return LBM_OK;
  return batch_step(*reinterpret_cast<Batch*>(hb), nsteps);
}

extern "C" void lbm_batch_destroy(lbm_batch* b) { delete reinterpret_cast<Batch*>(b); }

extern "C" int lbm_set_flux_shape(int32_t precision, int32_t shape) {
  if (precision != LBM_PREC_FP64 && precision != LBM_PREC_MIXED) return fail_with(LBM_ERR_ARG, "unknown precision");
  if (shape < 0 || shape >= kFluxShapes) return fail_with(LBM_ERR_ARG, "flux tile shape %d out of range", shape);
  g_flux_shape[precision == LBM_PREC_FP64 ? 0 : 1] = shape;
  return LBM_OK;
}

extern "C" int lbm_flux_shape_dims(int32_t shape, int32_t* w, int32_t* h) {
  if (shape < 0 || shape >= kFluxShapes || !w || !h) return fail_with(LBM_ERR_ARG, "bad flux shape query");
  int ww = 0, hh = 0;
  flux_tile_dims(shape, &ww, &hh);
  *w = ww;
  *h = hh;
  return LBM_OK;
}

// Tile-shape autotuner: times `steps` steps of the batch with each flux tile
// shape (after one untimed step that also captures the step graphs), keeps
// the lowest-numbered shape within kTuneTie of the fastest (shapes that close
// trade places from run to run on timing noise alone; the tie-break makes the
// choice repeatable), and restores every member's state, step count and
// failure flag, so tuning leaves the solution untouched. A batch whose members
// are all on strips launches the same kernels whatever the shape: it is timed
// once, and keeps its shape and the default (five timings of one sequence
// would choose between them by noise).
static constexpr double kTuneTie = 0.005;
extern "C" int lbm_batch_autotune(lbm_batch* hb, int32_t steps, int32_t* shape_out, double* ms_per_step_out) {
  if (!hb || steps < 1) return fail_with(LBM_ERR_ARG, "bad autotune arguments");
  Batch& b = *reinterpret_cast<Batch*>(hb);
  struct Saved {
    void* buf = nullptr;
    int cur = 0, step = 0, fail = INT_MAX;
    bool failed = false;
  };
  std::vector<Saved> saved(b.members.size());
  auto release = [&]() {
    for (auto& v : saved)
      if (v.buf) (void)hipFree(v.buf);
  };
  const size_t es = b.precision == LBM_PREC_FP64 ? sizeof(double) : sizeof(float);
  for (size_t k = 0; k < b.members.size(); k++) {
    Solver& s = *b.members[k];
    const size_t bytes = (size_t)s.pitch * s.ny * kPlanes * es;
    const size_t mbytes = s.mom[0] ? (size_t)s.pitch * s.ny * 4 * sizeof(double) : 0;
    if (hipMalloc(&saved[k].buf, bytes + mbytes) != hipSuccess) {
      release();
      return fail_with(LBM_ERR_NOMEM, "autotune: no room for a state snapshot");
    }
    HIP_TRY(hipMemcpyAsync(saved[k].buf, s.state[s.cur], bytes, hipMemcpyDeviceToDevice, b.stream));
    if (mbytes)
      HIP_TRY(hipMemcpyAsync((char*)saved[k].buf + bytes, s.mom[s.cur], mbytes, hipMemcpyDeviceToDevice, b.stream));
    HIP_TRY(hipMemcpyAsync(&saved[k].fail, s.fail, sizeof(int), hipMemcpyDeviceToHost, b.stream));
    saved[k].cur = s.cur;
    saved[k].step = s.step;
    saved[k].failed = s.failed;
  }
  HIP_TRY(hipStreamSynchronize(b.stream));
  const bool tiles = !strips_enabled() || b.tiles_rest > 0;
  double ms_of[kFluxShapes];
  for (int shape = 0; shape < kFluxShapes; shape++) {
    if (!tiles && shape > 0) {
      ms_of[shape] = ms_of[0];
      if (ms_per_step_out) ms_per_step_out[shape] = ms_of[0];
      continue;
    }
    int st = tiles ? batch_set_shape(b, shape) : LBM_OK;
    if (st == LBM_OK) st = batch_step(b, 1);
    if (st == LBM_OK) st = batch_step(b, steps);
    if (st < 0) {
      release();
      return st;
    }
    const double ms = g_last_timing.total_ms / steps;
    if (ms_per_step_out) ms_per_step_out[shape] = ms;
    ms_of[shape] = ms;
  }
  double fastest = ms_of[0];
  for (int shape = 1; shape < kFluxShapes; shape++) fastest = std::min(fastest, ms_of[shape]);
  int best_shape = 0;
  while (ms_of[best_shape] > fastest * (1.0 + kTuneTie)) best_shape++;
  if (!tiles) best_shape = b.flux_shape;
  for (size_t k = 0; k < b.members.size(); k++) {
    Solver& s = *b.members[k];
    const size_t bytes = (size_t)s.pitch * s.ny * kPlanes * es;
    const size_t mbytes = s.mom[0] ? (size_t)s.pitch * s.ny * 4 * sizeof(double) : 0;
    s.cur = saved[k].cur;
    s.step = saved[k].step;
    s.failed = saved[k].failed;
    HIP_TRY(hipMemcpyAsync(s.state[s.cur], saved[k].buf, bytes, hipMemcpyDeviceToDevice, b.stream));
    if (mbytes)
      HIP_TRY(hipMemcpyAsync(s.mom[s.cur], (char*)saved[k].buf + bytes, mbytes, hipMemcpyDeviceToDevice, b.stream));
    HIP_TRY(hipMemcpyAsync(s.fail, &saved[k].fail, sizeof(int), hipMemcpyHostToDevice, b.stream));
    HIP_TRY(hipStreamSynchronize(b.stream));
    const int st = upload_inst(s);
    if (st != LBM_OK) {
      release();
      return st;
    }
  }
  HIP_TRY(hipStreamSynchronize(b.stream));
  release();
  if (tiles) {
    const int st = batch_set_shape(b, best_shape);
    if (st != LBM_OK) return st;
    g_flux_shape[b.precision == LBM_PREC_FP64 ? 0 : 1] = best_shape;
  }
  if (shape_out) *shape_out = best_shape;
  return LBM_OK;
}


// lbm_fused.hip — the RK3 step of FP64 storage in two launches, for the
// instances on strips:
//
//   k_stage23  net fluxes of f2 (stage 2), then stage 3 of each cell -> f3 and
//              the stored net fluxes dF(f2)
//   k_stage31  net fluxes of f3 (stage 3), the new state f3 + (dF2 - dF3)/2,
//              then stages 1 and 2 of the next step -> f2
//
// Between the steps of a sequence the state lives only in f2, from which stage
// 3 takes what it needs of it (point_s3): a step reads and writes 76 values
// per cell and launch (f2 26 in, f3 26 and dF 24 out; f3 26 and dF 24 in, f2
// 26 out), 1216 B, where the four launches it replaces move 248 values. The
// state is written in the last two steps of a sequence (the residual compares
// them) and where an instance fails: the failing step's state goes to the
// buffer that does not hold the sequence's first state, so that the sequence
// can be taken again up to the step before (lone_step). Same values bit for
// bit as the four launches: the faces are the strip kernels' (March) and the
// pointwise stages those of lbm_point.hpp. us per step, four launches -> two
// (with the s12 launch that begins a sequence): 64^2 Couette 41 -> 29, 256^2
// shear wave 48 -> 40, 512^2 129 -> 98, ensemble of 48 1855 -> 1550, 3072^2
// Riemann 3865 -> 3165.
//
// Bounds at 3072^2: the 5.7 GB a launch moves take 1.25 ms at the rate of a
// large copy (4.6 TB/s); k_stage23 takes 1.70 ms, k_stage31 1.45. Without
// their loads or without their stores they took 1.3 and 1.0 ms (of 1.74 and
// 1.61 then), with the FP64 units busy for two thirds of it: neither alone
// bounds them, but the three wavefronts per SIMD that the registers leave room
// for, which wait for memory at the same places of a row.
//
// One workgroup per work item (a strip of kStripW columns by some rows); its
// four wavefronts march the rows in step, each with one direction along x, one
// along y and one diagonal (quad_x, quad_y, quad_d): four net faces for f and h
// each, equal work, and a quarter of the cell's equilibria, so that the
// stencil windows (three directions) and the pointwise temporaries fit the
// registers of three wavefronts per SIMD (3072^2, when first built: with two
// 3378 us, three 3266). Wavefronts whose x direction is negative take the columns in reverse
// lane order, in which the direction is positive: one x sign in the code. Per
// row the wavefronts exchange their parts of the cell's sums through LDS (one
// barrier; two buffers in turn, so that a part is overwritten only after every
// wavefront has passed the barrier behind its reads).
#include <type_traits>

#include "lbm_point.hpp"
#include "lbm_stencil.hpp"

namespace uqlbm {

#include "lbm_strip.hpp"

namespace {

constexpr int kQuadRows = 32;   // most rows of an item
constexpr int kWriteState = 1;  // k_stage31: write the new state
constexpr int kNextStages = 2;  // k_stage31: stages 1 and 2 of the next step
constexpr int kStateBit = 2;    // k_stage31: the buffer of the new state (one bit)

// The instance record through the constant address space: its fields (which no
// launch of the step changes) come in scalar loads wherever they are used.
using InstC = const __attribute__((address_space(4))) InstDev;

// Parts of a row's sums: N sums (as pairs of doubles) per wavefront, and the
// parts of the equilibrium mass, per column of the strip.
template <int N>
struct QuadRows {
  double2 v[2][4][N / 2][64];
  double mass[2][4][64];
  int rows[kQuadRows + 2 * kH];  // the row table (row_entry) of rows y0 - 3 .. y0 + nrows + 2
};

// Row table: the instance's row that a logical row maps to, and whether it is
// reached through a north or south mirror or clamped.
constexpr int kRowMir = 1 << 30, kRowClamp = 1 << 29, kRowMask = kRowClamp - 1;
__device__ __forceinline__ int row_entry(InstC& in, int yl) {
  unsigned m, c;
  const int flags = in.flags;
  const int r = map_axis(yl, in.ny, flags & kPeriodicY, flags & kMirrorS, flags & kMirrorN, m, c);
  return r | (m ? kRowMir : 0) | (c ? kRowClamp : 0);
}

__device__ __forceinline__ void quad_barrier() {
  // LDS only: global loads and stores stay in flight across the barrier
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// Buffer accesses: a descriptor per array (all its planes), the plane and row
// as a scalar offset, the column as the lane's 32-bit offset, so an access
// takes no vector instruction and no 64-bit address; a lane that takes no part
// has the offset kSkip, beyond every array: its load gives zero and its store
// is dropped, without a branch. The offsets reach 4 GiB: larger instances take
// the other kernels (fused_instance).
using Buf = __amdgpu_buffer_rsrc_t;
typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
constexpr unsigned kSkip = 0xFFFFFFF0u;

__device__ __forceinline__ Buf make_buf(const void* p, unsigned bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, bytes, 0x00027000);
}
__device__ __forceinline__ double ld(Buf b, unsigned col, unsigned row) {
  return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(b, col, row, 0));
}
__device__ __forceinline__ void st(Buf b, unsigned col, unsigned row, double v) {
  __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2, v), b, col, row, 0);
}
__device__ __forceinline__ unsigned ld32(Buf b, unsigned col, unsigned row) {
  return __builtin_amdgcn_raw_buffer_load_b32(b, col, row, 0);
}

template <int N>
__device__ __forceinline__ void put_sums(QuadRows<N>& X, int buf, int w, int col, int k, const Sums& s) {
  X.v[buf][w][2 * k][col] = double2{s.m, s.px};
  X.v[buf][w][2 * k + 1][col] = double2{s.py, s.e};
}
template <int N>
__device__ __forceinline__ Sums get_sums(const QuadRows<N>& X, int buf, int col, int k) {
  Sums s[4];
#pragma unroll
  for (int w = 0; w < 4; w++) {
    const double2 a = X.v[buf][w][2 * k][col], b = X.v[buf][w][2 * k + 1][col];
    s[w] = Sums{a.x, a.y, b.x, b.y};
  }
  return ((s[0] + s[1]) + s[2]) + s[3];
}

// Hides where a scalar value comes from: what is formed from it is formed
// again in every row, by scalar instructions and loads that run beside the
// vector ones, instead of being kept over the rows in scalar registers, which
// are too few for the descriptors, constants and signs of a row together. (Or
// as a flag per lane: QuadItem::upcol compared outside the rows took a vector
// register over all of them, and the compiler spilled it at the merge behind a
// wall's branch, before the other lanes were on again: their flag was lost.)
template <typename T>
__device__ __forceinline__ T again(T v) {
  asm volatile("" : "+s"(v));
  return v;
}

// quad_x, quad_y of a wavefront, four bits each.
constexpr int kDirX = quad_x(0) | quad_x(1) << 4 | quad_x(2) << 8 | quad_x(3) << 12;
constexpr int kDirY = quad_y(0) | quad_y(1) << 4 | quad_y(2) << 8 | quad_y(3) << 12;
__device__ __forceinline__ int dir_x(int w) { return (kDirX >> (4 * w)) & 15; }
__device__ __forceinline__ int dir_y(int w) { return (kDirY >> (4 * w)) & 15; }
// A wavefront's directions: signs and lattice velocities.
struct Quad {
  int w, Ix, Iy, Id;
  double sx, sy;    // signs
  double exx, eyy;  // lattice velocity of Ix along x, of Iy along y
  double aex, aey;  // their sizes
};
__device__ __forceinline__ Quad make_quad(int w) {
  Quad q;
  q.w = w;
  q.Ix = dir_x(w);
  q.Iy = dir_y(w);
  q.Id = 5 + w;
  q.sx = w == 0 || w == 3 ? 1.0 : -1.0;
  q.sy = w < 2 ? 1.0 : -1.0;
  q.aex = w < 2 ? 1.0 : 2.0;
  q.aey = (w & 1) ? 2.0 : 1.0;
  q.exx = q.aex * q.sx;
  q.eyy = q.aey * q.sy;
  return q;
}

// Equilibria of a wavefront's x and y direction (eq_point's arguments).
__device__ __forceinline__ void quad_eq_x(const Quad& q, const PointEq& e, double& fe, double& he) {
  const double a = q.sx * e.u;
  if (q.w < 2) eq_axis(e, a, e.v, fe, he);
  else eq_axis2(e, a, fe, he);
}
__device__ __forceinline__ void quad_eq_y(const Quad& q, const PointEq& e, double& fe, double& he) {
  const double b = q.sy * e.v;
  if (q.w & 1) eq_axis2(e, b, fe, he);
  else eq_axis(e, b, e.u, fe, he);
}

// A work item: the instance's arrays, offsets and edge rules, and the lane's
// column. Wavefronts of negative x sign take the columns in reverse.
struct QuadItem {
  InstC* in;
  const void *src, *out, *dfl, *type;  // src: f2 (k_stage23), f3 (k_stage31); out: the other
  double c;
  unsigned P8, pitch8;  // bytes of a plane, of a row
  const int* rows;  // the item's row table (LDS), from row y0 - 3
  int ytab;         // y0 - 3
  unsigned X8;      // byte offset of the lane's (mapped) column
  // ... with the planes from the lower one of an east/west pair of directions
  // to the lane's (a mirrored column takes the other one of the pair): of the x
  // direction, and of the diagonal at a row that is not or is mirrored
  unsigned Xx, Xd[2];
  int col;       // its column of the strip's 64
  int own;       // own column
  int upcol;     // the strip's column whose upwind column is clamped (of those within the instance at most one)
  double rdx;
};

// Cell type of a lane's column from the word that holds it (kept as loaded:
// taken apart where it is used, so that the wait for the load falls there).
__device__ __forceinline__ unsigned type_word(const QuadItem& Q, Buf type, unsigned row) {
  return ld32(type, (Q.X8 / 8u) & ~3u, row);
}
__device__ __forceinline__ int type_of(const QuadItem& Q, unsigned word) {
  return (int)((word >> (Q.X8 & 24u)) & 0xFFu);
}

template <bool STAGE31>
__device__ __forceinline__ void quad_setup(const InstDev* inst, const TileRef& sr, int w, const int* rows, QuadItem& Q) {
  const bool neg = w == 1 || w == 2;
  InstC* in = (InstC*)inst;
  Q.src = STAGE31 ? in->f3 : in->f2;
  Q.out = STAGE31 ? in->f2 : in->f3;
  Q.dfl = in->dflux;
  Q.type = in->ctype;
  Q.c = in->c;
  const int lane = threadIdx.x & 63, x0 = sr.tx * kStripW;
  Q.in = in;
  Q.P8 = (unsigned)in->plane * 8u;
  Q.pitch8 = (unsigned)in->pitch * 8u;
  const int flags = in->flags, nx = in->nx;
  Q.rows = rows;
  Q.ytab = sr.ty - kH;
  Q.col = neg ? 63 - lane : lane;
  const int xl = x0 - kH + Q.col;
  const int px = flags & kPeriodicX, mw = flags & kMirrorW, me = flags & kMirrorE;
  unsigned mx, cx;
  Q.X8 = (unsigned)map_axis(xl, nx, px, mw, me, mx, cx) * 8u;
  const unsigned pair = (unsigned)(w & 1) ^ mx;  // the pairs 1, 3; 9, 11 (two planes apart); 5, 6; 7, 8
  Q.Xx = Q.X8 + (w < 2 ? pair : 1u - pair) * 2u * Q.P8;
  Q.Xd[0] = Q.X8 + pair * Q.P8;
  Q.Xd[1] = Q.X8 + (1u - pair) * Q.P8;
  Q.upcol = __builtin_amdgcn_readfirstlane(neg ? (px || me ? -1 : nx - 1 - x0 + kH) : (px || mw ? -1 : kH - x0));
  Q.own = lane >= kH && lane < kH + kStripW && xl < nx;
  Q.rdx = Q.own ? (in->rdxs ? in->rdxs[xl] : in->rdx) : 0.0;
}

// Row table entry of logical row yl (the same for the whole wavefront).
__device__ __forceinline__ int quad_row(const QuadItem& Q, int yl) {
  return __builtin_amdgcn_readfirstlane(Q.rows[yl - Q.ytab]);
}

// The staged f and h of a wavefront's x direction at a row of the instance, and
// of its y and diagonal directions at a row table entry. A north or south
// mirror exchanges the y directions of wavefronts w and w ^ 2 and the diagonals
// of w and w ^ 3, an east or west mirror those along x and the diagonals of w
// and w ^ 1 (QuadItem::Xx, Xd).
__device__ __forceinline__ void quad_load_x(const QuadItem& Q, Buf src, int w, unsigned ro, double& f, double& h) {
  const unsigned o = (w < 2 ? 1u : 9u) * Q.P8 + ro;
  f = ld(src, Q.Xx, o);
  h = ld(src, Q.Xx, o + kQ * Q.P8);
}
__device__ __forceinline__ void quad_load_yd(const QuadItem& Q, Buf src, int w, int entry, double& fy, double& hy,
                                             double& fd, double& hd) {
  const int m = (entry & kRowMir) ? 1 : 0, wd = w ^ (3 * m);
  const unsigned ro = (unsigned)(entry & kRowMask) * Q.pitch8;
  const unsigned oy = (unsigned)dir_y(w ^ (2 * m)) * Q.P8 + ro, od = (unsigned)(5 + (wd & 2)) * Q.P8 + ro;
  const unsigned xd = m ? Q.Xd[1] : Q.Xd[0];
  fy = ld(src, Q.X8, oy);
  hy = ld(src, Q.X8, oy + kQ * Q.P8);
  fd = ld(src, xd, od);
  hd = ld(src, xd, od + kQ * Q.P8);
}

// The stencil window of a direction with a y component: the five rows of the y
// face F below row F, F - 3 .. F + 1 upwards (SY > 0: owner row F - 1) or F - 2
// .. F + 2 downwards (owner row F), and that face's values of the row before.
// The row that enters for the face above row y is y + 2 or y + 3.
struct QuadWin {
  double f[5], h[5], Ff, Fh;
};
template <int SY>
constexpr int kEnter = SY > 0 ? 2 : 3;

// Wall closure factor of the cells of a row (loaded where a wall owns a face).
__device__ __forceinline__ double quad_alpha(const QuadItem& Q, int yl) {
  return ld(make_buf(Q.in->alpha, Q.P8), Q.X8, (unsigned)(quad_row(Q, yl) & kRowMask) * Q.pitch8);
}

// y face F of a window.
template <bool SOLID, bool W5, int SY>
__device__ __forceinline__ void quad_yface(const QuadItem& Q, const QuadWin& W, unsigned solid, int F, double v,
                                           double& vf, double& vh) {
  double Lf[5], Lh[5];
  int sld[5];
#pragma unroll
  for (int k = 0; k < 5; k++) {
    const int r = SY > 0 ? k : 4 - k;
    Lf[k] = W.f[r];
    Lh[k] = W.h[r];
    sld[k] = SOLID ? (int)((solid >> r) & 1u) : 0;
  }
  if constexpr (SOLID) {
    if (__ballot(sld[2])) {
      const double a = quad_alpha(Q, SY > 0 ? F - 1 : F);
      if (sld[2]) {
        strip_wall<double>(a, v, Lf[2], Lh[2], 0.0, 0.0, vf, vh);
        return;
      }
    }
  }
  strip_line<double, SOLID, W5>(v, Lf, Lh, sld, vf, vh);
}

// x face upwind of the lane's column (owner lane l - 1) at row y.
template <bool SOLID, bool W5>
__device__ __forceinline__ void quad_xface(const QuadItem& Q, double f, double h, unsigned long long solid, int y,
                                           double v, double& vf, double& vh) {
  double Lf[5], Lh[5];
  int sld[5] = {0, 0, 0, 0, 0};
  Lf[3] = f;
  Lh[3] = h;
  Lf[2] = lane_shift<kDppShr1>(Lf[3]);
  Lh[2] = lane_shift<kDppShr1>(Lh[3]);
  Lf[1] = lane_shift<kDppShr1>(Lf[2]);
  Lh[1] = lane_shift<kDppShr1>(Lh[2]);
  Lf[0] = lane_shift<kDppShr1>(Lf[1]);
  Lh[0] = lane_shift<kDppShr1>(Lh[1]);
  Lf[4] = lane_shift<kDppShl1>(Lf[3]);
  Lh[4] = lane_shift<kDppShl1>(Lh[3]);
  if constexpr (SOLID) {
    // shifted as a scalar mask: five flags per lane, formed from the lane's
    // number, are kept over the rows in registers that k_stage23 does not have
    // (33 of them spilled; at most 5 this way)
#pragma unroll
    for (int k = 0; k < 5; k++)
      sld[k] = __builtin_amdgcn_inverse_ballot_w64(k < 3 ? solid << (3 - k) : solid >> (k - 3)) ? 1 : 0;
    if (solid) {
      const double a = lane_shift<kDppShr1>(quad_alpha(Q, y));
      if (sld[2]) {
        strip_wall<double>(a, v, Lf[2], Lh[2], 0.0, 0.0, vf, vh);
        return;
      }
    }
  }
  strip_line<double, SOLID, W5>(v, Lf, Lh, sld, vf, vh);
}

// Net fluxes of a row's cell in the direction of a window (HX: diagonal, with
// the x faces of the row's values) or of the x direction alone; the window
// moves on to row y + 4 (nf, nh). The grouping and roundings of March::net.
template <bool SOLID, bool W5, int SY, bool HX>
__device__ __forceinline__ void quad_net_y(const QuadItem& Q, QuadWin& W, unsigned solid, unsigned long long xsolid,
                                           int y, bool upclamp, double nf, double nh, double vx, double vy, double rdy,
                                           double& dF, double& dH, double& of, double& oh) {
#pragma clang fp contract(off)
#pragma unroll
  for (int k = 0; k < 4; k++) {
    W.f[k] = W.f[k + 1];
    W.h[k] = W.h[k + 1];
  }
  W.f[4] = nf;
  W.h[4] = nh;
  double Gf, Gh;
  quad_yface<SOLID, W5, SY>(Q, W, solid, y + 1, vy, Gf, Gh);  // face above row y
  of = W.f[SY > 0 ? 2 : 1];
  oh = W.h[SY > 0 ? 2 : 1];
  double oyf = SY > 0 ? Gf : W.Ff, oyh = SY > 0 ? Gh : W.Fh, iyf = SY > 0 ? W.Ff : Gf, iyh = SY > 0 ? W.Fh : Gh;
  if (upclamp) {
    iyf = oyf;
    iyh = oyh;
  }
  W.Ff = Gf;
  W.Fh = Gh;
  if constexpr (HX) {
    double ixf, ixh;
    quad_xface<SOLID, W5>(Q, of, oh, xsolid, y, vx, ixf, ixh);
    const double oxf = lane_shift<kDppShl1>(ixf), oxh = lane_shift<kDppShl1>(ixh);
    if (Q.col == again(Q.upcol)) {
      ixf = oxf;
      ixh = oxh;
    }
    dF = (Q.rdx * oxf + rdy * oyf) - (Q.rdx * ixf + rdy * iyf);
    dH = (Q.rdx * oxh + rdy * oyh) - (Q.rdx * ixh + rdy * iyh);
  } else {
    dF = rdy * oyf - rdy * iyf;
    dH = rdy * oyh - rdy * iyh;
  }
}
template <bool SOLID, bool W5>
__device__ __forceinline__ void quad_net_x(const QuadItem& Q, unsigned long long xsolid, int y, double f, double h,
                                           double vx, double& dF, double& dH) {
#pragma clang fp contract(off)
  double ixf, ixh;
  quad_xface<SOLID, W5>(Q, f, h, xsolid, y, vx, ixf, ixh);
  const double oxf = lane_shift<kDppShl1>(ixf), oxh = lane_shift<kDppShl1>(ixh);
  if (Q.col == again(Q.upcol)) {
    ixf = oxf;
    ixh = oxh;
  }
  dF = Q.rdx * oxf - Q.rdx * ixf;
  dH = Q.rdx * oxh - Q.rdx * ixh;
}

// What a row needs from memory, loaded one row ahead: the staged values (the x
// direction's of the row itself, the others' of the row entering the window),
// cell types, (k_stage31) the cell's stored dF2, the rest direction (wavefront
// 0), dt/dy.
template <bool STAGE31>
struct QuadRow {
  double x[2], y[2], d[2], r[2];
  double dF[STAGE31 ? 6 : 1];
  double rdy;
  unsigned type, ntype;  // words (type_word)
  bool upclamp;  // the upwind row is clamped
};

// Flag a failed equilibrium check of the row whose mass parts lie in X.mass[buf].
template <int N>
__device__ __forceinline__ void quad_check(const QuadItem& Q, const QuadRows<N>& X, int buf, int step, bool on,
                                           double rho) {
#pragma clang fp contract(off)
  if (!on) return;
  const double s = ((X.mass[buf][0][Q.col] + X.mass[buf][1][Q.col]) + X.mass[buf][2][Q.col]) + X.mass[buf][3][Q.col];
  if (!(fabs(s - rho) <= 1e-6) || !isfinite(rho)) atomicMin(Q.in->fail, Q.in->step_base + step);
}

template <bool STAGE31, bool SOLID, bool W5, int SY>
__device__ __forceinline__ void quad_rows(const InstDev& inst, const QuadItem& Q, const TileRef& sr, int w0,
                                          int step, int what, QuadRows<STAGE31 ? 4 : 8>& X) {
  const int y0 = sr.ty, nrows = sr.flags >> kStripRowsBit;
  QuadWin wy, wd;
  unsigned solid = 0;  // solid rows of the windows, bit k: row k

  auto fetch = [&](int y) {
    QuadRow<STAGE31> r;
    InstC* in = Q.in;
    const int w = again(w0);
    const Quad q = make_quad(w);
    const unsigned ro = (unsigned)y * Q.pitch8;
    const Buf src = make_buf(again(Q.src), kPlanes * Q.P8), type = make_buf(again(Q.type), Q.P8 / 8u);
    quad_load_x(Q, src, w, ro, r.x[0], r.x[1]);
    const int n = quad_row(Q, y + kEnter<SY>);
    quad_load_yd(Q, src, w, n, r.y[0], r.y[1], r.d[0], r.d[1]);
    r.upclamp = (quad_row(Q, y - SY) & kRowClamp) != 0;
    r.type = type_word(Q, type, ro / 8u);
    r.ntype = SOLID ? type_word(Q, type, (unsigned)(n & kRowMask) * (Q.pitch8 / 8u)) : 0u;
    if constexpr (STAGE31) {
      const Buf dfl = make_buf(again(Q.dfl), 24u * Q.P8);
      const unsigned ox = (unsigned)q.Ix * Q.P8 + ro, oy = (unsigned)q.Iy * Q.P8 + ro, od = (unsigned)q.Id * Q.P8 + ro;
      r.dF[0] = ld(dfl, Q.X8, ox - Q.P8);
      r.dF[1] = ld(dfl, Q.X8, ox + 11u * Q.P8);
      r.dF[2] = ld(dfl, Q.X8, oy - Q.P8);
      r.dF[3] = ld(dfl, Q.X8, oy + 11u * Q.P8);
      r.dF[4] = ld(dfl, Q.X8, od - Q.P8);
      r.dF[5] = ld(dfl, Q.X8, od + 11u * Q.P8);
    }
    const unsigned xr = w == 0 ? Q.X8 : kSkip;
    r.r[0] = ld(src, xr, ro);
    r.r[1] = ld(src, xr, ro + kQ * Q.P8);
    r.rdy = in->rdys ? ((const __attribute__((address_space(4))) double*)in->rdys)[y] : in->rdy;
    return r;
  };
  // three directions' values and (wavefront 0) the rest direction's
  auto put = [&](const Quad& q, const void* base, unsigned col, unsigned ro, const double* v, double f0, double h0) {
    const Buf b = make_buf(again(base), kPlanes * Q.P8);
    st(b, col, (unsigned)q.Ix * Q.P8 + ro, v[0]);
    st(b, col, (unsigned)(kQ + q.Ix) * Q.P8 + ro, v[1]);
    st(b, col, (unsigned)q.Iy * Q.P8 + ro, v[2]);
    st(b, col, (unsigned)(kQ + q.Iy) * Q.P8 + ro, v[3]);
    st(b, col, (unsigned)q.Id * Q.P8 + ro, v[4]);
    st(b, col, (unsigned)(kQ + q.Id) * Q.P8 + ro, v[5]);
    if (q.w == 0) {
      st(b, col, ro, f0);
      st(b, col, ro + kQ * Q.P8, h0);
    }
  };

  bool pon = false;  // the previous row: its check is due after the next barrier
  double prho = 0;
  const int cstep = STAGE31 ? step + 1 : step;  // the step whose equilibrium check this launch makes

  const int end = y0 + nrows;
  QuadRow<STAGE31> cc;
  auto row = [&](int y, int buf) {
#pragma clang fp contract(off)
    const int w = again(w0);
    const Quad q = make_quad(w);
    const double c = Q.c;
    double d[6], o[6];
    const unsigned long long xsolid = SOLID ? __ballot(type_of(Q, cc.type) == 2) : 0ull;
    if constexpr (SOLID) solid = (solid >> 1) | (type_of(Q, cc.ntype) == 2 ? 16u : 0u);
    o[0] = cc.x[0];
    o[1] = cc.x[1];
    quad_net_x<SOLID, W5>(Q, xsolid, y, o[0], o[1], q.aex * c, d[0], d[1]);
    __builtin_amdgcn_sched_barrier(0);  // one direction at a time: the temporaries of three at once spill
    quad_net_y<SOLID, W5, SY, false>(Q, wy, solid, 0ull, y, cc.upclamp, cc.y[0], cc.y[1], 0.0, q.aey * c, cc.rdy, d[2], d[3], o[2], o[3]);
    __builtin_amdgcn_sched_barrier(0);
    quad_net_y<SOLID, W5, SY, true>(Q, wd, solid, xsolid, y, cc.upclamp, cc.d[0], cc.d[1], c, c, cc.rdy, d[4], d[5], o[4], o[5]);
    __builtin_amdgcn_sched_barrier(0);
    const bool on = Q.own && type_of(Q, cc.type) == 0;
    const double rf = cc.r[0], rh = cc.r[1];
    const unsigned ro = (unsigned)y * Q.pitch8, oc = on ? Q.X8 : kSkip;
    if constexpr (STAGE31) {
#pragma unroll
      for (int k = 0; k < 6; k++) o[k] = o[k] + 0.5 * (cc.dF[k] - d[k]);  // the new state
    }
    // the next row's loads: they land while this row's cells are finished
    // (after the last row the same row again: no branch around the loads)
    cc = fetch(y + 1 < end ? y + 1 : y);
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (STAGE31) {
      if (what & kWriteState) put(q, Q.in->state[(what >> kStateBit) & 1], oc, ro, o, rf, rh);
      if (!(what & kNextStages)) return;
    } else {
      const Buf dfl = make_buf(again(Q.dfl), 24u * Q.P8);
      const unsigned ox = (unsigned)q.Ix * Q.P8 + ro, oy = (unsigned)q.Iy * Q.P8 + ro, od = (unsigned)q.Id * Q.P8 + ro;
      st(dfl, oc, ox - Q.P8, d[0]);
      st(dfl, oc, ox + 11u * Q.P8, d[1]);
      st(dfl, oc, oy - Q.P8, d[2]);
      st(dfl, oc, oy + 11u * Q.P8, d[3]);
      st(dfl, oc, od - Q.P8, d[4]);
      st(dfl, oc, od + 11u * Q.P8, d[5]);
    }
    Sums s = quad_sums(q.exx, q.sx, q.eyy, q.sy, o[0], o[2], o[4], o[1], o[3], o[5]);
    if (w == 0) {
      s.m = s.m + rf;
      s.e = s.e + rh;
    }
    put_sums(X, buf, w, Q.col, 0, s);
    if constexpr (!STAGE31)
      put_sums(X, buf, w, Q.col, 1, quad_sums(q.exx, q.sx, q.eyy, q.sy, d[0], d[2], d[4], d[1], d[3], d[5]));
    quad_barrier();
    InstC& k = *again(Q.in);
    if (w == 3) quad_check(Q, X, buf ^ 1, cstep, pon, prho);
    const Sums t = get_sums(X, buf, Q.col, 0);
    Macro m;
    point_macro(k, inst, t, m);
    const PointEq e = point_eq(k, m);
    // one direction at a time, stored as it is done: few values live at once
    const Quad qe = make_quad(again(w0));
    const Buf out = make_buf(again(Q.out), kPlanes * Q.P8);
    double mass = 0, fm0 = 0;
    auto keep = [&](int I, double f, double h) {
      st(out, oc, (unsigned)I * Q.P8 + ro, f);
      st(out, oc, (unsigned)(kQ + I) * Q.P8 + ro, h);
      __builtin_amdgcn_sched_barrier(0);
    };
    if constexpr (STAGE31) {
      const Relax12 R = make_relax12(k, m);
      __builtin_amdgcn_sched_barrier(0);
      double fe, he, f2, h2;
      quad_eq_x(qe, e, fe, he);
      point_s12(R, e, q.exx, 0.0, o[0], o[1], fe, he, f2, h2);
      mass = fe;
      keep(q.Ix, f2, h2);
      quad_eq_y(qe, e, fe, he);
      point_s12(R, e, 0.0, q.eyy, o[2], o[3], fe, he, f2, h2);
      mass = mass + fe;
      keep(q.Iy, f2, h2);
      eq_diag(e, q.sx * e.u, q.sy * e.v, fe, he);
      point_s12(R, e, q.sx, q.sy, o[4], o[5], fe, he, f2, h2);
      mass = mass + fe;
      keep(q.Id, f2, h2);
      if (w == 0) {
        eq_rest(e, fe, he);
        point_s12(R, e, 0.0, 0.0, rf, rh, fe, he, f2, h2);
        fm0 = fe;
        keep(0, f2, h2);
      }
      prho = m.rho;
    } else {
      Macro m3;
      point_macro(k, inst, t - get_sums(X, buf, Q.col, 1), m3);
      const Relax3 R = make_relax3(k, m, m3);
      const PointEq e3 = point_eq(k, m3);
      prho = m3.rho;
      __builtin_amdgcn_sched_barrier(0);
      double fe, he, fe3, he3, f3, h3;
      quad_eq_x(qe, e, fe, he);
      quad_eq_x(qe, e3, fe3, he3);
      point_s3(R, e, e3, q.exx, 0.0, o[0], o[1], d[0], d[1], fe, he, fe3, he3, f3, h3);
      mass = fe3;
      keep(q.Ix, f3, h3);
      quad_eq_y(qe, e, fe, he);
      quad_eq_y(qe, e3, fe3, he3);
      point_s3(R, e, e3, 0.0, q.eyy, o[2], o[3], d[2], d[3], fe, he, fe3, he3, f3, h3);
      mass = mass + fe3;
      keep(q.Iy, f3, h3);
      eq_diag(e, q.sx * e.u, q.sy * e.v, fe, he);
      eq_diag(e3, q.sx * e3.u, q.sy * e3.v, fe3, he3);
      point_s3(R, e, e3, q.sx, q.sy, o[4], o[5], d[4], d[5], fe, he, fe3, he3, f3, h3);
      mass = mass + fe3;
      keep(q.Id, f3, h3);
      if (w == 0) {
        eq_rest(e, fe, he);
        eq_rest(e3, fe3, he3);
        point_s3(R, e, e3, 0.0, 0.0, rf, rh, 0.0, 0.0, fe, he, fe3, he3, f3, h3);
        fm0 = fe3;
        keep(0, f3, h3);
      }
    }
    X.mass[buf][w][Q.col] = w == 0 ? mass + fm0 : mass;
    pon = on;
  };

  const Quad q = make_quad(w0);
  const Buf src = make_buf(Q.src, kPlanes * Q.P8);
#pragma unroll
  for (int k = 0; k < 5; k++) {
    const int n = quad_row(Q, y0 + kEnter<SY> - 5 + k);
    quad_load_yd(Q, src, w0, n, wy.f[k], wy.h[k], wd.f[k], wd.h[k]);
    if constexpr (SOLID)
      solid |= type_of(Q, type_word(Q, make_buf(Q.type, Q.P8 / 8u), (unsigned)(n & kRowMask) * (Q.pitch8 / 8u))) == 2 ? 1u << k : 0u;
  }
  cc = fetch(y0);
  quad_yface<SOLID, W5, SY>(Q, wy, solid, y0, q.aey * Q.in->c, wy.Ff, wy.Fh);
  quad_yface<SOLID, W5, SY>(Q, wd, solid, y0, Q.in->c, wd.Ff, wd.Fh);
  for (int y = y0, buf = 0; y < end; y++, buf ^= 1) row(y, buf);
  if (!STAGE31 || (what & kNextStages)) {
    quad_barrier();
    if (w0 == 3) quad_check(Q, X, (nrows - 1) & 1, cstep, pon, prho);
  }
}

template <bool STAGE31, int SY>
__device__ __forceinline__ void quad_item(const InstDev& inst, const QuadItem& Q, const TileRef& sr, int w,
                                          int step, int what, QuadRows<STAGE31 ? 4 : 8>& X) {
  if (sr.flags & kTileSolid) {
    if (inst.flux_method == 1) quad_rows<STAGE31, true, true, SY>(inst, Q, sr, w, step, what, X);
    else quad_rows<STAGE31, true, false, SY>(inst, Q, sr, w, step, what, X);
  } else {
    if (inst.flux_method == 1) quad_rows<STAGE31, false, true, SY>(inst, Q, sr, w, step, what, X);
    else quad_rows<STAGE31, false, false, SY>(inst, Q, sr, w, step, what, X);
  }
}

// A contiguous chunk of the items per XCD; ctr[0] is the step of k_stage23,
// ctr[1] that of k_stage31 (each launch sets the other's, which it does not
// read itself).
template <bool STAGE31>
__device__ __forceinline__ void quad_launch(const InstDev* __restrict__ insts, const TileRef* __restrict__ items, int n,
                                            int chunk, int what, int* ctr, QuadRows<STAGE31 ? 4 : 8>& X) {
  const int step = ctr[STAGE31 ? 1 : 0];
  if (blockIdx.x == 0 && threadIdx.x == 0) ctr[STAGE31 ? 0 : 1] = STAGE31 ? step + 1 : step;
  const int it = (int)(blockIdx.x % 8) * chunk + (int)(blockIdx.x / 8);
  if (it >= n) return;
  const TileRef sr = items[it];
  const InstDev& in = insts[sr.inst];
  // failures flagged while this launch runs are of its step or the next one:
  // every wavefront sees the same answers here
  const int fail = __builtin_amdgcn_readfirstlane(*in.fail), now = in.step_base + step;
  if (fail < now) return;
  if constexpr (STAGE31) {
    const bool stays = fail == now && (what & kNextStages);  // an inner step fails: its state stays
    what |= ((in.parity0 ^ (stays ? 1 : step)) & 1) << kStateBit;
    if (stays) what |= kWriteState;
  }
  const int w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  for (int k = threadIdx.x; k < (sr.flags >> kStripRowsBit) + 2 * kH; k += 256)
    X.rows[k] = row_entry(*(InstC*)&in, sr.ty - kH + k);
  __syncthreads();
  QuadItem Q;
  quad_setup<STAGE31>(&in, sr, w, X.rows, Q);
  if (w < 2) quad_item<STAGE31, 1>(in, Q, sr, w, step, what, X);
  else quad_item<STAGE31, -1>(in, Q, sr, w, step, what, X);
}

__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(3))) void k_stage23(
    const InstDev* __restrict__ insts, const TileRef* __restrict__ items, int n, int chunk, int* ctr) {
  __shared__ QuadRows<8> X;
  quad_launch<false>(insts, items, n, chunk, 0, ctr, X);
}
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(3))) void k_stage31(
    const InstDev* __restrict__ insts, const TileRef* __restrict__ items, int n, int chunk, int what, int* ctr) {
  __shared__ QuadRows<4> X;
  quad_launch<true>(insts, items, n, chunk, what, ctr, X);
}

}  // namespace

void launch_stage23(const StepLaunch& L, hipStream_t s) {
  const int chunk = (L.nmstrips + 7) / 8;
  k_stage23<<<8 * chunk, 256, 0, s>>>(L.insts, L.mstrips, L.nmstrips, chunk, L.step_ctr);
}
void launch_stage31(const StepLaunch& L, hipStream_t s, bool write_state, bool next_stages) {
  const int chunk = (L.nmstrips + 7) / 8;
  k_stage31<<<8 * chunk, 256, 0, s>>>(L.insts, L.mstrips, L.nmstrips, chunk,
                                      (write_state ? kWriteState : 0) | (next_stages ? kNextStages : 0), L.step_ctr);
}

}  // namespace uqlbm

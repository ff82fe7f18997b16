// lbm_strip.hpp — strip flux kernels (k_strip, k_strip_mom) of the D2Q13
// thermal FD-LBM, included by lbm_strip.hip after the face reconstructions.
//
// The net fluxes of every flux stage for the instances whose cells all take
// the logical stencil addressing. A strip is kStripW columns and some rows of
// one instance, marched row by row by one wavefront for one direction
// (k_strip) or by a workgroup of four wavefronts, three directions each
// (k_strip_mom: the stage-3 flux of FP32 storage, whose cells also sum the
// moments of their net fluxes over the directions). Lane l holds column
// x0 - 3 + l (a 3-column halo on each side fills the 64 lanes); a lane's y
// stencil is a window of six rows in its registers and its x stencil comes
// from the neighbouring lanes by whole-wave DPP shifts, so the faces need no
// LDS and no barrier. Each face is computed once: the x face left of a
// lane's column by that lane, the y face below a row when the window reaches
// it; a cell's net flux takes the face it shares with its right neighbour
// from that lane and the face below it from the previous row. The arithmetic
// of every face and net flux is that of the tile kernels (face_flux,
// flux_dir). The next row's loads are issued before the current row's faces,
// so their latency hides behind them.
// (Included inside namespace uqlbm, after the gptr global-pointer alias.)
#pragma once

// DPP controls of whole-wave shifts by one lane (GFX9 wave_shr:1 and
// wave_shl:1): lane l takes the value of lane l - 1, respectively l + 1;
// the lane shifted in at the end reads 0 (bound_ctrl: the zero comes from
// the instruction, so no register has to be cleared before each shift, as
// an "old" operand of 0 would need). Every shift runs with all 64 lanes
// active (never inside a divergent branch).
constexpr int kDppShr1 = 0x138;
constexpr int kDppShl1 = 0x130;

template <int CTRL>
__device__ __forceinline__ int lane_shift(int v) {
  return __builtin_amdgcn_update_dpp(0, v, CTRL, 0xF, 0xF, true);
}
template <int CTRL>
__device__ __forceinline__ float lane_shift(float v) {
  return __int_as_float(lane_shift<CTRL>(__float_as_int(v)));
}
template <int CTRL>
__device__ __forceinline__ double lane_shift(double v) {
  const long long b = __double_as_longlong(v);
  const int lo = lane_shift<CTRL>(int(b)), hi = lane_shift<CTRL>(int(b >> 32));
  return __longlong_as_double((long long)(((unsigned long long)(unsigned)hi << 32) | (unsigned)lo));
}

// One staged position of a direction: f, h and (solid items) its cell
// type, kept as loaded: compared only where used, so that the wait for the
// load falls there and not right after it (which would also wait for the
// loads of the next row in flight).
template <typename TC>
struct SPos {
  TC f, h;
  int type;
  TC a;  // solid items: the wall closure factor of the position
};

// Per-lane constants of a work item.
template <typename TC>
struct StripLane {
  unsigned X;      // mapped column of the lane's logical column
  int mx;          // the column is mirrored east/west
  int own;         // an own column of the item inside the instance
  int clampL;      // the logical column left of the lane is a clamped position
  int clampR;      // ... right of the lane
  TC rdx;          // dt/dx of the lane's column (own lanes)
  int xl;          // logical column
};

// Face flux of the line s0..s4 (WENO5; NND takes s1..s3), with the solid
// extrapolation of face_flux when a point of the line is solid.
template <typename TC, bool SOLID, bool W5>
__device__ __forceinline__ void strip_line(TC v, const TC (&Vf)[5], const TC (&Vh)[5], const int (&sld)[5], TC& vf,
                                           TC& vh) {
  if constexpr (W5) {
    TC F[5], H[5];
#pragma unroll
    for (int k = 0; k < 5; k++) { F[k] = Vf[k]; H[k] = Vh[k]; }
    if constexpr (SOLID) {
      if (sld[0] | sld[1] | sld[2] | sld[3] | sld[4]) {
        TC Ef[5], Eh[5];
#pragma unroll
        for (int k = 0; k < 5; k++) { Ef[k] = F[k]; Eh[k] = H[k]; }
        extrapolate<5>(sld, F, Ef);
        extrapolate<5>(sld, H, Eh);
#pragma unroll
        for (int k = 0; k < 5; k++) { F[k] = Ef[k]; H[k] = Eh[k]; }
      }
    }
    vf = weno5(v, F[0], F[1], F[2], F[3], F[4]);
    vh = weno5(v, H[0], H[1], H[2], H[3], H[4]);
  } else {
    TC F[3] = {Vf[1], Vf[2], Vf[3]}, H[3] = {Vh[1], Vh[2], Vh[3]};
    if constexpr (SOLID) {
      const int s3[3] = {sld[1], sld[2], sld[3]};
      if (s3[0] | s3[1] | s3[2]) {
        TC Ef[3] = {F[0], F[1], F[2]}, Eh[3] = {H[0], H[1], H[2]};
        extrapolate<3>(s3, F, Ef);
        extrapolate<3>(s3, H, Eh);
#pragma unroll
        for (int k = 0; k < 3; k++) { F[k] = Ef[k]; H[k] = Eh[k]; }
      }
    }
    vf = nnd(v, F[0], F[1], F[2]);
    vh = nnd(v, H[0], H[1], H[2]);
  }
}

// Wall closure face of a solid owner (face_flux): alpha |e| f, for FP32
// storage (deviations dev = f - ref staged) |e| (alpha dev + (alpha - 1) ref).
template <typename TS, typename TC>
__device__ __forceinline__ void strip_wall(TC a, TC v, TC wf, TC wh, TC rf, TC rh, TC& vf, TC& vh) {
#pragma clang fp contract(off)  // rounds as the tile kernels' wall faces
  if constexpr (sizeof(TS) == 4) {
    vf = v * (a * wf + (a - TC(1)) * rf);
    vh = v * (a * wh + (a - TC(1)) * rh);
  } else {
    (void)rf;
    (void)rh;
    vf = a * v * wf;
    vh = a * v * wh;
  }
}

// The instance fields the strip kernels read, copied once per work item:
// read through the instance table after the item's stores they would be
// reloaded (the stores might alias the table).
template <typename TS>
struct StripInst {
  gptr<const TS> src;
  gptr<TS> dst;
  gptr<const TS> dfl;  // MODE 1: the stored stage-2 net fluxes
  gptr<const uint8_t> ct;
  gptr<const double> alpha;
  gptr<const double> rdyp;  // dt/dy per row (rdy_stride 1) or the instance's one value (0)
  int rdy_stride;
  long long P;
  int pitch, ny, py, ms, mn;
  int inner;   // the item's rows and their 3-row halo lie inside the instance
  int colmir;  // some lane's column is mirrored east/west
  double c;
};

// Element at column X of the row `base` points at: base is the same for the
// whole wavefront (planes and rows are), so the access takes it from scalar
// registers with the lane's 32-bit byte offset, and neither 64-bit addresses
// per lane nor vector instructions to form them are needed.
template <typename T>
__device__ __forceinline__ gptr<T> at_col(gptr<T> base, unsigned X) {
  if constexpr (std::is_const<T>::value) return (gptr<T>)((gptr<const char>)base + X * unsigned(sizeof(T)));
  else return (gptr<T>)((gptr<char>)base + X * unsigned(sizeof(T)));
}

// The row order of a march: rows y0 .. y0 + nrows - 1 of the item, or (flip)
// the item turned upside down (row y of the march is row 2 y0 + nrows - 1 - y
// of the instance), the direction's y sign then negated: each face has the
// same upwind owner and the same stencil values in the same order either
// way, so the two orders give the same values bit for bit.
struct RowOrder {
  int flip, yflip;
  __device__ __forceinline__ int operator()(int y) const { return flip ? yflip - y : y; }
};

// One direction's march state: SX, SY the signs of its lattice velocity in
// the march's row order; SOLID: the item's region holds a solid cell; W5:
// WENO5 faces (else NND).
template <typename TS, typename TC, bool SOLID, bool W5, int SX, int SY>
struct March {
  static constexpr bool HX = SX != 0, HY = SY != 0;
  TC vx, vy;
  TC rf, rh;  // reference equilibrium of the direction for the wall faces of FP32 storage
              // (a mirror image of it has the same reference: it depends on |e|)
  gptr<const TS> pf0, ph0, pf1, ph1;  // planes staged at a row that is not (0) or is (1) mirrored north/south
  long long pew0, pew1;               // from them to the planes of an east/west mirrored column
  SPos<TC> W[HY ? 6 : 1];  // rows F - 3 .. F + 2 of the y face F below row F
  TC Fyf, Fyh;             // the y face below the next row

  __device__ __forceinline__ void setup(const StripInst<TS>& in, const StripLane<TC>& C, TC rf_, TC rh_, int I) {
    const int aex = c_lat_x[I] > 0 ? c_lat_x[I] : -c_lat_x[I];
    const int aey = c_lat_y[I] > 0 ? c_lat_y[I] : -c_lat_y[I];
    vx = TC(double(aex) * in.c);
    vy = TC(double(aey) * in.c);
    rf = rf_;
    rh = rh_;
    const int dns = c_mir_ns[I];
    pf0 = in.src + (long long)I * in.P;
    ph0 = in.src + (long long)(kQ + I) * in.P;
    pf1 = in.src + (long long)dns * in.P;
    ph1 = in.src + (long long)(kQ + dns) * in.P;
    pew0 = (long long)(c_mir_ew[I] - I) * in.P;
    pew1 = (long long)(c_mir_ew[dns] - dns) * in.P;
    Fyf = Fyh = TC(0);
  }

  // The staged position of logical row yl (an instance row).
  __device__ __forceinline__ SPos<TC> load(const StripInst<TS>& in, const StripLane<TC>& C, int yl) const {
    unsigned my = 0, cy;
    const int ro = (in.inner ? yl : map_axis(yl, in.ny, in.py, in.ms, in.mn, my, cy)) * in.pitch;
    const bool m = (in.ms | in.mn) != 0 && my;
    const gptr<const TS> pf = (m ? pf1 : pf0) + ro, ph = (m ? ph1 : ph0) + ro;
    TS f = *at_col(pf, C.X), h = *at_col(ph, C.X);
    if (in.colmir) {
      const long long ew = m ? pew1 : pew0;
      const TS fm = *at_col(pf + ew, C.X), hm = *at_col(ph + ew, C.X);
      f = C.mx ? fm : f;
      h = C.mx ? hm : h;
    }
    SPos<TC> p;
    p.f = TC(f);
    p.h = TC(h);
    p.type = SOLID ? int(*at_col(in.ct + ro, C.X)) : 0;
    p.a = SOLID ? TC(*at_col(in.alpha + ro, C.X)) : TC(0);
    return p;
  }
  static __device__ __forceinline__ int clamped_row(const StripInst<TS>& in, int yl) {
    if (in.inner) return 0;
    unsigned my, cy;
    (void)map_axis(yl, in.ny, in.py, in.ms, in.mn, my, cy);
    return (int)cy;
  }

  // x face left of this lane's column at a row: owner lane l - 1 (SX > 0) or
  // l (SX < 0); line owner - 2 sx .. owner + 2 sx across the lanes
  __device__ __forceinline__ void xface(const SPos<TC>& r, TC& vf, TC& vh) const {
    TC Lf[5], Lh[5];
    int sld[5] = {0, 0, 0, 0, 0};
    if constexpr (SX > 0) {
      Lf[3] = r.f;
      Lh[3] = r.h;
      Lf[2] = lane_shift<kDppShr1>(Lf[3]);
      Lh[2] = lane_shift<kDppShr1>(Lh[3]);
      Lf[1] = lane_shift<kDppShr1>(Lf[2]);
      Lh[1] = lane_shift<kDppShr1>(Lh[2]);
      Lf[0] = lane_shift<kDppShr1>(Lf[1]);
      Lh[0] = lane_shift<kDppShr1>(Lh[1]);
      Lf[4] = lane_shift<kDppShl1>(Lf[3]);
      Lh[4] = lane_shift<kDppShl1>(Lh[3]);
    } else {
      Lf[2] = r.f;
      Lh[2] = r.h;
      Lf[1] = lane_shift<kDppShl1>(Lf[2]);
      Lh[1] = lane_shift<kDppShl1>(Lh[2]);
      Lf[0] = lane_shift<kDppShl1>(Lf[1]);
      Lh[0] = lane_shift<kDppShl1>(Lh[1]);
      Lf[3] = lane_shift<kDppShr1>(Lf[2]);
      Lh[3] = lane_shift<kDppShr1>(Lh[2]);
      Lf[4] = lane_shift<kDppShr1>(Lf[3]);
      Lh[4] = lane_shift<kDppShr1>(Lh[3]);
    }
    if constexpr (SOLID) {
      const unsigned long long m = __ballot(r.type == 2);
      const int lane = threadIdx.x & 63;
#pragma unroll
      for (int k = 0; k < 5; k++) {
        const int pl = SX > 0 ? lane - 3 + k : lane + 2 - k;
        sld[k] = (pl >= 0 && pl < 64) ? int((m >> pl) & 1ull) : 0;
      }
      // the owner's wall closure factor, staged by the owner lane
      const TC ao = SX > 0 ? lane_shift<kDppShr1>(r.a) : r.a;
      if (sld[2]) {  // solid owner: wall closure
        strip_wall<TS>(ao, vx, Lf[2], Lh[2], rf, rh, vf, vh);
        return;
      }
    }
    strip_line<TC, SOLID, W5>(vx, Lf, Lh, sld, vf, vh);
  }

  // y face F below the window's row F (window rows F - 3 .. F + 2): owner
  // row F - 1 (SY > 0, window 2) or F (SY < 0, window 3)
  __device__ __forceinline__ void yface(TC& vf, TC& vh) const {
    TC Lf[5], Lh[5];
    int sld[5];
#pragma unroll
    for (int k = 0; k < 5; k++) {
      const int w = SY > 0 ? k : 5 - k;
      Lf[k] = W[w].f;
      Lh[k] = W[w].h;
      sld[k] = W[w].type == 2;
    }
    if constexpr (SOLID) {
      if (sld[2]) {
        strip_wall<TS>(W[SY > 0 ? 2 : 3].a, vy, Lf[2], Lh[2], rf, rh, vf, vh);
        return;
      }
    }
    strip_line<TC, SOLID, W5>(vy, Lf, Lh, sld, vf, vh);
  }

  // Fills the window for row y0 (call first_face once the loads have landed).
  __device__ __forceinline__ void fill(const StripInst<TS>& in, const StripLane<TC>& C, const RowOrder& ro, int y0) {
    if constexpr (HY) {
#pragma unroll
      for (int k = 0; k < 6; k++) W[k] = load(in, C, ro(y0 - 3 + k));
    }
  }
  __device__ __forceinline__ void first_face() {
    if constexpr (HY) yface(Fyf, Fyh);
  }
  // The position row y of the march needs from memory: the one entering the
  // window (row y + 3), without a y component row y itself.
  __device__ __forceinline__ SPos<TC> next(const StripInst<TS>& in, const StripLane<TC>& C, const RowOrder& ro,
                                               int y) const {
    return load(in, C, ro(HY ? y + 3 : y));
  }

  // Net flux of row y's cell from its prefetched position (registers only:
  // no memory access); own: the cell's staged values. No contraction: the net
  // flux rounds as the tile kernels (and the oracle) round it, so both paths
  // agree bit for bit.
  __device__ __forceinline__ void net(const StripInst<TS>& in, const StripLane<TC>& C, const RowOrder& ro, int y,
                                      const SPos<TC>& p, TC rdy, TC& dF, TC& dH, TC& ownf, TC& ownh) {
#pragma clang fp contract(off)
    TC Gf = 0, Gh = 0, Ff = 0, Fh = 0, Nf = 0, Nh = 0;
    SPos<TC> xr = p;
    if constexpr (HY) {
#pragma unroll
      for (int k = 0; k < 5; k++) W[k] = W[k + 1];
      W[5] = p;
      yface(Gf, Gh);  // face above row y
      xr = W[2];
    }
    ownf = xr.f;
    ownh = xr.h;
    if constexpr (HX) {
      xface(xr, Ff, Fh);
      Nf = lane_shift<kDppShl1>(Ff);  // face right of the column
      Nh = lane_shift<kDppShl1>(Fh);
    }
    TC oxf = 0, oxh = 0, ixf = 0, ixh = 0, oyf = 0, oyh = 0, iyf = 0, iyh = 0;
    if constexpr (HX) {
      oxf = SX > 0 ? Nf : Ff;
      oxh = SX > 0 ? Nh : Fh;
      ixf = SX > 0 ? Ff : Nf;
      ixh = SX > 0 ? Fh : Nh;
      if (SX > 0 ? C.clampL : C.clampR) {
        ixf = oxf;
        ixh = oxh;
      }
    }
    if constexpr (HY) {
      oyf = SY > 0 ? Gf : Fyf;
      oyh = SY > 0 ? Gh : Fyh;
      iyf = SY > 0 ? Fyf : Gf;
      iyh = SY > 0 ? Fyh : Gh;
      if (clamped_row(in, ro(y - SY))) {
        iyf = oyf;
        iyh = oyh;
      }
      Fyf = Gf;
      Fyh = Gh;
    }
    if constexpr (HX && HY) {
      dF = (C.rdx * oxf + rdy * oyf) - (C.rdx * ixf + rdy * iyf);
      dH = (C.rdx * oxh + rdy * oyh) - (C.rdx * ixh + rdy * iyh);
    } else if constexpr (HX) {
      dF = C.rdx * oxf - C.rdx * ixf;
      dH = C.rdx * oxh - C.rdx * ixh;
    } else {
      dF = rdy * oyf - rdy * iyf;
      dH = rdy * oyh - rdy * iyh;
    }
  }
};

// One direction over the rows of a work item.
template <typename TS, typename TC, int MODE, bool SOLID, bool W5, int SX, int SY>
__device__ __forceinline__ void strip_dir(const StripInst<TS>& in, const StripLane<TC>& C, TC rf, TC rh, int I,
                                          int y0, int nrows, int flip, bool alive) {
  using M = March<TS, TC, SOLID, W5, SX, SY>;
  M m;
  m.setup(in, C, rf, rh, I);
  const RowOrder ro{flip, 2 * y0 + nrows - 1};
  const int pitch = in.pitch;
  // the planes the item writes (MODE 0, 2: the dF planes of direction I;
  // MODE 1: the state planes) and, MODE 1, those of direction I it reads:
  // the stored dF(f2)
  const gptr<TS> of = in.dst + (MODE == 1 ? (long long)I : (long long)(I - 1)) * in.P;
  const gptr<TS> oh = in.dst + (MODE == 1 ? (long long)(kQ + I) : (long long)(12 + I - 1)) * in.P;
  const gptr<const TS> df2 = in.dfl + (long long)(I - 1) * in.P;
  const gptr<const TS> dh2 = in.dfl + (long long)(12 + I - 1) * in.P;

  // Everything a row needs from memory, loaded one row ahead: the staged
  // position, the own cell's type as loaded (0 fluid; 1 for lanes without an
  // own cell), its row offset, (MODE 1) its stored dF(f2), and dt/dy of the
  // row (on a uniform grid the instance's own value, read with stride 0, so
  // that every row issues the same loads).
  struct Pre {
    SPos<TC> p;
    int ro, type;
    TS f, h;
    TC rdy;
  };
  auto fetch = [&](int y) {
    Pre r;
    r.p = m.next(in, C, ro, y);
    r.ro = ro(y) * pitch;
    r.type = 1;
    r.f = r.h = TS(0);
    if (C.own) {
      r.type = *at_col(in.ct + r.ro, C.X);
      if (MODE == 1) {
        r.f = *at_col(df2 + r.ro, C.X);
        r.h = *at_col(dh2 + r.ro, C.X);
      }
    }
    r.rdy = TC(in.rdyp[ro(y) * in.rdy_stride]);
    return r;
  };
  // a row's results, stored at the start of the next half iteration
  struct Res {
    int ro, on;
    TS vf, vh;
  };
  auto store = [&](const Res& r) {
    if (r.on) {
      *at_col(of + r.ro, C.X) = r.vf;
      *at_col(oh + r.ro, C.X) = r.vh;
    }
  };
  // row y from its prefetched data (registers only: no memory access)
  auto row = [&](int y, const Pre& cc) {
#pragma clang fp contract(off)
    TC dF, dH, of3, oh3;
    m.net(in, C, ro, y, cc.p, cc.rdy, dF, dH, of3, oh3);
    Res r;
    r.ro = cc.ro;
    r.on = alive && cc.type == 0;
    if (MODE != 1) {
      r.vf = TS(dF);
      r.vh = TS(dH);
    } else {
      // the new state f3 + (dF2 - dF3)/2, the final combination of the
      // stage-3 kernel; the own cell's f3 is the staged value of row y
      r.vf = TS(of3 + TC(0.5) * (TC(cc.f) - dF));
      r.vh = TS(oh3 + TC(0.5) * (TC(cc.h) - dH));
    }
    return r;
  };
  // Rows two at a time with two prefetch slots. Each half iteration starts
  // with one wait for every load and store in flight (on this GPU loads and
  // stores share the vector-memory counter, so any wait for a load with a
  // store pending waits for everything), which finds the previous half's
  // loads and stores complete after a whole row of arithmetic; then it
  // stores the previous row, issues the next row's loads into the other
  // slot and computes its row from registers.
  const int end = y0 + nrows;
  m.fill(in, C, ro, y0);
  Pre A = fetch(y0), B;
  if constexpr (M::HY) {
    __builtin_amdgcn_s_waitcnt(kWaitVmem);
    m.first_face();
  }
  Res R{0, 0, TS(0), TS(0)};
  for (int y = y0;; y += 2) {
    __builtin_amdgcn_s_waitcnt(kWaitVmem);
    store(R);
    if (y + 1 < end) B = fetch(y + 1);
    R = row(y, A);
    if (y + 1 >= end) break;
    __builtin_amdgcn_s_waitcnt(kWaitVmem);
    store(R);
    if (y + 2 < end) A = fetch(y + 2);
    R = row(y + 1, B);
    if (y + 2 >= end) break;
  }
  store(R);
}

// The instance fields and lane constants of a work item.
template <typename TS, typename TC>
__device__ __forceinline__ void strip_setup(const InstDev& in, const TileRef& sr, const void* src, void* dst,
                                            StripInst<TS>& si, StripLane<TC>& C) {
  const int lane = threadIdx.x & 63;
  const int x0 = sr.tx * kStripW, y0 = sr.ty, nrows = sr.flags >> kStripRowsBit;
  si.src = (gptr<const TS>)src;
  si.dst = (gptr<TS>)dst;
  si.dfl = (gptr<const TS>)in.dflux;
  si.ct = (gptr<const uint8_t>)in.ctype;
  si.alpha = (gptr<const double>)in.alpha;
  si.rdyp = (gptr<const double>)(in.rdys ? in.rdys : &in.rdy);
  si.rdy_stride = in.rdys ? 1 : 0;
  si.P = in.plane;
  si.pitch = in.pitch;
  si.ny = in.ny;
  si.py = in.flags & kPeriodicY;
  si.ms = in.flags & kMirrorS;
  si.mn = in.flags & kMirrorN;
  si.inner = y0 - kH >= 0 && y0 + nrows + kH <= in.ny;
  si.c = in.c;
  C.xl = x0 - kH + lane;
  const int px = in.flags & kPeriodicX, mw = in.flags & kMirrorW, me = in.flags & kMirrorE;
  unsigned mx, cx, mt, cl, cr;
  C.X = (unsigned)map_axis(C.xl, in.nx, px, mw, me, mx, cx);
  C.mx = (int)mx;
  si.colmir = __ballot(C.mx != 0) != 0;
  (void)map_axis(C.xl - 1, in.nx, px, mw, me, mt, cl);
  (void)map_axis(C.xl + 1, in.nx, px, mw, me, mt, cr);
  C.clampL = (int)cl;
  C.clampR = (int)cr;
  C.own = lane >= kH && lane < kH + kStripW && C.xl < in.nx;
  C.rdx = C.own ? TC(in.rdxs ? in.rdxs[C.xl] : in.rdx) : TC(0);
}

// One direction of a work item. desc: the item takes its rows from the last
// to the first in the directions with a y component. Items alternate between
// the two orders down each strip column (kStripDesc), so that two items one
// above the other reach the rows they share (each one's rows next to the
// other, read by the other as its y halo) at about the same time: the first
// read of such a row leaves it in L2 for the second.
template <typename TS, typename TC, int MODE, bool SOLID, bool W5>
__device__ __forceinline__ void strip_item(const InstDev& in, const StripInst<TS>& si, const StripLane<TC>& C,
                                           const TileRef& sr, int I, bool alive) {
  const int y0 = sr.ty, nrows = sr.flags >> kStripRowsBit;
  const int sx = c_lat_x[I] > 0 ? 1 : (c_lat_x[I] < 0 ? -1 : 0);
  const int sy0 = c_lat_y[I] > 0 ? 1 : (c_lat_y[I] < 0 ? -1 : 0);
  const int fl = (sr.flags & kStripDesc) != 0 && sy0 != 0;
  const int sy = fl ? -sy0 : sy0;  // the sign in the march's row order
  const TC rf = sizeof(TS) == 4 ? TC(in.ref[I]) : TC(0);
  const TC rh = sizeof(TS) == 4 ? TC(in.ref[kQ + I]) : TC(0);
  if (sy == 0) {
    if (sx > 0) strip_dir<TS, TC, MODE, SOLID, W5, 1, 0>(si, C, rf, rh, I, y0, nrows, 0, alive);
    else strip_dir<TS, TC, MODE, SOLID, W5, -1, 0>(si, C, rf, rh, I, y0, nrows, 0, alive);
  } else if (sx == 0) {
    if (sy > 0) strip_dir<TS, TC, MODE, SOLID, W5, 0, 1>(si, C, rf, rh, I, y0, nrows, fl, alive);
    else strip_dir<TS, TC, MODE, SOLID, W5, 0, -1>(si, C, rf, rh, I, y0, nrows, fl, alive);
  } else if (sy > 0) {
    if (sx > 0) strip_dir<TS, TC, MODE, SOLID, W5, 1, 1>(si, C, rf, rh, I, y0, nrows, fl, alive);
    else strip_dir<TS, TC, MODE, SOLID, W5, -1, 1>(si, C, rf, rh, I, y0, nrows, fl, alive);
  } else {
    if (sx > 0) strip_dir<TS, TC, MODE, SOLID, W5, 1, -1>(si, C, rf, rh, I, y0, nrows, fl, alive);
    else strip_dir<TS, TC, MODE, SOLID, W5, -1, -1>(si, C, rf, rh, I, y0, nrows, fl, alive);
  }
}

// Directions in the order a chunk of items takes them: the four with both
// components, which cost twice the others, first.
static __constant__ int c_strip_dir[12] = {5, 6, 7, 8, 2, 4, 10, 12, 1, 3, 9, 11};

// One wavefront per work item and direction, four items of one direction per
// workgroup. The items (in memory order) are cut into one contiguous chunk
// per XCD, whose blocks take the chunk direction by direction: neighbouring
// strips of a direction run together and share their halos in that XCD's L2.
template <typename TS, typename TC, int MODE>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(3))) void k_strip(
    const InstDev* __restrict__ insts, const TileRef* __restrict__ strips, int nstrips, int chunk, int all, int par,
    const int* stepp) {
  const int step = *stepp;
  const int per = chunk / 4, b = blockIdx.x / 8;
  const int I = c_strip_dir[b / per];
  const int it = __builtin_amdgcn_readfirstlane((int)(blockIdx.x % 8) * chunk + (b % per) * 4 + (int)(threadIdx.x >> 6));
  if (it >= nstrips) return;
  const TileRef sr = strips[it];
  const InstDev& in = insts[sr.inst];
  if (!all && !eq_kernel_for<TS, TC>(in)) return;  // FP32 storage: the other compute type's instance
  const bool alive = !frozen_by_failure(in, step);
  StripInst<TS> si;
  StripLane<TC> C;
  const void* src = MODE == 0 ? in.f2 : (MODE == 1 ? in.f3 : in.state[in.parity0 ^ par]);
  strip_setup<TS, TC>(in, sr, src, MODE == 1 ? in.state[1 ^ in.parity0 ^ par] : in.dflux, si, C);
  if (sr.flags & kTileSolid) {
    if (in.flux_method == 1) strip_item<TS, TC, MODE, true, true>(in, si, C, sr, I, alive);
    else strip_item<TS, TC, MODE, true, false>(in, si, C, sr, I, alive);
  } else {
    if (in.flux_method == 1) strip_item<TS, TC, MODE, false, true>(in, si, C, sr, I, alive);
    else strip_item<TS, TC, MODE, false, false>(in, si, C, sr, I, alive);
  }
}

// ---------------------------------------------------------------------------
// k_strip_mom: the stage-3 flux of FP32 storage. Beside the new state
// G - dF/2, each cell's net fluxes of all twelve directions are summed into
// the FP64 moment planes, so one workgroup takes all of them: four
// wavefronts march the same strip in step, each with one direction along x,
// one along y and one diagonal (four net faces for f and h each: equal work),
// and exchange a row's net fluxes through LDS; wavefront k then adds moment k
// over the directions in their order (the tile kernel's order, the same
// bits). One barrier per row: the rows alternate between two LDS buffers, so
// a wavefront writes a buffer again only after every other one has passed
// the barrier that follows its reads. Three marches per wavefront also
// overlap each other's dependent arithmetic. Bound by HBM on large groups, by
// the latency of one march on small ones. Against the tile kernel (twelve
// directions one after the other per tile, two barriers each): 256-member
// ensemble 3490 -> 2328 us per launch (2.4 -> 3.6 TB/s of its 352 B per
// cell), Riemann 3072^2 1384 -> 920, shear 256^2 35 -> 20, couette 64^2 36 -> 17.
// ---------------------------------------------------------------------------
template <typename TC>
struct MomRows {
  TC v[2][2 * (kQ - 1)][64];  // [buffer][f and h net flux of directions 1..12][lane]
};

// Wavefront w: directions c_mom_dir[w] (x, y, diagonal), all of x sign
// (w == 0 || w == 3) and y sign (w < 2).
static __constant__ int c_mom_dir[4][3] = {{quad_x(0), quad_y(0), quad_d(0)},
                                           {quad_x(1), quad_y(1), quad_d(1)},
                                           {quad_x(2), quad_y(2), quad_d(2)},
                                           {quad_x(3), quad_y(3), quad_d(3)}};

// Moment k (0 mass, 1 and 2 x and y momentum, 3 energy) of a row's net fluxes.
template <typename TC>
__device__ __forceinline__ double mom_sum(const TC (&v)[2 * (kQ - 1)][64], int lane, int k, double c) {
#pragma clang fp contract(off)
  double s = 0;
  if (k == 0) {
#pragma unroll
    for (int I = 1; I < kQ; I++) s += double(v[2 * (I - 1)][lane]);
  } else if (k == 1) {
#pragma unroll
    for (int I = 1; I < kQ; I++) s += double(v[2 * (I - 1)][lane]) * (lat_x(I) * c);
  } else if (k == 2) {
#pragma unroll
    for (int I = 1; I < kQ; I++) s += double(v[2 * (I - 1)][lane]) * (lat_y(I) * c);
  } else {
#pragma unroll
    for (int I = 1; I < kQ; I++) s += double(v[2 * (I - 1) + 1][lane]);
  }
  return s;
}

template <typename TS, typename TC, bool SOLID, bool W5, int SX, int SY>
__device__ __forceinline__ void strip_mom_rows(const InstDev& inst, const StripInst<TS>& in, const StripLane<TC>& C,
                                               const TileRef& sr, int w, int flip, bool alive, gptr<double> momp,
                                               MomRows<TC>& X) {
  static_assert(kStage3G<TS>, "moment sums belong to the stage-3 flux of FP32 storage");
  const int lane = threadIdx.x & 63, y0 = sr.ty, nrows = sr.flags >> kStripRowsBit, pitch = in.pitch;
  const int Ix = c_mom_dir[w][0], Iy = c_mom_dir[w][1], Id = c_mom_dir[w][2];
  March<TS, TC, SOLID, W5, SX, 0> mx;
  March<TS, TC, SOLID, W5, 0, SY> my;
  March<TS, TC, SOLID, W5, SX, SY> md;
  mx.setup(in, C, TC(inst.ref[Ix]), TC(inst.ref[kQ + Ix]), Ix);
  my.setup(in, C, TC(inst.ref[Iy]), TC(inst.ref[kQ + Iy]), Iy);
  md.setup(in, C, TC(inst.ref[Id]), TC(inst.ref[kQ + Id]), Id);
  const RowOrder ro{flip, 2 * y0 + nrows - 1};
  const gptr<double> mom = momp + (long long)w * in.P;
  const gptr<TS> st[6] = {in.dst + Ix * in.P, in.dst + (kQ + Ix) * in.P, in.dst + Iy * in.P, in.dst + (kQ + Iy) * in.P,
                          in.dst + Id * in.P, in.dst + (kQ + Id) * in.P};

  // A row's data from memory: the three staged positions, the own cell's
  // type, its six G values and its moment w, dt/dy.
  struct Pre {
    SPos<TC> px, py, pd;
    int ro, type;
    TS g[6];
    double m;
    TC rdy;
  };
  auto fetch = [&](int y) {
    Pre r;
    r.px = mx.next(in, C, ro, y);
    r.py = my.next(in, C, ro, y);
    r.pd = md.next(in, C, ro, y);
    r.ro = ro(y) * pitch;
    r.type = 1;
    r.m = 0;
#pragma unroll
    for (int k = 0; k < 6; k++) r.g[k] = TS(0);
    if (C.own) {
      r.type = *at_col(in.ct + r.ro, C.X);
#pragma unroll
      for (int k = 0; k < 6; k++) r.g[k] = *at_col(st[k] + r.ro, C.X);
      r.m = *at_col(mom + r.ro, C.X);
    }
    r.rdy = TC(in.rdyp[ro(y) * in.rdy_stride]);
    return r;
  };
  struct Res {
    int ro, on;
    TS v[6];
    double m;
  };
  auto store = [&](const Res& r) {
    if (r.on) {
#pragma unroll
      for (int k = 0; k < 6; k++) *at_col(st[k] + r.ro, C.X) = r.v[k];
      *at_col(mom + r.ro, C.X) = r.m;
    }
  };
  auto row = [&](int y, const Pre& cc, int buf) {
#pragma clang fp contract(off)
    TC d[6], a, b;
    mx.net(in, C, ro, y, cc.px, cc.rdy, d[0], d[1], a, b);
    my.net(in, C, ro, y, cc.py, cc.rdy, d[2], d[3], a, b);
    md.net(in, C, ro, y, cc.pd, cc.rdy, d[4], d[5], a, b);
    TC(&v)[2 * (kQ - 1)][64] = X.v[buf];
    v[2 * (Ix - 1)][lane] = d[0];
    v[2 * (Ix - 1) + 1][lane] = d[1];
    v[2 * (Iy - 1)][lane] = d[2];
    v[2 * (Iy - 1) + 1][lane] = d[3];
    v[2 * (Id - 1)][lane] = d[4];
    v[2 * (Id - 1) + 1][lane] = d[5];
    Res r;
    r.ro = cc.ro;
    r.on = alive && cc.type == 0;
#pragma unroll
    for (int k = 0; k < 6; k++) r.v[k] = TS(TC(cc.g[k]) - TC(0.5) * d[k]);
    // LDS only: the row's global loads and stores stay in flight across the
    // barrier (each wavefront reads and writes its own planes)
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
    r.m = cc.m - 0.5 * mom_sum(v, lane, w, in.c);
    return r;
  };
  // as strip_dir: one wait, the stores of the row before, the next row's loads
  const int end = y0 + nrows;
  my.fill(in, C, ro, y0);
  md.fill(in, C, ro, y0);
  Pre A = fetch(y0), B;
  __builtin_amdgcn_s_waitcnt(kWaitVmem);
  my.first_face();
  md.first_face();
  Res R{0, 0, {}, 0.0};
  for (int y = y0;; y += 2) {
    __builtin_amdgcn_s_waitcnt(kWaitVmem);
    store(R);
    if (y + 1 < end) B = fetch(y + 1);
    R = row(y, A, 0);
    if (y + 1 >= end) break;
    __builtin_amdgcn_s_waitcnt(kWaitVmem);
    store(R);
    if (y + 2 < end) A = fetch(y + 2);
    R = row(y + 1, B, 1);
    if (y + 2 >= end) break;
  }
  store(R);
}

template <typename TS, typename TC, bool SOLID, bool W5>
__device__ __forceinline__ void strip_mom_item(const InstDev& inst, const StripInst<TS>& si, const StripLane<TC>& C,
                                               const TileRef& sr, int w, bool alive, gptr<double> momp,
                                               MomRows<TC>& X) {
  const int fl = (sr.flags & kStripDesc) != 0;
  const bool px = w == 0 || w == 3, py = (w < 2) != (fl != 0);  // signs in the march's row order
  if (px && py) strip_mom_rows<TS, TC, SOLID, W5, 1, 1>(inst, si, C, sr, w, fl, alive, momp, X);
  else if (py) strip_mom_rows<TS, TC, SOLID, W5, -1, 1>(inst, si, C, sr, w, fl, alive, momp, X);
  else if (px) strip_mom_rows<TS, TC, SOLID, W5, 1, -1>(inst, si, C, sr, w, fl, alive, momp, X);
  else strip_mom_rows<TS, TC, SOLID, W5, -1, -1>(inst, si, C, sr, w, fl, alive, momp, X);
}

// One workgroup per work item, a contiguous chunk of the items per XCD.
template <typename TS, typename TC>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(3))) void k_strip_mom(
    const InstDev* __restrict__ insts, const TileRef* __restrict__ strips, int nstrips, int chunk, int par,
    const int* stepp) {
  __shared__ MomRows<TC> X;
  const int step = *stepp;
  const int it = (int)(blockIdx.x % 8) * chunk + (int)(blockIdx.x / 8);
  if (it >= nstrips) return;
  const int w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const TileRef sr = strips[it];
  const InstDev& in = insts[sr.inst];
  const bool alive = !frozen_by_failure(in, step);
  const int nxt = 1 ^ in.parity0 ^ par;
  StripInst<TS> si;
  StripLane<TC> C;
  strip_setup<TS, TC>(in, sr, in.f3, in.state[nxt], si, C);
  const gptr<double> momp = (gptr<double>)in.mom[nxt];
  if (sr.flags & kTileSolid) {
    if (in.flux_method == 1) strip_mom_item<TS, TC, true, true>(in, si, C, sr, w, alive, momp, X);
    else strip_mom_item<TS, TC, true, false>(in, si, C, sr, w, alive, momp, X);
  } else {
    if (in.flux_method == 1) strip_mom_item<TS, TC, false, true>(in, si, C, sr, w, alive, momp, X);
    else strip_mom_item<TS, TC, false, false>(in, si, C, sr, w, alive, momp, X);
  }
}

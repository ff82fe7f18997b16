// lbm_strip.hip — strip flux kernels (lbm_strip.hpp) and the wall closure
// kernel of the D2Q13 thermal FD-LBM, with their launchers.
#include <type_traits>

#include "lbm_point.hpp"
#include "lbm_stencil.hpp"

namespace uqlbm {

#include "lbm_strip.hpp"

// ---------------------------------------------------------------------------
// k_alpha: wall closure factor of each wall cell with a non-solid axis
// neighbour, from the neighbours' face fluxes of `which` (0: f2 or f1,
// 1: f3, 2: the current state),
// following the reference's physical stencil addressing (cpuLBM.cpp:1171-1326,
// 1502-1590).
// ---------------------------------------------------------------------------
static __constant__ int c_wall_dx[4] = {-1, 1, 0, 0};
static __constant__ int c_wall_dy[4] = {0, 0, -1, 1};
static __constant__ int c_wall_in[4][4] = {{1, 5, 8, 9}, {3, 6, 7, 11}, {2, 5, 6, 10}, {4, 7, 8, 12}};
static __constant__ int c_wall_out[4][4] = {{3, 6, 7, 11}, {1, 5, 8, 9}, {4, 8, 7, 12}, {2, 6, 5, 10}};

// Sixteen lanes per wall cell: lane 4 j + k forms the face flux of incoming
// direction k of neighbour j and the outgoing flux of its partner; the first
// lane adds the sixteen terms in the reference's order (j, then k; a solid
// neighbour's terms are zero). Bound by latency, not by bytes: a few hundred
// wall cells leave the GPU idle, and a face is one chain (types, line,
// extrapolation points, reconstruction). One lane per wall cell ran the up to
// sixteen chains one after the other: 20 us per launch on the 64^2 Couette
// deck and 55 us around a block in 301^2, 9 and 10 us with sixteen lanes.
constexpr int kWallLanes = 16, kWallBlock = 128;

template <typename TS, typename TC>
__global__ __launch_bounds__(kWallBlock) void k_alpha(const InstDev* __restrict__ insts,
                                                      const WallRef* __restrict__ walls, int nwalls, int which, int par,
                                                      const int* stepp) {
  __shared__ double fin[kWallBlock], fout[kWallBlock];
  const int step = *stepp;
  const int w = (blockIdx.x * kWallBlock + threadIdx.x) / kWallLanes, q = threadIdx.x % kWallLanes;
  const WallRef wr = walls[w < nwalls ? w : nwalls - 1];
  const InstDev& in = insts[wr.inst];
  const bool on = w < nwalls && !frozen_by_failure(in, step);
  const long long ow = (long long)wr.y * in.pitch + wr.x;
  double tf = 0, to = 0;
  if (on) {
    const int j = q / 4, k = q % 4, axis = j < 2 ? 0 : 1;
    int mx, my;
    const int xn = ref_index(in, wr.x, c_wall_dx[j], 0, my);
    const int yn = ref_index(in, wr.y, c_wall_dy[j], 1, mx);
    const long long on_ = (long long)yn * in.pitch + xn;
    if (in.ctype[on_] < 2) {
      const TS* src =
          reinterpret_cast<const TS*>(which == 0 ? in.f2 : (which == 1 ? in.f3 : in.state[in.parity0 ^ par]));
      const auto fv = [&](int p, long long o) { return full_val(in, src, p, o); };
      // the wall cell's own spacing: its axis neighbours share its row (x
      // faces) or column (y faces), so the face-length weights of a
      // non-uniform grid reduce to it
      const double dd = axis == 0 ? (in.dxs ? in.dxs[wr.x] : in.dx) : (in.dys ? in.dys[wr.y] : in.dy);
      const int i = c_wall_in[j][k], io = c_wall_out[j][k];
      const double F = double(ref_line_flux<TC>(in, fv, 0, xn, yn, i, axis));
      const double vv = fabs(double(axis == 0 ? c_lat_x[io] : c_lat_y[io]) * in.c);
      const double fw = full_val(in, src, io, ow);
      tf = F / dd;
      to = fw * vv / dd;
    }
  }
  fin[threadIdx.x] = tf;
  fout[threadIdx.x] = to;
  __syncthreads();
  if (on && q == 0) {
    double in_f = 0, out_f = 0;
#pragma unroll
    for (int n = 0; n < kWallLanes; n++) {
      in_f += fin[threadIdx.x + n];
      out_f += fout[threadIdx.x + n];
    }
    in.alpha[ow] = in_f / out_f;
  }
}

template <typename TS>
void launch_alpha(const StepLaunch& L, hipStream_t s, int which, int par, const int* step) {
  constexpr int cells = kWallBlock / kWallLanes;
  k_alpha<TS, double><<<(L.nwalls + cells - 1) / cells, kWallBlock, 0, s>>>(L.insts, L.walls, L.nwalls, which, par,
                                                                            step);
}

// Compute type of the strip kernels: FP64 for FP64 storage; FP32 for FP32
// storage near the reference equilibrium; for the other FP32-storage
// instances FP64 in large launch groups (StepLaunch::far64: on the 4096^2
// Riemann deck FP32 stencil arithmetic ended the mixed run at step 1939, FP64
// arithmetic completes the 2000 steps) and FP32 in small ones. A group that
// needs both has a launch of each over the same item list.
template <typename TS, typename TC, int MODE>
static void launch_strips_as(const StepLaunch& L, hipStream_t s, int par, int all) {
  const int chunk = (L.nstrips + 31) / 32 * 4;  // items per XCD, a multiple of a block's four
  k_strip<TS, TC, MODE><<<8 * 12 * (chunk / 4), 256, 0, s>>>(L.insts, L.strips, L.nstrips, chunk, all, par,
                                                              L.step_ctr + par);
}

template <typename TS, int MODE>
void launch_strips(const StepLaunch& L, hipStream_t s, int par) {
  if constexpr (sizeof(TS) == 4) {
    if ((L.eq_kinds & 2) || !L.far64) launch_strips_as<TS, float, MODE>(L, s, par, !L.far64);
    if ((L.eq_kinds & 1) && L.far64) launch_strips_as<TS, double, MODE>(L, s, par, 0);
  } else {
    launch_strips_as<TS, double, MODE>(L, s, par, 1);
  }
}

// Stage-3 flux of FP32 storage: FP32 stencils for every instance.
void launch_strips_mom(const StepLaunch& L, hipStream_t s, int par) {
  const int chunk = (L.nmstrips + 7) / 8;
  k_strip_mom<float, float><<<8 * chunk, 256, 0, s>>>(L.insts, L.mstrips, L.nmstrips, chunk, par,
                                                       L.step_ctr + par);
}

template void launch_alpha<double>(const StepLaunch&, hipStream_t, int, int, const int*);
template void launch_alpha<float>(const StepLaunch&, hipStream_t, int, int, const int*);
template void launch_strips<double, 0>(const StepLaunch&, hipStream_t, int);
template void launch_strips<double, 1>(const StepLaunch&, hipStream_t, int);
template void launch_strips<double, 2>(const StepLaunch&, hipStream_t, int);
template void launch_strips<float, 0>(const StepLaunch&, hipStream_t, int);
template void launch_strips<float, 2>(const StepLaunch&, hipStream_t, int);

}  // namespace uqlbm

// lbm_stencil.hpp — device and launch helpers shared by the kernel sources
// (lbm_kernels.hip, lbm_strip.hip): boundary mapping, work order, global
// pointers, solid extrapolation and the reference's physical addressing.
#pragma once

#include <hip/hip_runtime.h>

#include "lbm_device.hpp"
#include "lbm_launch.hpp"

namespace uqlbm {

constexpr int kH = 3;                          // stencil halo (WENO5 reach)

static __constant__ int c_lat_x[13] = {0, 1, 0, -1, 0, 1, -1, -1, 1, 2, 0, -2, 0};
static __constant__ int c_lat_y[13] = {0, 0, 1, 0, -1, 1, 1, -1, -1, 0, 2, 0, -2};
static __constant__ int c_mir_ns[13] = {0, 1, 4, 3, 2, 8, 7, 6, 5, 9, 12, 11, 10};
static __constant__ int c_mir_ew[13] = {0, 3, 2, 1, 4, 6, 5, 8, 7, 11, 10, 9, 12};

// Reference index() along one axis (cpuLBM.cpp:1033-1113) for one position,
// then a clamp into the grid for positions no stencil reaches.
__device__ __forceinline__ int map_axis(int X, int n, int periodic, int mir_lo, int mir_hi, unsigned& mir,
                                        unsigned& clamped) {
  mir = 0;
  clamped = 0;
  if (X < 0) {
    if (periodic) X += n;
    else if (mir_lo) { X = -X - 1; mir = 1; }
    else { X = 0; clamped = 1; }
  } else if (X > n - 1) {
    if (periodic) X -= n;
    else if (mir_hi) { X = 2 * n - X - 1; mir = 1; }
    else { X = n - 1; clamped = 1; }
  }
  return X < 0 ? 0 : (X > n - 1 ? n - 1 : X);
}

// Grid-stride tile loop with an XCD-aware order: gfx950 hands consecutive
// workgroups to its 8 XCDs in turn, so block b is renumbered so that each
// XCD walks a contiguous run of tiles (neighbouring tiles share halos and
// that XCD's L2).
__device__ __forceinline__ int first_tile() {
  const int G = gridDim.x, b = blockIdx.x;
  if (G % 8 != 0) return b;
  return (b % 8) * (G / 8) + b / 8;
}

// `step` counts the steps of the current launch sequence from 1; the global
// step index of an instance is in.step_base + step. A failure flagged during
// step s freezes the instance for steps > s only, so this test gives the
// same answer to every thread of a launch.
__device__ __forceinline__ bool frozen_by_failure(const InstDev& in, int step) {
  return *in.fail < in.step_base + step;
}

// Global-memory pointers: loads and stores through them are global, not
// flat, operations (the pointers read out of the instance table are
// generic), so they count on the vector-memory counter only: a flat access
// also counts on the LDS/scalar counter, and every wait for a scalar load
// then waits for it too.
template <typename T>
using gptr = __attribute__((address_space(1))) T*;

template <typename T>
__device__ __forceinline__ gptr<T> as_global(T* p) {
  return (gptr<T>)p;
}
template <typename T>
__device__ __forceinline__ gptr<T> as_global(gptr<T> p) {
  return p;
}

// Whether the pointwise kernel instantiated for equilibrium type TE takes
// instance `in`: FP32 storage picks the equilibrium precision per instance
// (InstDev::eq32), and a launch group with both kinds launches each
// pointwise kernel once per kind.
template <typename TS, typename TE>
__device__ __forceinline__ bool eq_kernel_for(const InstDev& in) {
  if constexpr (sizeof(TS) == 4) return (in.eq32 != 0) == (sizeof(TE) == 4);
  else return true;
}

constexpr int kWaitVmem = 0x0F70;  // s_waitcnt vmcnt(0): this wave's loads (also those into LDS) done

// Reference stencil solid handling along one line (cpuLBM.cpp:1242-1322):
// the first solid/fluid transition's solid point becomes 2 V(m1) - V(m2) of
// the two nearest fluid points, and the point beyond it the same value. The
// addressing equivalence with the reference is checked on the host per
// geometry (lbm_runtime.hip, validate_geometry).
// (The transition is located in the unrolled loop and the line updated in
// the same unrolled iteration, so every index is a constant and the stencil
// stays in registers.)
template <int L, typename TC>
__device__ __forceinline__ void extrapolate(const int* sld, const TC* V, TC* S) {
#pragma clang fp contract(off)
  bool found = false;
#pragma unroll
  for (int j = 0; j < L - 1; j++) {
    const int d = sld[j] - sld[j + 1];
    if (!found && d != 0) {
      found = true;
      if (d > 0) {  // solid point j, fluid beyond it at j+1, j+2
        const TC e = TC(2) * V[j + 1 < L ? j + 1 : L - 1] - V[j + 2 < L ? j + 2 : L - 1];
        S[j] = e;
        if (j - 1 >= 0) S[j - 1] = e;
      } else {      // solid point j+1, fluid before it at j, j-1
        const TC e = TC(2) * V[j] - V[j - 1 >= 0 ? j - 1 : 0];
        S[j + 1] = e;
        if (j + 2 < L) S[j + 2] = e;
      }
    }
  }
}

__device__ __forceinline__ int ref_index(const InstDev& in, int i, int pm, int d, int& mir) {
  unsigned m, cl;
  int r;
  if (d == 0)
    r = map_axis(i + pm, in.nx, in.flags & kPeriodicX, in.flags & kMirrorW, in.flags & kMirrorE, m, cl);
  else
    r = map_axis(i + pm, in.ny, in.flags & kPeriodicY, in.flags & kMirrorS, in.flags & kMirrorN, m, cl);
  mir = (int)m;
  return r;
}

// Value of plane k at offset o in FP64 (FP32 storage: deviation + reference).
template <typename TS>
__device__ __forceinline__ double full_val(const InstDev& in, const TS* src, int k, long long o) {
  if constexpr (sizeof(TS) == 4) return double(src[in.plane * k + o]) + in.ref[k];
  else return double(src[in.plane * k + o]);
}

// Face flux of distribution k0 + i (k0 = 0: f, kQ: h) out of fluid cell
// (x, y) along `axis`, with the reference's physical addressing: the
// stencil line through the mapped neighbours (direction remapped at a
// mirror), its first solid run extrapolated from the two nearest fluid
// points of the line in direction i; val(k, o) gives the FP64 value of
// plane k at offset o.
// (The loops are unrolled over the L points, so a line's loads go out
// together and every array index is a constant.)
template <int L, typename TC, typename Val>
__device__ TC ref_line(const InstDev& in, const Val& val, int k0, int x, int y, int i, int axis, int e) {
  const int s = e > 0 ? 1 : -1;
  constexpr int low = (L - 1) / 2;
  const int start = (axis == 0 ? x : y) - s * low;
  TC V[L];
  int sld[L], any = 0;
#pragma unroll
  for (int j = 0; j < L; j++) {
    int mir;
    const int p = ref_index(in, start, s * j, axis, mir);
    const int d = mir ? (axis == 0 ? c_mir_ew[i] : c_mir_ns[i]) : i;
    const long long o = axis == 0 ? (long long)y * in.pitch + p : (long long)p * in.pitch + x;
    V[j] = TC(val(k0 + d, o));
    sld[j] = in.ctype[o] == 2;
    any |= sld[j];
  }
  if (any) {
    int diff = 0, jj = 0, pos = 0, mir;
#pragma unroll
    for (int j = 0; j < L - 1; j++) {
      const int d = sld[j] - sld[j + 1];
      if (diff == 0 && d != 0) {
        diff = d;
        jj = d > 0 ? j : j + 1;
        pos = ref_index(in, start, s * jj, axis, mir);
      }
    }
    const int m1 = ref_index(in, pos, s * diff, axis, mir);
    const int m2 = ref_index(in, pos, s * 2 * diff, axis, mir);
    const long long o1 = axis == 0 ? (long long)y * in.pitch + m1 : (long long)m1 * in.pitch + x;
    const long long o2 = axis == 0 ? (long long)y * in.pitch + m2 : (long long)m2 * in.pitch + x;
    const TC ex = TC(2) * TC(val(k0 + i, o1)) - TC(val(k0 + i, o2));
    const int nx = jj - diff;
#pragma unroll
    for (int j = 0; j < L; j++)
      if (j == jj || j == nx) V[j] = ex;
  }
  const TC v = TC(double(e > 0 ? e : -e) * in.c);
  if constexpr (L == 5) return weno5(v, V[0], V[1], V[2], V[3], V[4]);
  else return nnd(v, V[0], V[1], V[2]);
}

template <typename TC, typename Val>
__device__ __forceinline__ TC ref_line_flux(const InstDev& in, const Val& val, int k0, int x, int y, int i, int axis) {
  const int e = axis == 0 ? c_lat_x[i] : c_lat_y[i];
  if (e == 0) return TC(0);
  return in.flux_method == 1 ? ref_line<5, TC>(in, val, k0, x, y, i, axis, e)
                             : ref_line<3, TC>(in, val, k0, x, y, i, axis, e);
}

static int grid_for(const void* kernel, int threads, int max_per = 0) {
  int dev = 0, cus = 256, per = 4;
  (void)hipGetDevice(&dev);
  hipDeviceProp_t prop;
  if (hipGetDeviceProperties(&prop, dev) == hipSuccess) cus = prop.multiProcessorCount;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, kernel, threads, 0) != hipSuccess || per < 1) per = 1;
  if (max_per > 0 && per > max_per) per = max_per;
  long long g = (long long)cus * per;
  g -= g % 8;
  return (int)(g < 8 ? 8 : g);
}

static int blocks_for(int ntiles, int g) { return ntiles <= g ? ntiles : g; }

}  // namespace uqlbm

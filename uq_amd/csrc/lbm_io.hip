// lbm_io.hip — the boundary's arrays: distributions between the state planes
// and the caller's [x][y][i] order, transposed on the device, and the copies
// between device buffers and the caller's (pageable) host arrays.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cstring>
#include <exception>
#include <memory>
#include <mutex>
#include <thread>
#include <vector>

#include "lbm_runtime.hpp"
#include "lbm_stencil.hpp"

namespace uqlbm {

// ---------------------------------------------------------------------------
// Distributions in the boundary's order. One workgroup takes 16 x 16 cells:
// the planes are read and written in 16-cell row segments, the boundary's
// arrays (13 values per cell, y fastest) in runs of 16 x 13 values, through
// LDS (13 is odd: no bank conflicts either way). Bound by HBM; the transposes
// ran on one host core before, 3 ns per value.
// ---------------------------------------------------------------------------
constexpr int kIoT = 16;  // cells of a tile along x and y

// The values of a cell in FP64: as stored, or (FP32 storage) deviation plus
// reference with the moment correction of load_state (contraction off: the
// same roundings wherever this is evaluated).
template <typename TS>
__device__ __forceinline__ void cell_values(const InstDev& in, const TS* st, const double* mom, long long o, double* f,
                                            double* h) {
#pragma clang fp contract(off)
  const long long P = in.plane;
#pragma unroll
  for (int i = 0; i < kQ; i++) {
    f[i] = double(st[P * i + o]);
    h[i] = double(st[P * (kQ + i) + o]);
  }
  if constexpr (sizeof(TS) == 4) {
    double t[4] = {0, 0, 0, 0};
#pragma unroll
    for (int i = 0; i < kQ; i++) {
      f[i] += in.ref[i];
      h[i] += in.ref[kQ + i];
      t[0] += f[i];
      t[1] += f[i] * (lat_x(i) * in.c);
      t[2] += f[i] * (lat_y(i) * in.c);
      t[3] += h[i];
    }
    const double dx = (mom[P + o] - t[1]) * in.i2c, dy = (mom[2 * P + o] - t[2]) * in.i2c;
    f[0] += mom[o] - t[0];
    f[1] += dx;
    f[3] -= dx;
    f[2] += dy;
    f[4] -= dy;
    h[0] += mom[3 * P + o] - t[3];
  }
}

// A tile's values of f or h between the cells' lanes and an [x][y][i] array.
__device__ __forceinline__ void tile_to_array(double (&v)[kIoT * kIoT * kQ], double* out, int x0, int y0, int nx,
                                              int ny) {
  __syncthreads();
  for (int k = threadIdx.x; k < kIoT * kIoT * kQ; k += kIoT * kIoT) {
    const int lx = k / (kIoT * kQ), r = k % (kIoT * kQ), ly = r / kQ, i = r % kQ;
    if (x0 + lx < nx && y0 + ly < ny)
      out[((long long)(x0 + lx) * ny + y0) * kQ + r] = v[(ly * kIoT + lx) * kQ + i];
  }
  __syncthreads();
}

__device__ __forceinline__ void array_to_tile(double (&v)[kIoT * kIoT * kQ], const double* src, int x0, int y0, int nx,
                                              int ny) {
  __syncthreads();
  for (int k = threadIdx.x; k < kIoT * kIoT * kQ; k += kIoT * kIoT) {
    const int lx = k / (kIoT * kQ), r = k % (kIoT * kQ), ly = r / kQ, i = r % kQ;
    if (x0 + lx < nx && y0 + ly < ny)
      v[(ly * kIoT + lx) * kQ + i] = src[((long long)(x0 + lx) * ny + y0) * kQ + r];
  }
  __syncthreads();
}

template <typename TS>
__global__ __launch_bounds__(kIoT* kIoT) void k_dist_out(const InstDev* insts, const TS* st, const double* mom,
                                                         double* fo, double* ho) {
  __shared__ double v[kIoT * kIoT * kQ];
  const InstDev& in = insts[0];
  const int lx = threadIdx.x % kIoT, ly = threadIdx.x / kIoT;
  const int tw = (in.nx + kIoT - 1) / kIoT, n = tw * ((in.ny + kIoT - 1) / kIoT);
  for (int t = blockIdx.x; t < n; t += gridDim.x) {
    const int x0 = t % tw * kIoT, y0 = t / tw * kIoT;
    double f[kQ], h[kQ];
    if (x0 + lx < in.nx && y0 + ly < in.ny)
      cell_values(in, st, mom, (long long)(y0 + ly) * in.pitch + x0 + lx, f, h);
    else
      for (int i = 0; i < kQ; i++) f[i] = h[i] = 0.0;
    if (fo) {
#pragma unroll
      for (int i = 0; i < kQ; i++) v[threadIdx.x * kQ + i] = f[i];
      tile_to_array(v, fo, x0, y0, in.nx, in.ny);
    }
    if (ho) {
#pragma unroll
      for (int i = 0; i < kQ; i++) v[threadIdx.x * kQ + i] = h[i];
      tile_to_array(v, ho, x0, y0, in.nx, in.ny);
    }
  }
}

// fi, hi: the new values, or null to keep the cell's.
template <typename TS>
__global__ __launch_bounds__(kIoT* kIoT) void k_dist_in(const InstDev* insts, TS* st, double* mom, const double* fi,
                                                        const double* hi) {
#pragma clang fp contract(off)
  __shared__ double v[kIoT * kIoT * kQ];
  const InstDev& in = insts[0];
  const long long P = in.plane;
  const int lx = threadIdx.x % kIoT, ly = threadIdx.x / kIoT;
  const int tw = (in.nx + kIoT - 1) / kIoT, n = tw * ((in.ny + kIoT - 1) / kIoT);
  for (int t = blockIdx.x; t < n; t += gridDim.x) {
    const int x0 = t % tw * kIoT, y0 = t / tw * kIoT;
    const bool on = x0 + lx < in.nx && y0 + ly < in.ny;
    const long long o = on ? (long long)(y0 + ly) * in.pitch + x0 + lx : 0;
    double f[kQ], h[kQ];
    if (on && (!fi || !hi)) cell_values(in, st, mom, o, f, h);
    if (fi) {
      array_to_tile(v, fi, x0, y0, in.nx, in.ny);
      if (on)
#pragma unroll
        for (int i = 0; i < kQ; i++) f[i] = v[threadIdx.x * kQ + i];
    }
    if (hi) {
      array_to_tile(v, hi, x0, y0, in.nx, in.ny);
      if (on)
#pragma unroll
        for (int i = 0; i < kQ; i++) h[i] = v[threadIdx.x * kQ + i];
    }
    if (!on) continue;
    double m[4] = {0, 0, 0, 0};
#pragma unroll
    for (int i = 0; i < kQ; i++) {
      st[P * i + o] = TS(sizeof(TS) == 4 ? f[i] - in.ref[i] : f[i]);
      st[P * (kQ + i) + o] = TS(sizeof(TS) == 4 ? h[i] - in.ref[kQ + i] : h[i]);
      m[0] += f[i];
      m[1] += f[i] * (lat_x(i) * in.c);
      m[2] += f[i] * (lat_y(i) * in.c);
      m[3] += h[i];
    }
    if constexpr (sizeof(TS) == 4)
#pragma unroll
      for (int k = 0; k < 4; k++) mom[k * P + o] = m[k];
  }
}

static int io_blocks(const Solver& s) {
  const long long n = (long long)((s.nx + kIoT - 1) / kIoT) * ((s.ny + kIoT - 1) / kIoT);
  return (int)std::min<long long>(n, 4096);
}

void launch_dist_out(Solver& s, double* f, double* h) {
  if (s.precision == LBM_PREC_FP64)
    k_dist_out<double><<<io_blocks(s), kIoT * kIoT, 0, s.stream>>>(s.inst_dev, (const double*)s.state[s.cur], nullptr, f, h);
  else
    k_dist_out<float><<<io_blocks(s), kIoT * kIoT, 0, s.stream>>>(s.inst_dev, (const float*)s.state[s.cur], s.mom[s.cur], f, h);
}

void launch_dist_in(Solver& s, const double* f, const double* h) {
  if (s.precision == LBM_PREC_FP64)
    k_dist_in<double><<<io_blocks(s), kIoT * kIoT, 0, s.stream>>>(s.inst_dev, (double*)s.state[s.cur], nullptr, f, h);
  else
    k_dist_in<float><<<io_blocks(s), kIoT * kIoT, 0, s.stream>>>(s.inst_dev, (float*)s.state[s.cur], s.mom[s.cur], f, h);
}

// ---------------------------------------------------------------------------
// Copies between a device buffer and the caller's host arrays, through pinned
// slots: a piece of kSlotBytes is moved by DMA to or from a slot and by a host
// thread to or from the caller's memory. Up to kCopyThreads threads take the
// pieces in turn, each with a slot and a stream of its own, so that the DMA of
// one piece overlaps the host copies (and the first-touch page faults) of
// others; a copy of one piece runs on the solver's stream in the calling
// thread. The five fields of 3072^2 cells (377 MB) take 10 ms (38 GB/s; the DMA
// alone 57 GB/s), against 420 ms with one pageable copy and a transpose on one
// core; a 256^2 checkpoint in and out 1.5 ms against 18 ms.
//
// Slots are kept for later copies, at most kSlotsKept of them in all
// (lbm_release_cached returns them); a slot belongs to one copying thread at a
// time, so copies of several threads do not wait for each other.
// ---------------------------------------------------------------------------
namespace {
constexpr size_t kSlotBytes = size_t(2) << 20;
constexpr int kCopyThreads = 8;
constexpr size_t kSlotsKept = 16;

struct Slot {
  int dev = 0;
  char* buf = nullptr;
  hipStream_t stream = nullptr;
};

void free_slot(const Slot& s) {
  if (s.stream) (void)hipStreamDestroy(s.stream);
  if (s.buf) (void)hipHostFree(s.buf);
}

struct SlotPool {
  std::mutex mu;
  std::vector<Slot> free;
};
SlotPool& slot_pool() {
  static SlotPool* p = [] {
    SlotPool* q = new SlotPool();  // never destroyed: outlives every solver
    q->free.reserve(kSlotsKept);   // ~SlotUse gives slots back without an allocation
    return q;
  }();
  return *p;
}

// A slot of device `dev` for the lifetime of this object.
struct SlotUse {
  Slot s;
  hipError_t err = hipSuccess;
  explicit SlotUse(int dev) {
    SlotPool& p = slot_pool();
    {
      std::lock_guard<std::mutex> lock(p.mu);
      for (size_t k = 0; k < p.free.size(); k++)
        if (p.free[k].dev == dev) {
          s = p.free[k];
          p.free.erase(p.free.begin() + k);
          return;
        }
    }
    s.dev = dev;
    err = hipHostMalloc((void**)&s.buf, kSlotBytes, hipHostMallocDefault);
    if (err == hipSuccess) err = hipStreamCreateWithFlags(&s.stream, hipStreamNonBlocking);
  }
  ~SlotUse() {
    if (err == hipSuccess) {
      SlotPool& p = slot_pool();
      std::lock_guard<std::mutex> lock(p.mu);
      if (p.free.size() < kSlotsKept) {
        p.free.push_back(s);
        return;
      }
    }
    free_slot(s);
  }
};

// The part [a, b) of the device range between a slot and the host segments
// (`segs` cover the range in order; null host pointers are skipped).
void host_piece(const std::vector<HostSeg>& segs, bool out, char* slot, size_t a, size_t b) {
  size_t at = 0;
  for (const HostSeg& g : segs) {
    const size_t lo = std::max(a, at), hi = std::min(b, at + g.bytes);
    if (lo < hi && g.host) {
      char* host = (char*)g.host + (lo - at);
      if (out) std::memcpy(host, slot + (lo - a), hi - lo);
      else std::memcpy(slot + (lo - a), host, hi - lo);
    }
    at += g.bytes;
  }
}

// The same part between the device range and the host segments, without a slot.
hipError_t direct_piece(char* dev, const std::vector<HostSeg>& segs, bool out, size_t a, size_t b, hipStream_t stream) {
  size_t at = 0;
  for (const HostSeg& g : segs) {
    const size_t lo = std::max(a, at), hi = std::min(b, at + g.bytes);
    if (lo < hi && g.host) {
      char* host = (char*)g.host + (lo - at);
      const hipError_t e = out ? hipMemcpyAsync(host, dev + lo, hi - lo, hipMemcpyDeviceToHost, stream)
                               : hipMemcpyAsync(dev + lo, host, hi - lo, hipMemcpyHostToDevice, stream);
      const hipError_t e2 = hipStreamSynchronize(stream);
      if (e != hipSuccess || e2 != hipSuccess) return e != hipSuccess ? e : e2;
    }
    at += g.bytes;
  }
  return hipSuccess;
}
}  // namespace

void release_slots() {
  SlotPool& p = slot_pool();
  std::lock_guard<std::mutex> lock(p.mu);
  for (const Slot& s : p.free) free_slot(s);
  p.free.clear();
}

// out: device to host, else host to device. The device range is complete on
// `stream` when the copy starts, and the copy is complete on return.
hipError_t staged_copy(char* dev, const std::vector<HostSeg>& segs, bool out, hipStream_t stream) {
  size_t total = 0;
  for (const HostSeg& g : segs) total += g.bytes;
  const size_t n = (total + kSlotBytes - 1) / kSlotBytes;
  if (n == 0) return hipSuccess;
  int device = 0;
  (void)hipGetDevice(&device);
  std::atomic<int> err{(int)hipSuccess};
  auto pieces = [&](size_t first, size_t step, bool own_stream) {
    SlotUse u(device);
    if (u.err != hipSuccess) {  // no pinned memory to be had: pageable copies
      (void)hipGetLastError();
      hipError_t e = hipSuccess;
      for (size_t k = first; k < n && e == hipSuccess; k += step)
        e = direct_piece(dev, segs, out, k * kSlotBytes, std::min(total, (k + 1) * kSlotBytes), stream);
      if (e != hipSuccess) err.store((int)e);
      return;
    }
    hipError_t e = hipSuccess;
    const hipStream_t st = own_stream ? u.s.stream : stream;
    for (size_t k = first; k < n && e == hipSuccess && err.load() == (int)hipSuccess; k += step) {
      const size_t a = k * kSlotBytes, b = std::min(total, a + kSlotBytes);
      if (!out) host_piece(segs, out, u.s.buf, a, b);
      e = out ? hipMemcpyAsync(u.s.buf, dev + a, b - a, hipMemcpyDeviceToHost, st)
              : hipMemcpyAsync(dev + a, u.s.buf, b - a, hipMemcpyHostToDevice, st);
      const hipError_t e2 = hipStreamSynchronize(st);
      if (e == hipSuccess) e = e2;
      if (out && e == hipSuccess) host_piece(segs, out, u.s.buf, a, b);
    }
    if (e != hipSuccess) err.store((int)e);
  };
  if (n == 1) {
    pieces(0, 1, false);
    return (hipError_t)err.load();
  }
  hipError_t e = hipStreamSynchronize(stream);
  if (e != hipSuccess) return e;
  const unsigned hw = std::max(1u, std::thread::hardware_concurrency());
  const size_t workers = std::min({n, (size_t)kCopyThreads, (size_t)hw});
  std::vector<std::thread> threads;
  threads.reserve(workers);
  std::vector<size_t> here{0};  // shares of the calling thread: its own, and those no thread could be made for
  here.reserve(workers);
  for (size_t w = 1; w < workers; w++) {
    try {
      threads.emplace_back([&, w] {
        (void)hipSetDevice(device);
        pieces(w, workers, true);
      });
    } catch (const std::exception&) {  // std::system_error, std::bad_alloc
      here.push_back(w);
    }
  }
  for (size_t w : here) pieces(w, workers, true);
  for (std::thread& t : threads) t.join();
  return (hipError_t)err.load();
}

}  // namespace uqlbm

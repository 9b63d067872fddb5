// Step and right-hand-side kernels for any K: the march of channel groups (pf_device.h quad_march),
// and one thread per cell for K of more groups than a workgroup has threads.
#include "pf_host.h"

namespace pf {

template <class TS, bool ANISO, int MODE, int V, bool TAIL>
__global__ __launch_bounds__(kQuadT) void quad_kernel(const StepDev a, const StepDyn d, const RkStage rk) {
  __shared__ QuadLds<TS, V> lds;
  extern __shared__ __attribute__((aligned(16))) char axmem[];
  int run, layer;
  if (quad_tile(a, blockIdx.x, run, layer))
    quad_march<TS, ANISO, MODE, V, TAIL>(a, d, rk, run, layer, lds, (typename Traits<TS>::TC*)axmem);
}

// Batched: work items are (slot, workgroup of the slot's own launch).
template <class TS, bool ANISO, int V, bool TAIL>
__global__ __launch_bounds__(kQuadT) void batch_quad_kernel(const BatchView v, int cls, int step) {
  __shared__ QuadLds<TS, V> lds;
  extern __shared__ __attribute__((aligned(16))) char axmem[];
  const int2 ci = constant_at(v.cinfo, cls);
  for (int w = blockIdx.x; w < ci.y; w += gridDim.x) {
    const WorkItem it = constant_at(v.work, ci.x + w);
    const BatchSlot& s = constant_at(v.slots, it.slot);
    const StepDev& a = constant_at(v.descs, it.path ? (1LL + step) * v.inst + it.slot : it.slot);
    const StepDyn& d = constant_at(v.dyns, (long long)step * v.inst + it.slot);
    if (s.steps_left <= step || !s.active) continue;
    int run, layer;
    if (!quad_tile(a, it.tile, run, layer)) continue;
    quad_march<TS, ANISO, kStep, V, TAIL>(a, d, RkStage(), run, layer, lds,
                                              (typename Traits<TS>::TC*)axmem);
    lds_barrier();  // LDS is reused by the next item
  }
}

template <class TS, bool ANISO, bool RHS>
__global__ __launch_bounds__(256) void generic_kernel(const StepDev a, const StepDyn d) {
  const long long n = (long long)a.nz * a.ny * a.nx;
  const long long cell = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (cell < n) generic_cell<TS, ANISO, RHS>(a, d, cell);
}

// Batched, one thread per cell: work items are (slot, block of 256 cells).
template <class TS, bool ANISO>
__global__ __launch_bounds__(256) void batch_generic_kernel(const BatchView v, int cls, int step) {
  const int2 ci = constant_at(v.cinfo, cls);
  for (int w = blockIdx.x; w < ci.y; w += gridDim.x) {
    const WorkItem it = constant_at(v.work, ci.x + w);
    const BatchSlot& s = constant_at(v.slots, it.slot);
    const StepDev& a = constant_at(v.descs, it.path ? (1LL + step) * v.inst + it.slot : it.slot);
    const StepDyn& d = constant_at(v.dyns, (long long)step * v.inst + it.slot);
    if (s.steps_left <= step || !s.active) continue;
    const long long n = (long long)a.nz * a.ny * a.nx;
    const long long cell = (long long)it.tile * 256 + threadIdx.x;
    if (cell < n) generic_cell<TS, ANISO>(a, d, cell);
  }
}

// channels per thread: a full group where K holds one, else single channels
static int quad_v(int dtype, int K) {
  const int cap = dtype == PF_F64 ? 2 : 4;
  return K >= cap ? cap : 1;
}
// at most half a workgroup's threads per cell: the axis table of an anisotropic K stays under 25 KB
bool quad_fits(int dtype, int K) {
  const int V = quad_v(dtype, K);
  return (K + V - 1) / V <= kQuadT / 2;
}
static size_t ax_bytes(int k, int tc, bool aniso) { return aniso ? (size_t)12 * k * tc : 16; }

long long quad_threads(int dtype, int k, long long cells) {
  const int V = quad_v(dtype, k);
  return cells * ((k + V - 1) / V);
}

long long set_quads(StepDev& a, int dtype, int zc) {
  const long long nxy = (long long)a.nx * a.ny;
  if (!quad_fits(dtype, a.k)) return (nxy * a.nz + 255) / 256;
  const int V = quad_v(dtype, a.k), Q = (a.k + V - 1) / V, C = kQuadT / Q;
  const long long runs = (nxy + C - 1) / C;
  if (zc <= 0) {
    // the shortest marches whose workgroups are all resident at once
    const long long per = (runs + 7) / 8 * 8, chunks = kQuadBlocks > per ? kQuadBlocks / per : 1;
    zc = (int)((a.nz + chunks - 1) / chunks);
  }
  if (zc > kQuadTab / C) zc = kQuadTab / C;
  if (zc > a.nz) zc = a.nz;
  a.zc = a.zs = zc;
  a.zsplit = 0;
  a.tiles_x = (int)runs;
  a.tiles_y = (int)((runs + 7) / 8);
  a.tiles_z = (a.nz + zc - 1) / zc;
  return 8LL * a.tiles_y * a.tiles_z;
}

template <class TS, bool ANISO, bool RHS>
static hipError_t launch_cells(const StepDev& a, const StepDyn& d, hipStream_t s) {
  const long long n = (long long)a.nz * a.ny * a.nx;
  generic_kernel<TS, ANISO, RHS><<<dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s>>>(a, d);
  return hipGetLastError();
}

template <class TS, bool ANISO, int MODE>
static hipError_t launch_quad_mode(const StepDev& a, const StepDyn& d, const RkStage& rk, hipStream_t s) {
  using TC = typename Traits<TS>::TC;
  constexpr int dt = Traits<TS>::dtype;
  const unsigned nb = 8u * a.tiles_y * a.tiles_z;
  const size_t sh = ax_bytes(a.k, sizeof(TC), ANISO);
  const int V = quad_v(dt, a.k);
  if (V == 1) quad_kernel<TS, ANISO, MODE, 1, false><<<nb, kQuadT, sh, s>>>(a, d, rk);
  else if (a.k % V == 0) quad_kernel<TS, ANISO, MODE, quad_cap<TS>(), false><<<nb, kQuadT, sh, s>>>(a, d, rk);
  else quad_kernel<TS, ANISO, MODE, quad_cap<TS>(), true><<<nb, kQuadT, sh, s>>>(a, d, rk);
  return hipGetLastError();
}

template <class TS, bool ANISO, bool RHS>
static hipError_t launch_quad(const StepDev& a, const StepDyn& d, hipStream_t s) {
  // a launch has fewer than 2^32 threads; planes of a few cells by very many planes would need more
  if (8LL * a.tiles_y * a.tiles_z >= kQuadLaunch) return launch_cells<TS, ANISO, RHS>(a, d, s);
  return launch_quad_mode<TS, ANISO, RHS ? kRhs : kStep>(a, d, RkStage(), s);
}

template <class TS>
static hipError_t launch_rk(const StepDev& a, const StepDyn& d, const RkStage& rk, bool aniso, hipStream_t s) {
  return aniso ? launch_quad_mode<TS, true, kRk>(a, d, rk, s) : launch_quad_mode<TS, false, kRk>(a, d, rk, s);
}

hipError_t rk_stage(const StepDev& a, const StepDyn& d, const RkStage& rk, int dtype, bool aniso, hipStream_t s) {
  return dtype == PF_F64   ? launch_rk<double>(a, d, rk, aniso, s)
         : dtype == PF_F32 ? launch_rk<float>(a, d, rk, aniso, s)
                           : launch_rk<bf16_t>(a, d, rk, aniso, s);
}

template <class TS, bool ANISO, int V, bool TAIL>
static hipError_t launch_batch_quad(const BatchView& v, int cls, int i, int grid, int k, hipStream_t s) {
  batch_quad_kernel<TS, ANISO, V, TAIL>
      <<<dim3(grid), dim3(kQuadT), ax_bytes(k, sizeof(typename Traits<TS>::TC), ANISO), s>>>(v, cls, i);
  return hipGetLastError();
}

template <class TS, bool ANISO>
static hipError_t launch_batch_cells(const BatchView& v, int cls, int i, int grid, int, hipStream_t s) {
  batch_generic_kernel<TS, ANISO><<<dim3(grid), dim3(256), 0, s>>>(v, cls, i);
  return hipGetLastError();
}

template <class TS, bool RHS> static StepLaunch pick(int k, bool aniso) {
  if (quad_fits(Traits<TS>::dtype, k)) return aniso ? &launch_quad<TS, true, RHS> : &launch_quad<TS, false, RHS>;
  return aniso ? &launch_cells<TS, true, RHS> : &launch_cells<TS, false, RHS>;
}
template <class TS, bool ANISO> static BatchLaunch pick_batch(int k) {
  const int V = quad_v(Traits<TS>::dtype, k);
  if (!quad_fits(Traits<TS>::dtype, k)) return &launch_batch_cells<TS, ANISO>;
  if (V == 1) return &launch_batch_quad<TS, ANISO, 1, false>;
  return k % V == 0 ? &launch_batch_quad<TS, ANISO, quad_cap<TS>(), false>
                    : &launch_batch_quad<TS, ANISO, quad_cap<TS>(), true>;
}

StepLaunch generic_step(int dtype, int k, bool aniso) {
  return dtype == PF_F64   ? pick<double, false>(k, aniso)
         : dtype == PF_F32 ? pick<float, false>(k, aniso)
                           : pick<bf16_t, false>(k, aniso);
}
StepLaunch generic_rhs(int dtype, int k, bool aniso) {
  return dtype == PF_F64   ? pick<double, true>(k, aniso)
         : dtype == PF_F32 ? pick<float, true>(k, aniso)
                           : pick<bf16_t, true>(k, aniso);
}
BatchLaunch generic_batch(int dtype, int k, bool aniso) {
  switch (dtype) {
    case PF_F64: return aniso ? pick_batch<double, true>(k) : pick_batch<double, false>(k);
    case PF_F32: return aniso ? pick_batch<float, true>(k) : pick_batch<float, false>(k);
    default: return aniso ? pick_batch<bf16_t, true>(k) : pick_batch<bf16_t, false>(k);
  }
}

}  // namespace pf

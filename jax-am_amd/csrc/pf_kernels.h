// Kernel entry points of the fused step (single instance and batched), their
// launchers, and the dispatch-table entry type.  Instantiated per storage dtype in
// pf_inst_*.hip.
#pragma once

#include "pf_device.h"

namespace pf {

// Per-slot device state of the batched engine.  The step index n gives
// t_prev = t0 + n*dt and t_crt = t0 + (n+1)*dt (the reference's np.arange time grid,
// applications/phase_field/simple/example.py:52), so h = t_crt - t_prev per step.
struct BatchSlot {
  int steps_left;
  int parity;  // state lives in eta[parity]
  int n;
  int active;
  double t0, dt;
  void* eta[2];
  double tnow;         // time of the current state
  const double* path;  // per-step rows (PF_PATH_ROW values, include/pfhip.h) of a source table, or null
};

// A source-table row's position, direction, strength and speed into an instance description:
// the fields make_stepdev derives from pf_laser_t pos0, dir, Q (Rosenthal) or dT_peak
// (Gaussian) and vel, with the same expressions, so a row gives bitwise the description that
// pf_step builds from a descriptor holding those values.
__host__ __device__ inline void apply_path_row(StepDev& a, const double* r) {
  a.p0x = r[2];
  a.p0y = r[3];
  a.p0z = r[4];
  a.dirx = r[5];
  a.diry = r[6];
  a.dirz = r[7];
  a.vel = r[9];
  if (a.tmodel == PF_T_ROSENTHAL) {
    a.q_coef = rosenthal_q(r[8], a.kappa_T);
    a.pe = rosenthal_pe(r[9], a.alpha);
  } else {
    a.dT_peak = r[8];
  }
}

struct WorkItem {
  int slot;
  int tile;
  int path;  // 1: the slot has a source table (its descriptions are planned per step)
  int pad;
};

// The engine's device tables.  Slots change only between blocks of up to kPlan steps; the step arguments
// of a block's steps, and the descriptions of slots with a source table (whose source differs from step
// to step), are planned ahead by advance_kernel: dyns[i * inst + s] and descs[(1 + i) * inst + s] for
// step i of the block, descs[s] for every other slot.
constexpr int kPlan = 8;
struct BatchView {
  const StepDev* descs;
  const StepDyn* dyns;
  const BatchSlot* slots;
  const WorkItem* work;
  const int2* cinfo;  // per class (offset, count) of its work list
  int inst;
};

// An element of a table in the constant address space.  A launch does not change the tables it reads,
// but the compiler can not know: through ordinary pointers it reads what is uniform in a slot's description
// again after the first barrier by per-lane loads, into vector registers.  Loads from this address
// space are scalar and may be repeated anywhere, as those of kernel arguments.  A step of one 96x80x40,
// K = 20, FP32 instance: 24.0 -> 20.7 us (16x8 tiles), 27.2 -> 21.4 us (8x8 lane pairs); 64 instances of 32^3 to
// 128x128x64: 4.07e11 -> 4.27e11 updates/s with the engine's blocks of steps.
template <class T>
__device__ __forceinline__ const T& constant_at(const T* table, long long i) {
  typedef const __attribute__((address_space(4))) T CT;
  return *(const T*)((CT*)(uintptr_t)table + i);
}

template <int K, class TS, bool ANISO, int TX, int TY, int H>
__global__ __launch_bounds__(TX* TY* H) __attribute__((amdgpu_waves_per_eu(H + 1))) void step_kernel(const StepDev a,
                                                                                               const StepDyn d) {
  using TC = typename Traits<TS>::TC;
  using G = Tile<TS, K, TX, TY, H>;
  __shared__ __attribute__((aligned(16))) TC smem[G::NBUF * G::PSTR];
  __shared__ __attribute__((aligned(16))) TS stage[G::STAGE];
  __shared__ __attribute__((aligned(16))) TC ax[ANISO ? G::AXN : 4];
  __shared__ ZTab zt;
  int tx, ty, tz;
  if (!tile_coords(a, blockIdx.x, tx, ty, tz)) return;
  march_tile<K, TS, ANISO, TX, TY, H>(a, d, tx, ty, tz, smem, stage, ax, &zt);
}

// Persistent batched step: a fixed grid walks the device-resident work list (slot,
// tile) of one (dtype, K, anisotropy, tile shape) class.  Every workgroup exits after
// the list is exhausted; slots with no steps left are skipped.  Descriptions and step
// arguments are read in place (scalar loads), never copied into registers wholesale.
template <int K, class TS, bool ANISO, int TX, int TY, int H>
__global__ __launch_bounds__(TX* TY* H) __attribute__((amdgpu_waves_per_eu(2))) void batch_kernel(const BatchView v, int cls, int step) {
  using TC = typename Traits<TS>::TC;
  using G = Tile<TS, K, TX, TY, H>;
  __shared__ __attribute__((aligned(16))) TC smem[G::NBUF * G::PSTR];
  __shared__ __attribute__((aligned(16))) TS stage[G::STAGE];
  __shared__ __attribute__((aligned(16))) TC ax[ANISO ? G::AXN : 4];
  __shared__ ZTab zt;
  const int2 ci = constant_at(v.cinfo, cls);  // (offset, count) of this class's work list
  for (int w = blockIdx.x; w < ci.y; w += gridDim.x) {
    const WorkItem it = constant_at(v.work, ci.x + w);
    const BatchSlot& s = constant_at(v.slots, it.slot);
    const StepDev& a = constant_at(v.descs, it.path ? (1LL + step) * v.inst + it.slot : it.slot);
    const StepDyn& d = constant_at(v.dyns, (long long)step * v.inst + it.slot);
    if (s.steps_left <= step || !s.active) continue;
    int tx, ty, tz;
    item_coords(it.tile, a.tiles_x, a.tiles_y, a.tiles_z, tx, ty, tz);
    march_tile<K, TS, ANISO, TX, TY, H>(a, d, tx, ty, tz, smem, stage, ax, &zt);
    lds_barrier();  // LDS is reused by the next tile
  }
}

using StepLaunch = hipError_t (*)(const StepDev&, const StepDyn&, hipStream_t);
// Step `i` of the block for class `cls` (k: its number of orientations).
using BatchLaunch = hipError_t (*)(const BatchView&, int cls, int i, int grid, int k, hipStream_t);

struct StepEntry {
  int dtype, k, aniso, tile, tx, ty, h;
  StepLaunch step;
  BatchLaunch batch;
  size_t lds;
  const void* kernel;        // the step and batch kernels (occupancy queries)
  const void* batch_kernel;
};

template <int K, class TS, bool ANISO, int TX, int TY, int H>
hipError_t launch_step(const StepDev& a, const StepDyn& d, hipStream_t s) {
  const unsigned n = (unsigned)tile_launch(a);
  step_kernel<K, TS, ANISO, TX, TY, H><<<dim3(n), dim3(TX * TY * H), 0, s>>>(a, d);
  return hipGetLastError();
}

template <int K, class TS, bool ANISO, int TX, int TY, int H>
hipError_t launch_batch(const BatchView& v, int cls, int i, int grid, int, hipStream_t s) {
  batch_kernel<K, TS, ANISO, TX, TY, H><<<dim3(grid), dim3(TX * TY * H), 0, s>>>(v, cls, i);
  return hipGetLastError();
}

#define PF_ENTRY(DT, TS, K, A, T, TX, TY, H)                                      \
  {DT,                                                                           \
   K,                                                                            \
   A,                                                                            \
   T,                                                                            \
   TX,                                                                           \
   TY,                                                                           \
   H,                                                                            \
   &launch_step<K, TS, (A != 0), TX, TY, H>,                                     \
   &launch_batch<K, TS, (A != 0), TX, TY, H>,                                    \
   Tile<TS, K, TX, TY, H>::LDS_BYTES,                                            \
   (const void*)&step_kernel<K, TS, (A != 0), TX, TY, H>,                         \
   (const void*)&batch_kernel<K, TS, (A != 0), TX, TY, H>}

// instantiation tables, one per compiled part of pf_inst.hip (see Makefile):
// parts 0-3 F32, 4-7 BF16, 8-11 F64, each over a K range
constexpr int kInstParts = 12;
const StepEntry* step_table_part_0(int* n);
const StepEntry* step_table_part_1(int* n);
const StepEntry* step_table_part_2(int* n);
const StepEntry* step_table_part_3(int* n);
const StepEntry* step_table_part_4(int* n);
const StepEntry* step_table_part_5(int* n);
const StepEntry* step_table_part_6(int* n);
const StepEntry* step_table_part_7(int* n);
const StepEntry* step_table_part_8(int* n);
const StepEntry* step_table_part_9(int* n);
const StepEntry* step_table_part_10(int* n);
const StepEntry* step_table_part_11(int* n);
// Kernels for any K (pf_quad.hip): the march of channel groups, and one thread per cell for K of more
// groups than a workgroup's threads.  set_quads fills a's tile fields for (dtype, K) and returns the
// number of workgroups (work items of the batched kernel) of a launch; quad_threads is the number
// of its threads' channel groups in one pass over the grid.
long long set_quads(StepDev& a, int dtype, int zc);
constexpr int kQuadBlocks = 1280;  // five workgroups of the march on each of 256 CUs (what the registers allow)
constexpr long long kQuadLaunch = 1LL << 24;  // a launch has fewer workgroups of the march than this
long long quad_threads(int dtype, int k, long long cells);
bool quad_fits(int dtype, int k);  // K runs on the march of channel groups
// one Runge-Kutta stage on the march of channel groups (quad_fits, set_quads)
hipError_t rk_stage(const StepDev& a, const StepDyn& d, const RkStage& rk, int dtype, bool aniso, hipStream_t s);
StepLaunch generic_step(int dtype, int k, bool aniso);
StepLaunch generic_rhs(int dtype, int k, bool aniso);
BatchLaunch generic_batch(int dtype, int k, bool aniso);

}  // namespace pf

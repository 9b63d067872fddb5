// Grain segmentation on the GPU (include/pfhip.h pf_segment, pf_segment_moments):
// connected components of face-adjacent non-liquid cells with equal orientation index, the
// graph search of jax_am/phase_field/utils.py:217-265 done by joining trees.
//
// Labels are parents of a union-find forest in which every cell points to a cell of its own
// component with a smaller or the same index, so that the root of a component ends as its smallest
// cell.  One launch joins the cells of each tile in LDS, one joins the tiles across their faces
// with atomic minima, and one points every cell at its root, numbers the roots and, in the end,
// exact int64 moments are summed per tile in LDS and added up (independent of summation order).
// 128x128x64, 110 grains: 18 us in the tiles, 45 across their faces (the chains of finds and the minima
// on few roots bound it; tiles of 8 or 16 planes measured slower), 8 for the roots, 20 for the moments.  Label propagation by
// whole-grid passes (each label the minimum of its neighbours', four passes between host checks)
// took 92 passes of 9.1 us in 23 round trips, and moments by global atomics from runs of 16 cells 620 us.
#include "pf_host.h"

namespace pf {

constexpr int SX = 32, SY = 8, SZ = 4;      // cells of a tile: rows of half a wavefront
constexpr int ST = 256;                     // threads per block
constexpr int SC = SX * SY * SZ;

// Root of i in a forest of which other threads may be joining trees (values only ever decrease,
// and each is a cell of the same component, so a value read late is still an ancestor).
template <int SCOPE>
__device__ __forceinline__ int32_t seg_find(const int32_t* parent, int32_t i) {
  for (;;) {
    const int32_t q = __hip_atomic_load(parent + i, __ATOMIC_RELAXED, SCOPE);
    if (q == i) return i;
    i = q;
  }
}

// Joins the trees of a and b: the larger root is pointed at the smaller.  If another thread has
// pointed it elsewhere first, the tree that it went to is joined instead; every round ends at a
// smaller index, so this ends.
template <int SCOPE>
__device__ __forceinline__ void seg_join(int32_t* parent, int32_t a, int32_t b) {
  for (;;) {
    a = seg_find<SCOPE>(parent, a);
    b = seg_find<SCOPE>(parent, b);
    if (a == b) return;
    if (a < b) {
      const int32_t t = a;
      a = b;
      b = t;
    }
    const int32_t old = __hip_atomic_fetch_min(parent + a, b, __ATOMIC_RELAXED, SCOPE);
    if (old == a) return;
    a = old;
  }
}

// Cell of a tile by its place i = (z * SY + y) * SX + x, which orders a tile's cells as their indices do.
struct SegTiles {
  int nx, ny, nz, tx, ty;
  long long tiles, mtiles;  // tiles of the joins, tiles of the moments
};

__global__ __launch_bounds__(ST) void seg_tile_kernel(const StepDev a, SegTiles g, double t,
                                                     const int32_t* __restrict__ ori, int32_t* __restrict__ label,
                                                     int32_t* __restrict__ counter) {
  constexpr int W = __HIP_MEMORY_SCOPE_WORKGROUP;
  __shared__ int32_t key[SC];  // orientation
  __shared__ int32_t lab[SC];  // parent within the tile, -1: liquid or outside the grid
  if (blockIdx.x == 0 && threadIdx.x == 0) *counter = 0;
  for (long long w = blockIdx.x; w < g.tiles; w += gridDim.x) {
    const long long r = w / g.tx;
    const int x0 = (int)(w - r * g.tx) * SX, y0 = (int)(r % g.ty) * SY, z0 = (int)(r / g.ty) * SZ;
    for (int i = threadIdx.x; i < SC; i += ST) {
      const int ix = x0 + i % SX, iy = y0 + i / SX % SY, iz = z0 + i / (SX * SY);
      int32_t k = 0;
      bool solid = false;
      if (ix < g.nx && iy < g.ny && iz < g.nz) {
        const long long c = ((long long)iz * g.ny + iy) * g.nx + ix;
        k = ori[c];
        solid = cell_temperature(a, ix, iy, iz, c, t) < a.T_l;  // utils.py:193: non-liquid = T < T_liquidus
      }
      key[i] = k;
      // runs along x are joined from the start: each cell points at the first of its run
      const int lane = threadIdx.x & 63;
      const int left = __shfl_up(k, 1, 64);
      const unsigned long long solids = __ballot(solid);
      const bool lsolid = lane > 0 && (solids >> (lane - 1) & 1);
      const unsigned long long same = __ballot(i % SX != 0 && solid && lsolid && left == k);
      const unsigned long long starts = ~same & ((2ULL << lane) - 1);
      lab[i] = solid ? i - (lane - (63 - __clzll(starts))) : -1;
    }
    __syncthreads();
    for (int i = threadIdx.x; i < SC; i += ST) {
      if (lab[i] < 0) continue;
      const int32_t k = key[i];
      const int x = i % SX, y = i / SX % SY, z = i / (SX * SY);
      const bool left = x > 0 && lab[i - 1] >= 0 && key[i - 1] == k;
      // a pair whose left pair is of the same two runs is joined already
      const auto joins = [&](int b) {
        return lab[b] >= 0 && key[b] == k && !(left && lab[b - 1] >= 0 && key[b - 1] == k);
      };
      if (y > 0 && joins(i - SX)) seg_join<W>(lab, i, i - SX);
      if (z > 0 && joins(i - SX * SY)) seg_join<W>(lab, i, i - SX * SY);
    }
    __syncthreads();
    for (int i = threadIdx.x; i < SC; i += ST) {
      const int ix = x0 + i % SX, iy = y0 + i / SX % SY, iz = z0 + i / (SX * SY);
      if (ix >= g.nx || iy >= g.ny || iz >= g.nz) continue;
      int32_t l = -1;
      if (lab[i] >= 0) {
        const int q = seg_find<W>(lab, i);
        l = ((z0 + q / (SX * SY)) * g.ny + y0 + q / SX % SY) * g.nx + x0 + q % SX;
      }
      label[((long long)iz * g.ny + iy) * g.nx + ix] = l;
    }
    __syncthreads();
  }
}

// Joins across the low faces of the tiles, one thread per cell.
__global__ __launch_bounds__(ST) void seg_merge_kernel(SegTiles g, const int32_t* __restrict__ ori, int32_t* label) {
  constexpr int A = __HIP_MEMORY_SCOPE_AGENT;
  const long long n = (long long)g.nx * g.ny * g.nz;
  const long long c = (long long)blockIdx.x * ST + threadIdx.x;
  if (c >= n) return;
  const int u = (int)c, ix = u % g.nx, iy = u / g.nx % g.ny, iz = u / g.nx / g.ny;
  const bool fx = ix > 0 && ix % SX == 0, fy = iy > 0 && iy % SY == 0, fz = iz > 0 && iz % SZ == 0;
  if (!(fx || fy || fz)) return;
  const auto solid = [&](int i) { return __hip_atomic_load(label + i, __ATOMIC_RELAXED, A) >= 0; };
  if (!solid(u)) return;
  const int32_t o = ori[u];
  const bool lefts = ix % SX != 0 && ori[u - 1] == o && solid(u - 1);  // the cell to the left is of the same run
  const int step[3] = {1, g.nx, g.nx * g.ny};
  const bool face[3] = {fx, fy, fz};
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    if (!face[k]) continue;
    const int b = u - step[k];
    if (ori[b] != o || !solid(b)) continue;
    if (k > 0 && lefts && ori[b - 1] == o && solid(b - 1)) continue;  // joined by the pair to the left
    seg_join<A>(label, u, b);
  }
}

// Every cell to its root, and the roots numbered.
__global__ __launch_bounds__(ST) void seg_roots_kernel(long long n, int32_t* label, int32_t* __restrict__ cid,
                                                      int32_t* __restrict__ root, int32_t* __restrict__ counter) {
  const long long c = (long long)blockIdx.x * ST + threadIdx.x;
  if (c >= n) return;
  constexpr int A = __HIP_MEMORY_SCOPE_AGENT;
  const int32_t l = __hip_atomic_load(label + c, __ATOMIC_RELAXED, A);
  if (l < 0) return;
  const int32_t q = seg_find<A>(label, l);
  if (q == (int32_t)c) {
    const int32_t g = atomicAdd(counter, 1);
    cid[c] = g;
    root[g] = (int32_t)c;
  } else if (q != l) {
    __hip_atomic_store(label + c, q, __ATOMIC_RELAXED, A);
  }
}

constexpr int NMOM = 10;
constexpr int MZ = 16;     // planes of a moments tile (SX x SY columns)
constexpr int MSLOT = 64;  // grains of a tile summed in LDS; those past them go straight to memory

__global__ __launch_bounds__(ST) void seg_zero_kernel(unsigned long long* __restrict__ p, long long n) {
  for (long long i = (long long)blockIdx.x * ST + threadIdx.x; i < n; i += (long long)gridDim.x * ST) p[i] = 0;
}

__device__ __forceinline__ void seg_flush(unsigned long long* mom, int32_t g, const long long (&s)[NMOM],
                                          int32_t* slot, unsigned long long (*sum)[NMOM]) {
#pragma unroll 1
  for (int k = 0; k < MSLOT; ++k) {
    const int h = (g + k) % MSLOT;
    const int32_t was = atomicCAS(slot + h, -1, g);
    if (was == -1 || was == g) {
#pragma unroll
      for (int m = 0; m < NMOM; ++m)
        if (s[m] != 0) atomicAdd(&sum[h][m], (unsigned long long)s[m]);
      return;
    }
  }
#pragma unroll
  for (int m = 0; m < NMOM; ++m)
    if (s[m] != 0) atomicAdd(mom + (long long)g * NMOM + m, (unsigned long long)s[m]);
}

// One thread per column of a tile: sums are kept in registers while the planes belong to the same
// grain, then go to the tile's sums in LDS, one slot per grain (open addressing).
__global__ __launch_bounds__(ST) void seg_moments_kernel(SegTiles g, const int32_t* __restrict__ label,
                                                        const int32_t* __restrict__ cid,
                                                        unsigned long long* __restrict__ mom) {
  __shared__ int32_t slot[MSLOT];
  __shared__ unsigned long long sum[MSLOT][NMOM];
  for (long long w = blockIdx.x; w < g.mtiles; w += gridDim.x) {
    for (int i = threadIdx.x; i < MSLOT * NMOM; i += ST) sum[i / NMOM][i % NMOM] = 0;
    if (threadIdx.x < MSLOT) slot[threadIdx.x] = -1;
    __syncthreads();
    const long long r = w / g.tx;
    const int ix = (int)(w - r * g.tx) * SX + threadIdx.x % SX, iy = (int)(r % g.ty) * SY + threadIdx.x / SX;
    const int z0 = (int)(r / g.ty) * MZ, z1 = min(g.nz, z0 + MZ);
    if (ix < g.nx && iy < g.ny) {
      // a column's cells share x and y: their sums follow from the number of cells and the sums over z
      long long n = 0, sz = 0, szz = 0;
      int32_t cur = -1;
      for (int iz = z0; iz <= z1; ++iz) {
        int32_t gr = -1;
        if (iz < z1) {
          const int32_t l = label[((long long)iz * g.ny + iy) * g.nx + ix];
          if (l < 0) continue;
          gr = cid[l];
        }
        if (gr != cur) {
          if (cur >= 0) {
            const long long s[NMOM] = {n,      n * ix,      n * iy,  sz,      n * ix * ix, n * iy * iy,
                                       szz,    n * ix * iy, sz * ix, sz * iy};
            seg_flush(mom, cur, s, slot, sum);
          }
          n = sz = szz = 0;
          cur = gr;
        }
        n += 1;
        sz += iz;
        szz += (long long)iz * iz;
      }
    }
    __syncthreads();
    for (int i = threadIdx.x; i < MSLOT * NMOM; i += ST) {
      const int h = i / NMOM, m = i % NMOM;
      if (slot[h] >= 0 && sum[h][m] != 0) atomicAdd(mom + (long long)slot[h] * NMOM + m, sum[h][m]);
    }
    __syncthreads();
  }
}

static SegTiles seg_tiles(const pf_params_t* p) {
  SegTiles g{p->nx, p->ny, p->nz, (p->nx + SX - 1) / SX, (p->ny + SY - 1) / SY, 0, 0};
  g.tiles = (long long)g.tx * g.ty * ((p->nz + SZ - 1) / SZ);
  g.mtiles = (long long)g.tx * g.ty * ((p->nz + MZ - 1) / MZ);
  return g;
}
// blocks of a loop over tiles (a launch has fewer than 2^32 threads)
static unsigned seg_blocks(long long tiles) { return (unsigned)(tiles < (1 << 20) ? tiles : 1 << 20); }

}  // namespace pf

using namespace pf;

extern "C" {

int pf_segment(const int32_t* ori_dev, const void* T_dev, const pf_params_t* p, double t, int32_t* labels_dev,
               int32_t* cid_dev, int32_t* root_dev, int32_t* ws_dev, int64_t max_passes, int32_t* n_grains,
               void* stream) {
  if (!ori_dev || !labels_dev || !cid_dev || !root_dev || !ws_dev || !n_grains) return fail(PF_E_ARG, "NULL argument");
  StepDev a;
  int rc = make_stepdev(p, PF_F64, T_dev, (const void*)1, 0, a);
  if (rc) return rc;
  const long long n = (long long)p->nz * p->ny * p->nx;
  if (n >= (1LL << 31) - 1) return fail(PF_E_ARG, "pf_segment supports fewer than 2^31 cells");
  if (max_passes < 1) return fail(PF_E_ARG, "max_passes must be >= 1");
  hipStream_t s = (hipStream_t)stream;
  const SegTiles g = seg_tiles(p);
  const unsigned nb = (unsigned)((n + ST - 1) / ST);
  seg_tile_kernel<<<seg_blocks(g.tiles), ST, 0, s>>>(a, g, t, ori_dev, labels_dev, ws_dev);
  seg_merge_kernel<<<nb, ST, 0, s>>>(g, ori_dev, labels_dev);
  seg_roots_kernel<<<nb, ST, 0, s>>>(n, labels_dev, cid_dev, root_dev, ws_dev);
  hipError_t e = hipGetLastError();
  int32_t count = 0;
  if (e == hipSuccess) e = hipMemcpyAsync(&count, ws_dev, sizeof(int32_t), hipMemcpyDeviceToHost, s);
  if (e == hipSuccess) e = hipStreamSynchronize(s);
  if (e != hipSuccess) return hip_fail(e, "pf_segment roots");
  *n_grains = count;
  return PF_OK;
}

int pf_segment_moments(const int32_t* labels_dev, const int32_t* cid_dev, const pf_params_t* p, int32_t n_grains,
                       int64_t* moments_dev, void* stream) {
  if (!labels_dev || !cid_dev || !p || (!moments_dev && n_grains > 0)) return fail(PF_E_ARG, "NULL argument");
  if (n_grains < 0) return fail(PF_E_ARG, "n_grains must be >= 0");
  if (p->nz < 1 || p->ny < 1 || p->nx < 1) return fail(PF_E_ARG, "grid dimensions must be >= 1");
  if (n_grains == 0) return PF_OK;
  hipStream_t s = (hipStream_t)stream;
  const SegTiles g = seg_tiles(p);
  const long long nm = (long long)n_grains * NMOM;
  seg_zero_kernel<<<seg_blocks((nm + ST - 1) / ST), ST, 0, s>>>((unsigned long long*)moments_dev, nm);
  seg_moments_kernel<<<seg_blocks(g.mtiles), ST, 0, s>>>(g, labels_dev, cid_dev, (unsigned long long*)moments_dev);
  hipError_t e = hipGetLastError();
  return e == hipSuccess ? PF_OK : hip_fail(e, "pf_segment_moments");
}

}  // extern "C"

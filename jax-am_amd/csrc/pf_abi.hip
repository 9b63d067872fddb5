// C ABI of libpfhip.so (include/pfhip.h): single-instance step, temperature,
// and initial condition.  Argmax and the diagnostics are in pf_reduce.hip, the batched engine in
// pf_batch.hip, the register-tiled instantiations in pf_inst_*.hip.
#include <math.h>
#include <string.h>

#include <atomic>
#include <memory>
#include <string>
#include <vector>

#include "pf_host.h"

namespace pf {

// ------------------------------------------------------------------ errors
static thread_local std::string g_err;

void set_error(const std::string& msg) { g_err = msg; }
int fail(int code, const std::string& msg) {
  g_err = msg;
  return code;
}
int hip_fail(hipError_t e, const char* what) {
  g_err = std::string(what) + ": " + hipGetErrorName(e) + " (" + hipGetErrorString(e) + ")";
  return PF_E_HIP;
}

size_t dtype_size(int dtype) { return dtype == PF_F64 ? 8 : dtype == PF_F32 ? 4 : dtype == PF_BF16 ? 2 : 0; }
bool valid_dtype(int dtype) { return dtype == PF_F64 || dtype == PF_F32 || dtype == PF_BF16; }

// ------------------------------------------------------------------ parameters
int make_stepdev(const pf_params_t* p, int dtype, const void* T_dev, const void* axes_dev, int zc, StepDev& a) {
  if (!p) return fail(PF_E_ARG, "params pointer is NULL");
  if (!valid_dtype(dtype)) return fail(PF_E_ARG, "dtype must be PF_F64, PF_F32 or PF_BF16");
  if (p->nz < 1 || p->ny < 1 || p->nx < 1 || p->num_oris < 1)
    return fail(PF_E_ARG, "grid dimensions and num_oris must be >= 1");
  const long long n = (long long)p->nz * p->ny * p->nx;
  if (n * p->num_oris >= (1LL << 40)) return fail(PF_E_ARG, "grid too large");
  if ((long long)p->ny * p->nx * p->num_oris >= (1LL << 31))
    return fail(PF_E_ARG, "one z-plane must hold fewer than 2^31 values");
  for (int d = 0; d < 3; ++d)
    if (!(p->h[d] > 0.0)) return fail(PF_E_ARG, "mesh_h_xyz must be positive");
  if (!(p->ad_hoc != 0.0)) return fail(PF_E_ARG, "ad_hoc must be non-zero");
  if (!(p->T_liquidus > 0.0) || !(p->gas_const != 0.0)) return fail(PF_E_ARG, "T_liquidus and gas_const must be set");
  const pf_laser_t& L = p->laser;
  if (L.model < PF_T_BUFFER || L.model > PF_T_QUENCH) return fail(PF_E_ARG, "unknown temperature model");
  if (L.model == PF_T_BUFFER) {
    if (!T_dev) return fail(PF_E_ARG, "temperature model PF_T_BUFFER needs a T buffer");
    if (L.T_dtype != PF_F64 && L.T_dtype != PF_F32) return fail(PF_E_ARG, "T buffer dtype must be PF_F64 or PF_F32");
  }
  if (L.model == PF_T_ROSENTHAL && (!(L.kappa_T != 0.0) || !(L.alpha != 0.0)))
    return fail(PF_E_ARG, "Rosenthal model needs kappa_T and alpha");
  if (L.model == PF_T_GAUSSIAN && (!(L.sigma_xy > 0.0) || !(L.sigma_z > 0.0)))
    return fail(PF_E_ARG, "Gaussian model needs sigma_xy, sigma_z > 0");
  const bool aniso = p->anisotropy > 0.0;
  if (aniso && !axes_dev) return fail(PF_E_ARG, "anisotropy > 0 needs the grain-direction table");

  memset(&a, 0, sizeof(a));
  a.T = T_dev;
  a.axes = axes_dev;
  a.nz = p->nz;
  a.ny = p->ny;
  a.nx = p->nx;
  a.k = p->num_oris;
  a.zc = zc;
  a.tmodel = L.model;
  a.t_f64 = L.T_dtype == PF_F64;
  a.force_liquid = p->force_liquid != 0;
  a.hx = p->h[0];
  a.hy = p->h[1];
  a.hz = p->h[2];
  a.ihx2 = 1.0 / (p->h[0] * p->h[0]);
  a.ihy2 = 1.0 / (p->h[1] * p->h[1]);
  a.ihz2 = 1.0 / (p->h[2] * p->h[2]);
  a.m_over_ad = p->m_g / p->ad_hoc;
  a.kappa_ad = p->kappa_g * p->ad_hoc;
  a.gamma4 = 4.0 * p->gamma;
  a.B = 1.0 - 4.0 * p->gamma;
  a.ihx2f = (float)a.ihx2;
  a.ihy2f = (float)a.ihy2;
  a.ihz2f = (float)a.ihz2;
  a.Bf = (float)a.B;
  a.L0 = p->L0;
  a.Qg = p->Qg;
  a.gas_const = p->gas_const;
  a.T_l = p->T_liquidus;
  a.T_clip = p->T_clip;
  a.theta = p->zeta_sharpness;
  // |theta*(Tc/T_l - 1)| >= 20 (tanh == +-1 exactly in FP64) holds for |Tc - T_l| > 20*T_l/theta;
  // use twice that as the compare window.
  a.zeta_window = p->zeta_sharpness > 0.0 ? 40.0 * p->T_liquidus / p->zeta_sharpness : INFINITY;
  a.eps = aniso ? p->anisotropy : 0.0;
  a.liquid_T = p->T_liquidus + p->liquid_shift;
  a.stiff = fabs(a.m_over_ad) * (4.0 + 4.0 * fabs(p->gamma)) +
            4.0 * fabs(a.kappa_ad) * (1.0 + a.eps) * (a.ihx2 + a.ihy2 + a.ihz2);
  a.T_amb = L.T_ambient;
  a.p0x = L.pos0[0];
  a.p0y = L.pos0[1];
  a.p0z = L.pos0[2];
  a.dirx = L.dir[0];
  a.diry = L.dir[1];
  a.dirz = L.dir[2];
  a.vel = L.vel;
  if (L.model == PF_T_ROSENTHAL) {
    a.kappa_T = L.kappa_T;
    a.alpha = L.alpha;
    a.q_coef = rosenthal_q(L.Q, L.kappa_T);  // simple/example.py:35 Q / (2*pi*kappa)
    a.pe = rosenthal_pe(L.vel, L.alpha);     // vel / (2*alpha)
  }
  a.T_cap = L.T_cap;
  a.dT_peak = L.dT_peak;
  if (L.model == PF_T_GAUSSIAN) {
    a.g_sxy = 1.0 / (2.0 * L.sigma_xy * L.sigma_xy);
    a.g_sz = 1.0 / (2.0 * L.sigma_z * L.sigma_z);
  }
  a.T_ref = L.T_ref;
  a.grad_T = L.grad_T;
  a.cool_rate = L.cool_rate;
  return PF_OK;
}

// ------------------------------------------------------------------ dispatch tables
namespace {
struct Tables {
  std::vector<StepEntry> t[3];
  static constexpr int kMaxK = 32, kMaxTile = 8;
  const StepEntry* at[3][kMaxK + 1][2][kMaxTile] = {};  // [dtype][K][anisotropic][tile]
  std::unique_ptr<std::atomic<int>[]> held[3];  // per entry and kernel (step, batch): workgroups the GPU holds at once (0: not asked yet)
  Tables() {
    using PartFn = const StepEntry* (*)(int*);
    const PartFn parts[kInstParts] = {&step_table_part_0, &step_table_part_1, &step_table_part_2,
                                      &step_table_part_3, &step_table_part_4, &step_table_part_5,
                                      &step_table_part_6, &step_table_part_7, &step_table_part_8,
                                      &step_table_part_9, &step_table_part_10, &step_table_part_11};
    for (PartFn f : parts) {
      int n = 0;
      const StepEntry* e = f(&n);
      for (int i = 0; i < n; ++i) t[e[i].dtype].push_back(e[i]);
    }
    for (int d = 0; d < 3; ++d)
      for (const StepEntry& e : t[d]) at[d][e.k][e.aniso != 0][e.tile] = &e;
    for (int d = 0; d < 3; ++d) held[d] = std::make_unique<std::atomic<int>[]>(2 * t[d].size());
  }
};
const Tables& tables() {
  static Tables tb;
  return tb;
}
}  // namespace

int entry_count(int dtype, int k, bool aniso) {
  if (!valid_dtype(dtype)) return 0;
  const Tables& tb = tables();
  int c = 0;
  for (const StepEntry& e : tb.t[dtype])
    if (e.k == k && (e.aniso != 0) == aniso) ++c;
  return c;
}

const StepEntry* find_entry(int dtype, int k, bool aniso, int tile) {
  if (tile < 0) tile = 0;
  if (!valid_dtype(dtype) || k < 0 || k > Tables::kMaxK || tile >= Tables::kMaxTile) return nullptr;
  return tables().at[dtype][k][aniso ? 1 : 0][tile];
}

// Asked of the runtime once per kernel.
int held_workgroups(const StepEntry* e, bool batch) {
  const Tables& tb = tables();
  std::atomic<int>& c = tb.held[e->dtype][2 * (e - tb.t[e->dtype].data()) + (batch ? 1 : 0)];
  int n = c.load(std::memory_order_relaxed);
  if (n == 0) {
    int per = 0, dev = 0, cus = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, batch ? e->batch_kernel : e->kernel, e->tx * e->ty * e->h, 0) !=
            hipSuccess ||
        hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) {
      (void)hipGetLastError();
      return 1024;
    }
    n = per * cus;
    if (n < 1) n = 1;
    c.store(n, std::memory_order_relaxed);
  }
  return n;
}

// Planes per march for `cols` tile columns when the GPU holds `held` workgroups: the shortest marches
// that fill it a whole number of times, once if they then have at most 12 planes, else as often as
// that takes.  Each march reads two planes more than it writes, so longer is better, but only while
// no CU idles at the launch's end: 128x96x48, K = 20, FP64 (16x4 lane pairs) 46.6 us at 12 planes, one
// filling, against 51.4 at 6; 203x197x59, K = 17, FP32 (16x8) 85.8 us at 10, two fillings, against 98 at 16.
// A tall grid whose columns alone fill the GPU's half takes 16 planes with the tail split (PF_ZCHUNK_TAIL), whose
// short marches end the launch: 256x256x64 in FP32 K = 13 104.6 -> 100.0 us, BF16 K = 10 57.8 -> 54.4, K = 17 112.2 -> 105.7, FP64
// K = 12 189 -> 182.5, against fillings; on 203x197x59 (a third) it is slower, FP32 K = 17 91 against 85.8.
static int fill_zchunk(int nz, long long cols, int held) {
  if (nz >= 40 && 2 * cols >= held) return 16 | PF_ZCHUNK_TAIL;
  const long long kmin = (nz + 11) / 12;
  const long long m = (kmin * cols + held - 1) / held;  // fillings: the fewest whose chunks have at most 12 planes
  const long long k = m * held / cols;
  const long long zc = (nz + k - 1) / k;
  return (int)(zc < 2 ? (nz < 2 ? nz : 2) : zc);
}

// The kernel of a step whose caller leaves the choice open, for K with tiled kernels: a tile shape,
// or nullptr for the march of channel groups.  That one has a workgroup for every few hundred
// cells and no LDS planes to fill first, which wins while the grid leaves the tiled kernels short of
// workgroups, and for odd K in FP64, where a tile has one lane per cell and its registers spill; in
// larger grids the tiles' exact skips of all-zero channels win.  Measured in us, groups against the best
// tile (its best z-chunk): FP32 K = 10: 32^3 5.7/7.1, 64x64x32 8.7/8.3, 64^3 12.8/10.5; K = 20: 48x48x40 8.9/10.4,
// 64x64x32 11.5/10.0; K = 17: 64x64x32 11.3/11.3, 64^3 17.5/14.2.  BF16 K = 20: 48x48x40 8.3/9.1; K = 10: 7.5/6.9;
// K = 13: 64x64x32 9.1/9.3.  FP64 K = 10: 64x64x32 11.5/10.7 (isotropic 9.2/8.9), 48x48x40 9.3/10.2; K = 16: 64x64x32
// 13.7/14.3, 64^3 20.3/21.2; K = 13: 96x96x48 30.9/33.2, 128x96x48 43.1/41.2; K = 17: 128x96x48 54.4/54.2.
bool small_step(int dtype, int k, long long cells) {
  if (!quad_fits(dtype, k)) return false;
  const bool odd = k % 2 != 0;
  long long most;
  if (dtype == PF_F64) most = odd && k >= 11 ? 4000000 : k >= 16 ? 1100000 : 500000;
  else if (dtype == PF_F32) most = odd ? 530000 : 470000;
  else most = odd || k >= 16 ? 480000 : 250000;
  return quad_threads(dtype, k, cells) <= most;
}

// Whether a step's tiles go to the XCDs by whole rows (tile_coords): where the XCD with the most rows needs no
// more fillings than an even share would, `held` workgroups being resident on the GPU at once, and none
// stays empty.  Sharing an L2 along a row is worth 3 to 7 % (us a step, rows against even shares: 203x197x59,
// K = 20, FP32 85.0/91.4, 300x100x80 85.3/91.6, 100x300x40 48.3/51.3); a filling more costs far more than
// that (320x72x48, 36 rows of 40 tiles, 192 held per XCD: 54.9/44.8; 200x56x64, K = 17, 77 rows of 13, 128 held:
// 35.8/33.9), and so do XCDs without work (4096x32x1, K = 20, 4 rows: 16.5/10.4).
static bool deal_rows(const StepDev& a, int held) {
  const long long rows = (long long)a.tiles_y * a.tiles_z;
  if (rows < 8) return false;
  const long long most = (rows + 7) / 8 * a.tiles_x, even = (rows * a.tiles_x + 7) / 8;
  const long long cap = held >= 8 ? held / 8 : 1;
  return (most + cap - 1) / cap == (even + cap - 1) / cap;
}

// Share of the GPU's workgroups that a launch of kernel e keeps busy: its marches, the shortest that fill the GPU a
// whole number of times (fill_zchunk) but of two planes or more, against the fillings they take.
static double filled(const StepEntry* e, int nz, int ny, int nx) {
  const long long held = held_workgroups(e, false);
  const long long cols = (long long)((nx + e->tx - 1) / e->tx) * ((ny + e->ty - 1) / e->ty);
  const long long m = ((nz + 11) / 12 * cols + held - 1) / held;
  const long long most = (nz + 1) / 2, k = m * held / cols < most ? m * held / cols : most;
  return (double)(k * cols) / (double)(m * held);
}

// Flat grids in FP32 and BF16 (us, other tile / this one).  A single plane has nothing to march through and takes
// the tile with the least halo, 32x8: 1024x1024x1, FP32 K = 16 52.7/48.0, BF16 K = 13 47.4/46.1, and the march of
// channel groups only up to half as many values (64x2048x1, FP32 K = 13 10.5/8.3); so do up to four planes in BF16
// for odd K where it fills the GPU as well: 512x512x3, K = 13 27.3/24.0.  Lane pairs lose to 16x8 tiles on few planes
// if they keep under 0.7 of the GPU busy and those more: 256x256x8, two thirds, BF16 K = 16 20.3/16.4, 256x256x4, FP32
// K = 20 15.4/14.3, 64x2048x2 16.5/13.8; but 300x700x6, 0.73, BF16 K = 20 33.8/38.9, and on more planes the marches are
// cut to fill it (256x256x16, BF16 K = 16 28.5/29.0).
static const StepEntry* choose_step(int dtype, int k, bool aniso, int nz, int ny, int nx) {
  const long long cells = (long long)nz * ny * nx;
  const bool odd = k % 2 != 0, bf16 = dtype == PF_BF16, flat = dtype != PF_F64 && nz == 1;
  if (small_step(dtype, k, flat ? 2 * cells : cells)) return nullptr;
  const StepEntry* wide = find_entry(dtype, k, aniso, 0);
  const StepEntry* e = find_entry(dtype, k, aniso, 2);
  if (dtype == PF_F64) {
    e = find_entry(dtype, k, aniso, !odd ? 2 : k >= 17 ? 0 : 1);  // 16x4 lane pairs; 32x4; 16x4
  } else if (flat) {
    e = wide;
  } else if (k % 4 == 0 && (k >= 16 || (bf16 && k == 12 && cells < 2000000))) {
    // 8x8 lane pairs (whole vectors in each half need K % 4 = 0; BF16 K = 12: 256x256x64 65.1 against 58.9 us)
    const StepEntry* pairs = find_entry(dtype, k, aniso, 4);
    if (pairs && e && nz <= (bf16 ? 12 : 6)) {
      const double share = filled(pairs, nz, ny, nx);
      if (share >= 0.7 || share >= filled(e, nz, ny, nx)) e = pairs;
    } else {
      e = pairs;
    }
  } else if (bf16 && odd && nz <= 4 && e && wide && filled(wide, nz, ny, nx) >= filled(e, nz, ny, nx)) {
    e = wide;
  }
  return e ? e : wide;  // 16x8
}

int default_zchunk(int nz, int ny, int nx, int tx, int ty) {
  // about 2048 workgroups (four rounds of 2 per CU on 256 CUs: shorter marches balance the
  // data-dependent work better), at least 4 planes per march
  const long long txy = (long long)((nx + tx - 1) / tx) * ((ny + ty - 1) / ty);
  long long chunks = (2048 + txy / 2) / txy;
  if (chunks < 1) chunks = 1;
  int zc = (int)((nz + chunks - 1) / chunks);
  if (zc < 4) zc = 4;
  if (zc > nz) zc = nz;
  return zc;
}

// The tiled kernels (the march) address a z-plane with 32-bit byte offsets and write it
// back through raw buffer stores whose out-of-range offsets (2^31 and above) are dropped.
int march_fits(const pf_params_t* p, int dtype) {
  if ((long long)p->ny * p->nx * p->num_oris * (long long)dtype_size(dtype) >= (1LL << 31))
    return fail(PF_E_ARG, "the tiled kernels need a z-plane of fewer than 2^31 bytes (tile -2 runs the generic kernel)");
  return PF_OK;
}

void set_tiles(StepDev& a, int tx, int ty, int zchunk) {
  const bool tail = (zchunk & PF_ZCHUNK_TAIL) != 0;
  int zc = zchunk & ~PF_ZCHUNK_TAIL;
  if (zc <= 0) zc = default_zchunk(a.nz, a.ny, a.nx, tx, ty);
  if (zc > a.nz) zc = a.nz;
  a.zc = zc;
  a.zs = zc;
  a.zsplit = 0;
  if (tail) {
    // the lowest quarter of the planes in whole chunks of ceil(zc / 2), at least one full chunk above
    const int zs = (zc + 1) / 2;
    int nbot = (a.nz / 4 + zs - 1) / zs * zs;
    if (nbot > a.nz - zc) nbot = (a.nz - zc) / zs * zs;
    if (zs < zc && nbot > 0) {
      a.zs = zs;
      a.zsplit = nbot;
    }
  }
  a.tiles_x = (a.nx + tx - 1) / tx;
  a.tiles_y = (a.ny + ty - 1) / ty;
  a.tiles_z = (a.zsplit > 0 ? (a.zsplit + a.zs - 1) / a.zs : 0) + (a.nz - a.zsplit + zc - 1) / zc;
}

// ------------------------------------------------------------------ auxiliary kernels
template <class TT>
__global__ __launch_bounds__(256) void temperature_kernel(const StepDev a, TT* __restrict__ out, double t) {
  const long long n = (long long)a.nz * a.ny * a.nx;
  const long long c = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= n) return;
  int ix, iy, iz;
  if (n <= 0xffffffffLL) {  // 32-bit divisions: a fraction of the cost of the 64-bit ones
    const unsigned u = (unsigned)c, r = u / (unsigned)a.nx;
    ix = (int)(u - r * (unsigned)a.nx);
    iz = (int)(r / (unsigned)a.ny);
    iy = (int)(r - (unsigned)iz * (unsigned)a.ny);
  } else {
    ix = (int)(c % a.nx);
    iy = (int)((c / a.nx) % a.ny);
    iz = (int)(c / ((long long)a.nx * a.ny));
  }
  out[c] = (TT)cell_temperature(a, ix, iy, iz, c, t);
}

// One-hot state of a run of OC cells per block: the cells' orientations go through LDS and the block
// writes its values as one contiguous piece, 16 bytes a thread and store.  Bound by the writes:
// 256x256x64, K = 20, FP32 60 us, 5.6 TB/s (a 64-bit division and a 4-byte store per value: 122 us).
constexpr int OC = 256;

template <class TS>
__global__ __launch_bounds__(256) void onehot_kernel(TS* __restrict__ eta, const int32_t* __restrict__ ori,
                                                    long long n_cells, int k) {
  using TC = typename Traits<TS>::TC;
  constexpr int V = 16 / (int)sizeof(TS);
  __shared__ int32_t so[OC];
  const TS one = from_tc<TS>((TC)1), zero = from_tc<TS>((TC)0);
  for (long long c0 = (long long)blockIdx.x * OC; c0 < n_cells; c0 += (long long)gridDim.x * OC) {
    const int m = (int)min((long long)OC, n_cells - c0);
    __syncthreads();
    if ((int)threadIdx.x < m) so[threadIdx.x] = ori[c0 + threadIdx.x];
    __syncthreads();
    TS* out = eta + c0 * k;
    const long long ne = (long long)m * k;
    for (long long e = (long long)threadIdx.x * V; e < ne; e += 256 * V) {
      int c = ne < (1LL << 31) ? (int)((unsigned)e / (unsigned)k) : (int)(e / k);
      int i = (int)(e - (long long)c * k);
      VecA<TS, V, (int)sizeof(TS)> v;
#pragma unroll
      for (int q = 0; q < V; ++q) {
        v.v[q] = so[min(c, m - 1)] == i ? one : zero;
        if (++i == k) {
          i = 0;
          ++c;
        }
      }
      if (e + V <= ne) {
        *(VecA<TS, V, (int)sizeof(TS)>*)(out + e) = v;
      } else {
#pragma unroll
        for (int q = 0; q < V; ++q)
          if (e + q < ne) out[e + q] = v.v[q];
      }
    }
  }
}

// Nearest seed of each cell centroid.  A block owns a box of cells and first keeps the seeds that can
// be nearest to any of them: those no further from the box than the least of the seeds' greatest
// distances to it.  Both bounds are formed by the operations of a cell's own distance on the box's
// first and last centroids; rounding is monotonic, so no cell's distance is below the one or above the
// other and the result is that of trying every seed.  The list keeps the seeds' order (ties go to the
// lower index).  256x256x64 cells, 500 seeds: 61 us (every seed for every cell: 792 us).
constexpr int VX = 16, VY = 8, VZ = 4;  // cells of a box, two per thread
constexpr int VCAND = 512;              // seeds kept at most; more: every seed is tried

__global__ __launch_bounds__(256) void voronoi_kernel(const double* __restrict__ seeds, int ns,
                                                     const int32_t* __restrict__ gori, int nz, int ny, int nx,
                                                     double hx, double hy, double hz, long long boxes,
                                                     int32_t* __restrict__ out) {
  __shared__ double cx[VCAND], cy[VCAND], cz[VCAND];
  __shared__ int cid[VCAND];
  __shared__ double wmin[4];
  __shared__ int wcount[4];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int bx = (nx + VX - 1) / VX, by = (ny + VY - 1) / VY;
  for (long long b = blockIdx.x; b < boxes; b += gridDim.x) {
    const long long r = b / bx;
    const int x0 = (int)(b - r * bx) * VX, y0 = (int)(r % by) * VY, z0 = (int)(r / by) * VZ;
    // first and last centroids of the box along each axis, in either order (h of any sign)
    const auto ends = [](int i0, int i1, double h, double& l, double& u) {
      const double a = ((double)i0 + 0.5) * h, c = ((double)i1 + 0.5) * h;
      l = fmin(a, c);
      u = fmax(a, c);
    };
    double lx, ux, ly, uy, lz, uz;
    ends(x0, min(x0 + VX - 1, nx - 1), hx, lx, ux);
    ends(y0, min(y0 + VY - 1, ny - 1), hy, ly, uy);
    ends(z0, min(z0 + VZ - 1, nz - 1), hz, lz, uz);
    const auto least = [](double l, double u, double s) { return s < l ? l - s : s > u ? s - u : 0.0; };
    const auto most = [](double l, double u, double s) { return fmax(fabs(l - s), fabs(u - s)); };
    double bound = INFINITY;
    for (int s = tid; s < ns; s += 256) {
      const double dx = most(lx, ux, seeds[3 * (long long)s]), dy = most(ly, uy, seeds[3 * (long long)s + 1]),
                   dz = most(lz, uz, seeds[3 * (long long)s + 2]);
      bound = fmin(bound, dx * dx + dy * dy + dz * dz);
    }
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) bound = fmin(bound, __shfl_xor(bound, o, 64));
    __syncthreads();  // the candidates of the box before
    if (lane == 0) wmin[wave] = bound;
    __syncthreads();
    bound = fmin(fmin(wmin[0], wmin[1]), fmin(wmin[2], wmin[3]));
    int n = 0;
    for (int s0 = 0; s0 < ns; s0 += 256) {
      const int s = s0 + tid;
      double px = 0.0, py = 0.0, pz = 0.0;
      bool keep = false;
      if (s < ns) {
        px = seeds[3 * (long long)s];
        py = seeds[3 * (long long)s + 1];
        pz = seeds[3 * (long long)s + 2];
        const double dx = least(lx, ux, px), dy = least(ly, uy, py), dz = least(lz, uz, pz);
        keep = dx * dx + dy * dy + dz * dz <= bound;
      }
      const unsigned long long m = __ballot(keep);
      if (lane == 0) wcount[wave] = __popcll(m);
      __syncthreads();
      int at = n + __popcll(m & ((1ULL << lane) - 1));
      for (int w = 0; w < wave; ++w) at += wcount[w];
      if (keep && at < VCAND) {
        cx[at] = px;
        cy[at] = py;
        cz[at] = pz;
        cid[at] = s;
      }
      n += wcount[0] + wcount[1] + wcount[2] + wcount[3];
      __syncthreads();
    }
    const bool all = n > VCAND;
    for (int i = tid; i < VX * VY * VZ; i += 256) {
      const int ix = x0 + i % VX, iy = y0 + i / VX % VY, iz = z0 + i / (VX * VY);
      if (ix >= nx || iy >= ny || iz >= nz) continue;
      const double gx = ((double)ix + 0.5) * hx, gy = ((double)iy + 0.5) * hy, gz = ((double)iz + 0.5) * hz;
      double best = INFINITY;
      int bi = 0;
      const int m = all ? ns : n;
      for (int j = 0; j < m; ++j) {
        const double dx = gx - (all ? seeds[3 * (long long)j] : cx[j]), dy = gy - (all ? seeds[3 * (long long)j + 1] : cy[j]),
                     dz = gz - (all ? seeds[3 * (long long)j + 2] : cz[j]);
        const double d = dx * dx + dy * dy + dz * dz;
        if (d < best) {
          best = d;
          bi = all ? j : cid[j];
        }
      }
      out[((long long)iz * ny + iy) * nx + ix] = gori ? gori[bi] : bi;
    }
  }
}

// CFD coupling (coupled/example.py:31-42): T_pf[(z, y, x)] = r T_past[(x, y, z)] + (1 - r) T_future[(x, y, z)].
// A block transposes a square of CT x CT cells (x, z) of one y through LDS, so that both the snapshots (z
// fastest) and the result (x fastest) are read and written in contiguous rows.  128x96x48, FP64: 6.0 us
// (each thread reading its two values at a stride of ny nz: 8.5 us).
constexpr int CT = 32;

template <class TT>
__global__ __launch_bounds__(256) void cfd_temperature_kernel(const TT* __restrict__ past, const TT* __restrict__ fut,
                                                             int nz, int ny, int nx, double r, long long tiles,
                                                             TT* __restrict__ out) {
  __shared__ TT tile[CT][CT + 1];
  const int tx = (nx + CT - 1) / CT, tz = (nz + CT - 1) / CT;
  const int l = threadIdx.x % CT, m = threadIdx.x / CT;  // 8 rows at a time
  for (long long w = blockIdx.x; w < tiles; w += gridDim.x) {
    const long long q = w / tx;
    const int x0 = (int)(w - q * tx) * CT, z0 = (int)(q % tz) * CT, iy = (int)(q / tz);
#pragma unroll
    for (int k = 0; k < CT; k += 8) {
      const int ix = x0 + m + k, iz = z0 + l;
      if (ix < nx && iz < nz) {
        const long long src = ((long long)ix * ny + iy) * nz + iz;
        tile[m + k][l] = (TT)(r * (double)past[src] + (1.0 - r) * (double)fut[src]);
      }
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < CT; k += 8) {
      const int ix = x0 + l, iz = z0 + m + k;
      if (ix < nx && iz < nz) out[((long long)iz * ny + iy) * nx + ix] = tile[l][m + k];
    }
    __syncthreads();
  }
}

static bool grid_ok(long long n, long long threads_per_item) {
  return (n + 255) / 256 * threads_per_item < (1LL << 31);
}

// The launch of a step: checks the arguments that do not concern the state buffers, fills the
// instance description with the tiling and names the kernel.
static int plan_step(const pf_params_t* p, int dtype, const void* T_dev, const void* axes_dev, int tile, int zchunk,
                     StepDev& a, StepLaunch& fn) {
  int rc = make_stepdev(p, dtype, T_dev, axes_dev, zchunk, a);
  if (rc) return rc;
  const bool aniso = p->anisotropy > 0.0;
  if (tile < -2) return fail(PF_E_ARG, "tile must be >= -2");
  const StepEntry* e = tile == -2 ? nullptr : find_entry(dtype, p->num_oris, aniso, tile);
  const long long n = (long long)p->nz * p->ny * p->nx;
  if (e) {
    if (zchunk < 0 || (zchunk & ~(PF_ZCHUNK_TAIL | 0xffff)) != 0)
      return fail(PF_E_ARG, "zchunk must be a plane count in [0, 65535], optionally | PF_ZCHUNK_TAIL");
    if (march_fits(p, dtype)) return PF_E_ARG;
    if (tile == -1) e = choose_step(dtype, p->num_oris, aniso, p->nz, p->ny, p->nx);
  } else if (tile > 0 && entry_count(dtype, p->num_oris, aniso) > 0) {
    return fail(PF_E_ARG, "no such tile shape");
  }
  if (e) {
    const long long cols = (long long)((p->nx + e->tx - 1) / e->tx) * ((p->ny + e->ty - 1) / e->ty);
    if ((zchunk & 0xffff) == 0) zchunk |= fill_zchunk(p->nz, cols, held_workgroups(e, false));
    set_tiles(a, e->tx, e->ty, zchunk);
    a.rsh = deal_rows(a, held_workgroups(e, false)) ? 3 : 0;
    if (tile_launch(a) >= (1LL << 31)) return fail(PF_E_ARG, "too many tiles");
    fn = e->step;
  } else {
    if (!grid_ok(n, 1)) return fail(PF_E_ARG, "grid too large for the generic kernel");
    set_quads(a, dtype, zchunk > 0 ? zchunk & 0xffff : 0);
    fn = generic_step(dtype, p->num_oris, aniso);
  }
  return PF_OK;
}

}  // namespace pf

using namespace pf;

// ====================================================================== C ABI
extern "C" {

int pf_version(void) { return PFHIP_ABI_VERSION; }

const char* pf_last_error(void) { return g_err.c_str(); }

int pf_abi_sizes(size_t* params, size_t* laser, size_t* batch_inst) {
  if (params) *params = sizeof(pf_params_t);
  if (laser) *laser = sizeof(pf_laser_t);
  if (batch_inst) *batch_inst = sizeof(pf_batch_inst_t);
  return PF_OK;
}

int pf_device_count(void) {
  int n = 0;
  if (hipGetDeviceCount(&n) != hipSuccess) {
    (void)hipGetLastError();
    return 0;
  }
  return n;
}

int pf_tile_count(int32_t dtype, int32_t k) { return entry_count(dtype, k, false); }

int pf_tile_shape(int32_t dtype, int32_t k, int32_t tile, int32_t* tx, int32_t* ty) {
  const StepEntry* e = find_entry(dtype, k, false, tile);
  if (!e) return fail(PF_E_ARG, "no such tile shape for this (dtype, K)");
  if (tx) *tx = e->tx;
  if (ty) *ty = e->ty;
  return PF_OK;
}

int pf_tile_lanes(int32_t dtype, int32_t k, int32_t tile) {
  const StepEntry* e = find_entry(dtype, k, false, tile);
  if (!e) return fail(PF_E_ARG, "no such tile shape for this (dtype, K)");
  return e->h;
}

int pf_fast_path(int32_t dtype, int32_t k) { return entry_count(dtype, k, false) > 0 ? 1 : 0; }

int pf_step(const void* eta_in_dev, void* eta_out_dev, int32_t dtype, const void* T_dev, const pf_params_t* p,
            const void* axes_dev, double t_prev, double t_crt, int32_t tile, int32_t zchunk, void* stream) {
  if (!eta_in_dev || !eta_out_dev) return fail(PF_E_ARG, "eta buffers must be non-NULL");
  if (eta_in_dev == eta_out_dev) return fail(PF_E_ARG, "eta_in and eta_out must not alias");
  if (((uintptr_t)eta_in_dev | (uintptr_t)eta_out_dev) & 15)
    return fail(PF_E_ARG, "eta buffers must be 16-byte aligned");
  StepDev a;
  StepLaunch fn;
  int rc = plan_step(p, dtype, T_dev, axes_dev, tile, zchunk, a, fn);
  if (rc) return rc;
  hipError_t err = fn(a, make_dyn(a, eta_in_dev, eta_out_dev, t_prev, t_crt - t_prev), (hipStream_t)stream);  // allen_cahn.py:112
  return err == hipSuccess ? PF_OK : hip_fail(err, "pf_step launch");
}

int pf_run(const void* eta_in_dev, void* buf0_dev, void* buf1_dev, int32_t dtype, const void* T_dev,
           const pf_params_t* p, const void* axes_dev, const double* ts, int32_t steps, int32_t tile, int32_t zchunk,
           void* stream) {
  if (!eta_in_dev || !buf0_dev || !buf1_dev || !ts) return fail(PF_E_ARG, "NULL argument");
  // eta_in may be buf1: step 1 has read it before step 2 writes it
  if (eta_in_dev == buf0_dev || buf0_dev == buf1_dev)
    return fail(PF_E_ARG, "buf0 must alias neither eta_in nor buf1");
  if (((uintptr_t)eta_in_dev | (uintptr_t)buf0_dev | (uintptr_t)buf1_dev) & 15)
    return fail(PF_E_ARG, "eta buffers must be 16-byte aligned");
  if (steps < 1) return fail(PF_E_ARG, "steps must be >= 1");
  StepDev a;
  StepLaunch fn;
  int rc = plan_step(p, dtype, T_dev, axes_dev, tile, zchunk, a, fn);
  if (rc) return rc;
  const void* in = eta_in_dev;
  for (int i = 0; i < steps; ++i) {
    void* out = i % 2 == 0 ? buf0_dev : buf1_dev;
    hipError_t err = fn(a, make_dyn(a, in, out, ts[i], ts[i + 1] - ts[i]), (hipStream_t)stream);
    if (err != hipSuccess) return hip_fail(err, "pf_run launch");
    in = out;
  }
  return PF_OK;
}

int pf_rhs(const void* eta_in_dev, void* rhs_out_dev, int32_t dtype, const void* T_dev, const pf_params_t* p,
           const void* axes_dev, double t, void* stream) {
  if (!eta_in_dev || !rhs_out_dev) return fail(PF_E_ARG, "eta/rhs buffers must be non-NULL");
  if (eta_in_dev == rhs_out_dev) return fail(PF_E_ARG, "eta_in and rhs_out must not alias");
  StepDev a;
  int rc = make_stepdev(p, dtype, T_dev, axes_dev, 0, a);
  if (rc) return rc;
  const StepDyn d = make_dyn(a, eta_in_dev, rhs_out_dev, t, 1.0);  // c1, c2 carry L only: rhs = -L (grad + laplace)
  const long long n = (long long)p->nz * p->ny * p->nx;
  if (!grid_ok(n, 1)) return fail(PF_E_ARG, "grid too large");
  set_quads(a, dtype, 0);
  hipError_t err = generic_rhs(dtype, p->num_oris, p->anisotropy > 0.0)(a, d, (hipStream_t)stream);
  return err == hipSuccess ? PF_OK : hip_fail(err, "pf_rhs launch");
}

int pf_rk4(const void* eta_in_dev, void* eta_out_dev, void* work_dev, void* sum_dev, int32_t dtype, const void* T_dev,
           const pf_params_t* p, const void* axes_dev, double t_prev, double t_crt, void* stream) {
  if (!eta_in_dev || !eta_out_dev || !work_dev || !sum_dev) return fail(PF_E_ARG, "NULL buffer");
  const void* bufs[4] = {eta_in_dev, eta_out_dev, work_dev, sum_dev};
  for (int i = 0; i < 4; ++i)
    for (int j = 0; j < i; ++j)
      if (bufs[i] == bufs[j]) return fail(PF_E_ARG, "the buffers must not alias");
  StepDev a;
  int rc = make_stepdev(p, dtype, T_dev, axes_dev, 0, a);
  if (rc) return rc;
  if (!quad_fits(dtype, p->num_oris)) return fail(PF_E_UNSUPPORTED, "pf_rk4: too many orientations");
  if (!grid_ok((long long)p->nz * p->ny * p->nx, 1)) return fail(PF_E_ARG, "grid too large");
  if (set_quads(a, dtype, 0) >= kQuadLaunch) return fail(PF_E_UNSUPPORTED, "pf_rk4: too many planes");
  const double h = t_crt - t_prev;
  const double t[4] = {t_prev, t_prev + h / 2.0, t_prev + h / 2.0, t_prev + h};  // allen_cahn.py:93-99
  const double c[4] = {h / 2.0, h / 2.0, h, h / 6.0};
  const void* in[4] = {eta_in_dev, work_dev, eta_out_dev, work_dev};
  void* out[4] = {work_dev, eta_out_dev, work_dev, eta_out_dev};
  for (int i = 0; i < 4; ++i) {
    hipError_t err = rk_stage(a, make_dyn(a, in[i], out[i], t[i], 1.0), RkStage{eta_in_dev, sum_dev, c[i], i + 1}, dtype,
                              p->anisotropy > 0.0, (hipStream_t)stream);
    if (err != hipSuccess) return hip_fail(err, "pf_rk4 launch");
  }
  return PF_OK;
}

int pf_temperature(void* T_dev, int32_t T_dtype, const pf_params_t* p, double t, void* stream) {
  if (!T_dev) return fail(PF_E_ARG, "T buffer is NULL");
  if (T_dtype != PF_F64 && T_dtype != PF_F32) return fail(PF_E_ARG, "T dtype must be PF_F64 or PF_F32");
  if (p && p->laser.model == PF_T_BUFFER) return fail(PF_E_ARG, "PF_T_BUFFER has no closed-form temperature");
  StepDev a;
  int rc = make_stepdev(p, PF_F64, nullptr, (const void*)1, 0, a);
  if (rc) return rc;
  const long long n = (long long)p->nz * p->ny * p->nx;
  if (!grid_ok(n, 1)) return fail(PF_E_ARG, "grid too large");
  const dim3 g((unsigned)((n + 255) / 256));
  if (T_dtype == PF_F64)
    temperature_kernel<double><<<g, 256, 0, (hipStream_t)stream>>>(a, (double*)T_dev, t);
  else
    temperature_kernel<float><<<g, 256, 0, (hipStream_t)stream>>>(a, (float*)T_dev, t);
  hipError_t err = hipGetLastError();
  return err == hipSuccess ? PF_OK : hip_fail(err, "pf_temperature launch");
}

int pf_cfd_temperature(const void* T_past_dev, const void* T_future_dev, int32_t T_dtype, int32_t nz, int32_t ny,
                       int32_t nx, double t_pf, double t_cfd, double dt_cfd, void* T_out_dev, void* stream) {
  if (!T_past_dev || !T_future_dev || !T_out_dev) return fail(PF_E_ARG, "NULL buffer");
  if (T_dtype != PF_F64 && T_dtype != PF_F32) return fail(PF_E_ARG, "T dtype must be PF_F64 or PF_F32");
  if (nz < 1 || ny < 1 || nx < 1) return fail(PF_E_ARG, "grid dimensions must be >= 1");
  if (!(dt_cfd != 0.0)) return fail(PF_E_ARG, "dt_cfd must be non-zero");
  const long long n = (long long)nz * ny * nx;
  if (!grid_ok(n, 1)) return fail(PF_E_ARG, "grid too large");
  const double r = (t_cfd - t_pf) / dt_cfd;  // coupled/example.py:40
  const long long tiles = (long long)((nx + CT - 1) / CT) * ((nz + CT - 1) / CT) * ny;
  const dim3 g((unsigned)(tiles < (1 << 20) ? tiles : 1 << 20));
  hipStream_t s = (hipStream_t)stream;
  if (T_dtype == PF_F64)
    cfd_temperature_kernel<double><<<g, 256, 0, s>>>((const double*)T_past_dev, (const double*)T_future_dev, nz, ny,
                                                     nx, r, tiles, (double*)T_out_dev);
  else
    cfd_temperature_kernel<float><<<g, 256, 0, s>>>((const float*)T_past_dev, (const float*)T_future_dev, nz, ny, nx,
                                                    r, tiles, (float*)T_out_dev);
  hipError_t err = hipGetLastError();
  return err == hipSuccess ? PF_OK : hip_fail(err, "pf_cfd_temperature launch");
}

int pf_init_onehot(void* eta_dev, int32_t dtype, const int32_t* ori_dev, int64_t n_cells, int32_t k, void* stream) {
  if (!eta_dev || !ori_dev) return fail(PF_E_ARG, "NULL buffer");
  if (!valid_dtype(dtype)) return fail(PF_E_ARG, "bad dtype");
  if (n_cells < 1 || k < 1) return fail(PF_E_ARG, "n_cells and k must be >= 1");
  const long long ne = (long long)n_cells * k;
  if (!grid_ok(ne, 1)) return fail(PF_E_ARG, "state too large");
  const long long blocks = (n_cells + OC - 1) / OC;
  const dim3 g((unsigned)(blocks < (1 << 20) ? blocks : 1 << 20));
  hipStream_t s = (hipStream_t)stream;
  switch (dtype) {
    case PF_F64: onehot_kernel<double><<<g, 256, 0, s>>>((double*)eta_dev, ori_dev, n_cells, k); break;
    case PF_F32: onehot_kernel<float><<<g, 256, 0, s>>>((float*)eta_dev, ori_dev, n_cells, k); break;
    case PF_BF16: onehot_kernel<bf16_t><<<g, 256, 0, s>>>((bf16_t*)eta_dev, ori_dev, n_cells, k); break;
  }
  hipError_t err = hipGetLastError();
  return err == hipSuccess ? PF_OK : hip_fail(err, "pf_init_onehot launch");
}

int pf_voronoi(const double* seeds_dev, int32_t n_seeds, const int32_t* grain_ori_dev, const pf_params_t* p,
               int32_t* out_dev, void* stream) {
  if (!seeds_dev || !out_dev || !p) return fail(PF_E_ARG, "NULL argument");
  if (n_seeds < 1) return fail(PF_E_ARG, "n_seeds must be >= 1");
  if (p->nz < 1 || p->ny < 1 || p->nx < 1) return fail(PF_E_ARG, "grid dimensions must be >= 1");
  const long long n = (long long)p->nz * p->ny * p->nx;
  if (!grid_ok(n, 1)) return fail(PF_E_ARG, "grid too large");
  const long long boxes = (long long)((p->nx + VX - 1) / VX) * ((p->ny + VY - 1) / VY) * ((p->nz + VZ - 1) / VZ);
  voronoi_kernel<<<(unsigned)(boxes < (1 << 20) ? boxes : 1 << 20), 256, 0, (hipStream_t)stream>>>(
      seeds_dev, n_seeds, grain_ori_dev, p->nz, p->ny, p->nx, p->h[0], p->h[1], p->h[2], boxes, out_dev);
  hipError_t err = hipGetLastError();
  return err == hipSuccess ? PF_OK : hip_fail(err, "pf_voronoi launch");
}

}  // extern "C"

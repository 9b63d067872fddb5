// State diagnostics of libpfhip.so: argmax over orientations and the FP64 reductions
// (pf_argmax, pf_reduce, pf_reduce_noalloc).
//
// Both passes have to read eta once.  The K channels of a cell are dealt to Q = ceil(K / V) threads
// of V consecutive channels each, so that a wavefront reads a contiguous run of memory whatever K is;
// the per-cell quantities (sum of squares, argmax) are combined through LDS by one thread per cell.
//   argmax, 256x256x64, K = 20, FP32: 62 us, 5.7 TB/s, the rate of a copy (one thread per cell reading
//   its row value by value: 256 us; BF16 34 us, FP64 on half the cells 61 us).
//   reduce, the same state: 127 us (a thread per cell with its three neighbour rows, a second
//   pass for the volumes and one block adding up the partials: 1648 + 1593 + 1463 us).  Bound by the
//   issue of VALU instructions, 46 a value, which keep the SIMDs busy 83 % of the time: 14 are FP64
//   arithmetic, 4 conversions, 8 integer arithmetic, the rest the compares and selects of argmax and
//   finiteness and copies.  The reads take 57 us, LDS bank conflicts 5 % of the time.
#include <math.h>

#include <mutex>
#include <string>

#include "pf_host.h"

namespace pf {

constexpr int RB = 256;     // threads per block of both passes
constexpr int RMAXK = 256;  // pf_reduce handles K <= RMAXK
constexpr int NF = 4;       // F_local, F_grad, max T, sum eta
constexpr int NI = 3;       // changed, liquid, nonfinite

// numpy.argmax semantics among a thread's own channels: first maximum; a NaN is the maximum (first
// NaN wins).
template <class TS, int V, bool TAIL>
__device__ __forceinline__ void quad_argmax(const QuadAt<TS, V, TAIL>& at, const typename Traits<TS>::TC (&v)[V],
                                            typename Traits<TS>::TC& best, int& bi) {
  typename Traits<TS>::TC b = v[0];
  int i = at.s;
#pragma unroll
  for (int e = 1; e < V; ++e) {
    const bool take = ((b == b) & !(v[e] <= b) & (e > at.e0)) | (TAIL & (e == at.e0));
    b = take ? v[e] : b;
    i = take ? at.s + e : i;
  }
  best = b;
  bi = i;
}

// Best of a cell's groups in order of their channels.
template <class TC>
__device__ __forceinline__ int merge_argmax(const TC* __restrict__ mx, const int* __restrict__ ix, int Q) {
  TC best = mx[0];
  int bi = ix[0];
#pragma unroll 4
  for (int q = 1; q < Q; ++q) {
    const TC v = mx[q];
    const int i = ix[q];
    const bool take = (best == best) & !(v <= best);
    best = take ? v : best;
    bi = take ? i : bi;
  }
  return bi;
}

// ------------------------------------------------------------------ argmax
// A block takes AR runs of C = RB / Q cells (one contiguous piece of memory); every thread issues
// its AR loads before the first use.
constexpr int AR = 4;

template <class TS, int V, bool TAIL>
__global__ __launch_bounds__(RB) void argmax_kernel(const TS* __restrict__ eta, long long n_cells, int K, int Q, int C,
                                                   int32_t* __restrict__ out) {
  using TC = typename Traits<TS>::TC;
  __shared__ TC mx[AR][RB];
  __shared__ int ix[AR][RB];
  const int j = threadIdx.x / Q;
  const QuadAt<TS, V, TAIL> at(K, threadIdx.x - j * Q);
  const long long c0 = (long long)blockIdx.x * (C * AR);
  const int n = (int)min((long long)(C * AR), n_cells - c0);
  const TS* base = eta + (c0 + j) * K;
  TC v[AR][V];
  // the last block's missing cells read its last one again (their results are not used)
#pragma unroll
  for (int r = 0; r < AR; ++r) at.load(base + (long long)min(r * C, n - 1 - j) * K, v[r]);
#pragma unroll
  for (int r = 0; r < AR; ++r) quad_argmax(at, v[r], mx[r][threadIdx.x], ix[r][threadIdx.x]);
  __syncthreads();
  for (int i = threadIdx.x; i < n; i += RB) {
    const int r = i / C, cj = i - r * C;
    out[c0 + i] = merge_argmax(&mx[r][cj * Q], &ix[r][cj * Q], Q);
  }
}

// One thread per cell: K of more than RB groups.
template <class TS>
__global__ __launch_bounds__(RB) void argmax_rows_kernel(const TS* __restrict__ eta, long long n_cells, int K,
                                                        int32_t* __restrict__ out) {
  using TC = typename Traits<TS>::TC;
  const long long c = (long long)blockIdx.x * RB + threadIdx.x;
  if (c >= n_cells) return;
  const TS* row = eta + c * K;
  TC best = to_tc(row[0]);
  int bi = 0;
  for (int i = 1; i < K && best == best; ++i) {
    const TC v = to_tc(row[i]);
    if (v != v || v > best) {
      best = v;
      bi = i;
    }
  }
  out[c] = bi;
}

// ------------------------------------------------------------------ FP64 diagnostics
__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}
__device__ __forceinline__ double wave_max(double v) {
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) v = fmax(v, __shfl_xor(v, o, 64));
  return v;
}
__device__ __forceinline__ long long wave_sum_i(long long v) {
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}

// Shape of a reduction: tiles of C cells of a z-plane (a contiguous run) by zc planes, walked by nb
// blocks.  Block b takes tiles b, b + nb, ...; tile t belongs to XCD t % 8 (workgroups are dealt
// round-robin), which walks its own eighth of the plane's runs, so that the y-neighbours of a run are
// read into the same L2 that has them.
struct RedGeo {
  int Q, C, nrun, m, zc, nb;
  long long tiles;
};

constexpr int kRedBlocks = 1024;  // four blocks of 256 threads on each of 256 CUs (what registers and LDS allow)
constexpr int RG = 4;             // planes whose cells are summed up together, by all threads of a block
constexpr int kRedTab = 1024;     // (cell, plane) pairs of a tile at most

static long long red_block_cap(long long n) {
  const long long b = (n + 31) / 32;
  return b < 1 ? 1 : b > kRedBlocks ? kRedBlocks : b;
}

static RedGeo red_geo(int nz, int ny, int nx, int K, int V) {
  RedGeo g;
  const long long nxy = (long long)nx * ny;
  g.Q = (K + V - 1) / V;
  g.C = RB / g.Q;
  g.nrun = (int)((nxy + g.C - 1) / g.C);
  g.m = (g.nrun + 7) / 8;
  const long long cap = red_block_cap(nxy * nz);
  // number of z-chunks: the best product of how evenly the tiles fill the blocks and the share of a
  // tile's planes that is not its extra plane below
  const int zmax = kRedTab / g.C < nz ? kRedTab / g.C : nz;
  double best = -1.0;
  g.zc = 1;
  for (int zc = zmax; zc >= 1; --zc) {
    const double t = (double)g.nrun * ((nz + zc - 1) / zc);
    const double eff = t / (ceil(t / (double)cap) * (double)cap) * zc / (zc + 1.0);
    if (eff > best) {
      best = eff;
      g.zc = zc;
    }
  }
  g.tiles = 8LL * g.m * ((nz + g.zc - 1) / g.zc);
  g.nb = (int)(g.tiles < cap ? g.tiles : cap);
  return g;
}

// s += |a - b|^2 in FP64
template <class TC, int V>
__device__ __forceinline__ void sq_diff(const TC (&a)[V], const TC (&b)[V], double& s) {
#pragma unroll
  for (int e = 0; e < V; ++e) {
    const double d = (double)a[e] - (double)b[e];
    s = fma(d, d, s);
  }
}

// A block marches its run of cells up through the planes of a tile with the plane below in registers
// (the z-differences), the next plane requested one plane ahead; x- and y-neighbours are read again
// from the caches.  The cells of RG planes are summed up together: one plane at a time, a single
// wavefront's chain of LDS reads per plane set the time (282 us against 134).  The temperatures of a
// tile are evaluated before its march by all threads.
// Partial results of nb blocks: double [NF][nb], double [K][nb], int32 [K + NI][nb].
template <class TS, int V, bool TAIL>
__global__ __launch_bounds__(RB) __attribute__((amdgpu_waves_per_eu(4))) void reduce_kernel(const StepDev a, const TS* __restrict__ eta,
                                                   const int32_t* __restrict__ argmax0, double t, double m_g,
                                                   double gamma, double ad_hoc, double half_kappa_ad, RedGeo g,
                                                   double* __restrict__ part_f, double* __restrict__ part_v,
                                                   int32_t* __restrict__ part_i) {
  using TC = typename Traits<TS>::TC;
  // per-group results of RG planes
  __shared__ double s2[RG * RB], s4[RG * RB];
  __shared__ TC mx[RG * RB];
  __shared__ int ix[RG * RB];
  __shared__ int hist[RMAXK];
  __shared__ double sf[RB / 64][NF];
  __shared__ long long si[RB / 64][NI];
  __shared__ double tab[kRedTab];  // (1 - zeta)^2 of the tile's cells; at the end the volumes' partial sums
  static_assert(RB * V <= kRedTab, "volume sums fit the table");
  const int tid = threadIdx.x;
  const int K = a.k, nx = a.nx, ny = a.ny, nz = a.nz, Q = g.Q, C = g.C;
  const int nxy = nx * ny;
  const int j = tid / Q;
  const QuadAt<TS, V, TAIL> at(K, tid - j * Q);
  for (int i = tid; i < K; i += RB) hist[i] = 0;
  double f_loc = 0.0, gx = 0.0, gy = 0.0, gz = 0.0, tmax = -INFINITY;
  double vs[V];
#pragma unroll
  for (int e = 0; e < V; ++e) vs[e] = 0.0;
  int changed = 0, liquid = 0, nonfinite = 0;
  const long long plane = (long long)nxy * K;
  for (long long w = blockIdx.x; w < g.tiles; w += g.nb) {
    const int i8 = (int)(w >> 3), layer = i8 / g.m;
    const int run = (int)(w & 7) * g.m + (i8 - layer * g.m);
    if (run >= g.nrun) continue;
    const int zb = layer * g.zc, len = min(nz - zb, g.zc);
    const int p0 = run * C;
    // this thread's channels of cell p0 + j
    const int p = p0 + j;
    const bool on = j < C && p < nxy;
    const int py = p / nx, px = p - py * nx;
    const bool hasx = on && px + 1 < nx, hasy = on && py + 1 < ny;
    const TS* r = eta + ((long long)zb * nxy + p) * K;
    const int dx = K, dy = nx * K;  // a z-plane holds fewer than 2^31 values
    TC prev[V], n[V], nx_[V], ny_[V];
    if (on) {
      if (zb > 0) at.load(r - plane, prev);
      at.load(r, n);
    }
    if (hasx) at.load(r + dx, nx_);
    if (hasy) at.load(r + dy, ny_);
    lds_barrier();  // hist; the table of the tile before
    // temperatures of the tile, before the march over its planes: every thread takes part, and the
    // constants of the source and of exp and tanh hold no registers during the march
    for (int i = tid; i < len * C; i += RB) {
      const int l = i / C, cp = p0 + (i - l * C);
      if (cp < nxy) {
        const StepDev& ac = reload(a);
        const int cy = cp / nx, cx = cp - cy * nx;
        const double T = cell_temperature(ac, cx, cy, zb + l, (long long)(zb + l) * nxy + cp, t);
        const double Tc = T > ac.T_clip ? ac.T_clip : T;
        // zeta as in cell_coef64: tanh only inside the window where it is not exactly +-1
        double zeta;
        if (fabs(Tc - ac.T_l) > ac.zeta_window) zeta = Tc < ac.T_l ? 1.0 : 0.0;
        else zeta = 0.5 * (1.0 - tanh(ac.theta * (Tc / ac.T_l - 1.0)));
        const double omz = 1.0 - zeta;
        tab[i] = omz * omz;
        if (T >= ac.T_l) ++liquid;
        tmax = fmax(tmax, T);
      }
    }
    for (int l0 = 0; l0 < len; l0 += RG) {
#pragma unroll
      for (int k = 0; k < RG; ++k) {
        const int l = l0 + k;
        if (l < len && on) {
          // take over the plane requested one plane ago, and request the next one before using it
          TC v[V], vx[V], vy[V];
#pragma unroll
          for (int e = 0; e < V; ++e) {
            v[e] = n[e];
            vx[e] = nx_[e];
            vy[e] = ny_[e];
          }
          r += plane;
          if (l + 1 < len) {
            at.load(r, n);
            if (hasx) at.load(r + dx, nx_);
            if (hasy) at.load(r + dy, ny_);
          }
          double S = 0.0, F = 0.0;
#pragma unroll
          for (int e = 0; e < V; ++e) {
            const double x = (double)v[e];
            const double x2 = x * x;
            S += x2;
            F = fma(x2, x2, F);
            vs[e] += x;
            nonfinite += isfinite(v[e]) ? 0 : 1;
          }
          if (hasx) sq_diff(vx, v, gx);
          if (hasy) sq_diff(vy, v, gy);
          if (zb + l > 0) sq_diff(v, prev, gz);
          s2[k * RB + tid] = S;
          s4[k * RB + tid] = F;
          quad_argmax(at, v, mx[k * RB + tid], ix[k * RB + tid]);
#pragma unroll
          for (int e = 0; e < V; ++e) prev[e] = v[e];
        }
      }
      lds_barrier();
      for (int i = tid; i < min(RG, len - l0) * C; i += RB) {
        const int k = i / C, ci = i - k * C;
        if (p0 + ci < nxy) {
          const long long cell = (long long)(zb + l0 + k) * nxy + p0 + ci;
          const int am0 = argmax0 ? argmax0[cell] : 0;
          const int at0 = k * RB + ci * Q;
          double S1 = 0.0, F1 = 0.0;
#pragma unroll 4
          for (int c = 0; c < Q; ++c) {
            S1 += s2[at0 + c];
            F1 += s4[at0 + c];
          }
          const int am = merge_argmax(&mx[at0], &ix[at0], Q);
          // allen_cahn.py:45-48 with sum_ij (eta_i eta_j)^2 = S^2
          f_loc += F1 / 4.0 - S1 / 2.0 + gamma * (S1 * S1 - F1) + tab[(l0 + k) * C + ci] * S1;
          atomicAdd(&hist[am], 1);
          if (argmax0 && am0 != am) ++changed;
        }
      }
      lds_barrier();
    }
  }
  // fixed-order block reduction: wave butterflies, then waves in index order
  __syncthreads();
#pragma unroll
  for (int e = 0; e < V; ++e) tab[tid * V + e] = vs[e];
  f_loc = wave_sum(f_loc);
  const double f_grad = wave_sum(fma(gz, a.ihz2, fma(gy, a.ihy2, gx * a.ihx2)));
  tmax = wave_max(tmax);
  const long long nchanged = wave_sum_i(changed), nliquid = wave_sum_i(liquid), nbad = wave_sum_i(nonfinite);
  const int wv = tid / 64;
  if ((tid & 63) == 0) {
    sf[wv][0] = f_loc;
    sf[wv][1] = f_grad;
    sf[wv][2] = tmax;
    si[wv][0] = nchanged;
    si[wv][1] = nliquid;
    si[wv][2] = nbad;
  }
  __syncthreads();
  // channel i of the block: group min(i / V, Q - 1) of every cell slot, element i - s of it
  double* cs = s2;  // K <= RB values
  for (int i = tid; i < K; i += RB) {
    const int gq = i / V, gs = TAIL ? min(V * gq, K - V) : V * gq;
    double sum = 0.0;
    for (int c = 0; c < C; ++c) sum += tab[(c * Q + gq) * V + (i - gs)];
    part_v[(long long)i * g.nb + blockIdx.x] = sum;
    part_i[(long long)i * g.nb + blockIdx.x] = hist[i];
    cs[i] = sum;
  }
  __syncthreads();
  if (tid == 0) {
    double r[NF] = {0.0, 0.0, -INFINITY, 0.0};
    long long ri[NI] = {0, 0, 0};
    for (int k = 0; k < RB / 64; ++k) {
      r[0] += sf[k][0];
      r[1] += sf[k][1];
      r[2] = fmax(r[2], sf[k][2]);
      for (int c = 0; c < NI; ++c) ri[c] += si[k][c];
    }
    r[0] = m_g * r[0] / ad_hoc;
    r[1] *= half_kappa_ad;
    for (int i = 0; i < K; ++i) r[3] += cs[i];
    for (int c = 0; c < NF; ++c) part_f[(long long)c * g.nb + blockIdx.x] = r[c];
    // fewer than 2^40 values over at least min(n / 32, 1024) blocks: a block's counts fit 32 bits
    for (int c = 0; c < NI; ++c) part_i[(long long)(K + c) * g.nb + blockIdx.x] = (int32_t)ri[c];
  }
}

// One block per output value; fixed order (thread strides, wave butterflies, waves in index order).
__global__ __launch_bounds__(RB) void reduce_final_kernel(int nb, int K, double dV, const double* __restrict__ part_f,
                                                         const double* __restrict__ part_v,
                                                         const int32_t* __restrict__ part_i,
                                                         double* __restrict__ out_f, long long* __restrict__ out_i) {
  __shared__ double sd[RB / 64];
  __shared__ long long sl[RB / 64];
  const int tid = threadIdx.x, o = blockIdx.x;
  if (o < NF + K) {
    const double* src = o < NF ? part_f + (long long)o * nb : part_v + (long long)(o - NF) * nb;
    const bool mxo = o == 2;
    double r = mxo ? -INFINITY : 0.0;
    for (int b = tid; b < nb; b += RB) r = mxo ? fmax(r, src[b]) : r + src[b];
    r = mxo ? wave_max(r) : wave_sum(r);
    if ((tid & 63) == 0) sd[tid / 64] = r;
    __syncthreads();
    if (tid == 0) {
      r = sd[0];
      for (int k = 1; k < RB / 64; ++k) r = mxo ? fmax(r, sd[k]) : r + sd[k];
      out_f[o] = (o == 2 || o == 3) ? r : r * dV;
    }
  } else {
    const int i = o - NF - K;
    long long r = 0;
    for (int b = tid; b < nb; b += RB) r += part_i[(long long)i * nb + b];
    r = wave_sum_i(r);
    if ((tid & 63) == 0) sl[tid / 64] = r;
    __syncthreads();
    if (tid == 0) {
      r = sl[0];
      for (int k = 1; k < RB / 64; ++k) r += sl[k];
      out_i[i] = r;
    }
  }
}

template <class TS>
static void launch_argmax(const TS* eta, long long n_cells, int K, int V, int32_t* out, hipStream_t s) {
  const int Q = (K + V - 1) / V, C = RB / Q;
  const unsigned nb = (unsigned)((n_cells + C * AR - 1) / (C * AR));
  with_quad<TS>(K, V, [&](auto v, auto tail) {
    argmax_kernel<TS, decltype(v)::value, decltype(tail)::value><<<nb, RB, 0, s>>>(eta, n_cells, K, Q, C, out);
  });
}

template <class TS>
static void launch_reduce(const StepDev& a, const TS* eta, const int32_t* argmax0, const pf_params_t* p, double t,
                          const RedGeo& g, int V, double* part_f, double* part_v, int32_t* part_i, hipStream_t s) {
  const double hk = 0.5 * p->kappa_g * p->ad_hoc;
  with_quad<TS>(a.k, V, [&](auto v, auto tail) {
    reduce_kernel<TS, decltype(v)::value, decltype(tail)::value><<<g.nb, RB, 0, s>>>(
        a, eta, argmax0, t, p->m_g, p->gamma, p->ad_hoc, hk, g, part_f, part_v, part_i);
  });
}

static size_t red_bytes(long long nb, int K) {
  return (size_t)(nb * (NF + K) * 8 + (nb * (K + NI) * 4 + 7) / 8 * 8);
}

}  // namespace pf

using namespace pf;

extern "C" {

int pf_argmax(const void* eta_dev, int32_t dtype, int64_t n_cells, int32_t k, int32_t* out_dev, void* stream) {
  if (!eta_dev || !out_dev) return fail(PF_E_ARG, "NULL buffer");
  if (!valid_dtype(dtype)) return fail(PF_E_ARG, "bad dtype");
  if (n_cells < 1 || k < 1) return fail(PF_E_ARG, "n_cells and k must be >= 1");
  if ((n_cells + RB - 1) / RB >= (1LL << 31)) return fail(PF_E_ARG, "grid too large");
  hipStream_t s = (hipStream_t)stream;
  const int V = quad_of(dtype, k), Q = (k + V - 1) / V, C = Q <= RB ? RB / Q : 0;
  if (C > 0 && (n_cells + C * AR - 1) / (C * AR) < (1LL << 24)) {  // a launch has fewer than 2^32 threads
    switch (dtype) {
      case PF_F64: launch_argmax((const double*)eta_dev, n_cells, k, V, out_dev, s); break;
      case PF_F32: launch_argmax((const float*)eta_dev, n_cells, k, V, out_dev, s); break;
      case PF_BF16: launch_argmax((const bf16_t*)eta_dev, n_cells, k, V, out_dev, s); break;
    }
  } else {
    const dim3 g((unsigned)((n_cells + RB - 1) / RB));
    switch (dtype) {
      case PF_F64: argmax_rows_kernel<double><<<g, RB, 0, s>>>((const double*)eta_dev, n_cells, k, out_dev); break;
      case PF_F32: argmax_rows_kernel<float><<<g, RB, 0, s>>>((const float*)eta_dev, n_cells, k, out_dev); break;
      case PF_BF16: argmax_rows_kernel<bf16_t><<<g, RB, 0, s>>>((const bf16_t*)eta_dev, n_cells, k, out_dev); break;
    }
  }
  hipError_t err = hipGetLastError();
  return err == hipSuccess ? PF_OK : hip_fail(err, "pf_argmax launch");
}

// The partial results of the blocks, at most 1024 of them: 0.4 MB for K = 20, 3.2 MB for K = 256.  Never
// less than the tables of ceil(n / 2048) rows and ceil(n / 4096) column sums of an earlier layout, so that the grids
// that pf_reduce_noalloc refuses for their size stay the same.
size_t pf_reduce_workspace_bytes(int64_t n_cells, int32_t k) {
  if (n_cells < 1 || k < 1) return 0;
  long long rows = (n_cells + 2047) / 2048;
  if (rows > 2048) rows = 2048;
  const long long cols = (n_cells + 4095) / 4096;
  const size_t floor_bytes = (size_t)(rows * (NF + k + NI) * 8 + cols * k * 8);
  const size_t need = red_bytes(red_block_cap(n_cells), k);
  return need > floor_bytes ? need : floor_bytes;
}

}  // extern "C"

namespace {

// Argument checks shared by pf_reduce and pf_reduce_noalloc (host only, no HIP call):
// fills the instance description and the workspace size the reduction needs.
int reduce_check(const void* eta_dev, int32_t dtype, const void* T_dev, const pf_params_t* p,
                 const double* out_f64_dev, const int64_t* out_i64_dev, StepDev& a, size_t& need) {
  if (!eta_dev || !out_f64_dev || !out_i64_dev) return fail(PF_E_ARG, "NULL buffer");
  int rc = make_stepdev(p, dtype, T_dev, (const void*)1, 0, a);
  if (rc) return rc;
  if (p->num_oris > RMAXK) return fail(PF_E_UNSUPPORTED, "pf_reduce supports K <= 256");
  need = pf_reduce_workspace_bytes((long long)p->nz * p->ny * p->nx, p->num_oris);
  return PF_OK;
}

// The two reduction launches over a workspace of at least pf_reduce_workspace_bytes bytes.
// Every partial result is written before it is read, so the workspace needs no clearing.
int reduce_launch(const StepDev& a, const void* eta_dev, int32_t dtype, const int32_t* argmax0_dev,
                  const pf_params_t* p, double t, double* out_f64_dev, int64_t* out_i64_dev, void* ws_dev,
                  void* stream) {
  const int K = p->num_oris;
  const int V = quad_of(dtype, K);
  const RedGeo g = red_geo(p->nz, p->ny, p->nx, K, V);
  double* part_f = (double*)ws_dev;
  double* part_v = part_f + (long long)g.nb * NF;
  int32_t* part_i = (int32_t*)(part_v + (long long)g.nb * K);
  hipStream_t s = (hipStream_t)stream;
  switch (dtype) {
    case PF_F64: launch_reduce(a, (const double*)eta_dev, argmax0_dev, p, t, g, V, part_f, part_v, part_i, s); break;
    case PF_F32: launch_reduce(a, (const float*)eta_dev, argmax0_dev, p, t, g, V, part_f, part_v, part_i, s); break;
    case PF_BF16: launch_reduce(a, (const bf16_t*)eta_dev, argmax0_dev, p, t, g, V, part_f, part_v, part_i, s); break;
  }
  const double dV = p->h[0] * p->h[1] * p->h[2];
  reduce_final_kernel<<<NF + K + K + NI, RB, 0, s>>>(g.nb, K, dV, part_f, part_v, part_i, out_f64_dev,
                                                     (long long*)out_i64_dev);
  hipError_t err = hipGetLastError();
  return err == hipSuccess ? PF_OK : hip_fail(err, "pf_reduce launch");
}

}  // namespace

// ---- allocation-free diagnostics (pf_reduce_noalloc)
// The reduction's partial results live in this fixed array instead of a caller workspace.
// Each GPU holds its own copy from code-object load until the process ends.  In host code
// `scratch` names a host-side stand-in, not device memory: kernels get the device address
// that hipGetSymbolAddress returns for the current device (scratch_dev below).
static __device__ __align__(256) unsigned char scratch[PF_REDUCE_SCRATCH_BYTES];

namespace {

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
void* g_scratch_dev[kMaxDevices];  // device address of `scratch` per device, looked up once

// Device address of `scratch` on the current device (set up on the first call per device).
int scratch_dev(void** out) {
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return hip_fail(e, "hipGetDevice");
  if (dev < 0 || dev >= kMaxDevices) return fail(PF_E_UNSUPPORTED, "pf_reduce_noalloc supports devices 0..63");
  std::lock_guard<std::mutex> lk(g_scratch_mu);
  if (!g_scratch_dev[dev]) {
    void* ptr = nullptr;
    e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
    if (e != hipSuccess) return hip_fail(e, "hipGetSymbolAddress(scratch)");
    if (!ptr) return fail(PF_E_HIP, "hipGetSymbolAddress(scratch) returned NULL");
    g_scratch_dev[dev] = ptr;
  }
  *out = g_scratch_dev[dev];
  return PF_OK;
}

}  // namespace

extern "C" {

int pf_reduce(const void* eta_dev, int32_t dtype, const void* T_dev, const int32_t* argmax0_dev,
              const pf_params_t* p, double t, double* out_f64_dev, int64_t* out_i64_dev, void* ws_dev,
              size_t ws_bytes, void* stream) {
  StepDev a;
  size_t need = 0;
  int rc = reduce_check(eta_dev, dtype, T_dev, p, out_f64_dev, out_i64_dev, a, need);
  if (rc) return rc;
  if (!ws_dev) return fail(PF_E_ARG, "NULL workspace");
  if (ws_bytes < need) return fail(PF_E_ARG, "workspace too small");
  return reduce_launch(a, eta_dev, dtype, argmax0_dev, p, t, out_f64_dev, out_i64_dev, ws_dev, stream);
}

int pf_reduce_noalloc(const void* eta_dev, int32_t dtype, const void* T_dev, const int32_t* argmax0_dev,
                      const pf_params_t* p, double t, double* out_f64_dev, int64_t* out_i64_dev, void* stream) {
  StepDev a;
  size_t need = 0;
  int rc = reduce_check(eta_dev, dtype, T_dev, p, out_f64_dev, out_i64_dev, a, need);
  if (rc) return rc;
  if (need > (size_t)PF_REDUCE_SCRATCH_BYTES)
    return fail(PF_E_ARG, "pf_reduce_noalloc: the reduction needs " + std::to_string(need) +
                              " bytes of scratch, more than its fixed " + std::to_string(PF_REDUCE_SCRATCH_BYTES) +
                              " (use pf_reduce with a workspace)");
  void* ws = nullptr;
  rc = scratch_dev(&ws);
  if (rc) return rc;
  return reduce_launch(a, eta_dev, dtype, argmax0_dev, p, t, out_f64_dev, out_i64_dev, ws, stream);
}

}  // extern "C"

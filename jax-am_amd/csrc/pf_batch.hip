// Batched engine of libpfhip.so: many independent phase-field instances advanced
// together.  Design:
//   - Slot table (StepDev descriptors, BatchSlot step counters and each slot's StepDyn
//     step arguments) lives in device memory; after each block of up to kPlan steps the device
//     advances each slot's step index and ping-pong parity and plans its next kPlan steps,
//     so a captured graph stays valid while instances come and go.
//   - Instances are grouped into classes (dtype, K, anisotropy, tile shape).  Each
//     class has a device-resident work list of (slot, tile) items walked by one
//     persistent launch per step with a fixed grid; in a captured block of steps the classes (or the parts
//     of a lone large one) run on branches of the graph.
//   - A class whose instances together leave the GPU short of workgroups runs shorter marches than its
//     instances ask for, or the march of channel groups (rebuild_work).
//   - `chunk` steps (launches of the classes that have work, an advance per block) are captured
//     into one HIP graph and replayed.  Graphs are cached by (chunk, set of classes with
//     work and their kernels): admitting or removing an instance only rewrites table entries and work
//     lists, and a new capture happens only for a class set not seen before.
// The kernel and march length of an instance may change from rebuild to rebuild as others of its class come
// and go.  Its trajectory does not: every kernel (tile shape, lane split, channel groups, one thread per cell) and
// every march length gives bitwise the same step (test_gpu_parity, test_gpu_anyk, test_gpu_batch_blocks).
#include <string.h>

#include <algorithm>
#include <mutex>
#include <vector>

#include "pf_host.h"

namespace pf {

// After a block of `steps` steps (0 when slots have come or gone): advance every active slot's counters
// and plan its next kPlan steps.  A block's threads are eight slots by kPlan steps: every thread has read
// its slot before the first of them writes it.  One launch per block of steps: one per step took
// 5.0 us of each, for two dependent reads and a few stores.
__global__ __launch_bounds__(8 * kPlan) void advance_kernel(StepDev* __restrict__ descs, BatchSlot* __restrict__ slots,
                                                           StepDyn* __restrict__ dyns, int n, int steps) {
  const int s = blockIdx.x * 8 + threadIdx.x / kPlan, i = threadIdx.x % kPlan;
  BatchSlot b;
  b.active = 0;
  if (s < n) b = slots[s];
  __syncthreads();
  if (!b.active) return;
  const int done = min(steps, b.steps_left);
  if (done > 0) {
    b.steps_left -= done;
    b.parity ^= done & 1;
    b.n += done;
    b.tnow = b.path ? b.path[PF_PATH_ROW * (long long)(b.n - 1) + 1] : b.t0 + (double)b.n * b.dt;
    if (i == 0) slots[s] = b;
  }
  if (i >= b.steps_left) return;
  const int m = b.n + i, par = b.parity ^ (i & 1);
  StepDyn* d = dyns + i * n + s;
  if (b.path) {
    StepDev a = descs[s];
    const double* r = b.path + PF_PATH_ROW * (long long)m;
    apply_path_row(a, r);
    descs[(1 + i) * n + s] = a;
    *d = make_dyn(a, b.eta[par], b.eta[par ^ 1], r[0], r[1] - r[0]);
  } else {
    const double tp = b.t0 + (double)m * b.dt, tc = b.t0 + (double)(m + 1) * b.dt;
    *d = make_dyn(descs[s], b.eta[par], b.eta[par ^ 1], tp, tc - tp);  // allen_cahn.py:112  h = t_crt - t_prev
  }
}

// A slot's description and counters, passed by value: nothing of the caller's is read after the launch.
__global__ void put_kernel(StepDev* desc, BatchSlot* slot, const StepDev a, const BatchSlot b) {
  if (threadIdx.x == 0) *desc = a;
  if (threadIdx.x == 1) *slot = b;
}

// Tiling of every slot (rebuild_work) into its description and those of its planned steps.
struct SlotTiles {
  int tiles_x, tiles_y, tiles_z, zc, zs, zsplit;
};
__global__ __launch_bounds__(64) void tiles_kernel(StepDev* __restrict__ descs, const SlotTiles* __restrict__ t, int n) {
  const int s = blockIdx.x * 64 + threadIdx.x;
  if (s >= n) return;
  const SlotTiles v = t[s];
  StepDev& a = descs[s];
  a.tiles_x = v.tiles_x;
  a.tiles_y = v.tiles_y;
  a.tiles_z = v.tiles_z;
  a.zc = v.zc;
  a.zs = v.zs;
  a.zsplit = v.zsplit;
}

struct BatchClass {
  int dtype, k, aniso, tile;
  const StepEntry* entry;  // tile shape, null for K without tiled kernels
  bool quads;              // the class runs the march of channel groups (always for a null entry)
  int count;  // host copy of the work-item count
  int users;  // slots in this class; a class without users is retired and its index reused
};

struct SlotHost {
  bool used = false;
  int cls = -1;
  int charge = 0;  // what the slot counts for against max_tiles: its tiles, or its blocks of 256 cells
  int zchunk = 0;  // planes per march at most (0: the default), as the instance asked
  int path = 0;    // 1: it has a source table
  StepDev a;       // its description with the tiling it was given last
};

}  // namespace pf

using namespace pf;

struct pf_batch {
  int max_inst = 0, max_tiles = 0;
  static constexpr int kMaxClasses = 64;
  hipStream_t stream = nullptr;
  StepDev* d_desc = nullptr;
  StepDyn* d_dyn = nullptr;
  BatchSlot* d_slots = nullptr;
  WorkItem* d_work = nullptr;
  size_t work_cap = 0;     // items that d_work holds (at least max_tiles)
  int2* d_info = nullptr;  // per class (work-list offset, count), then those of a lone class's parts
  SlotTiles* d_tiles = nullptr;
  std::vector<SlotHost> slots;
  std::vector<BatchClass> classes;
  bool work_dirty = false;
  int parts = 1;  // that a lone class's instances are dealt to (rebuild_work)
  struct Graph {
    int chunk;
    unsigned long long mask, quads;  // classes with work, and those of them on channel groups
    int parts;                       // of a lone class
    hipGraph_t def;
    hipGraphExec_t exec;
  };
  static constexpr int kMaxGraphs = 16;
  std::vector<Graph> graphs;  // most recently used last
  static constexpr int kSide = 2;  // streams that a captured block of steps forks to (launch_steps)
  hipStream_t side[kSide] = {};
  hipEvent_t forked = nullptr, joined[kSide] = {};
  std::mutex mu;
};

namespace {

// Values (cells x orientations) from which a lone tiled class's launches are split over the branches: 21 million of
// eight 64x64x32 48.2 -> 44.7 us a step; below, three of 36x36x30 (2.3 million) 14.3 -> 16.0, twelve of 32^3, K = 10
// (3.9 million) 17.6 -> 18.9.  On channel groups a split loses at any size measured (50x50x34, K = 33 38 -> 42).
constexpr long long kSplitValues = 12000000;
constexpr int kForkSteps = 4;  // steps of a block from which its launches fork (launch_steps)
constexpr int kBatchQuads = 1024;  // workgroups of the batched march of channel groups on 256 CUs

void drop_graphs(pf_batch* b) {
  for (pf_batch::Graph& g : b->graphs) {
    (void)hipGraphExecDestroy(g.exec);
    (void)hipGraphDestroy(g.def);
  }
  b->graphs.clear();
}

// Tiling of class c's slots.  A class with more than three fillings of the GPU (held workgroups) is tiled as its
// instances asked (short marches balance the work, long ones read less: the autotuner's choice).  Below
// that the length that ends with every CU busy is best: of the shortest marches that need one,
// two and three fillings, the least fillings times planes (two more than a march writes are read).  A
// class small enough for the march of channel groups (small_step) runs that.
// Eight requests of 36x36x30 to 72x72x40 cells, K = 10, 16, 20, FP32: 80 us a step at the asked 6 and 8 planes,
// 63 us here (of both without the scalar reads of constant_at; 52 us with them).
void tile_class(pf_batch* b, int c) {
  BatchClass& k = b->classes[c];
  long long cells = 0;
  for (const SlotHost& s : b->slots)
    if (s.used && s.cls == c) cells += (long long)s.a.nz * s.a.ny * s.a.nx;
  k.quads = !k.entry || small_step(k.dtype, k.k, cells);
  if (k.quads) {
    long long runs = 0;
    for (SlotHost& s : b->slots)
      if (s.used && s.cls == c) {
        set_quads(s.a, k.dtype, 1);
        runs += 8LL * s.a.tiles_y;
      }
    for (SlotHost& s : b->slots)
      if (s.used && s.cls == c) {
        const long long chunks = runs > 0 && kBatchQuads > runs ? kBatchQuads / runs : 1;
        set_quads(s.a, k.dtype, (int)((s.a.nz + chunks - 1) / chunks));
      }
    return;
  }
  const int tx = k.entry->tx, ty = k.entry->ty;
  const auto tile_all = [&](int zc) {  // 0: as asked
    long long items = 0;
    for (SlotHost& s : b->slots)
      if (s.used && s.cls == c) {
        set_tiles(s.a, tx, ty, zc == 0 || (s.zchunk & PF_ZCHUNK_TAIL) ? s.zchunk : zc);
        items += (long long)s.a.tiles_x * s.a.tiles_y * s.a.tiles_z;
      }
    return items;
  };
  const long long held = held_workgroups(k.entry, true);
  if (tile_all(0) > 3 * held) return;
  int best = 0, best_cost = 0;
  for (int m = 1, zc = 16; m <= 3; ++m) {
    if (tile_all(zc) > m * held) continue;
    while (zc > 2 && tile_all(zc - 1) <= m * held) --zc;
    if (best == 0 || m * (zc + 2) < best_cost) {
      best = zc;
      best_cost = m * (zc + 2);
    }
  }
  tile_all(best);
}

int rebuild_work(pf_batch* b) {
  for (size_t c = 0; c < b->classes.size(); ++c)
    if (b->classes[c].users > 0) tile_class(b, (int)c);
  // pack each class's work items contiguously, in slot order; of a lone class, each part's: a slot goes to the
  // part with the fewest items so far
  int live = 0, used = 0;
  for (const BatchClass& k : b->classes) live += k.users > 0;
  long long values = 0;
  for (const SlotHost& sh : b->slots)
    if (sh.used && !b->classes[sh.cls].quads) {
      used += 1;
      values += (long long)sh.a.nz * sh.a.ny * sh.a.nx * b->classes[sh.cls].k;
    }
  b->parts = live == 1 && values >= kSplitValues ? std::min(used, 1 + pf_batch::kSide) : 1;
  std::vector<std::vector<WorkItem>> per(pf_batch::kMaxClasses + 1 + pf_batch::kSide);
  std::vector<SlotTiles> tiles(b->max_inst, SlotTiles{0, 0, 0, 0, 0, 0});
  for (int s = 0; s < b->max_inst; ++s) {
    const SlotHost& sh = b->slots[s];
    if (!sh.used) continue;
    const StepDev& a = sh.a;
    tiles[s] = SlotTiles{a.tiles_x, a.tiles_y, a.tiles_z, a.zc, a.zs, a.zsplit};
    const BatchClass& k = b->classes[sh.cls];
    const long long items = !k.quads                  ? (long long)a.tiles_x * a.tiles_y * a.tiles_z
                            : quad_fits(k.dtype, k.k) ? 8LL * a.tiles_y * a.tiles_z
                                                      : sh.charge;
    if (items >= (1LL << 31)) return fail(PF_E_ARG, "instance too large");
    int to = b->parts > 1 ? pf_batch::kMaxClasses : sh.cls;
    for (int p = 1; p < b->parts; ++p)
      if (per[pf_batch::kMaxClasses + p].size() < per[to].size()) to = pf_batch::kMaxClasses + p;
    for (int t = 0; t < (int)items; ++t) per[to].push_back(WorkItem{s, t, sh.path, 0});
  }
  std::vector<WorkItem> all;
  std::vector<int2> info(per.size());
  for (size_t c = 0; c < per.size(); ++c) {
    if (c < b->classes.size()) b->classes[c].count = (int)per[c].size();
    info[c] = make_int2((int)all.size(), (int)per[c].size());
    all.insert(all.end(), per[c].begin(), per[c].end());
  }
  if (b->parts > 1)  // the class's own entry spans its parts, which lie one after the other
    for (size_t c = 0; c < b->classes.size(); ++c)
      if (b->classes[c].users > 0) {
        b->classes[c].count = (int)all.size();
        info[c] = make_int2(0, (int)all.size());
      }
  hipError_t e = hipSuccess;
  if (all.size() > b->work_cap) {
    // more items than max_tiles, by which slots are charged as they asked to be tiled: a longer list;
    // the graphs that hold the old one's address go with it
    WorkItem* grown = nullptr;
    const size_t cap = all.size() + all.size() / 2;
    e = hipMalloc((void**)&grown, sizeof(WorkItem) * cap);
    if (e != hipSuccess) return hip_fail(e, "pf_batch work list");
    e = hipStreamSynchronize(b->stream);
    drop_graphs(b);
    (void)hipFree(b->d_work);
    b->d_work = grown;
    b->work_cap = cap;
    if (e != hipSuccess) return hip_fail(e, "pf_batch work list");
  }
  if (!all.empty())
    e = hipMemcpyAsync(b->d_work, all.data(), all.size() * sizeof(WorkItem), hipMemcpyHostToDevice, b->stream);
  if (e == hipSuccess)
    e = hipMemcpyAsync(b->d_info, info.data(), info.size() * sizeof(int2), hipMemcpyHostToDevice, b->stream);
  if (e == hipSuccess)
    e = hipMemcpyAsync(b->d_tiles, tiles.data(), tiles.size() * sizeof(SlotTiles), hipMemcpyHostToDevice, b->stream);
  if (e == hipSuccess) {
    tiles_kernel<<<(b->max_inst + 63) / 64, 64, 0, b->stream>>>(b->d_desc, b->d_tiles, b->max_inst);
    advance_kernel<<<(b->max_inst + 7) / 8, 8 * kPlan, 0, b->stream>>>(b->d_desc, b->d_slots, b->d_dyn, b->max_inst, 0);
    e = hipGetLastError();
  }
  // the host vectors above are pageable and local: finish the copies before they go away
  if (e == hipSuccess) e = hipStreamSynchronize(b->stream);
  if (e != hipSuccess) return hip_fail(e, "pf_batch work-list upload");
  b->work_dirty = false;
  return PF_OK;
}

unsigned long long active_mask(const pf_batch* b) {
  unsigned long long m = 0;
  for (size_t c = 0; c < b->classes.size(); ++c)
    if (b->classes[c].count > 0) m |= 1ULL << c;
  return m;
}

unsigned long long quad_mask(const pf_batch* b) {
  unsigned long long m = 0;
  for (size_t c = 0; c < b->classes.size(); ++c)
    if (b->classes[c].count > 0 && b->classes[c].quads) m |= 1ULL << c;
  return m;
}

// `steps` steps of every class with work, in blocks of up to kPlan with an advance after each.  The classes' slots
// have nothing in common but the tables, which only the advance writes: with `fork` (a capture) a block's
// launches of different classes, or of a lone class's parts, run on branches of the graph, each step after step,
// and their tails and latencies overlap.  us a step, on one stream -> forked: eighteen requests of 36x36x30 to
// 72x72x40 in six classes 87 -> 60, 64 instances of 32^3 to 128x128x64 4.41e11 -> 5.06e11 updates/s; a lone class
// of K = 20: eight of 64x64x32 in FP32 48.2 -> 44.7, eight of 72x72x40 in BF16 51.5 -> 43.6, four in FP64 133 -> 108.  The fork and the
// join take about 13 us a block: three classes of one 32^3 instance each 26.9 -> 46.3 in blocks of one step, 22.2 -> 30.3 of
// two, 19.8 -> 18.3 of four, 18.9 -> 15.3 of eight; hence kForkSteps.  More branches than three gained nothing.
int launch_steps(pf_batch* b, int steps, bool fork) {
  const BatchView v{b->d_desc, b->d_dyn, b->d_slots, b->d_work, b->d_info, b->max_inst};
  struct Launch {
    int cls, info;  // class, and which entry of d_info holds its items
  };
  std::vector<Launch> whole, parts;
  for (size_t c = 0; c < b->classes.size(); ++c) {
    if (b->classes[c].count == 0) continue;
    whole.push_back(Launch{(int)c, (int)c});
    for (int p = 0; p < b->parts; ++p)
      parts.push_back(Launch{(int)c, b->parts > 1 ? pf_batch::kMaxClasses + p : (int)c});
  }
  for (int done = 0; done < steps;) {
    const int n = std::min(kPlan, steps - done);
    const bool forked = fork && n >= kForkSteps;
    const std::vector<Launch>& live = forked ? parts : whole;
    const int branches = forked ? std::max(1, std::min((int)live.size(), 1 + pf_batch::kSide)) : 1;
    hipError_t e = hipSuccess;
    if (branches > 1) e = hipEventRecord(b->forked, b->stream);
    for (int s = 1; s < branches && e == hipSuccess; ++s) e = hipStreamWaitEvent(b->side[s - 1], b->forked, 0);
    if (e != hipSuccess) return hip_fail(e, "pf_batch fork");
    for (int i = 0; i < n; ++i) {
      for (size_t l = 0; l < live.size(); ++l) {
        const BatchClass& k = b->classes[live[l].cls];
        // (workgroups: tiled classes 1024 / 2048 / 4096 / 8192: c3 4.73 / 4.90 / 5.06 / 5.10e11 updates/s, two of
        // 256x256x64 271 / 279 / 267 / 265 us, but six small classes 59.9 / 59.3 / 60.6 / 64.7 us)
        const BatchLaunch fn = k.quads ? generic_batch(k.dtype, k.k, k.aniso != 0) : k.entry->batch;
        const int s = (int)(l % branches);
        e = fn(v, live[l].info, i, k.quads ? 2048 : 4096, k.k, s ? b->side[s - 1] : b->stream);
        if (e != hipSuccess) return hip_fail(e, "pf_batch step launch");
      }
    }
    for (int s = 1; s < branches && e == hipSuccess; ++s) {
      e = hipEventRecord(b->joined[s - 1], b->side[s - 1]);
      if (e == hipSuccess) e = hipStreamWaitEvent(b->stream, b->joined[s - 1], 0);
    }
    if (e != hipSuccess) return hip_fail(e, "pf_batch join");
    advance_kernel<<<(b->max_inst + 7) / 8, 8 * kPlan, 0, b->stream>>>(b->d_desc, b->d_slots, b->d_dyn, b->max_inst, n);
    e = hipGetLastError();
    if (e != hipSuccess) return hip_fail(e, "pf_batch advance launch");
    done += n;
  }
  return PF_OK;
}

// Destroy the cached graphs that launch class c (its index is about to be retired).  The
// caller has synchronized the stream, so none of them is in flight.
void drop_graphs_of_class(pf_batch* b, int c) {
  const unsigned long long bit = 1ULL << c;
  for (size_t i = 0; i < b->graphs.size();) {
    if (b->graphs[i].mask & bit) {
      (void)hipGraphExecDestroy(b->graphs[i].exec);
      (void)hipGraphDestroy(b->graphs[i].def);
      b->graphs.erase(b->graphs.begin() + i);
    } else {
      ++i;
    }
  }
}

// The graph of `chunk` steps for the current class set (captured on first use).
int get_graph(pf_batch* b, int chunk, hipGraphExec_t* out) {
  const unsigned long long mask = active_mask(b), quads = quad_mask(b);
  for (size_t i = 0; i < b->graphs.size(); ++i) {
    if (b->graphs[i].chunk == chunk && b->graphs[i].mask == mask && b->graphs[i].quads == quads &&
        b->graphs[i].parts == b->parts) {
      pf_batch::Graph g = b->graphs[i];
      b->graphs.erase(b->graphs.begin() + i);
      b->graphs.push_back(g);
      *out = g.exec;
      return PF_OK;
    }
  }
  hipError_t e = hipStreamBeginCapture(b->stream, hipStreamCaptureModeThreadLocal);
  if (e != hipSuccess) return hip_fail(e, "hipStreamBeginCapture");
  const int rc = launch_steps(b, chunk, true);
  hipGraph_t g = nullptr;
  e = hipStreamEndCapture(b->stream, &g);
  if (rc) {
    if (g) (void)hipGraphDestroy(g);
    return rc;
  }
  if (e != hipSuccess) return hip_fail(e, "hipStreamEndCapture");
  hipGraphExec_t ex = nullptr;
  e = hipGraphInstantiate(&ex, g, nullptr, nullptr, 0);
  if (e != hipSuccess) {
    (void)hipGraphDestroy(g);
    return hip_fail(e, "hipGraphInstantiate");
  }
  if ((int)b->graphs.size() >= pf_batch::kMaxGraphs) {
    // the oldest graph may still be in flight: finish the stream before destroying it
    (void)hipStreamSynchronize(b->stream);
    (void)hipGraphExecDestroy(b->graphs.front().exec);
    (void)hipGraphDestroy(b->graphs.front().def);
    b->graphs.erase(b->graphs.begin());
  }
  b->graphs.push_back(pf_batch::Graph{chunk, mask, quads, b->parts, g, ex});
  *out = ex;
  return PF_OK;
}

}  // namespace

extern "C" {

pf_batch_t* pf_batch_create(int32_t max_instances, int32_t max_tiles, void* stream) {
  if (max_instances < 1 || max_tiles < 1) {
    set_error("max_instances and max_tiles must be >= 1");
    return nullptr;
  }
  pf_batch* b = new pf_batch();
  b->max_inst = max_instances;
  b->max_tiles = max_tiles;
  b->stream = (hipStream_t)stream;
  b->work_cap = max_tiles;
  b->slots.resize(max_instances);
  hipError_t e = hipMalloc((void**)&b->d_desc, sizeof(StepDev) * (1 + kPlan) * max_instances);
  if (e == hipSuccess) e = hipMalloc((void**)&b->d_dyn, sizeof(StepDyn) * kPlan * max_instances);
  if (e == hipSuccess) e = hipMalloc((void**)&b->d_slots, sizeof(BatchSlot) * max_instances);
  if (e == hipSuccess) e = hipMalloc((void**)&b->d_work, sizeof(WorkItem) * max_tiles);
  if (e == hipSuccess) e = hipMalloc((void**)&b->d_info, sizeof(int2) * (pf_batch::kMaxClasses + 1 + pf_batch::kSide));
  if (e == hipSuccess) e = hipMalloc((void**)&b->d_tiles, sizeof(SlotTiles) * max_instances);
  if (e == hipSuccess) e = hipEventCreateWithFlags(&b->forked, hipEventDisableTiming);
  for (int s = 0; s < pf_batch::kSide && e == hipSuccess; ++s) {
    e = hipStreamCreateWithFlags(&b->side[s], hipStreamNonBlocking);
    if (e == hipSuccess) e = hipEventCreateWithFlags(&b->joined[s], hipEventDisableTiming);
  }
  if (e == hipSuccess) {
    std::vector<BatchSlot> z(max_instances);
    memset(z.data(), 0, z.size() * sizeof(BatchSlot));
    std::vector<int2> zc(pf_batch::kMaxClasses + 1 + pf_batch::kSide, make_int2(0, 0));
    e = hipMemcpyAsync(b->d_slots, z.data(), z.size() * sizeof(BatchSlot), hipMemcpyHostToDevice, b->stream);
    if (e == hipSuccess)
      e = hipMemcpyAsync(b->d_info, zc.data(), zc.size() * sizeof(int2), hipMemcpyHostToDevice, b->stream);
    if (e == hipSuccess) e = hipStreamSynchronize(b->stream);
  }
  if (e != hipSuccess) {
    hip_fail(e, "pf_batch_create");
    pf_batch_destroy(b);
    return nullptr;
  }
  return b;
}

void pf_batch_destroy(pf_batch_t* b) {
  if (!b) return;
  if (b->stream) (void)hipStreamSynchronize(b->stream);
  drop_graphs(b);
  if (b->forked) (void)hipEventDestroy(b->forked);
  for (int s = 0; s < pf_batch::kSide; ++s) {
    if (b->joined[s]) (void)hipEventDestroy(b->joined[s]);
    if (b->side[s]) (void)hipStreamDestroy(b->side[s]);
  }
  if (b->d_desc) (void)hipFree(b->d_desc);
  if (b->d_dyn) (void)hipFree(b->d_dyn);
  if (b->d_slots) (void)hipFree(b->d_slots);
  if (b->d_work) (void)hipFree(b->d_work);
  if (b->d_info) (void)hipFree(b->d_info);
  if (b->d_tiles) (void)hipFree(b->d_tiles);
  delete b;
}

int pf_batch_add(pf_batch_t* b, const pf_batch_inst_t* inst) {
  if (!b || !inst) return fail(PF_E_ARG, "NULL batch or instance");
  std::lock_guard<std::mutex> lk(b->mu);
  if (!inst->eta_dev[0] || !inst->eta_dev[1] || inst->eta_dev[0] == inst->eta_dev[1])
    return fail(PF_E_ARG, "an instance needs two distinct state buffers");
  if (((uintptr_t)inst->eta_dev[0] | (uintptr_t)inst->eta_dev[1]) & 15)
    return fail(PF_E_ARG, "eta buffers must be 16-byte aligned");
  if (inst->steps < 0) return fail(PF_E_ARG, "steps must be >= 0");
  if (inst->zchunk < 0 || (inst->zchunk & ~(PF_ZCHUNK_TAIL | 0xffff)) != 0)
    return fail(PF_E_ARG, "zchunk must be a plane count in [0, 65535], optionally | PF_ZCHUNK_TAIL");
  if (inst->path_dev && inst->p.laser.model != PF_T_ROSENTHAL && inst->p.laser.model != PF_T_GAUSSIAN)
    return fail(PF_E_ARG, "a source table needs a Rosenthal or Gaussian source");
  int slot = -1;
  for (int s = 0; s < b->max_inst; ++s)
    if (!b->slots[s].used) {
      slot = s;
      break;
    }
  if (slot < 0) return fail(PF_E_STATE, "no free batch slot");
  StepDev a;
  int rc = make_stepdev(&inst->p, inst->dtype, inst->T_dev, inst->axes_dev, inst->zchunk, a);
  if (rc) return rc;
  const bool aniso = inst->p.anisotropy > 0.0;
  const StepEntry* e = find_entry(inst->dtype, inst->p.num_oris, aniso, inst->tile);
  int charge, tile = -1;
  if (e) {
    if (march_fits(&inst->p, inst->dtype)) return PF_E_ARG;
    set_tiles(a, e->tx, e->ty, inst->zchunk);
    charge = a.tiles_x * a.tiles_y * a.tiles_z;
    tile = e->tile;
  } else {
    if (inst->tile > 0 && entry_count(inst->dtype, inst->p.num_oris, aniso) > 0)
      return fail(PF_E_ARG, "no such tile shape");
    const long long n = (long long)inst->p.nz * inst->p.ny * inst->p.nx;
    if ((n + 255) / 256 >= (1LL << 31)) return fail(PF_E_ARG, "instance too large");
    charge = (int)((n + 255) / 256);
  }
  int total = 0;
  for (const SlotHost& sh : b->slots)
    if (sh.used) total += sh.charge;
  if (total + charge > b->max_tiles) return fail(PF_E_STATE, "batch work list full (max_tiles)");
  int cls = -1, free_cls = -1;
  for (size_t c = 0; c < b->classes.size(); ++c) {
    const BatchClass& k = b->classes[c];
    if (k.users == 0) {
      if (free_cls < 0) free_cls = (int)c;
    } else if (k.dtype == inst->dtype && k.k == inst->p.num_oris && k.aniso == (int)aniso && k.tile == tile) {
      cls = (int)c;
    }
  }
  if (cls < 0) {
    // a new class takes a retired index (its graphs were dropped when it retired) or a new one
    const BatchClass nc{inst->dtype, inst->p.num_oris, (int)aniso, tile, e, !e, 0, 0};
    if (free_cls >= 0) {
      b->classes[free_cls] = nc;
      cls = free_cls;
    } else {
      if ((int)b->classes.size() >= pf_batch::kMaxClasses)
        return fail(PF_E_STATE, "too many instance classes at once (64)");
      b->classes.push_back(nc);
      cls = (int)b->classes.size() - 1;
    }
  }
  BatchSlot st;
  memset(&st, 0, sizeof(st));
  st.steps_left = inst->steps;
  st.parity = 0;
  st.n = 0;
  st.active = 1;
  st.t0 = inst->t0;
  st.dt = inst->dt;
  st.eta[0] = inst->eta_dev[0];
  st.eta[1] = inst->eta_dev[1];
  st.tnow = inst->t0;
  st.path = inst->path_dev;
  put_kernel<<<1, 64, 0, b->stream>>>(b->d_desc + slot, b->d_slots + slot, a, st);
  hipError_t he = hipGetLastError();
  if (he != hipSuccess) return hip_fail(he, "pf_batch_add upload");
  b->slots[slot].used = true;
  b->slots[slot].cls = cls;
  b->slots[slot].charge = charge;
  b->slots[slot].zchunk = inst->zchunk;
  b->slots[slot].path = inst->path_dev ? 1 : 0;
  b->slots[slot].a = a;
  b->classes[cls].users += 1;
  b->work_dirty = true;
  return slot;
}

int pf_batch_remove(pf_batch_t* b, int32_t slot) {
  if (!b) return fail(PF_E_ARG, "NULL batch");
  std::lock_guard<std::mutex> lk(b->mu);
  if (slot < 0 || slot >= b->max_inst || !b->slots[slot].used) return fail(PF_E_ARG, "slot not in use");
  BatchSlot st;
  memset(&st, 0, sizeof(st));
  hipError_t he = hipMemcpyAsync(b->d_slots + slot, &st, sizeof(BatchSlot), hipMemcpyHostToDevice, b->stream);
  if (he == hipSuccess) he = hipStreamSynchronize(b->stream);  // st is a local
  if (he != hipSuccess) return hip_fail(he, "pf_batch_remove");
  const int cls = b->slots[slot].cls;
  b->slots[slot] = SlotHost();
  if (--b->classes[cls].users == 0) drop_graphs_of_class(b, cls);  // retired: its index is free again
  b->work_dirty = true;
  return PF_OK;
}

int pf_batch_run(pf_batch_t* b, int32_t steps, int32_t chunk) {
  if (!b) return fail(PF_E_ARG, "NULL batch");
  if (steps < 0) return fail(PF_E_ARG, "steps must be >= 0");
  std::lock_guard<std::mutex> lk(b->mu);
  if (b->work_dirty) {
    int rc = rebuild_work(b);
    if (rc) return rc;
  }
  int done = 0;
  if (chunk > 0 && steps >= chunk) {
    hipGraphExec_t g = nullptr;
    int rc = get_graph(b, chunk, &g);
    if (rc) return rc;
    for (; done + chunk <= steps; done += chunk) {
      hipError_t e = hipGraphLaunch(g, b->stream);
      if (e != hipSuccess) return hip_fail(e, "hipGraphLaunch");
    }
  }
  return launch_steps(b, steps - done, false);
}

int pf_batch_status(pf_batch_t* b, int32_t* steps_left, double* t, int32_t* parity, int32_t n) {
  if (!b) return fail(PF_E_ARG, "NULL batch");
  std::lock_guard<std::mutex> lk(b->mu);
  if (n > b->max_inst) n = b->max_inst;
  std::vector<BatchSlot> h(b->max_inst);
  hipError_t e = hipMemcpyAsync(h.data(), b->d_slots, sizeof(BatchSlot) * b->max_inst, hipMemcpyDeviceToHost,
                                b->stream);
  if (e == hipSuccess) e = hipStreamSynchronize(b->stream);
  if (e != hipSuccess) return hip_fail(e, "pf_batch_status");
  for (int s = 0; s < n; ++s) {
    if (steps_left) steps_left[s] = b->slots[s].used ? h[s].steps_left : -1;
    if (t) t[s] = h[s].tnow;
    if (parity) parity[s] = h[s].parity;
  }
  return PF_OK;
}

int pf_batch_active(const pf_batch_t* b) {
  if (!b) return 0;
  int c = 0;
  for (const SlotHost& s : b->slots) c += s.used ? 1 : 0;
  return c;
}

}  // extern "C"

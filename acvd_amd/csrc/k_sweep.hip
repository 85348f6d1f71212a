// Boundary sweep of the vertex clustering, one pass =
//   scan     : the boundary items whose clusters changed recently (or whose
//              last proposal lost) form the work list;
//   evaluate : each evaluates its best move to a neighbouring cluster
//              (isotropic or QEM energy, vtkUniformClustering.h:922-991) and,
//              if it lowers the energy, registers its accept key at the source
//              and target clusters (minimum per cluster) and joins the
//              candidate list;
//   rounds   : kMatchRounds accept rounds.  In each, a candidate whose key is
//              the minimum at both of its clusters is applied (label, int64
//              fixed-point accumulators of the two clusters, then their
//              centroid, W and FP64 rank-truncated QEM point); the remaining
//              candidates are re-evaluated against the new state when one of
//              their clusters moved, and register their next-round key;
//   controller: per-mesh phase logic of MinimizeEnergy
//              (vtkUniformClustering.h:724-830) after the pass.
// A cluster takes part in at most one applied move per round, so every
// applied dE is exact with respect to the state at the start of its round and
// the energy decreases monotonically.  Between convergences the host runs the
// clean (largest connected component per cluster, vtkUniformClustering.h:405-549)
// and fill (regrowth of null items, :551-633) kernels below.

#include <hip/hip_runtime.h>
#include <hipcub/hipcub.hpp>

#include "acvd_ctx.h"

namespace acvd {

namespace {

inline unsigned grid_for(int64_t n) { return unsigned((n + kBlock - 1) / kBlock); }

__device__ inline int mesh_of_item(const SweepArgs& a, int64_t i) { return a.item_mesh ? a.item_mesh[i] : 0; }
__device__ inline int mesh_of_cluster(const SweepArgs& a, int64_t c) { return a.clus_mesh ? a.clus_mesh[c] : 0; }

__device__ inline int64_t ld_i64(const unsigned long long* p) { return int64_t(*p); }

// ----------------------------------------------------------------- statistics
__global__ void k_zero_clusters(SweepArgs a, const int32_t* __restrict__ mask) {
  int64_t c = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (c >= a.n_clusters) return;
  if (!mask[mesh_of_cluster(a, c)]) return;
  for (int k = 0; k < 4; ++k) a.acc_ws[4 * c + k] = 0ull;
  if (a.acc_q)
    for (int k = 0; k < 10; ++k) a.acc_q[10 * c + k] = 0ull;
  a.sizes[c] = 0;
}

template <int CTRL>
__device__ inline unsigned long long dpp_u64(unsigned long long x) {
  const uint32_t lo = uint32_t(__builtin_amdgcn_update_dpp(0, int(uint32_t(x)), CTRL, 0xf, 0xf, true));
  const uint32_t hi = uint32_t(__builtin_amdgcn_update_dpp(0, int(uint32_t(x >> 32)), CTRL, 0xf, 0xf, true));
  return (uint64_t(hi) << 32) | lo;
}

// One doubling step of the segmented sum over runs of equal clusters: lane l adds
// lane l + D (of its 16-lane row) when rem lanes of its run follow it.
template <int D, int V>
__device__ inline void merge_step(unsigned long long (&v)[V], int n, int rem) {
  const bool take = rem >= D;
  if (__ballot(take) == 0ull) return;
#pragma unroll
  for (int k = 0; k < V; ++k) {
    if (k >= n) break;  // wave-uniform
    const unsigned long long t = dpp_u64<0x100 | D>(v[k]);  // row_shl:D
    v[k] += take ? t : 0ull;
  }
}

// Lanes that follow in the lane's run, given the run heads of the wave.
__device__ inline int run_left(unsigned long long heads) {
  const int lane = __lane_id();
  const unsigned long long after = lane == 63 ? 0ull : heads >> (lane + 1);
  return after ? __builtin_ctzll(after) : 63 - lane;
}

// Item contributions in int64 fixed point (order-independent sums).  Each block
// takes a contiguous range of items, 512 at a time: runs of equal clusters merge
// in registers (at most 8 lanes), each run adds once into the block's LDS table
// keyed by cluster, and the table goes to the global sums, consecutive threads to
// consecutive words, when it is three quarters full and at the end.  The quadrics
// are summed only while the mesh is constrained (nothing reads them before, and
// the recompute of the convergence that constrains it sums them).
// One table per 256 items, an LDS atomic per item and value and a global one per
// cluster and table took 870 us at 8.39 M items; now 268 us (178 without quadrics;
// a copy of the bytes read takes 100).
constexpr int kAccBlock = 512;
constexpr int kAccBlocks = 512;  // 2 per CU (61 KB of LDS each)
__global__ __launch_bounds__(kAccBlock) void k_accumulate(SweepArgs a, const int32_t* __restrict__ mask,
                                                          unsigned long long* mesh_count, int64_t chunk) {
  constexpr int V = 15;  // W, S[3], count, Q[10]
  constexpr int kSlots = 512, kSlotBits = 9, kFlushAt = kSlots * 3 / 4, kProbes = 32, kCheckSteps = 4;
  __shared__ int32_t keys[kSlots];
  __shared__ unsigned long long vals[kSlots * V];
  __shared__ int32_t n_keys;
  for (int k = threadIdx.x; k < kSlots; k += kAccBlock) keys[k] = -1;
  for (int k = threadIdx.x; k < kSlots * V; k += kAccBlock) vals[k] = 0ull;
  if (threadIdx.x == 0) n_keys = 0;
  __syncthreads();
  auto add_global = [&](int64_t c, int k, unsigned long long x) {
    if (k < 4) atomicAdd(&a.acc_ws[4 * c + k], x);
    else if (k == 4) atomicAdd(&a.sizes[c], int32_t(x));
    else atomicAdd(&a.acc_q[10 * c + k - 5], x);
  };
  auto flush = [&]() {  // every thread of the block; the table is complete
    for (int k = threadIdx.x; k < kSlots * V; k += kAccBlock) {
      const int32_t key = keys[k / V];
      const unsigned long long x = vals[k];
      vals[k] = 0ull;
      if (key >= 0 && x != 0ull) add_global(key, k % V, x);
    }
    __syncthreads();
    for (int k = threadIdx.x; k < kSlots; k += kAccBlock) keys[k] = -1;
    if (threadIdx.x == 0) n_keys = 0;
    __syncthreads();
  };
  const int64_t begin = int64_t(blockIdx.x) * chunk, end = min(begin + chunk, a.n_items);
  const int lane = __lane_id();
  const int m0 = mesh_of_item(a, begin), m1 = mesh_of_item(a, end - 1);
  int step = 0;
  for (int m = m0; m <= m1; ++m) {
    if (!mask[m]) continue;  // block-uniform
    const DevMesh& dm = a.meshes[m];
    const Scales sc = dm.scales;
    const bool with_q = dm.metric == 1 && a.state[m].constrained;
    const int64_t first = max(begin, dm.item_off), last = min(end, dm.item_off + dm.n_items);
    int counted = 0;  // items of clusters that are not frozen, per wave
    for (int64_t base = first; base < last; base += kAccBlock) {
      const int64_t i = base + threadIdx.x;
      const int32_t c = i < last ? a.labels[i] : kNull;
      unsigned long long v[V];
#pragma unroll
      for (int k = 0; k < V; ++k) v[k] = 0ull;
      if (c != kNull) {
        const float4 p = a.xw[i];
        v[0] = (unsigned long long)fix_w(p.w, sc);
        v[1] = (unsigned long long)fix_s(p.w, p.x, sc);
        v[2] = (unsigned long long)fix_s(p.w, p.y, sc);
        v[3] = (unsigned long long)fix_s(p.w, p.z, sc);
        v[4] = 1ull;
        if (with_q)
          for (int k = 0; k < 10; ++k) v[5 + k] = (unsigned long long)fix_q(a.q[10 * i + k], sc);
      }
      counted += __popcll(__ballot(c != kNull && !(a.frozen && a.frozen[c])));
      const int32_t prev = __builtin_amdgcn_update_dpp(-2, c, 0x111, 0xf, 0xf, false);  // row_shr:1
      const bool head = prev != c || (lane & 7) == 0;
      const int rem = run_left(__ballot(head));
      const int n = with_q ? V : 5;
      merge_step<1>(v, n, rem);
      merge_step<2>(v, n, rem);
      merge_step<4>(v, n, rem);
      if (head && c != kNull) {
        uint32_t h = (uint32_t(c) * 2654435761u) >> (32 - kSlotBits);
        int slot = -1;
        for (int probe = 0; probe < kProbes; ++probe) {
          const int32_t old = atomicCAS(&keys[h], -1, c);
          if (old == -1) atomicAdd(&n_keys, 1);
          if (old == -1 || old == c) {
            slot = int(h);
            break;
          }
          h = (h + 1) & (kSlots - 1);
        }
#pragma unroll
        for (int k = 0; k < V; ++k) {
          if (k >= n) break;
          if (slot >= 0) atomicAdd(&vals[slot * V + k], v[k]);
          else if (v[k] != 0ull) add_global(c, k, v[k]);  // no free slot near by
        }
      }
      if (++step % kCheckSteps == 0) {  // block-uniform
        __syncthreads();
        const bool full = n_keys > kFlushAt;
        __syncthreads();
        if (full) flush();
      }
    }
    if (mesh_count && lane == 0 && counted) atomicAdd(&mesh_count[m], (unsigned long long)counted);
  }
  __syncthreads();
  flush();
}

// Centroid, W and (QEM, constrained) T of cluster c from its accumulators;
// the solve leaves the cluster's eigenvectors in evec, which warm-start the
// trial solves on the cluster and, with warm = true, this solve itself (the
// derive after a move, whose quadric differs from the last one by one item).
// kExtras = false: no mesh has fixed clusters (the anchor test is compiled out).
template <bool kExtras = true>
__device__ void derive_cluster(const SweepArgs& a, int64_t c, const DevMesh& dm, int constrained, bool warm) {
  const int64_t W = ld_i64(&a.acc_ws[4 * c]);
  const ClusterGeom g = geom_from_fixed(W, ld_i64(&a.acc_ws[4 * c + 1]), ld_i64(&a.acc_ws[4 * c + 2]),
                                        ld_i64(&a.acc_ws[4 * c + 3]), dm.scales);
  a.geom[c] = g;
  if (dm.metric == 1) {
    double T = 0.0;
    const int32_t an = (kExtras && a.anchor) ? a.anchor[c] : -1;
    if (an >= 0) {  // a fixed cluster: its point is its anchor item's position
      const float4 p = a.xw[an];
      T = anchored_T(g, AnchorPos{double(p.x), double(p.y), double(p.z), true});
    } else if (constrained) {
      int64_t q10[10];
      for (int k = 0; k < 10; ++k) q10[k] = ld_i64(&a.acc_q[10 * c + k]);
      double V0[9];
      if (warm)
        for (int k = 0; k < 9; ++k) V0[k] = a.evec[9 * c + k];
      T = qem_T_from_fixed(q10, g, dm.scales, dm.level, nullptr, warm ? V0 : nullptr, a.evec + 9 * c);
    }
    a.T[c] = T;
  }
}

__global__ void k_derive(SweepArgs a, const int32_t* __restrict__ mask, int set_stamp) {
  int64_t c = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (c >= a.n_clusters) return;
  const int m = mesh_of_cluster(a, c);
  if (!mask[m]) return;
  const DevMesh dm = a.meshes[m];
  derive_cluster(a, c, dm, a.state[m].constrained, false);
  if (set_stamp) a.stamp[c] = a.state[m].loops;  // SetAllClustersToModified
}

// ------------------------------------------------------------------- propose
// kExtras = false: no fixed or frozen cluster exists in the context, and the
// view says so at compile time (the kernels' anchor and freeze tests fold
// away; the host picks the instantiation).
template <bool kExtras>
__device__ inline SweepView make_view(const SweepArgs& a) {
  SweepView v;
  v.row_ptr = a.row_ptr;
  v.col = a.col;
  v.labels = a.labels;
  v.xw = reinterpret_cast<const float*>(a.xw);
  v.q = a.q;
  v.acc_ws = a.acc_ws;
  v.acc_q = a.acc_q;
  v.evec = a.evec;
  v.geom = a.geom;
  v.T = a.T;
  v.sizes = a.sizes;
  v.stamp = a.stamp;
  v.cand_pass = a.cand_pass;
  v.ring_adj = a.ring_adj;
  v.anchor = kExtras ? a.anchor : nullptr;
  v.frozen = kExtras ? a.frozen : nullptr;
  return v;
}

// Neighbours of item i from the short rows (kRowPad past the row); false for a
// row of more than kRingCache neighbours, which is in the CSR alone.
__device__ inline bool load_row8(const SweepArgs& a, int64_t i, int32_t* nbr) {
  const int4 u = a.row8[2 * i], v = a.row8[2 * i + 1];
  nbr[0] = u.x;
  nbr[1] = u.y;
  nbr[2] = u.z;
  nbr[3] = u.w;
  nbr[4] = v.x;
  nbr[5] = v.y;
  nbr[6] = v.z;
  nbr[7] = v.w;
  return nbr[0] != kRowLong;
}

// Labels of the neighbours of a short row (kNull past it); returns their number.
__device__ inline int32_t load_labels8(const SweepArgs& a, const int32_t* nbr, int32_t* nb) {
  int32_t deg = 0;
#pragma unroll
  for (int p = 0; p < kRingCache; ++p) {
    nb[p] = nbr[p] >= 0 ? a.labels[nbr[p]] : kNull;
    deg += nbr[p] >= 0;
  }
  return deg;
}

// needs_eval of acvd_math.h with the neighbour loads issued together so that the
// label and stamp gathers overlap.
__device__ inline bool needs_eval_fast(const SweepArgs& a, int64_t i, int32_t lab, int32_t L) {
  int32_t nbr[kRingCache], lb[kRingCache];
  const bool is_short = load_row8(a, i, nbr);
  bool dirty = (a.cand_pass[i] == L - 1);
  if (lab != kNull) dirty |= (a.stamp[lab] + 1 >= L);
  bool boundary = false;
#pragma unroll
  for (int k = 0; k < kRingCache; ++k) lb[k] = nbr[k] >= 0 ? a.labels[nbr[k]] : lab;
  // neighbour stamps are read only while the item is not already dirty
#pragma unroll
  for (int k = 0; k < kRingCache; ++k) {
    if (lb[k] != lab) {
      boundary = true;
      if (!dirty && lb[k] != kNull && a.stamp[lb[k]] + 1 >= L) dirty = true;
    }
  }
  if (!is_short)
    for (int32_t k = a.row_ptr[i]; k < a.row_ptr[i + 1]; ++k) {
      const int32_t b = a.labels[a.col[k]];
      if (b != lab) {
        boundary = true;
        if (!dirty && b != kNull && a.stamp[b] + 1 >= L) dirty = true;
      }
    }
  return boundary && dirty;
}

// Control values of a mesh that the sweep kernels read per item.  In a context of
// one mesh (kB = false) they are read once, at the kernel's start, with its
// other first loads.
struct MeshCtl {
  int64_t item_off;
  uint32_t seed;
  int32_t metric, level;
  int32_t loops, connexity, constrained, mode, rounds;
};
__device__ inline MeshCtl load_mesh(const SweepArgs& a, int32_t m) {
  const DevMesh& dm = a.meshes[m];
  const MeshState& st = a.state[m];
  return MeshCtl{dm.item_off, dm.seed, dm.metric, dm.level, st.loops, st.connexity, st.constrained, qem_mode(st),
                 pass_rounds(st)};
}
template <bool kB>
struct MeshReader {
  const SweepArgs& a;
  MeshCtl one;
  __device__ explicit MeshReader(const SweepArgs& args) : a(args) {
    if constexpr (!kB) one = load_mesh(a, 0);
  }
  __device__ int32_t of_item(int64_t i) const { return kB ? mesh_of_item(a, i) : 0; }
  __device__ MeshCtl operator()(int32_t m) const {
    if constexpr (kB) return load_mesh(a, m);
    else return one;
  }
};

// Scan while the tile sets are off (nearly every tile holds a changed
// cluster): every item in id order, so that the item words and CSR rows are
// read in order.  Block b takes items [b * kBlock, (b + 1) * kBlock) and
// appends to work slice b % kWorkSlices (at most one tile's worth per block,
// within the slice capacity).  The evaluate's results do not depend on the
// order of the work list.  C3 torus: 139 -> 127 us per full scan.
__global__ __launch_bounds__(kBlock) void k_scan_linear(SweepArgs a) {
  __shared__ int32_t s_cnt[kBlock / 64], s_base;
  const int64_t i = int64_t(blockIdx.x) * kBlock + threadIdx.x;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  bool want = false;
  if (i < a.n_items) {
    const MeshState& st = a.state[mesh_of_item(a, i)];
    if (st.phase == kPhaseSweep) want = needs_eval_fast(a, i, a.labels[i], st.loops);
  }
  const unsigned long long bal = __ballot(want);
  if (lane == 0) s_cnt[w] = __popcll(bal);
  __syncthreads();
  if (threadIdx.x == 0) {
    int tot = 0;
    for (int k = 0; k < kBlock / 64; ++k) {
      const int c = s_cnt[k];
      s_cnt[k] = tot;
      tot += c;
    }
    s_base = tot ? atomicAdd(&a.work_count[blockIdx.x % kWorkSlices], tot) : 0;
  }
  __syncthreads();
  if (want) {
    const int32_t pos = s_base + s_cnt[w] + __popcll(bal & ((1ull << lane) - 1ull));
    a.work[int64_t(blockIdx.x % kWorkSlices) * a.work_cap + pos] = int32_t(i);
  }
}

// Scan: items of sweeping meshes that must be evaluated this pass are
// compacted into the work list (slice t % kWorkSlices of tile t).  One
// wavefront per tile: the lanes first test the tile's cluster set against the
// cluster stamps (and the tile's last proposal loop); only an active tile
// reads its items and CSR rows.  The test is conservative: every item
// needs_eval would select lies in an active tile.
// It runs while the tile sets are kept; before that k_scan_linear scans every
// item.
static_assert(kTileSet == 64, "k_scan: one set entry per lane");
__global__ __launch_bounds__(kBlock) void k_scan(SweepArgs a) {
  // one wavefront per tile, kTilesPerScanBlock tiles per block (the waves
  // are independent: no block-level synchronisation)
  const int32_t t = int32_t(blockIdx.x) * kTilesPerScanBlock + int32_t(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (t >= a.n_tiles) return;  // wave-uniform
  const int m = a.item_mesh ? a.tile_mesh[t] : 0;
  // the tile's count, last proposal and set entry of this lane (the set holds
  // kTileSet = 64 entries; entries past cnt are ignored) read with the state
  const int32_t cnt = a.tile_cnt[t];
  const int32_t prop = a.tile_prop[t];
  const int32_t c_lane = a.tile_set[int64_t(t) * kTileSet + lane];
  const MeshState& st = a.state[m];
  if (st.phase != kPhaseSweep) return;
  const int32_t L = st.loops;
  bool active = cnt > kTileSet || prop == L - 1;
  if (!active) {  // wave-uniform branch
    bool hit = false;
    if (lane < cnt) hit = a.stamp[c_lane] + 1 >= L;
    active = __ballot(hit) != 0ull;
  }
  if (!active) return;
  constexpr int R = kTileItems / 64;
  int32_t it[R];
  bool want[R];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    it[r] = a.tile_items[int64_t(t) * kTileItems + r * 64 + lane];
    want[r] = it[r] >= 0 && needs_eval_fast(a, it[r], a.labels[it[r]], L);
  }
  unsigned long long bal[R];
  int32_t tot = 0;
#pragma unroll
  for (int r = 0; r < R; ++r) {
    bal[r] = __ballot(want[r]);
    tot += __popcll(bal[r]);
  }
  if (tot == 0) return;
  const int slice = t % kWorkSlices;
  int32_t base = 0;
  if (lane == 0) base = atomicAdd(&a.work_count[slice], tot);
  base = __shfl(base, 0);
  const unsigned long long below = (1ull << lane) - 1ull;
  int32_t off = 0;
#pragma unroll
  for (int r = 0; r < R; ++r) {
    if (want[r]) a.work[int64_t(slice) * a.work_cap + base + off + __popcll(bal[r] & below)] = it[r];
    off += __popcll(bal[r]);
  }
}

// Cluster set of a tile, rebuilt from scratch: labels of its items and of
// their neighbours, gathered in an LDS hash table (linear probing, bounded).
__global__ __launch_bounds__(64) void k_tile_sets(SweepArgs a, const int32_t* __restrict__ mask) {
  constexpr int kTab = 256;
  constexpr int32_t kEmpty = -2;
  __shared__ int32_t tab[kTab];
  __shared__ int32_t n_uniq, overflow, n_out;
  const int32_t t = blockIdx.x;
  const int m = a.item_mesh ? a.tile_mesh[t] : 0;
  if (mask && !mask[m]) return;
  for (int k = threadIdx.x; k < kTab; k += 64) tab[k] = kEmpty;
  if (threadIdx.x == 0) {
    n_uniq = 0;
    overflow = 0;
    n_out = 0;
  }
  __syncthreads();
  auto insert = [&](int32_t c) {
    if (c == kNull) return;
    uint32_t h = (uint32_t(c) * 2654435761u) >> 24;  // top 8 bits
    for (int probe = 0; probe < kTab; ++probe) {
      const int32_t old = atomicCAS(&tab[h], kEmpty, c);
      if (old == kEmpty) {
        atomicAdd(&n_uniq, 1);
        return;
      }
      if (old == c) return;
      h = (h + 1) & (kTab - 1);
    }
    atomicOr(&overflow, 1);
  };
  for (int r = 0; r < kTileItems / 64; ++r) {
    const int32_t i = a.tile_items[int64_t(t) * kTileItems + r * 64 + threadIdx.x];
    if (i < 0) continue;
    insert(a.labels[i]);
    for (int32_t k = a.row_ptr[i]; k < a.row_ptr[i + 1]; ++k) insert(a.labels[a.col[k]]);
  }
  __syncthreads();
  const bool big = overflow || n_uniq > kTileSet;
  if (!big) {
    for (int k = threadIdx.x; k < kTab; k += 64) {
      const int32_t c = tab[k];
      if (c != kEmpty) a.tile_set[int64_t(t) * kTileSet + atomicAdd(&n_out, 1)] = c;
    }
    // the free slots hold a value no cluster id equals: tile_insert may read a
    // slot another insert has reserved but not written yet, and must not
    // mistake a stale id left there for its own cluster
    for (int k = threadIdx.x; k < kTileSet; k += 64)
      if (k >= n_uniq) a.tile_set[int64_t(t) * kTileSet + k] = kEmpty;
  }
  if (threadIdx.x == 0) a.tile_cnt[t] = big ? kTileSet + 1 : n_uniq;
}
// ------------------------------------------------------------------ propose
// Work slices: a scan tile appends its work items to slice t % kWorkSlices;
// many slices keep the same-address counter atomics few.  A consumer block
// maps a position of the concatenation to its entry with an LDS index of the
// slice starts.
struct WorkIndex {
  int32_t start[kWorkSlices + 1];
};

__device__ inline void load_work_index(const int32_t* counts, WorkIndex* wi) {
  constexpr int kPer = kWorkSlices / kBlock;
  static_assert(kWorkSlices % kBlock == 0, "work slices per thread");
  __shared__ int32_t s_wave[kBlock / 64];
  int32_t v[kPer];
  int32_t tot = 0;
  for (int k = 0; k < kPer; ++k) {
    v[k] = counts[threadIdx.x * kPer + k];
    tot += v[k];
  }
  // inclusive scan of the thread totals over the wave, then over the waves
  const int lane = __lane_id(), wv = threadIdx.x >> 6;
  int32_t inc = tot;
  for (int off = 1; off < 64; off <<= 1) {
    const int32_t u = __shfl_up(inc, off);
    if (lane >= off) inc += u;
  }
  if (lane == 63) s_wave[wv] = inc;
  __syncthreads();
  int32_t before = inc - tot;
  for (int w = 0; w < wv; ++w) before += s_wave[w];
  for (int k = 0; k < kPer; ++k) {
    wi->start[threadIdx.x * kPer + k] = before;
    before += v[k];
  }
  if (threadIdx.x == kBlock - 1) wi->start[kWorkSlices] = before;
  __syncthreads();
}

__device__ inline int32_t work_entry(const SweepArgs& a, const WorkIndex* wi, int32_t p) {
  int lo = 0, hi = kWorkSlices;  // slice k with start[k] <= p < start[k+1]
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (wi->start[mid] <= p) lo = mid;
    else hi = mid;
  }
  return a.work[int64_t(lo) * a.work_cap + (p - wi->start[lo])];
}

// Candidate segments seen as one list: an LDS index of the segment starts
// (prefix of the n_seg <= kMaxSeg fill counts), so that consumer blocks walk
// all candidates evenly whatever their segments.
struct SegIndex {
  int32_t start[kMaxSeg + 1];
};

__device__ inline void load_seg_index(const int32_t* counts, int32_t n_seg, SegIndex* si) {
  constexpr int kPer = kMaxSeg / kBlock;
  __shared__ int32_t s_wave[kBlock / 64];
  int32_t v[kPer];
  int32_t tot = 0;
  for (int k = 0; k < kPer; ++k) {
    const int32_t j = threadIdx.x * kPer + k;
    v[k] = j < n_seg ? counts[j] : 0;
    tot += v[k];
  }
  const int lane = __lane_id(), wv = threadIdx.x >> 6;
  int32_t inc = tot;
  for (int off = 1; off < 64; off <<= 1) {
    const int32_t u = __shfl_up(inc, off);
    if (lane >= off) inc += u;
  }
  if (lane == 63) s_wave[wv] = inc;
  __syncthreads();
  int32_t before = inc - tot;
  for (int w = 0; w < wv; ++w) before += s_wave[w];
  for (int k = 0; k < kPer; ++k) {
    si->start[threadIdx.x * kPer + k] = before;
    before += v[k];
  }
  if (threadIdx.x == kBlock - 1) si->start[kMaxSeg] = before;
  __syncthreads();
}

// Storage index (segment * cap + offset) of position p of the list.
__device__ inline int64_t seg_pos(const SegIndex* si, int32_t cap, int32_t p) {
  int lo = 0, hi = kMaxSeg;  // segment k with start[k] <= p < start[k+1]
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (si->start[mid] <= p) lo = mid;
    else hi = mid;
  }
  return int64_t(lo) * cap + (p - si->start[lo]);
}

// True (in every lane) when round r applied no move: the later rounds of the
// pass then apply nothing either and are skipped.  Every wave reads the counters
// itself, with its first loads: no barrier stands before the candidates.
__device__ inline bool round_was_empty(const SweepArgs& a, int r) {
  static_assert(kSlices == 64, "one slice per lane");
  return __ballot(a.ctrl->mods[r][__lane_id()] != 0) == 0ull;
}

// Metric of the meshes a kernel instantiation sweeps: 0 isotropic, 1 QEM,
// 2 QEM while unconstrained (isotropic rule, no FP64 solves compiled in).
constexpr int mesh_metric(int kernel_metric) { return kernel_metric == 2 ? 1 : kernel_metric; }

// Positions 0..n-1 of a list over the whole grid, one per thread and step (every
// thread of the block takes every step): for (base = w.first; base < n; base +=
// w.stride), thread position base + w.off when w.valid(base).  A list of fewer
// positions than kSpread blocks have threads is spread evenly over those blocks
// and their waves instead of filling the first ones: the step's time is its chain
// of loads and, for the QEM rule, the solves of its busiest wave.  One block per CU:
// over more of them a block's key table merges fewer keys and more blocks start.
// To convergence, not spread / 128 / 256 / 512 / 768 / 1152 blocks: QEM torus of
// 8.39M vertices 243.9 / 241.7 / 240.4 / 242.1 / 245.8 / 257.4 ms, of 260,533 32.9 /
// 32.3 / 31.6 / 32.4 / 33.0 / 35.4.
constexpr int32_t kSpread = 256;
struct EvenWalk {
  int32_t n, first, stride, off;
  bool mine;
  __device__ explicit EvenWalk(int32_t count) : n(count) {
    const int32_t grid = int32_t(gridDim.x);
    const int32_t blocks = grid < kSpread ? grid : kSpread;
    const bool full = n >= blocks * kBlock;  // block-uniform
    const int32_t per = full ? kBlock : (n + blocks - 1) / blocks;  // positions per block and step, then per wave
    const int32_t wave = (per + kBlock / 64 - 1) / (kBlock / 64);
    first = int32_t(blockIdx.x) * per;
    stride = full ? grid * kBlock : n;  // a spread list takes one step
    off = int32_t(threadIdx.x >> 6) * wave + __lane_id();
    mine = int32_t(__lane_id()) < wave && off < per;
  }
  __device__ bool valid(int32_t base) const { return mine && base + off < n; }
};

// Walks the candidate list, calling f(valid, entry) for one position per
// thread per step (every thread of the block takes part in every step).  A
// long list (last pass's proposals above kSegWalkMax) is walked evenly by all
// blocks through the LDS index; a short one by block b over segment b alone,
// which spares the index (grid = n_seg).  The results do not depend on the
// walk.
// Control values of the candidate walk, loaded by a kernel before its first
// barrier so that they share a memory round trip with its other first loads.
struct WalkCtl {
  bool by_seg;    // this pass walks one segment per block
  int32_t n_own;  // fill count of this block's segment
};
__device__ inline WalkCtl load_walk_ctl(const SweepArgs& a) {
  WalkCtl w;
  w.by_seg = a.ctrl->seg_walk != 0;
  w.n_own = a.seg_cand[blockIdx.x];
  return w;
}

// A candidate entry: item, its label (a live candidate has not moved), its live
// target (< 0: none) and the loop and round of its last evaluation.
struct CandRec {
  int32_t b, i, lab, since;
};
__device__ inline CandRec load_cand(const SweepArgs& a, int64_t e) {
  return CandRec{a.cand_tgt[e], a.cand[e], a.cand_lab[e], a.cand_since[e]};
}

// f(valid, entry, record); first: this thread's record of its block's segment,
// read by the kernel with its first loads (any value past the fill count).
template <class F>
__device__ inline void walk_candidates(const SweepArgs& a, const WalkCtl& w, SegIndex* si, const CandRec& first_rec,
                                       F&& f) {
  if (w.by_seg) {  // block-uniform
    const int64_t seg = int64_t(blockIdx.x) * a.cand_cap;
    for (int32_t base = 0; base < w.n_own; base += kBlock) {
      const int32_t k = base + int32_t(threadIdx.x);
      const bool valid = k < w.n_own;
      CandRec c = first_rec;
      if (base > 0 && valid) c = load_cand(a, seg + k);
      f(valid, seg + k, c);
    }
    return;
  }
  load_seg_index(a.seg_cand, a.n_seg, si);
  const EvenWalk ew(si->start[kMaxSeg]);
  for (int32_t base = ew.first; base < ew.n; base += ew.stride) {
    const bool valid = ew.valid(base);
    int64_t e = 0;
    CandRec c{-1, 0, kNull, 0};
    if (valid) {
      e = seg_pos(si, a.cand_cap, base + ew.off);
      c = load_cand(a, e);
    }
    f(valid, e, c);
  }
}

// Block-local minimum of the accept keys registered per cluster: an
// open-addressing table in LDS, flushed with one global atomicMin per distinct
// cluster.  Candidates of a block lie close together on the mesh and share
// few clusters, so this replaces most same-address global atomics.  The
// minimum does not depend on the order, so the keys are those of direct
// atomics.  A block registers at most 2 * kBlock keys between flushes, which
// keeps the table at most half full (every probe sequence ends).
constexpr int kKeyAggBits = 10;
constexpr int kKeyAggSlots = 1 << kKeyAggBits;
static_assert(2 * kBlock <= kKeyAggSlots / 2, "key table must stay at most half full");
struct KeyAgg {
  int32_t cl[kKeyAggSlots];
  unsigned long long key[kKeyAggSlots];
};

__device__ inline void keyagg_clear(KeyAgg* g) {
  for (int k = threadIdx.x; k < kKeyAggSlots; k += blockDim.x) {
    g->cl[k] = -1;
    g->key[k] = ~0ull;
  }
}

__device__ inline void keyagg_min(KeyAgg* g, int32_t c, unsigned long long key) {
  uint32_t h = (uint32_t(c) * 2654435761u) >> (32 - kKeyAggBits);
  while (true) {
    const int32_t prev = atomicCAS(&g->cl[h], -1, c);
    if (prev == -1 || prev == c) {
      atomicMin(&g->key[h], key);
      return;
    }
    h = (h + 1) & (kKeyAggSlots - 1);
  }
}

// Flushes the table to the global keys and clears it; all threads of the
// block call it (it synchronises the block before and after).
__device__ inline void keyagg_flush(KeyAgg* g, unsigned long long* prio) {
  __syncthreads();
  for (int k = threadIdx.x; k < kKeyAggSlots; k += blockDim.x) {
    const int32_t c = g->cl[k];
    if (c >= 0) {
      atomicMin(&prio[c], g->key[k]);
      g->cl[k] = -1;
      g->key[k] = ~0ull;
    }
  }
  __syncthreads();
}

// Wave-aggregated append of v to a block-owned list segment (fill count in
// LDS); every lane of the wave calls it.  Returns the entry index (when want).
__device__ inline int64_t seg_append(int64_t seg, int32_t* s_n, bool want) {
  const unsigned long long bal = __ballot(want);
  if (bal == 0ull) return -1;
  const int lane = __lane_id();
  const int leader = __ffsll((long long)bal) - 1;
  int32_t base = 0;
  if (lane == leader) base = atomicAdd(s_n, __popcll(bal));
  base = __shfl(base, leader);
  return want ? seg + base + __popcll(bal & ((1ull << lane) - 1ull)) : -1;
}

// ------------------------------------------------------ QEM solve pool (wave)
// The constrained QEM rule needs one FP64 solve for the item leaving its
// cluster and one per open target (qem_propose_short_row runs them one after
// the other in the item's lane).  Here the lanes of a wave put these solves
// into a shared pool and take them one per lane: a wave whose items need S
// solves in all runs ceil(S / 64) solve steps instead of as many as its
// busiest lane, and an item's solves run side by side.  The choice among the
// targets is the lexicographic minimum of (dE, cluster id), which does not
// depend on the order the solves finish in, so the move is the one of
// qem_propose_short_row.
constexpr int kPoolTasks = 64 * (1 + kRingCache);  // solves of one wave at most
struct QemPool {
  int32_t cl[kPoolTasks];     // target cluster, or ~a for the leave solve of cluster a
  uint8_t owner[kPoolTasks];  // lane of the item
  // results of one solve step (one per lane)
  float tb[64];   // join term of the target
  double Tn[64];  // T of the trial cluster
  double Tb[64];  // T of the target
};

// Orders the LDS accesses of the lanes of one wave (their DS operations
// execute in issue order; this keeps the compiler from moving them).
__device__ inline void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Wave-inclusive prefix sum of v.
__device__ inline int wave_prefix(int v) {
  const int lane = __lane_id();
  for (int off = 1; off < 64; off <<= 1) {
    const int u = __shfl_up(v, off);
    if (lane >= off) v += u;
  }
  return v;
}

// Owner kinds of the pool: a labelled item of a constrained QEM mesh whose
// screen passed, with a row of at most kRingCache neighbours (open targets in
// nb / open) or a longer one (open targets found again by walking the row).
enum PoolKind : int { kPoolNone = 0, kPoolShort = 1, kPoolLong = 2 };

// Screen of a labelled item with a long row for the pool: its kind (kPoolNone
// when no target is open) and its number of solves.
__device__ inline int pool_screen_long(const SweepView& v, int64_t i, int32_t lab, int connexity, QemItem* s,
                                       int* ntask) {
  *ntask = 0;
  if (!qem_screen(v, i, lab, connexity, 1, s)) return kPoolNone;
  int n = 1;
  for (int32_t k = qem_next_open(v, lab, *s, 1, s->r0 - 1); k < s->r1; k = qem_next_open(v, lab, *s, 1, k)) ++n;
  *ntask = n;
  return kPoolLong;
}

// Posts solves [j0, j1) of a long-row owner at pool index first (solve 0 is
// the leave, solve j > 0 the j-th open target in CSR order).
__device__ inline void pool_post_long(const SweepView& v, QemPool* pool, int64_t i, int32_t lab, int j0, int j1,
                                      int first) {
  QemItem s;
  qem_item_terms(v, i, lab, 1, &s);
  int32_t k = s.r0 - 1;
  for (int j = 1; j < j0; ++j) k = qem_next_open(v, lab, s, 1, k);
  for (int j = j0; j < j1; ++j) {
    int32_t c = ~lab;
    if (j > 0) {
      k = qem_next_open(v, lab, s, 1, k);
      c = k < s.r1 ? v.labels[v.col[k]] : ~lab;  // the state is frozen: the count of pool_screen_long holds
    }
    pool->cl[first + j - j0] = c;
    pool->owner[first + j - j0] = uint8_t(__lane_id());
  }
}

// Every lane of the wave calls it.  An owner (kind != kPoolNone, from
// its screen, mesh m) receives its item's move as qem_propose_short_row /
// the generic QEM rule would return it.  Short-row owners post all their
// solves first (a wave posts at most kPoolTasks of them), so that the lanes
// keep only the choice state across the solve steps; long-row owners post
// after them what fits and the rest in later fills.
template <bool kExtras, bool kB>
__device__ bool qem_pool_choose(const SweepArgs& a, const SweepView& v, QemPool* pool, int kind, int ntask,
                                int64_t i, int32_t lab, int32_t m, const int32_t* nb, const QemItem& s,
                                uint32_t open, int32_t* target_out) {
  const int lane = __lane_id();
  int first, total, post;
  {
    const int cs = kind == kPoolShort ? ntask : 0, cl = kind == kPoolLong ? ntask : 0;
    const int is = wave_prefix(cs), il = wave_prefix(cl);
    const int ts = __shfl(is, 63), tl = __shfl(il, 63);
    first = kind == kPoolShort ? is - cs : ts + il - cl;
    total = ts + tl < kPoolTasks ? ts + tl : kPoolTasks;
    post = total - first < ntask ? total - first : ntask;
    if (post < 0) post = 0;
  }
  if (kind == kPoolShort) {
    pool->cl[first] = ~lab;
    pool->owner[first] = uint8_t(lane);
    for (int j = 1; j < ntask; ++j) {
      pool->cl[first + j] = ring_label(nb, __builtin_ctz(open));
      pool->owner[first + j] = uint8_t(lane);
      open &= open - 1;
    }
  } else if (kind == kPoolLong && post > 0) {
    pool_post_long(v, pool, i, lab, 0, post, first);
  }
  const float pw = s.pw, ta = s.ta;
  const double Ta = s.Ta;
  double Ta_new = 0.0, best_d = 0.0, best_m = 0.0;
  int32_t target = kNull;
  int done = 0;
  while (total > 0) {
    wave_lds_sync();
    for (int base = 0; base < total; base += 64) {
      const bool solve = lane < total - base;
      const int ow = solve ? pool->owner[base + lane] : lane;
      const int64_t ti = __shfl(int32_t(i), ow);
      const int32_t tm = kB ? __shfl(m, ow) : 0;
      if (solve) {
        const int32_t tc = pool->cl[base + lane];
        const int32_t c = tc < 0 ? ~tc : tc;
        const DevMesh& dm = a.meshes[tm];
        const Scales sc = dm.scales;
        const AnchorPos an = kExtras ? anchor_pos(v, c) : AnchorPos{0.0, 0.0, 0.0, false};
        double Tn = 0.0;  // a centroid point (an unconstrained mesh's unanchored cluster)
        if (an.valid || a.state[tm].constrained) {
          int64_t iw, is[3], iq[10], ws[4], q10[10];
          item_fixed(v, ti, sc, &iw, is, iq);
          load_acc(v, c, ws, q10);
          Tn = qem_T_trial(ws, q10, iw, is, iq, tc < 0 ? -1 : 1, sc, dm.level, v.evec + 9 * int64_t(c), an);
        }
        pool->Tn[lane] = Tn;
        if (tc >= 0) {
          pool->tb[lane] =
              join_term(v.xw[4 * ti], v.xw[4 * ti + 1], v.xw[4 * ti + 2], v.xw[4 * ti + 3], v.geom[tc]);
          pool->Tb[lane] = v.T[tc];
        }
      }
      wave_lds_sync();
      // collect this lane's solves among pool entries [base, base + 64)
      const int j0 = first > base ? first : base;
      const int j1 = first + post < base + 64 ? first + post : base + 64;
      for (int j = j0; j < j1; ++j) {
        if (j - first + done == 0) {
          Ta_new = pool->Tn[j - base];
          continue;
        }
        const int32_t b = pool->cl[j];
        const float tb = pool->tb[j - base];
        const double Tb_new = pool->Tn[j - base], Tb = pool->Tb[j - base];
        const double d = qem_delta(pw, ta, tb, Ta_new, Ta, Tb_new, Tb);
        if (target == kNull || d < best_d || (d == best_d && b < target)) {
          best_d = d;
          best_m = qem_mag(pw, ta, tb, Ta_new, Ta, Tb_new, Tb);
          target = b;
        }
      }
      wave_lds_sync();
    }
    // next fill: long-row solves that did not fit
    done += post;
    const int rem = kind == kPoolLong ? ntask - done : 0;
    const int inc = wave_prefix(rem);
    const int tot = __shfl(inc, 63);
    first = inc - rem;
    total = tot < kPoolTasks ? tot : kPoolTasks;
    post = total - first < rem ? total - first : rem;
    if (post < 0) post = 0;
    if (post > 0) pool_post_long(v, pool, i, lab, done, done + post, first);
  }
  *target_out = target;
  return target != kNull && qem_accept(best_d, best_m);
}

// Adds one to counter(m) for every lane of the wave with `want`: one atomic per
// distinct mesh of the wave (its lanes mostly lie in one).  Every lane calls it.
template <class Counter>
__device__ inline void count_per_mesh(bool want, int32_t m, Counter&& counter) {
  unsigned long long todo = __ballot(want);
  while (todo) {
    const int leader = __ffsll((long long)todo) - 1;
    const int32_t m0 = __shfl(m, leader);
    const unsigned long long same = __ballot(want && m == m0);
    if (int(__lane_id()) == leader) atomicAdd(counter(m0), __popcll(same));
    todo &= ~same;
  }
}

// Evaluate (round 0) of item i (when valid): its best move (shared rules of
// acvd_math.h) against the state at the pass start; a proposal registers its
// round-0 accept key at both clusters and joins the block's candidate segment.
// Every lane of the block calls it (the QEM solve pool is shared by the wave).
// Bound by its chain of dependent loads: a short row's chain is item -> neighbour
// ids, label -> neighbour labels, own cluster -> neighbour clusters, each step's
// loads side by side (walked neighbour by neighbour it was three per neighbour).
template <int METRIC, bool kExtras, bool kB>
__device__ inline void eval_item(const SweepArgs& a, const SweepView& v, const MeshReader<kB>& mesh, QemPool* pool,
                                 KeyAgg* agg, bool direct, int64_t seg, int32_t* s_n, bool valid, int32_t i) {
  bool want = false;
  int32_t lab = kNull, target = kNull, m = 0;
  int32_t nb[kRingCache];
  MeshCtl mc{};
  QemItem s;
  uint32_t open = 0;
  int kind = kPoolNone, ntask = 0;
  if (valid) {
    m = mesh.of_item(i);
    mc = mesh(m);
    if (mc.metric == mesh_metric(METRIC)) {
      int32_t nbr[kRingCache];
      lab = a.labels[i];
      const bool is_short = load_row8(a, i, nbr);
      const float4 p = a.xw[i];
      const bool qem = METRIC == 1 && mc.mode != 0;
      if (lab != kNull && is_short) {
        ShortItem t{p.x, p.y, p.z, p.w, 0, a.sizes[lab], a.ring_adj[i], a.geom[lab]};
        const double Ta = qem ? a.T[lab] : 0.0;
        t.deg = load_labels8(a, nbr, nb);
        if (!qem) {  // no FP64 solve: the isotropic rule
          want = iso_propose_short(v, t, lab, mc.connexity, nb, &target);
        } else if (!is_anchor(v, i, lab) && qem_screen_short(v, t, lab, mc.connexity, Ta, 1, nb, &s, &open)) {
          kind = kPoolShort;
          ntask = 1 + __popc(open);
        }
      } else if (lab != kNull && qem) {
        kind = pool_screen_long(v, i, lab, mc.connexity, &s, &ntask);
      } else {  // the null-item rule, or the isotropic one over a long row
        want = propose_item<METRIC == 1 ? 2 : METRIC>(v, i, lab, mc.connexity, mc.constrained, mc.level,
                                                      a.meshes[m].scales, &target);
      }
    }
  }
  if constexpr (METRIC == 1) {
    int32_t pt = kNull;
    const bool r = qem_pool_choose<kExtras, kB>(a, v, pool, kind, ntask, i, lab, m, nb, s, open, &pt);
    if (kind != kPoolNone) {
      want = r;
      target = pt;
    }
  }
  if (want) {
    const unsigned long long key = accept_key(mc.seed, mc.loops, 0, uint32_t(i - mc.item_off));
    if (direct) {
      if (lab != kNull) atomicMin(&a.prio[lab], key);
      atomicMin(&a.prio[target], key);
    } else {
      if (lab != kNull) keyagg_min(agg, lab, key);
      keyagg_min(agg, target, key);
    }
    a.cand_pass[i] = mc.loops;
    a.tile_prop[a.item_tile[i]] = mc.loops;
  }
  if constexpr (kB) count_per_mesh(want, m, [&](int32_t mm) { return &a.state[mm].pass_props; });
  const int64_t e = seg_append(seg, s_n, want);
  if (want) {
    a.cand[e] = i;
    a.cand_lab[e] = lab;
    a.cand_tgt[e] = target;
    a.cand_since[e] = mc.loops * kMatchRounds;
  }
  if (!direct) keyagg_flush(agg, a.prio);
}

// Evaluate the work list of the scan.  Block b owns segment b (capacity
// cand_cap, count seg_cand[b]); the second launch of a mixed batch (append = 1)
// continues the segments of the first.
template <int METRIC, bool kExtras, bool kB>
__global__ __launch_bounds__(kBlock, METRIC == 1 ? 3 : 4) void k_eval(SweepArgs a, int append) {
  __shared__ WorkIndex wi;
  __shared__ KeyAgg agg;
  __shared__ QemPool pools[METRIC == 1 ? kBlock / 64 : 1];
  __shared__ int32_t s_n;
  const MeshReader<kB> mesh(a);
  if (threadIdx.x == 0) s_n = append ? a.seg_cand[blockIdx.x] : 0;
  keyagg_clear(&agg);
  load_work_index(a.work_count, &wi);
  const int32_t n = wi.start[kWorkSlices];
  const SweepView v = make_view<kExtras>(a);
  const int64_t seg = int64_t(blockIdx.x) * a.cand_cap;
  QemPool* pool = &pools[METRIC == 1 ? threadIdx.x >> 6 : 0];
  const bool direct = n <= kSegWalkMax && !a.crowded;  // few keys apart are not worth the table's barriers
  const EvenWalk ew(n);
  for (int32_t base = ew.first; base < n; base += ew.stride) {
    const bool valid = ew.valid(base);
    const int32_t i = valid ? work_entry(a, &wi, base + ew.off) : 0;
    eval_item<METRIC, kExtras, kB>(a, v, mesh, pool, &agg, direct, seg, &s_n, valid, i);
  }
  __syncthreads();
  if (threadIdx.x == 0) a.seg_cand[blockIdx.x] = s_n;
}

// Scan and evaluate in one launch, on contexts of at most kFusedItems items:
// block b takes the item blocks b, b + n_seg, ... , compacts the items to
// evaluate in LDS and evaluates them.  The work list, its index of slice starts
// and a launch go; what they give, an even share of the work items for every
// block, counts only where the blocks have more than a step or two of them.
// The keys go straight to the clusters (kTable: a crowded chunk): the LDS table's
// clearing, flush and barriers cost more than its merging saves here (2,562 items
// into 170 clusters to convergence 1.23 / 1.16 ms, 163,842 into 10,900 7.87 / 7.83).
template <int METRIC, bool kExtras, bool kB, bool kTable>
__global__ __launch_bounds__(kBlock, METRIC == 1 ? 3 : 4) void k_scan_eval(SweepArgs a, int append) {
  __shared__ KeyAgg agg;  // kTable
  __shared__ QemPool pools[METRIC == 1 ? kBlock / 64 : 1];
  __shared__ int32_t s_n, s_cnt[kBlock / 64], s_item[kBlock];
  const MeshReader<kB> mesh(a);
  if (kTable) keyagg_clear(&agg);  // made visible by the barriers of the first step
  if (threadIdx.x == 0) s_n = append ? a.seg_cand[blockIdx.x] : 0;
  const SweepView v = make_view<kExtras>(a);
  const int64_t seg = int64_t(blockIdx.x) * a.cand_cap;
  QemPool* pool = &pools[METRIC == 1 ? threadIdx.x >> 6 : 0];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  for (int64_t base = int64_t(blockIdx.x) * kBlock; base < a.n_items; base += int64_t(gridDim.x) * kBlock) {
    const int64_t i = base + threadIdx.x;
    bool want = false;
    if (i < a.n_items) {
      const int m = mesh_of_item(a, i);
      const MeshState& st = a.state[m];
      if (st.phase == kPhaseSweep && a.meshes[m].metric == mesh_metric(METRIC))
        want = needs_eval_fast(a, i, a.labels[i], st.loops);
    }
    const unsigned long long bal = __ballot(want);
    if (lane == 0) s_cnt[w] = __popcll(bal);
    __syncthreads();
    int32_t before = 0, n = 0;
    for (int k = 0; k < kBlock / 64; ++k) {
      if (k < w) before += s_cnt[k];
      n += s_cnt[k];
    }
    if (want) s_item[before + __popcll(bal & ((1ull << lane) - 1ull))] = int32_t(i);
    if (n && threadIdx.x == 0) atomicAdd(&a.work_count[blockIdx.x % kWorkSlices], n);  // items evaluated
    __syncthreads();
    if (n) {  // block-uniform
      // spread over the waves (EvenWalk)
      const int32_t per = (n + kBlock / 64 - 1) / (kBlock / 64);
      const int32_t off = w * per + lane;
      const bool valid = lane < per && off < n;
      eval_item<METRIC, kExtras, kB>(a, v, mesh, pool, kTable ? &agg : nullptr, !kTable, seg, &s_n, valid,
                                     valid ? s_item[off] : 0);
    }
  }
  __syncthreads();
  if (threadIdx.x == 0) a.seg_cand[blockIdx.x] = s_n;
}

// Block sum of v (the result is valid in thread 0; synchronises the block).
__device__ inline int block_sum(int v) {
  __shared__ int s_red[kBlock / 64];
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off);
  if (__lane_id() == 0) s_red[threadIdx.x / 64] = v;
  __syncthreads();
  int tot = 0;
  if (threadIdx.x == 0)
    for (int w = 0; w < kBlock / 64; ++w) tot += s_red[w];
  __syncthreads();
  return tot;  // valid in thread 0
}

// Re-evaluation of candidate entry e (record c, when valid) for round `round`;
// every lane of the wave calls it (the QEM solve pool is shared by the wave).
// reg(c, key) registers an accept key at cluster c.  Two candidates in three are
// stale, and the rounds wait on their chain of dependent loads: what a stale
// candidate reads of its item and cluster is read with the clusters' round tags,
// before it is known to be stale.
template <int METRIC, bool kExtras, bool kB, bool kCount, class Reg>
__device__ inline void reeval_entry(const SweepArgs& a, const SweepView& v, const MeshReader<kB>& mesh, QemPool* pool,
                                    bool valid, int64_t e, const CandRec& c, int round, Reg&& reg, int* n_live,
                                    int* n_stale, int* n_recheck) {
  const int32_t b = valid ? c.b : -1;
  bool live = false, stale = false, use_pool = false, recheck = false;
  int32_t i = 0, lab = kNull, target = b, m = 0;
  unsigned long long key = 0;
  int32_t nb[kRingCache];
  QemItem s;
  uint32_t open = 0;
  int kind = kPoolNone, ntask = 0;
  if (b >= 0) {
    i = c.i;
    lab = c.lab;
    m = mesh.of_item(i);
    const MeshCtl mc = mesh(m);
    // a mesh past its last round of the pass registers nothing (no move); a
    // context of one mesh has left the kernel already
    if (mc.metric == mesh_metric(METRIC) && (!kB || round < mc.rounds)) {
      const bool qem = METRIC == 1 && mc.mode != 0;
      const int32_t ra = lab != kNull ? a.cl_round[lab] : -1, rb = a.cl_round[b];
      int32_t nbr[kRingCache];
      const bool is_short = load_row8(a, i, nbr);
      const float4 p = a.xw[i];
      const int32_t la = lab != kNull ? lab : b;
      ShortItem t{p.x, p.y, p.z, p.w, 0, a.sizes[la], a.ring_adj[i], a.geom[la]};
      ClusterGeom gb{0.0, 0.0, 0.0, 0.0};
      double Ta = 0.0;
      if (METRIC == 1) Ta = a.T[la];
      else gb = a.geom[b];
      stale = ra >= c.since || rb >= c.since;
      key = accept_key(mc.seed, mc.loops, round, uint32_t(i - mc.item_off));
      live = true;
      if (stale) {
        a.cand_since[e] = mc.loops * kMatchRounds + round;
        target = kNull;
        use_pool = qem && lab != kNull;
        if (lab != kNull && is_short) {
          t.deg = load_labels8(a, nbr, nb);
          if (qem) {
            if (!is_anchor(v, i, lab) && qem_screen_short(v, t, lab, mc.connexity, Ta, 1, nb, &s, &open)) {
              kind = kPoolShort;
              ntask = 1 + __popc(open);
            }
          } else {  // the isotropic rule: the move itself is checked again
            if (METRIC == 1) gb = a.geom[b];
            target = b;
            recheck = true;
            live = iso_recheck_short(v, t, lab, b, mc.connexity, nb, gb);
          }
        } else if (use_pool) {
          kind = pool_screen_long(v, i, lab, mc.connexity, &s, &ntask);
        } else if (lab != kNull) {
          target = b;
          recheck = true;
          live = iso_recheck(v, i, lab, b, mc.connexity);
        } else {  // the null-item rule
          live = propose_item<METRIC == 1 ? 2 : METRIC>(v, i, lab, mc.connexity, mc.constrained, mc.level,
                                                        a.meshes[m].scales, &target);
        }
      }
    }
  }
  if constexpr (METRIC == 1) {
    int32_t pt = kNull;
    const bool r = qem_pool_choose<kExtras, kB>(a, v, pool, kind, ntask, i, lab, m, nb, s, open, &pt);
    if (use_pool) {
      live = r;
      target = pt;
    }
  }
  if (stale) a.cand_tgt[e] = live ? target : -3;
  if (live) {
    if (lab != kNull) reg(lab, key);
    reg(target, key);
  }
  if constexpr (kCount) {
    *n_live += live;
    *n_stale += stale && !recheck;
    *n_recheck += recheck;
  }
}

// Measured and left out: 4 waves per SIMD for the QEM kernels (128 registers):
// 237.3 against 236.7 ms on the 8.39M-vertex torus; the item read only once it is
// known to be stale in long lists: 238.1; a look at the global key before the
// table's atomicMin: 255.4 (it costs what the atomic does).
//
// Re-evaluate (round r > 0): a live candidate (cand_tgt >= 0) whose own
// cluster or target moved since its last evaluation is evaluated again
// against the state left by round r-1: it registers its round-r key with its
// (possibly new) target or is dropped (-3).  The others keep their move, whose
// dE depends only on the two unchanged clusters, and register it again.
// A short list (one segment per block) registers straight at the global keys
// (kTable, a crowded chunk: not): its few keys are not worth the LDS table's barriers.
// kCount: count the registered and re-evaluated candidates (timed runs).
template <int METRIC, bool kExtras, bool kB, bool kCount, bool kTable>
__global__ __launch_bounds__(kBlock, METRIC == 1 ? 3 : 4) void k_reeval(SweepArgs a, int round) {
  __shared__ KeyAgg agg;
  __shared__ SegIndex si;
  __shared__ QemPool pools[METRIC == 1 ? kBlock / 64 : 1];
  const WalkCtl w = load_walk_ctl(a);
  const CandRec rec = load_cand(a, int64_t(blockIdx.x) * a.cand_cap + threadIdx.x);
  const MeshReader<kB> mesh(a);
  const bool empty = round_was_empty(a, round - 1);
  if (empty || (!kB && round >= mesh.one.rounds)) return;
  const SweepView v = make_view<kExtras>(a);
  QemPool* pool = &pools[METRIC == 1 ? threadIdx.x >> 6 : 0];
  int n_live = 0, n_stale = 0, n_recheck = 0;
  if (kTable || !w.by_seg) keyagg_clear(&agg);  // made visible by the index's barrier
  if (kTable && w.by_seg) __syncthreads();      // (without an index by this one)
  walk_candidates(a, w, &si, rec, [&](bool valid, int64_t e, const CandRec& c) {
    reeval_entry<METRIC, kExtras, kB, kCount>(
        a, v, mesh, pool, valid, e, c, round,
        [&](int32_t cl, unsigned long long key) {
          if (!kTable && w.by_seg) atomicMin(&a.prio[cl], key);
          else keyagg_min(&agg, cl, key);
        },
        &n_live, &n_stale, &n_recheck);
    if (kTable || !w.by_seg) keyagg_flush(&agg, a.prio);
  });
  // candidates registered and re-evaluated in this round (statistics of the
  // timed runs: the block sums cost a few barriers per round)
  if constexpr (kCount) {
    const int tl = block_sum(n_live);
    const int ts = block_sum(n_stale);
    const int tr = block_sum(n_recheck);
    if (threadIdx.x == 0) {
      if (tl) atomicAdd(&a.ctrl->live[round][blockIdx.x % kSlices], tl);
      if (ts) atomicAdd(&a.ctrl->stale[round][blockIdx.x % kSlices], ts);
      if (tr) atomicAdd(&a.ctrl->recheck[round][blockIdx.x % kSlices], tr);
    }
  }
}

// --------------------------------------------------------------------- apply
// Adds cluster c to the set of tile t unless present (sets only grow between
// rebuilds; duplicates from concurrent inserts only use capacity).
__device__ inline void tile_insert(const SweepArgs& a, int32_t t, int32_t c) {
  // the count and all set entries read at once (16-byte loads; the set holds
  // kTileSet entries), entries past cnt ignored
  const int32_t cnt = a.tile_cnt[t];
  const int4* set4 = reinterpret_cast<const int4*>(a.tile_set + int64_t(t) * kTileSet);
  int4 sv[kTileSet / 4];
#pragma unroll
  for (int q = 0; q < kTileSet / 4; ++q) sv[q] = set4[q];
  if (cnt > kTileSet) return;
  bool found = false;
#pragma unroll
  for (int q = 0; q < kTileSet / 4; ++q) {
    const int4 v = sv[q];
    found |= (4 * q < cnt && v.x == c) || (4 * q + 1 < cnt && v.y == c) || (4 * q + 2 < cnt && v.z == c) ||
             (4 * q + 3 < cnt && v.w == c);
  }
  if (found) return;
  const int32_t slot = atomicAdd(&a.tile_cnt[t], 1);
  if (slot < kTileSet) a.tile_set[int64_t(t) * kTileSet + slot] = c;
}


// Apply round `round`: a live candidate holding the minimum round key at both
// of its clusters moves: label, fixed-point accumulator deltas (plain
// read-modify-write: the round owns both clusters), sizes and stamps; then the
// centroid, W and (QEM) T of both clusters are derived from their final
// accumulators (the round's only writer of them).  The blocks walk all
// candidates evenly; the item joins its block's moved segment (tile sets are
// extended by k_tile_update after the pass).
//  kSolve = false (no mesh constrained): a derive is a centroid, computed by
//    the mover itself;
//  kSolve = true: a derive may need an FP64 solve; the clusters the movers of
//    a wave modified are listed in LDS and derived one per lane.
struct DeriveList {
  int32_t cl[2 * 64];
};

// Apply of candidate entry e (when valid) in round `round`; every lane of the
// wave calls it.  Returns true when the candidate moved (item *moved_item).
template <bool kSolve, bool kExtras, bool kB>
__device__ inline bool apply_entry(const SweepArgs& a, const MeshReader<kB>& mesh, DeriveList* dl, bool valid,
                                   int64_t e, const CandRec& c, int round, int32_t* moved_item) {
  bool win = false;
  int64_t i = 0;
  int32_t lab = kNull;
  const int32_t b = valid ? c.b : -1;
  int32_t m = 0;
  if (b >= 0) {
    i = c.i;
    lab = c.lab;
    m = mesh.of_item(i);
    const MeshCtl mc = mesh(m);
    const int32_t L = mc.loops;
    const DevMesh& dm = a.meshes[m];
    const unsigned long long key = accept_key(mc.seed, L, round, uint32_t(i - mc.item_off));
    const unsigned long long pa = lab != kNull ? a.prio[lab] : key, pb = a.prio[b];
    win = pa == key && pb == key;
    if (win) {
      // exclusive owner of clusters lab and b for this round
      a.labels[i] = b;
      a.cand_tgt[e] = -3;
      const float4 p = a.xw[i];
      const Scales sc = dm.scales;
      const unsigned long long iw = (unsigned long long)fix_w(p.w, sc);
      const unsigned long long is[3] = {(unsigned long long)fix_s(p.w, p.x, sc),
                                        (unsigned long long)fix_s(p.w, p.y, sc),
                                        (unsigned long long)fix_s(p.w, p.z, sc)};
      const int32_t rtag = L * kMatchRounds + round;
      if (lab != kNull) {
        unsigned long long* wa = a.acc_ws + 4 * int64_t(lab);
        wa[0] -= iw;
        for (int q = 0; q < 3; ++q) wa[1 + q] -= is[q];
        a.sizes[lab] -= 1;
        a.stamp[lab] = L;
        a.cl_round[lab] = rtag;
      }
      unsigned long long* wb = a.acc_ws + 4 * int64_t(b);
      wb[0] += iw;
      for (int q = 0; q < 3; ++q) wb[1 + q] += is[q];
      // quadric accumulators: while no mesh is constrained (kSolve = false)
      // nothing reads them, and the recompute at the convergence that
      // constrains a mesh rebuilds them from the labels
      if (kSolve && dm.metric == 1) {
        unsigned long long* qa = lab != kNull ? a.acc_q + 10 * int64_t(lab) : nullptr;
        unsigned long long* qb = a.acc_q + 10 * int64_t(b);
        for (int q = 0; q < 10; ++q) {
          const unsigned long long iq = (unsigned long long)fix_q(a.q[10 * i + q], sc);
          if (qa) qa[q] -= iq;
          qb[q] += iq;
        }
      }
      a.sizes[b] += 1;
      a.stamp[b] = L;
      a.cl_round[b] = rtag;
      if (!kSolve) {
        if (lab != kNull) derive_cluster<kExtras>(a, lab, dm, 0, false);
        derive_cluster<kExtras>(a, b, dm, 0, false);
      }
    }
  }
  if constexpr (kB) count_per_mesh(win, m, [&](int32_t mm) { return &a.state[mm].pass_mods; });
  if constexpr (kSolve) {
    const int cnt = win ? (lab != kNull ? 2 : 1) : 0;
    const int inc = wave_prefix(cnt);
    const int total = __shfl(inc, 63);
    if (cnt) {
      dl->cl[inc - cnt] = b;
      if (cnt == 2) dl->cl[inc - 1] = lab;
    }
    // the movers' accumulator stores before the other lanes' loads (one
    // CU: workgroup scope orders them through its L1)
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
    for (int k = __lane_id(); k < total; k += 64) {
      const int64_t c = dl->cl[k];
      const int mm = kB ? mesh_of_cluster(a, c) : 0;
      derive_cluster<kExtras>(a, c, a.meshes[mm], mesh(mm).constrained, true);
    }
    wave_lds_sync();
  }
  *moved_item = int32_t(i);
  return win;
}

// Apply of a short list (one segment per block) whose derives may need a solve:
// two lanes per candidate, one for the cluster it leaves (side 0) and one for the
// cluster it joins.  Each lane updates and derives its own cluster from registers:
// no accumulator store is waited for and read back, and what a winner needs is
// read with the keys that say whether it wins (a short list's losers cost little).
// Returns true on both lanes of a candidate that moves.
template <bool kExtras, bool kB>
__device__ inline bool apply_pair(const SweepArgs& a, const MeshReader<kB>& mesh, bool valid, int64_t e,
                                  const CandRec& rec, int round) {
  const int side = threadIdx.x & 1;
  const bool live = valid && rec.b >= 0;
  const int32_t c = side ? rec.b : rec.lab;
  const bool has = live && c != kNull;
  bool ok = live;
  int32_t m = 0, size = 0;
  MeshCtl mc{};
  float4 p = make_float4(0.f, 0.f, 0.f, 0.f);
  float q[10];
  unsigned long long ws[4], q10[10];
  double V0[9];
  if (live) {
    m = mesh.of_item(rec.i);
    mc = mesh(m);
  }
  if (has) {
    const unsigned long long key = a.prio[c];
    size = a.sizes[c];
    p = a.xw[rec.i];
    for (int k = 0; k < 4; ++k) ws[k] = a.acc_ws[4 * int64_t(c) + k];
    if (mc.metric == 1) {
      for (int k = 0; k < 10; ++k) q[k] = a.q[10 * int64_t(rec.i) + k];
      for (int k = 0; k < 10; ++k) q10[k] = a.acc_q[10 * int64_t(c) + k];
      for (int k = 0; k < 9; ++k) V0[k] = a.evec[9 * int64_t(c) + k];
    }
    ok = key == accept_key(mc.seed, mc.loops, round, uint32_t(rec.i - mc.item_off));
  }
  const bool other = __shfl_xor(int(ok), 1) != 0;  // every lane takes part
  const bool win = live && ok && other;
  if (win && side) {
    a.labels[rec.i] = rec.b;
    a.cand_tgt[e] = -3;
  }
  if (win && has) {  // exclusive owner of cluster c for this round
    const DevMesh& dm = a.meshes[m];
    const Scales sc = dm.scales;
    const unsigned long long d[4] = {(unsigned long long)fix_w(p.w, sc), (unsigned long long)fix_s(p.w, p.x, sc),
                                     (unsigned long long)fix_s(p.w, p.y, sc), (unsigned long long)fix_s(p.w, p.z, sc)};
    for (int k = 0; k < 4; ++k) {
      ws[k] = side ? ws[k] + d[k] : ws[k] - d[k];
      a.acc_ws[4 * int64_t(c) + k] = ws[k];
    }
    a.sizes[c] = side ? size + 1 : size - 1;
    a.stamp[c] = mc.loops;
    a.cl_round[c] = mc.loops * kMatchRounds + round;
    const ClusterGeom g = geom_from_fixed(int64_t(ws[0]), int64_t(ws[1]), int64_t(ws[2]), int64_t(ws[3]), sc);
    a.geom[c] = g;
    if (mc.metric == 1) {
      int64_t Q[10];
      for (int k = 0; k < 10; ++k) {
        const unsigned long long iq = (unsigned long long)fix_q(q[k], sc);
        q10[k] = side ? q10[k] + iq : q10[k] - iq;
        a.acc_q[10 * int64_t(c) + k] = q10[k];
        Q[k] = int64_t(q10[k]);
      }
      double T = 0.0;
      const int32_t an = (kExtras && a.anchor) ? a.anchor[c] : -1;
      if (an >= 0) {
        const float4 x = a.xw[an];
        T = anchored_T(g, AnchorPos{double(x.x), double(x.y), double(x.z), true});
      } else if (mc.constrained) {
        T = qem_T_from_fixed(Q, g, sc, dm.level, nullptr, V0, a.evec + 9 * int64_t(c));
      }
      a.T[c] = T;
    }
  }
  if constexpr (kB) count_per_mesh(win && side, m, [&](int32_t mm) { return &a.state[mm].pass_mods; });
  return win;
}

template <bool kSolve, bool kExtras, bool kB>
__global__ __launch_bounds__(kBlock, kSolve ? 3 : 4) void k_apply(SweepArgs a, int round) {
  __shared__ int32_t s_moved;
  __shared__ SegIndex si;
  __shared__ DeriveList dlist[kSolve ? kBlock / 64 : 1];
  const int64_t mseg = int64_t(blockIdx.x) * a.cand_cap;
  const WalkCtl w = load_walk_ctl(a);
  const CandRec rec = load_cand(a, mseg + (kSolve ? threadIdx.x >> 1 : threadIdx.x));
  const MeshReader<kB> mesh(a);
  const int32_t moved0 = round == 0 ? 0 : a.seg_moved[blockIdx.x];
  const bool empty = round > 0 && round_was_empty(a, round - 1);
  if (empty || (!kB && round >= mesh.one.rounds)) return;
  if (threadIdx.x == 0) s_moved = moved0;
  __syncthreads();
  DeriveList* dl = &dlist[kSolve ? threadIdx.x >> 6 : 0];
  int mods = 0;
  if (kSolve && w.by_seg) {  // block-uniform
    for (int32_t base = 0; base < w.n_own; base += kBlock / 2) {
      const int32_t k = base + int32_t(threadIdx.x >> 1);
      const bool valid = k < w.n_own;
      CandRec c = rec;
      if (base > 0 && valid) c = load_cand(a, mseg + k);
      const bool won = apply_pair<kExtras, kB>(a, mesh, valid, mseg + k, c, round) && (threadIdx.x & 1);
      mods += won;
      const int64_t em = seg_append(mseg, &s_moved, won);
      if (em >= 0) a.moved[em] = c.i;
    }
  } else {
    walk_candidates(a, w, &si, rec, [&](bool valid, int64_t e, const CandRec& c) {
      int32_t i;
      const bool win = apply_entry<kSolve, kExtras, kB>(a, mesh, dl, valid, e, c, round, &i);
      mods += win;
      const int64_t em = seg_append(mseg, &s_moved, win);
      if (em >= 0) a.moved[em] = i;
    });
  }
  const int tm = block_sum(mods);  // synchronises the block
  if (threadIdx.x == 0) {
    a.seg_moved[blockIdx.x] = s_moved;
    if (tm) atomicAdd(&a.ctrl->mods[round][blockIdx.x % kSlices], tm);
  }
}

// Tile sets after a pass: an item that moved to cluster b shows b to its own
// tile and to the tiles of its neighbours (k_scan of the next pass reads them).
__global__ __launch_bounds__(kBlock) void k_tile_update(SweepArgs a) {
  const int32_t n = a.seg_moved[blockIdx.x];
  const int64_t seg = int64_t(blockIdx.x) * a.cand_cap;
  for (int32_t k = threadIdx.x; k < n; k += kBlock) {
    const int64_t i = a.moved[seg + k];
    const int32_t b = a.labels[i];
    const int32_t ti = a.item_tile[i];
    const int32_t r0 = a.row_ptr[i], r1 = a.row_ptr[i + 1];
    // the tiles of the first kRingCache neighbours read at once; each distinct
    // tile other than the item's gets one insert
    int32_t tj[kRingCache];
    ACVD_UNROLL
    for (int p = 0; p < kRingCache; ++p) tj[p] = r0 + p < r1 ? a.item_tile[a.col[r0 + p]] : ti;
    tile_insert(a, ti, b);
    ACVD_UNROLL
    for (int p = 0; p < kRingCache; ++p) {
      bool first = tj[p] != ti;
      ACVD_UNROLL
      for (int q = 0; q < p; ++q) first = first && tj[q] != tj[p];
      if (first) tile_insert(a, tj[p], b);
    }
    for (int32_t r = r0 + kRingCache; r < r1; ++r) {
      const int32_t t = a.item_tile[a.col[r]];
      if (t != ti) tile_insert(a, t, b);
    }
  }
}

// ---------------------------------------------------------------- controller
// One block after every pass: the pass's counts, then each sweeping mesh's phase
// logic.  Bound by its dependent loads (7 us of every pass, whatever its work):
// the state and the control words are read with the counters, and a context of
// one mesh is stepped from registers (5.1 -> 3.7 us on an icosphere of 2,562).
__global__ __launch_bounds__(kBlock) void k_controller(SweepArgs a) {
  __shared__ int any_sweep, any_clean;
  __shared__ int s_part[2][kBlock / 64], s_round_mods[kMatchRounds], s_count[3];
  __shared__ int s_flags;   // phase flags of mesh 0 during this pass
  __shared__ int s_rounds;  // most accept rounds a sweeping mesh ran this pass
  static_assert(kSlices == 64, "one wave sums the slice counters");
  Ctrl* ctrl = a.ctrl;
  MeshState s0{};
  unsigned long long c_eval = 0, c_prop = 0, c_acc = 0, c_accq = 0, c_pass = 0, c_rounds = 0, c_walked = 0;
  if (threadIdx.x == 0) {
    s0 = a.state[0];
    c_eval = ctrl->evaluated;
    c_prop = ctrl->proposed;
    c_acc = ctrl->accepted;
    c_accq = ctrl->accepted_constrained;
    c_pass = ctrl->passes;
    c_rounds = ctrl->rounds;
    c_walked = ctrl->walked;
    any_sweep = 0;
    any_clean = 0;
    s_rounds = 1;
    s_count[0] = s_count[1] = s_count[2] = 0;
  }
  {  // items evaluated and proposals of the pass: sums over the work slices
     // (cleared for the next scan) and the candidate segments
    int w = 0, p = 0;
    int wv[kWorkSlices / kBlock];
#pragma unroll
    for (int k = 0; k < kWorkSlices / kBlock; ++k) wv[k] = a.work_count[k * kBlock + threadIdx.x];
    for (int k = threadIdx.x; k < a.n_seg; k += kBlock) p += a.seg_cand[k];
#pragma unroll
    for (int k = 0; k < kWorkSlices / kBlock; ++k) {
      w += wv[k];
      if (wv[k]) a.work_count[k * kBlock + threadIdx.x] = 0;
    }
    for (int off = 32; off > 0; off >>= 1) {
      w += __shfl_xor(w, off);
      p += __shfl_xor(p, off);
    }
    if (__lane_id() == 0) {
      s_part[0][threadIdx.x >> 6] = w;
      s_part[1][threadIdx.x >> 6] = p;
    }
  }
  // wave k sums the move counters of rounds k, k + 4, ... (lane l reads slice l)
  {
    constexpr int kPer = kMatchRounds / (kBlock / 64);
    static_assert(kMatchRounds % (kBlock / 64) == 0, "rounds per wave");
    const int w = threadIdx.x >> 6, lane = __lane_id();
    int dr[kPer];
#pragma unroll
    for (int k = 0; k < kPer; ++k) dr[k] = ctrl->mods[w + k * (kBlock / 64)][lane];
#pragma unroll
    for (int k = 0; k < kPer; ++k) {
      if (dr[k]) ctrl->mods[w + k * (kBlock / 64)][lane] = 0;
      for (int off = 32; off > 0; off >>= 1) dr[k] += __shfl_xor(dr[k], off);
      if (lane == 0) s_round_mods[w + k * (kBlock / 64)] = dr[k];
    }
  }
  __syncthreads();
  if (a.count_rounds) {  // timed runs: the registered, re-evaluated and re-checked candidates
    int v[3] = {0, 0, 0};
    for (int k = threadIdx.x; k < kMatchRounds * kSlices; k += kBlock) {
      v[0] += ctrl->live[0][k];
      v[1] += ctrl->stale[0][k];
      v[2] += ctrl->recheck[0][k];
      ctrl->live[0][k] = 0;
      ctrl->stale[0][k] = 0;
      ctrl->recheck[0][k] = 0;
    }
    for (int j = 0; j < 3; ++j)
      if (v[j]) atomicAdd(&s_count[j], v[j]);
  }
  int work = 0, props = 0, mods = 0;
  for (int k = 0; k < kBlock / 64; ++k) {
    work += s_part[0][k];
    props += s_part[1][k];
  }
  for (int r = 0; r < kMatchRounds; ++r) mods += s_round_mods[r];
  for (int m = threadIdx.x; m < a.n_meshes; m += kBlock) {
    MeshState s = m == 0 ? s0 : a.state[m];
    if (m == 0) s_flags = (s.constrained ? 1 : 0) | (s.connexity ? 2 : 0);
    if (s.phase == kPhaseSweep) {
      atomicMax(&s_rounds, pass_rounds(s));
      atomicOr(&any_sweep, 2);
      if (!a.item_mesh) {  // one mesh: the sliced counters are its own
        s.pass_props = props;
        s.pass_mods = mods;
      }
      if (s.pass_props > kCrowdedProps * (a.item_mesh ? int64_t(a.meshes[m].K) : a.n_clusters)) atomicOr(&any_sweep, 4);
      controller_step(s);
      a.state[m] = s;
    }
    if (s.phase == kPhaseSweep) atomicOr(&any_sweep, 1);
    if (s.phase == kPhaseNeedClean) atomicOr(&any_clean, 1);
  }
  __syncthreads();
  if (threadIdx.x != 0) return;
  const bool ran = any_sweep & 2;
  ctrl->evaluated = c_eval + (unsigned long long)work;
  ctrl->proposed = c_prop + (unsigned long long)props;
  ctrl->accepted = c_acc + (unsigned long long)mods;
  if (s_flags & 1) ctrl->accepted_constrained = c_accq + (unsigned long long)mods;
  if (ran) {
    int32_t* e = ctrl->pass_log[c_pass % kPassLogCap];
    e[0] = int32_t(c_pass);
    e[1] = work;
    e[2] = props;
    e[3] = mods;
    for (int r = 0; r < kMatchRounds; ++r) e[4 + r] = s_round_mods[r];
    e[4 + kMatchRounds] = s_flags;
    // accept rounds that walked the candidate list: round 0, and each later
    // round whose predecessor applied a move (a round after one without moves
    // exits at once); the re-evaluate kernels walked the list in all but one
    int walked = 1;
    while (walked < s_rounds && s_round_mods[walked - 1] > 0) ++walked;
    ctrl->rounds = c_rounds + (unsigned long long)walked;
    ctrl->walked = c_walked + (unsigned long long)props * (unsigned long long)(2 * walked - 1);
    if (a.count_rounds) {
      ctrl->reeval_live += (unsigned long long)s_count[0];
      ctrl->reevaluated += (unsigned long long)s_count[1];
      ctrl->rechecked += (unsigned long long)s_count[2];
    }
    ctrl->passes = c_pass + 1;
  }
  ctrl->any_sweep = any_sweep & 1;
  ctrl->seg_walk = props <= kSegWalkMax ? 1 : 0;
  ctrl->crowded = any_sweep & 4 ? 1 : 0;
  ctrl->any_need_clean = any_clean;
}

// ---------------------------------------------------------------------- fill
// One synchronous round: every null item with a labelled neighbour takes the
// label of its lowest-id labelled neighbour (as of the start of the round).
__global__ void k_fill_pick(SweepArgs a, const int32_t* __restrict__ mask, int32_t* pending) {
  int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  bool changed = false;
  if (i < a.n_items && mask[mesh_of_item(a, i)] && a.labels[i] == kNull) {
    int32_t pick = kNull;
    for (int32_t k = a.row_ptr[i]; k < a.row_ptr[i + 1]; ++k) {
      const int32_t b = a.labels[a.col[k]];
      if (b != kNull) {
        pick = b;
        break;
      }
    }
    pending[i] = pick;
    changed = pick != kNull;
  }
  if (__ballot(changed) != 0 && __lane_id() == 0) a.ctrl->fill_changed = 1;
}

__global__ void k_fill_commit(SweepArgs a, const int32_t* __restrict__ mask, const int32_t* __restrict__ pending) {
  int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= a.n_items || !mask[mesh_of_item(a, i)] || a.labels[i] != kNull) return;
  a.labels[i] = pending[i];
}

// --------------------------------------------------- connected components
// Union-find over same-label edges; a root is always the smallest item id of
// its tree (larger roots are hooked under smaller ones), so the final
// representative of a component is its minimum item id.
__device__ int32_t cc_find(int32_t* parent, int32_t x) {
  while (true) {
    int32_t p = parent[x];
    if (p == x) return x;
    int32_t gp = parent[p];
    if (gp != p) parent[x] = gp;  // path halving (benign race: ancestors only)
    x = gp;
  }
}

// f(j) for every neighbour j of item i.
template <class F>
__device__ inline void for_each_neighbour(const SweepArgs& a, int64_t i, F&& f) {
  int32_t nbr[kRingCache];
  if (load_row8(a, i, nbr)) {
#pragma unroll
    for (int p = 0; p < kRingCache; ++p)
      if (nbr[p] >= 0) f(nbr[p]);
  } else {
    for (int32_t k = a.row_ptr[i]; k < a.row_ptr[i + 1]; ++k) f(a.col[k]);
  }
}

// Every item starts below its smallest neighbour of the same label, so that most
// of a component is one tree before the first compare-and-swap.
__global__ void k_cc_init(SweepArgs a, const int32_t* __restrict__ mask, int32_t* parent, int32_t* comp_size) {
  int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= a.n_items || !mask[mesh_of_item(a, i)]) return;
  const int32_t lab = a.labels[i];
  int32_t low = int32_t(i);
  if (lab != kNull)
    for_each_neighbour(a, i, [&](int32_t j) {
      if (j < low && a.labels[j] == lab) low = j;
    });
  parent[i] = low;
  comp_size[i] = 0;
}

// Every item straight below the root of its tree, so that the ends of most edges
// show the same root at the first look.
__global__ void k_cc_flatten(SweepArgs a, const int32_t* __restrict__ mask, int32_t* parent) {
  int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= a.n_items || !mask[mesh_of_item(a, i)]) return;
  int32_t r = parent[i];
  for (int32_t p = parent[r]; p != r; p = parent[r]) r = p;
  parent[i] = r;
}

// Joins the trees of items x and y.  A root that a stale read shows may have been
// hooked meanwhile: the compare-and-swap then returns what it is hooked under, and
// the walk goes on from there (ids only fall, so it ends).
__device__ inline void cc_join(int32_t* parent, int32_t x, int32_t y) {
  int32_t u = x, v = y;
  while (true) {
    u = cc_find(parent, u);
    v = cc_find(parent, v);
    if (u == v) return;
    if (u > v) {
      int32_t t = u;
      u = v;
      v = t;
    }
    // hook root v under the smaller root u
    const int32_t old = atomicCAS(&parent[v], v, u);
    if (old == v) return;
    v = old;
  }
}

// Joins the two ends of every edge inside a cluster (each edge at its larger
// end).  The labels of a short row and then the roots of its ends are read side
// by side; only an edge between two trees takes the walk.  8.39 M items: 1118 us
// edge by edge from single items, 600 from the trees of k_cc_init, 397 so (and
// k_cc_count 479 -> 65 us).
__global__ void k_cc_hook(SweepArgs a, const int32_t* __restrict__ mask, int32_t* parent) {
  int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= a.n_items || !mask[mesh_of_item(a, i)]) return;
  const int32_t lab = a.labels[i];
  if (lab == kNull) return;
  int32_t nbr[kRingCache];
  if (load_row8(a, i, nbr)) {
    const int32_t root = parent[i];
    int32_t r[kRingCache];
#pragma unroll
    for (int p = 0; p < kRingCache; ++p) r[p] = nbr[p] >= 0 && nbr[p] < i ? a.labels[nbr[p]] : kNull;
#pragma unroll
    for (int p = 0; p < kRingCache; ++p) r[p] = r[p] == lab ? parent[nbr[p]] : root;
    int32_t last = root;  // the ends of a row mostly show one other root
#pragma unroll 1
    for (int p = 0; p < kRingCache; ++p) {
      int32_t q = root;
#pragma unroll
      for (int k = 0; k < kRingCache; ++k)
        if (k == p) q = r[k];
      if (q == root || q == last) continue;
      cc_join(parent, root, q);
      last = q;
    }
  } else {
    for (int32_t k = a.row_ptr[i]; k < a.row_ptr[i + 1]; ++k) {
      const int32_t j = a.col[k];
      if (j < i && a.labels[j] == lab) cc_join(parent, int32_t(i), j);
    }
  }
}

// Sizes of the components, one atomic per run of equal roots in a wave; the items
// keep their root.
__global__ void k_cc_count(SweepArgs a, const int32_t* __restrict__ mask, int32_t* parent, int32_t* comp_size) {
  int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  int32_t r = -1;
  if (i < a.n_items && mask[mesh_of_item(a, i)] && a.labels[i] != kNull) {
    r = cc_find(parent, int32_t(i));
    parent[i] = r;
  }
  const int32_t prev = __shfl_up(r, 1);
  const bool head = __lane_id() == 0 || prev != r;
  const int len = 1 + run_left(__ballot(head));
  if (head && r >= 0) atomicAdd(&comp_size[r], len);
}

__global__ void k_cc_best(SweepArgs a, const int32_t* __restrict__ mask, const int32_t* __restrict__ parent,
                          const int32_t* __restrict__ comp_size, unsigned long long* best, int32_t* ncomp) {
  int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= a.n_items || !mask[mesh_of_item(a, i)]) return;
  const int32_t lab = a.labels[i];
  if (lab == kNull || parent[i] != i) return;
  // the component holding the cluster's fixed item first (its size counts 1e9
  // in CleanClustering, vtkUniformClustering.h:441-447), then the larger
  // component, then the smaller first item
  uint32_t size = uint32_t(comp_size[i]);
  const int32_t an = a.anchor ? a.anchor[lab] : -1;
  if (an >= 0) {
    int32_t r = an;
    while (parent[r] != r) r = parent[r];  // read-only find (the hooks are done)
    if (r == int32_t(i)) size |= 0x80000000u;
  }
  const unsigned long long key = (uint64_t(size) << 32) | uint64_t(0xFFFFFFFFu - uint32_t(i));
  atomicMax(&best[lab], key);
  atomicAdd(&ncomp[lab], 1);
}

__global__ void k_cc_reset(SweepArgs a, const int32_t* __restrict__ mask, int32_t* parent,
                           const unsigned long long* __restrict__ best) {
  int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= a.n_items || !mask[mesh_of_item(a, i)]) return;
  const int32_t lab = a.labels[i];
  if (lab == kNull) return;
  const int32_t r = cc_find(parent, int32_t(i));
  const uint32_t keep = 0xFFFFFFFFu - uint32_t(best[lab] & 0xFFFFFFFFull);
  if (uint32_t(r) != keep) a.labels[i] = kNull;
}

__global__ void k_cc_zero(SweepArgs a, const int32_t* __restrict__ mask, unsigned long long* best, int32_t* ncomp) {
  int64_t c = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (c >= a.n_clusters || !mask[mesh_of_cluster(a, c)]) return;
  best[c] = 0ull;
  ncomp[c] = 0;
}

__global__ void k_cc_disc(SweepArgs a, const int32_t* __restrict__ mask, const int32_t* __restrict__ ncomp,
                          int32_t* ndisc) {
  int64_t c = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  int m = 0;
  bool split = false;
  if (c < a.n_clusters) {
    m = mesh_of_cluster(a, c);
    split = mask[m] && ncomp[c] > 1;
  }
  count_per_mesh(split, m, [&](int32_t mm) { return &ndisc[mm]; });
}

// ----------------------------------------------------------------- seeding
// Weighted random seeds: key_i = E_i / w_i with E_i ~ Exp(1); the K smallest
// keys of a mesh (one sort) seed its clusters, so that denser regions get
// more seeds.
__global__ void k_seed_keys(SweepArgs a, int64_t off, int64_t n, uint32_t seed, uint32_t* keys, int32_t* vals) {
  int64_t t = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (t >= n) return;
  const int64_t i = off + t;
  uint32_t h = prio_hash(seed ^ 0x5EEDu, 0x9E37u, uint32_t(t));
  double u = (double(h) + 0.5) * (1.0 / 4294967296.0);
  double w = a.xw[i].w;
  float k = float(-log(u) / (w > 0 ? w : 1e-300));
  keys[t] = __float_as_uint(k);  // positive floats order like their bits
  vals[t] = int32_t(t);
}

__global__ void k_seed_assign(int32_t* labels, int64_t item_off, int64_t clus_off, int32_t K,
                              const int32_t* __restrict__ sorted_vals) {
  int64_t r = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (r >= K) return;
  labels[item_off + sorted_vals[r]] = int32_t(clus_off + r);
}

// ----------------------------------------------------------------- outputs
// Cluster point of mesh `mesh`: centroid (isotropic) or the QEM point when the
// metric is constrained (GetClusterCentroid semantics).
__global__ void k_cluster_points(SweepArgs a, int32_t mesh, double* pts) {
  const DevMesh dm = a.meshes[mesh];
  int64_t r = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (r >= dm.K) return;
  const int64_t c = dm.clus_off + r;
  const int64_t W = ld_i64(&a.acc_ws[4 * c]);
  const ClusterGeom g = geom_from_fixed(W, ld_i64(&a.acc_ws[4 * c + 1]), ld_i64(&a.acc_ws[4 * c + 2]),
                                        ld_i64(&a.acc_ws[4 * c + 3]), dm.scales);
  double q[3] = {g.cx, g.cy, g.cz};
  const int32_t an = a.anchor && dm.metric == 1 ? a.anchor[c] : -1;
  if (!(g.W > 0.0)) {
    q[0] = q[1] = q[2] = __builtin_nan("");
  } else if (an >= 0) {  // fixed cluster: the anchor (exact input coordinates are set by the host)
    const float4 p = a.xw[an];
    q[0] = p.x;
    q[1] = p.y;
    q[2] = p.z;
  } else if (dm.metric == 1 && a.state[mesh].constrained) {
    int64_t q10[10];
    for (int k = 0; k < 10; ++k) q10[k] = ld_i64(&a.acc_q[10 * c + k]);
    qem_T_from_fixed(q10, g, dm.scales, dm.level, q);
  }
  pts[3 * r] = q[0];
  pts[3 * r + 1] = q[1];
  pts[3 * r + 2] = q[2];
}

// Per-item unshifted energy w |x - p_c|^2 with p_c given per global cluster.
__global__ void k_item_energy(SweepArgs a, const double* __restrict__ pts_all, double* e_item) {
  int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= a.n_items) return;
  const int32_t c = a.labels[i];
  if (c == kNull) {
    e_item[i] = 0.0;
    return;
  }
  const float4 p = a.xw[i];
  double dx = double(p.x) - pts_all[3 * int64_t(c)];
  double dy = double(p.y) - pts_all[3 * int64_t(c) + 1];
  double dz = double(p.z) - pts_all[3 * int64_t(c) + 2];
  e_item[i] = double(p.w) * (dx * dx + dy * dy + dz * dz);
}

// Energy log, step 1 (WriteToGlobalEnergyLog, vtkUniformClustering.h:1383-1395):
// the energy of every cluster from its exact accumulators, the point solved
// from scratch (no warm start, so the value depends on the labels only).
__global__ void k_log_cluster_energy(SweepArgs a, double* __restrict__ e) {
  int64_t c = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (c >= a.n_clusters) return;
  const int m = mesh_of_cluster(a, c);
  const DevMesh dm = a.meshes[m];
  const int64_t W = ld_i64(&a.acc_ws[4 * c]);
  const ClusterGeom g = geom_from_fixed(W, ld_i64(&a.acc_ws[4 * c + 1]), ld_i64(&a.acc_ws[4 * c + 2]),
                                        ld_i64(&a.acc_ws[4 * c + 3]), dm.scales);
  double T = 0.0;
  if (dm.metric == 1) {
    const int32_t an = a.anchor ? a.anchor[c] : -1;
    if (an >= 0) {
      const float4 p = a.xw[an];
      T = anchored_T(g, AnchorPos{double(p.x), double(p.y), double(p.z), true});
    } else if (a.state[m].constrained) {
      int64_t q10[10];
      for (int k = 0; k < 10; ++k) q10[k] = ld_i64(&a.acc_q[10 * c + k]);
      T = qem_T_from_fixed(q10, g, dm.scales, dm.level, nullptr);
    }
  }
  e[c] = log_cluster_energy(g, T);
}

// Energy log, step 2: one block per mesh sums its clusters in the order of
// kLogThreads (acvd_math.h).  In a pass (final_e null) a sweeping mesh writes
// its energy and the device wall clock to entry `loops % ring` of its ring of
// log entries, before the controller counts the pass; the final call writes
// every mesh's energy to final_e.
__global__ void __launch_bounds__(kLogThreads) k_log_reduce(SweepArgs a, const double* __restrict__ e,
                                                            EnergyLogEntry* log, int32_t ring, double* final_e) {
  const int m = blockIdx.x;
  const int32_t phase = a.state[m].phase, loop = a.state[m].loops;
  if (!final_e && (phase != kPhaseSweep || loop < 0)) return;  // uniform over the block
  const DevMesh dm = a.meshes[m];
  __shared__ double part[kLogThreads];
  double s = 0.0;
  for (int64_t r = threadIdx.x; r < dm.K; r += kLogThreads) s += e[dm.clus_off + r];
  part[threadIdx.x] = s;
  __syncthreads();
  for (int h = kLogThreads / 2; h > 0; h >>= 1) {
    if (int(threadIdx.x) < h) part[threadIdx.x] += part[threadIdx.x + h];
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    if (final_e) {
      final_e[m] = part[0];
    } else {
      EnergyLogEntry& x = log[int64_t(m) * ring + loop % ring];
      x.energy = part[0];
      x.clock = (unsigned long long)wall_clock64();
    }
  }
}

__global__ void k_clock_stamp(unsigned long long* t) { *t = (unsigned long long)wall_clock64(); }

// Labels between the caller's numbering (0..K-1, anything else none; K = none on
// the way out) and the context's (global cluster ids, kNull).  A pass over device
// memory costs 15 us at 8.39 M items; the loop over host memory, with the fresh
// buffer it filled, took 5 ms each way.
__global__ void k_labels_in(int64_t n, int32_t K, int32_t clus_off, int32_t* labels) {
  int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int32_t l = labels[i];
  labels[i] = (l < 0 || l >= K) ? kNull : l + clus_off;
}
__global__ void k_labels_out(int64_t n, int32_t K, int32_t clus_off, const int32_t* __restrict__ labels,
                             int32_t* __restrict__ out) {
  int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i < n) out[i] = labels[i] == kNull ? K : labels[i] - clus_off;
}

__global__ void k_fill_i32(int32_t* p, int64_t n, int32_t v) {
  int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}
__global__ void k_fill_u64(unsigned long long* p, int64_t n, unsigned long long v) {
  int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}

}  // namespace

// ------------------------------------------------------------------ launchers
hipError_t launch_zero_clusters(hipStream_t s, const SweepArgs& a, const int32_t* mask) {
  if (a.n_clusters == 0) return hipSuccess;
  hipLaunchKernelGGL(k_zero_clusters, dim3(grid_for(a.n_clusters)), dim3(kBlock), 0, s, a, mask);
  return hipGetLastError();
}

hipError_t launch_accumulate(hipStream_t s, const SweepArgs& a, const int32_t* mask, unsigned long long* mesh_count) {
  if (a.n_items == 0) return hipSuccess;
  const int64_t per = (a.n_items + kAccBlocks - 1) / kAccBlocks;
  const int64_t chunk = (per + kAccBlock - 1) / kAccBlock * kAccBlock;
  hipLaunchKernelGGL(k_accumulate, dim3(unsigned((a.n_items + chunk - 1) / chunk)), dim3(kAccBlock), 0, s, a, mask,
                     mesh_count, chunk);
  return hipGetLastError();
}

hipError_t launch_derive(hipStream_t s, const SweepArgs& a, const int32_t* mask, int set_stamp) {
  if (a.n_clusters == 0) return hipSuccess;
  hipLaunchKernelGGL(k_derive, dim3(grid_for(a.n_clusters)), dim3(kBlock), 0, s, a, mask, set_stamp);
  return hipGetLastError();
}

hipError_t launch_tile_sets(hipStream_t s, const SweepArgs& a, const int32_t* mesh_mask) {
  if (a.n_tiles == 0) return hipSuccess;
  hipLaunchKernelGGL(k_tile_sets, dim3(unsigned(a.n_tiles)), dim3(64), 0, s, a, mesh_mask);
  return hipGetLastError();
}

hipError_t launch_scan(hipStream_t s, const SweepArgs& a, bool tiles) {
  if (a.n_items == 0) return hipSuccess;
  const dim3 grid(unsigned((a.n_tiles + kTilesPerScanBlock - 1) / kTilesPerScanBlock));
  // blocks of kBlock items never outnumber the scan tiles (each mesh's tiles
  // cover its items), so the linear scan stays within the slice capacity
  static_assert(kBlock == kTileItems, "one scan block per tile's worth of items");
  if (tiles) hipLaunchKernelGGL(k_scan, grid, dim3(kBlock), 0, s, a);
  else hipLaunchKernelGGL(k_scan_linear, dim3(unsigned((a.n_items + kBlock - 1) / kBlock)), dim3(kBlock), 0, s, a);
  return hipGetLastError();
}

// One evaluate block per candidate segment: block b writes segment b's count.
// qem_unconstrained: no QEM mesh is constrained (the QEM meshes take the
// isotropic rule, METRIC 2).
// The kernels come in three builds: with the anchor and freeze tests (some mesh
// has fixed or frozen clusters), without them, and without them for a context of
// one mesh (kB = false: no mesh lookups).
template <bool kX, bool kB>
void launch_eval_x(hipStream_t s, const SweepArgs& a, bool any_iso, bool any_qem, bool qem_unconstrained) {
  const dim3 g(unsigned(a.n_seg)), b(kBlock);
  if (any_iso) hipLaunchKernelGGL((k_eval<0, kX, kB>), g, b, 0, s, a, 0);
  if (any_qem && qem_unconstrained) hipLaunchKernelGGL((k_eval<2, kX, kB>), g, b, 0, s, a, any_iso ? 1 : 0);
  else if (any_qem) hipLaunchKernelGGL((k_eval<1, kX, kB>), g, b, 0, s, a, any_iso ? 1 : 0);
}

hipError_t launch_eval(hipStream_t s, const SweepArgs& a, bool any_iso, bool any_qem, bool qem_unconstrained) {
  if (a.anchor || a.frozen) launch_eval_x<true, true>(s, a, any_iso, any_qem, qem_unconstrained);
  else if (a.item_mesh) launch_eval_x<false, true>(s, a, any_iso, any_qem, qem_unconstrained);
  else launch_eval_x<false, false>(s, a, any_iso, any_qem, qem_unconstrained);
  return hipGetLastError();
}

template <bool kX, bool kB, bool kT>
void launch_scan_eval_t(hipStream_t s, const SweepArgs& a, bool any_iso, bool any_qem, bool qem_unconstrained) {
  const dim3 g(unsigned(a.n_seg)), b(kBlock);
  if (any_iso) hipLaunchKernelGGL((k_scan_eval<0, kX, kB, kT>), g, b, 0, s, a, 0);
  if (any_qem && qem_unconstrained) hipLaunchKernelGGL((k_scan_eval<2, kX, kB, kT>), g, b, 0, s, a, any_iso ? 1 : 0);
  else if (any_qem) hipLaunchKernelGGL((k_scan_eval<1, kX, kB, kT>), g, b, 0, s, a, any_iso ? 1 : 0);
}
template <bool kX, bool kB>
void launch_scan_eval_x(hipStream_t s, const SweepArgs& a, bool any_iso, bool any_qem, bool qem_unconstrained) {
  if (a.crowded) launch_scan_eval_t<kX, kB, true>(s, a, any_iso, any_qem, qem_unconstrained);
  else launch_scan_eval_t<kX, kB, false>(s, a, any_iso, any_qem, qem_unconstrained);
}

hipError_t launch_scan_eval(hipStream_t s, const SweepArgs& a, bool any_iso, bool any_qem, bool qem_unconstrained) {
  if (a.anchor || a.frozen) launch_scan_eval_x<true, true>(s, a, any_iso, any_qem, qem_unconstrained);
  else if (a.item_mesh) launch_scan_eval_x<false, true>(s, a, any_iso, any_qem, qem_unconstrained);
  else launch_scan_eval_x<false, false>(s, a, any_iso, any_qem, qem_unconstrained);
  return hipGetLastError();
}

// One apply block per candidate segment (its moved segment has the same
// index).  constrained: some mesh is constrained (derives may need a solve).
template <bool kX, bool kB>
void launch_apply_x(hipStream_t s, const SweepArgs& a, int round, bool constrained) {
  const dim3 g(unsigned(a.n_seg)), b(kBlock);
  if (constrained) hipLaunchKernelGGL((k_apply<true, kX, kB>), g, b, 0, s, a, round);
  else hipLaunchKernelGGL((k_apply<false, kX, kB>), g, b, 0, s, a, round);
}

hipError_t launch_apply(hipStream_t s, const SweepArgs& a, int round, bool constrained) {
  if (a.anchor || a.frozen) launch_apply_x<true, true>(s, a, round, constrained);
  else if (a.item_mesh) launch_apply_x<false, true>(s, a, round, constrained);
  else launch_apply_x<false, false>(s, a, round, constrained);
  return hipGetLastError();
}

hipError_t launch_tile_update(hipStream_t s, const SweepArgs& a) {
  hipLaunchKernelGGL(k_tile_update, dim3(unsigned(a.n_seg)), dim3(kBlock), 0, s, a);
  return hipGetLastError();
}

template <bool kX, bool kB, bool kC, bool kT>
void launch_reeval_t(hipStream_t s, const SweepArgs& a, bool any_iso, bool any_qem, bool qem_unconstrained,
                     int round) {
  const dim3 g(unsigned(a.n_seg)), b(kBlock);
  if (any_iso) hipLaunchKernelGGL((k_reeval<0, kX, kB, kC, kT>), g, b, 0, s, a, round);
  if (any_qem && qem_unconstrained) hipLaunchKernelGGL((k_reeval<2, kX, kB, kC, kT>), g, b, 0, s, a, round);
  else if (any_qem) hipLaunchKernelGGL((k_reeval<1, kX, kB, kC, kT>), g, b, 0, s, a, round);
}
template <bool kX, bool kB, bool kC>
void launch_reeval_x(hipStream_t s, const SweepArgs& a, bool any_iso, bool any_qem, bool qem_unconstrained,
                     int round) {
  if (a.crowded) launch_reeval_t<kX, kB, kC, true>(s, a, any_iso, any_qem, qem_unconstrained, round);
  else launch_reeval_t<kX, kB, kC, false>(s, a, any_iso, any_qem, qem_unconstrained, round);
}

hipError_t launch_reeval(hipStream_t s, const SweepArgs& a, bool any_iso, bool any_qem, bool qem_unconstrained,
                         int round) {
  const bool x = a.anchor || a.frozen, c = a.count_rounds != 0;
  if (x && c) launch_reeval_x<true, true, true>(s, a, any_iso, any_qem, qem_unconstrained, round);
  else if (x) launch_reeval_x<true, true, false>(s, a, any_iso, any_qem, qem_unconstrained, round);
  else if (c) launch_reeval_x<false, true, true>(s, a, any_iso, any_qem, qem_unconstrained, round);
  else if (a.item_mesh) launch_reeval_x<false, true, false>(s, a, any_iso, any_qem, qem_unconstrained, round);
  else launch_reeval_x<false, false, false>(s, a, any_iso, any_qem, qem_unconstrained, round);
  return hipGetLastError();
}

hipError_t launch_controller(hipStream_t s, const SweepArgs& a) {
  hipLaunchKernelGGL(k_controller, dim3(1), dim3(kBlock), 0, s, a);
  return hipGetLastError();
}

hipError_t launch_fill_round(hipStream_t s, const SweepArgs& a, const int32_t* mask, int32_t* pending) {
  if (a.n_items == 0) return hipSuccess;
  hipLaunchKernelGGL(k_fill_pick, dim3(grid_for(a.n_items)), dim3(kBlock), 0, s, a, mask, pending);
  hipLaunchKernelGGL(k_fill_commit, dim3(grid_for(a.n_items)), dim3(kBlock), 0, s, a, mask, pending);
  return hipGetLastError();
}

hipError_t launch_cc(hipStream_t s, const SweepArgs& a, const int32_t* mask, int32_t* parent, int32_t* comp_size,
                     unsigned long long* best, int32_t* ncomp, int32_t* ndisc) {
  if (a.n_items == 0) return hipSuccess;
  const dim3 gi(grid_for(a.n_items)), gc(grid_for(a.n_clusters)), b(kBlock);
  hipLaunchKernelGGL(k_cc_init, gi, b, 0, s, a, mask, parent, comp_size);
  hipLaunchKernelGGL(k_cc_zero, gc, b, 0, s, a, mask, best, ncomp);
  hipLaunchKernelGGL(k_cc_flatten, gi, b, 0, s, a, mask, parent);
  hipLaunchKernelGGL(k_cc_hook, gi, b, 0, s, a, mask, parent);
  hipLaunchKernelGGL(k_cc_count, gi, b, 0, s, a, mask, parent, comp_size);
  hipLaunchKernelGGL(k_cc_best, gi, b, 0, s, a, mask, parent, comp_size, best, ncomp);
  hipLaunchKernelGGL(k_cc_reset, gi, b, 0, s, a, mask, parent, best);
  hipLaunchKernelGGL(k_cc_disc, gc, b, 0, s, a, mask, ncomp, ndisc);
  return hipGetLastError();
}

hipError_t launch_seed_keys(hipStream_t s, const SweepArgs& a, int64_t off, int64_t n, uint32_t seed,
                            uint32_t* keys, int32_t* vals) {
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(k_seed_keys, dim3(grid_for(n)), dim3(kBlock), 0, s, a, off, n, seed, keys, vals);
  return hipGetLastError();
}

hipError_t launch_seed_assign(hipStream_t s, int32_t* labels, int64_t item_off, int64_t clus_off, int32_t K,
                              const int32_t* sorted_vals) {
  if (K == 0) return hipSuccess;
  hipLaunchKernelGGL(k_seed_assign, dim3(grid_for(K)), dim3(kBlock), 0, s, labels, item_off, clus_off, K,
                     sorted_vals);
  return hipGetLastError();
}

hipError_t sort_pairs_u32(hipStream_t s, const uint32_t* kin, uint32_t* kout, const int32_t* vin, int32_t* vout,
                          int64_t n, void** tmp, size_t* tmp_bytes) {
  size_t need = 0;
  hipError_t e = hipcub::DeviceRadixSort::SortPairs(nullptr, need, kin, kout, vin, vout, int(n), 0, 32, s);
  if (e != hipSuccess) return e;
  if (need > *tmp_bytes) {
    if (*tmp) (void)hipFree(*tmp);
    *tmp = nullptr;
    e = hipMalloc(tmp, need);
    if (e != hipSuccess) return e;
    *tmp_bytes = need;
  }
  return hipcub::DeviceRadixSort::SortPairs(*tmp, need, kin, kout, vin, vout, int(n), 0, 32, s);
}

hipError_t launch_cluster_points(hipStream_t s, const SweepArgs& a, int32_t mesh, double* pts) {
  hipLaunchKernelGGL(k_cluster_points, dim3(unsigned((a.n_clusters + kBlock - 1) / kBlock) + 1), dim3(kBlock), 0, s,
                     a, mesh, pts);
  return hipGetLastError();
}

hipError_t launch_item_energy(hipStream_t s, const SweepArgs& a, const double* pts_all, double* e_item) {
  if (a.n_items == 0) return hipSuccess;
  hipLaunchKernelGGL(k_item_energy, dim3(grid_for(a.n_items)), dim3(kBlock), 0, s, a, pts_all, e_item);
  return hipGetLastError();
}

hipError_t launch_energy_log(hipStream_t s, const SweepArgs& a, double* e_cluster, EnergyLogEntry* log, int32_t ring,
                             double* final_e) {
  if (a.n_clusters == 0 || a.n_meshes == 0) return hipSuccess;
  hipLaunchKernelGGL(k_log_cluster_energy, dim3(grid_for(a.n_clusters)), dim3(kBlock), 0, s, a, e_cluster);
  hipLaunchKernelGGL(k_log_reduce, dim3(unsigned(a.n_meshes)), dim3(kLogThreads), 0, s, a, e_cluster, log, ring,
                     final_e);
  return hipGetLastError();
}

hipError_t launch_clock_stamp(hipStream_t s, unsigned long long* t) {
  hipLaunchKernelGGL(k_clock_stamp, dim3(1), dim3(1), 0, s, t);
  return hipGetLastError();
}

hipError_t launch_labels_in(hipStream_t s, int64_t n, int32_t K, int64_t clus_off, int32_t* labels) {
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(k_labels_in, dim3(grid_for(n)), dim3(kBlock), 0, s, n, K, int32_t(clus_off), labels);
  return hipGetLastError();
}

hipError_t launch_labels_out(hipStream_t s, int64_t n, int32_t K, int64_t clus_off, const int32_t* labels,
                             int32_t* out) {
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(k_labels_out, dim3(grid_for(n)), dim3(kBlock), 0, s, n, K, int32_t(clus_off), labels, out);
  return hipGetLastError();
}

hipError_t launch_fill_i32(hipStream_t s, int32_t* p, int64_t n, int32_t v) {
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(k_fill_i32, dim3(grid_for(n)), dim3(kBlock), 0, s, p, n, v);
  return hipGetLastError();
}

hipError_t launch_fill_u64(hipStream_t s, unsigned long long* p, int64_t n, unsigned long long v) {
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(k_fill_u64, dim3(grid_for(n)), dim3(kBlock), 0, s, p, n, v);
  return hipGetLastError();
}

}  // namespace acvd

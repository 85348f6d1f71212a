// Fixed-assignment clustering energy and its adjoint.
//
// For a labelling l (frozen) of the vertices of one or more meshes:
//   isotropic (ACVD):  E = sum_i w_i |x_i - c_l(i)|^2,  c = S/W,
//                      S = sum w x, W = sum w over the cluster
//                      (vtkIsotropicMetricForClustering.h:114-121 unshifted);
//   QEM (ACVDQ):       E = sum_i w_i |x_i - q_l(i)|^2,
//                      q = c + A+_trunc (b - A c), with (A, b) from the cluster
//                      quadric Q_c = sum_{i in c} sum_{f ni i} Q_f(x),
//                      Q_f = [n; d][n; d]^T, n = (x2-x1) x (x3-x1), d = -n.x1
//                      (vtkQEMetricForClustering.h:151-167, 194-208,
//                      Common/vtkQuadricTools.cxx:56-177).
// Everything is computed in FP64 from FP32 positions and weights; the face
// quadrics are recomputed from the positions (so that they are differentiable),
// unlike the sweep, which uses FP32 vertex quadrics.
//
// Forward: cluster sums (W, S, Q), cluster points, per-mesh energy.  The
// points kernel also computes the adjoint of each QEM cluster for a unit
// upstream gradient (dE/dq = -2 (S - W q) pulled back through q(c, A, b); the
// truncated pseudo-inverse's derivative includes the coupling of kept and
// dropped eigen-directions) into dE/dQ (9 entries) and dE/dc: the adjoint is
// linear in the gradient, and the eigen-decomposition is at hand.  Backward:
// per vertex the direct terms, the centroid path and the face-quadric path
// (over the faces around the vertex, recomputed, no per-item partials stored)
// give dE/dx and dE/dw.
//
// The faces around a vertex v are read as a chain of neighbour ids (the ring):
// two ids in a row are the other two vertices of a face, in its orientation, so
// an interior vertex of valence d takes d + 1 ids and one position gather per
// neighbour, instead of d face ids, 3 d vertex ids and 3 d positions.  The rings
// of 64 consecutive vertices are stored slot by slot (slot s of all 64, then
// slot s + 1): one 256-byte load per slot and wave.

#include <hip/hip_runtime.h>

#include <algorithm>
#include <mutex>

#include "acvd_energy.h"

namespace acvd {

namespace {

constexpr int kEBlock = 256;
constexpr int kAccBlock = 512;          // threads of ke_accumulate and ke_energy
constexpr int kAccMaxBlocks = 512;      // 2 blocks of ke_accumulate per CU (its registers)
constexpr double kThreshold = 1e-3;

inline unsigned egrid(int64_t n) { return unsigned((n + kEBlock - 1) / kEBlock); }

__device__ inline int mesh_of(const EnergyArgs& a, int64_t i) { return a.item_mesh ? a.item_mesh[i] : 0; }

// What the kernels over items use of a mesh: uniform over the block, or (kMany)
// each lane's own.
struct ItemMesh {
  int32_t off, K;  // clusters
  bool qem;
};

__device__ inline ItemMesh item_mesh(const EnergyMesh& em) {
  return ItemMesh{int32_t(em.clus_off), em.K, em.metric == 1};
}

// global cluster of an item labelled l, or -1
__device__ inline int32_t cluster_of(const ItemMesh& im, int32_t l) {
  return (l < 0 || l >= im.K) ? -1 : im.off + l;
}

// Lanes that follow in the lane's run, given the run heads of the wave.
__device__ inline int run_left(unsigned long long heads) {
  const int lane = threadIdx.x & 63;
  const unsigned long long after = lane == 63 ? 0ull : heads >> (lane + 1);
  return after ? __builtin_ctzll(after) : 63 - lane;
}

struct Vec3 {
  double x, y, z;
};

__device__ inline Vec3 load_point(const float* __restrict__ xyz, int64_t i) {
  return Vec3{double(xyz[3 * i]), double(xyz[3 * i + 1]), double(xyz[3 * i + 2])};
}

__device__ inline Vec3 sub(const Vec3& a, const Vec3& b) { return Vec3{a.x - b.x, a.y - b.y, a.z - b.z}; }

// Normal of the face (v, v + u, v + w) (plain products, so that a degenerate
// face gives an exact zero).
__device__ inline Vec3 cross(const Vec3& u, const Vec3& w) {
  return Vec3{u.y * w.z - u.z * w.y, u.z * w.x - u.x * w.z, u.x * w.y - u.y * w.x};
}

struct RingPoint {
  float x, y, z;
};

__device__ inline Vec3 ring_point(const EnergyArgs& a, int32_t e) {
  return load_point(a.xyz, int64_t(e & kRingId));
}

// The first kRingChunk ring entries of item i (64 consecutive items per wave:
// i = 64 g + lane), loaded together; returns the group's slots.
__device__ inline int32_t load_ring(const EnergyArgs& a, int64_t i, int32_t e[kRingChunk]) {
  const int64_t g = __builtin_amdgcn_readfirstlane(int32_t(i >> 6));
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int k = 0; k < kRingChunk; ++k) e[k] = kRingEnd;
  if (64 * g >= a.n_items) return 0;  // a wave past the last group
  const int32_t s0 = a.ring_slot[g], n = a.ring_slot[g + 1] - s0;  // scalar loads
#pragma unroll
  for (int k = 0; k < kRingChunk; ++k)
    if (k < n) e[k] = a.ring[int64_t(s0 + k) * 64 + lane];
  return n;
}

// Faces around item i past its first `from` ring entries (u: the previous ring
// vertex less the item's position, cu: its tag), and those of a vertex with more
// faces than a ring holds: the paths of rare vertices, an entry at a time.
// tag(id) labels a ring vertex; face(u, cu, s, cs) takes a face.
template <class Tag, class Face>
__device__ inline void walk_rest(const EnergyArgs& a, int64_t i, const Vec3& x, int32_t first, int from, Vec3 u,
                                 int32_t cu, Tag&& tag, Face&& face) {
  if (first == kRingLong) {
    for (int32_t k = a.vfptr[i]; k < a.vfptr[i + 1]; ++k) {
      const int64_t f = a.vfcol[k];
      // the corner of this entry: a face listed more than once for the vertex
      // (a degenerate face, whose normal is zero) takes its first corner
      int j = 0;
      while (j < 2 && a.tri[3 * f + j] != int32_t(i)) ++j;
      const int32_t v1 = a.tri[3 * f + (j + 1) % 3], v2 = a.tri[3 * f + (j + 2) % 3];
      face(sub(load_point(a.xyz, v1), x), tag(v1), sub(load_point(a.xyz, v2), x), tag(v2));
    }
    return;
  }
  const int32_t s0 = a.ring_slot[i >> 6], s1 = a.ring_slot[(i >> 6) + 1];
  for (int32_t s = s0 + from; s < s1; ++s) {
    const int32_t e = a.ring[int64_t(s) * 64 + (i & 63)];
    if (e == kRingEnd) break;
    const Vec3 t = sub(ring_point(a, e), x);
    const int32_t ct = tag(e & kRingId);
    if (e >= 0) face(u, cu, t, ct);
    u = t;
    cu = ct;
  }
}

// Symmetric 3x3 eigen-decomposition by cyclic Jacobi to convergence.
// A = (a00, a01, a02, a11, a12, a22); V columns are eigenvectors (V[3*r + k]).
__device__ void eig_sym3(const double* A, double lam[3], double V[9]) {
  double a[3][3] = {{A[0], A[1], A[2]}, {A[1], A[3], A[4]}, {A[2], A[4], A[5]}};
  for (int k = 0; k < 9; ++k) V[k] = (k % 4 == 0) ? 1.0 : 0.0;
  for (int sweep = 0; sweep < 16; ++sweep) {
    const double off = fabs(a[0][1]) + fabs(a[0][2]) + fabs(a[1][2]);
    const double dia = fabs(a[0][0]) + fabs(a[1][1]) + fabs(a[2][2]);
    if (!(off > dia * 1e-18)) break;
    for (int p = 0; p < 2; ++p)
      for (int q = p + 1; q < 3; ++q) {
        const double apq = a[p][q];
        if (apq == 0.0) continue;
        const double theta = (a[q][q] - a[p][p]) / (2.0 * apq);
        const double t = (fabs(theta) > 1e150) ? 0.5 / theta
                                                : (theta >= 0 ? 1.0 : -1.0) / (fabs(theta) + sqrt(theta * theta + 1.0));
        const double cs = 1.0 / sqrt(t * t + 1.0), sn = t * cs;
        // A <- J^T A J with J the (p,q) rotation
        for (int k = 0; k < 3; ++k) {
          const double akp = a[k][p], akq = a[k][q];
          a[k][p] = cs * akp - sn * akq;
          a[k][q] = sn * akp + cs * akq;
        }
        for (int k = 0; k < 3; ++k) {
          const double apk = a[p][k], aqk = a[q][k];
          a[p][k] = cs * apk - sn * aqk;
          a[q][k] = sn * apk + cs * aqk;
        }
        a[p][q] = a[q][p] = 0.0;
        for (int r = 0; r < 3; ++r) {
          const double vp = V[3 * r + p], vq = V[3 * r + q];
          V[3 * r + p] = cs * vp - sn * vq;
          V[3 * r + q] = sn * vp + cs * vq;
        }
      }
  }
  lam[0] = a[0][0];
  lam[1] = a[1][1];
  lam[2] = a[2][2];
}

// Kept eigen-directions: by decreasing |lambda| (first index on ties) while
// |lambda| / max|lambda| > 1e-3 and at most `level` of them
// (vtkQuadricTools.cxx:119-154).
__device__ inline void kept_set(const double lam[3], int level, bool keep[3]) {
  double aw[3] = {fabs(lam[0]), fabs(lam[1]), fabs(lam[2])};
  const double mx = fmax(aw[0], fmax(aw[1], aw[2]));
  keep[0] = keep[1] = keep[2] = false;
  int left = level;
  for (int it = 0; it < 3; ++it) {
    int idx = -1;
    double best = -1.0;
    for (int k = 0; k < 3; ++k)
      if (!keep[k] && aw[k] > best && aw[k] >= 0.0) {
        // skip indices already decided as dropped
        best = aw[k];
        idx = k;
      }
    if (idx < 0) break;
    if (mx > 0.0 && best * (1.0 / mx) > kThreshold && left > 0) {
      keep[idx] = true;
      --left;
    } else {
      break;  // every remaining value is smaller
    }
  }
}

__device__ inline double dot3(const double* a, const double* b) { return a[0] * b[0] + a[1] * b[1] + a[2] * b[2]; }

// ---------------------------------------------------------------- ring build
__global__ void ke_offset_tri(int64_t n, int32_t off, int32_t* tri) {
  const int64_t k = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (k < n) tri[k] += off;
}

__global__ void ke_vf_count(int64_t n3, const int32_t* __restrict__ tri, int32_t* deg) {
  const int64_t k = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (k < n3) atomicAdd(&deg[tri[k]], 1);
}

__global__ void ke_vf_fill(int64_t n3, const int32_t* __restrict__ tri, const int32_t* __restrict__ vfptr,
                           int32_t* fill, int32_t* vfcol) {
  const int64_t k = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (k >= n3) return;
  const int32_t v = tri[k];
  vfcol[vfptr[v] + atomicAdd(&fill[v], 1)] = int32_t(k / 3);
}

// Sorts the vertex -> face rows by face id (heap sort: a row of any length in
// n log n steps), so that a ring does not depend on the order of the atomics.
__global__ void ke_vf_sort(int64_t n, const int32_t* __restrict__ vfptr, int32_t* vfcol) {
  const int64_t v = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (v >= n) return;
  int32_t* r = vfcol + vfptr[v];
  const int32_t len = vfptr[v + 1] - vfptr[v];
  if (len <= 32) {
    for (int32_t i = 1; i < len; ++i) {
      const int32_t x = r[i];
      int32_t j = i - 1;
      for (; j >= 0 && r[j] > x; --j) r[j + 1] = r[j];
      r[j + 1] = x;
    }
    return;
  }
  for (int32_t half = len / 2, end = len; end > 1;) {
    int32_t x;
    if (half > 0) {
      x = r[--half];
    } else {
      x = r[--end];
      r[end] = r[0];
    }
    int32_t p = half;
    for (int32_t c = 2 * p + 1; c < end; c = 2 * p + 1) {
      if (c + 1 < end && r[c + 1] > r[c]) ++c;
      if (r[c] <= x) break;
      r[p] = r[c];
      p = c;
    }
    r[p] = x;
  }
}

// Ring of vertex v (at most kRingFaces faces): the links a -> b of its faces
// (v, a, b) strung into chains.  A chain starts at a link no unused link leads
// to (a boundary vertex, a bowtie), else at the first unused one (a closed fan).
// emit(k, entry) is called for every entry; returns their number.
template <class Emit>
__device__ int ring_chains(const EnergyArgs& a, int64_t v, Emit&& emit) {
  const int32_t k0 = a.vfptr[v], d = a.vfptr[v + 1] - k0;
  int32_t la[kRingFaces], lb[kRingFaces];
  for (int k = 0; k < d; ++k) {
    const int64_t f = a.vfcol[k0 + k];
    int j = 0;
    while (j < 2 && a.tri[3 * f + j] != int32_t(v)) ++j;
    la[k] = a.tri[3 * f + (j + 1) % 3];
    lb[k] = a.tri[3 * f + (j + 2) % 3];
  }
  uint32_t left = d == 32 ? ~0u : (1u << d) - 1u;
  int n = 0;
  while (left) {
    int s = -1;
    for (int k = 0; k < d && s < 0; ++k) {
      if (!(left >> k & 1u)) continue;
      bool led = false;
      for (int t = 0; t < d; ++t) led = led || (t != k && (left >> t & 1u) && lb[t] == la[k]);
      if (!led) s = k;
    }
    if (s < 0) s = __builtin_ctz(left);
    emit(n++, int32_t(uint32_t(la[s]) | 0x80000000u));
    while (s >= 0) {
      left &= ~(1u << s);
      const int32_t cur = lb[s];
      emit(n++, cur);
      s = -1;
      for (int t = 0; t < d && s < 0; ++t)
        if ((left >> t & 1u) && la[t] == cur) s = t;
    }
  }
  return n;
}

// Slots of each group of 64 vertices: the longest ring of its QEM vertices.
__global__ __launch_bounds__(64) void ke_ring_slots(EnergyArgs a, int32_t* slots) {
  const int64_t v = int64_t(blockIdx.x) * 64 + threadIdx.x;
  int n = 0;
  if (v < a.n_items && a.meshes[mesh_of(a, v)].metric == 1) {
    if (a.vfptr[v + 1] - a.vfptr[v] > kRingFaces) n = 1;
    else n = ring_chains(a, v, [](int, int32_t) {});
  }
  for (int off = 32; off > 0; off >>= 1) n = max(n, __shfl_xor(n, off));
  if (threadIdx.x == 0) slots[blockIdx.x] = n;
}

__global__ __launch_bounds__(64) void ke_ring_fill(EnergyArgs a, const int32_t* __restrict__ slot, int32_t* ring) {
  const int64_t v = int64_t(blockIdx.x) * 64 + threadIdx.x;
  const int32_t s0 = slot[blockIdx.x], s1 = slot[blockIdx.x + 1];
  int32_t* r = ring + int64_t(s0) * 64 + threadIdx.x;
  int n = 0;
  if (v < a.n_items && a.meshes[mesh_of(a, v)].metric == 1) {
    if (a.vfptr[v + 1] - a.vfptr[v] > kRingFaces) {
      r[0] = kRingLong;
      n = 1;
    } else {
      n = ring_chains(a, v, [&](int k, int32_t e) { r[int64_t(k) * 64] = e; });
    }
  }
  for (; n < s1 - s0; ++n) r[int64_t(n) * 64] = kRingEnd;
}

// ------------------------------------------------------------------ forward
// Clears the cluster sums and the energies (one launch; stores of 16 bytes).
__global__ __launch_bounds__(kEBlock) void ke_zero(int64_t n_acc, double* acc, int64_t n_meshes, double* energy) {
  const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (2 * i + 1 < n_acc) reinterpret_cast<double2*>(acc)[i] = make_double2(0.0, 0.0);
  else if (2 * i < n_acc) acc[2 * i] = 0.0;
  if (i < n_meshes) energy[i] = 0.0;
}

template <int CTRL>
__device__ inline double dpp_f64(double x) {
  const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(x), CTRL, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(x), CTRL, 0xf, 0xf, true);
  return __hiloint2double(hi, lo);
}

// One doubling step of the segmented sum over runs of equal keys: lane l adds
// lane l + D when that lane belongs to its run (rem = lanes left in the run).
template <int D, int V>
__device__ inline void merge_step(double (&v)[V], int rem) {
  const bool take = rem >= D;
  if (__ballot(take) == 0ull) return;
#pragma unroll
  for (int k = 0; k < V; ++k) {
    const double t = dpp_f64<0x100 | D>(v[k]);  // row_shl:D
    v[k] += take ? t : 0.0;
  }
}

// Cluster sums.  Block b takes a contiguous range of items, 512 at a time: the
// lanes of a wave first merge runs of equal clusters in registers (aligned runs
// of at most 8 lanes), each run then adds once into the block's LDS table keyed
// by cluster, and the table goes to the global sums when it is three quarters
// full and at the end, consecutive threads to consecutive words.
// A table of 256 items (one mesh row's worth) flushed every cluster about 7
// times, 34 M f64 atomics for 16.8 M QEM vertices and most of the kernel's time;
// kept over a block's range it flushes each 1 to 2 times.  Now bound by the f64
// work (580 instructions a step of 64 items, 60 % of the time) and the gathers'
// latency at 4 waves per SIMD: 16.8 M QEM vertices 2328 -> 372 us (a copy of the
// bytes takes 168 us), 1 M isotropic ones 45.7 -> 16.7 us.
template <bool kQem, bool kMany>
__global__ __launch_bounds__(kAccBlock) void ke_accumulate(EnergyArgs a, int64_t chunk) {
  constexpr int V = kQem ? 13 : 4;  // W, S[3], Q[9]
  constexpr int kSlots = kQem ? 512 : 1024;
  constexpr int kSlotBits = kQem ? 9 : 10;
  constexpr int kFlushAt = kSlots * 3 / 4;
  constexpr int kProbes = 32;
  constexpr int kRun = 8;         // lanes merged at most (16 M QEM vertices: 1 592 us, 2 467, 4 429, 8 432, 16 425)
  constexpr int kCheckSteps = 4;  // steps between looks at the table's fill (1: 432 us, 4: 407)
  __shared__ int32_t keys[kSlots];
  __shared__ double vals[kSlots * V];
  __shared__ int32_t n_keys;
  for (int k = threadIdx.x; k < kSlots; k += kAccBlock) keys[k] = -1;
  for (int k = threadIdx.x; k < kSlots * V; k += kAccBlock) vals[k] = 0.0;
  if (threadIdx.x == 0) n_keys = 0;
  __syncthreads();
  const int64_t begin = int64_t(blockIdx.x) * chunk;
  const int64_t end = min(begin + chunk, a.n_items);
  const int lane = threadIdx.x & 63;
  auto flush = [&]() {  // every thread of the block; the table is complete
    for (int k = threadIdx.x; k < kSlots * V; k += kAccBlock) {
      const int32_t key = keys[k / V];
      const double x = vals[k];
      vals[k] = 0.0;
      if (key >= 0 && x != 0.0) atomicAdd(&a.acc[int64_t(key) * a.acc_stride + k % V], x);
    }
    __syncthreads();
    for (int k = threadIdx.x; k < kSlots; k += kAccBlock) keys[k] = -1;
    if (threadIdx.x == 0) n_keys = 0;
    __syncthreads();
  };
  const int m0 = kMany ? 0 : mesh_of(a, begin), m1 = kMany ? 0 : mesh_of(a, end - 1);
  int step = 0;
  for (int m = m0; m <= m1; ++m) {
    const EnergyMesh em = a.meshes[m];
    const int64_t first = kMany ? begin : max(begin, em.item_off);
    const int64_t last = kMany ? end : min(end, em.item_off + em.n_items);
    ItemMesh im = item_mesh(em);
    const bool rings = kQem && (kMany || im.qem);  // block-uniform
    // steps stay aligned to the chunk (and so to the ring groups)
    const int64_t base0 = begin + (first - begin) / kAccBlock * kAccBlock;
    int32_t e[kRingChunk];
    int32_t slots = 0, lab = -1, mi = 0;
    // the ring entries, labels and (kMany) meshes of a step are read during the step before it
    if (rings && base0 < last) slots = load_ring(a, base0 + threadIdx.x, e);
    if (base0 + int64_t(threadIdx.x) >= first && base0 + int64_t(threadIdx.x) < last) {
      lab = a.labels[base0 + threadIdx.x];
      if (kMany) mi = a.item_mesh[base0 + threadIdx.x];
    }
    for (int64_t base = base0; base < last; base += kAccBlock) {
      const int64_t i = base + threadIdx.x;
      const bool active = i >= first && i < last;
      if (kMany) im = item_mesh(a.meshes[mi]);
      const int32_t c = active ? cluster_of(im, lab) : -1;
      const bool qem = kQem && im.qem;
      double v[V];
#pragma unroll
      for (int k = 0; k < V; ++k) v[k] = 0.0;
      Vec3 x{0.0, 0.0, 0.0};
      RingPoint q[kRingChunk];
      const int32_t e0 = e[0], cur_slots = slots;
      uint32_t faces = 0;  // entries that close a face
      if (qem && c >= 0) {
#pragma unroll
        for (int k = 0; k < kRingChunk; ++k) {
          const int64_t j = (e[k] == kRingEnd || e0 == kRingLong) ? i : int64_t(e[k] & kRingId);
          q[k] = RingPoint{a.xyz[3 * j], a.xyz[3 * j + 1], a.xyz[3 * j + 2]};
          if (e[k] >= 0) faces |= 1u << k;
        }
      }
      const bool more = qem && c >= 0 && (e0 == kRingLong || (cur_slots > kRingChunk && e[kRingChunk - 1] != kRingEnd));
      if (c >= 0) {
        const double w = double(a.w[i]);
        x = load_point(a.xyz, i);
        v[0] = w;
        v[1] = w * x.x;
        v[2] = w * x.y;
        v[3] = w * x.z;
      }
      if (base + kAccBlock < last) {
        if (rings) slots = load_ring(a, i + kAccBlock, e);
        lab = i + kAccBlock < last ? a.labels[i + kAccBlock] : -1;
        if (kMany && i + kAccBlock < last) mi = a.item_mesh[i + kAccBlock];
      }
      if constexpr (kQem) {
        if (qem && c >= 0) {
          auto add = [&](const Vec3& n) {
            v[4] = __builtin_fma(n.x, n.x, v[4]);
            v[5] = __builtin_fma(n.x, n.y, v[5]);
            v[6] = __builtin_fma(n.x, n.z, v[6]);
            v[8] = __builtin_fma(n.y, n.y, v[8]);
            v[9] = __builtin_fma(n.y, n.z, v[9]);
            v[11] = __builtin_fma(n.z, n.z, v[11]);
          };
          Vec3 u{0.0, 0.0, 0.0};
#pragma unroll
          for (int k = 0; k < kRingChunk; ++k) {
            const Vec3 t = sub(Vec3{double(q[k].x), double(q[k].y), double(q[k].z)}, x);
            if (faces >> k & 1u) add(cross(u, t));
            u = t;
          }
          if (more)
            walk_rest(
                a, i, x, e0, kRingChunk, u, 0, [](int32_t) { return 0; },
                [&](const Vec3& r, int32_t, const Vec3& t, int32_t) { add(cross(r, t)); });
          // every plane passes through the vertex (d = -n . x): sum n d = -(sum n n^T) x
          v[7] = -(v[4] * x.x + v[5] * x.y + v[6] * x.z);
          v[10] = -(v[5] * x.x + v[8] * x.y + v[9] * x.z);
          v[12] = -(v[6] * x.x + v[9] * x.y + v[11] * x.z);
        }
      }
      // runs of equal clusters
      const int32_t prev = __builtin_amdgcn_update_dpp(-2, c, 0x111, 0xf, 0xf, false);  // row_shr:1
      const bool head = prev != c || (lane & (kRun - 1)) == 0;
      const int rem = run_left(__ballot(head));
      static_assert(kRun == 8, "three doubling steps");
      merge_step<1>(v, rem);
      merge_step<2>(v, rem);
      merge_step<4>(v, rem);
      if (head && c >= 0) {
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
        if (slot >= 0) {
#pragma unroll
          for (int k = 0; k < V; ++k) atomicAdd(&vals[slot * V + k], v[k]);
        } else {  // no free slot near by: straight to the global sums
#pragma unroll
          for (int k = 0; k < V; ++k)
            if (v[k] != 0.0) atomicAdd(&a.acc[int64_t(c) * a.acc_stride + k], v[k]);
        }
      }
      if (++step % kCheckSteps == 0) {  // block-uniform
        __syncthreads();
        const bool full = n_keys > kFlushAt;
        __syncthreads();
        if (full) flush();
      }
    }
  }
  __syncthreads();
  flush();
}

// Cluster points: q, and for QEM meshes the unit adjoint (adj: dE/dQ at 0..8,
// (dE/dc) / W at 9..11, the centroid at 12..14).
__global__ __launch_bounds__(64) void ke_points(EnergyArgs a) {
  const int64_t c = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (c >= a.n_clusters) return;
  const EnergyMesh& em = a.meshes[a.clus_mesh ? a.clus_mesh[c] : 0];
  const double* s = a.acc + c * a.acc_stride;
  const double W = s[0];
  double cc[3] = {0.0, 0.0, 0.0}, q[3] = {0.0, 0.0, 0.0};
  double adj[12] = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
  const bool some = W > 0.0;
  if (some)
    for (int k = 0; k < 3; ++k) q[k] = cc[k] = s[1 + k] / W;
  if (some && em.metric == 1) {
    double Q[9];
    for (int k = 0; k < 9; ++k) Q[k] = s[4 + k];
    const double A[6] = {Q[0], Q[1], Q[2], Q[4], Q[5], Q[7]};
    double lam[3], V[9];
    bool keep[3];
    eig_sym3(A, lam, V);
    kept_set(lam, em.level, keep);
    const double r[3] = {-Q[3] - (Q[0] * cc[0] + Q[1] * cc[1] + Q[2] * cc[2]),
                         -Q[6] - (Q[1] * cc[0] + Q[4] * cc[1] + Q[5] * cc[2]),
                         -Q[8] - (Q[2] * cc[0] + Q[5] * cc[1] + Q[7] * cc[2])};
    double vr[3];
    for (int k = 0; k < 3; ++k) {
      const double vk[3] = {V[k], V[3 + k], V[6 + k]};
      vr[k] = dot3(vk, r);
      if (!keep[k]) continue;
      const double f = vr[k] / lam[k];
      for (int e = 0; e < 3; ++e) q[e] += f * vk[e];
    }
    // dE/dq = -2 (S - W q)
    const double gq[3] = {-2.0 * (s[1] - W * q[0]), -2.0 * (s[2] - W * q[1]), -2.0 * (s[3] - W * q[2])};
    double vg[3];
    // y = A+ r = q - c; h = A+ gq; P gq = gq - sum_kept v_k (v_k . gq)
    double h[3] = {0, 0, 0}, pg[3] = {gq[0], gq[1], gq[2]};
    for (int k = 0; k < 3; ++k) {
      const double vk[3] = {V[k], V[3 + k], V[6 + k]};
      vg[k] = dot3(vk, gq);
      if (!keep[k]) continue;
      for (int e = 0; e < 3; ++e) {
        h[e] += V[3 * e + k] * vg[k] / lam[k];
        pg[e] -= V[3 * e + k] * vg[k];
      }
    }
    // G = -h (y + c)^T + sum_{k kept, j dropped} coef_kj v_j v_k^T, y + c = q
    double G[3][3];
    for (int r0 = 0; r0 < 3; ++r0)
      for (int c0 = 0; c0 < 3; ++c0) G[r0][c0] = -h[r0] * q[c0];
    for (int k = 0; k < 3; ++k) {
      if (!keep[k]) continue;
      for (int j = 0; j < 3; ++j) {
        if (keep[j]) continue;
        const double gap = lam[k] - lam[j];
        if (gap == 0.0) continue;
        const double coef = (vg[j] * vr[k] + vg[k] * vr[j]) / (lam[k] * gap);
        for (int r0 = 0; r0 < 3; ++r0)
          for (int c0 = 0; c0 < 3; ++c0) G[r0][c0] += coef * V[3 * r0 + j] * V[3 * c0 + k];
      }
    }
    // dE/dA as the symmetric matrix B with dE = n^T B dn for a plane normal n
    // (00, 01, 02, 11, 12, 22), then dE/d(n d) = -A+ gq
    adj[0] = 2.0 * G[0][0];
    adj[1] = G[0][1] + G[1][0];
    adj[2] = G[0][2] + G[2][0];
    adj[3] = 2.0 * G[1][1];
    adj[4] = G[1][2] + G[2][1];
    adj[5] = 2.0 * G[2][2];
    for (int e = 0; e < 3; ++e) adj[6 + e] = -h[e];
    for (int e = 0; e < 3; ++e) adj[9 + e] = pg[e] / W;
  }
  double* out = a.pts + 4 * c;
  for (int k = 0; k < 3; ++k) out[k] = q[k];
  if (a.adj) {
    double* o = a.adj + kAdjStride * c;
    for (int k = 0; k < 12; ++k) o[k] = adj[k];
    for (int k = 0; k < 3; ++k) o[12 + k] = cc[k];
  }
}

// Per-mesh energy.  Few blocks, each over a contiguous range of items, add
// their sums to the mesh's energy: one atomic per block and mesh (atomics on one
// address take 12.7 ns each; with one per 256 items they were this kernel's
// time: 1 M vertices 52 -> 8 us, 16 x 1 M 694 -> 92 us, 3.6 TB/s).
template <bool kMany>
__global__ __launch_bounds__(kAccBlock) void ke_energy(EnergyArgs a, int64_t chunk, double* energy) {
  constexpr int kWaves = kAccBlock / 64;
  __shared__ double red[kWaves];
  const int64_t begin = int64_t(blockIdx.x) * chunk;
  const int64_t end = min(begin + chunk, a.n_items);
  auto term = [&](const ItemMesh& im, int64_t i) {
    const int32_t c = cluster_of(im, a.labels[i]);
    const Vec3 x = load_point(a.xyz, i);
    const double w = double(a.w[i]);
    if (c < 0) return 0.0;
    const double* q = a.pts + 4 * int64_t(c);
    const double dx = x.x - q[0], dy = x.y - q[1], dz = x.z - q[2];
    return w * (dx * dx + dy * dy + dz * dz);
  };
  if constexpr (kMany) {
    // A wave adds up the items of one mesh while its lanes lie in it (cur), and
    // else the runs of its lanes in each mesh.
    __shared__ int32_t mesh[kWaves];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    double e = 0.0;
    int32_t cur = -1;
    auto wave_sum = [&]() {
      for (int off = 32; off > 0; off >>= 1) e += __shfl_xor(e, off);
    };
    for (int64_t base = begin; base < end; base += kAccBlock) {
      const int64_t i = base + threadIdx.x;
      const int32_t m = i < end ? a.item_mesh[i] : -1;
      double t = m >= 0 ? term(item_mesh(a.meshes[m]), i) : 0.0;
      const int32_t m0 = __builtin_amdgcn_readfirstlane(m);
      if (__ballot(m != m0) == 0ull) {
        if (m0 != cur) {
          wave_sum();
          if (lane == 0 && cur >= 0) atomicAdd(&energy[cur], e);
          e = 0.0;
          cur = m0;
        }
        e += t;
      } else {
        const int32_t prev = __shfl_up(m, 1);
        const bool head = lane == 0 || prev != m;
        const int rem = run_left(__ballot(head));
        for (int off = 1; off < 64; off <<= 1) {
          const double u = __shfl_down(t, off);
          if (rem >= off) t += u;
        }
        if (head && m >= 0) atomicAdd(&energy[m], t);
      }
    }
    wave_sum();
    if (lane == 0) {
      red[wave] = e;
      mesh[wave] = cur;
    }
    __syncthreads();
    if (threadIdx.x == 0)  // one atomic for neighbouring waves of one mesh
      for (int k = 0; k < kWaves;) {
        const int32_t m = mesh[k];
        double sum = 0.0;
        for (; k < kWaves && mesh[k] == m; ++k) sum += red[k];
        if (m >= 0) atomicAdd(&energy[m], sum);
      }
  } else {
    const int m0 = mesh_of(a, begin), m1 = mesh_of(a, end - 1);
    for (int m = m0; m <= m1; ++m) {
      const EnergyMesh em = a.meshes[m];
      const ItemMesh im = item_mesh(em);
      const int64_t first = max(begin, em.item_off), last = min(end, em.item_off + em.n_items);
      double e = 0.0;
#pragma unroll 4
      for (int64_t i = first + threadIdx.x; i < last; i += kAccBlock) e += term(im, i);
      for (int off = 32; off > 0; off >>= 1) e += __shfl_xor(e, off);
      __syncthreads();  // red of the previous mesh has been read
      if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = e;
      __syncthreads();
      if (threadIdx.x == 0) {
        for (int k = 1; k < kWaves; ++k) e += red[k];
        atomicAdd(&energy[m], e);
      }
    }
  }
}

// The whole forward of one small isotropic mesh in one block: sums, points and
// energy in turn, the sums in LDS by cluster.  The four launches of the general
// forward cost the host more than this block takes (2,562 vertices, a call from
// Python: 21.8 -> 13.4 us).
constexpr int kSmallBlock = 1024;
constexpr int64_t kSmallItems = 4096;
constexpr int64_t kSmallClusters = 1024;
__global__ __launch_bounds__(kSmallBlock) void ke_forward_small(EnergyArgs a, double* energy) {
  __shared__ double acc[kSmallClusters * 4];
  __shared__ double red[kSmallBlock / 64];
  const ItemMesh em = item_mesh(a.meshes[0]);
  const int lane = threadIdx.x & 63;
  for (int k = threadIdx.x; k < em.K * 4; k += kSmallBlock) acc[k] = 0.0;
  __syncthreads();
  for (int64_t base = 0; base < a.n_items; base += kSmallBlock) {
    const int64_t i = base + threadIdx.x;
    const int32_t c = i < a.n_items ? cluster_of(em, a.labels[i]) : -1;
    double v[4] = {0.0, 0.0, 0.0, 0.0};
    if (c >= 0) {
      const Vec3 x = load_point(a.xyz, i);
      v[0] = double(a.w[i]);
      v[1] = v[0] * x.x;
      v[2] = v[0] * x.y;
      v[3] = v[0] * x.z;
    }
    const int32_t prev = __builtin_amdgcn_update_dpp(-2, c, 0x111, 0xf, 0xf, false);  // row_shr:1
    const bool head = prev != c || (lane & 7) == 0;
    const int rem = run_left(__ballot(head));
    merge_step<1>(v, rem);
    merge_step<2>(v, rem);
    merge_step<4>(v, rem);
    if (head && c >= 0)
      for (int k = 0; k < 4; ++k) atomicAdd(&acc[4 * c + k], v[k]);
  }
  __syncthreads();
  for (int c = threadIdx.x; c < em.K; c += kSmallBlock) {
    const double W = acc[4 * c];
    for (int k = 0; k < 3; ++k) {
      const double q = W > 0.0 ? acc[4 * c + 1 + k] / W : 0.0;
      acc[4 * c + 1 + k] = q;
      a.pts[4 * c + k] = q;
    }
  }
  __syncthreads();
  double e = 0.0;
  for (int64_t i = threadIdx.x; i < a.n_items; i += kSmallBlock) {
    const int32_t c = cluster_of(em, a.labels[i]);
    if (c < 0) continue;
    const Vec3 x = load_point(a.xyz, i);
    const double* q = acc + 4 * c + 1;
    const double dx = x.x - q[0], dy = x.y - q[1], dz = x.z - q[2];
    e += double(a.w[i]) * (dx * dx + dy * dy + dz * dz);
  }
  for (int off = 32; off > 0; off >>= 1) e += __shfl_xor(e, off);
  if (lane == 0) red[threadIdx.x >> 6] = e;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int k = 1; k < kSmallBlock / 64; ++k) e += red[k];
    energy[0] = e;
  }
}

// ----------------------------------------------------------------- backward
// Adjoint of one cluster's quadric as the planes through a vertex x see it.  With
// d = -n . x, dE = n^T B dn + g . d(n d) pulls back to dE/dn = M n with
// M = B - g x^T - x g^T, and x receives -(g . n) n: both depend on the vertex,
// not on the face.
struct PlaneAdjoint {
  double m[6];  // M: 00, 01, 02, 11, 12, 22
  double g[3];
};

__device__ inline PlaneAdjoint plane_adjoint(const double* __restrict__ adj, const Vec3& x) {
  PlaneAdjoint r;
  for (int k = 0; k < 3; ++k) r.g[k] = adj[6 + k];
  r.m[0] = adj[0] - 2.0 * (r.g[0] * x.x);
  r.m[1] = adj[1] - (r.g[0] * x.y + r.g[1] * x.x);
  r.m[2] = adj[2] - (r.g[0] * x.z + r.g[2] * x.x);
  r.m[3] = adj[3] - 2.0 * (r.g[1] * x.y);
  r.m[4] = adj[4] - (r.g[1] * x.z + r.g[2] * x.y);
  r.m[5] = adj[5] - 2.0 * (r.g[2] * x.z);
  return r;
}

__device__ inline PlaneAdjoint no_adjoint() {
  PlaneAdjoint r;
  for (int k = 0; k < 6; ++k) r.m[k] = 0.0;
  for (int k = 0; k < 3; ++k) r.g[k] = 0.0;
  return r;
}

// Per vertex: dE/dx (3) and dE/dw.  QEM: the faces around the vertex v, each as
// (v, v + u, v + s), feed the clusters of their three vertices.  The adjoints of
// the vertex's cluster and of the first two others its ring meets are read
// before the faces are visited: read face by face, behind the labels, they were
// most of this kernel's waits.  A wave with a ring of more clusters visits the
// faces again for the next two (against reading them face by face: labels of a
// graded clustering of 4 x 1 M vertices 296 -> 257 us, 12 vertices a cluster
// 306 -> 266, 42 a cluster 708 -> 715).  Consecutive blocks run on one XCD, whose
// L2 then holds the rows a block shares with its neighbours (HBM reads 1.27 ->
// 0.87 GB).  Bound by the f64 work (950
// instructions per 64 vertices, half of the time) and by gather latency at 3
// waves per SIMD (168 registers; held to 128 the spills cost more: 1359 us;
// a loop over the faces that keeps one position in flight: 831 us).
// 16.8 M QEM vertices 2050 -> 765 us, 1 M isotropic ones 10.5 -> 8.6 us.
template <bool kQem, bool kMany>
__global__ __launch_bounds__(kEBlock) void ke_item_grad(EnergyArgs a, const double* __restrict__ gE,
                                                        float* __restrict__ dxyz, float* __restrict__ dw) {
  constexpr int kXcd = 8;
  const int64_t nb = gridDim.x, xcd = blockIdx.x % kXcd;
  const int64_t block = xcd * (nb / kXcd) + min(xcd, nb % kXcd) + blockIdx.x / kXcd;
  const int64_t begin = block * kEBlock;
  const int64_t end = min(begin + kEBlock, a.n_items);
  const int64_t i = begin + threadIdx.x;
  // what does not depend on the mesh is read with the mesh's number
  const int64_t ic = min(i, a.n_items - 1);
  const int32_t lab = a.labels[ic];
  const float wf = a.w[ic];
  const Vec3 x = load_point(a.xyz, ic);
  int32_t e[kRingChunk];
  int32_t slots = 0;
  if constexpr (kQem) slots = load_ring(a, i, e);
  const int m0 = kMany ? 0 : mesh_of(a, begin), m1 = kMany ? 0 : mesh_of(a, end - 1);
  for (int m = m0; m <= m1; ++m) {
    const EnergyMesh& mesh = a.meshes[kMany ? a.item_mesh[ic] : m];
    const ItemMesh em = item_mesh(mesh);
    const bool active = i < end && (kMany || (i >= mesh.item_off && i < mesh.item_off + mesh.n_items));
    const double g = gE[kMany ? a.item_mesh[ic] : m];
    double gx[3] = {0, 0, 0}, gw = 0.0;
    const int32_t c = active ? cluster_of(em, lab) : -1;
    const bool qem = kQem && em.qem;  // block-uniform unless kMany
    if (c >= 0) {
      const double w = double(wf);
      const double* q = a.pts + 4 * int64_t(c);
      const double d[3] = {x.x - q[0], x.y - q[1], x.z - q[2]};
      for (int k = 0; k < 3; ++k) gx[k] = 2.0 * w * d[k];
      gw = d[0] * d[0] + d[1] * d[1] + d[2] * d[2];
      if (qem) {
        const double* adj = a.adj + kAdjStride * int64_t(c);
        for (int k = 0; k < 3; ++k) gx[k] += w * adj[9 + k];
        gw += adj[9] * (x.x - adj[12]) + adj[10] * (x.y - adj[13]) + adj[11] * (x.z - adj[14]);
      }
    }
    if (qem && active) {
      // clusters of the ring's first entries: bit k of own_bits the vertex's own, of
      // todo another one whose part is still to be taken
      const bool is_long = e[0] == kRingLong;
      const bool more = is_long || (slots > kRingChunk && e[kRingChunk - 1] != kRingEnd);
      int32_t cl[kRingChunk];
      uint32_t own_bits = 0, todo = 0;
#pragma unroll
      for (int k = 0; k < kRingChunk; ++k) {
        if (k >= slots) break;  // wave-uniform
        if (e[k] == kRingEnd || is_long) e[k] = int32_t(uint32_t(i) | 0x80000000u);  // no face
        cl[k] = a.labels[e[k] & kRingId];
      }
#pragma unroll
      for (int k = 0; k < kRingChunk; ++k) {
        if (k >= slots) break;
        cl[k] = cluster_of(em, cl[k]);
        if (cl[k] >= 0) (cl[k] == c ? own_bits : todo) |= 1u << k;
      }
      PlaneAdjoint A0 = c >= 0 ? plane_adjoint(a.adj + kAdjStride * int64_t(c), x) : no_adjoint();
      double own = c >= 0 ? 1.0 : 0.0;
      // the face (v, v + u, v + s) with adjoint F: n = u x s; u receives s x dn,
      // s receives dn x u, and v minus both (dn x (u - s)) and minus (g . n) n
      auto pull = [&](const PlaneAdjoint& F, const Vec3& u, const Vec3& s) {
        const Vec3 n = cross(u, s), t = sub(u, s);
        const double n0 = __builtin_fma(F.m[2], n.z, __builtin_fma(F.m[1], n.y, F.m[0] * n.x));
        const double n1 = __builtin_fma(F.m[4], n.z, __builtin_fma(F.m[3], n.y, F.m[1] * n.x));
        const double n2 = __builtin_fma(F.m[5], n.z, __builtin_fma(F.m[4], n.y, F.m[2] * n.x));
        const double gn = __builtin_fma(F.g[2], n.z, __builtin_fma(F.g[1], n.y, F.g[0] * n.x));
        gx[0] -= __builtin_fma(gn, n.x, __builtin_fma(n1, t.z, -(n2 * t.y)));
        gx[1] -= __builtin_fma(gn, n.y, __builtin_fma(n2, t.x, -(n0 * t.z)));
        gx[2] -= __builtin_fma(gn, n.z, __builtin_fma(n0, t.y, -(n1 * t.x)));
      };
      Vec3 u{0.0, 0.0, 0.0};
      while (true) {
        int32_t c1 = -1, c2 = -1;
        uint32_t bits1 = 0, bits2 = 0;
#pragma unroll
        for (int k = 0; k < kRingChunk; ++k) {
          if (k >= slots) break;
          if (!(todo >> k & 1u)) continue;
          if (c1 < 0) c1 = cl[k];
          if (cl[k] == c1) bits1 |= 1u << k;
          else {
            if (c2 < 0) c2 = cl[k];
            if (cl[k] == c2) bits2 |= 1u << k;
          }
        }
        todo &= ~(bits1 | bits2);
        const PlaneAdjoint A1 = c1 >= 0 ? plane_adjoint(a.adj + kAdjStride * int64_t(c1), x) : no_adjoint();
        const PlaneAdjoint A2 = c2 >= 0 ? plane_adjoint(a.adj + kAdjStride * int64_t(c2), x) : no_adjoint();
#pragma unroll
        for (int k = 0; k < kRingChunk; ++k) {
          if (k >= slots) break;
          const Vec3 s = sub(ring_point(a, e[k]), x);
          if (k > 0 && e[k] >= 0) {
            const double w0 = own + ((own_bits >> (k - 1) & 1u) ? 1.0 : 0.0) + ((own_bits >> k & 1u) ? 1.0 : 0.0);
            const double w1 = ((bits1 >> (k - 1) & 1u) ? 1.0 : 0.0) + ((bits1 >> k & 1u) ? 1.0 : 0.0);
            const double w2 = ((bits2 >> (k - 1) & 1u) ? 1.0 : 0.0) + ((bits2 >> k & 1u) ? 1.0 : 0.0);
            PlaneAdjoint F;
            for (int j = 0; j < 6; ++j)
              F.m[j] = __builtin_fma(w2, A2.m[j], __builtin_fma(w1, A1.m[j], w0 * A0.m[j]));
            for (int j = 0; j < 3; ++j)
              F.g[j] = __builtin_fma(w2, A2.g[j], __builtin_fma(w1, A1.g[j], w0 * A0.g[j]));
            pull(F, u, s);
          }
          u = s;
        }
        if (__ballot(todo != 0) == 0ull) break;
        // rings of more clusters: the faces again for the next two, the own part done
        A0 = no_adjoint();
        own = 0.0;
        own_bits = 0;
      }
      if (more) {  // faces past the first entries, in full
        auto pull_of = [&](int32_t cj, const Vec3& r, const Vec3& s) {
          if (cj >= 0) pull(plane_adjoint(a.adj + kAdjStride * int64_t(cj), x), r, s);
        };
        const int32_t cu = is_long ? -1 : cl[kRingChunk - 1];
        walk_rest(
            a, i, x, is_long ? kRingLong : 0, kRingChunk, u, cu,
            [&](int32_t j) { return cluster_of(em, a.labels[j]); },
            [&](const Vec3& r, int32_t cr, const Vec3& s, int32_t cs) {
              pull_of(c, r, s);
              pull_of(cr, r, s);
              pull_of(cs, r, s);
            });
      }
    }
    if (active) {
      for (int k = 0; k < 3; ++k) dxyz[3 * i + k] = float(g * gx[k]);
      dw[i] = float(g * gw);
    }
  }
}

}  // namespace

// Items per block of ke_accumulate and ke_energy: a multiple of the block, at
// least 4,096 where that still leaves a block per CU, so that a block's table
// sees several mesh rows; at most `max_blocks` blocks.
static int64_t item_chunk(int64_t n, int64_t max_blocks) {
  int64_t blocks = (n + kAccBlock - 1) / kAccBlock;
  blocks = std::min(blocks, std::max<int64_t>(256, std::min(max_blocks, n / 4096)));
  const int64_t per = (n + blocks - 1) / blocks;
  return (per + kAccBlock - 1) / kAccBlock * kAccBlock;
}

hipError_t energy_forward(hipStream_t s, const EnergyArgs& a, double* energy, int n_meshes) {
  if (!a.adj && n_meshes == 1 && a.n_items > 0 && a.n_items <= kSmallItems && a.n_clusters <= kSmallClusters) {
    hipLaunchKernelGGL(ke_forward_small, dim3(1), dim3(kSmallBlock), 0, s, a, energy);
    return hipGetLastError();
  }
  const int64_t nacc = a.n_clusters * a.acc_stride;
  hipLaunchKernelGGL(ke_zero, dim3(egrid(std::max<int64_t>((nacc + 1) / 2, n_meshes))), dim3(kEBlock), 0, s, nacc,
                     a.acc, int64_t(n_meshes), energy);
  if (a.n_items > 0) {
    const int64_t chunk = item_chunk(a.n_items, kAccMaxBlocks);
    const dim3 grid(unsigned((a.n_items + chunk - 1) / chunk));
    const auto k = a.adj ? (a.many ? ke_accumulate<true, true> : ke_accumulate<true, false>)
                         : (a.many ? ke_accumulate<false, true> : ke_accumulate<false, false>);
    hipLaunchKernelGGL(k, grid, dim3(kAccBlock), 0, s, a, chunk);
  }
  if (a.n_clusters > 0)
    hipLaunchKernelGGL(ke_points, dim3(unsigned((a.n_clusters + 63) / 64)), dim3(64), 0, s, a);
  if (a.n_items > 0) {
    const int64_t chunk = item_chunk(a.n_items, 512);
    hipLaunchKernelGGL(a.many ? ke_energy<true> : ke_energy<false>, dim3(unsigned((a.n_items + chunk - 1) / chunk)),
                       dim3(kAccBlock), 0, s, a, chunk, energy);
  }
  return hipGetLastError();
}

hipError_t energy_offset_tri(hipStream_t s, int64_t n3, int32_t off, int32_t* tri) {
  if (n3 == 0 || off == 0) return hipSuccess;
  hipLaunchKernelGGL(ke_offset_tri, dim3(egrid(n3)), dim3(kEBlock), 0, s, n3, off, tri);
  return hipGetLastError();
}

hipError_t energy_vf_count(hipStream_t s, int64_t n3, const int32_t* tri, int32_t* deg) {
  if (n3 == 0) return hipSuccess;
  hipLaunchKernelGGL(ke_vf_count, dim3(egrid(n3)), dim3(kEBlock), 0, s, n3, tri, deg);
  return hipGetLastError();
}

hipError_t energy_vf_fill(hipStream_t s, int64_t n, int64_t n3, const int32_t* tri, const int32_t* vfptr,
                          int32_t* fill, int32_t* vfcol) {
  if (n3 == 0) return hipSuccess;
  hipLaunchKernelGGL(ke_vf_fill, dim3(egrid(n3)), dim3(kEBlock), 0, s, n3, tri, vfptr, fill, vfcol);
  hipLaunchKernelGGL(ke_vf_sort, dim3(egrid(n)), dim3(kEBlock), 0, s, n, vfptr, vfcol);
  return hipGetLastError();
}

hipError_t energy_ring_slots(hipStream_t s, const EnergyArgs& a, int32_t* slots) {
  hipLaunchKernelGGL(ke_ring_slots, dim3(unsigned((a.n_items + 63) / 64)), dim3(64), 0, s, a, slots);
  return hipGetLastError();
}

hipError_t energy_ring_fill(hipStream_t s, const EnergyArgs& a, const int32_t* slot, int32_t* ring) {
  hipLaunchKernelGGL(ke_ring_fill, dim3(unsigned((a.n_items + 63) / 64)), dim3(64), 0, s, a, slot, ring);
  return hipGetLastError();
}

// ------------------------------------------------- forward without allocation
namespace {

// Scratch of energy_forward_cvt_noalloc: the mesh descriptor, then the
// per-cluster sums (4 doubles) and points (4 doubles) of at most
// kNoAllocMaxClusters clusters; one copy per device, held until the process
// ends.  Host code never passes `scratch` itself to a kernel (in host code the
// name is only a stand-in): it uses the device address found once per device
// by hipGetSymbolAddress.
constexpr size_t kNoAllocMeshBytes = 256;
constexpr size_t kNoAllocBytes =
    kNoAllocMeshBytes + size_t(kNoAllocMaxClusters) * size_t(4 + 4) * sizeof(double);
static_assert(sizeof(EnergyMesh) <= kNoAllocMeshBytes, "mesh descriptor slot");
static __device__ __align__(256) unsigned char scratch[kNoAllocBytes];

constexpr int kNoAllocMaxDevices = 64;

// Device address of `scratch` on the current device (looked up once per device).
hipError_t noalloc_scratch(unsigned char** out) {
  static std::mutex mu;
  static unsigned char* ptr[kNoAllocMaxDevices] = {};
  int dev = 0;
  hipError_t err = hipGetDevice(&dev);
  if (err != hipSuccess) return err;
  if (dev < 0 || dev >= kNoAllocMaxDevices) return hipErrorInvalidDevice;
  std::lock_guard<std::mutex> lock(mu);
  if (!ptr[dev]) {
    void* p = nullptr;
    err = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (err != hipSuccess) return err;
    ptr[dev] = static_cast<unsigned char*>(p);
  }
  *out = ptr[dev];
  return hipSuccess;
}

__global__ void ke_set_mesh(EnergyMesh m, EnergyMesh* dst) { *dst = m; }

}  // namespace

hipError_t energy_forward_cvt_noalloc(hipStream_t s, int64_t n, int32_t K, const float* xyz, const float* w,
                                      const int32_t* labels, double* energy) {
  unsigned char* base = nullptr;
  hipError_t err = noalloc_scratch(&base);
  if (err != hipSuccess) return err;
  EnergyMesh* mesh = reinterpret_cast<EnergyMesh*>(base);
  double* acc = reinterpret_cast<double*>(base + kNoAllocMeshBytes);
  EnergyArgs a{};
  a.n_items = n;
  a.n_clusters = K;
  a.meshes = mesh;
  a.xyz = xyz;
  a.w = w;
  a.labels = labels;
  a.acc = acc;
  a.acc_stride = 4;
  a.pts = acc + size_t(kNoAllocMaxClusters) * 4;
  // the descriptor is written by a kernel (no host copy: the call may be captured)
  hipLaunchKernelGGL(ke_set_mesh, dim3(1), dim3(1), 0, s, EnergyMesh{0, n, 0, 0, K, 0, 0, 0}, mesh);
  return energy_forward(s, a, energy, 1);
}

hipError_t energy_backward(hipStream_t s, const EnergyArgs& a, const double* grad_energy, float* dxyz, float* dw) {
  if (a.n_items > 0) {
    const auto k = a.adj ? (a.many ? ke_item_grad<true, true> : ke_item_grad<true, false>)
                         : (a.many ? ke_item_grad<false, true> : ke_item_grad<false, false>);
    hipLaunchKernelGGL(k, dim3(egrid(a.n_items)), dim3(kEBlock), 0, s, a, grad_energy, dxyz, dw);
  }
  return hipGetLastError();
}

}  // namespace acvd

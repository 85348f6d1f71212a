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

// What the kernels over items use of a mesh.  A block whose items lie in one mesh
// reads it once; in another each lane reads its own item's (its meshes taken one
// after the other, a pass of the block each, batches of small meshes took several
// times as long: forward and backward of 33,333 QEM meshes of 12 vertices 720 us,
// by lane 112, 3,125 of 128 115 / 78, 64 of 4,095 54 / 46).
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

// kRingChunk ring entries of item i from entry `from` on (64 consecutive items per
// wave: i = 64 g + lane), loaded together; returns the group's slots.
__device__ inline int32_t load_ring(const EnergyArgs& a, int64_t i, int from, int32_t e[kRingChunk]) {
  const int64_t g = __builtin_amdgcn_readfirstlane(int32_t(i >> 6));
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int k = 0; k < kRingChunk; ++k) e[k] = kRingEnd;
  if (64 * g >= a.n_items) return 0;  // a wave past the last group
  const int2 slot = a.ring_slot[g];  // a scalar load
  const int32_t s0 = slot.x, n = slot.y;
#pragma unroll
  for (int k = 0; k < kRingChunk; ++k)
    if (from + k < n) e[k] = a.ring[int64_t(s0 + from + k) * 64 + lane];
  return n;
}

// The faces of a vertex with more faces than a ring holds, from its vertex -> face
// row: visit(n, v1, v2) takes kFaceBatch of them at a time, n real ones in the
// face's orientation behind the vertex.  A face listed more than once for the
// vertex (a degenerate one, whose normal is zero) takes its first corner.
constexpr int kFaceBatch = 4;
template <class Visit>
__device__ inline void walk_faces(const EnergyArgs& a, int64_t i, Visit&& visit) {
  const int32_t begin = a.vfptr[i], end = a.vfptr[i + 1];
  for (int32_t base = begin; base < end; base += kFaceBatch) {
    int32_t v1[kFaceBatch], v2[kFaceBatch];
#pragma unroll
    for (int k = 0; k < kFaceBatch; ++k) {
      const int64_t f = a.vfcol[min(base + k, end - 1)];
      const int32_t t0 = a.tri[3 * f], t1 = a.tri[3 * f + 1], t2 = a.tri[3 * f + 2];
      const int j = t0 == int32_t(i) ? 0 : t1 == int32_t(i) ? 1 : 2;
      v1[k] = j == 0 ? t1 : j == 1 ? t2 : t0;
      v2[k] = j == 0 ? t2 : j == 1 ? t0 : t1;
    }
    visit(min(end - base, kFaceBatch), v1, v2);
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
__global__ void ke_set_mesh(EnergyMesh m, EnergyMesh* dst) { *dst = m; }

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

// Sorts a vertex -> face row by face id (heap sort: a row of any length in
// n log n steps), so that a ring does not depend on the order of the atomics.
__device__ inline void sort_row(int32_t* r, int32_t len) {
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

__global__ void ke_vf_sort(int64_t n, const int32_t* __restrict__ vfptr, int32_t* vfcol) {
  const int64_t v = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (v < n) sort_row(vfcol + vfptr[v], vfptr[v + 1] - vfptr[v]);
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

// Entries of the ring of vertex v (0 past the end and outside QEM meshes).
template <class Emit>
__device__ inline int ring_of(const EnergyArgs& a, int64_t v, Emit&& emit) {
  if (v >= a.n_items || a.meshes[mesh_of(a, v)].metric != 1) return 0;
  if (a.vfptr[v + 1] - a.vfptr[v] <= kRingFaces) return ring_chains(a, v, emit);
  emit(0, kRingLong);
  return 1;
}

__device__ inline int wave_max(int n) {
  for (int off = 32; off > 0; off >>= 1) n = max(n, __shfl_xor(n, off));
  return n;
}

// Slots of each group of 64 vertices: the longest ring of its QEM vertices.
__global__ __launch_bounds__(64) void ke_ring_slots(EnergyArgs a, int32_t* slots) {
  const int n = wave_max(ring_of(a, int64_t(blockIdx.x) * 64 + threadIdx.x, [](int, int32_t) {}));
  if (threadIdx.x == 0) slots[blockIdx.x] = n;
}

__global__ __launch_bounds__(64) void ke_ring_fill(EnergyArgs a, const int32_t* start, int2* ring_slot, int32_t* ring) {
  const int32_t s0 = start ? start[blockIdx.x] : ring_slot[blockIdx.x].x;
  int32_t* r = ring + int64_t(s0) * 64 + threadIdx.x;
  int n = ring_of(a, int64_t(blockIdx.x) * 64 + threadIdx.x, [&](int k, int32_t e) { r[int64_t(k) * 64] = e; });
  const int most = wave_max(n);
  for (; n < most; ++n) r[int64_t(n) * 64] = kRingEnd;
  if (threadIdx.x == 0) ring_slot[blockIdx.x] = make_int2(s0, most);
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
// latency at 4 waves per SIMD: 16.8 M QEM vertices 2328 -> 377 us (a copy of the
// bytes takes 168 us), 1 M isotropic ones 45.7 -> 16.7 us.
template <bool kQem>
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
  const int m0 = mesh_of(a, begin);
  const bool one = m0 == mesh_of(a, end - 1);  // block-uniform
  ItemMesh im = item_mesh(a.meshes[m0]);
  const bool rings = kQem && (!one || im.qem);
  int32_t e[kRingChunk];
  int32_t slots = 0, lab = -1, mi = m0;
  // the ring entries, labels and meshes of a step are read during the step before it
  if (rings) slots = load_ring(a, begin + threadIdx.x, 0, e);
  if (begin + int64_t(threadIdx.x) < end) {
    lab = a.labels[begin + threadIdx.x];
    if (!one) mi = a.item_mesh[begin + threadIdx.x];
  }
  if (!one) im = item_mesh(a.meshes[mi]);
  int step = 0;
  for (int64_t base = begin; base < end; base += kAccBlock) {
    const int64_t i = base + threadIdx.x;
    const int32_t c = i < end ? cluster_of(im, lab) : -1;
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
    if (base + kAccBlock < end) {
      if (rings) slots = load_ring(a, i + kAccBlock, 0, e);
      lab = i + kAccBlock < end ? a.labels[i + kAccBlock] : -1;
      if (!one && i + kAccBlock < end) mi = a.item_mesh[i + kAccBlock];
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
        if (more && e0 != kRingLong) {
          int32_t f[kRingChunk];
          for (int from = kRingChunk; from < cur_slots; from += kRingChunk) {
            load_ring(a, i, from, f);
            if (f[0] == kRingEnd) break;
#pragma unroll
            for (int k = 0; k < kRingChunk; ++k) {
              const int64_t j = f[k] == kRingEnd ? i : int64_t(f[k] & kRingId);
              q[k] = RingPoint{a.xyz[3 * j], a.xyz[3 * j + 1], a.xyz[3 * j + 2]};
            }
#pragma unroll
            for (int k = 0; k < kRingChunk; ++k) {
              const Vec3 t = sub(Vec3{double(q[k].x), double(q[k].y), double(q[k].z)}, x);
              if (f[k] >= 0) add(cross(u, t));
              u = t;
            }
          }
        } else if (more) {
          walk_faces(a, i, [&](int n, const int32_t* v1, const int32_t* v2) {
            Vec3 r[kFaceBatch], t[kFaceBatch];
#pragma unroll
            for (int k = 0; k < kFaceBatch; ++k) {
              r[k] = sub(load_point(a.xyz, v1[k]), x);
              t[k] = sub(load_point(a.xyz, v2[k]), x);
            }
#pragma unroll
            for (int k = 0; k < kFaceBatch; ++k)
              if (k < n) add(cross(r[k], t[k]));
          });
        }
        // every plane passes through the vertex (d = -n . x): sum n d = -(sum n n^T) x
        v[7] = -(v[4] * x.x + v[5] * x.y + v[6] * x.z);
        v[10] = -(v[5] * x.x + v[8] * x.y + v[9] * x.z);
        v[12] = -(v[6] * x.x + v[9] * x.y + v[11] * x.z);
      }
    }
    if (!one) im = item_mesh(a.meshes[mi]);  // of the next step
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
__global__ __launch_bounds__(kAccBlock) void ke_energy(EnergyArgs a, int64_t chunk, double* energy) {
  constexpr int kWaves = kAccBlock / 64;
  constexpr int kLoopMeshes = 3;  // a block of so few meshes takes them one after the other
  __shared__ double red[kWaves];
  __shared__ int32_t mesh[kWaves];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int64_t begin = int64_t(blockIdx.x) * chunk;
  const int64_t end = min(begin + chunk, a.n_items);
  auto term = [&](const ItemMesh& im, int64_t i) {
    const int32_t c = cluster_of(im, a.labels[i]);
    const Vec3 x = load_point(a.xyz, i);
    const double w = double(a.w[i]);
    double t = 0.0;
    if (c >= 0) {
      const double* q = a.pts + 4 * int64_t(c);
      const double dx = x.x - q[0], dy = x.y - q[1], dz = x.z - q[2];
      t = w * (dx * dx + dy * dy + dz * dz);
    }
    return t;
  };
  double e = 0.0;
  auto wave_sum = [&]() {
    for (int off = 32; off > 0; off >>= 1) e += __shfl_xor(e, off);
  };
  const int m0 = mesh_of(a, begin), m1 = mesh_of(a, end - 1);
  if (m1 - m0 < kLoopMeshes) {  // block-uniform
    for (int m = m0; m <= m1; ++m) {
      const EnergyMesh em = a.meshes[m];
      const ItemMesh im = item_mesh(em);
      const int64_t last = min(end, em.item_off + em.n_items);
      e = 0.0;
#pragma unroll 4
      for (int64_t i = max(begin, em.item_off) + threadIdx.x; i < last; i += kAccBlock) e += term(im, i);
      wave_sum();
      __syncthreads();  // red of the previous mesh has been read
      if (lane == 0) red[wave] = e;
      __syncthreads();
      if (threadIdx.x == 0) {
        for (int k = 1; k < kWaves; ++k) e += red[k];
        atomicAdd(&energy[m], e);
      }
    }
    return;
  }
  // a wave adds up the items of one mesh (cur) while its lanes lie in it, and else
  // the runs of its lanes in each mesh
  int32_t cur = -1;
  for (int64_t base = begin; base < end; base += kAccBlock) {
    const int64_t i = base + threadIdx.x;
    const int32_t m = i < end ? a.item_mesh[i] : -1;
    double t = m >= 0 ? term(item_mesh(a.meshes[m]), i) : 0.0;
    const int32_t first = __builtin_amdgcn_readfirstlane(m);
    if (__ballot(m != first) == 0ull) {
      if (first != cur) {
        wave_sum();
        if (lane == 0 && cur >= 0) atomicAdd(&energy[cur], e);
        e = 0.0;
        cur = first;
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
  if (threadIdx.x == 0)
    for (int k = 0; k < kWaves;) {  // one atomic for neighbouring waves of one mesh
      const int32_t m = mesh[k];
      double sum = 0.0;
      for (; k < kWaves && mesh[k] == m; ++k) sum += red[k];
      if (m >= 0) atomicAdd(&energy[m], sum);
    }
}

// The whole forward of one small isotropic mesh in one block: sums, points and
// energy in turn, the sums in LDS by cluster.  The four launches of the general
// forward cost the host more than this block takes (2,562 vertices, a call from
// Python: 21.8 -> 13.4 us).  On the device alone one block / four launches take 3.5 /
// 8.2 us at 64 items, 5.8 / 9.4 at 2,562, 7.4 / 9.4 at 4,096 (random labels 10.1 /
// 10.0), 11.8 / 9.4 at 8,192 (17.2 / 10.0): the line is at 4,096; the clusters' sums
// of kSmallClusters take 32 KB of LDS.
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
// 306 -> 266, 42 a cluster 708 -> 715).  A ring of more than eight entries takes
// them eight at a time, faces past 32 come four at a time from the vertex's row (one
// by one behind its loads, and from the row past 16: a sphere of 368,642 vertices of
// valence 3 to 24, labels of a clustering, 303 us, so 95; the forward 232, 101).  Consecutive blocks run on one XCD, whose
// L2 then holds the rows a block shares with its neighbours (HBM reads 1.27 ->
// 0.89 GB).  Bound by the f64 work (980
// instructions per 64 vertices, half of the time) and by gather latency at 3
// waves per SIMD (168 registers; held to 128 the spills cost more: 1359 us;
// a loop over the faces that keeps one position in flight: 831 us).
// 16.8 M QEM vertices 2050 -> 752 us, 1 M isotropic ones 10.5 -> 8.6 us.
template <bool kQem>
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
  if constexpr (kQem) slots = load_ring(a, i, 0, e);
  const int m0 = mesh_of(a, begin);
  const bool one = m0 == mesh_of(a, end - 1);  // block-uniform
  // (a build of it with the mesh in scalar registers and one without)
  auto grad = [&](const ItemMesh& em, double g) {
    const bool active = i < end;
    double gx[3] = {0, 0, 0}, gw = 0.0;
    const int32_t c = active ? cluster_of(em, lab) : -1;
    const bool qem = kQem && em.qem;
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
      auto adjoint_of = [&](int32_t cl) {
        return cl >= 0 ? plane_adjoint(a.adj + kAdjStride * int64_t(cl), x) : no_adjoint();
      };
      const bool is_long = e[0] == kRingLong;
      // kRingChunk entries at a time; a further chunk starts at the last entry of the
      // one before, whose face with the next entry it takes
      for (int from = 0;;) {
        // clusters of the entries: bit k of own_bits the vertex's own, of todo another
        // one whose part is still to be taken
        const bool more = !is_long && slots - from > kRingChunk && e[kRingChunk - 1] != kRingEnd;
        int32_t cl[kRingChunk];
        uint32_t own_bits = 0, todo = 0;
#pragma unroll
        for (int k = 0; k < kRingChunk; ++k) {
          if (k >= slots - from) break;  // wave-uniform
          if (e[k] == kRingEnd || is_long) e[k] = int32_t(uint32_t(i) | 0x80000000u);  // no face
          cl[k] = a.labels[e[k] & kRingId];
        }
#pragma unroll
        for (int k = 0; k < kRingChunk; ++k) {
          if (k >= slots - from) break;
          cl[k] = cluster_of(em, cl[k]);
          if (cl[k] >= 0) (cl[k] == c ? own_bits : todo) |= 1u << k;
        }
        PlaneAdjoint A0 = adjoint_of(c);
        double own = c >= 0 ? 1.0 : 0.0;
        Vec3 u{0.0, 0.0, 0.0};
        while (true) {
          int32_t c1 = -1, c2 = -1;
          uint32_t bits1 = 0, bits2 = 0;
#pragma unroll
          for (int k = 0; k < kRingChunk; ++k) {
            if (k >= slots - from) break;
            if (!(todo >> k & 1u)) continue;
            if (c1 < 0) c1 = cl[k];
            if (cl[k] == c1) bits1 |= 1u << k;
            else {
              if (c2 < 0) c2 = cl[k];
              if (cl[k] == c2) bits2 |= 1u << k;
            }
          }
          todo &= ~(bits1 | bits2);
          const PlaneAdjoint A1 = adjoint_of(c1), A2 = adjoint_of(c2);
#pragma unroll
          for (int k = 0; k < kRingChunk; ++k) {
            if (k >= slots - from) break;
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
        if (!more) break;
        from += kRingChunk - 1;
        load_ring(a, i, from, e);
      }
      if (is_long) {
        const PlaneAdjoint A0 = adjoint_of(c);
        walk_faces(a, i, [&](int n, const int32_t* v1, const int32_t* v2) {
          Vec3 r[kFaceBatch], t[kFaceBatch];
          int32_t c1[kFaceBatch], c2[kFaceBatch];
#pragma unroll
          for (int k = 0; k < kFaceBatch; ++k) {
            r[k] = sub(load_point(a.xyz, v1[k]), x);
            t[k] = sub(load_point(a.xyz, v2[k]), x);
            c1[k] = a.labels[v1[k]];
            c2[k] = a.labels[v2[k]];
          }
#pragma unroll
          for (int k = 0; k < kFaceBatch; ++k) {
            if (k >= n) break;
            const PlaneAdjoint A1 = adjoint_of(cluster_of(em, c1[k])), A2 = adjoint_of(cluster_of(em, c2[k]));
            PlaneAdjoint F;
            for (int j = 0; j < 6; ++j) F.m[j] = A0.m[j] + A1.m[j] + A2.m[j];
            for (int j = 0; j < 3; ++j) F.g[j] = A0.g[j] + A1.g[j] + A2.g[j];
            pull(F, r[k], t[k]);
          }
        });
      }
    }
    if (active) {
      for (int k = 0; k < 3; ++k) dxyz[3 * i + k] = float(g * gx[k]);
      dw[i] = float(g * gw);
    }
  };
  if (one) {
    grad(item_mesh(a.meshes[m0]), gE[m0]);
  } else {
    const int32_t m = a.item_mesh[ic];
    grad(item_mesh(a.meshes[m]), gE[m]);
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
    const auto k = a.adj ? ke_accumulate<true> : ke_accumulate<false>;
    hipLaunchKernelGGL(k, grid, dim3(kAccBlock), 0, s, a, chunk);
  }
  if (a.n_clusters > 0)
    hipLaunchKernelGGL(ke_points, dim3(unsigned((a.n_clusters + 63) / 64)), dim3(64), 0, s, a);
  if (a.n_items > 0) {
    const int64_t chunk = item_chunk(a.n_items, 512);
    hipLaunchKernelGGL(ke_energy, dim3(unsigned((a.n_items + chunk - 1) / chunk)), dim3(kAccBlock), 0, s, a, chunk,
                       energy);
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

hipError_t energy_ring_fill(hipStream_t s, const EnergyArgs& a, const int32_t* start, int2* ring_slot, int32_t* ring) {
  hipLaunchKernelGGL(ke_ring_fill, dim3(unsigned((a.n_items + 63) / 64)), dim3(64), 0, s, a, start, ring_slot, ring);
  return hipGetLastError();
}

hipError_t energy_set_mesh(hipStream_t s, const EnergyMesh& m, EnergyMesh* dst) {
  hipLaunchKernelGGL(ke_set_mesh, dim3(1), dim3(1), 0, s, m, dst);
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
  err = energy_set_mesh(s, EnergyMesh{0, n, 0, 0, K, 0, 0, 0}, mesh);
  return err != hipSuccess ? err : energy_forward(s, a, energy, 1);
}

hipError_t energy_backward(hipStream_t s, const EnergyArgs& a, const double* grad_energy, float* dxyz, float* dw) {
  if (a.n_items > 0) {
    const auto k = a.adj ? ke_item_grad<true> : ke_item_grad<false>;
    hipLaunchKernelGGL(k, dim3(egrid(a.n_items)), dim3(kEBlock), 0, s, a, grad_energy, dxyz, dw);
  }
  return hipGetLastError();
}

}  // namespace acvd

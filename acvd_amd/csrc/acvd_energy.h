// Device layout of the fixed-assignment energy (k_energy.hip): meshes packed
// back to back, items [item_off, item_off + n), clusters [clus_off, + K),
// faces [face_off, + nf) with global vertex ids.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace acvd {

struct EnergyMesh {
  int64_t item_off;
  int64_t n_items;
  int64_t clus_off;
  int64_t face_off;
  int32_t K;
  int32_t metric;  // 0 isotropic (CVT), 1 QEM
  int32_t level;   // rank truncation of the QEM point
  int32_t pad;
};

struct EnergyArgs {
  int64_t n_items;
  int64_t n_clusters;
  const EnergyMesh* meshes;
  const int32_t* item_mesh;  // null for one mesh
  const int32_t* clus_mesh;  // null for one mesh
  const int32_t* tri;        // 3 global vertex ids per face (contexts with QEM meshes; else null)
  const int32_t* vfptr;      // vertex -> incident faces, one entry per corner
  const int32_t* vfcol;
  // rings (faces around each QEM vertex as chains of neighbour ids): group g of
  // 64 items holds ring_slot[g].y slots of 64 ids from slot ring_slot[g].x on
  const int2* ring_slot;
  const int32_t* ring;
  // inputs of one call
  const float* xyz;          // 3 per item
  const float* w;            // 1 per item
  const int32_t* labels;     // mesh-local cluster ids, K or out of range = none
  // state kept from the forward for the backward
  int32_t acc_stride;        // 13 with QEM meshes, else 4
  double* acc;               // per cluster: W, S[3] and (QEM) Q[9]
  double* pts;               // 4 per cluster: point, unused
  double* adj;               // kAdjStride per cluster (null without QEM meshes): for a unit gradient
                             // dE/dQ[9], (dE/dc)/W [3]; centroid [3]
};

constexpr int kAdjStride = 16;
// Ring entries: a neighbour id; with the sign bit set the first id of a chain;
// kRingEnd past the end; kRingLong (first entry alone) for a vertex of more than
// kRingFaces faces, whose faces are read from its vertex -> face row.
constexpr int32_t kRingEnd = -1;
constexpr int32_t kRingLong = -2;
constexpr int32_t kRingId = 0x7fffffff;
constexpr int kRingFaces = 32;
constexpr int kRingChunk = 8;  // ids read at once

// Device build of the vertex -> face rows and rings.
hipError_t energy_offset_tri(hipStream_t s, int64_t n3, int32_t off, int32_t* tri);
hipError_t energy_vf_count(hipStream_t s, int64_t n3, const int32_t* tri, int32_t* deg);
hipError_t energy_vf_fill(hipStream_t s, int64_t n, int64_t n3, const int32_t* tri, const int32_t* vfptr,
                          int32_t* fill, int32_t* vfcol);
hipError_t energy_ring_slots(hipStream_t s, const EnergyArgs& a, int32_t* slots);
// start: first slot of each group; null: those in ring_slot[g].x
hipError_t energy_ring_fill(hipStream_t s, const EnergyArgs& a, const int32_t* start, int2* ring_slot, int32_t* ring);
hipError_t energy_set_mesh(hipStream_t s, const EnergyMesh& m, EnergyMesh* dst);

hipError_t energy_forward(hipStream_t s, const EnergyArgs& a, double* energy, int n_meshes);
// Largest cluster count of energy_forward_cvt_noalloc (its static scratch).
constexpr int32_t kNoAllocMaxClusters = 65536;
// energy_forward for one isotropic mesh with every per-call buffer in the
// library's static device scratch of the current device (no allocation).
hipError_t energy_forward_cvt_noalloc(hipStream_t s, int64_t n, int32_t K, const float* xyz, const float* w,
                                      const int32_t* labels, double* energy);
hipError_t energy_backward(hipStream_t s, const EnergyArgs& a, const double* grad_energy, float* dxyz, float* dw);

}  // namespace acvd

// Element clusters and their slots on the device, as the cluster passes of the
// fused step and of the adjoint read them (plan: wfx_cluster.hpp).
#pragma once

#include "wfx_cluster.hpp"
#include "wfx_internal.hpp"

namespace wfx {
namespace {

// Slots each thread of a cluster pass stages (slot_cap = kSlotsPerThread *
// kCluster): the staging rows past the cluster's slot count are written with
// a repeat of its last slot and never read, so that no load or store of the
// staging waits behind a branch
template <int NN>
constexpr int kSlotsPerThread = slot_cap(NN) / kCluster;

// Cluster tables of the fused element pass on the device (wfx_cluster.hpp)
struct ClusterArgs {
  const ClusterDesc *desc;  // this and the tables as DevMesh::cl_*
  const uint16_t *goff;
  const uint2 *ent;
  const int *snode;      // [S] slot -> node
  const uint16_t *lslot;
  const int *nrel;
  const int *spos;       // [S] slot -> where its partial sum is stored when node-major
  long S;                // slots: the row length of the partial sums
  int nm;                // partial sums node-major (FP32-mixed always, FP64 with the paired passes)
};

inline ClusterArgs cluster_args(const wfx_ctx *c) {
  return ClusterArgs{c->ms.cl_desc, c->ms.cl_goff, c->ms.cl_ent, c->ms.cl_snode,
                     c->ms.cl_lslot, c->ms.cl_nrel, c->ms.spos, c->ms.nslot, c->ms.spos != nullptr};
}

// One element's nodes as slot indices of its cluster (a 16- or 8-byte load)
template <int NN>
__device__ __forceinline__ void load_lslot(const uint16_t *p, int (&ls)[NN]) {
  typedef unsigned int u32v __attribute__((ext_vector_type(NN / 2)));
  const u32v w = *reinterpret_cast<const u32v *>(p);  // clusters share the table
#pragma unroll
  for (int k = 0; k < NN / 2; ++k) {
    ls[2 * k] = (int)(w[k] & 0xffffu);
    ls[2 * k + 1] = (int)(w[k] >> 16);
  }
}

}  // namespace
}  // namespace wfx

// Per-frame refit kernels for gfx950.
//
// The refit is DynBVH::updateBounds<false> without rotations (DynBVH.cc:2084-2117), done
// level-synchronously:
//   k_refit_slots: one lane per object slot rebuilds the slot's triangle record from the
//     current vertices; the lane at a leaf's first slot forms the leaf box from its slots'
//     boxes (Mesh::getBBox + BBox::extendByBox, Model/Groups/Mesh.cc:228-237,
//     DynBVH.cc:2091-2097). Loaded trees whose leaves do not partition the slots take
//     k_refit_leaves, one lane per leaf record, instead;
//   k_refit_level: one launch per even depth, deepest first; each lane unions the boxes of
//     one inner record's children that are inner records (the odd depth below), then its
//     own two child boxes (DynBVH.cc:2110-2116), and stores the four boxes of its wide node;
//   k_refit_top: the small depths at the top of the tree (even depths of at most kTopNodes
//     records) in one workgroup, deepest first, with a barrier between depths.
// Kernel boundaries on the stream order the levels, so no cross-workgroup synchronisation
// is needed (agent-scope acquire/release would write back and invalidate the per-XCD L2s).
// Box arithmetic is exact (min/max of the same fp32 values), so the result is
// bit-identical to a serial recomputation.

#include <hip/hip_runtime.h>

#include <cfloat>

#include "mh_device.h"
#include "prim_setup.h"
#include "wide_node.h"

namespace mh {
namespace {

constexpr int kBlock = 256;

__device__ __forceinline__ float pick_lo(float a, float b) { return a < b ? a : b; }
__device__ __forceinline__ float pick_hi(float a, float b) { return a > b ? a : b; }


__device__ __forceinline__ void write_record(const DevRefit& r, int slot, const Tri& t) {
  store_tri_record(r.tris, r.prim_kind, slot, t);
}

__global__ __launch_bounds__(kBlock) void k_prim_setup(DevRefit r) {
  const int64_t s = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (s >= r.n_slots) return;
  write_record(r, (int)s, load_tri(r.verts, r.idx, r.obj_ids[s]));
}

__device__ __forceinline__ void store_box(const DevRefit& r, int rec, const NodeBox& b) {
  RefNode* nd = r.refs + rec;
  *reinterpret_cast<float4*>(nd) = make_float4(b.lo[0], b.lo[1], b.lo[2], b.hi[0]);
  *reinterpret_cast<float2*>(reinterpret_cast<float*>(nd) + 4) = make_float2(b.hi[1], b.hi[2]);
}

// Adds triangle t's box to leaf box b.
__device__ __forceinline__ void extend_tri(NodeBox& b, const Tri& t) {
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    const float tlo = pick_lo(pick_lo(t.p[0][a], t.p[1][a]), t.p[2][a]);
    const float thi = pick_hi(pick_hi(t.p[0][a], t.p[1][a]), t.p[2][a]);
    b.lo[a] = pick_lo(b.lo[a], tlo);
    b.hi[a] = pick_hi(b.hi[a], thi);
  }
}

__device__ __forceinline__ void store_leaf_box(const DevRefit& r, int rec, const NodeBox& b) {
  store_box(r, rec, b);
  bool nan = false;
#pragma unroll
  for (int a = 0; a < 3; ++a) nan = nan || b.lo[a] != b.lo[a] || b.hi[a] != b.hi[a];
  if (nan) r.irregular[1] = 1;
}

__global__ __launch_bounds__(kBlock) void k_refit_leaves(DevRefit r) {
  const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (i >= r.n_leaves) return;
  const int rec = r.leaves[i];
  const int first = r.refs[rec].child, count = r.refs[rec].children;
  NodeBox b = empty_box();
  for (int k = 0; k < count; ++k) {
    const Tri t = load_tri(r.verts, r.idx, r.obj_ids[first + k]);
    write_record(r, first + k, t);
    extend_tri(b, t);
  }
  store_leaf_box(r, rec, b);
}

// The gathers of a leaf list's lanes scatter over the mesh and chain their leaf's objects;
// by slots each lane gathers one triangle, beside its neighbours' (they lie close together
// in leaf order), once for the record and the box, and a leaf reads its other objects'
// boxes from LDS. Only a leaf that runs past its workgroup's slots gathers those again.
// 8M-triangle heightfield: 477 us by leaves, 228 us by slots (1.08 GB moved, 4.5 TB/s).
__global__ __launch_bounds__(kBlock) void k_refit_slots(DevRefit r) {
  __shared__ float s_lo[3][kBlock], s_hi[3][kBlock];
  const int tid = threadIdx.x;
  const int64_t i = (int64_t)blockIdx.x * kBlock + tid;
  int rec = -1;
  if (i < r.n_slots) {
    const Tri t = load_tri(r.verts, r.idx, r.obj_ids[i]);
    rec = r.leaf_at[i];
    write_record(r, (int)i, t);
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      s_lo[a][tid] = pick_lo(pick_lo(t.p[0][a], t.p[1][a]), t.p[2][a]);
      s_hi[a][tid] = pick_hi(pick_hi(t.p[0][a], t.p[1][a]), t.p[2][a]);
    }
  }
  __syncthreads();
  if (rec < 0) return;
  const int count = r.refs[rec].children;
  NodeBox b = empty_box();
  const int here = count < kBlock - tid ? count : kBlock - tid;
  for (int k = 0; k < here; ++k) {
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      b.lo[a] = pick_lo(b.lo[a], s_lo[a][tid + k]);
      b.hi[a] = pick_hi(b.hi[a], s_hi[a][tid + k]);
    }
  }
  for (int k = here; k < count; ++k) extend_tri(b, load_tri(r.verts, r.idx, r.obj_ids[i + k]));
  store_leaf_box(r, rec, b);
}

// Entry `e` of an even level list: the boxes of its record and of that record's inner
// children, and its wide node's planes.
__device__ __forceinline__ void refit_entry(const DevRefit& r, int64_t e) {
  const int rec = r.levels[e];
  const int c = r.refs[rec].child;
  NodeBox own[2], slot[4];
#pragma unroll
  for (int side = 0; side < 2; ++side) {
    const NodeWords w = load_node(r.refs, c + side);
    if (node_children(w) != 0) {
      own[side] = slot[2 * side] = node_box(w);
      slot[2 * side + 1] = empty_box();
    } else {
      slot[2 * side] = node_box(load_node(r.refs, node_child(w)));
      slot[2 * side + 1] = node_box(load_node(r.refs, node_child(w) + 1));
      own[side] = unite_boxes(slot[2 * side], slot[2 * side + 1]);
      store_box(r, c + side, own[side]);
    }
  }
  store_box(r, rec, unite_boxes(own[0], own[1]));
  store_planes(r.wide + e, slot);
}

__global__ __launch_bounds__(kBlock) void k_refit_level(DevRefit r, int64_t first, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (i >= n) return;
  refit_entry(r, first + i);
}

// The top even depths, deepest first, in one workgroup with a barrier between depths (its
// waves share one compute unit and its L1, so the boxes stored before the barrier are
// seen by the loads after it). The last launch of a refit: it takes the leaf pass's NaN
// mark over for the traces that follow.
__global__ __launch_bounds__(kBlock) void k_refit_top(DevRefit r, TopLevels t) {
  for (int d = t.n - 1; d >= 0; --d) {
    for (int i = (int)threadIdx.x; i < t.cnt[d]; i += kBlock) refit_entry(r, t.first[d] + i);
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    r.irregular[0] = r.fixed | (r.irregular[1] != 0);
    r.irregular[1] = 0;
  }
}

__global__ __launch_bounds__(kBlock) void k_displace_sine(float* verts, const float* base,
                                                          int64_t n, float amp, float freq,
                                                          float phase) {
  const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (i >= n) return;
  const float x = base[3 * i + 0];
  verts[3 * i + 0] = x;
  verts[3 * i + 1] = base[3 * i + 1] + amp * sinf(freq * x + phase);
  verts[3 * i + 2] = base[3 * i + 2];
}

}  // namespace

int launch_prim_setup(const DevRefit& r, void* stream) {
  if (r.n_slots <= 0) return 0;
  const unsigned blocks = (unsigned)((r.n_slots + kBlock - 1) / kBlock);
  hipLaunchKernelGGL(k_prim_setup, dim3(blocks), dim3(kBlock), 0,
                     reinterpret_cast<hipStream_t>(stream), r);
  return (int)hipGetLastError();
}

int launch_refit(const DevRefit& r, const LevelList* lev, int n_levels, void* stream) {
  if (r.n_leaves <= 0) return 0;
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  auto grid = [](int64_t n) { return dim3((unsigned)((n + kBlock - 1) / kBlock)); };
  if (r.leaf_at)
    hipLaunchKernelGGL(k_refit_slots, grid(r.n_slots), dim3(kBlock), 0, s, r);
  else
    hipLaunchKernelGGL(k_refit_leaves, grid(r.n_leaves), dim3(kBlock), 0, s, r);
  TopLevels t;
  const int top = 2 * top_levels(lev, n_levels, 2, t);
  for (int d = (n_levels - 1) & ~1; d >= top; d -= 2)
    if (lev[d].n > 0)
      hipLaunchKernelGGL(k_refit_level, grid(lev[d].n), dim3(kBlock), 0, s, r, lev[d].first,
                         lev[d].n);
  // (also where the root is a leaf and there is no level: the NaN mark)
  hipLaunchKernelGGL(k_refit_top, dim3(1), dim3(kBlock), 0, s, r, t);
  return (int)hipGetLastError();
}

int launch_displace_sine(float* verts, const float* base, int64_t n_verts, float amp, float freq,
                         float phase, void* stream) {
  if (n_verts <= 0) return 0;
  const unsigned blocks = (unsigned)((n_verts + kBlock - 1) / kBlock);
  hipLaunchKernelGGL(k_displace_sine, dim3(blocks), dim3(kBlock), 0,
                     reinterpret_cast<hipStream_t>(stream), verts, base, n_verts, amp, freq,
                     phase);
  return (int)hipGetLastError();
}

}  // namespace mh

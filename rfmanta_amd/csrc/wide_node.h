// Wide nodes from reference records (mh_device.h), shared by the refit and the passes that
// write a new tree's nodes.
#pragma once

#include <hip/hip_runtime.h>

#include <cfloat>

#include "mh_device.h"

namespace mh {
namespace {

// A record as two 16-byte words: lo.x lo.y lo.z hi.x | hi.y hi.z child word, where word
// holds axis (byte 0), bits (byte 1) and children (int16, bytes 2-3).
struct NodeWords {
  float4 a, b;
};
__device__ __forceinline__ NodeWords load_node(const RefNode* refs, int64_t r) {
  const float4* p = reinterpret_cast<const float4*>(refs + r);
  return NodeWords{p[0], p[1]};
}
__device__ __forceinline__ int node_child(const NodeWords& w) { return __float_as_int(w.b.z); }
__device__ __forceinline__ int node_word(const NodeWords& w) { return __float_as_int(w.b.w); }
__device__ __forceinline__ int node_children(const NodeWords& w) { return node_word(w) >> 16; }

struct NodeBox {
  float lo[3], hi[3];
};
__device__ __forceinline__ NodeBox node_box(const NodeWords& w) {
  return NodeBox{{w.a.x, w.a.y, w.a.z}, {w.a.w, w.b.x, w.b.y}};
}
__device__ __forceinline__ NodeBox empty_box() {
  return NodeBox{{FLT_MAX, FLT_MAX, FLT_MAX}, {-FLT_MAX, -FLT_MAX, -FLT_MAX}};
}
// BBox::extendByBox from an empty box: the select forms of the reference's min and max.
__device__ __forceinline__ NodeBox unite_boxes(const NodeBox& a, const NodeBox& b) {
  NodeBox u;
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    const float l = FLT_MAX < a.lo[k] ? FLT_MAX : a.lo[k];
    u.lo[k] = l < b.lo[k] ? l : b.lo[k];
    const float h = -FLT_MAX > a.hi[k] ? -FLT_MAX : a.hi[k];
    u.hi[k] = h > b.hi[k] ? h : b.hi[k];
  }
  return u;
}

__device__ __forceinline__ void store_planes(WideNode* w, const NodeBox (&s)[4]) {
  float4* p = reinterpret_cast<float4*>(w);
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    p[2 * k] = make_float4(s[0].lo[k], s[1].lo[k], s[2].lo[k], s[3].lo[k]);
    p[2 * k + 1] = make_float4(s[0].hi[k], s[1].hi[k], s[2].hi[k], s[3].hi[k]);
  }
}

}  // namespace
}  // namespace mh

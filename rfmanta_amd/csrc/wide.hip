// Level lists, leaf list, leaf starts and wide nodes of a tree, top down (gfx950), after a
// build, a load or a rotating update.
//
// One pass per even depth: each lane takes one inner record of the depth, reads its two
// children and, of those that are inner records, the grandchildren (64 bytes each), writes
// its wide node, and appends the inner children to the odd level list, the inner
// grandchildren to the even one and the leaves met to the leaf list. A wide node's index is
// its record's place in the even list, so a grandchild's reference is the place it has just
// been given. Beside each even entry lies its record's first child and word, copied when
// the record was read, so that no depth loads its own records again. A workgroup ranks its
// appends with a wave scan over packed counts and takes its ranges with one atomic per list
// and loop iteration; the order inside a list is free, since the nodes of one depth are
// independent. The passes read scattered records and are bound by those reads and, at the
// top, by their latency: the depths that are small run in one workgroup, in one launch.

#include <hip/hip_runtime.h>

#include "mh_device.h"
#include "wide_node.h"

namespace mh {
namespace {

constexpr int kBlock = 256;

// Counts of one lane's appends packed into a word: odd entries (at most 2 a lane, 512 a
// workgroup), even entries and leaves (at most 4 a lane, 1024 a workgroup).
constexpr int kEvenShift = 10, kLeafShift = 21;
__device__ __forceinline__ unsigned odd_of(unsigned p) { return p & 1023u; }
__device__ __forceinline__ unsigned even_of(unsigned p) { return (p >> kEvenShift) & 2047u; }
__device__ __forceinline__ unsigned leaves_of(unsigned p) { return p >> kLeafShift; }

// Order bits of split axis a (WideNode::order, j = 0): set for the octants whose bit a is
// clear.
__device__ __forceinline__ unsigned axis_order(int a) {
  return a == 0 ? 0x041041u : (a == 1 ? 0x009009u : 0x000249u);
}
// Those and the any-hit bit (set unless isLeftCheaper) of a record's word.
__device__ __forceinline__ unsigned word_order(int word) {
  return axis_order(word & 3) | (((word >> 8) & 1) ? 0u : 1u << 24);
}

// Leaf code of a leaf record, with big_count set for leaves of 15 or more objects.
__device__ __forceinline__ int32_t leaf_code(const DevUpdate& u, const NodeWords& w) {
  const int n = node_children(w), first = node_child(w);
  if (n >= kLeafCountInline) u.big_count[first] = n;
  return ~((first << kLeafCountBits) | (n < kLeafCountInline ? n : kLeafCountInline));
}

struct Bases {
  unsigned odd, even, leaf;
};

// One workgroup's share of an even depth whose entries are even[first, first + n): items
// i_begin, i_begin + stride, ... Depth d + 1 starts at odd[first_odd], depth d + 2 at
// even[first + n]; reserve(counts) returns the workgroup's ranges in the three lists.
template <class Reserve>
__device__ __forceinline__ void wide_depth(const DevUpdate& u, const DevFrontier& f,
                                           unsigned first, unsigned n, unsigned first_odd,
                                           unsigned i_begin, unsigned stride, Reserve reserve) {
  __shared__ unsigned s_wave[kBlock / 64];
  __shared__ Bases s_base;
  const unsigned next = first + n;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  for (unsigned i0 = i_begin; i0 < n; i0 += stride) {  // uniform over the workgroup
    const unsigned i = i0 + threadIdx.x, at = first + i;
    // past the capacities only after an overflow (flagged)
    const bool live = i < n && at < f.cap && at < f.cap_wide;
    int2 self = make_int2(0, 0);
    NodeWords kid[2], slot[4];
    bool inner[2] = {false, false}, used[4] = {false, false, false, false};
    unsigned mine = 0;
    if (live) {
      self = f.aux[at];
#pragma unroll
      for (int side = 0; side < 2; ++side) {
        kid[side] = load_node(u.refs, self.x + side);
        inner[side] = node_children(kid[side]) == 0;
      }
#pragma unroll
      for (int side = 0; side < 2; ++side) {
        used[2 * side] = true;
        used[2 * side + 1] = inner[side];
        if (inner[side]) {
          mine += 1u;
          slot[2 * side] = load_node(u.refs, node_child(kid[side]));
          slot[2 * side + 1] = load_node(u.refs, node_child(kid[side]) + 1);
        } else {
          slot[2 * side] = slot[2 * side + 1] = kid[side];
        }
      }
#pragma unroll
      for (int k = 0; k < 4; ++k)
        if (used[k]) mine += node_children(slot[k]) == 0 ? 1u << kEvenShift : 1u << kLeafShift;
    }
    unsigned sum = mine;  // inclusive over the wave
    for (int m = 1; m < 64; m <<= 1) {
      const unsigned y = __shfl_up(sum, m, 64);
      if (lane >= m) sum += y;
    }
    if (lane == 63) s_wave[wave] = sum;
    __syncthreads();
    if (threadIdx.x == 0) {
      unsigned t = 0;
      for (int w = 0; w < kBlock / 64; ++w) {
        const unsigned x = s_wave[w];
        s_wave[w] = t;
        t += x;
      }
      s_base = reserve(t);
    }
    __syncthreads();
    if (live) {
      const unsigned before = s_wave[wave] + sum - mine;
      unsigned po = first_odd + s_base.odd + odd_of(before);
      unsigned pe = next + s_base.even + even_of(before);
      unsigned pl = s_base.leaf + leaves_of(before);
      bool over = false;
      NodeBox box[4];
      int ref[4];
      unsigned order = word_order(self.y);
#pragma unroll
      for (int side = 0; side < 2; ++side)
        if (inner[side]) {
          order |= word_order(node_word(kid[side])) << (1 + side);
          if (po < f.cap)
            f.odd[po] = self.x + side;
          else
            over = true;
          ++po;
        }
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        box[k] = empty_box();
        ref[k] = kWideEmpty;
        if (!used[k]) continue;
        box[k] = node_box(slot[k]);
        const int rec = inner[k >> 1] ? node_child(kid[k >> 1]) + (k & 1) : self.x + (k >> 1);
        if (node_children(slot[k]) == 0) {
          ref[k] = (int)pe;
          if (pe < f.cap && pe < f.cap_wide) {
            f.even[pe] = rec;
            f.aux[pe] = make_int2(node_child(slot[k]), node_word(slot[k]));
          } else {
            over = true;
          }
          ++pe;
        } else {
          ref[k] = leaf_code(u, slot[k]);
          if (pl < f.cap)
            f.leaves[pl] = rec;
          else
            over = true;
          ++pl;
          if (u.leaf_at && node_child(slot[k]) < u.n_objects) u.leaf_at[node_child(slot[k])] = rec;
        }
      }
      if (over) f.fr[kFrOver] = 1u;
      WideNode* w = f.wide + at;
      store_planes(w, box);
      *reinterpret_cast<int4*>(w->ref) = make_int4(ref[0], ref[1], ref[2], ref[3]);
      w->order = order;
    }
    __syncthreads();  // s_wave and s_base are rewritten by the next iteration
  }
}

// The even depths below n_top in one workgroup, from the root: it clears fr, counts in LDS
// (a barrier ends each depth; the workgroup's waves share one compute unit and its L1, so
// the list entries stored before it are seen after it) and leaves the counts and offsets
// of depths 0 .. n_top and the leaf count for the launches of the deeper depths.
__global__ __launch_bounds__(kBlock) void k_wide_top(DevUpdate u, DevFrontier f, int n_top) {
  __shared__ unsigned s_cnt[kTopLevels + 3], s_off[kTopLevels + 3], s_leaf;
  for (int i = threadIdx.x; i < kFrontierWords; i += kBlock) f.fr[i] = 0u;
  if (threadIdx.x == 0) {
    s_cnt[0] = 1u;  // depth 0: the root
    s_off[0] = s_off[1] = 0u;
    s_leaf = 0u;
    f.even[0] = 0;
    const NodeWords root = load_node(u.refs, 0);
    f.aux[0] = make_int2(node_child(root), node_word(root));
    f.irregular[0] = f.fixed | (f.irregular[1] != 0);
    f.irregular[1] = 0;
  }
  __syncthreads();
  for (int d = 0; d < n_top; d += 2) {
    const unsigned n = s_cnt[d], first = s_off[d], first_odd = s_off[d + 1];
    __syncthreads();  // every lane has read the depth's count before lane 0 opens the next
    if (threadIdx.x == 0) {
      s_cnt[d + 1] = s_cnt[d + 2] = 0u;
      s_off[d + 2] = first + n;
    }
    __syncthreads();
    wide_depth(u, f, first, n, first_odd, 0u, kBlock, [&](unsigned t) {
      const Bases b{s_cnt[d + 1], s_cnt[d + 2], s_leaf};
      s_cnt[d + 1] = b.odd + odd_of(t);
      s_cnt[d + 2] = b.even + even_of(t);
      s_leaf = b.leaf + leaves_of(t);
      return b;
    });
    __syncthreads();
    if (threadIdx.x == 0) s_off[d + 3] = first_odd + s_cnt[d + 1];
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    for (int d = 0; d <= n_top; ++d) {
      f.fr[d] = s_cnt[d];
      f.fr[kFrOff + d] = s_off[d];
    }
    f.fr[kFrOff + n_top + 1] = s_off[n_top + 1];
    f.fr[kFrLeaves] = s_leaf;
  }
}

// Even depth d (>= the depths of k_wide_top) over the whole grid, counters in fr.
__global__ __launch_bounds__(kBlock) void k_wide_level(DevUpdate u, DevFrontier f, int d) {
  unsigned* off = f.fr + kFrOff;
  const unsigned n = f.fr[d], first = off[d];
  // (off[d + 1] was left by the depths above, which closed depth d - 1)
  const unsigned first_odd = d > 0 ? off[d - 1] + f.fr[d - 1] : 0u;
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    off[d + 1] = first_odd;
    off[d + 2] = first + n;
  }
  wide_depth(u, f, first, n, first_odd, blockIdx.x * kBlock, gridDim.x * kBlock,
             [&](unsigned t) {
               const unsigned o = odd_of(t), e = even_of(t), l = leaves_of(t);
               return Bases{o ? atomicAdd(f.fr + d + 1, o) : 0u, e ? atomicAdd(f.fr + d + 2, e) : 0u,
                            l ? atomicAdd(f.fr + kFrLeaves, l) : 0u};
             });
}

}  // namespace

int launch_wide_top(const DevUpdate& u, const DevFrontier& f, int n_top, void* stream) {
  if (n_top < 2 || n_top > kTopLevels || (n_top & 1)) return (int)hipErrorInvalidValue;
  hipLaunchKernelGGL(k_wide_top, dim3(1), dim3(kBlock), 0, reinterpret_cast<hipStream_t>(stream), u,
                     f, n_top);
  return (int)hipGetLastError();
}

int launch_wide_level(const DevUpdate& u, const DevFrontier& f, int d, unsigned blocks,
                      void* stream) {
  if (d < 2 || d >= kMaxDepth || (d & 1)) return (int)hipErrorInvalidValue;
  hipLaunchKernelGGL(k_wide_level, dim3(blocks ? blocks : 1), dim3(kBlock), 0,
                     reinterpret_cast<hipStream_t>(stream), u, f, d);
  return (int)hipGetLastError();
}

}  // namespace mh

// Device build for gfx950: DynBVH::rebuild (Model/Groups/DynBVH.cc:1699-1793) as the
// reference builds it with USE_APPROXIMATE_BUILD set (its MANTA_USE_DYNBVH_APPROXIMATE
// option, include/CMakeLists.txt:134-147, DynBVH.cc:1815-1822): every node is partitioned
// by partitionApproxSAH (16 bins over the longest centroid axis), leaves are sorted, then
// computeSubTreeSizes, the RTSAH pass and computeCost<true>. The tree is the reference's
// record for record, numbering included.
//
// Phase 1, level-synchronous, for nodes of more than kBuildSerial objects. The objects of a
// node are a contiguous range of slots; each slot carries its object's centroid, id and
// box (48 bytes, moved with the id), so every pass streams. A level's nodes are cut into
// virtual blocks of kVB slots; per level:
//   k_level_open   node of each virtual block, accumulators cleared
//   k_bins         16 bins: counts and boxes
//   k_seg_split    the binned SAH sweep: split position or leaf (16 lanes per node)
//   k_count_less   objects left of the position; from their number the split slot, or the
//                  middle when everything fell on one side (seg_mid)
//   k_mis_count, k_scan_mis, k_mis_scatter, k_swap   partitionObjects
//   k_child_bounds boxes and centroid boxes of the two sides
//   k_seg_children new record pair, child nodes to the next level or to phase 2
// The node count of a level stays on the device; the host only bounds it (2^level at most).
// Reductions must give what the reference's serial loops give. Its min/max are select
// forms (a < b ? a : b) applied in slot order, so of equal values (+0 and -0) the last one
// wins; the values that records keep are reduced as 64-bit keys (order-preserving value
// bits, then the slot number) with integer atomics, which makes the result exact and
// independent of order. Bin and centroid boxes only feed differences and comparisons, where
// the sign of a zero makes no difference, and are reduced as 32-bit keys.
// partitionObjects (Hoare's scheme) exchanges the k-th slot from the left whose key is on
// the right side with the k-th slot from the right whose key is on the left side; the
// ranks come from a scan, and the exchanges are independent.
// Phase 2: one wave per node of at most kBuildSerial objects builds its subtree
// (k_subtrees). Phase 3 renumbers the records in the reference's allocation order
// (pairs in preorder of their parents) and computes sizes, marks, costs and RTSAH bottom up.

#include <hip/hip_runtime.h>

#include <cfloat>
#include <climits>
#include <vector>

#include "approx_sah.h"
#include "mh_device.h"
#include "rtsah.h"

namespace mh {
namespace {

constexpr int kBlock = 256;
constexpr int kPer = kBuildVB / kBlock;
constexpr int kVB = kBuildVB;
constexpr int kBins = kSamples;
static_assert(kBins == kBuildBins, "bins");
constexpr int kSetupVB = 2048;  // objects or vertices a workgroup of the set-up passes

// 32-bit key that orders floats as numbers, with -0 and +0 equal.
__device__ __forceinline__ uint32_t ord(float f) {
  uint32_t u = __float_as_uint(f);
  if ((u << 1) == 0) u = 0;
  return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}
__device__ __forceinline__ float unord(uint32_t e) {
  return __uint_as_float((e & 0x80000000u) ? (e & 0x7FFFFFFFu) : ~e);
}
constexpr uint32_t kOrdZero = 0x80000000u;
// Smallest value, then the largest slot. Maxima are minima of the negated values.
__device__ __forceinline__ unsigned long long kmin(float v, uint32_t slot) {
  return ((unsigned long long)ord(v) << 32) | (0xFFFFFFFFu - slot);
}
__device__ __forceinline__ uint32_t kmin_slot(unsigned long long k) {
  return 0xFFFFFFFFu - (uint32_t)k;
}

template <int kCtrl>
__device__ __forceinline__ float dpp_mov(float x) {
  return __int_as_float(
      __builtin_amdgcn_update_dpp(0, __float_as_int(x), kCtrl, 0xF, 0xF, true));
}
template <int kCtrl, int kRows>
__device__ __forceinline__ int dpp_or_own(int x) {
  return __builtin_amdgcn_update_dpp(x, x, kCtrl, kRows, 0xF, false);
}
// Smallest of the wave's values, by row shifts and row broadcasts, in every lane.
template <int kCtrl, int kRows>
__device__ __forceinline__ uint32_t umin_step(uint32_t x) {
  const uint32_t t = (uint32_t)dpp_or_own<kCtrl, kRows>((int)x);
  return t < x ? t : x;
}
__device__ __forceinline__ uint32_t wave_umin(uint32_t x) {
  x = umin_step<0x111, 0xF>(x);
  x = umin_step<0x112, 0xF>(x);
  x = umin_step<0x114, 0xF>(x);
  x = umin_step<0x118, 0xF>(x);
  x = umin_step<0x142, 0xA>(x);
  x = umin_step<0x143, 0xC>(x);
  return (uint32_t)__builtin_amdgcn_readlane((int)x, 63);
}
// A lane's smallest value, the later of equal ones; slots come in ascending order.
struct MinSlot {
  float v = FLT_MAX;
  uint32_t at = 0;
  __device__ __forceinline__ void take(float x, uint32_t slot) {
    at = x <= v ? slot : at;
    v = x <= v ? x : v;
  }
};
// The wave's key: the slot only matters where the value is a zero (key_value).
__device__ __forceinline__ unsigned long long wave_kmin(const MinSlot& m) {
  const uint32_t o = ord(m.v), least = wave_umin(o);
  uint32_t inv = 0;
  if (least == kOrdZero) inv = wave_umin(o == kOrdZero ? 0xFFFFFFFFu - m.at : 0xFFFFFFFFu);
  return ((unsigned long long)least << 32) | inv;
}

// Slot record: centroid, object id, box.
struct alignas(16) Slot {
  float c[3];
  int32_t id;
  float lo[3];
  float hi[3];
  float pad[2];
};
static_assert(sizeof(Slot) == 48, "slot record is 48 bytes");
__device__ __forceinline__ Slot* SL(const DevBuild& d) { return reinterpret_cast<Slot*>(d.slots); }

__device__ __forceinline__ void load_slot(const Slot* s, int64_t i, Slot& o) {
  const float4* p = reinterpret_cast<const float4*>(s + i);
  const float4 a = p[0], b = p[1], c = p[2];
  o.c[0] = a.x;
  o.c[1] = a.y;
  o.c[2] = a.z;
  o.id = __float_as_int(a.w);
  o.lo[0] = b.x;
  o.lo[1] = b.y;
  o.lo[2] = b.z;
  o.hi[0] = b.w;
  o.hi[1] = c.x;
  o.hi[2] = c.y;
  o.pad[0] = c.z;
  o.pad[1] = c.w;
}
__device__ __forceinline__ float slot_c(const Slot* s, int64_t i, int a) {
  return reinterpret_cast<const float*>(s + i)[a];
}

// The level node that owns virtual block v.
__device__ __forceinline__ int find_seg(const DevBuild& d, int64_t v) { return d.vbseg[v]; }

// Boxes are held as six minima (lo, -hi); negating is exact.
__device__ __forceinline__ Box min_box(const float* m) {
  Box b;
  for (int a = 0; a < 3; ++a) {
    b.lo[a] = m[a];
    b.hi[a] = -m[3 + a];
  }
  return b;
}

struct VRange {
  int s;
  int64_t first, end;  // slots of this virtual block
};
__device__ __forceinline__ bool vrange(const DevBuild& d, VRange& r) {
  const int64_t v = blockIdx.x;
  if (v >= (int64_t)d.ctr[kCtrNvb + d.level]) return false;
  r.s = d.vbseg[v];
  const BuildSeg sg = d.seg[r.s];
  r.first = sg.b + (v - sg.vb0) * (int64_t)kVB;
  r.end = r.first + kVB < sg.e ? r.first + kVB : sg.e;
  return true;
}
__device__ __forceinline__ int n_segs(const DevBuild& d) { return (int)d.ctr[kCtrSegs + d.level]; }

// Accumulators of a level node (kAcc*).
__device__ __forceinline__ unsigned* acc(const DevBuild& d, int s) {
  return d.acc + (int64_t)s * kAccWords;
}
__device__ __forceinline__ unsigned long long* acc_box(const DevBuild& d, int s) {
  return reinterpret_cast<unsigned long long*>(acc(d, s));
}
// Split slot of a node and whether slots move (not in the middle fallback): when 0 or all
// objects lie left of the position, partitionObjects moves nothing and the reference
// splits at the middle (DynBVH.cc:2250-2261).
__device__ __forceinline__ int seg_mid(const DevBuild& d, int s, const BuildSeg& sg, bool& moves) {
  const int n = sg.e - sg.b, m = (int)acc(d, s)[kAccLess];
  moves = m != 0 && m != n;
  return moves ? sg.b + m : sg.b + n / 2;
}
// Value of a reduced key; a zero is read back from the winning slot for its sign.
__device__ __forceinline__ float key_value(unsigned long long k, const float* slots, int stride,
                                           int field, bool negated) {
  const uint32_t o = (uint32_t)(k >> 32);
  if (o == kOrdZero) return slots[(int64_t)kmin_slot(k) * stride + field];
  return negated ? -unord(o) : unord(o);
}

// The binning of a node with centroid box keys c (three minima, three negated maxima):
// its longest axis (BBox::longestAxis), start, width and scale.
__device__ __forceinline__ BuildPlan make_plan(const unsigned* c) {
  BuildPlan p{};
  float lo[3], w[3];
  for (int a = 0; a < 3; ++a) {
    lo[a] = unord(c[a]);
    w[a] = -unord(c[3 + a]) - lo[a];
  }
  p.axis = index_of_max(w[0], w[1], w[2]);
  p.width = p.axis == 0 ? w[0] : (p.axis == 1 ? w[1] : w[2]);
  p.lo_c = p.axis == 0 ? lo[0] : (p.axis == 1 ? lo[1] : lo[2]);
  p.scale = ((float)kBins / p.width) * .999f;
  return p;
}

// ---------------------------------------------------------------------------------------
// Set-up

// Box of all vertices (Mesh::computeBounds, Model/Groups/Mesh.cc:195-225); a non-finite
// coordinate sets err = 2.
__global__ __launch_bounds__(kBlock) void k_root_box(DevBuild d) {
  __shared__ unsigned long long sk[6];
  if (threadIdx.x < 6) sk[threadIdx.x] = ~0ull;
  __syncthreads();
  const int64_t first = (int64_t)blockIdx.x * kSetupVB;
  MinSlot m[6];
  bool bad = false;
  for (int k = 0; k < kSetupVB / kBlock; ++k) {
    int64_t i = first + k * kBlock + threadIdx.x;
    i = i < d.n_verts ? i : d.n_verts - 1;
    for (int a = 0; a < 3; ++a) {
      const float x = d.verts[3 * i + a];
      bad |= !(x >= -FLT_MAX && x <= FLT_MAX);
      m[a].take(x, (uint32_t)i);
      m[3 + a].take(-x, (uint32_t)i);
    }
  }
  if (__ballot(bad) && (threadIdx.x & 63) == 0) atomicExch(d.u.err, 2);
  for (int k = 0; k < 6; ++k) {
    const unsigned long long key = wave_kmin(m[k]);
    if ((threadIdx.x & 63) == 0) atomicMin(&sk[k], key);
  }
  __syncthreads();
  if (threadIdx.x < 6) atomicMin(&d.rootk[threadIdx.x], sk[threadIdx.x]);
}

// Slot records, in object order as object_ids starts out: object box (Mesh::getBBox,
// Mesh.cc:228-237) and centroid (BBox::center, BBox.h:63-65), and the box of the centroids.
__global__ __launch_bounds__(kBlock) void k_slots(DevBuild d) {
  __shared__ unsigned sc[6];
  if (threadIdx.x < 6) sc[threadIdx.x] = ~0u;
  __syncthreads();
  const int64_t first = (int64_t)blockIdx.x * kSetupVB;
  uint32_t least[6];
  for (int k = 0; k < 6; ++k) least[k] = ~0u;
  for (int k = 0; k < kSetupVB / kBlock; ++k) {
    const int64_t i = first + k * kBlock + threadIdx.x;
    if (i >= d.u.n_objects) break;
    const Box b = obj_box(d.u, (int)i);
    float c[3];
    for (int a = 0; a < 3; ++a) {
      c[a] = box_cen(b, a);
      const uint32_t lo = ord(c[a]), hi = ord(-c[a]);
      least[a] = lo < least[a] ? lo : least[a];
      least[3 + a] = hi < least[3 + a] ? hi : least[3 + a];
    }
    float4* p = reinterpret_cast<float4*>(SL(d) + i);
    p[0] = make_float4(c[0], c[1], c[2], __int_as_float((int)i));
    p[1] = make_float4(b.lo[0], b.lo[1], b.lo[2], b.hi[0]);
    p[2] = make_float4(b.hi[1], b.hi[2], 0.f, 0.f);
  }
  for (int k = 0; k < 6; ++k) {
    const uint32_t x = wave_umin(least[k]);
    if ((threadIdx.x & 63) == 0) atomicMin(&sc[k], x);
  }
  __syncthreads();
  if (threadIdx.x < 6) atomicMin(&d.rootc[threadIdx.x], sc[threadIdx.x]);
}

// Record 0 gets the vertex box; the root becomes the first node of phase 1 or 2.
__global__ void k_root_init(DevBuild d, int serial) {
  RefNode& r = d.u.refs[0];
  for (int a = 0; a < 3; ++a) {
    r.box.lo[a] = key_value(d.rootk[a], d.verts, 3, a, false);
    r.box.hi[a] = key_value(d.rootk[3 + a], d.verts, 3, a, true);
  }
  r.child = 0;
  r.children = 0;
  r.axis = 0;
  r.bits = 0;
  *d.u.next_free = 1;
  const BuildSeg root{0, 0, d.u.n_objects, 0};
  if (serial) {
    d.small[0] = root;
    d.ctr[kCtrSmall] = 1;
  } else {
    d.seg[0] = root;
    d.plan[0] = make_plan(d.rootc);
    d.ctr[kCtrSegs] = 1;
    d.ctr[kCtrNvb] = (unsigned)((d.u.n_objects + kVB - 1) / kVB);
  }
}

// ---------------------------------------------------------------------------------------
// Phase 1: one level

// vbseg[v] = the node of virtual block v, and cleared accumulators: 16 lanes per node.
__global__ __launch_bounds__(kBlock) void k_level_open(DevBuild d) {
  const int s = (int)(((int64_t)blockIdx.x * kBlock + threadIdx.x) >> 4);
  const int j = threadIdx.x & 15;
  if (s >= n_segs(d)) return;
  const BuildSeg sg = d.seg[s];
  const int nvb = (sg.e - sg.b + kVB - 1) / kVB;
  for (int k = j; k < nvb; k += 16) d.vbseg[sg.vb0 + k] = s;
  uint4* p = reinterpret_cast<uint4*>(acc(d, s));
  for (int k = j; k < kAccWords / 4; k += 16) {
    const unsigned x = 4 * k < kAccCounts ? ~0u : 0u;
    p[k] = make_uint4(x, x, x, x);
  }
}

__device__ __forceinline__ int bin_of(float c, float lo_c, float scale) {
  const float f = (c - lo_c) * scale;
  // int(f) as the reference's x86 build converts it (cvttss2si): NaN and values outside
  // the int range give INT_MIN, i.e. bin 0 after the clamp.
  int which = (f >= -2147483648.f && f < 2147483648.f) ? (int)f : INT_MIN;
  return which < 0 ? 0 : (which > kBins - 1 ? kBins - 1 : which);
}

// Bins of a virtual block in LDS, four copies by lane (lanes of one bin spread over four
// words), then one global atomic per value.
__global__ __launch_bounds__(kBlock) void k_bins(DevBuild d) {
  constexpr int kCopies = 4;
  __shared__ unsigned least[6 * kBins * kCopies], cnt[kBins * kCopies];
  VRange r;
  if (!vrange(d, r)) return;
  for (int k = threadIdx.x; k < 6 * kBins * kCopies; k += kBlock) least[k] = ~0u;
  if (threadIdx.x < kBins * kCopies) cnt[threadIdx.x] = 0;
  __syncthreads();
  const BuildPlan p = d.plan[r.s];
  const int copy = threadIdx.x & (kCopies - 1);
#pragma unroll
  for (int k = 0; k < kPer; ++k) {
    const int64_t i = r.first + k * kBlock + threadIdx.x;
    if (i >= r.end) break;
    Slot o;
    load_slot(SL(d), i, o);
    const float cen = p.axis == 0 ? o.c[0] : (p.axis == 1 ? o.c[1] : o.c[2]);
    const int w = bin_of(cen, p.lo_c, p.scale) * kCopies + copy;
    atomicAdd(&cnt[w], 1u);
    for (int a = 0; a < 3; ++a) {
      atomicMin(&least[a * kBins * kCopies + w], ord(o.lo[a]));
      atomicMin(&least[(3 + a) * kBins * kCopies + w], ord(-o.hi[a]));
    }
  }
  __syncthreads();
  if (threadIdx.x < 7 * kBins) {
    const int w = threadIdx.x & (kBins - 1), f = threadIdx.x / kBins;
    unsigned n = 0;
    for (int k = 0; k < kCopies; ++k) n += cnt[w * kCopies + k];
    if (n) {
      if (f == 6) {
        atomicAdd(&acc(d, r.s)[kAccCounts + w], n);
      } else {
        unsigned x = ~0u;
        for (int k = 0; k < kCopies; ++k) {
          const unsigned y = least[threadIdx.x * kCopies + k];
          x = y < x ? y : x;
        }
        atomicMin(&acc(d, r.s)[kAccBins + threadIdx.x], x);
      }
    }
  }
}

// The sweep of partitionApproxSAH (DynBVH.cc:2196-2236) over the reduced bins, one lane per
// bin: a node's 16 lanes are a row, whose scans are row shifts. (One lane per node, with
// its bins in private memory, took 35 to 50 us a level.)
template <int kCtrl>
__device__ __forceinline__ float row_min(float x, bool c) {
  const float t = dpp_mov<kCtrl>(x);
  return c && t < x ? t : x;
}
__global__ __launch_bounds__(kBlock) void k_seg_split(DevBuild d) {
  const int s = (int)(((int64_t)blockIdx.x * kBlock + threadIdx.x) >> 4);
  const int w = threadIdx.x & 15, lane = threadIdx.x & 63;
  const bool in = s < n_segs(d);
  if (!__ballot(in)) return;
  const int at = in ? s : 0;
  const BuildSeg sg = d.seg[at];
  BuildPlan p = d.plan[at];
  const unsigned* A = acc(d, at);
  const int n = sg.e - sg.b;
  int nl = (int)A[kAccCounts + w];
  float l[6], r[6];
  for (int f = 0; f < 6; ++f)
    l[f] = r[f] = nl ? unord(A[kAccBins + f * kBins + w]) : FLT_MAX;
  for (int f = 0; f < 6; ++f) {
    l[f] = row_min<0x111>(l[f], w >= 1);
    l[f] = row_min<0x112>(l[f], w >= 2);
    l[f] = row_min<0x114>(l[f], w >= 4);
    l[f] = row_min<0x118>(l[f], w >= 8);
    r[f] = row_min<0x101>(r[f], w < 15);
    r[f] = row_min<0x102>(r[f], w < 14);
    r[f] = row_min<0x104>(r[f], w < 12);
    r[f] = row_min<0x108>(r[f], w < 8);
    r[f] = dpp_mov<0x101>(r[f]);  // bins behind this one
  }
  for (int off = 1; off < 16; off <<= 1) {
    const int t = __shfl_up(nl, off, 16);
    nl += w >= off ? t : 0;
  }
  const float inv_parent_area = (float)(1.0 / (double)area(rbox(d.u.refs[sg.rec])));
  const float left_area = area(min_box(l)), right_area = area(min_box(r));
  const float cost =
      (left_area * nl + right_area * (n - nl)) * inv_parent_area * kCIsec + kCTrav;
  float best = w < kBins - 1 && cost < n * kCIsec ? cost : FLT_MAX;
  const float own = best;
  for (int off = 8; off; off >>= 1) {
    const float t = __shfl_xor(best, off, 16);
    best = t < best ? t : best;
  }
  const unsigned long long first = __ballot(own == best && own < FLT_MAX);
  const unsigned mine = (unsigned)(first >> (lane & 48)) & 0xFFFFu;
  if (!in || w != 0) return;
  p.leaf = mine == 0;
  const int i = mine ? __ffs((int)mine) - 1 : 0;
  p.pos = p.lo_c + p.width * (static_cast<float>(i + 1) / kBins);
  d.plan[s] = p;
}

// A wave takes kVB / 4 consecutive slots of a virtual block, 64 at a time.
constexpr int kWaveSlots = kVB / (kBlock / 64);
constexpr int kWaveSteps = kWaveSlots / 64;
__device__ __forceinline__ int64_t wave_slot(const VRange& r, int k) {
  return r.first + (int64_t)(threadIdx.x >> 6) * kWaveSlots + k * 64 + (threadIdx.x & 63);
}

__global__ __launch_bounds__(kBlock) void k_count_less(DevBuild d) {
  __shared__ unsigned tot;
  VRange r;
  if (!vrange(d, r)) return;
  const BuildPlan p = d.plan[r.s];
  if (p.leaf) return;  // uniform over the block
  if (threadIdx.x == 0) tot = 0;
  __syncthreads();
  unsigned c = 0;
#pragma unroll
  for (int k = 0; k < kWaveSteps; ++k) {
    const int64_t i = wave_slot(r, k), j = i < r.end ? i : r.end - 1;
    c += __popcll(__ballot(slot_c(SL(d), j, p.axis) < p.pos && i < r.end));
  }
  if (c && (threadIdx.x & 63) == 0) atomicAdd(&tot, c);
  __syncthreads();
  if (threadIdx.x == 0) {
    d.vcnt[2 * (int64_t)blockIdx.x] = tot;
    if (tot) atomicAdd(&acc(d, r.s)[kAccLess], tot);
  }
}

// A slot is misplaced on the left if it lies before the split with a key >= the position,
// on the right if it lies at or after the split with a key < the position. No slot moves
// in the middle fallback. Only the virtual block that holds the split counts its slots
// again; the others have all of theirs on one side.
__global__ __launch_bounds__(kBlock) void k_mis_count(DevBuild d) {
  __shared__ unsigned tl, tr;
  VRange r;
  if (!vrange(d, r)) return;
  const int64_t v = blockIdx.x;
  const BuildPlan p = d.plan[r.s];
  const BuildSeg sg = d.seg[r.s];
  bool moves;
  const int mid = seg_mid(d, r.s, sg, moves);
  if (p.leaf || !moves || mid >= r.end || mid <= r.first) {
    if (threadIdx.x == 0) {
      const unsigned less = p.leaf || !moves ? 0u : d.vcnt[2 * v];
      const bool before = mid >= r.end;
      d.vcnt[2 * v] = p.leaf || !moves || !before ? 0u : (unsigned)(r.end - r.first) - less;
      d.vcnt[2 * v + 1] = before ? 0u : less;
    }
    return;
  }
  if (threadIdx.x == 0) tl = tr = 0;
  __syncthreads();
  unsigned cl = 0, cr = 0;
  for (int k = 0; k < kWaveSteps; ++k) {
    const int64_t i = wave_slot(r, k);
    const bool less = i < r.end && slot_c(SL(d), i, p.axis) < p.pos;
    cl += __popcll(__ballot(i < mid && !less));
    cr += __popcll(__ballot(i >= mid && less));
  }
  if ((threadIdx.x & 63) == 0) {
    if (cl) atomicAdd(&tl, cl);
    if (cr) atomicAdd(&tr, cr);
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    d.vcnt[2 * v] = tl;
    d.vcnt[2 * v + 1] = tr;
  }
}

// Exclusive scans over all virtual blocks of the left and right counts (one workgroup, four
// virtual blocks a thread): gscan[v] (left) and gscan[vcap + 1 + v] (right), v in [0, nvb].
__global__ __launch_bounds__(1024) void k_scan_mis(DevBuild d) {
  __shared__ unsigned wl[16], wr[16];
  const int64_t nvb = d.ctr[kCtrNvb + d.level];
  unsigned* gl = d.gscan;
  unsigned* gr = d.gscan + d.vcap + 1;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  unsigned cl = 0, cr = 0;  // before this round
  for (int64_t base = 0; base < nvb; base += 4096) {
    const int64_t v0 = base + 4 * (int64_t)threadIdx.x;
    unsigned a[4], b[4], sl = 0, sr = 0;
    for (int k = 0; k < 4; ++k) {
      a[k] = v0 + k < nvb ? d.vcnt[2 * (v0 + k)] : 0u;
      b[k] = v0 + k < nvb ? d.vcnt[2 * (v0 + k) + 1] : 0u;
      sl += a[k];
      sr += b[k];
    }
    unsigned il = sl, ir = sr;  // inclusive over the wave
    for (int off = 1; off < 64; off <<= 1) {
      const unsigned x = (unsigned)__shfl_up((int)il, off), y = (unsigned)__shfl_up((int)ir, off);
      il += lane >= off ? x : 0u;
      ir += lane >= off ? y : 0u;
    }
    if (lane == 63) {
      wl[wave] = il;
      wr[wave] = ir;
    }
    __syncthreads();
    unsigned pl = cl + il - sl, pr = cr + ir - sr;
    for (int w = 0; w < 16; ++w) {
      pl += w < wave ? wl[w] : 0u;
      pr += w < wave ? wr[w] : 0u;
      cl += wl[w];
      cr += wr[w];
    }
    for (int k = 0; k < 4 && v0 + k < nvb; ++k) {
      gl[v0 + k] = pl;
      gr[v0 + k] = pr;
      pl += a[k];
      pr += b[k];
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    gl[nvb] = cl;
    gr[nvb] = cr;
  }
}

// Slots of the misplaced objects by rank: from the left in lpos, from the right in rpos.
__global__ __launch_bounds__(kBlock) void k_mis_scatter(DevBuild d) {
  __shared__ unsigned wl[kBlock / 64], wr[kBlock / 64];
  VRange r;
  if (!vrange(d, r)) return;
  const int64_t v = blockIdx.x;
  const BuildPlan p = d.plan[r.s];
  const BuildSeg sg = d.seg[r.s];
  bool moves;
  const int mid = seg_mid(d, r.s, sg, moves);
  if (p.leaf || !moves) return;  // uniform over the block
  const unsigned* gl = d.gscan;
  const unsigned* gr = d.gscan + d.vcap + 1;
  const int nvb_s = (sg.e - sg.b + kVB - 1) / kVB;
  const unsigned totR = gr[sg.vb0 + nvb_s] - gr[sg.vb0];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const unsigned long long below = (1ull << lane) - 1ull;
  unsigned long long ml[kWaveSteps], mr[kWaveSteps];
  unsigned cl = 0, cr = 0;
#pragma unroll
  for (int k = 0; k < kWaveSteps; ++k) {
    const int64_t i = wave_slot(r, k), j = i < r.end ? i : r.end - 1;
    const bool less = slot_c(SL(d), j, p.axis) < p.pos;
    ml[k] = __ballot(i < r.end && i < mid && !less);
    mr[k] = __ballot(i < r.end && i >= mid && less);
    cl += __popcll(ml[k]);
    cr += __popcll(mr[k]);
  }
  if (lane == 0) {
    wl[wave] = cl;
    wr[wave] = cr;
  }
  __syncthreads();
  unsigned rl = gl[v] - gl[sg.vb0], rr = gr[v] - gr[sg.vb0];
  for (int w = 0; w < wave; ++w) {
    rl += wl[w];
    rr += wr[w];
  }
#pragma unroll
  for (int k = 0; k < kWaveSteps; ++k) {
    const int32_t i = (int32_t)wave_slot(r, k);
    if ((ml[k] >> lane) & 1) d.lpos[sg.b + rl + __popcll(ml[k] & below)] = i;
    if ((mr[k] >> lane) & 1) d.rpos[sg.b + (totR - 1 - (rr + __popcll(mr[k] & below)))] = i;
    rl += __popcll(ml[k]);
    rr += __popcll(mr[k]);
  }
}

__global__ __launch_bounds__(kBlock) void k_swap(DevBuild d) {
  VRange r;
  if (!vrange(d, r)) return;
  const BuildPlan p = d.plan[r.s];
  const BuildSeg sg = d.seg[r.s];
  bool moves;
  (void)seg_mid(d, r.s, sg, moves);
  if (p.leaf || !moves) return;
  const unsigned* gl = d.gscan;
  const int nvb_s = (sg.e - sg.b + kVB - 1) / kVB;
  const int64_t nswap = gl[sg.vb0 + nvb_s] - gl[sg.vb0];
  for (int k = 0; k < kPer; ++k) {
    const int64_t i = r.first + k * kBlock + threadIdx.x;
    if (i >= r.end) break;
    const int64_t j = i - sg.b;
    if (j >= nswap) break;
    const int64_t a = d.lpos[sg.b + j], b = d.rpos[sg.b + j];
    float4* pa = reinterpret_cast<float4*>(SL(d) + a);
    float4* pb = reinterpret_cast<float4*>(SL(d) + b);
    const float4 a0 = pa[0], a1 = pa[1], a2 = pa[2];
    const float4 b0 = pb[0], b1 = pb[1], b2 = pb[2];
    pa[0] = b0;
    pa[1] = b1;
    pa[2] = b2;
    pb[0] = a0;
    pb[1] = a1;
    pb[2] = a2;
  }
}

// Boxes and centroid boxes of the two sides: reduced in registers over the wave (by lanes
// into one LDS word of 64 bits, as before, 50 to 130 us a level), then in LDS over the
// workgroup, then one global atomic per value.
__global__ __launch_bounds__(kBlock) void k_child_bounds(DevBuild d) {
  __shared__ unsigned long long sk[12];
  __shared__ unsigned sc[12];
  VRange r;
  if (!vrange(d, r)) return;
  const BuildPlan p = d.plan[r.s];
  if (p.leaf) return;
  const BuildSeg sg = d.seg[r.s];
  bool moves;
  const int mid = seg_mid(d, r.s, sg, moves);
  if (threadIdx.x < 12) {
    sk[threadIdx.x] = ~0ull;
    sc[threadIdx.x] = ~0u;
  }
  __syncthreads();
  for (int side = 0; side < 2; ++side) {
    const int64_t lo = side && mid > r.first ? mid : r.first;
    const int64_t hi = !side && mid < r.end ? mid : r.end;
    if (lo + (threadIdx.x & ~63) >= hi) continue;  // nothing for this wave
    MinSlot m[6];
    uint32_t c[6];
    for (int k = 0; k < 6; ++k) c[k] = ~0u;
    for (int64_t first = lo; first < hi; first += kBlock) {
      int64_t i = first + threadIdx.x;
      i = i < hi ? i : hi - 1;  // the last slot again: changes no minimum
      Slot o;
      load_slot(SL(d), i, o);
      for (int a = 0; a < 3; ++a) {
        m[a].take(o.lo[a], (uint32_t)i);
        m[3 + a].take(-o.hi[a], (uint32_t)i);
        const uint32_t x = ord(o.c[a]), y = ord(-o.c[a]);
        c[a] = x < c[a] ? x : c[a];
        c[3 + a] = y < c[3 + a] ? y : c[3 + a];
      }
    }
    for (int k = 0; k < 6; ++k) {
      const unsigned long long key = wave_kmin(m[k]);
      const uint32_t x = wave_umin(c[k]);
      if ((threadIdx.x & 63) == 0) {
        atomicMin(&sk[6 * side + k], key);
        atomicMin(&sc[6 * side + k], x);
      }
    }
  }
  __syncthreads();
  if (threadIdx.x < 12) {
    if (sk[threadIdx.x] != ~0ull) atomicMin(&acc_box(d, r.s)[threadIdx.x], sk[threadIdx.x]);
  } else if (threadIdx.x < 24) {
    const unsigned x = sc[threadIdx.x - 12];
    if (x != ~0u) atomicMin(&acc(d, r.s)[kAccCen + threadIdx.x - 12], x);
  }
}

// One lane per node; a wave's nodes take their places from each counter with one atomic
// (an atomic per node and counter took up to 137 us a level).
__global__ __launch_bounds__(kBlock) void k_seg_children(DevBuild d) {
  const int s = blockIdx.x * kBlock + threadIdx.x;
  const int lane = threadIdx.x & 63;
  const unsigned long long below = (1ull << lane) - 1ull;
  const bool in = s < n_segs(d);
  if (!__ballot(in)) return;
  const int at = in ? s : 0;
  const BuildPlan p = d.plan[at];
  const BuildSeg sg = d.seg[at];
  bool moves;
  const int mid = seg_mid(d, at, sg, moves);
  const bool inner = in && !p.leaf, leaf = in && p.leaf;
  const int b[2] = {sg.b, mid}, e[2] = {mid, sg.e};
  unsigned long long next[2], small[2];
  int vbs = 0;  // virtual blocks of this node's children
  for (int side = 0; side < 2; ++side) {
    const bool large = e[side] - b[side] > kBuildSerial;
    next[side] = __ballot(inner && large);
    small[side] = __ballot(inner && !large);
    if (inner && large) vbs += (e[side] - b[side] + kVB - 1) / kVB;
  }
  int vb_end = vbs;
  for (int off = 1; off < 64; off <<= 1) {
    const int t = __shfl_up(vb_end, off);
    vb_end += lane >= off ? t : 0;
  }
  const unsigned long long inners = __ballot(inner), leaves = __ballot(leaf);
  const unsigned amount[5] = {2u * (unsigned)__popcll(inners),
                              (unsigned)(__popcll(next[0]) + __popcll(next[1])),
                              (unsigned)(__popcll(small[0]) + __popcll(small[1])),
                              (unsigned)__popcll(leaves), (unsigned)__shfl(vb_end, 63)};
  unsigned* const counter[5] = {d.u.next_free, d.ctr + kCtrSegs + d.level + 1, d.ctr + kCtrSmall,
                                d.ctr + kCtrBig, d.ctr + kCtrNvb + d.level + 1};
  unsigned got = 0;
  for (int k = 0; k < 5; ++k)
    if (lane == k && amount[k]) got = atomicAdd(counter[k], amount[k]);
  unsigned base[5];
  for (int k = 0; k < 5; ++k) base[k] = (unsigned)__shfl((int)got, k);
  if (!in) return;
  RefNode& nd = d.u.refs[sg.rec];
  if (leaf) {  // sorted later, with the other large leaves
    const int n = sg.e - sg.b;
    if (n > 32767) atomicExch(d.u.err, 3);
    nd.child = sg.b;
    nd.children = (int16_t)n;
    nd.axis = 0;
    d.big[base[3] + __popcll(leaves & below)] = sg;
    return;
  }
  unsigned spot = base[0] + 2u * (unsigned)__popcll(inners & below);
  if (spot + 1 >= (unsigned)d.u.n_records) {  // cannot happen: N objects need < 2N records
    atomicExch(d.u.err, 1);
    spot = 0;
  }
  nd.child = (int32_t)spot;
  nd.children = 0;
  nd.axis = (uint8_t)p.axis;
  int vb = (int)base[4] + vb_end - vbs;
  unsigned q_next = base[1], q_small = base[2];
  for (int side = 0; side < 2; ++side) {
    RefNode& c = d.u.refs[spot + side];
    const unsigned long long* k = acc_box(d, s) + 6 * side;
    for (int a = 0; a < 3; ++a) {
      c.box.lo[a] = key_value(k[a], d.slots, 12, 4 + a, false);
      c.box.hi[a] = key_value(k[3 + a], d.slots, 12, 7 + a, true);
    }
    c.child = 0;
    c.children = 0;
    c.axis = 0;
    c.bits = 0;
    const BuildSeg child{(int32_t)spot + side, b[side], e[side], vb};
    if ((next[side] >> lane) & 1) {
      const unsigned q = q_next + (unsigned)__popcll(next[side] & below);
      d.seg_next[q] = child;
      d.plan_next[q] = make_plan(acc(d, s) + kAccCen + 6 * side);
      vb += (e[side] - b[side] + kVB - 1) / kVB;
    } else {
      d.small[q_small + (unsigned)__popcll(small[side] & below)] = child;
    }
    q_next += (unsigned)__popcll(next[side]);
    q_small += (unsigned)__popcll(small[side]);
  }
}

// ---------------------------------------------------------------------------------------
// Phase 2 and large leaves

// One wave builds the subtree of a small node (at most 64 objects), one object per lane in
// slot order, all nodes of a depth in one step. A node is a run of lanes; its reductions
// are segmented scans over the wave (SegScan), its bins a stable sort by bin number. The
// data of a subtree is read once and the work is VALU issue: about 900 instructions a
// depth whatever the number of nodes in it. One lane per subtree running the reference's
// recursion (bins in private memory, a depth-first chain of loads) took 3742 us for the
// 28 thousand subtrees of a million triangles, and 3300 to 6900 us with 32 to 1 lanes of a
// wave in use; this takes 193 us.

__device__ __forceinline__ float lane_get(float x, int src) {
  return __int_as_float(__builtin_amdgcn_ds_bpermute(src << 2, __float_as_int(x)));
}
__device__ __forceinline__ int lane_get(int x, int src) {
  return __builtin_amdgcn_ds_bpermute(src << 2, x);
}
__device__ __forceinline__ float lane_put(float x, int dst) {
  return __int_as_float(__builtin_amdgcn_ds_permute(dst << 2, __float_as_int(x)));
}
__device__ __forceinline__ int lane_put(int x, int dst) {
  return __builtin_amdgcn_ds_permute(dst << 2, x);
}

// Inclusive minimum over the lanes [sb, lane], with the select form a < b ? a : b applied
// in lane order (so the sign of a zero is the one the reference's loop leaves). Four steps
// inside the rows of 16 lanes, then the last lanes of the rows before.
struct SegScan {
  bool c1, c2, c4, c8, row, half;
  __device__ __forceinline__ SegScan(int lane, int sb) {
    const int p = lane & 15, reach = lane - sb;
    c1 = p >= 1 && reach >= 1;
    c2 = p >= 2 && reach >= 2;
    c4 = p >= 4 && reach >= 4;
    c8 = p >= 8 && reach >= 8;
    row = (lane & 16) && reach > p;
    half = lane >= 32 && sb <= 31;
  }
  __device__ __forceinline__ static void step(float& x, float t, bool c) {
    x = c && t < x ? t : x;
  }
  __device__ __forceinline__ float min(float x) const {
    step(x, dpp_mov<0x111>(x), c1);
    step(x, dpp_mov<0x112>(x), c2);
    step(x, dpp_mov<0x114>(x), c4);
    step(x, dpp_mov<0x118>(x), c8);
    step(x, dpp_mov<0x142>(x), row);   // lane 15 of the row before
    step(x, dpp_mov<0x143>(x), half);  // lane 31
    return x;
  }
};

__device__ __forceinline__ void put_record(RefNode* r, const float* m, int child, int children,
                                           int axis) {
  float4* p = reinterpret_cast<float4*>(r);
  p[0] = make_float4(m[0], m[1], m[2], -m[3]);
  p[1] = make_float4(-m[4], -m[5], __int_as_float(child),
                     __int_as_float((children << 16) | axis));
}
__device__ __forceinline__ int place(unsigned long long m) { return __popcll(m); }

__global__ __launch_bounds__(kBlock) void k_subtrees(DevBuild d, int64_t n_small) {
  constexpr int kWaves = kBlock / 64;
  __shared__ unsigned need_of[kWaves], base_of;
  __shared__ int partner[kWaves][2][64];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int64_t k = (int64_t)blockIdx.x * kWaves + wave;
  const bool has = k < n_small;
  const BuildSeg sg = has ? d.small[k] : BuildSeg{0, 0, 1, 0};
  const int n = sg.e - sg.b;
  // A subtree of n objects has at most n - 1 inner nodes: reserve their pairs at once, for
  // the workgroup's waves together.
  const unsigned need = 2u * (unsigned)(n - 1);
  if (lane == 0) need_of[wave] = need;
  __syncthreads();
  if (threadIdx.x == 0) {
    unsigned sum = 0;
    for (int w = 0; w < kWaves; ++w) sum += need_of[w];
    base_of = sum ? atomicAdd(d.u.next_free, sum) : 0u;
  }
  __syncthreads();
  if (!has) return;
  unsigned base = base_of;
  for (int w = 0; w < wave; ++w) base += need_of[w];
  if (need && base + need > (unsigned)d.u.n_records) {
    if (lane == 0) atomicExch(d.u.err, 1);
    return;
  }

  const bool in = lane < n;
  float c[3] = {0.f, 0.f, 0.f}, v[6] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f}, nb[6];
  int id = 0;
  if (in) {
    Slot o;
    load_slot(SL(d), sg.b + lane, o);
    id = o.id;
    for (int a = 0; a < 3; ++a) {
      c[a] = o.c[a];
      v[a] = o.lo[a];
      v[3 + a] = -o.hi[a];
    }
  }
  {
    const RefNode& top = d.u.refs[sg.rec];
    for (int a = 0; a < 3; ++a) {
      nb[a] = top.box.lo[a];
      nb[3 + a] = -top.box.hi[a];
    }
  }
  // This lane's node: its lanes [sb, se), its record and its box nb.
  int sb = in ? 0 : lane, se = in ? n : lane + 1, rec = sg.rec;
  bool live = in;
  unsigned used = 0;  // pairs handed out
  const unsigned long long below = (1ull << lane) - 1ull;
  while (__ballot(live)) {
    const int m = se - sb;
    const unsigned long long seg = (~0ull >> (64 - m)) << sb;
    const Box node_box = min_box(nb);
    bool split = false;
    int axis = 0, mid = sb, src = lane;
    const bool many = live && m >= 3;
    if (__ballot(many)) {  // partitionApproxSAH (DynBVH.cc:2125-2246)
      const SegScan scan(lane, sb);
      float cm[6];
      for (int a = 0; a < 3; ++a) {
        cm[a] = lane_get(scan.min(c[a]), se - 1);
        cm[3 + a] = lane_get(scan.min(-c[a]), se - 1);
      }
      const float w0 = -cm[3] - cm[0], w1 = -cm[4] - cm[1], w2 = -cm[5] - cm[2];
      const int ax = index_of_max(w0, w1, w2);
      const float width = ax == 0 ? w0 : (ax == 1 ? w1 : w2);
      const float lo_c = ax == 0 ? cm[0] : (ax == 1 ? cm[1] : cm[2]);
      const float cen = ax == 0 ? c[0] : (ax == 1 ? c[1] : c[2]);
      const float scale = ((float)kBins / width) * .999f;
      const int w = bin_of(cen, lo_c, scale);
      // Place among the node's objects by (bin, lane).
      unsigned long long less = 0, same = seg;
      for (int bit = 8; bit; bit >>= 1) {
        const unsigned long long one = __ballot((w & bit) != 0);
        if (w & bit) {
          less |= same & ~one;
          same &= one;
        } else {
          same &= ~one;
        }
      }
      const int to = many ? sb + place(less) + place(same & below) : lane;
      const int rto = many ? sb + se - 1 - to : lane;
      const int sw = lane_put(w, to);
      float l[6], r[6];
      for (int a = 0; a < 6; ++a) {
        l[a] = scan.min(lane_put(v[a], to));
        r[a] = scan.min(lane_put(v[a], rto));
      }
      // A cost changes only behind a bin that holds objects, so the last object of each
      // bin stands for the reference's candidates up to the next such bin; behind the last
      // bin that holds any the right side's area is NaN times zero objects.
      const int back = sb + se - lane - 2;
      for (int a = 0; a < 6; ++a) r[a] = lane_get(r[a], back >= sb ? back : lane);
      const int next_w = lane_get(sw, lane < 63 ? lane + 1 : lane);
      const bool cand = many && lane + 1 < se && sw != next_w;
      const float inv_parent_area = (float)(1.0 / (double)area(node_box));
      const float left_area = area(min_box(l)), right_area = area(min_box(r));
      const float cost = (left_area * (lane + 1 - sb) + right_area * (se - 1 - lane)) *
                             inv_parent_area * kCIsec + kCTrav;
      const float key = cand && cost < m * kCIsec ? cost : FLT_MAX;
      const float best = lane_get(scan.min(key), se - 1);
      const unsigned long long at = __ballot(cand && key == best && key < FLT_MAX) & seg;
      const int bin = lane_get(sw, at ? __ffsll((long long)at) - 1 : lane);
      const float pos = lo_c + width * (static_cast<float>(bin + 1) / kBins);
      const bool cut = many && at != 0;
      // partitionObjects (DynBVH.cc:1369-1396), or the middle (DynBVH.cc:2250-2261)
      const bool left = cut && cen < pos;
      const int nl = place(__ballot(left) & seg);
      const bool fallback = nl == 0 || nl == m;
      if (cut) {
        split = true;
        axis = ax;
        mid = fallback ? sb + m / 2 : sb + nl;
      }
      const bool out_l = cut && !fallback && lane < mid && !left;
      const bool out_r = cut && !fallback && lane >= mid && left;
      const unsigned long long ml = __ballot(out_l) & seg, mr = __ballot(out_r) & seg;
      if (ml | mr) {
        const int kl = sb + place(ml & below);
        const int kr = sb + place(mr & ~below & ~(1ull << lane));
        if (out_l) partner[wave][0][kl] = lane;
        if (out_r) partner[wave][1][kr] = lane;
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        if (out_l) src = partner[wave][1][kl];
        if (out_r) src = partner[wave][0][kr];
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      }
    }
    const bool two = live && m == 2;
    if (__ballot(two)) {  // partition2Objs (DynBVH.cc:2277-2308)
      const int other = two ? sb + se - 1 - lane : lane;
      const float mine = area(min_box(v));
      const float theirs = lane_get(mine, other);
      const float new_cost = kCTrav + (mine * kCIsec + theirs * kCIsec) / area(node_box);
      const int ax = longest_axis(node_box);
      const float lo = ax == 0 ? v[0] : (ax == 1 ? v[1] : v[2]);
      const float lo_other = lane_get(lo, other);
      if (two && new_cost < kCIsec * 2) {
        split = true;
        axis = ax;
        mid = sb + 1;
        if (lane == sb ? lo > lo_other : lo_other > lo) src = other;
      }
    }
    const unsigned long long heads = __ballot(split && lane == sb);
    const unsigned spot = base + 2u * (used + (unsigned)place(heads & ((1ull << sb) - 1ull)));
    used += (unsigned)place(heads);
    if (live && lane == sb)
      put_record(d.u.refs + rec, nb, split ? (int)spot : sg.b + sb, split ? 0 : m,
                 split ? axis : 0);
    live = split;
    if (!heads) break;
    id = lane_get(id, src);
    for (int a = 0; a < 3; ++a) c[a] = lane_get(c[a], src);
    for (int a = 0; a < 6; ++a) v[a] = lane_get(v[a], src);
    if (split) {
      const bool right = lane >= mid;
      rec = (int)spot + (right ? 1 : 0);
      sb = right ? mid : sb;
      se = right ? se : mid;
    }
    const SegScan sides(lane, sb);
    for (int a = 0; a < 6; ++a) {
      const float x = lane_get(sides.min(v[a]), se - 1);
      if (split) nb[a] = x;
    }
  }
  // Leaves' ids in ascending order (std::sort); each node is now a leaf.
  const int m = se - sb;
  int less = 0;
  for (int t = 0; __ballot(in && t < m); ++t) {
    const int o = lane_get(id, t < m ? sb + t : lane);
    less += o < id ? 1 : 0;
  }
  if (in) d.u.ids[sg.b + sb + less] = id;
  for (unsigned r = base + 2 * used + lane; r < base + need; r += 64) {
    // unused records: marked as holes
    RefNode& h = d.u.refs[r];
    h.child = 0;
    h.children = kHole;
    h.axis = 0;
    h.bits = 0;
  }
}

// std::sort of a large leaf's ids: bitonic sort of the range padded to a power of two
// in scratch (two ints per slot of the range, so leaves never share scratch).
__global__ __launch_bounds__(1024) void k_sort_big(DevBuild d, int32_t* scratch) {
  const BuildSeg sg = d.big[blockIdx.x];
  const int n = sg.e - sg.b;
  int P = 1;
  while (P < n) P <<= 1;
  int32_t* a = scratch + 2 * (int64_t)sg.b;
  for (int i = threadIdx.x; i < P; i += blockDim.x) a[i] = i < n ? SL(d)[sg.b + i].id : INT_MAX;
  __syncthreads();
  for (int k = 2; k <= P; k <<= 1) {
    for (int j = k >> 1; j > 0; j >>= 1) {
      for (int i = threadIdx.x; i < P; i += blockDim.x) {
        const int l = i ^ j;
        if (l > i) {
          const int32_t x = a[i], y = a[l];
          const bool up = (i & k) == 0;
          if (up ? x > y : x < y) {
            a[i] = y;
            a[l] = x;
          }
        }
      }
      __syncthreads();
    }
  }
  for (int i = threadIdx.x; i < n; i += blockDim.x) d.u.ids[sg.b + i] = a[i];
}

// ---------------------------------------------------------------------------------------
// Phase 3: reference numbering and the bottom-up passes

__global__ __launch_bounds__(kBlock) void k_ic_leaves(DevFinish f, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (i < n) f.ic[f.leaves[i]] = 0;
}
// The small depths at the top run in one workgroup (k_*_top): the barrier between depths
// orders them as separate launches would (the workgroup's waves share one compute unit and
// its L1, so stores before the barrier are seen by loads after it).
template <class F>
__device__ __forceinline__ void top_up(const TopLevels& t, F node) {
  for (int d = t.n - 1; d >= 0; --d) {
    for (int i = (int)threadIdx.x; i < t.cnt[d]; i += kBlock) node((int64_t)t.first[d] + i);
    __syncthreads();
  }
}
__device__ __forceinline__ void ic_node(const DevFinish& f, int64_t i) {
  const int x = f.levels[i];
  const int c = f.trefs[x].child;
  f.ic[x] = 1 + f.ic[c] + f.ic[c + 1];
}
__global__ __launch_bounds__(kBlock) void k_ic_level(DevFinish f, int64_t first, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (i < n) ic_node(f, first + i);
}
// Pairs are handed out in preorder of their parents (DynBVH::build recursion).
__device__ __forceinline__ void rank_node(const DevFinish& f, int64_t i) {
  const int x = f.levels[i];
  const int c = f.trefs[x].child;
  const int rk = f.rank[x];
  f.fin[c] = 2 * rk + 1;
  f.fin[c + 1] = 2 * rk + 2;
  f.rank[c] = rk + 1;
  f.rank[c + 1] = rk + 1 + f.ic[c];
}
__global__ __launch_bounds__(kBlock) void k_rank_level(DevFinish f, int64_t first, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (i < n) rank_node(f, first + i);
}
// Counts up and ranks down through the top depths.
__global__ __launch_bounds__(kBlock) void k_ic_rank_top(DevFinish f, TopLevels t) {
  top_up(t, [&](int64_t i) { ic_node(f, i); });
  if (threadIdx.x == 0) {
    f.rank[0] = 0;
    f.fin[0] = 0;
  }
  __syncthreads();
  for (int d = 0; d < t.n; ++d) {
    for (int i = (int)threadIdx.x; i < t.cnt[d]; i += kBlock) rank_node(f, (int64_t)t.first[d] + i);
    __syncthreads();
  }
}
// Records in use move to their reference numbers; records from the node count on are
// left as DynBVH::allocate leaves them after a reset. Holes (records that the
// small nodes' subtrees reserved but did not use) have no number and vanish.
__global__ __launch_bounds__(kBlock) void k_emit(DevFinish f) {
  const int64_t x = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (x >= f.n_records) return;
  if (x >= f.n_final) {
    RefNode b;
    for (int a = 0; a < 3; ++a) {
      b.box.lo[a] = FLT_MAX;
      b.box.hi[a] = -FLT_MAX;
    }
    b.child = 0;
    b.axis = 0;
    b.bits = 0;
    b.children = 0;
    f.refs[x] = b;
  }
  if (x >= (int64_t)*f.tcount) return;
  const int32_t to = f.fin[x];
  if (to < 0 || to >= f.n_final) return;  // a hole
  RefNode t = f.trefs[x];
  t.bits = 0;
  if (t.children == 0) t.child = 2 * f.rank[x] + 1;
  f.refs[to] = t;
}
__global__ __launch_bounds__(kBlock) void k_map_lists(DevFinish f, int64_t n_inner,
                                                      int64_t n_leaves) {
  const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (i < n_inner) f.levels[i] = f.fin[f.levels[i]];
  if (i < n_leaves) f.leaves[i] = f.fin[f.leaves[i]];
}
// computeSubTreeSizes, computeCost<true> and the RTSAH pass (DynBVH.cc:1971-1996,
// 3388-3415, 1594-1678) for the leaves, then one launch per depth, deepest first.
__global__ __launch_bounds__(kBlock) void k_fin_leaves(DevFinish f, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (i >= n) return;
  const int r = f.leaves[i];
  RefNode& nd = f.refs[r];
  nd.bits &= ~2;
  f.ssize[r] = 1;
  f.costs[r] = nd.children * kCIsec;
  const rtsah::CostPair c = rtsah::leaf_cost(nd.children);
  f.rt[2 * r] = c.c0;
  f.rt[2 * r + 1] = c.c1;
}
__device__ __forceinline__ Aabb aabb(const RefNode& n) {
  Aabb b;
  for (int a = 0; a < 3; ++a) {
    b.lo[a] = n.box.lo[a];
    b.hi[a] = n.box.hi[a];
  }
  return b;
}
// The crossing probabilities of every inner node. They depend on the boxes alone, so all
// depths go in one launch: some 30 us of dependent float work that each depth's launch
// would otherwise wait for (12 to 87 us a depth, 1160 us of a million triangles' build).
__global__ __launch_bounds__(kBlock) void k_fin_probs(DevFinish f, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (i >= n) return;
  const RefNode nd = f.refs[f.levels[i]];
  const Aabb L = aabb(f.refs[nd.child]), R = aabb(f.refs[nd.child + 1]);
  float lr, jl, jr;
  rtsah::probabilities(f.logtab, aabb(nd), L, R, lr, jl, jr);
  f.prob[0][i] = lr;
  f.prob[1][i] = jl;
  f.prob[2][i] = jr;
}
__device__ __forceinline__ void fin_node(const DevFinish& f, int64_t i) {
  const int r = f.levels[i];
  RefNode& nd = f.refs[r];
  const int c = nd.child;
  const uint32_t size = 1 + f.ssize[c] + f.ssize[c + 1];
  f.ssize[r] = size;
  uint8_t bits = nd.bits & ~3;
  if (size > f.large) bits |= 2;
  const float ar = area(rbox(nd)), al = area(rbox(f.refs[c])), arr = area(rbox(f.refs[c + 1]));
  f.costs[r] = kCTrav + (al * f.costs[c] + arr * f.costs[c + 1]) / ar;
  if (f.rtsah) {
    bool left_cheaper = false;
    const rtsah::CostPair cl{f.rt[2 * c], f.rt[2 * c + 1]};
    const rtsah::CostPair cr{f.rt[2 * c + 2], f.rt[2 * c + 3]};
    const rtsah::CostPair o =
        rtsah::combine(f.prob[0][i], f.prob[1][i], f.prob[2][i], cl, cr, left_cheaper);
    if (left_cheaper) bits |= 1;
    f.rt[2 * r] = o.c0;
    f.rt[2 * r + 1] = o.c1;
  }
  nd.bits = bits;
}
__global__ __launch_bounds__(kBlock) void k_fin_level(DevFinish f, int64_t first, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (i < n) fin_node(f, first + i);
}
__global__ __launch_bounds__(kBlock) void k_fin_top(DevFinish f, TopLevels t) {
  top_up(t, [&](int64_t i) { fin_node(f, i); });
}

unsigned grid(int64_t n, int block = kBlock) { return (unsigned)((n + block - 1) / block); }

}  // namespace

// ---------------------------------------------------------------------------------------
// Launchers (the host drives the level loop; see build_device in mh_api.cpp)

int build_launch_setup(const DevBuild& d, int serial, void* stream) {
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  hipLaunchKernelGGL(k_root_box, dim3(grid(d.n_verts, kSetupVB)), dim3(kBlock), 0, s, d);
  hipLaunchKernelGGL(k_slots, dim3(grid(d.u.n_objects, kSetupVB)), dim3(kBlock), 0, s, d);
  hipLaunchKernelGGL(k_root_init, dim3(1), dim3(1), 0, s, d, serial);
  return (int)hipGetLastError();
}

int build_launch_level(const DevBuild& d, int64_t nseg_bound, int64_t nvb_bound, void* stream) {
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  const unsigned gs = grid(nseg_bound), g16 = grid(nseg_bound, kBlock / 16);
  const unsigned gv = (unsigned)nvb_bound;
  hipLaunchKernelGGL(k_level_open, dim3(g16), dim3(kBlock), 0, s, d);
  hipLaunchKernelGGL(k_bins, dim3(gv), dim3(kBlock), 0, s, d);
  hipLaunchKernelGGL(k_seg_split, dim3(g16), dim3(kBlock), 0, s, d);
  hipLaunchKernelGGL(k_count_less, dim3(gv), dim3(kBlock), 0, s, d);
  hipLaunchKernelGGL(k_mis_count, dim3(gv), dim3(kBlock), 0, s, d);
  hipLaunchKernelGGL(k_scan_mis, dim3(1), dim3(1024), 0, s, d);
  hipLaunchKernelGGL(k_mis_scatter, dim3(gv), dim3(kBlock), 0, s, d);
  hipLaunchKernelGGL(k_swap, dim3(gv), dim3(kBlock), 0, s, d);
  hipLaunchKernelGGL(k_child_bounds, dim3(gv), dim3(kBlock), 0, s, d);
  hipLaunchKernelGGL(k_seg_children, dim3(gs), dim3(kBlock), 0, s, d);
  return (int)hipGetLastError();
}

int build_launch_serial(const DevBuild& d, int64_t n_small, int64_t n_big, int32_t* scratch,
                        void* stream) {
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  if (n_small > 0)
    hipLaunchKernelGGL(k_subtrees, dim3(grid(n_small, kBlock / 64)), dim3(kBlock), 0, s, d,
                       n_small);
  if (n_big > 0) hipLaunchKernelGGL(k_sort_big, dim3((unsigned)n_big), dim3(1024), 0, s, d, scratch);
  return (int)hipGetLastError();
}

int build_launch_ranks(const DevFinish& f, const int64_t* level_off, int n_levels,
                       int64_t n_leaves, void* stream) {
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  std::vector<LevelList> lev;
  for (int d = 0; d < n_levels; ++d)
    lev.push_back(LevelList{level_off[d], level_off[d + 1] - level_off[d]});
  TopLevels t;
  const int top = top_levels(lev.data(), n_levels, 1, t);
  if (n_leaves > 0)
    hipLaunchKernelGGL(k_ic_leaves, dim3(grid(n_leaves)), dim3(kBlock), 0, s, f, n_leaves);
  for (int d = n_levels - 1; d >= top; --d)
    if (lev[d].n > 0)
      hipLaunchKernelGGL(k_ic_level, dim3(grid(lev[d].n)), dim3(kBlock), 0, s, f, lev[d].first,
                         lev[d].n);
  hipLaunchKernelGGL(k_ic_rank_top, dim3(1), dim3(kBlock), 0, s, f, t);
  for (int d = top; d < n_levels; ++d)
    if (lev[d].n > 0)
      hipLaunchKernelGGL(k_rank_level, dim3(grid(lev[d].n)), dim3(kBlock), 0, s, f, lev[d].first,
                         lev[d].n);
  hipLaunchKernelGGL(k_emit, dim3(grid(f.n_records)), dim3(kBlock), 0, s, f);
  const int64_t n_inner = level_off[n_levels];
  const int64_t m = n_inner > n_leaves ? n_inner : n_leaves;
  if (m > 0)
    hipLaunchKernelGGL(k_map_lists, dim3(grid(m)), dim3(kBlock), 0, s, f, n_inner, n_leaves);
  if (n_leaves > 0)
    hipLaunchKernelGGL(k_fin_leaves, dim3(grid(n_leaves)), dim3(kBlock), 0, s, f, n_leaves);
  if (f.rtsah && n_inner > 0)
    hipLaunchKernelGGL(k_fin_probs, dim3(grid(n_inner)), dim3(kBlock), 0, s, f, n_inner);
  for (int d = n_levels - 1; d >= top; --d)
    if (lev[d].n > 0)
      hipLaunchKernelGGL(k_fin_level, dim3(grid(lev[d].n)), dim3(kBlock), 0, s, f, lev[d].first,
                         lev[d].n);
  if (top > 0) hipLaunchKernelGGL(k_fin_top, dim3(1), dim3(kBlock), 0, s, f, t);
  return (int)hipGetLastError();
}

}  // namespace mh

// Packet traversal for gfx950 (wave64), and the entry of plain traces: single rays take
// k_wide_whole (wide_trace.h).
//
// k_trace_packet: one RayPacket of up to 64 consecutive rays per wave, the reference's
//   packet recursion (intersectNode/firstIntersects/lastIntersects, DynBVH.cc:274-905,
//   scalar branch). Node and triangle records are read with uniform (scalar) loads, each
//   lane tests its own ray, and everything about the packet (rays still looking, rays that
//   hit, firstActive/lastActive, child order) is kept as wave-uniform masks. The
//   interval-arithmetic frustum test (DynBVH.cc:682-721) runs on wave-reduced ray bounds.
//   A wave visits one record at a time and waits for its scalar loads (vector instructions
//   take 45% of their slots), and what is uniform stays in scalar registers (vector loads of
//   the records, vector masks and a stack in LDS took 1.16 times as long: 801 against
//   706 us for 2.07M camera rays in packets of 64 over a 1M-triangle heightfield). Testing
//   both children at their parent, so that the farther one need not be pushed, was slower
//   (849 us): a child that is hit is then tested twice.
//
// Arithmetic follows the reference's scalar build operation for operation: no
// contraction (the library is compiled with -ffp-contract=off), IEEE division for
// 1/direction and the triangle reciprocal, and the reference's select-based min/max.

#include <hip/hip_runtime.h>

#include <cfloat>

#include "mh_device.h"
#include "trace_common.h"
#include "traverse.h"

namespace mh {

// wide_ks.hip, wide_wald.hip
int launch_wide_one_ks(const DevScene& sc, const BatchDev& rays, const LaunchCfg& cfg,
                       hipStream_t s);
int launch_wide_one_wald(const DevScene& sc, const BatchDev& rays, const LaunchCfg& cfg,
                         hipStream_t s);

namespace {

constexpr int kBlock = 256;
constexpr int kWaves = kBlock / 64;

// ---------------------------------------------------------------------------
// Packet traversal (one RayPacket per wave)
// ---------------------------------------------------------------------------
__device__ __forceinline__ int uni(int x) { return __builtin_amdgcn_readfirstlane(x); }
__device__ __forceinline__ float uni(float x) { return __int_as_float(uni(__float_as_int(x))); }
using Mask = unsigned long long;
__device__ __forceinline__ Mask mask_of(bool x) { return __builtin_amdgcn_ballot_w64(x); }
__device__ __forceinline__ int lowest(unsigned long long m) { return __builtin_ctzll(m); }
__device__ __forceinline__ int highest(unsigned long long m) { return 63 - __builtin_clzll(m); }

// The packet's IAData loop folds its rays in order with selects (DynBVH.cc:246-266):
//   min: acc = (acc < x) ? acc : x from FLT_MAX;  max: acc = (acc < x) ? x : acc from -FLT_MAX.
// The min fold takes a NaN (and restarts from the next ray after it) and keeps the later
// of two equal values (+0/-0); the max fold skips NaNs and keeps the earlier. A butterfly
// over (value, lane) pairs with those tie rules gives the fold's exact bits in any order.
__device__ __forceinline__ float fold_min(float x, bool contrib, int lane) {
  const unsigned long long nan = __ballot(contrib && x != x);
  const int j = nan ? highest(nan) : -1;  // the last NaN: the fold restarts after it
  float v = (contrib && lane > j) ? x : __builtin_inff();
  int p = (contrib && lane > j) ? lane : -1;
  for (int m = 32; m >= 1; m >>= 1) {
    const float y = __shfl_xor(v, m, 64);
    const int q = __shfl_xor(p, m, 64);
    const bool take = (y < v) || (!(v < y) && q > p);
    v = take ? y : v;
    p = take ? q : p;
  }
  if (j < 0) return (FLT_MAX < v) ? FLT_MAX : v;  // from the initial FLT_MAX
  if (p < 0) return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), j));
  return v;
}
__device__ __forceinline__ float fold_max(float x, bool contrib, int lane) {
  const bool use = contrib && x == x;
  float v = use ? x : -__builtin_inff();
  int p = use ? lane : 64;
  for (int m = 32; m >= 1; m >>= 1) {
    const float y = __shfl_xor(v, m, 64);
    const int q = __shfl_xor(p, m, 64);
    const bool take = (v < y) || (!(y < v) && q < p);
    v = take ? y : v;
    p = take ? q : p;
  }
  return (-FLT_MAX < v) ? v : -FLT_MAX;  // from the initial -FLT_MAX
}
__device__ __forceinline__ unsigned long long above(int b) {
  return b >= 63 ? 0ull : (~0ull << (b + 1));
}

struct IA {
  float min_rcp[3], max_rcp[3], min_org[3], max_org[3];
};

// Records at wave-uniform indices, through the scalar cache.
typedef float Float4 __attribute__((ext_vector_type(4)));
typedef const __attribute__((address_space(4))) Float4* UniformWords;
__device__ __forceinline__ UniformWords uniform_words(const void* p) {
  return (UniformWords)reinterpret_cast<unsigned long long>(p);
}
struct UniformNode {
  float lo[3], hi[3];
  int child, word;
  __device__ __forceinline__ UniformNode(const RefNode* refs, int i) {
    const UniformWords p = uniform_words(refs + i);
    const Float4 a = p[0], b = p[1];
    lo[0] = a.x;
    lo[1] = a.y;
    lo[2] = a.z;
    hi[0] = a.w;
    hi[1] = b.x;
    hi[2] = b.y;
    child = __float_as_int(b.z);
    word = __float_as_int(b.w);
  }
  __device__ __forceinline__ int children() const { return word >> 16; }
  __device__ __forceinline__ int axis() const { return word & 255; }
  __device__ __forceinline__ int left_cheaper() const { return (word >> 8) & 1; }
};
__device__ __forceinline__ PrimRecord uniform_prim(const DevScene& sc, int slot) {
  const UniformWords p = uniform_words(sc.tris + 12 * (int64_t)slot);
  const Float4 a = p[0], b = p[1], c = p[2];
  return PrimRecord{make_float4(a.x, a.y, a.z, a.w), make_float4(b.x, b.y, b.z, b.w),
                    make_float4(c.x, c.y, c.z, c.w)};
}

// Interval-arithmetic frustum exit of the scalar firstIntersects (DynBVH.cc:682-721).
__device__ __forceinline__ bool frustum_miss(const UniformNode& nd, const IA& ia) {
  float tmin_f = 1e-5f, tmax_f = FLT_MAX;
#pragma unroll
  for (int axis = 0; axis < 3; ++axis) {
    float a = nd.lo[axis] - ia.max_org[axis];
    float b = nd.hi[axis] - ia.min_org[axis];
    const float ar0 = a * ia.min_rcp[axis];
    const float ar1 = a * ia.max_rcp[axis];
    const float br0 = b * ia.min_rcp[axis];
    const float br1 = b * ia.max_rcp[axis];
    a = (br0 < br1) ? br0 : br1;
    a = (a < ar1) ? a : ar1;
    a = (a < ar0) ? a : ar0;
    b = (br0 < br1) ? br1 : br0;
    b = (b < ar1) ? ar1 : b;
    b = (b < ar0) ? ar0 : b;
    tmin_f = (tmin_f < a) ? a : tmin_f;
    tmax_f = (tmax_f > b) ? b : tmax_f;
  }
  return tmin_f > tmax_f;
}

template <bool ANY, int PRIM, bool STATS>
__global__ __launch_bounds__(kBlock) void k_trace_packet(DevScene sc, DevRays rays,
                                                         DevHits hits, int64_t n, int psize,
                                                         unsigned long long* counters) {
  const int lane = threadIdx.x & 63;
  const int wv = threadIdx.x >> 6;
  const int64_t pk = (int64_t)blockIdx.x * kWaves + wv;
  const int64_t first = pk * psize;
  if (first >= n) return;
  const int cnt = (int)((n - first) < psize ? (n - first) : psize);
  const bool in = lane < cnt;
  const int64_t ri = first + lane;

  Ray r;
  float minT;
  int st;  // 0 not hit, 1 hit, -1 masked, -3 outside the packet
  if (in) {
    load_ray(rays, ri, r);
    const bool m = rays.masked && rays.masked[ri];
    st = m ? -1 : 0;
    minT = m ? -kMaxT : rays.tmax[ri];
  } else {
    r.o[0] = r.o[1] = r.o[2] = 0.f;
    r.d[0] = r.d[1] = r.d[2] = 1.f;
    r.inv[0] = r.inv[1] = r.inv[2] = 1.f;
    st = -3;
    minT = -kMaxT;
  }
  // DynBVH::intersect IAData over the packet's unmasked rays (DynBVH.cc:246-266)
  IA ia;
  const bool contrib = st == 0;
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    ia.min_rcp[a] = uni(fold_min(r.inv[a], contrib, lane));
    ia.max_rcp[a] = uni(fold_max(r.inv[a], contrib, lane));
    ia.min_org[a] = uni(fold_min(r.o[a], contrib, lane));
    ia.max_org[a] = uni(fold_max(r.o[a], contrib, lane));
  }

  int pos = -1;
  float hu = 0.f, hv = 0.f;
  unsigned long long nbox = 0, ntri = 0;
  // Rays and boxes for which the min/max form of the slab test is exact: no product is a
  // NaN with finite origins, finite reciprocals other than zero and boxes without NaNs.
  bool plain = regular_ray(r, minT) && r.inv[0] != 0.f && r.inv[1] != 0.f && r.inv[2] != 0.f;
  plain = mask_of(in && !plain) == 0 && *sc.irregular == 0;
  Mask alive = mask_of(st == 0);  // rays still looking
  const Mask pos_x = mask_of(r.d[0] > 0.f), pos_y = mask_of(r.d[1] > 0.f),
             pos_z = mask_of(r.d[2] > 0.f);
  // The stack of (node, firstActive), at most 126 entries (the host refuses deeper trees):
  // entry k in lane k % 64 of a register pair, written and read at a wave-uniform index.
  int stk_node[2] = {0, 0}, stk_b[2] = {0, 0};
  int sp = 0, nid = 0, b = 0;
  for (;;) {
    const UniformNode nd(sc.refs, nid);
    const Mask E = alive & (~(Mask)0 << b);
    float tn;
    Mask H;
    if (plain)
      H = mask_of(slab_fast(nd.lo[0], nd.hi[0], nd.lo[1], nd.hi[1], nd.lo[2], nd.hi[2], r, minT,
                            tn));
    else
      H = mask_of(slab(nd.lo[0], nd.hi[0], nd.lo[1], nd.hi[1], nd.lo[2], nd.hi[2], r, minT, tn));
    H &= E;
    // (a node that no ray hits is left either way; the frustum test only counts then)
    if (E != 0 && !((H >> lowest(E)) & 1) && (STATS || H != 0)) {
      if (frustum_miss(nd, ia)) {
        if (STATS) nbox += 1;
        H = 0;
      } else if (STATS && H == 0) {
        nbox += __popcll(E);
      }
    }
    if (H != 0) {
      const int fa = lowest(H);
      if (STATS) nbox += __popcll(E & (fa >= 63 ? ~0ull : ((2ull << fa) - 1)));
      if (nd.children() == 0) {
        int front;
        if (ANY) {
          front = nd.left_cheaper() ? 0 : 1;
        } else {
          const int axis = nd.axis();
          const Mask ahead = axis == 0 ? pos_x : (axis == 1 ? pos_y : pos_z);
          front = ((ahead >> fa) & 1) ? 0 : 1;
        }
        const int other = nd.child + 1 - front;
        const bool here = lane == (sp & 63);
        if (sp < 64) {
          stk_node[0] = here ? other : stk_node[0];
          stk_b[0] = here ? fa : stk_b[0];
        } else {
          stk_node[1] = here ? other : stk_node[1];
          stk_b[1] = here ? fa : stk_b[1];
        }
        ++sp;
        nid = nd.child + front;
        b = fa;
        continue;
      }
      const Mask Lm = H & above(b);
      const int la = Lm ? highest(Lm) : b;
      int sb = fa, se = la + 1;
      const int end = nd.child + nd.children();
      PrimRecord next = uniform_prim(sc, nd.child);
      for (int slot = nd.child; slot < end; ++slot) {
        const PrimRecord tri = next;
        if (slot + 1 < end) next = uniform_prim(sc, slot + 1);
        if (STATS) ntri += (unsigned long long)(se - sb);
        const bool act = lane >= sb && lane < se;
        if (act) {
          float t, u, v;
          if (record_test<PRIM>(tri, r, minT, t, u, v)) {
            minT = t;
            st = 1;
            pos = slot;
            hu = u;
            hv = v;
          }
        }
        if (ANY) {
          // DynBVH.cc:329-374: opaque hits end the ray (minT = T_EPSILON); the
          // subpacket shrinks to the rays still unoccluded.
          const bool hit_here = act && st == 1;
          if (hit_here) minT = kEps;
          if (mask_of(hit_here)) {
            alive &= ~mask_of(hit_here);
            const Mask left = mask_of(act && st == 0);
            if (!left) break;
            sb = lowest(left);
            se = highest(left) + 1;
          }
        }
      }
    }
    if (sp == 0) break;
    --sp;
    if (sp < 64) {
      nid = __builtin_amdgcn_readlane(stk_node[0], sp);
      b = __builtin_amdgcn_readlane(stk_b[0], sp);
    } else {
      nid = __builtin_amdgcn_readlane(stk_node[1], sp & 63);
      b = __builtin_amdgcn_readlane(stk_b[1], sp & 63);
    }
  }
  if (in) {
    const int32_t prim = st == 1 ? sc.obj_ids[pos] : (st == -1 ? -2 : -1);
    store_hit(hits, ri, prim, minT, hu, hv, st != 0);
  }
  if (STATS && counters && lane == 0) {
    atomicAdd(counters + 0, nbox);
    atomicAdd(counters + 1, ntri);
  }
}

template <bool ANY, int PRIM>
int launch_packets(const DevScene& sc, const DevRays& rays, const DevHits& hits, int64_t n,
                   const LaunchCfg& cfg, hipStream_t s) {
  const int64_t packets = (n + cfg.packet_size - 1) / cfg.packet_size;
  const int64_t blocks = (packets + kWaves - 1) / kWaves;
  unsigned long long* c = reinterpret_cast<unsigned long long*>(cfg.counters);
  if (c)
    hipLaunchKernelGGL((k_trace_packet<ANY, PRIM, true>), dim3((unsigned)blocks), dim3(kBlock), 0,
                       s, sc, rays, hits, n, cfg.packet_size, c);
  else
    hipLaunchKernelGGL((k_trace_packet<ANY, PRIM, false>), dim3((unsigned)blocks), dim3(kBlock), 0,
                       s, sc, rays, hits, n, cfg.packet_size, c);
  return (int)hipGetLastError();
}

}  // namespace

int launch_trace(const DevScene& sc, const DevRays& rays, const DevHits& hits, int64_t n,
                 const LaunchCfg& cfg, void* stream) {
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  if (cfg.packet_size <= 1) {
    const BatchDev b{rays, hits, n, 0, cfg.any_hit ? 1u : 0u, 0};
    return sc.prim_kind == 1 ? launch_wide_one_wald(sc, b, cfg, s) : launch_wide_one_ks(sc, b, cfg, s);
  }
  if (cfg.any_hit) {
    return sc.prim_kind == 1 ? launch_packets<true, 1>(sc, rays, hits, n, cfg, s)
                             : launch_packets<true, 0>(sc, rays, hits, n, cfg, s);
  }
  return sc.prim_kind == 1 ? launch_packets<false, 1>(sc, rays, hits, n, cfg, s)
                           : launch_packets<false, 0>(sc, rays, hits, n, cfg, s);
}

}  // namespace mh

// Single-ray traversal over the four-wide nodes for gfx950 (wave64): DynBVH::intersect on
// one-ray packets (Model/Groups/DynBVH.cc:101-404), with the reference's results bit for
// bit. Included by wide_ks.hip and wide_wald.hip, one per triangle test.
//
// What has to match. The reference visits the leaves in an order fixed by the split axes
// and the direction's signs (isLeftCheaper for any hit, DynBVH.cc:386-398), and enters a
// leaf if its slab test and those of the inner records above it pass with the minT of that
// moment. Boxes nest and every step of the slab test is monotone (products that are not
// numbers aside, see leaf_entered), so a leaf whose own test passes passes it all the way up:
// which leaves are entered depends on the leaf boxes alone, and inner boxes may be tested with
// any arithmetic that never rejects what the reference accepts. So here an inner test is one
// fused multiply-add a plane, widened by more than all rounding errors (WideRay), two tree
// levels are tested at a time, and the exact test of a leaf is run only for leaves that gave a
// hit: when a later hit replaces it or the ray ends, with the minT of the hit's acceptance (a
// leaf that passes with that one passes with the larger one of its visit). While every such
// leaf passes, minT is the reference's at every leaf, and the leaves visited here are its
// leaves and others that accepted nothing. Should one fail, which takes a hit within rounding
// of its leaf's box, the ray is traced again, as are rays outside the bounds below. Nothing is
// assumed of where triangles lie in their boxes: a grazing ray's computed distance may lie
// before the box, and a loaded tree's boxes may be those of another pose. (Leaving out the
// test of a hit replaced by one that is clearly nearer gained up to 0.8%: 1,593 against 1,606
// us for 12 uneven batches in a 300,000-triangle soup, nothing on a heightfield.)
//
// Rays that are traced again, and trees whose boxes do not nest, are traversed on the 32-byte
// records, the two children of a record a step, every box tested exactly (wide_pair_step;
// k_wide_lanes, whose lanes are at different rays, runs the reference's own steps in one loop
// instead, wide_redo). A whole wave may need it: of vertical rays from a heightfield's
// vertices, which lie on box planes, every one with positive zero components hits a leaf that
// the reference does not enter (500,000: 149 us, 172 with wide_redo, 47 on binary nodes alone,
// which visit no such leaf; 61 from between the vertices).
//
// How the wave works. A node visit costs about 110 vector instructions and a triangle test
// about 95, and each waits about 850 cycles for its record (L2 and MALL; a 10,000-triangle
// tree as well). Every step the wave votes: node visits for the lanes at a node, or
// triangle tests for the lanes at a leaf, whichever more lanes wait for; the others keep
// their place. Walking every lane to its leaf before any triangle is tested (two loops, as
// in batch_kernel.h) took 84 node visits and 21 tests a wave on a 10,000-triangle soup's
// camera rays against 61 and 10 by vote, 147 and 59 against 100 and 44 at 200,000. Then one
// stack entry is taken off for every lane that needs it: a loop until each lane has one that
// is still in front of its hit cost more (up to three LDS round trips a step) than the
// steps that the lanes with a culled entry sit out.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cfloat>

#include "batch_kernel.h"
#include "mh_device.h"
#include "trace_common.h"
#include "traverse.h"

namespace mh {

// A plane at p of axis k is met at p * inv[k] + c, with c = cn[k] for a near plane and cf[k]
// for a far one.
struct WideRay {
  float inv[3], cn[3], cf[3];
  int on[3], of[3];  // byte offsets of the near and the far row among an axis's two rows
};

// Sets w up for a ray; false if the bounds do not hold for it. reach is the largest
// |coordinate| of the root box. With R = reach + max|o| every product below is at most
// R |inv|; its roundings and those of the reference's (p - o) * inv come to at most six
// times 2^-24 R |inv|, and c is moved outward by eight. A reciprocal is cut at 2^40 times
// the smallest one (a direction component of zero has an infinite one): the cut plane
// distances keep their signs, and the widening of such an axis alone, 2^19 R m, is beyond
// any distance inside the root box, so a ray between the planes still passes. The bounds on
// R m keep every product along the longest component finite, so every box the reference
// enters is left at a finite distance, also for a ray with an infinite minT.
__device__ __forceinline__ bool wide_setup(float reach, const Ray& r, float minT, WideRay& w) {
  const float m = fminf(fminf(fabsf(r.inv[0]), fabsf(r.inv[1])), fabsf(r.inv[2]));
  const float R = reach + fmaxf(fmaxf(fabsf(r.o[0]), fabsf(r.o[1])), fabsf(r.o[2]));
  const float q = R * m, lim = m * 0x1p40f;
  bool ok = q >= 0x1p-60f && q <= 0x1p60f && m >= 0x1p-60f && m <= 0x1p60f && !(minT != minT);
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    ok = ok && !(r.o[k] != r.o[k]) && !(r.d[k] != r.d[k]);
    const float a = fminf(fabsf(r.inv[k]), lim);
    w.inv[k] = __builtin_copysignf(a, r.inv[k]);
    const float p = R * 0x1p-21f * a;
    const float c = -(r.o[k] * w.inv[k]);
    w.cn[k] = c - p;
    w.cf[k] = c + p;
    w.on[k] = w.inv[k] < 0.f ? 16 : 0;
    w.of[k] = 16 - w.on[k];
  }
  return ok;
}

// A condition as the mask of the wave's lanes, and back: logic on masks is scalar work.
__device__ __forceinline__ unsigned long long wave_mask(bool b) {
  return __builtin_amdgcn_ballot_w64(b);
}
__device__ __forceinline__ bool lane_bit(unsigned long long m) {
  return __builtin_amdgcn_inverse_ballot_w64(m);
}

constexpr int kIdle = (int)0x80000000;  // no ray
constexpr int kPop = (int)0x80000001;   // takes its next node from the stack

// One lane's ray.
struct WideLane {
  Ray r;  // inv is only live while the ray is set up
  WideRay w;
  RayHit h;
  float enter;   // minT when the hit in h was accepted
  unsigned ord;  // where the ray's visit order lies in WideNode::order (kAnyOrder: any hit)
  int cur;       // node (>= 0), leaf code, kPop or kIdle
  bool bad;      // the reference's own steps have to trace it
  unsigned nbox, ntri;  // COUNT: box and triangle tests
};
constexpr unsigned kAnyOrder = 24;

// Whether the ray passes the reference's slab test of the leaf that holds object slot `slot`,
// or false where that test and those of the boxes around the leaf may differ:
//   - along a component so small that its reciprocal may have been cut (wide_setup), the
//     origin has to lie between the leaf's planes, or on the near one: then the cut reciprocal
//     changes no near distance and brings the far one closer, so a box that passes passes uncut
//     as well (without forming the reciprocal again);
//   - across a zero component the leaf must not be flat in the origin's plane: products that
//     are not numbers drop out of the reference's test there, and a box around such a leaf
//     need not pass.
__device__ __forceinline__ bool leaf_entered(const DevScene& sc, const WideLane& L, int slot,
                                             float minT) {
  int rec = sc.leaf_at[slot];
  while (rec < 0) rec = sc.leaf_at[--slot];
  const RefNode& nd = sc.refs[rec];
  Ray r = L.r;
#pragma unroll
  for (int k = 0; k < 3; ++k) r.inv[k] = L.w.inv[k];
  const float dmin = fminf(fminf(fabsf(r.d[0]), fabsf(r.d[1])), fabsf(r.d[2]));
  const float dmax = fmaxf(fmaxf(fabsf(r.d[0]), fabsf(r.d[1])), fabsf(r.d[2]));
  if (dmin * 0x1p39f < dmax) {
    bool same = true;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      const float o = r.o[k], lo = nd.box.lo[k], hi = nd.box.hi[k];
      const bool zero = r.d[k] == 0.f, neg = r.inv[k] < 0.f;
      const bool between = neg ? (lo < o) & (o <= hi) : (lo <= o) & (o < hi);
      same &= (fabsf(r.d[k]) * 0x1p39f >= dmax) | (zero ? (lo != o) | (hi != o) : between);
      r.inv[k] = zero ? __builtin_copysignf(__builtin_inff(), r.inv[k]) : r.inv[k];
    }
    if (!same) return false;
  }
  float tn;
  return slab(nd.box.lo[0], nd.box.hi[0], nd.box.lo[1], nd.box.hi[1], nd.box.lo[2], nd.box.hi[2],
              r, minT, tn);
}

// The lanes that meet one box of a node.
__device__ __forceinline__ unsigned long long wide_box(float nx, float fx, float ny, float fy,
                                                       float nz, float fz, const WideRay& w,
                                                       float minT, float& tn) {
  const float ax = __builtin_fmaf(nx, w.inv[0], w.cn[0]), bx = __builtin_fmaf(fx, w.inv[0], w.cf[0]);
  const float ay = __builtin_fmaf(ny, w.inv[1], w.cn[1]), by = __builtin_fmaf(fy, w.inv[1], w.cf[1]);
  const float az = __builtin_fmaf(nz, w.inv[2], w.cn[2]), bz = __builtin_fmaf(fz, w.inv[2], w.cf[2]);
  tn = fmaxf(fmaxf(fmaxf(ax, ay), az), kEps);
  const float tf = fminf(fminf(bx, by), bz);
  return wave_mask(tn <= tf) & wave_mask(tn <= minT);
}

// Per-lane stack, its newest S entries in LDS ([entry][lane], no bank conflicts), older ones
// in the thread's spill column, which holds n - S for a stack of at most n (three a wide node;
// one a level on the records). sp and base count in steps of U bytes.
template <int S, int BLOCK>
struct WideStack {
  static_assert((S & (S - 1)) == 0 && S > 4, "ring size is a power of two");
  static constexpr int U = BLOCK * 8, RM = (S - 1) * U;
  MH_LDS char* col;
  MH_GLOBAL unsigned long long* spill;  // [depth][spill_stride], this thread's column
  int64_t spill_stride;
  int sp = 0, base = 0;  // entries [base, sp) are in the ring, [0, base) spilled

  __device__ __forceinline__ WideStack(unsigned long long* lds, unsigned long long* area,
                                       int64_t stride, int64_t gtid, int tid)
      : col((MH_LDS char*)(MH_LDS unsigned long long*)lds + 8 * tid),
        spill((MH_GLOBAL unsigned long long*)area + gtid), spill_stride(stride) {}

  __device__ __forceinline__ MH_LDS unsigned long long* at(int p) const {
    return (MH_LDS unsigned long long*)(col + (p & RM));
  }
  __device__ __forceinline__ MH_GLOBAL unsigned long long* spilled(int p) const {
    return spill + (int64_t)(p / U) * spill_stride;
  }
  __device__ __forceinline__ void reset() { sp = base = 0; }
  // Up to three entries, the deepest first; each is written, and kept for the lanes of its
  // mask. Room is made for three whatever is kept.
  __device__ __forceinline__ void push3(unsigned long long ma, int ra, float ta,
                                        unsigned long long mb, int rb, float tb,
                                        unsigned long long mc, int rc, float tc) {
    if (wave_mask(sp - base > (S - 3) * U)) {
      while (sp - base > (S - 3) * U) {
        *spilled(base) = *at(base);
        base += U;
      }
    }
    *at(sp) = stack_entry(ra, ta);
    sp += lane_bit(ma) ? U : 0;
    *at(sp) = stack_entry(rb, tb);
    sp += lane_bit(mb) ? U : 0;
    *at(sp) = stack_entry(rc, tc);
    sp += lane_bit(mc) ? U : 0;
  }
  // One entry.
  __device__ __forceinline__ void push1(unsigned long long m, int r, float t) {
    if (wave_mask(sp - base > RM)) {
      if (sp - base > RM) {
        *spilled(base) = *at(base);
        base += U;
      }
    }
    *at(sp) = stack_entry(r, t);
    sp += lane_bit(m) ? U : 0;
  }
  // The newest entry of the lanes that have one (`have`); the caller takes it off.
  __device__ __forceinline__ unsigned long long top(bool have) {
    unsigned long long e = *at(sp - U);
    const unsigned long long low = wave_mask(have) & wave_mask(sp == base);
    if (low) {
      if (lane_bit(low)) {
        base -= U;
        e = *spilled(base);
      }
    }
    return e;
  }
};

// Visits node L.cur: the boxes two levels down, the nearest in visit order next, the others
// on the stack.
template <int S, int BLOCK>
__device__ __forceinline__ void wide_node_step(const DevScene& sc, WideLane& L,
                                               WideStack<S, BLOCK>& st) {
  const MhBufRsrc wt = record_table(sc.wide, sizeof(WideNode), sc.n_wide);
  const WideRay& w = L.w;
  const float4 NX = fetch_record_at(wt, L.cur, w.on[0], 0), FX = fetch_record_at(wt, L.cur, w.of[0], 0);
  const float4 NY = fetch_record_at(wt, L.cur, w.on[1], 32), FY = fetch_record_at(wt, L.cur, w.of[1], 32);
  const float4 NZ = fetch_record_at(wt, L.cur, w.on[2], 64), FZ = fetch_record_at(wt, L.cur, w.of[2], 64);
  const float4 D = fetch_record(wt, L.cur, 96);
  const unsigned order = __float_as_uint(fetch_record(wt, L.cur, 112).x) >> L.ord;
  float t0, t1, t2, t3;
  const unsigned long long H0 = wide_box(NX.x, FX.x, NY.x, FY.x, NZ.x, FZ.x, w, L.h.minT, t0);
  const unsigned long long H1 = wide_box(NX.y, FX.y, NY.y, FY.y, NZ.y, FZ.y, w, L.h.minT, t1);
  const unsigned long long H2 = wide_box(NX.z, FX.z, NY.z, FY.z, NZ.z, FZ.z, w, L.h.minT, t2);
  const unsigned long long H3 = wide_box(NX.w, FX.w, NY.w, FY.w, NZ.w, FZ.w, w, L.h.minT, t3);
  const int r0 = __float_as_int(D.x), r1 = __float_as_int(D.y), r2 = __float_as_int(D.z),
            r3 = __float_as_int(D.w);
  // into visit order: swap inside the left pair, inside the right pair, and the pairs
  const unsigned long long P = wave_mask((order & 1u) != 0), Lm = wave_mask((order & 2u) != 0),
                           Rm = wave_mask((order & 4u) != 0);
  const bool sp = lane_bit(P), sl = lane_bit(Lm), sr = lane_bit(Rm);
  const float ta = sl ? t1 : t0, tb = sl ? t0 : t1, tc = sr ? t3 : t2, td = sr ? t2 : t3;
  const int ra = sl ? r1 : r0, rb = sl ? r0 : r1, rc = sr ? r3 : r2, rd = sr ? r2 : r3;
  const float u1 = sp ? td : tb, u2 = sp ? ta : tc, u3 = sp ? tb : td;
  const int q0 = sp ? rc : ra, q1 = sp ? rd : rb, q2 = sp ? ra : rc, q3 = sp ? rb : rd;
  const unsigned long long a = (Lm & H1) | (~Lm & H0), b = (Lm & H0) | (~Lm & H1),
                           c = (Rm & H3) | (~Rm & H2), d = (Rm & H2) | (~Rm & H3);
  const unsigned long long G0 = (P & c) | (~P & a), G1 = (P & d) | (~P & b),
                           G2 = (P & a) | (~P & c), G3 = (P & b) | (~P & d);
  st.push3(G3 & (G0 | G1 | G2), q3, u3, G2 & (G0 | G1), q2, u2, G1 & G0, q1, u1);
  int cur = lane_bit(G3) ? q3 : kPop;
  cur = lane_bit(G2) ? q2 : cur;
  cur = lane_bit(G1) ? q1 : cur;
  L.cur = lane_bit(G0) ? q0 : cur;
}

// Tests the triangle of `slot`; true when that ends an any-hit ray.
template <int PRIM>
__device__ __forceinline__ bool wide_tri(const DevScene& sc, WideLane& L, int slot,
                                         const PrimRecord& p) {
  float t, u, v;
  if (!record_test<PRIM>(p, L.r, L.h.minT, t, u, v)) return false;
  L.enter = L.h.minT;
  L.h = RayHit{t, slot, u, v};
  return L.ord == kAnyOrder;
}

// Tests two triangles of leaf L.cur (every one where it holds kLeafCountInline or more), both
// fetched at once: a surface's leaves hold two as a rule, and a second step for the second
// one would wait for its record again. (One a step: 1M incoherent rays over the 1M-triangle
// heightfield 228 against 205 us, shadow rays 239 against 214. Past the last slot the
// descriptor reads zeros.)
// PAIRS: the leaf's own box has been tested. COUNT: the tests are counted.
template <int PRIM, bool PAIRS, bool COUNT>
__device__ __forceinline__ void wide_leaf_step(const DevScene& sc, WideLane& L) {
  const int code = ~L.cur;
  const int slot = code >> kLeafCountBits;
  const int count = code & kLeafCountInline;  // left in the leaf; 0 in an empty slot's code
  const int old = PAIRS ? -1 : L.h.best;
  const float entered = L.enter;
  const PrimRecord p = fetch_prim(sc, slot), q = fetch_prim(sc, slot + 1);
  hold_prim(p);
  hold_prim(q);
  bool done = count > 0 && wide_tri<PRIM>(sc, L, slot, p);
  if (COUNT) L.ntri += count > 1 && !done ? 2 : 1;
  if (!done && count > 1) done = wide_tri<PRIM>(sc, L, slot + 1, q);
  if (!done && count == kLeafCountInline) {
    const int end = slot + sc.big_count[slot];
    for (int k = slot + 2; k < end && !done; ++k) {
      if (COUNT) ++L.ntri;
      done = wide_tri<PRIM>(sc, L, k, fetch_prim(sc, k));
    }
  }
  // (of two hits in this leaf the later one's test covers both: its minT is the smaller one)
  if (old >= 0 && L.h.best != old) L.bad |= !leaf_entered(sc, L, old, entered);
  if (done)
    L.cur = kIdle;
  else if (count > 2 && count < kLeafCountInline)
    L.cur -= 2 * ((1 << kLeafCountBits) - 1);  // code: two slots on, two triangles fewer
  else
    L.cur = kPop;
}

// wide_pair_step's reference of a record: twice its first child, plus one if the ray visits
// the second child first, or the leaf code.
__device__ __forceinline__ int pair_ref(const WideLane& L, int child, int word) {
  const int n = word >> 16;
  if (n != 0) return ~((child << kLeafCountBits) | (n < kLeafCountInline ? n : kLeafCountInline));
  const int first = L.ord == kAnyOrder ? (word >> 8) & 1 : (L.r.dpos >> (word & 3)) & 1;
  return 2 * child + 1 - first;
}

// Visits the children L.cur of an inner record: the boxes of both are tested as the reference
// tests them (the farther one's distance again when it is taken off the stack, which is its
// later test with the minT of that moment).
template <bool COUNT, int S, int BLOCK>
__device__ __forceinline__ void wide_pair_step(const DevScene& sc, WideLane& L,
                                               WideStack<S, BLOCK>& st) {
  if (COUNT) L.nbox += 2;
  const float4* p = reinterpret_cast<const float4*>(sc.refs + (L.cur >> 1));
  const float4 A = p[0], B = p[1], C = p[2], D = p[3];
  Ray r = L.r;
#pragma unroll
  for (int k = 0; k < 3; ++k) r.inv[k] = L.w.inv[k];
  float t0, t1;
  const unsigned long long H0 = wave_mask(slab(A.x, A.w, A.y, B.x, A.z, B.y, r, L.h.minT, t0)),
                           H1 = wave_mask(slab(C.x, C.w, C.y, D.x, C.z, D.y, r, L.h.minT, t1)),
                           F = wave_mask((L.cur & 1) != 0);
  const int r0 = pair_ref(L, __float_as_int(B.z), __float_as_int(B.w)),
            r1 = pair_ref(L, __float_as_int(D.z), __float_as_int(D.w));
  const bool f = lane_bit(F);
  st.push1(H0 & H1, f ? r0 : r1, f ? t0 : t1);
  L.cur = lane_bit(H0 & H1) ? (f ? r1 : r0) : (lane_bit(H0) ? r0 : (lane_bit(H1) ? r1 : kPop));
}

// One step of the wave; a lane at a leaf weighs `weight` quarters of one at a node.
template <int PRIM, bool PAIRS, bool COUNT, int S, int BLOCK>
__device__ __forceinline__ void wide_step(const DevScene& sc, WideLane& L, int weight,
                                          WideStack<S, BLOCK>& st) {
  const unsigned long long at_node = wave_mask(L.cur >= 0);
  const unsigned long long at_leaf = wave_mask(L.cur < 0) & wave_mask(L.cur > kPop);
  if (weight * __popcll(at_leaf) >= 4 * __popcll(at_node)) {
    if (lane_bit(at_leaf)) wide_leaf_step<PRIM, PAIRS, COUNT>(sc, L);
  } else if (lane_bit(at_node)) {
    if constexpr (PAIRS)
      wide_pair_step<COUNT, S, BLOCK>(sc, L, st);
    else
      wide_node_step<S, BLOCK>(sc, L, st);
  }
  if (L.cur == kPop) {
    const bool have = st.sp > 0;
    const unsigned long long e = st.top(have);
    st.sp -= have ? st.U : 0;
    L.cur = !have ? kIdle
                  : (__uint_as_float((unsigned)(e >> 32)) <= L.h.minT ? (int)(unsigned)e : kPop);
  }
}

// The reference's own traversal of ray i, on its 32-byte records.
template <int PRIM, bool COUNT, int S, int BLOCK, class Index>
__device__ __forceinline__ void wide_redo(const DevScene& sc, const GRays& rays, Index i,
                                          WideLane& L, WideStack<S, BLOCK>& st) {
  const bool any = L.ord == kAnyOrder;
  Ray r;
  load_ray(rays, i, r);
  RayHit h{rays.tmax[i], -1, 0.f, 0.f};
  int cur = 0;
  st.reset();
  for (;;) {
    const RefNode nd = sc.refs[cur];
    float tn;
    if (slab(nd.box.lo[0], nd.box.hi[0], nd.box.lo[1], nd.box.hi[1], nd.box.lo[2], nd.box.hi[2], r,
             h.minT, tn)) {
      if (nd.children != 0) {
        bool done = false;
        for (int k = 0; k < nd.children && !done; ++k) {
          float t, u, v;
          if (COUNT) ++L.ntri;
          if (prim_test<PRIM>(sc, nd.child + k, r, h.minT, t, u, v)) {
            h = RayHit{t, nd.child + k, u, v};
            done = any;
          }
        }
        if (done) break;
      } else {
        if (COUNT) L.nbox += 2;
        const int front = any ? ((nd.bits & 1) ? 0 : 1) : (((r.dpos >> (nd.axis & 3)) & 1) ? 0 : 1);
        st.push1(~0ull, nd.child + 1 - front, 0.f);
        cur = nd.child + front;
        continue;
      }
    }
    if (st.sp == 0) break;
    cur = (int)(unsigned)st.top(true);
    st.sp -= st.U;
  }
  L.h = h;
}

// Starts ray L.r on the records.
__device__ __forceinline__ void pair_start(const DevScene& sc, WideLane& L) {
#pragma unroll
  for (int k = 0; k < 3; ++k) L.w.inv[k] = L.r.inv[k];
  const RefNode& nd = sc.refs[0];
  float tn;
  const bool in = slab(nd.box.lo[0], nd.box.hi[0], nd.box.lo[1], nd.box.hi[1], nd.box.lo[2],
                       nd.box.hi[2], L.r, L.h.minT, tn);
  L.bad = false;
  L.cur = in ? pair_ref(L, nd.child, (nd.children << 16) | (nd.bits << 8) | nd.axis) : kIdle;
}

// Starts ray i of `rays` in an idle lane (Index: 32 bits where the views were moved to the
// wave's first ray, so that the addresses are a scalar base and a lane offset).
template <int S, int BLOCK, class Index>
__device__ __forceinline__ void wide_start(const DevScene& sc, float reach, const GRays& rays,
                                           Index i, bool any, int irregular, WideLane& L,
                                           WideStack<S, BLOCK>& st) {
  load_ray(rays, i, L.r);
  L.h = RayHit{rays.tmax[i], -1, 0.f, 0.f};
  L.enter = L.h.minT;
  st.reset();
  L.ord = any ? kAnyOrder : 3u * (L.r.dpos & 7u);
  L.nbox = 1;  // the root's
  L.ntri = 0;
  if (irregular == 1) {
    pair_start(sc, L);
    return;
  }
  const bool ok = (irregular == 0) & wide_setup(reach, L.r, L.h.minT, L.w);
  L.bad = !ok;
  L.cur = ok ? sc.root_ref : kIdle;
}

// Whether the leaf of the ray's hit has yet to show that the reference enters it, and does not.
__device__ __forceinline__ bool last_leaf_missed(const DevScene& sc, const WideLane& L) {
  return !L.bad && L.h.best >= 0 && !leaf_entered(sc, L, L.h.best, L.enter);
}

// Stores the hit of a lane that has come to the end of ray i.
template <int PRIM, bool COUNT, int S, int BLOCK, class Index>
__device__ __forceinline__ void wide_finish(const DevScene& sc, const GRays& rays,
                                            const GHits& hits, Index i, WideLane& L,
                                            WideStack<S, BLOCK>& st) {
  if (L.bad) wide_redo<PRIM, COUNT, S, BLOCK>(sc, rays, i, L, st);
  const bool hit = L.h.best >= 0;
  store_hit(hits, i, hit ? sc.obj_ids[L.h.best] : -1, (L.ord == kAnyOrder && hit) ? kEps : L.h.minT, L.h.u,
            L.h.v, hit);
}

struct WideArgs {
  DevScene sc;
  const BatchTable* table;  // a table of batches, or null
  BatchDev one;             // table null: the only batch
  unsigned long long* ctr;  // u64[2], zero between launches; null with a static stride
  unsigned long long* counters;  // COUNT: box and triangle tests
  unsigned long long* spill;
  int64_t spill_stride;
  int nb;       // batches of the table, as the host counted them
  int refill;   // k_wide_lanes: idle lanes of a wave that make it take rays
  int chunk;    // rays a wave takes at a time ...
  int fair;     // ... at most total / fair where fair > 0, at least 64
  int remap;    // give each XCD a contiguous share of the first chunks
  int reverse;  // hand chunks out from the end of the table
  int weight;   // wide_step
  int pairs;    // table null: traverse the records whatever the tree
};

// The kernel's arguments, to be read again (by scalar loads) where they are used: held in
// registers from the start they crowd out others, and filling them in costs a wave of one
// chunk more than it saves.
__device__ __forceinline__ const WideArgs& args_again() {
  auto p = __builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(p));
  return *(const WideArgs*)p;
}

__device__ __forceinline__ float root_reach(const DevScene& sc) {
  const RefNode& root = sc.refs[0];
  float reach = 0.f;
#pragma unroll
  for (int k = 0; k < 3; ++k)
    reach = fmaxf(reach, fmaxf(fabsf(root.box.lo[k]), fabsf(root.box.hi[k])));
  return reach;
}

__device__ __forceinline__ GRays moved(GRays r, int64_t n) {
  return GRays{r.ox + n, r.oy + n, r.oz + n, r.dx + n, r.dy + n,
               r.dz + n, r.tmax + n, r.masked ? r.masked + n : nullptr};
}
__device__ __forceinline__ GHits moved(GHits h, int64_t n) {
  return GHits{h.prim ? h.prim + n : nullptr, h.t ? h.t + n : nullptr, h.u ? h.u + n : nullptr,
               h.v ? h.v + n : nullptr, h.occluded ? h.occluded + n : nullptr};
}

// Waves that trace their rays 64 at a time, a ray to a lane: chunks of `chunk` consecutive
// rays by a static stride, each cut where a batch ends. A wave lives for about ten steps
// on camera rays, so what it does beside them is kept short: no lane hand-out, batch
// arrays read where a group starts and where it ends. Five waves a SIMD. COUNT: on the
// records, whose tests are the reference's, adding up box and triangle tests.
template <int PRIM, int S, int BLOCK, bool TABLE, bool COUNT>
__global__ __launch_bounds__(BLOCK) __attribute__((amdgpu_waves_per_eu(5, 8))) void k_wide_whole(
    WideArgs a) {
  __shared__ unsigned long long s_ring[S * BLOCK];
  extern __shared__ int64_t s_start[];  // TABLE: nb entries (dynamic LDS)
  const int tid = threadIdx.x, lane = tid & 63;
  int nb = 1;
  int64_t total = a.one.count;
  if constexpr (TABLE) {
    // The dynamic LDS holds a.nb offsets; a table with more entries is cut to that.
    const BatchTable* table = a.table;
    nb = table->nb < a.nb ? table->nb : a.nb;
    total = nb == table->nb ? table->total
                            : table->batches[nb - 1].start + table->batches[nb - 1].count;
    for (int i = tid; i < nb; i += BLOCK) s_start[i] = table->batches[i].start;
    __syncthreads();
  }
  int blk = blockIdx.x;
  if (TABLE && a.remap && (gridDim.x & 7) == 0) blk = (blk & 7) * (gridDim.x >> 3) + (blk >> 3);
  WideStack<S, BLOCK> st(s_ring, a.spill, a.spill_stride, (int64_t)blockIdx.x * BLOCK + tid, tid);
  const float reach = root_reach(a.sc);
  int irregular = *a.sc.irregular;
  if (!TABLE && a.pairs && irregular == 0) irregular = 1;
  unsigned long long nbox = 0, ntri = 0;
  const int C = a.chunk;
  const int64_t stride = (int64_t)gridDim.x * (BLOCK / 64) * C;
  // (the wave's number is the same in all its lanes: kept in scalar registers)
  int64_t next = ((int64_t)blk * (BLOCK / 64) + __builtin_amdgcn_readfirstlane(tid >> 6)) * C;
  for (; next < total; next += stride) {
    int64_t pos = a.reverse ? (total - next - C > 0 ? total - next - C : 0) : next;
    const int64_t stop = a.reverse ? total - next : (next + C < total ? next + C : total);
    while (pos < stop) {
      const BatchDev* B;
      int64_t first = 0, end = stop;
      int bi = 0;
      if constexpr (TABLE) {
        bi = __builtin_amdgcn_readfirstlane(find_batch(s_start, nb, pos));
        B = a.table->batches + bi;
        first = B->start;
        end = first + B->count < stop ? first + B->count : stop;
      } else {
        B = &args_again().one;
      }
      const int n = (int)(end - pos < 64 ? end - pos : 64);
      WideLane L;
      L.cur = kIdle;
      bool live = lane < n;
      if (live) {
        const GRays rays = moved(global_view(B->rays), pos - first);
        if (rays.masked && rays.masked[lane]) {
          store_hit(moved(global_view(B->hits), pos - first), lane, -2, -kMaxT, 0.f, 0.f, true);
          live = false;
        } else {
          wide_start<S, BLOCK>(a.sc, reach, rays, (unsigned)lane, (B->flags & 1u) != 0, irregular,
                               L, st);
        }
      }
      if (!COUNT && irregular == 0) {
        while (wave_mask(L.cur != kIdle))
          wide_step<PRIM, false, COUNT, S, BLOCK>(a.sc, L, a.weight, st);
        if (live) L.bad |= last_leaf_missed(a.sc, L);
        if (wave_mask(live && L.bad)) {  // again, on the records
          const BatchDev* E = TABLE ? args_again().table->batches + bi : &args_again().one;
          const GRays rays = moved(global_view(E->rays), pos - first);
          if (live && L.bad) {
            wide_start<S, BLOCK>(a.sc, reach, rays, (unsigned)lane, L.ord == kAnyOrder, 1, L, st);
          }
        }
      }
      while (wave_mask(L.cur != kIdle))
        wide_step<PRIM, true, COUNT, S, BLOCK>(a.sc, L, a.weight, st);
      if (live) {
        const WideArgs& again = args_again();
        const BatchDev* E = TABLE ? again.table->batches + bi : &again.one;
        wide_finish<PRIM, COUNT, S, BLOCK>(again.sc, moved(global_view(E->rays), pos - first),
                                           moved(global_view(E->hits), pos - first),
                                           (unsigned)lane, L, st);
        if (COUNT) {
          nbox += L.nbox;
          ntri += L.ntri;
        }
      }
      pos += n;
    }
  }
  if (COUNT) {
    for (int m = 1; m < 64; m <<= 1) {
      nbox += __shfl_xor(nbox, m, 64);
      ntri += __shfl_xor(ntri, m, 64);
    }
    if (lane == 0) {
      atomicAdd(a.counters + 0, nbox);
      atomicAdd(a.counters + 1, ntri);
    }
  }
}

// Persistent waves over the rays of a table of batches, numbered through, whose idle lanes
// take the wave's next rays as soon as `refill` of them are idle. A wave takes `chunk` ray
// numbers at a time: first those at its own place, then by a shared counter, asked ahead of
// time. The last wave to leave clears the counter, so launches and graph replays need no
// clearing pass. Five waves a SIMD (80 registers, for six, spill). PAIRS as a whole loop of
// its own: both kinds of step in one loop cost the wide ones 5% (scalar registers).
template <int PRIM, bool PAIRS, int S, int BLOCK>
__device__ __forceinline__ void wide_lanes(const WideArgs& a, unsigned long long* s_ring,
                                           int64_t* s_start) {
  const int tid = threadIdx.x, lane = tid & 63;
  // The dynamic LDS holds a.nb offsets; a table with more entries is cut to that.
  const BatchTable* table = a.table;
  const int nb = table->nb < a.nb ? table->nb : a.nb;
  const BatchDev* batches = table->batches;
  const int64_t total =
      nb == table->nb ? table->total : batches[nb - 1].start + batches[nb - 1].count;
  for (int i = tid; i < nb; i += BLOCK) s_start[i] = batches[i].start;
  __syncthreads();
  int blk = blockIdx.x;
  if (a.remap && (gridDim.x & 7) == 0) blk = (blk & 7) * (gridDim.x >> 3) + (blk >> 3);
  const int64_t n_waves = (int64_t)gridDim.x * (BLOCK / 64);
  const int64_t wave_id = (int64_t)blk * (BLOCK / 64) + __builtin_amdgcn_readfirstlane(tid >> 6);
  WideStack<S, BLOCK> st(s_ring, a.spill, a.spill_stride, (int64_t)blockIdx.x * BLOCK + tid, tid);
  const DevScene& sc = a.sc;
  const float reach = root_reach(sc);
  const int irregular = PAIRS ? 1 : *sc.irregular;

  int64_t C = a.chunk;
  if (a.fair > 0) {  // no more than a quarter of a resident wave's share of the rays
    const int64_t share = (total / a.fair) & ~(int64_t)63;
    C = share < 64 ? 64 : (share < C ? share : C);
  }
  int64_t next = wave_id * C;      // hand-out number of the wave's next chunk
  int64_t pos = 0, end = 0;        // rays in hand
  unsigned long long ahead = 0;    // lane 0: the counter's answer, the chunk after this one
  bool asked = false;              // `next` has to be taken from it
  WideLane L;
  L.cur = kIdle;
  int64_t li = -1;  // ray in its batch, -1 none
  int bi = 0;       // its batch
  // Runs fn(rays, hits, flags, start) for the lanes of `who`, batch by batch (nearly always
  // one), so that a batch's record is read by scalar loads.
  auto by_batch = [&](bool who, auto fn) {
    for (unsigned long long todo = wave_mask(who); todo;) {
      const int b = __builtin_amdgcn_readlane(bi, __builtin_ctzll(todo));
      const unsigned long long m = wave_mask(bi == b) & todo;
      const BatchDev& B = batches[b];
      if (lane_bit(m)) fn(global_view(B.rays), global_view(B.hits), B.flags);
      todo &= ~m;
    }
  };

  for (;;) {
    const unsigned long long idle = wave_mask(L.cur == kIdle);
    const int n_idle = __popcll(idle);
    bool take_rays = n_idle >= a.refill, more = true;
    if (take_rays) {
      if (pos >= end && asked) {
        next = (int64_t)__shfl((long long)ahead, 0, 64) + n_waves * C;
        asked = false;
      }
      more = pos < end || next < total;
      take_rays = more || n_idle == 64;
    }
    if (take_rays) {
      by_batch(lane_bit(idle) && li >= 0, [&](const GRays& rays, const GHits& hits, uint32_t) {
        if (!PAIRS && irregular == 0) L.bad |= last_leaf_missed(sc, L);
        wide_finish<PRIM, false, S, BLOCK>(sc, rays, hits, li, L, st);
      });
      if (lane_bit(idle)) li = -1;
      if (!more) break;  // every lane is idle
      if (pos >= end) {
        pos = a.reverse ? (total - next - C > 0 ? total - next - C : 0) : next;
        end = a.reverse ? total - next : (next + C < total ? next + C : total);
        if (lane == 0) ahead = atomicAdd(a.ctr, (unsigned long long)C);
        asked = true;
      }
      const int64_t g = pos + __popcll(idle & ((1ull << lane) - 1ull));
      const bool take = lane_bit(idle) && g < end;
      int64_t i = 0;
      if (take) {
        bi = find_batch(s_start, nb, g);
        i = g - s_start[bi];
      }
      by_batch(take, [&](const GRays& rays, const GHits& hits, uint32_t flags) {
        if (rays.masked && rays.masked[i]) {
          store_hit(hits, i, -2, -kMaxT, 0.f, 0.f, true);
        } else {
          li = i;
          wide_start<S, BLOCK>(sc, reach, rays, i, (flags & 1u) != 0, irregular, L, st);
        }
      });
      pos = pos + n_idle < end ? pos + n_idle : end;
    }
    wide_step<PRIM, PAIRS, false, S, BLOCK>(sc, L, a.weight, st);
  }
  if (lane == 0) {
    const unsigned long long left = atomicAdd(a.ctr + 1, 1ull);
    if (left == (unsigned long long)n_waves - 1) {
      atomicExch(a.ctr, 0ull);
      atomicExch(a.ctr + 1, 0ull);
    }
  }
}

template <int PRIM, int S, int BLOCK>
__global__ __launch_bounds__(BLOCK) __attribute__((amdgpu_waves_per_eu(5, 8))) void k_wide_lanes(
    WideArgs a) {
  __shared__ unsigned long long s_ring[S * BLOCK];
  extern __shared__ int64_t s_start[];  // nb entries (dynamic LDS)
  if (*a.sc.irregular == 1)
    wide_lanes<PRIM, true, S, BLOCK>(a, s_ring, s_start);
  else
    wide_lanes<PRIM, false, S, BLOCK>(a, s_ring, s_start);
}

namespace {

template <int PRIM, int S, int BLOCK>
void launch_table(const WideArgs& a, dim3 g, hipStream_t s) {
  const size_t lds = sizeof(int64_t) * (size_t)a.nb;  // batch start offsets
  if (a.ctr)
    hipLaunchKernelGGL((k_wide_lanes<PRIM, S, BLOCK>), g, dim3(BLOCK), lds, s, a);
  else
    hipLaunchKernelGGL((k_wide_whole<PRIM, S, BLOCK, true, false>), g, dim3(BLOCK), lds, s, a);
}
template <int PRIM, int BLOCK>
int launch_table(const WideArgs& a, dim3 g, int stack_lds, hipStream_t s) {
  if (stack_lds == 8)
    launch_table<PRIM, 8, BLOCK>(a, g, s);
  else if (stack_lds == 32)
    launch_table<PRIM, 32, BLOCK>(a, g, s);
  else
    launch_table<PRIM, 16, BLOCK>(a, g, s);
  return (int)hipGetLastError();
}

// A lane at a leaf weighs as much as one at a node: a triangle test costs about what a node
// visit does. (Half of that is 4% better on camera rays and 6% worse on a soup's.)
constexpr int kLeafWeight = 4;
template <int PRIM>
int launch_wide_table(const DevScene& sc, const BatchLaunch& bl, hipStream_t s) {
  WideArgs a{};
  a.sc = sc;
  a.table = bl.table;
  a.ctr = bl.chunk == 0 ? nullptr : bl.counters;
  a.spill = reinterpret_cast<unsigned long long*>(bl.spill);
  a.spill_stride = bl.spill_stride;
  a.nb = bl.nb;
  a.refill = wide_refill(bl.refill, bl.chunk);
  a.chunk = bl.chunk == 0 ? 64 : bl.chunk;
  a.fair = bl.chunk > 64 ? 4 * bl.resident : 0;
  a.remap = bl.xcd_remap;
  a.reverse = bl.reverse;
  a.weight = kLeafWeight;
  const dim3 g(bl.blocks);
  if (bl.block == 64) return launch_table<PRIM, 64>(a, g, bl.stack_lds, s);
  if (bl.block == 128) return launch_table<PRIM, 128>(a, g, bl.stack_lds, s);
  return launch_table<PRIM, 256>(a, g, bl.stack_lds, s);
}

template <int PRIM, bool COUNT>
int launch_one(const WideArgs& a, const LaunchCfg& cfg, hipStream_t s) {
  const dim3 g(cfg.blocks), b(64);
  if (cfg.stack_lds == 8)
    hipLaunchKernelGGL((k_wide_whole<PRIM, 8, 64, false, COUNT>), g, b, 0, s, a);
  else if (cfg.stack_lds == 32)
    hipLaunchKernelGGL((k_wide_whole<PRIM, 32, 64, false, COUNT>), g, b, 0, s, a);
  else
    hipLaunchKernelGGL((k_wide_whole<PRIM, 16, 64, false, COUNT>), g, b, 0, s, a);
  return (int)hipGetLastError();
}

template <int PRIM>
int launch_wide_one(const DevScene& sc, const BatchDev& rays, const LaunchCfg& cfg, hipStream_t s) {
  WideArgs a{};
  a.sc = sc;
  a.one = rays;
  a.counters = reinterpret_cast<unsigned long long*>(cfg.counters);
  a.spill = reinterpret_cast<unsigned long long*>(cfg.spill);
  a.spill_stride = cfg.spill_stride;
  a.chunk = cfg.chunk;
  a.pairs = cfg.pairs;
  a.reverse = 1;
  a.weight = kLeafWeight;
  return a.counters ? launch_one<PRIM, true>(a, cfg, s) : launch_one<PRIM, false>(a, cfg, s);
}

}  // namespace

// One launcher per triangle test (wide_ks.hip, wide_wald.hip).
int launch_wide_table_ks(const DevScene& sc, const BatchLaunch& bl, hipStream_t s);
int launch_wide_table_wald(const DevScene& sc, const BatchLaunch& bl, hipStream_t s);
int launch_wide_one_ks(const DevScene& sc, const BatchDev& rays, const LaunchCfg& cfg,
                       hipStream_t s);
int launch_wide_one_wald(const DevScene& sc, const BatchDev& rays, const LaunchCfg& cfg,
                         hipStream_t s);

}  // namespace mh

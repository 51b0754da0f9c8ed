// Device data layout shared by the HIP kernels and the host library.
//
// HBM layout of one scene (all arrays 256-byte aligned, one allocation each):
//   refs      RefNode[2T]      reference DynBVH records, 32 B (packet traversal, refit)
//   wide      WideNode[]       one 128-B record per inner record of even depth, with the
//                              boxes of its grandchildren (single-ray traversal); record k
//                              belongs to entry k of the even level list
//   pairs     PairNode[T]      made for MH_LAYOUT_SOA launches only: one 64-B record per
//                              pair of sibling records (2p+1, 2p+2). Sibling records are
//                              allocated in pairs (nextFree += 2 from 1), so record r sits
//                              in pair (r - 1) / 2 on side (r - 1) & 1, and a node whose
//                              children are (c, c + 1) refers to pair (c - 1) / 2.
//   tris      float4[3T]       per object slot (object_ids order), 48 B:
//                              Kensler-Shirley: p0, e0 = p1-p0, e1 = p0-p2, n = e0 x e1
//                              Wald: n_u n_v n_d k | b_nu b_nv b_d n_k | c_nu c_nv c_d 0
//   obj_ids   int32[T]         object_ids
//   big_count int32[T]         leaf size at a leaf's first slot when it is >= 15
//   verts     float[3V], idx uint32[3T], base_verts float[3V]    mesh (refit, animation)
//   leaves int32[L], levels int32[I]   leaf records; inner records grouped by depth, the
//                              even depths in one list and the odd depths in another
//   leaf_at int32[T]           per object slot, the leaf record that starts there, else -1
//   costs float[2T], ssize uint32[2T], parent int32[2T]   rotating update state (parent:
//                              allocated at the first mh_scene_update)
#pragma once

#include <cstdint>

#include "sah_builder.h"

namespace mh {

// Child reference inside a PairNode: >= 0 is an inner-node (pair) index; < 0 is a leaf,
// ~((first_slot << 4) | c) with c = min(count, 15); c == 15 means "read big_count".
constexpr int kLeafCountBits = 4;
constexpr int kLeafCountInline = 15;
// Fewer than 2^26 objects: leaf codes hold first_slot << 4 in an int, and the triangle and
// pair tables (48 and 64 B per object) stay within the 4 GiB that a buffer descriptor's byte
// offsets reach.
constexpr uint32_t kMaxObjects = 1u << 26;

struct alignas(16) PairNode {
  // child 0: lo.x hi.x lo.y hi.y | lo.z hi.z ; child 1: lo.x hi.x | lo.y hi.y lo.z hi.z
  float b[12];
  int32_t ref[2];
  int32_t meta;  // bits 0-1 split axis, bit 2 isLeftCheaper
  int32_t node;  // reference record id of this inner node
};
static_assert(sizeof(PairNode) == 64, "pair node is 64 bytes");

// Inner record of even depth with the boxes two levels below it. Slots 0 and 1 are the left
// child's children, 2 and 3 the right child's; a child that is a leaf takes its side's
// first slot itself and leaves the other empty. An empty slot's box is inverted, so that no
// ray meets it, and its reference is a leaf of no objects. One cache line: the node is
// fetched whole, and a lane takes the near and the far row of each axis by its own offsets.
struct alignas(128) WideNode {
  float plane[6][4];  // lo.x, hi.x, lo.y, hi.y, lo.z, hi.z of the four boxes
  int32_t ref[4];     // wide node (>= 0) or leaf code
  // Visit order: bit 3 o + j for direction octant o (bit k set iff d[k] > 0), bit 24 + j for
  // any-hit rays: the second of the pair is visited first, for the pair of children (j = 0),
  // the left child's pair (1) and the right child's (2).
  uint32_t order;
  int32_t pad[3];
};
static_assert(sizeof(WideNode) == 128, "wide node is one cache line");
// Wide nodes within the 4 GiB that a buffer descriptor's byte offsets reach. Trees of more
// (from about 50M triangles on) are traversed on their records.
constexpr uint32_t kMaxWide = 1u << 25;
constexpr int32_t kWideEmpty = -1;  // ~((0 << kLeafCountBits) | 0)

struct DevScene {
  const WideNode* wide;
  uint32_t n_wide;         // the bound of the wide table's descriptor
  const int32_t* leaf_at;
  // 1: single rays traverse the records instead of the wide nodes. The tree's boxes do not
  // nest or its leaves overlap (a loaded tree), a box is not a number, or there are more
  // than kMaxWide wide nodes. Beyond 1: big_count does not hold either (leaves of
  // kLeafCountInline or more objects that start at one slot), every ray takes the
  // reference's own steps.
  const int32_t* irregular;
  const RefNode* refs;
  const float* tris;  // 12 floats per slot
  const int32_t* obj_ids;
  const int32_t* big_count;
  int32_t root_ref;   // record 0: its wide node (0), or its leaf code
  int32_t prim_kind;  // 0 KS, 1 Wald
  uint32_t n_pairs;   // PairNodes of the SOA copy
  const void* pairs_soa;  // kLayoutSoa: 16-byte field k of pair p at [k * n_pairs + p], or null
  uint32_t n_slots;   // triangle records allocated (the bound of the triangle table's)
};

struct DevRays {
  const float *ox, *oy, *oz, *dx, *dy, *dz, *tmax;
  const uint8_t* masked;
};

struct DevHits {
  int32_t* prim;
  float *t, *u, *v;
  uint8_t* occluded;
};

struct LaunchCfg {
  int any_hit;
  int packet_size;    // 1 = single-ray kernels
  int stack_lds;      // 8/16/32 (single-ray)
  int blocks;         // grid size in blocks of 64 lanes (single-ray)
  int64_t* counters;  // device int64[2] or null: box and triangle tests
  int32_t* spill;     // per-thread stack spill (single-ray)
  int64_t spill_stride;
  int chunk;          // rays a wave takes at a time, 1..64 (single-ray)
  int pairs;          // traverse the records, on a stack of one entry a level (single-ray)
};

// Node layouts of the single-ray traversal (MH_LAYOUT_*). A non-root record r's box is
// also held by PairNode (r - 1) / 2, side (r - 1) & 1.
constexpr int kLayoutPair = 0;  // 128-byte WideNodes, four boxes per fetch
constexpr int kLayoutRef = 1;   // 32-byte reference records, own box tested at visit
constexpr int kLayoutSoa = 2;   // the PairNodes as four arrays of their 16-byte fields

// One ray batch of a persistent launch: rays [start, start + count) of the launch's
// global numbering are rays [0, count) of this batch.
struct BatchDev {
  DevRays rays;
  DevHits hits;
  int64_t count;
  int64_t start;
  uint32_t flags;  // bit 0: any-hit
  uint32_t pad;
};

// Device-resident batch table: the kernel reads the batch count and total from here, so a
// captured graph stays valid when the table's contents change.
struct BatchTable {
  int64_t total;
  int32_t nb;
  int32_t pad;
  BatchDev batches[1];  // nb entries
};

// Bytes of a batch launch's counters (ray counters, exit count; zero between launches).
constexpr size_t kBatchCounterBytes = 10 * sizeof(unsigned long long);

struct BatchLaunch {
  const BatchTable* table;
  int nb;  // host copy, for argument checks only
  unsigned long long* counters;  // device u64[10], zero between launches (self-resetting)
  int32_t* spill;
  int64_t spill_stride;  // blocks * block
  int blocks;
  int block;      // 64, 128 or 256 lanes
  int stack_lds;  // 8, 16 or 32
  int layout;     // kLayoutPair, kLayoutRef or kLayoutSoa
  int refill;     // idle lanes that trigger a refill, 1..63; 64 = whole-wave chunks
  int chunk;      // rays per counter grab (multiple of 64); 0 = static stride, no counter
  int xcd_remap;  // contiguous ray shares per XCD
  int reverse;    // hand chunks out from the end of the table
  int resident;   // waves of the wide kernel the device holds at once (kLayoutPair)
  int kinds;      // 0 mixed table, 1 closest-hit batches only, 2 any-hit batches only
};

// Idle lanes that make a wave of the wide kernel take rays (kLayoutPair): the caller's, but
// whole-wave chunks of more than 64 rays go by this many instead of waiting for the last lane,
// and no chunk is more than a quarter of a resident wave's share of the rays. (12 uneven
// batches, 3M rays in a 300,000-triangle soup, 256-ray chunks: 1,691 us; 2,928 with 64 idle
// lanes and whole chunks. At 8, 16, 24, 32, 40, 48 and 56 idle lanes that frame takes 1634,
// 1546, 1525, 1482, 1513, 1571 and 1658 us, and 4.1M primary and bounce rays over a
// 1M-triangle heightfield 793, 747, 715, 701, 700, 702 and 748; five to eight batches of 0.5
// to 1.5M rays in 20,000 to 1M triangles differ by 1% from 24 to 48.)
constexpr int kChunkRefill = 40;
inline int wide_refill(int refill, int chunk) {
  return refill == 64 && chunk > 64 ? kChunkRefill : refill;
}
int launch_trace_batch(const DevScene& sc, const BatchLaunch& bl, void* stream);

// Launchers (trace.hip). Return hipError_t as int.
int launch_trace(const DevScene& sc, const DevRays& rays, const DevHits& hits, int64_t n,
                 const LaunchCfg& cfg, void* stream);

// The inner records of one depth: entries [first, first + n) of the level lists. The lists
// of the even depths lie one after the other from entry 0, those of the odd depths from
// entry list_cap.
struct LevelList {
  int64_t first, n;
};

struct DevRefit {
  RefNode* refs;
  WideNode* wide;
  float* tris;
  const int32_t* obj_ids;
  const float* verts;
  const uint32_t* idx;
  const int32_t* leaves;   // leaf record ids
  const int32_t* leaf_at;  // null: the leaves do not partition the slots, take the leaf list
  const int32_t* levels;
  int32_t* irregular;      // [0] DevScene::irregular, [1] set by a pass that met a NaN box
  int32_t fixed;           // DevScene::irregular without NaN boxes
  int32_t n_leaves;
  int32_t n_slots;        // T
  int32_t prim_kind;
};

// rotate.hip: DynBVH::update with tree rotations and leaf splits.
constexpr int kMaxDepth = 256;  // deepest tree the level lists hold

// The top depths of a tree that one workgroup runs in one launch, with a barrier between
// depths (refit and update): depths [0, n), each of at most kTopNodes records.
constexpr int kTopLevels = 32;
constexpr int kTopNodes = 512;
struct TopLevels {
  int32_t first[kTopLevels], cnt[kTopLevels];
  int32_t n;
};
// The top depths (every `step`-th one) that fit: fills t, returns t.n.
inline int top_levels(const LevelList* lev, int n_levels, int step, TopLevels& t) {
  int n = 0;
  for (int d = 0; d < n_levels && n < kTopLevels && lev[d].n <= kTopNodes; d += step, ++n) {
    t.first[n] = (int32_t)lev[d].first;
    t.cnt[n] = (int32_t)lev[d].n;
  }
  t.n = n;
  return n;
}

struct DevUpdate {
  RefNode* refs;
  PairNode* pairs;
  int32_t* big_count;
  float* costs;          // DynBVH::costs (Real), per record
  uint32_t* ssize;       // DynBVH::subtree_size, per record
  int32_t* parent;       // parent links of records built by leaf splits
  int32_t* ids;          // object_ids (leaf splits permute ranges)
  const float* verts;
  const uint32_t* idx;
  unsigned* next_free;   // records in use (nextFree)
  int* err;              // set when the record array is full
  int32_t* split_list;   // update: leaves whose parent's rotation may split them
  unsigned* split_count; // update: entries of split_list (cleared by the host)
  int32_t* leaf_at;      // per slot, the leaf whose first slot it is, else -1
  int32_t* irregular;    // update: [1] is set by the leaf pass for an object with a NaN box
  int32_t n_records;     // capacity, 2T
  int32_t n_old;         // update: records in use before the frame's leaf splits
  int32_t n_objects;     // T
  uint32_t large;        // largeSubtreeSize
};
// Leaf pass over the object slots (u.leaf_at), leaf splits, then one launch per two depths
// (deepest first).
int launch_update_tree(const DevUpdate& u, int64_t n_leaves, const int32_t* levels,
                       const LevelList* lev, int n_levels, void* stream);
// The PairNodes of the n inner records of a level list.
int launch_list_pairs(const DevUpdate& u, const int32_t* levels, int64_t n, void* stream);
// Depth of every record in use by pointer jumping; hist[d] inner records at depth d,
// hist[kMaxDepth] leaves, hist[kMaxDepth + 1] the deepest depth (hist, kDepthHist entries,
// cleared by the caller). Depths in dep0.
constexpr int kDepthHist = kMaxDepth + 2;
int launch_depths(const DevUpdate& u, int32_t* anc0, int32_t* dep0, int32_t* anc1, int32_t* dep1,
                  unsigned* hist, void* stream);
int launch_depth_scatter(const DevUpdate& u, const int32_t* dep, unsigned* cursor,
                         int32_t* levels, int32_t* leaves, void* stream);
// wide.hip: level lists, leaf list, leaf starts and wide nodes of a tree, top down from an
// inner root. Counters fr: [d] inner records at depth d, [kFrLeaves] leaves, [kFrOver] set
// when a list would pass its capacity, [kFrOff + d] where depth d starts in its list.
// launch_wide_top clears them and runs the even depths below n_top in one workgroup;
// launch_wide_level(d) then runs an even depth d in `blocks` workgroups: it writes the wide
// nodes of depth d and lists depths d + 1 and d + 2 and the leaves met on the way.
constexpr int kFrLeaves = kMaxDepth + 2;
constexpr int kFrOver = kMaxDepth + 3;
constexpr int kFrOff = kMaxDepth + 4;
constexpr int kFrontierWords = kFrOff + kMaxDepth + 4;
struct DevFrontier {
  unsigned* fr;
  int32_t* even;    // even level list (a wide node's index is its place here)
  int32_t* odd;
  int2* aux;        // beside each even entry, its record's first child and word
  int32_t* leaves;
  WideNode* wide;
  int32_t* irregular;  // [0] is set from `fixed` and the NaN mark [1], which is cleared
  int32_t fixed;
  unsigned cap;        // entries each list holds
  unsigned cap_wide;   // wide nodes
};
int launch_wide_top(const DevUpdate& u, const DevFrontier& f, int n_top, void* stream);
int launch_wide_level(const DevUpdate& u, const DevFrontier& f, int d, unsigned blocks,
                      void* stream);

// refit.hip
int launch_prim_setup(const DevRefit& r, void* stream);  // tris from verts (all slots)
// tris + leaf boxes, then one launch per even depth from the deepest up: the boxes of its
// records and of their children, and its wide nodes.
int launch_refit(const DevRefit& r, const LevelList* lev, int n_levels, void* stream);
int launch_displace_sine(float* verts, const float* base, int64_t n_verts, float amp, float freq,
                         float phase, void* stream);

// genrays.hip: camera rays and secondary rays from hit records.
struct RayOut {
  float *ox, *oy, *oz, *dx, *dy, *dz, *tmax;
  uint8_t* masked;  // may be null for camera rays
};
struct CameraDev {
  float eye[3], U[3], V[3], W[3];  // up * tan(vfov/2) * |W|, right * tan(hfov/2) * |W|, lookat-eye
  int xres, yres, spp;             // xres, yres multiples of 8
  unsigned long long seed;
};
struct SecondaryArgs {
  DevRays in;            // the primary rays
  const int32_t* hit_prim;
  const float* hit_t;
  const float* verts;
  const uint32_t* idx;
  float light[3];
  unsigned long long seed;
  int64_t n;
  RayOut out;
};
int launch_camera(const CameraDev& c, const RayOut& out, void* stream);
int launch_secondary(const SecondaryArgs& a, int kind /*0 shadow, 1 bounce*/, void* stream);

// util.hip: streaming copy with 16-byte vector accesses (plus a byte tail).
int launch_copy(void* dst, const void* src, size_t bytes, int cu_count, void* stream);


// Device build (build.hip): DynBVH::rebuild with the approximate SAH at every node.
constexpr int16_t kHole = -1;     // children of a temporary record no node uses
constexpr int kBuildSerial = 64;  // nodes of at most this many objects: one wave each
constexpr int kBuildVB = 1024;     // slots per virtual block of the level passes
constexpr int kBuildBins = 16;     // BVH_num_samples (DynBVH.cc:34)

// Accumulators of one level node, in 32-bit words: keys that reduce by minimum (maxima
// negated), all cleared to ones, then counts, cleared to zero.
enum : int {
  kAccBox = 0,                             // 64-bit keys: left and right box, 6 each
  kAccCen = kAccBox + 2 * 12,              // left and right centroid box, 6 each
  kAccBins = kAccCen + 12,                 // [6][bin] bin boxes
  kAccCounts = kAccBins + 6 * kBuildBins,  // objects of each bin
  kAccLess = kAccCounts + kBuildBins,      // objects left of the position
  kAccWords = (kAccLess + 1 + 31) / 32 * 32,
};
static_assert(kAccCounts % 4 == 0, "cleared four words at a time");

struct BuildSeg {  // a node of the current level: its temporary record and slot range
  int32_t rec, b, e, vb0;
};
struct BuildPlan {  // its binning and split
  int32_t axis, leaf;
  float lo_c, scale, pos, width;
};

// Counters: records in use, error, small nodes, large leaves, then the nodes and the
// virtual blocks of each level.
enum : int {
  kCtrRecords = 0,
  kCtrErr = 1,
  kCtrSmall = 2,
  kCtrBig = 3,
  kCtrSegs = 4,
  kCtrNvb = kCtrSegs + kMaxDepth + 2,
  kCtrCount = kCtrNvb + kMaxDepth + 2,
};

struct DevBuild {
  DevUpdate u;                    // temporary records, ids, mesh, counters
  float* slots;                   // 12 floats per slot: centroid, id, box
  const float* verts;
  int64_t n_verts;
  BuildSeg* seg;
  BuildSeg* seg_next;
  BuildSeg* small;
  BuildSeg* big;
  BuildPlan* plan;
  BuildPlan* plan_next;
  unsigned* acc;                  // [node][kAccWords]
  unsigned* ctr;                  // kCtr*
  int32_t* vbseg;                 // per virtual block: its node
  unsigned* vcnt;                 // per virtual block: objects left of the position (first
                                  // word), then left, right misplaced counts
  unsigned* gscan;                // exclusive scans of vcnt (left at [0, nvb], right after)
  int64_t vcap;                   // capacity of the virtual block arrays
  int32_t* lpos;
  int32_t* rpos;
  unsigned long long* rootk;      // 6 keys: vertex box
  unsigned* rootc;                // 6 keys: box of the object centroids
  int32_t level;
};

struct DevFinish {
  const RefNode* trefs;    // temporary records
  RefNode* refs;           // final records
  const unsigned* tcount;  // records in use
  int32_t* ic;             // inner records per temporary subtree
  int32_t* rank;           // preorder rank of a temporary record among inner records
  int32_t* fin;            // final number of a temporary record
  int32_t* levels;
  int32_t* leaves;
  float* costs;
  uint32_t* ssize;
  float* rt;               // RTSAH pairs (c0, c1) per final record
  float* prob[3];          // crossing probabilities per entry of levels
  const float* logtab;
  int32_t n_records;
  int32_t n_final;         // records of the tree (inner + leaves)
  uint32_t large;
  int rtsah;
};

int build_launch_setup(const DevBuild& d, int serial, void* stream);
int build_launch_level(const DevBuild& d, int64_t nseg_bound, int64_t nvb_bound, void* stream);
int build_launch_serial(const DevBuild& d, int64_t n_small, int64_t n_big, int32_t* scratch,
                        void* stream);
int build_launch_ranks(const DevFinish& f, const int64_t* level_off, int n_levels,
                       int64_t n_leaves, void* stream);

// shade.hip: hit positions, normals and texture coordinates of traced rays.
struct DevShade {
  DevRays rays;
  const int32_t* prim;
  const float *t, *u, *v;
  const float* verts;
  const uint32_t* idx;
  const float* normals;        // null: face normals
  const uint32_t* normal_idx;
  const float* tex;            // null: barycentric weights
  const uint32_t* tex_idx;
  float* out[12];              // px py pz, nx ny nz, gx gy gz, tu tv tw (each may be null)
  int64_t n;
  int32_t n_tris;
  int32_t prim_kind;
};
int launch_shade(const DevShade& s, void* stream);

}  // namespace mh

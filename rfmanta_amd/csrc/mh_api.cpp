// C ABI of libmh.so (declared in include/mh.h): scene ownership, device upload, tree
// import/export, refit and trace dispatch. No C++ exception leaves this file; every
// entry point returns a status code and records a thread-local message.

#include "mh.h"

#include <hip/hip_runtime_api.h>

#include <algorithm>
#include <cstdarg>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <fstream>
#include <map>
#include <mutex>
#include <new>
#include <stdexcept>
#include <string>
#include <vector>

#include "internal.h"
#include "mh_device.h"
#include "rtsah.h"
#include "sah_builder.h"

namespace mh_internal {

namespace {
thread_local std::string g_err;

struct Lib {
  std::mutex mu;
  bool ready = false;
  int device = 0;
  int cu_count = 0;
  size_t hbm = 0;
  char name[256] = {0};
};
Lib g_lib;
}  // namespace

int fail(int code, const char* fmt, ...) {
  char buf[512];
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(buf, sizeof(buf), fmt, ap);
  va_end(ap);
  g_err = buf;
  // The failure is reported here: take it off the thread's HIP error state too, or the
  // check after this thread's next kernel launch (hipGetLastError) would report it again.
  (void)hipGetLastError();
  return code;
}

int ensure_init() {
  std::lock_guard<std::mutex> lk(g_lib.mu);
  if (g_lib.ready) {
    HIP_OK(hipSetDevice(g_lib.device));
    return MH_OK;
  }
  int count = 0;
  HIP_OK(hipGetDeviceCount(&count));
  if (g_lib.device < 0 || g_lib.device >= count)
    return fail(MH_E_INVALID, "device %d out of range (%d devices)", g_lib.device, count);
  HIP_OK(hipSetDevice(g_lib.device));
  hipDeviceProp_t p;
  HIP_OK(hipGetDeviceProperties(&p, g_lib.device));
  g_lib.cu_count = p.multiProcessorCount;
  g_lib.hbm = p.totalGlobalMem;
  std::snprintf(g_lib.name, sizeof(g_lib.name), "%s", p.gcnArchName);
  scratch_setup(g_lib.device);
  g_lib.ready = true;
  return MH_OK;
}

int cu_count() { return g_lib.cu_count; }
const char* device_name() { return g_lib.name; }

}  // namespace mh_internal

using mh_internal::DevBuf;
using mh_internal::ensure_init;
using mh_internal::fail;
using mh_internal::g_err;
using mh_internal::g_lib;

namespace {

// Rotation state after DynBVH::rebuild with TREE_ROT: computeCost<true>(0)
// (DynBVH.cc:3388-3415) and subtree sizes (DynBVH.cc:1971-1996) of the reachable records.
void rotation_state(const std::vector<mh::RefNode>& nodes, std::vector<float>& costs,
                    std::vector<uint32_t>& ssize) {
  costs.assign(nodes.size(), 0.f);
  ssize.assign(nodes.size(), 0u);
  auto area = [](const mh::Aabb& b) {  // BBox::computeArea, float arithmetic
    const float dx = b.hi[0] - b.lo[0], dy = b.hi[1] - b.lo[1], dz = b.hi[2] - b.lo[2];
    return 2 * (dx * dy + dy * dz + dx * dz);
  };
  struct It {
    int32_t rec;
    bool done;
  };
  std::vector<It> st{{0, false}};
  while (!st.empty()) {
    const It it = st.back();
    st.pop_back();
    const mh::RefNode& n = nodes[it.rec];
    if (n.leaf()) {
      costs[it.rec] = n.children * 1.f;
      ssize[it.rec] = 1;
      continue;
    }
    if (!it.done) {
      st.push_back({it.rec, true});
      st.push_back({n.child + 1, false});
      st.push_back({n.child, false});
      continue;
    }
    const int l = n.child, r = n.child + 1;
    costs[it.rec] = 1.f + (area(nodes[l].box) * costs[l] + area(nodes[r].box) * costs[r]) /
                              area(n.box);
    ssize[it.rec] = 1 + ssize[l] + ssize[r];
  }
}

// Room for the device tree of T objects and nrec records with n_inner inner records and
// n_leaves leaves: level and leaf lists of T entries, which the rotating update needs (a
// partition of T objects has at most T leaves and T - 1 inner records), and of every record
// of a loaded tree whose leaves overlap (it can hold more leaves than objects). Of I inner
// records at most (2 I + 1) / 3 lie at even depths: all but the root have an inner parent
// at an odd depth, and that has at most two such children.
int reserve_tree(mh_scene* s, size_t nrec, size_t n_inner, size_t n_leaves) {
  const size_t T = s->nt;
  s->list_cap = std::max<size_t>({1, T, n_inner, n_leaves});
  const size_t n_wide = (2 * std::max(T, n_inner) + 1) / 3 + 1;
  int rc;
  if ((rc = s->refs.reserve(nrec * sizeof(mh::RefNode))) ||
      (rc = s->wide.reserve(n_wide * sizeof(mh::WideNode))) ||
      (rc = s->tris.reserve(T * 48)) || (rc = s->ids.reserve(T * 4)) ||
      (rc = s->big.reserve(T * 4)) || (rc = s->leaf_at.reserve(T * 4)) ||
      (rc = s->leaves.reserve(s->list_cap * 4)) || (rc = s->levels.reserve(2 * s->list_cap * 4)) ||
      (rc = s->levels_aux.reserve(s->list_cap * 8)) || (rc = s->costs.reserve(nrec * 4)) ||
      (rc = s->ssize.reserve(nrec * 4)) || (rc = s->hist.reserve(mh::kFrontierWords * 4)) ||
      (rc = s->counters.reserve(16)) || (rc = s->irregular.reserve(8)))
    return rc;
  if (!s->host_ctr) {
    void* h = nullptr;
    if (hipHostMalloc(&h, (mh::kFrontierWords + 2) * 4, hipHostMallocDefault) != hipSuccess)
      return fail(MH_E_NOMEM, "hipHostMalloc of the level counters' copy");
    s->host_ctr = static_cast<unsigned*>(h);
  }
  return MH_OK;
}

mh::DevUpdate tree_view(mh_scene* s) {
  mh::DevUpdate u{};
  u.refs = s->refs.as<mh::RefNode>();
  u.pairs = s->pairs.as<mh::PairNode>();
  u.big_count = s->big.as<int32_t>();
  u.costs = s->costs.as<float>();
  u.ssize = s->ssize.as<uint32_t>();
  u.parent = s->parent.as<int32_t>();
  u.ids = s->ids.as<int32_t>();
  u.verts = s->d_verts.as<float>();
  u.idx = s->d_idx.as<uint32_t>();
  u.leaf_at = s->leaf_at.as<int32_t>();
  u.irregular = s->irregular.as<int32_t>();
  u.n_objects = (int32_t)s->nt;
  return u;
}

// The level lists, leaf list, leaf starts and wide nodes of the tree in `refs`, whose root
// is an inner record, top down, one pass per even depth (the small depths at the top in one
// launch). sizes: the expected inner records per depth, which set the grids. The first
// batch of passes covers the expected depth with two levels to spare; a tree that turns out
// deeper gets more passes after the counters are read back. MH_UPDATE_FRONTIER_LEVELS (1 or
// more) sets the first batch's size instead, so that tests can reach the later batches.
// Copies `extra` (two words) back along with the counters; synchronises the stream.
// MH_OK, MH_E_UNSUPPORTED (inner records at more than max_levels depths) or MH_E_STATE (not
// a binary tree).
int wide_pass(mh_scene* s, const std::vector<mh::LevelList>& sizes, unsigned max_levels,
              int irregular, const unsigned* extra, unsigned extra_out[2], hipStream_t st) {
  const mh::DevUpdate u = tree_view(s);
  mh::DevFrontier f{};
  f.fr = s->hist.as<unsigned>();
  f.even = s->levels.as<int32_t>();
  f.odd = f.even + s->list_cap;
  f.aux = s->levels_aux.as<int2>();
  f.leaves = s->leaves.as<int32_t>();
  f.wide = s->wide.as<mh::WideNode>();
  f.irregular = s->irregular.as<int32_t>();
  f.fixed = irregular;
  f.cap = (unsigned)s->list_cap;
  f.cap_wide = (unsigned)(s->wide.bytes / sizeof(mh::WideNode));
  unsigned* hc = s->host_ctr;
  const int n_sizes = (int)sizes.size();
  constexpr int kEnd = mh::kMaxDepth;  // passes run at even depths below it
  int d_end = n_sizes + 2;
  if (const char* e = std::getenv("MH_UPDATE_FRONTIER_LEVELS"))
    if (const int v = std::atoi(e); v >= 1) d_end = v;
  d_end = std::min((d_end + 1) & ~1, kEnd);
  mh::TopLevels t;
  const int top = mh::top_levels(sizes.data(), n_sizes, 2, t);
  int d = std::max(2, std::min({2 * top, d_end, mh::kTopLevels}));
  HIP_OK((hipError_t)mh::launch_wide_top(u, f, d, st));
  for (;;) {
    for (; d < d_end; d += 2) {
      // workgroups for the expected size (a grid-stride loop covers any other)
      const int64_t n = d < n_sizes ? sizes[d].n : 256;
      const unsigned blocks = (unsigned)std::min<int64_t>(2048, (n + n / 4 + 255) / 256);
      HIP_OK((hipError_t)mh::launch_wide_level(u, f, d, blocks, st));
    }
    HIP_OK(hipMemcpyAsync(hc, f.fr, mh::kFrontierWords * 4, hipMemcpyDeviceToHost, st));
    if (extra)
      HIP_OK(hipMemcpyAsync(hc + mh::kFrontierWords, extra, 8, hipMemcpyDeviceToHost, st));
    HIP_OK(hipStreamSynchronize(st));
    if (hc[d_end] == 0 || d_end >= kEnd) break;
    d_end = std::min(d_end + 16, kEnd);
  }
  if (extra) {
    extra_out[0] = hc[mh::kFrontierWords];
    extra_out[1] = hc[mh::kFrontierWords + 1];
  }
  unsigned deepest = 0;
  while ((int)deepest < d_end && hc[deepest]) ++deepest;
  if (hc[d_end] || deepest > max_levels)
    return fail(MH_E_UNSUPPORTED, "tree deeper than %d levels", mh::kMaxDepth - 1);
  s->lev.clear();
  int64_t at[2] = {0, (int64_t)s->list_cap};
  uint64_t n_inner = 0;
  for (unsigned k = 0; k < deepest; ++k) {
    s->lev.push_back(mh::LevelList{at[k & 1], (int64_t)hc[k]});
    at[k & 1] += hc[k];
    n_inner += hc[k];
  }
  if (at[0] > (int64_t)s->max_wide) {
    s->fixed_irregular |= 1;
    const int32_t word = irregular | 1;
    HIP_OK(hipMemcpyAsync(s->irregular.p, &word, 4, hipMemcpyHostToDevice, st));
    HIP_OK(hipStreamSynchronize(st));
  }
  const uint64_t n_leaves = hc[mh::kFrLeaves];
  if (hc[mh::kFrOver] || n_leaves != n_inner + 1 || n_leaves > s->list_cap)
    return fail(MH_E_STATE, "the records are not a binary tree (%llu inner, %llu leaves)",
                (unsigned long long)n_inner, (unsigned long long)n_leaves);
  s->n_inner = (uint32_t)n_inner;
  s->n_leaves = (uint32_t)n_leaves;
  s->depth = deepest;
  return MH_OK;
}

// The state of a tree whose root is a leaf: no levels, one leaf at slot 0.
int leaf_root(mh_scene* s, int irregular, hipStream_t st) {
  const int32_t zero = 0, mark[2] = {irregular, 0};
  HIP_OK(hipMemcpyAsync(s->leaves.p, &zero, 4, hipMemcpyHostToDevice, st));
  HIP_OK(hipMemcpyAsync(s->irregular.p, mark, 8, hipMemcpyHostToDevice, st));
  HIP_OK(hipStreamSynchronize(st));
  s->lev.clear();
  s->n_inner = 0;
  s->n_leaves = 1;
  s->depth = 0;
  return MH_OK;
}

// Lays the reference tree out for the device: checks it, uploads its records and rotation
// state, then has the device make the lists and wide nodes. With rtsah, isLeftCheaper is
// recomputed once the records are known to form a tree (DynBVH::buildFromFile runs
// computeTraversalCost after reading, DynBVH.cc:2469-2472).
int upload(mh_scene* s, bool rtsah = false) {
  std::vector<mh::RefNode>& nodes = s->bvh.nodes;
  const uint32_t nrec = (uint32_t)nodes.size();
  const uint32_t T = s->nt;
  std::vector<int32_t> leaves;
  std::vector<mh::LevelList> sizes;  // inner records per depth
  struct It {
    int32_t rec;
    uint32_t depth;
  };
  std::vector<It> st;
  st.push_back({0, 0});
  uint32_t n_inner = 0, max_rec = 0, n_reached = 0;
  uint64_t leaf_objects = 0;
  bool nested = true;  // every box holds its children's
  std::vector<uint8_t> seen(nrec, 0);
  while (!st.empty()) {
    It it = st.back();
    st.pop_back();
    const mh::RefNode& n = nodes[it.rec];
    if (seen[it.rec]) return fail(MH_E_INVALID, "record %d is reached twice: not a tree", it.rec);
    seen[it.rec] = 1;
    ++n_reached;
    max_rec = std::max(max_rec, (uint32_t)it.rec);
    if (n.leaf()) {
      if (n.children < 0) return fail(MH_E_INVALID, "record %d: negative leaf size", it.rec);
      if ((uint32_t)n.child + (uint32_t)n.children > T || n.child < 0)
        return fail(MH_E_INVALID, "record %d: leaf range outside object_ids", it.rec);
      leaves.push_back(it.rec);
      leaf_objects += (uint32_t)n.children;
      continue;
    }
    if (n.child < 1 || (uint32_t)n.child + 1 >= nrec)
      return fail(MH_E_INVALID, "record %d: child %d outside the node array", it.rec, n.child);
    if ((n.child & 1) == 0)
      return fail(MH_E_INVALID, "record %d: child %d is not the first record of a pair "
                  "(DynBVH allocates sibling records in pairs from 1)", it.rec, n.child);
    if (n.axis > 2) return fail(MH_E_INVALID, "record %d: axis %d", it.rec, (int)n.axis);
    if (++n_inner > nrec) return fail(MH_E_INVALID, "node graph is not a tree");
    if (it.depth >= (uint32_t)mh::kMaxDepth - 1)
      return fail(MH_E_UNSUPPORTED, "tree deeper than %d levels", mh::kMaxDepth - 1);
    if (sizes.size() <= it.depth) sizes.resize(it.depth + 1, mh::LevelList{0, 0});
    ++sizes[it.depth].n;
    for (int side = 0; side < 2; ++side) {
      const mh::Aabb &b = n.box, &c = nodes[n.child + side].box;
      for (int k = 0; k < 3; ++k) nested = nested && c.lo[k] >= b.lo[k] && c.hi[k] <= b.hi[k];
    }
    st.push_back({n.child + 1, it.depth + 1});
    st.push_back({n.child, it.depth + 1});
  }
  if (rtsah) mh::compute_rtsah(nodes, 0);
  // Leaf ranges lie inside [0, T); they partition it iff their sizes sum to T and no slot
  // is covered twice.
  bool partition = leaf_objects == T;
  if (partition) {
    std::vector<uint8_t> cover(T, 0);
    for (int32_t r : leaves)
      for (int k = 0; k < nodes[r].children && partition; ++k)
        partition = !cover[nodes[r].child + k]++;
  }
  std::vector<float> costs;
  std::vector<uint32_t> ssize;
  rotation_state(nodes, costs, ssize);

  int rc;
  if ((rc = reserve_tree(s, nrec, n_inner, leaves.size()))) return rc;
  s->partition = partition;
  s->fixed_irregular = partition ? 0 : 1;
  if (!partition) {  // one big_count entry for two large leaves that start at one slot?
    std::vector<int32_t> big(T, 0);
    for (int32_t r : leaves) {
      const int n = nodes[r].children;
      if (n < mh::kLeafCountInline) continue;
      int32_t& b = big[nodes[r].child];
      if (b && b != n) s->fixed_irregular = 2;
      b = n;
    }
  }
  s->updatable = partition && n_reached == max_rec + 1;
  s->next_free = max_rec + 1;
  s->n_records = nrec;
  ++s->tree_gen;
  HIP_OK(hipMemcpy(s->refs.p, nodes.data(), nrec * sizeof(mh::RefNode), hipMemcpyHostToDevice));
  HIP_OK(hipMemcpy(s->ids.p, s->bvh.ids.data(), (size_t)T * 4, hipMemcpyHostToDevice));
  HIP_OK(hipMemcpy(s->costs.p, costs.data(), nrec * sizeof(float), hipMemcpyHostToDevice));
  HIP_OK(hipMemcpy(s->ssize.p, ssize.data(), nrec * sizeof(uint32_t), hipMemcpyHostToDevice));
  HIP_OK(hipMemset(s->leaf_at.p, 0xFF, (size_t)T * 4));
  HIP_OK(hipMemset(s->irregular.p, 0, 8));
  if (n_inner > 0) {
    if ((rc = wide_pass(s, sizes, mh::kMaxDepth - 1, s->fixed_irregular | !nested, nullptr, nullptr,
                        nullptr)))
      return rc;
    s->root_ref = 0;
  } else {
    const mh::RefNode& n = nodes[0];
    bool nan = false;
    for (int k = 0; k < 3; ++k)
      nan = nan || n.box.lo[k] != n.box.lo[k] || n.box.hi[k] != n.box.hi[k];
    if ((rc = leaf_root(s, s->fixed_irregular | nan, nullptr))) return rc;
    const int32_t zero = 0, count = n.children;
    HIP_OK(hipMemcpy(s->leaf_at.as<int32_t>() + n.child, &zero, 4, hipMemcpyHostToDevice));
    HIP_OK(hipMemcpy(s->big.as<int32_t>() + n.child, &count, 4, hipMemcpyHostToDevice));
    s->root_ref = ~((n.child << mh::kLeafCountBits) |
                    std::min<int>(n.children, mh::kLeafCountInline));
  }
  mh::DevRefit r{};
  r.tris = s->tris.as<float>();
  r.obj_ids = s->ids.as<int32_t>();
  r.verts = s->d_verts.as<float>();
  r.idx = s->d_idx.as<uint32_t>();
  r.n_slots = (int32_t)T;
  r.prim_kind = s->prim_kind;
  HIP_OK((hipError_t)mh::launch_prim_setup(r, nullptr));
  HIP_OK(hipDeviceSynchronize());
  s->built = true;
  return MH_OK;
}

int validate_ids(const std::vector<int32_t>& ids, uint32_t T) {
  if (ids.size() != T) return fail(MH_E_INVALID, "object_ids has %zu entries for %u triangles",
                                   ids.size(), T);
  std::vector<uint8_t> seen(T, 0);
  for (int32_t id : ids) {
    if (id < 0 || (uint32_t)id >= T || seen[id])
      return fail(MH_E_INVALID, "object_ids is not a permutation of the triangles");
    seen[id] = 1;
  }
  return MH_OK;
}

mh::DevScene dev_scene(const mh_scene* s) { return s->dev(); }

// mh_trace. The wide kernel gets a wave of its own for every 64 rays, up to kTraceBlocksPerCu
// times four waves per compute unit (the spill area has a column per lane), and takes them
// by a static stride from the end of the set: the hardware then starts waves as others end.
// 2M camera rays of the 1M-triangle heightfield: 161 us; 202 with half as many waves, 267
// with the resident ones alone (a wave's share of the rays fixed up front), 504 with those
// and a ray counter (its atomics come from all XCDs, about 15 ns each). From the end, since a
// camera image's rays come bottom row first and the long ones, along the ground to the
// horizon, would start late: 256 us in the other order.
constexpr int kTraceBlocksPerCu = 32;
// Sets too small to give every SIMD a wave are cut into waves of fewer rays, which wait for
// fewer others: 4,096 rays in a 10,000-triangle soup 98 us at 64 rays a wave, 67 at 4.
constexpr int64_t kMinWaveRays = 4;
// Ring entries unless the caller says: 16 (five waves per SIMD fill the LDS) spill less than
// 8 (786,432 camera and bounce rays in a 200,000-triangle soup 1274 against 1337 us), and
// where there are few waves 32 need no spill area up to a depth of 20 (allocating one takes
// a first call about 300 us). 32 with waves to spare cost occupancy: 199,023 rays 68
// against 57 us.
constexpr int kWideRing = 16, kFewWavesRing = 32;
constexpr int64_t kFewWaves = 8;  // per compute unit
// A stream's spill area, unless the resident waves alone need more: trees of up to 32 levels
// (a heightfield of 8M triangles has 25) get all the waves below this, a tree of 60 levels
// 2.8 times the resident ones, and no tree more than 965 MB.
constexpr int64_t kSpillBytes = int64_t(512) << 20;

// fixed_spill / fixed_bytes: a stack spill area the caller provides (mh_trace_noalloc);
// null = the scene's per-stream spill buffer, grown here as needed.
int trace_impl(const mh_scene* cs, const mh_rays* rays, const mh_hits* hits, int64_t n,
               uint32_t flags, const mh_trace_opts* opts, void* stream,
               void* fixed_spill = nullptr, size_t fixed_bytes = 0) {
  mh_scene* s = const_cast<mh_scene*>(cs);
  if (!s || !rays || !hits) return fail(MH_E_INVALID, "null scene, rays or hits");
  if (!s->built) return fail(MH_E_STATE, "scene has no tree: call mh_scene_build first");
  if (n < 0) return fail(MH_E_INVALID, "negative ray count");
  if (flags & ~MH_ANY_HIT) return fail(MH_E_INVALID, "unknown trace flags 0x%x", flags);
  if (n == 0) return MH_OK;
  if (!rays->ox || !rays->oy || !rays->oz || !rays->dx || !rays->dy || !rays->dz || !rays->tmax)
    return fail(MH_E_INVALID, "ray arrays must be non-null");
  const bool any = flags & MH_ANY_HIT;
  if (any ? !hits->occluded : !hits->prim)
    return fail(MH_E_INVALID, any ? "any-hit needs hits.occluded" : "closest-hit needs hits.prim");
  const int psize = opts && opts->packet_size ? opts->packet_size : 1;
  if (psize < 1 || psize > 64) return fail(MH_E_INVALID, "packet_size %d not in 1..64", psize);
  int rc;
  if ((rc = ensure_init())) return rc;

  mh::LaunchCfg cfg{};
  cfg.any_hit = any;
  cfg.packet_size = psize;
  cfg.counters = opts ? opts->counters : nullptr;
  if (psize > 1) {
    if (s->depth + 2 > 128)
      return fail(MH_E_UNSUPPORTED, "tree depth %u exceeds the packet stack (126)", s->depth);
  } else {
    const int bpc = (opts && opts->blocks_per_cu > 0) ? opts->blocks_per_cu : kTraceBlocksPerCu;
    const int64_t cus = g_lib.cu_count;
    const int64_t chunk =
        std::min<int64_t>(64, std::max<int64_t>(kMinWaveRays, (n + 4 * cus - 1) / (4 * cus)));
    const int64_t waves = (n + chunk - 1) / chunk;
    const int own = opts ? opts->stack_lds : 0;  // the caller's ring
    const int S = own == 8 || own == 16 || own == 32 ? own
                  : waves <= kFewWaves * cus         ? kFewWavesRing
                                                     : kWideRing;
    // Entries of a spill column: the wide nodes' stack, or the records' one entry a level.
    const int64_t wide_need = std::max<int64_t>(0, (int64_t)s->stack_bound(MH_LAYOUT_PAIR) - S);
    const int64_t pairs_need = std::max<int64_t>(0, (int64_t)s->stack_bound(MH_LAYOUT_REF) - S);
    cfg.pairs = cfg.counters != nullptr;  // (the tests counted are those of the records' boxes)
    int64_t need = cfg.pairs ? pairs_need : wide_need;
    int64_t blocks = std::min(waves, 4 * cus * bpc);
    auto fit = [&] { return (int64_t)(fixed_bytes / (size_t)(need * 64 * 8)); };
    if (fixed_spill) {
      // Refused where columns of an entry a level beyond the ring (8 entries unless the caller
      // says) do not fit for every 256 rays, up to 256 lanes per compute unit.
      const int64_t deep = std::max<int64_t>(0, (int64_t)s->depth - (own == S ? S : 8));
      const int64_t per_block = deep * 256 * 8, least = std::min<int64_t>((n + 255) / 256, cus);
      if (per_block * least > (int64_t)fixed_bytes)
        return fail(MH_E_UNSUPPORTED,
                    "tree depth %u needs %lld bytes of stack spill for %lld workgroups; the "
                    "fixed area holds %zu (use mh_trace, or a larger stack_lds)",
                    s->depth, (long long)(per_block * least), (long long)least, fixed_bytes);
      // Where four waves per compute unit do not fit with the wide nodes, the records do.
      if (need > 0 && fit() < std::min(waves, 4 * cus)) {
        cfg.pairs = 1;
        need = pairs_need;
      }
      if (need > 0) blocks = std::min(blocks, fit());
    } else if (need > 0) {
      blocks = std::min(blocks, std::max<int64_t>(mh_internal::resident_waves(),
                                                  kSpillBytes / (need * 64 * 8)));
    }
    cfg.stack_lds = S;
    cfg.chunk = (int)chunk;
    cfg.blocks = (int)blocks;
    cfg.spill_stride = blocks * 64;
    if (need > 0 && fixed_spill) {
      cfg.spill = reinterpret_cast<int32_t*>(fixed_spill);
    } else if (need > 0) {
      std::lock_guard<std::mutex> lk(s->spill_mu);
      DevBuf*& b = s->spill[stream];
      if (!b) b = new (std::nothrow) DevBuf();
      if (!b) return fail(MH_E_NOMEM, "spill descriptor");
      rc = b->reserve((size_t)need * cfg.spill_stride * 8);
      if (rc == MH_E_NOMEM && cfg.blocks > mh_internal::resident_waves()) {
        cfg.blocks = mh_internal::resident_waves();
        cfg.spill_stride = (int64_t)cfg.blocks * 64;
        rc = b->reserve((size_t)need * cfg.spill_stride * 8);
      }
      if (rc) return rc;
      cfg.spill = b->as<int32_t>();
    }
  }
  mh::DevRays dr{rays->ox, rays->oy, rays->oz, rays->dx, rays->dy, rays->dz, rays->tmax,
                 rays->masked};
  mh::DevHits dh{hits->prim, hits->t, hits->u, hits->v, hits->occluded};
  HIP_OK((hipError_t)mh::launch_trace(dev_scene(s), dr, dh, n, cfg, stream));
  return MH_OK;
}

}  // namespace

int mh_internal::ensure_soa(mh_scene* s, void* stream) {
  const size_t n = std::max<size_t>(1, s->n_records / 2);  // (a single record has no pair)
  int rc;
  if ((rc = s->pairs.reserve(n * sizeof(mh::PairNode)))) return rc;
  if (s->pairs_soa.bytes != n * sizeof(mh::PairNode)) {
    s->pairs_soa.release();
    if ((rc = s->pairs_soa.reserve(n * sizeof(mh::PairNode)))) return rc;
    s->soa_gen = ~0ull;
  }
  if (s->soa_gen == s->tree_gen) return MH_OK;
  const mh::DevUpdate u = tree_view(s);
  for (const mh::LevelList& l : s->lev)
    HIP_OK((hipError_t)mh::launch_list_pairs(u, s->levels.as<int32_t>() + l.first, l.n, stream));
  // field k (16 bytes at offset 16k of every 64-byte pair) into array k
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  for (size_t k = 0; k < 4; ++k)
    HIP_OK(hipMemcpy2DAsync(s->pairs_soa.as<char>() + k * n * 16, 16, s->pairs.as<char>() + 16 * k,
                            sizeof(mh::PairNode), 16, n, hipMemcpyDeviceToDevice, st));
  s->soa_gen = s->tree_gen;
  return MH_OK;
}

int mh_internal::trace_fixed_spill(const mh_scene* s, const mh_rays* rays, const mh_hits* hits,
                                   int64_t n, uint32_t flags, const mh_trace_opts* opts,
                                   void* stream, void* spill, size_t spill_bytes) {
  if (!spill) return fail(MH_E_STATE, "no spill area");
  return trace_impl(s, rays, hits, n, flags, opts, stream, spill, spill_bytes);
}

extern "C" {

int mh_abi_version(void) { return MH_ABI_VERSION; }

const char* mh_last_error(void) { return g_err.c_str(); }

int mh_init(int device) {
  {
    std::lock_guard<std::mutex> lk(g_lib.mu);
    if (g_lib.ready && g_lib.device != device)
      return fail(MH_E_STATE, "already initialised on device %d", g_lib.device);
    g_lib.device = device;
  }
  return ensure_init();
}

int mh_device_info(char* name, int name_len, int* cu_count, size_t* hbm_bytes) {
  int rc = ensure_init();
  if (rc) return rc;
  if (name && name_len > 0) std::snprintf(name, (size_t)name_len, "%s", g_lib.name);
  if (cu_count) *cu_count = g_lib.cu_count;
  if (hbm_bytes) *hbm_bytes = g_lib.hbm;
  return MH_OK;
}

int mh_scene_create(const float* verts, uint32_t n_verts, const uint32_t* idx, uint32_t n_tris,
                    mh_scene** out) {
  if (!out) return fail(MH_E_INVALID, "null output pointer");
  *out = nullptr;
  if (!verts || !idx || n_verts == 0 || n_tris == 0)
    return fail(MH_E_INVALID, "empty mesh (%u vertices, %u triangles)", n_verts, n_tris);
  if (n_tris >= mh::kMaxObjects)
    return fail(MH_E_UNSUPPORTED, "%u triangles exceeds the limit %u", n_tris, mh::kMaxObjects);
  for (size_t i = 0; i < 3 * (size_t)n_tris; ++i)
    if (idx[i] >= n_verts) return fail(MH_E_INVALID, "index %zu = %u out of range", i, idx[i]);
  int rc = ensure_init();
  if (rc) return rc;
  mh_scene* s = new (std::nothrow) mh_scene();
  if (!s) return fail(MH_E_NOMEM, "scene");
  try {
    s->verts.assign(verts, verts + 3 * (size_t)n_verts);
    s->idx.assign(idx, idx + 3 * (size_t)n_tris);
  } catch (...) {
    delete s;
    return fail(MH_E_NOMEM, "host copy of the mesh");
  }
  s->nv = n_verts;
  s->nt = n_tris;
  const size_t vb = 3 * (size_t)n_verts * 4, ib = 3 * (size_t)n_tris * 4;
  if ((rc = s->d_verts.reserve(vb)) || (rc = s->d_base.reserve(vb)) ||
      (rc = s->d_idx.reserve(ib))) {
    delete s;
    return rc;
  }
  hipError_t e = hipMemcpy(s->d_verts.p, verts, vb, hipMemcpyHostToDevice);
  if (e == hipSuccess) e = hipMemcpy(s->d_base.p, verts, vb, hipMemcpyHostToDevice);
  if (e == hipSuccess) e = hipMemcpy(s->d_idx.p, idx, ib, hipMemcpyHostToDevice);
  if (e != hipSuccess) {
    delete s;
    return fail(MH_E_HIP, "mesh upload: %s", hipGetErrorString(e));
  }
  *out = s;
  return MH_OK;
}

int mh_scene_destroy(mh_scene* scene) {
  if (!scene) return MH_OK;
  (void)ensure_init();
  (void)hipDeviceSynchronize();
  delete scene;
  return MH_OK;
}

// DynBVH::rebuild with USE_APPROXIMATE_BUILD, on the device (build.hip): object boxes,
// the level loop over nodes of many objects, one wave per small node, then the reference
// numbering and the bottom-up passes.
int build_device(mh_scene* s, int rtsah) {
  using mh_internal::DevBuf;
  const uint32_t T = s->nt;
  const size_t nrec = 2 * (size_t)T;
  const int64_t cap = (int64_t)T / (mh::kBuildSerial + 1) + 2;
  const int64_t vcap = (int64_t)T / mh::kBuildVB + cap + 2;
  int rc;
  if ((rc = reserve_tree(s, nrec, 0, 0)) || (rc = s->parent.reserve(nrec * 4)) ||
      (rc = s->anc0.reserve(nrec * 4)) || (rc = s->dep0.reserve(nrec * 4)) ||
      (rc = s->anc1.reserve(nrec * 4)) || (rc = s->dep1.reserve(nrec * 4)) ||
      (rc = s->hist.reserve(mh::kDepthHist * 4)))
    return rc;
  if (!s->logtab.p) {
    std::vector<float> tab(mh::rtsah::kLogTable);
    mh::rtsah::fill_log_table(tab.data());
    if ((rc = s->logtab.reserve(tab.size() * 4))) return rc;
    HIP_OK(hipMemcpy(s->logtab.p, tab.data(), tab.size() * 4, hipMemcpyHostToDevice));
  }
  // Work arrays of this build only, in one allocation.
  size_t held = 0;
  auto place = [&](size_t bytes) {
    const size_t at = held;
    held += (bytes + 255) & ~(size_t)255;
    return at;
  };
  const size_t o_slots = place((size_t)T * 48), o_trefs = place(nrec * 32),
               o_seg0 = place(cap * sizeof(mh::BuildSeg)),
               o_seg1 = place(cap * sizeof(mh::BuildSeg)),
               o_small = place((size_t)T * sizeof(mh::BuildSeg)),
               o_big = place(cap * sizeof(mh::BuildSeg)),
               o_plan0 = place(cap * sizeof(mh::BuildPlan)),
               o_plan1 = place(cap * sizeof(mh::BuildPlan)),
               o_acc = place((size_t)cap * mh::kAccWords * 4), o_ctr = place(mh::kCtrCount * 4),
               o_vbseg = place(vcap * 4), o_vcnt = place(vcap * 8),
               o_gscan = place(2 * (vcap + 1) * 4), o_scratch = place(nrec * 4),
               o_root = place(48 + 24), o_ic = place(nrec * 4), o_rank = place(nrec * 4),
               o_fin = place(nrec * 4), o_rt = place(nrec * 8);
  DevBuf work;
  if ((rc = work.reserve(held))) return rc;
  auto at = [&](size_t offset) { return static_cast<void*>(work.as<char>() + offset); };
  hipStream_t st = nullptr;
  HIP_OK(hipMemsetAsync(at(o_ctr), 0, mh::kCtrCount * 4, st));
  HIP_OK(hipMemsetAsync(at(o_root), 0xFF, 48 + 24, st));

  mh::DevBuild d{};
  unsigned* ctr = static_cast<unsigned*>(at(o_ctr));
  d.u.refs = static_cast<mh::RefNode*>(at(o_trefs));
  d.u.ids = s->ids.as<int32_t>();
  d.u.verts = s->d_verts.as<float>();
  d.u.idx = s->d_idx.as<uint32_t>();
  d.u.next_free = ctr + mh::kCtrRecords;
  d.u.err = reinterpret_cast<int*>(ctr + mh::kCtrErr);
  d.u.n_records = (int32_t)nrec;
  d.u.n_objects = (int32_t)T;
  d.slots = static_cast<float*>(at(o_slots));
  d.verts = s->d_verts.as<float>();
  d.n_verts = s->nv;
  d.small = static_cast<mh::BuildSeg*>(at(o_small));
  d.big = static_cast<mh::BuildSeg*>(at(o_big));
  d.acc = static_cast<unsigned*>(at(o_acc));
  d.ctr = ctr;
  d.vbseg = static_cast<int32_t*>(at(o_vbseg));
  d.vcnt = static_cast<unsigned*>(at(o_vcnt));
  d.gscan = static_cast<unsigned*>(at(o_gscan));
  d.vcap = vcap;
  d.lpos = static_cast<int32_t*>(at(o_scratch));
  d.rpos = d.lpos + T;
  d.rootk = static_cast<unsigned long long*>(at(o_root));
  d.rootc = reinterpret_cast<unsigned*>(d.rootk + 6);
  const bool serial_root = T <= (uint32_t)mh::kBuildSerial;
  d.seg = static_cast<mh::BuildSeg*>(at(o_seg0));
  d.plan = static_cast<mh::BuildPlan*>(at(o_plan0));
  HIP_OK((hipError_t)mh::build_launch_setup(d, serial_root ? 1 : 0, st));
  d.seg_next = static_cast<mh::BuildSeg*>(at(o_seg1));
  d.plan_next = static_cast<mh::BuildPlan*>(at(o_plan1));
  // Level k holds at most 2^k nodes, which is a tight bound until nodes of few objects
  // appear: those levels are launched one after the other, and only from then on does the
  // host read the number of nodes back before it launches a level.
  unsigned back[mh::kCtrCount] = {};
  int64_t bound = serial_root ? 0 : 1;
  bool counted = false;
  for (int level = 0; bound > 0; ++level) {
    if (level == mh::kMaxDepth)
      return fail(MH_E_UNSUPPORTED, "tree deeper than %d levels", mh::kMaxDepth - 1);
    d.level = level;
    HIP_OK((hipError_t)mh::build_launch_level(d, bound, (int64_t)T / mh::kBuildVB + bound + 1, st));
    std::swap(d.seg, d.seg_next);
    std::swap(d.plan, d.plan_next);
    bound = std::min(2 * bound, cap);
    if (!counted && bound < cap) continue;
    counted = true;
    HIP_OK(hipMemcpyAsync(back, ctr, sizeof(back), hipMemcpyDeviceToHost, st));
    HIP_OK(hipStreamSynchronize(st));
    if (back[mh::kCtrErr]) break;
    bound = back[mh::kCtrSegs + level + 1];
  }
  HIP_OK(hipMemcpyAsync(back, ctr, sizeof(back), hipMemcpyDeviceToHost, st));
  HIP_OK(hipStreamSynchronize(st));
  const unsigned err = back[mh::kCtrErr];
  if (err == 2) return fail(MH_E_INVALID, "non-finite vertex coordinate");
  if (err == 3) return fail(MH_E_UNSUPPORTED, "a leaf of more than 32767 objects");
  if (err) return fail(MH_E_STATE, "device build ran out of node records");
  HIP_OK((hipError_t)mh::build_launch_serial(d, back[mh::kCtrSmall], back[mh::kCtrBig],
                                             static_cast<int32_t*>(at(o_scratch)), st));
  // Depths of the temporary tree, then its per-depth lists.
  HIP_OK(hipMemsetAsync(s->hist.p, 0, mh::kDepthHist * 4, st));
  HIP_OK((hipError_t)mh::launch_depths(d.u, s->anc0.as<int32_t>(), s->dep0.as<int32_t>(),
                                       s->anc1.as<int32_t>(), s->dep1.as<int32_t>(),
                                       s->hist.as<unsigned>(), st));
  std::vector<unsigned> hist(mh::kDepthHist);
  unsigned used[2];
  HIP_OK(hipMemcpyAsync(hist.data(), s->hist.p, hist.size() * 4, hipMemcpyDeviceToHost, st));
  HIP_OK(hipMemcpyAsync(used, ctr, 8, hipMemcpyDeviceToHost, st));
  HIP_OK(hipStreamSynchronize(st));
  if (used[1]) return fail(MH_E_STATE, "device build ran out of node records");
  const unsigned deepest = hist[mh::kMaxDepth + 1];
  if (deepest >= (unsigned)mh::kMaxDepth - 1)
    return fail(MH_E_UNSUPPORTED, "tree deeper than %d levels", mh::kMaxDepth - 1);
  std::vector<unsigned> cursor(mh::kMaxDepth + 1, 0u);
  std::vector<int64_t> level_off(1, 0);
  for (unsigned dd = 0; dd < deepest; ++dd) {
    cursor[dd] = (unsigned)level_off.back();
    level_off.push_back(level_off.back() + hist[dd]);
  }
  const int64_t n_leaves = hist[mh::kMaxDepth];
  HIP_OK(hipMemcpyAsync(s->hist.p, cursor.data(), cursor.size() * 4, hipMemcpyHostToDevice, st));
  HIP_OK((hipError_t)mh::launch_depth_scatter(d.u, s->dep0.as<int32_t>(), s->hist.as<unsigned>(),
                                              s->levels.as<int32_t>(), s->leaves.as<int32_t>(),
                                              st));
  HIP_OK(hipMemsetAsync(at(o_fin), 0xFF, nrec * 4, st));
  mh::DevFinish f{};
  f.trefs = d.u.refs;
  f.refs = s->refs.as<mh::RefNode>();
  f.tcount = ctr;
  f.ic = static_cast<int32_t*>(at(o_ic));
  f.rank = static_cast<int32_t*>(at(o_rank));
  f.fin = static_cast<int32_t*>(at(o_fin));
  // written after the numbering, when these three are free
  f.prob[0] = static_cast<float*>(at(o_ic));
  f.prob[1] = static_cast<float*>(at(o_rank));
  f.prob[2] = static_cast<float*>(at(o_scratch));
  f.levels = s->levels.as<int32_t>();
  f.leaves = s->leaves.as<int32_t>();
  f.costs = s->costs.as<float>();
  f.ssize = s->ssize.as<uint32_t>();
  f.rt = static_cast<float*>(at(o_rt));
  f.logtab = s->logtab.as<float>();
  const uint32_t n_final = (uint32_t)(level_off.back() + n_leaves);
  f.n_records = (int32_t)nrec;
  f.n_final = (int32_t)n_final;
  f.large = (uint32_t)(nrec / (20 * (size_t)s->workers));
  f.rtsah = rtsah;
  const int n_levels = (int)level_off.size() - 1;
  ++s->tree_gen;
  HIP_OK((hipError_t)mh::build_launch_ranks(f, level_off.data(), n_levels, n_leaves, st));
  HIP_OK(hipMemcpyAsync(s->counters.p, &n_final, 4, hipMemcpyHostToDevice, st));
  mh::DevRefit r{};
  r.tris = s->tris.as<float>();
  r.obj_ids = s->ids.as<int32_t>();
  r.verts = s->d_verts.as<float>();
  r.idx = s->d_idx.as<uint32_t>();
  r.n_slots = (int32_t)T;
  r.prim_kind = s->prim_kind;
  HIP_OK((hipError_t)mh::launch_prim_setup(r, st));
  HIP_OK(hipMemsetAsync(s->leaf_at.p, 0xFF, (size_t)T * 4, st));
  HIP_OK(hipMemsetAsync(s->irregular.p, 0, 8, st));
  s->fixed_irregular = 0;
  if (n_final > 1) {
    std::vector<mh::LevelList> sizes;
    for (int k = 0; k < n_levels; ++k)
      sizes.push_back(mh::LevelList{0, level_off[k + 1] - level_off[k]});
    if ((rc = wide_pass(s, sizes, mh::kMaxDepth - 2, 0, nullptr, nullptr, st))) return rc;
    s->root_ref = 0;
  } else {
    if ((rc = leaf_root(s, 0, st))) return rc;
    const int32_t zero = 0, n = (int32_t)T;
    HIP_OK(hipMemcpy(s->leaf_at.p, &zero, 4, hipMemcpyHostToDevice));
    HIP_OK(hipMemcpy(s->big.p, &n, 4, hipMemcpyHostToDevice));
    s->root_ref = ~(int)std::min<uint32_t>(T, mh::kLeafCountInline);
  }
  s->next_free = n_final;
  s->n_records = (uint32_t)nrec;
  s->bvh = mh::DynBvh();
  s->partition = s->updatable = true;
  s->built = true;
  return MH_OK;
}

int mh_scene_build(mh_scene* s, const mh_build_opts* opts) {
  if (!s) return fail(MH_E_INVALID, "null scene");
  const int kind = opts ? opts->prim_kind : MH_PRIM_KENSLER_SHIRLEY;
  if (kind != MH_PRIM_KENSLER_SHIRLEY && kind != MH_PRIM_WALD)
    return fail(MH_E_INVALID, "unknown prim_kind %d", kind);
  const int rtsah = opts ? opts->rtsah : 1;
  const int threads = opts ? opts->threads : 0;
  int rc = ensure_init();
  if (rc) return rc;
  if (opts && opts->approximate) {
    s->built = s->updatable = false;
    s->prim_kind = kind;
    return build_device(s, rtsah);
  }
  try {
    s->bvh = mh::build_dynbvh(s->verts.data(), s->nv, s->idx.data(), s->nt, threads);
    if (s->workers != 1) mh::mark_large_subtrees(s->bvh.nodes, s->workers);
    if (rtsah) mh::compute_rtsah(s->bvh.nodes, threads);
  } catch (const std::bad_alloc&) {
    return fail(MH_E_NOMEM, "host memory for the SAH build");
  } catch (const std::exception& ex) {
    return fail(MH_E_INVALID, "build: %s", ex.what());
  }
  s->prim_kind = kind;
  return upload(s);
}

int mh_scene_set_workers(mh_scene* s, int workers) {
  if (!s) return fail(MH_E_INVALID, "null scene");
  if (workers < 1 || workers > 4096) return fail(MH_E_INVALID, "workers %d not in 1..4096", workers);
  s->workers = workers;
  if (!s->built) return MH_OK;  // applies to the next build
  int rc = ensure_init();
  if (rc) return rc;
  // computeSubTreeSizes over the current tree with the new threshold (DynBVH.cc:941-950,
  // 1971-1996): reachable records only, sizes counted in records.
  const uint32_t nn = s->n_records;
  std::vector<mh::RefNode> nodes(nn);
  HIP_OK(hipMemcpy(nodes.data(), s->refs.p, (size_t)nn * sizeof(mh::RefNode),
                   hipMemcpyDeviceToHost));
  const uint32_t limit = s->large_limit();
  std::vector<uint32_t> size(nn, 0);
  std::vector<std::pair<int32_t, bool>> st{{0, false}};
  while (!st.empty()) {
    auto [id, done] = st.back();
    st.pop_back();
    if (id < 0 || (uint32_t)id >= nn) return fail(MH_E_STATE, "record %d outside the tree", id);
    mh::RefNode& n = nodes[id];
    if (n.leaf()) {
      size[id] = 1;
      n.bits &= (uint8_t)~2;
      continue;
    }
    if (!done) {
      if ((uint32_t)n.child + 1 >= nn) return fail(MH_E_STATE, "record %d: child outside", id);
      st.push_back({id, true});
      st.push_back({n.child + 1, false});
      st.push_back({n.child, false});
      continue;
    }
    size[id] = size[n.child] + size[n.child + 1] + 1;
    if (size[id] > limit)
      n.bits |= 2;
    else
      n.bits &= (uint8_t)~2;
  }
  HIP_OK(hipMemcpy(s->refs.p, nodes.data(), (size_t)nn * sizeof(mh::RefNode),
                   hipMemcpyHostToDevice));
  if (s->bvh.nodes.size() == nodes.size()) s->bvh.nodes = nodes;
  return MH_OK;
}

int mh_dynbvh_build_host(const float* verts, uint32_t n_verts, const uint32_t* idx,
                         uint32_t n_tris, const mh_build_opts* opts, int32_t* ids, void* nodes,
                         uint32_t* num_nodes) {
  if (!verts || !idx || !ids || !nodes) return fail(MH_E_INVALID, "null argument");
  if (n_verts == 0 || n_tris == 0) return fail(MH_E_INVALID, "empty mesh");
  if (n_tris >= mh::kMaxObjects)
    return fail(MH_E_UNSUPPORTED, "%u triangles exceeds the limit %u", n_tris, mh::kMaxObjects);
  for (size_t i = 0; i < 3 * (size_t)n_tris; ++i)
    if (idx[i] >= n_verts) return fail(MH_E_INVALID, "index %zu = %u out of range", i, idx[i]);
  const int rtsah = opts ? opts->rtsah : 1;
  const int threads = opts ? opts->threads : 0;
  try {
    mh::DynBvh b = mh::build_dynbvh(verts, n_verts, idx, n_tris, threads);
    if (rtsah) mh::compute_rtsah(b.nodes, threads);
    std::memcpy(ids, b.ids.data(), b.ids.size() * 4);
    std::memcpy(nodes, b.nodes.data(), b.nodes.size() * sizeof(mh::RefNode));
    if (num_nodes) *num_nodes = (uint32_t)b.num_nodes;
  } catch (const std::bad_alloc&) {
    return fail(MH_E_NOMEM, "host memory for the SAH build");
  } catch (const std::exception& ex) {
    return fail(MH_E_INVALID, "build: %s", ex.what());
  }
  return MH_OK;
}

namespace {

int load_tree(mh_scene* s, const int32_t* ids, uint32_t n_ids, const void* nodes,
              uint32_t n_nodes, int prim_kind, bool rtsah) {
  if (!s || !ids || !nodes) return fail(MH_E_INVALID, "null argument");
  if (prim_kind != MH_PRIM_KENSLER_SHIRLEY && prim_kind != MH_PRIM_WALD)
    return fail(MH_E_INVALID, "unknown prim_kind %d", prim_kind);
  if (n_nodes == 0) return fail(MH_E_INVALID, "empty node array");
  int rc = ensure_init();
  if (rc) return rc;
  std::vector<int32_t> idv(ids, ids + n_ids);
  if ((rc = validate_ids(idv, s->nt))) return rc;
  s->bvh.ids = std::move(idv);
  const mh::RefNode* nn = static_cast<const mh::RefNode*>(nodes);
  s->bvh.nodes.assign(nn, nn + n_nodes);
  s->bvh.num_nodes = 0;
  s->prim_kind = prim_kind;
  s->built = false;
  return upload(s, rtsah);
}

}  // namespace

int mh_scene_load_dynbvh(mh_scene* s, const int32_t* ids, uint32_t n_ids, const void* nodes,
                         uint32_t n_nodes, int prim_kind) {
  return load_tree(s, ids, n_ids, nodes, n_nodes, prim_kind, false);
}

int mh_scene_load_dynbvh_file(mh_scene* s, const char* path, int prim_kind) {
  if (!s || !path) return fail(MH_E_INVALID, "null argument");
  std::ifstream in(path, std::ios::binary);
  if (!in) return fail(MH_E_IO, "cannot open %s", path);
  uint32_t n_ids = 0, n_nodes = 0;
  in.read(reinterpret_cast<char*>(&n_ids), 4);
  if (!in || n_ids != s->nt) return fail(MH_E_IO, "%s: bad object_ids count", path);
  std::vector<int32_t> ids(n_ids);
  in.read(reinterpret_cast<char*>(ids.data()), (std::streamsize)n_ids * 4);
  in.read(reinterpret_cast<char*>(&n_nodes), 4);
  if (!in || n_nodes == 0 || n_nodes > 4u * n_ids + 4u) return fail(MH_E_IO, "%s: bad node count", path);
  std::vector<mh::RefNode> nodes(n_nodes);
  in.read(reinterpret_cast<char*>(nodes.data()), (std::streamsize)n_nodes * 32);
  if (!in) return fail(MH_E_IO, "%s: truncated", path);
  return load_tree(s, ids.data(), n_ids, nodes.data(), n_nodes, prim_kind, true);
}

int mh_scene_export_dynbvh(const mh_scene* s, int32_t* ids, uint32_t* n_ids, void* nodes,
                           uint32_t* n_nodes) {
  if (!s || !n_ids || !n_nodes) return fail(MH_E_INVALID, "null argument");
  if (!s->built) return fail(MH_E_STATE, "scene has no tree");
  const uint32_t ni = s->nt, nn = s->n_records;
  if (!ids && !nodes) {
    *n_ids = ni;
    *n_nodes = nn;
    return MH_OK;
  }
  if (*n_ids < ni || *n_nodes < nn) return fail(MH_E_INVALID, "export arrays too small");
  int rc = ensure_init();
  if (rc) return rc;
  if (ids) HIP_OK(hipMemcpy(ids, s->ids.p, (size_t)ni * 4, hipMemcpyDeviceToHost));
  if (nodes) HIP_OK(hipMemcpy(nodes, s->refs.p, (size_t)nn * 32, hipMemcpyDeviceToHost));
  *n_ids = ni;
  *n_nodes = nn;
  return MH_OK;
}

int mh_scene_save_dynbvh_file(const mh_scene* s, const char* path) {
  if (!s || !path) return fail(MH_E_INVALID, "null argument");
  uint32_t ni = 0, nn = 0;
  int rc = mh_scene_export_dynbvh(s, nullptr, &ni, nullptr, &nn);
  if (rc) return rc;
  std::vector<int32_t> ids(ni);
  std::vector<mh::RefNode> nodes(nn);
  if ((rc = mh_scene_export_dynbvh(s, ids.data(), &ni, nodes.data(), &nn))) return rc;
  std::ofstream out(path, std::ios::binary);
  if (!out) return fail(MH_E_IO, "cannot create %s", path);
  out.write(reinterpret_cast<const char*>(&ni), 4);
  out.write(reinterpret_cast<const char*>(ids.data()), (std::streamsize)ni * 4);
  out.write(reinterpret_cast<const char*>(&nn), 4);
  out.write(reinterpret_cast<const char*>(nodes.data()), (std::streamsize)nn * 32);
  if (!out) return fail(MH_E_IO, "write to %s failed", path);
  return MH_OK;
}

int mh_scene_bounds(const mh_scene* s, float lo[3], float hi[3]) {
  if (!s || !lo || !hi) return fail(MH_E_INVALID, "null argument");
  if (!s->built) return fail(MH_E_STATE, "scene has no tree");
  int rc = ensure_init();
  if (rc) return rc;
  mh::RefNode root;
  HIP_OK(hipMemcpy(&root, s->refs.p, sizeof(root), hipMemcpyDeviceToHost));
  for (int k = 0; k < 3; ++k) {
    lo[k] = root.box.lo[k];
    hi[k] = root.box.hi[k];
  }
  return MH_OK;
}

int mh_scene_stats(const mh_scene* s, uint32_t* n_nodes, uint32_t* n_inner, uint32_t* depth,
                   size_t* device_bytes) {
  if (!s) return fail(MH_E_INVALID, "null scene");
  if (!s->built) return fail(MH_E_STATE, "scene has no tree");
  if (n_nodes) *n_nodes = s->n_inner + s->n_leaves;
  if (n_inner) *n_inner = s->n_inner;
  if (depth) *depth = s->depth;
  if (device_bytes) *device_bytes = s->device_bytes();
  return MH_OK;
}

int mh_scene_set_vertices(mh_scene* s, const float* verts, int on_device, void* stream) {
  if (!s || !verts) return fail(MH_E_INVALID, "null argument");
  int rc = ensure_init();
  if (rc) return rc;
  const size_t vb = 3 * (size_t)s->nv * 4;
  HIP_OK(hipMemcpyAsync(s->d_verts.p, verts, vb,
                        on_device ? hipMemcpyDeviceToDevice : hipMemcpyHostToDevice,
                        reinterpret_cast<hipStream_t>(stream)));
  if (!on_device) std::memcpy(s->verts.data(), verts, vb);
  return MH_OK;
}

int mh_scene_vertices_device(mh_scene* s, float** verts) {
  if (!s || !verts) return fail(MH_E_INVALID, "null argument");
  *verts = s->d_verts.as<float>();
  return MH_OK;
}

int mh_scene_displace_sine(mh_scene* s, float amp, float freq, float phase, void* stream) {
  if (!s) return fail(MH_E_INVALID, "null scene");
  int rc = ensure_init();
  if (rc) return rc;
  HIP_OK((hipError_t)mh::launch_displace_sine(s->d_verts.as<float>(), s->d_base.as<float>(),
                                              s->nv, amp, freq, phase, stream));
  return MH_OK;
}

int mh_scene_refit(mh_scene* s, void* stream) {
  if (!s) return fail(MH_E_INVALID, "null scene");
  if (!s->built) return fail(MH_E_STATE, "scene has no tree");
  int rc = ensure_init();
  if (rc) return rc;
  mh::DevRefit r{};
  r.refs = s->refs.as<mh::RefNode>();
  r.wide = s->wide.as<mh::WideNode>();
  r.leaf_at = s->partition ? s->leaf_at.as<int32_t>() : nullptr;
  r.irregular = s->irregular.as<int32_t>();
  r.fixed = s->fixed_irregular;
  r.tris = s->tris.as<float>();
  r.obj_ids = s->ids.as<int32_t>();
  r.verts = s->d_verts.as<float>();
  r.idx = s->d_idx.as<uint32_t>();
  r.leaves = s->leaves.as<int32_t>();
  r.levels = s->levels.as<int32_t>();
  r.n_leaves = (int32_t)s->n_leaves;
  r.n_slots = (int32_t)s->nt;
  r.prim_kind = s->prim_kind;
  ++s->tree_gen;
  HIP_OK((hipError_t)mh::launch_refit(r, s->lev.data(), (int)s->lev.size(), stream));
  return MH_OK;
}

int mh_scene_update(mh_scene* s, void* stream) {
  if (!s) return fail(MH_E_INVALID, "null scene");
  if (!s->built) return fail(MH_E_STATE, "scene has no tree");
  if (!s->updatable)
    return fail(MH_E_UNSUPPORTED, "the tree has records outside it or leaves that do not "
                "partition the objects; use mh_scene_refit");
  int rc = ensure_init();
  if (rc) return rc;
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  const uint32_t T = s->nt;
  const size_t nrec = s->refs.bytes / sizeof(mh::RefNode);
  // Work arrays, allocated at the first update.
  if ((rc = s->parent.reserve(nrec * 4)) ||
      (rc = s->split_list.reserve((size_t)std::max<uint32_t>(1u, T) * 4)))
    return rc;
  unsigned* nfree = s->counters.as<unsigned>();
  const unsigned init[3] = {s->next_free, 0u, 0u};  // next_free, err, split list entries
  HIP_OK(hipMemcpyAsync(nfree, init, sizeof(init), hipMemcpyHostToDevice, st));
  mh::DevUpdate u = tree_view(s);  // (object boxes are formed from the vertices)
  u.next_free = nfree;
  u.err = reinterpret_cast<int*>(nfree + 1);
  u.split_list = s->split_list.as<int32_t>();
  u.split_count = nfree + 2;
  u.n_records = (int32_t)nrec;
  u.n_old = (int32_t)s->next_free;
  // largeSubtreeSize = nodes.size() / (20 * numProcs) (DynBVH.cc:1776)
  u.large = (uint32_t)(nrec / (20 * (size_t)s->workers));
  ++s->tree_gen;
  // leaf pass (triangle records and leaf boxes from the current vertices), leaf splits,
  // rotations depth by depth
  HIP_OK((hipError_t)mh::launch_update_tree(u, s->n_leaves, s->levels.as<int32_t>(),
                                            s->lev.data(), (int)s->lev.size(), st));
  mh::DevRefit r{};  // triangle records in slot order from the current vertices
  r.tris = s->tris.as<float>();
  r.obj_ids = s->ids.as<int32_t>();
  r.verts = s->d_verts.as<float>();
  r.idx = s->d_idx.as<uint32_t>();
  r.n_slots = (int32_t)T;
  r.prim_kind = s->prim_kind;
  HIP_OK((hipError_t)mh::launch_prim_setup(r, st));
  // Lists and wide nodes of the new topology.
  unsigned now[2] = {0, 0};  // records in use, error
  rc = MH_OK;
  if (s->n_inner > 0) {  // rotations never turn a leaf root inner
    const std::vector<mh::LevelList> sizes = s->lev;
    s->fixed_irregular = 0;
    rc = wide_pass(s, sizes, mh::kMaxDepth - 2, 0, nfree, now, st);
  } else {
    int32_t mark[2];  // the leaf pass's NaN mark, which wide_pass takes over otherwise
    HIP_OK(hipMemcpyAsync(s->host_ctr, nfree, 8, hipMemcpyDeviceToHost, st));
    HIP_OK(hipMemcpyAsync(mark, s->irregular.p, 8, hipMemcpyDeviceToHost, st));
    HIP_OK(hipStreamSynchronize(st));
    now[0] = s->host_ctr[0];
    now[1] = s->host_ctr[1];
    mark[0] = mark[1];
    mark[1] = 0;
    HIP_OK(hipMemcpyAsync(s->irregular.p, mark, 8, hipMemcpyHostToDevice, st));
    HIP_OK(hipStreamSynchronize(st));
  }
  // Either failure leaves a device tree that must not be traced: the scene needs a build.
  if (now[1]) {
    s->built = s->updatable = false;
    return fail(MH_E_STATE, "leaf splits ran out of node records; build the scene again");
  }
  if (rc) {
    s->built = s->updatable = false;
    return rc;
  }
  s->next_free = now[0];
  return MH_OK;
}

int mh_scene_set_attributes(mh_scene* s, const float* normals, uint32_t n_normals,
                            const uint32_t* normal_idx, const float* texcoords,
                            uint32_t n_texcoords, const uint32_t* tex_idx) {
  if (!s) return fail(MH_E_INVALID, "null scene");
  if (!normals != !normal_idx || !texcoords != !tex_idx)
    return fail(MH_E_INVALID, "an attribute needs both its values and its indices");
  const size_t n3 = 3 * (size_t)s->nt;
  if (normals) {
    for (size_t k = 0; k < n3; ++k)
      if (normal_idx[k] >= n_normals)
        return fail(MH_E_INVALID, "normal index %zu = %u out of range", k, normal_idx[k]);
  }
  if (texcoords) {
    for (size_t t = 0; t < s->nt; ++t) {
      if (tex_idx[3 * t] == MH_NO_TEXTURE_INDEX) continue;
      for (int k = 0; k < 3; ++k)
        if (tex_idx[3 * t + k] >= n_texcoords)
          return fail(MH_E_INVALID, "texture index %zu = %u out of range", 3 * t + k,
                      tex_idx[3 * t + k]);
    }
  }
  int rc = ensure_init();
  if (rc) return rc;
  s->normals.release();
  s->normal_idx.release();
  s->texcoords.release();
  s->tex_idx.release();
  if (normals) {
    if ((rc = s->normals.reserve(std::max<size_t>(1, n_normals) * 12)) ||
        (rc = s->normal_idx.reserve(n3 * 4)))
      return rc;
    HIP_OK(hipMemcpy(s->normals.p, normals, (size_t)n_normals * 12, hipMemcpyHostToDevice));
    HIP_OK(hipMemcpy(s->normal_idx.p, normal_idx, n3 * 4, hipMemcpyHostToDevice));
  }
  if (texcoords) {
    if ((rc = s->texcoords.reserve(std::max<size_t>(1, n_texcoords) * 12)) ||
        (rc = s->tex_idx.reserve(n3 * 4)))
      return rc;
    HIP_OK(hipMemcpy(s->texcoords.p, texcoords, (size_t)n_texcoords * 12,
                     hipMemcpyHostToDevice));
    HIP_OK(hipMemcpy(s->tex_idx.p, tex_idx, n3 * 4, hipMemcpyHostToDevice));
  }
  return MH_OK;
}

int mh_shade(const mh_scene* s, const mh_rays* rays, const mh_hits* hits, int64_t n,
             const mh_shading* out, void* stream) {
  if (!s || !rays || !hits || !out) return fail(MH_E_INVALID, "null argument");
  if (n < 0) return fail(MH_E_INVALID, "negative ray count");
  if (!rays->ox || !rays->oy || !rays->oz || !rays->dx || !rays->dy || !rays->dz)
    return fail(MH_E_INVALID, "ray origin and direction arrays are required");
  if (!hits->prim || !hits->t || !hits->u || !hits->v)
    return fail(MH_E_INVALID, "hits need prim, t, u and v");
  if (n == 0) return MH_OK;
  int rc = ensure_init();
  if (rc) return rc;
  mh::DevShade d{};
  d.rays.ox = rays->ox;
  d.rays.oy = rays->oy;
  d.rays.oz = rays->oz;
  d.rays.dx = rays->dx;
  d.rays.dy = rays->dy;
  d.rays.dz = rays->dz;
  d.prim = hits->prim;
  d.t = hits->t;
  d.u = hits->u;
  d.v = hits->v;
  d.verts = s->d_verts.as<float>();
  d.idx = s->d_idx.as<uint32_t>();
  d.normals = s->normals.as<float>();
  d.normal_idx = s->normal_idx.as<uint32_t>();
  d.tex = s->texcoords.as<float>();
  d.tex_idx = s->tex_idx.as<uint32_t>();
  float* o[12] = {out->px, out->py, out->pz, out->nx, out->ny, out->nz,
                  out->gx, out->gy, out->gz, out->tu, out->tv, out->tw};
  for (int k = 0; k < 12; ++k) d.out[k] = o[k];
  d.n = n;
  d.n_tris = (int32_t)s->nt;
  d.prim_kind = s->prim_kind;
  HIP_OK((hipError_t)mh::launch_shade(d, stream));
  return MH_OK;
}

int mh_trace(const mh_scene* s, const mh_rays* rays, const mh_hits* hits, int64_t n,
             uint32_t flags, const mh_trace_opts* opts, void* stream) {
  return trace_impl(s, rays, hits, n, flags, opts, stream);
}

// Ray count up to which mh_trace_host packs rays and results into pinned host memory.
constexpr int64_t kPinnedStageRays = int64_t(1) << 16;

int mh_trace_host(const mh_scene* cs, const mh_rays* rays, const mh_hits* hits, int64_t n,
                  uint32_t flags, const mh_trace_opts* opts) {
  mh_scene* s = const_cast<mh_scene*>(cs);
  if (!s || !rays || !hits) return fail(MH_E_INVALID, "null argument");
  if (n <= 0) return n == 0 ? MH_OK : fail(MH_E_INVALID, "negative ray count");
  int rc = ensure_init();
  if (rc) return rc;
  std::lock_guard<std::mutex> lk(s->stage_mu);
  // One staging layout in device memory (and, for small sets, in pinned host memory): 7
  // float arrays and the mask bytes in, 4 result arrays and the occluded bytes out, on the
  // scene's own stream.
  const size_t f = (size_t)n * 4, al = 256;
  auto up = [&](size_t x) { return (x + al - 1) / al * al; };
  const size_t in_bytes = 7 * up(f) + up((size_t)n);
  const size_t out_bytes = 4 * up(f) + up((size_t)n);
  if ((rc = s->stage.reserve(in_bytes + out_bytes))) return rc;
  // A blocking stream: work the caller queued on the null stream (a refit, an upload)
  // comes first, as it did for the null-stream copies of this entry point.
  if (!s->stage_stream) HIP_OK(hipStreamCreateWithFlags(&s->stage_stream, hipStreamDefault));
  hipStream_t st = s->stage_stream;
  char* base = s->stage.as<char>();
  if (n > kPinnedStageRays) {
    // Large sets: the runtime's own pipelined copies from pageable memory, array by array.
    const float* src[7] = {rays->ox, rays->oy, rays->oz, rays->dx, rays->dy, rays->dz, rays->tmax};
    float* d[7];
    for (int i = 0; i < 7; ++i) {
      if (!src[i]) return fail(MH_E_INVALID, "ray array %d is null", i);
      d[i] = reinterpret_cast<float*>(base + i * up(f));
      HIP_OK(hipMemcpyAsync(d[i], src[i], f, hipMemcpyHostToDevice, st));
    }
    uint8_t* dm = nullptr;
    if (rays->masked) {
      dm = reinterpret_cast<uint8_t*>(base + 7 * up(f));
      HIP_OK(hipMemcpyAsync(dm, rays->masked, (size_t)n, hipMemcpyHostToDevice, st));
    }
    char* ob = base + in_bytes;
    mh_hits dh{};
    dh.prim = hits->prim ? reinterpret_cast<int32_t*>(ob) : nullptr;
    dh.t = hits->t ? reinterpret_cast<float*>(ob + up(f)) : nullptr;
    dh.u = hits->u ? reinterpret_cast<float*>(ob + 2 * up(f)) : nullptr;
    dh.v = hits->v ? reinterpret_cast<float*>(ob + 3 * up(f)) : nullptr;
    dh.occluded = hits->occluded ? reinterpret_cast<uint8_t*>(ob + 4 * up(f)) : nullptr;
    mh_rays dr{d[0], d[1], d[2], d[3], d[4], d[5], d[6], dm};
    if ((rc = trace_impl(s, &dr, &dh, n, flags, opts, st))) return rc;
    if (hits->prim) HIP_OK(hipMemcpyAsync(hits->prim, dh.prim, f, hipMemcpyDeviceToHost, st));
    if (hits->t) HIP_OK(hipMemcpyAsync(hits->t, dh.t, f, hipMemcpyDeviceToHost, st));
    if (hits->u) HIP_OK(hipMemcpyAsync(hits->u, dh.u, f, hipMemcpyDeviceToHost, st));
    if (hits->v) HIP_OK(hipMemcpyAsync(hits->v, dh.v, f, hipMemcpyDeviceToHost, st));
    if (hits->occluded)
      HIP_OK(hipMemcpyAsync(hits->occluded, dh.occluded, (size_t)n, hipMemcpyDeviceToHost, st));
    HIP_OK(hipStreamSynchronize(st));
    return MH_OK;
  }
  // Small sets (the packets of a render thread gathered by HipDynBVH): packed into pinned
  // host memory, one copy each way.
  if (s->host_stage_bytes < in_bytes + out_bytes) {
    if (s->host_stage) (void)hipHostFree(s->host_stage);
    s->host_stage = nullptr;
    s->host_stage_bytes = 0;
    HIP_OK(hipHostMalloc(&s->host_stage, in_bytes + out_bytes, hipHostMallocDefault));
    s->host_stage_bytes = in_bytes + out_bytes;
  }
  char* hbase = static_cast<char*>(s->host_stage);
  const float* src[7] = {rays->ox, rays->oy, rays->oz, rays->dx, rays->dy, rays->dz, rays->tmax};
  float* d[7];
  for (int i = 0; i < 7; ++i) {
    if (!src[i]) return fail(MH_E_INVALID, "ray array %d is null", i);
    std::memcpy(hbase + i * up(f), src[i], f);
    d[i] = reinterpret_cast<float*>(base + i * up(f));
  }
  uint8_t* dm = nullptr;
  if (rays->masked) {
    std::memcpy(hbase + 7 * up(f), rays->masked, (size_t)n);
    dm = reinterpret_cast<uint8_t*>(base + 7 * up(f));
  }
  HIP_OK(hipMemcpyAsync(base, hbase, rays->masked ? in_bytes : 7 * up(f), hipMemcpyHostToDevice,
                        st));
  char* ob = base + in_bytes;
  mh_hits dh{};
  dh.prim = hits->prim ? reinterpret_cast<int32_t*>(ob) : nullptr;
  dh.t = hits->t ? reinterpret_cast<float*>(ob + up(f)) : nullptr;
  dh.u = hits->u ? reinterpret_cast<float*>(ob + 2 * up(f)) : nullptr;
  dh.v = hits->v ? reinterpret_cast<float*>(ob + 3 * up(f)) : nullptr;
  dh.occluded = hits->occluded ? reinterpret_cast<uint8_t*>(ob + 4 * up(f)) : nullptr;
  mh_rays dr{d[0], d[1], d[2], d[3], d[4], d[5], d[6], dm};
  if ((rc = trace_impl(s, &dr, &dh, n, flags, opts, st))) return rc;
  HIP_OK(hipMemcpyAsync(hbase + in_bytes, ob, out_bytes, hipMemcpyDeviceToHost, st));
  HIP_OK(hipStreamSynchronize(st));
  const char* ho = hbase + in_bytes;
  if (hits->prim) std::memcpy(hits->prim, ho, f);
  if (hits->t) std::memcpy(hits->t, ho + up(f), f);
  if (hits->u) std::memcpy(hits->u, ho + 2 * up(f), f);
  if (hits->v) std::memcpy(hits->v, ho + 3 * up(f), f);
  if (hits->occluded) std::memcpy(hits->occluded, ho + 4 * up(f), (size_t)n);
  return MH_OK;
}

int mh_malloc(void** ptr, size_t bytes) {
  if (!ptr) return fail(MH_E_INVALID, "null argument");
  int rc = ensure_init();
  if (rc) return rc;
  hipError_t e = hipMalloc(ptr, bytes);
  if (e != hipSuccess) return fail(MH_E_NOMEM, "hipMalloc(%zu): %s", bytes, hipGetErrorString(e));
  return MH_OK;
}

int mh_free(void* ptr) {
  if (!ptr) return MH_OK;
  int rc = ensure_init();
  if (rc) return rc;
  HIP_OK(hipFree(ptr));
  return MH_OK;
}

int mh_memcpy_h2d(void* dst, const void* src, size_t bytes) {
  int rc = ensure_init();
  if (rc) return rc;
  HIP_OK(hipMemcpy(dst, src, bytes, hipMemcpyHostToDevice));
  return MH_OK;
}

int mh_memcpy_d2h(void* dst, const void* src, size_t bytes) {
  int rc = ensure_init();
  if (rc) return rc;
  HIP_OK(hipMemcpy(dst, src, bytes, hipMemcpyDeviceToHost));
  return MH_OK;
}

int mh_device_copy(void* dst, const void* src, size_t bytes, void* stream) {
  if ((!dst || !src) && bytes) return fail(MH_E_INVALID, "null argument");
  int rc = ensure_init();
  if (rc) return rc;
  HIP_OK((hipError_t)mh::launch_copy(dst, src, bytes, g_lib.cu_count, stream));
  return MH_OK;
}

int mh_stream_create(void** stream) {
  if (!stream) return fail(MH_E_INVALID, "null argument");
  int rc = ensure_init();
  if (rc) return rc;
  hipStream_t s;
  HIP_OK(hipStreamCreateWithFlags(&s, hipStreamNonBlocking));
  *stream = s;
  return MH_OK;
}

int mh_stream_destroy(void* stream) {
  if (!stream) return MH_OK;
  HIP_OK(hipStreamDestroy(reinterpret_cast<hipStream_t>(stream)));
  return MH_OK;
}

int mh_stream_sync(void* stream) {
  int rc = ensure_init();
  if (rc) return rc;
  HIP_OK(hipStreamSynchronize(reinterpret_cast<hipStream_t>(stream)));
  return MH_OK;
}

int mh_time_trace(const mh_scene* s, const mh_rays* rays, const mh_hits* hits, int64_t n,
                  uint32_t flags, const mh_trace_opts* opts, void* stream, int iters, float* ms) {
  if (!ms || iters < 1) return fail(MH_E_INVALID, "bad timing arguments");
  int rc = ensure_init();
  if (rc) return rc;
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  hipEvent_t a, b;
  HIP_OK(hipEventCreate(&a));
  HIP_OK(hipEventCreate(&b));
  HIP_OK(hipEventRecord(a, st));
  for (int i = 0; i < iters; ++i)
    if ((rc = trace_impl(s, rays, hits, n, flags, opts, stream))) {
      (void)hipEventDestroy(a);
      (void)hipEventDestroy(b);
      return rc;
    }
  HIP_OK(hipEventRecord(b, st));
  HIP_OK(hipEventSynchronize(b));
  HIP_OK(hipEventElapsedTime(ms, a, b));
  (void)hipEventDestroy(a);
  (void)hipEventDestroy(b);
  return MH_OK;
}

}  // extern "C"

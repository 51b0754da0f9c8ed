// Drives a scene of the C ABI on the host (simt.h): loads, refits, updates, exports, run by
// mh_api.cpp, refit.hip, rotate.hip and wide.hip as they are. Traces and device builds are
// not linked.
//
// usage: scene_host DIR OP...
//   DIR holds verts.bin and idx.bin; OP is one of
//   load:NAME    NAME.ids and NAME.nodes into the scene
//   verts:FILE   the vertices of FILE
//   trace:N,BLOCKS,RING,COUNT  mh_trace of N rays with blocks_per_cu, stack_lds and, if COUNT,
//                counters: prints "blocks B ring R spill BYTES pairs P" of its launch
//   refill:R,C   prints "refill N", the idle lanes that a launch configuration's refill and
//                chunk come to in the default layout
//   soa          the node arrays of the SOA layout
//   fixed:BYTES  later traces use a spill area of the caller's, as mh_trace_noalloc does
//   room:BYTES   no device allocation beyond BYTES succeeds from here on
//   limit:N      trees of more than N wide nodes are traversed on their records
//   refit, update
//   save:NAME    the tree to NAME.ids and NAME.nodes, after checking what the traversal
//                reads beside it: prints "irregular I nested N inner X leaves L depth D"
#include <cstdio>
#include <cstdlib>
#include <string>
#include <vector>

#include "internal.h"
#include "prim_setup.h"

mh::LaunchCfg g_launch;
size_t g_fixed = 0;

namespace mh {
int launch_trace(const DevScene&, const DevRays&, const DevHits&, int64_t, const LaunchCfg& c, void*) {
  g_launch = c;
  return 0;
}
int launch_shade(const DevShade&, void*) { return 1; }
int launch_copy(void*, const void*, size_t, int, void*) { return 1; }
int build_launch_setup(const DevBuild&, int, void*) { return 1; }
int build_launch_level(const DevBuild&, int64_t, int64_t, void*) { return 1; }
int build_launch_serial(const DevBuild&, int64_t, int64_t, int32_t*, void*) { return 1; }
int build_launch_ranks(const DevFinish&, const int64_t*, int, int64_t, void*) { return 1; }
}  // namespace mh
void mh_internal::scratch_setup(int) {}

namespace {

template <class T>
std::vector<T> read(const std::string& path) {
  FILE* f = std::fopen(path.c_str(), "rb");
  if (!f) {
    std::fprintf(stderr, "cannot read %s\n", path.c_str());
    std::exit(2);
  }
  std::vector<T> v;
  T x;
  while (std::fread(&x, sizeof(T), 1, f) == 1) v.push_back(x);
  std::fclose(f);
  return v;
}
template <class T>
void write(const std::string& path, const std::vector<T>& v) {
  FILE* f = std::fopen(path.c_str(), "wb");
  std::fwrite(v.data(), sizeof(T), v.size(), f);
  std::fclose(f);
}
void need(bool ok, const char* what, int64_t at) {
  if (ok) return;
  std::fprintf(stderr, "%s (%lld)\n", what, (long long)at);
  std::exit(3);
}
void check(int rc, const std::string& op) {
  if (rc == MH_OK) return;
  std::fprintf(stderr, "%s: %d %s\n", op.c_str(), rc, mh_last_error());
  std::exit(4);
}

// The wide nodes, big leaf counts, leaf starts and triangle records against the records.
// Returns whether every box holds its children's.
bool check_tree(const mh_scene* s) {
  const mh::DevScene d = s->dev();
  const mh::RefNode* refs = d.refs;
  auto same = [](float a, float b) { return std::memcmp(&a, &b, 4) == 0; };
  auto leaf = [&](int ref, int rec) {
    const int n = refs[rec].children, first = refs[rec].child;
    const int c = n < mh::kLeafCountInline ? n : mh::kLeafCountInline;
    need(ref == ~((first << mh::kLeafCountBits) | c), "leaf code", rec);
    if (n >= mh::kLeafCountInline) need(d.big_count[first] == n, "big leaf count", rec);
    need(d.leaf_at[first] == rec, "leaf start", rec);
    for (int k = 1; k < n; ++k) need(d.leaf_at[first + k] == -1, "slot inside a leaf", rec);
  };
  bool nested = true;
  size_t inner = 0;
  struct At {
    int rec, wide;
  };
  std::vector<At> todo;
  if (refs[0].children)
    leaf(d.root_ref, 0);
  else
    todo.push_back({0, d.root_ref});
  auto holds = [&](int p, int c) {
    for (int a = 0; a < 3; ++a)
      nested = nested && refs[c].box.lo[a] >= refs[p].box.lo[a] &&
               refs[c].box.hi[a] <= refs[p].box.hi[a];
  };
  while (!todo.empty()) {
    const At t = todo.back();
    todo.pop_back();
    need(t.wide >= 0 && (uint32_t)t.wide < d.n_wide, "wide reference", t.rec);
    const mh::WideNode& w = d.wide[t.wide];
    ++inner;
    auto order = [&](int rec, int j) {
      for (int o = 0; o < 8; ++o)
        need((w.order >> (3 * o + j) & 1) == !(o >> refs[rec].axis & 1), "visit order", rec);
      need((w.order >> (24 + j) & 1) == !(refs[rec].bits & 1), "any-hit order", rec);
    };
    order(t.rec, 0);
    for (int side = 0; side < 2; ++side) {
      const int kid = refs[t.rec].child + side;
      holds(t.rec, kid);
      int rec[2] = {kid, -1};
      if (refs[kid].children == 0) {
        ++inner;
        order(kid, 1 + side);
        rec[0] = refs[kid].child;
        rec[1] = rec[0] + 1;
        holds(kid, rec[0]);
        holds(kid, rec[1]);
      }
      for (int k = 0; k < 2; ++k) {
        const int at = 2 * side + k;
        if (rec[k] < 0) {
          need(w.ref[at] == mh::kWideEmpty, "empty slot", t.rec);
          for (int a = 0; a < 3; ++a)
            need(w.plane[2 * a][at] > w.plane[2 * a + 1][at], "empty slot's box", t.rec);
          continue;
        }
        for (int a = 0; a < 3; ++a)
          need(same(w.plane[2 * a][at], refs[rec[k]].box.lo[a]) &&
                   same(w.plane[2 * a + 1][at], refs[rec[k]].box.hi[a]),
               "wide box", rec[k]);
        if (refs[rec[k]].children)
          leaf(w.ref[at], rec[k]);
        else
          todo.push_back({rec[k], w.ref[at]});
      }
    }
  }
  need(inner == s->n_inner, "inner records", (int64_t)inner);
  for (uint32_t k = 0; k < s->nt; ++k) {
    float rec[12];
    mh::ks_record(mh::load_tri(s->verts.data(), s->idx.data(), d.obj_ids[k]), rec);
    for (int j = 0; j < 12; ++j)
      need(same(rec[j], d.tris[12 * (size_t)k + j]) || (rec[j] != rec[j] && d.tris[12 * (size_t)k + j] != d.tris[12 * (size_t)k + j]),
           "triangle record", k);
  }
  return nested;
}

}  // namespace

int main(int argc, char** argv) {
  if (argc < 3) return 2;
  const std::string dir = std::string(argv[1]) + "/";
  const auto verts = read<float>(dir + "verts.bin");
  const auto idx = read<uint32_t>(dir + "idx.bin");
  mh_scene* s = nullptr;
  check(mh_scene_create(verts.data(), (uint32_t)(verts.size() / 3), idx.data(),
                        (uint32_t)(idx.size() / 3), &s), "create");
  for (int k = 2; k < argc; ++k) {
    const std::string op = argv[k];
    const size_t colon = op.find(':');
    const std::string what = op.substr(0, colon);
    const std::string name = colon == std::string::npos ? "" : dir + op.substr(colon + 1);
    if (what == "load") {
      const auto ids = read<int32_t>(name + ".ids");
      const auto nodes = read<mh::RefNode>(name + ".nodes");
      check(mh_scene_load_dynbvh(s, ids.data(), (uint32_t)ids.size(), nodes.data(),
                                 (uint32_t)nodes.size(), MH_PRIM_KENSLER_SHIRLEY), op);
    } else if (what == "verts") {
      check(mh_scene_set_vertices(s, read<float>(name).data(), 0, nullptr), op);
    } else if (what == "trace") {
      long n = 0;
      mh_trace_opts o{};
      int count = 0;
      if (std::sscanf(op.c_str() + colon + 1, "%ld,%d,%d,%d", &n, &o.blocks_per_cu, &o.stack_lds,
                      &count) != 4)
        return 2;
      int64_t counters[2];
      if (count) o.counters = counters;
      float f = 0.f;  // never read: the launch is only recorded
      int32_t prim = 0;
      const mh_rays rays{&f, &f, &f, &f, &f, &f, &f, nullptr};
      const mh_hits hits{&prim, nullptr, nullptr, nullptr, nullptr};
      static char fixed;
      check(g_fixed ? mh_internal::trace_fixed_spill(s, &rays, &hits, n, 0, &o, nullptr, &fixed, g_fixed)
                    : mh_trace(s, &rays, &hits, n, 0, &o, nullptr), op);
      const mh::LaunchCfg& c = g_launch;
      const int64_t stack =
          (int64_t)s->stack_bound(c.pairs ? MH_LAYOUT_REF : MH_LAYOUT_PAIR) - c.stack_lds;
      need(c.blocks > 0 && c.spill_stride == (int64_t)c.blocks * 64, "spill columns", c.blocks);
      const size_t area = stack <= 0 ? 0 : g_fixed ? g_fixed : s->spill[nullptr]->bytes;
      if (stack > 0) need((size_t)stack * c.spill_stride * 8 <= area, "spill area", stack);
      std::printf("blocks %d ring %d spill %zu pairs %d\n", c.blocks, c.stack_lds, area, c.pairs);
    } else if (what == "fixed") {
      g_fixed = (size_t)std::atoll(op.c_str() + colon + 1);
    } else if (what == "refill") {
      int r = 0, c = 0;
      if (std::sscanf(op.c_str() + colon + 1, "%d,%d", &r, &c) != 2) return 2;
      std::printf("refill %d\n", mh::wide_refill(r, c));
    } else if (what == "soa") {
      check(mh_internal::ensure_soa(s, nullptr), op);
    } else if (what == "room") {
      simt::room = (size_t)std::atoll(op.c_str() + colon + 1);
    } else if (what == "limit") {
      s->max_wide = (uint32_t)std::atol(op.c_str() + colon + 1);
    } else if (what == "refit") {
      check(mh_scene_refit(s, nullptr), op);
    } else if (what == "update") {
      check(mh_scene_update(s, nullptr), op);
    } else if (what == "save") {
      const bool nested = check_tree(s);
      uint32_t ni = 0, nn = 0;
      check(mh_scene_export_dynbvh(s, nullptr, &ni, nullptr, &nn), op);
      std::vector<int32_t> ids(ni);
      std::vector<mh::RefNode> nodes(nn);
      check(mh_scene_export_dynbvh(s, ids.data(), &ni, nodes.data(), &nn), op);
      write(name + ".ids", ids);
      write(name + ".nodes", nodes);
      std::printf("irregular %d nested %d inner %u leaves %u depth %u\n",
                  s->irregular.as<int32_t>()[0], (int)nested, s->n_inner, s->n_leaves, s->depth);
    } else {
      return 2;
    }
  }
  check(mh_scene_destroy(s), "destroy");
  return 0;
}

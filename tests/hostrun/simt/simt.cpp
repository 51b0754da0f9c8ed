// The lane scheduler and memory of simt.h.
#include "simt.h"

#include <sanitizer/common_interface_defs.h>
#include <ucontext.h>

#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <memory>
#include <random>
#include <vector>

dim3 threadIdx, blockIdx, gridDim, blockDim;

namespace simt {

size_t room = ~(size_t)0;

namespace {

constexpr size_t kStack = 256 << 10;

struct Lane {
  std::unique_ptr<char[]> stack{new char[kStack]};
  ucontext_t ctx;
  void* fake = nullptr;
  enum { kReady, kWaiting, kDone } state = kDone;
  Op op = Op::kBarrier;
  int src = 0, site = 0;
  unsigned long long value = 0;
};

std::vector<Lane> lanes;
ucontext_t main_ctx;
void* main_fake = nullptr;
const void* main_stack = nullptr;
size_t main_size = 0;
int running = -1;
const std::function<void()>* body = nullptr;
std::mt19937 order(1);

void to_main(bool last) {
  Lane& l = lanes[running];
  __sanitizer_start_switch_fiber(last ? nullptr : &l.fake, main_stack, main_size);
  swapcontext(&l.ctx, &main_ctx);
  __sanitizer_finish_switch_fiber(l.fake, &main_stack, &main_size);
}

void entry() {
  __sanitizer_finish_switch_fiber(nullptr, &main_stack, &main_size);
  (*body)();
  lanes[running].state = Lane::kDone;
  to_main(true);
}

void resume(int k) {
  Lane& l = lanes[k];
  running = k;
  threadIdx = dim3((unsigned)k);
  __sanitizer_start_switch_fiber(&main_fake, l.stack.get(), kStack);
  swapcontext(&main_ctx, &l.ctx);
  __sanitizer_finish_switch_fiber(main_fake, nullptr, nullptr);
  running = -1;
}

// Releases the lanes of one wave that wait at its first ballot or shuffle, in program order.
bool release_wave(int first, int end) {
  int site = -1;
  for (int k = first; k < end; ++k)
    if (lanes[k].state == Lane::kWaiting && lanes[k].op != Op::kBarrier &&
        (site < 0 || lanes[k].site < site))
      site = lanes[k].site;
  if (site < 0) return false;
  unsigned long long mask = 0, here = 0, in[64];
  auto at = [&](int k) {
    return lanes[k].state == Lane::kWaiting && lanes[k].op != Op::kBarrier && lanes[k].site == site;
  };
  for (int k = first; k < end; ++k)
    if (at(k)) {
      here |= 1ull << (k - first);
      in[k - first] = lanes[k].value;
      if (lanes[k].value) mask |= 1ull << (k - first);
    }
  for (int k = first; k < end; ++k)
    if (here >> (k - first) & 1) {
      Lane& l = lanes[k];
      if (l.op == Op::kBallot) {
        l.value = mask;
      } else {
        if (!(here >> l.src & 1)) {
          std::fprintf(stderr, "line %d: lane %d reads lane %d, which is not there\n", site,
                       k - first, l.src);
          std::abort();
        }
        l.value = in[l.src];
      }
      l.state = Lane::kReady;
    }
  return true;
}

void run_block(int n, std::vector<int>& turn) {
  for (int k = 0; k < n; ++k) {
    Lane& l = lanes[k];
    getcontext(&l.ctx);
    l.ctx.uc_stack.ss_sp = l.stack.get();
    l.ctx.uc_stack.ss_size = kStack;
    l.ctx.uc_link = nullptr;
    l.fake = nullptr;
    makecontext(&l.ctx, entry, 0);
    l.state = Lane::kReady;
  }
  for (;;) {
    std::shuffle(turn.begin(), turn.end(), order);
    for (int k : turn)
      if (lanes[k].state == Lane::kReady) resume(k);
    bool any = false, left = false;
    for (int w = 0; w < n; w += 64) any |= release_wave(w, std::min(n, w + 64));
    if (any) continue;
    int site = 0;
    for (int k = 0; k < n; ++k)  // every lane left is at a barrier, which must be the same one
      if (lanes[k].state == Lane::kWaiting) {
        if (left && lanes[k].site != site) {
          std::fprintf(stderr, "lanes wait at the barriers of lines %d and %d\n", site, lanes[k].site);
          std::abort();
        }
        lanes[k].state = Lane::kReady;
        site = lanes[k].site;
        left = true;
      }
    if (!left) return;
  }
}

}  // namespace

unsigned long long wait(Op op, unsigned long long value, int src, int site) {
  Lane& l = lanes[running];
  l.op = op;
  l.value = value;
  l.src = src;
  l.site = site;
  l.state = Lane::kWaiting;
  to_main(false);
  return l.value;
}

void launch(dim3 grid, dim3 block, const std::function<void()>& lane) {
  const int n = (int)block.x;
  if ((int)lanes.size() < n) lanes = std::vector<Lane>(n);
  body = &lane;
  gridDim = grid;
  blockDim = block;
  std::vector<int> blocks(grid.x), turn(n);
  for (unsigned b = 0; b < grid.x; ++b) blocks[b] = (int)b;
  for (int k = 0; k < n; ++k) turn[k] = k;
  std::shuffle(blocks.begin(), blocks.end(), order);
  for (int b : blocks) {
    blockIdx = dim3((unsigned)b);
    run_block(n, turn);
  }
}

}  // namespace simt

hipError_t hipMalloc(void** p, size_t n) {
  *p = n <= simt::room ? std::malloc(n) : nullptr;
  if (*p && n < (64 << 20)) std::memset(*p, 0xA5, n);  // whatever was there before
  return *p ? hipSuccess : hipErrorOutOfMemory;
}
hipError_t hipFree(void* p) {
  std::free(p);
  return hipSuccess;
}
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) {
  std::memcpy(d, s, n);
  return hipSuccess;
}
hipError_t hipMemset(void* d, int v, size_t n) {
  std::memset(d, v, n);
  return hipSuccess;
}
hipError_t hipMemcpy2DAsync(void* d, size_t dp, const void* s, size_t sp, size_t w, size_t h,
                            hipMemcpyKind, hipStream_t) {
  for (size_t k = 0; k < h; ++k)
    std::memcpy((char*)d + k * dp, (const char*)s + k * sp, w);
  return hipSuccess;
}
hipError_t hipGetDeviceProperties(hipDeviceProp_t* p, int) {
  *p = hipDeviceProp_t{256, size_t(1) << 30, "host"};
  return hipSuccess;
}

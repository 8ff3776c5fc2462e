// The depth order's kernels (csrc/gs_sample_sort.h) on the CPU, under a schedule of the caller's
// choice: every thread of a workgroup is a fiber, the 64 lanes of a wavefront meet at every
// wavefront operation, and between two workgroup barriers the wavefronts run one after the other,
// each as far as it gets. With the first wavefront first (or the last one first) any word that one
// wavefront writes and another still has to read, with no barrier between, is read too late.
// Workgroups run one after the other; LDS keeps what the previous one left.
#include <stdint.h>
#include <string.h>
#include <ucontext.h>

#include <algorithm>
#include <functional>
#include <memory>
#include <vector>

namespace emu {

struct Idx {
  unsigned x;
};

struct Wave {  // a meeting point of 64 lanes; the values of two meetings, so that none is overwritten early
  uint32_t val[2][64];
  unsigned arrived = 0, gen = 0;
};

struct Fiber {
  ucontext_t ctx;
  std::unique_ptr<char[]> stack;
  bool done = false;
};

constexpr size_t kStack = 48 << 10;
static std::vector<Fiber> fibers;
static std::vector<Wave> waves;
static ucontext_t scheduler;
static std::function<void()> body;
static Idx thread_idx, block_idx, grid_dim;
static unsigned threads, at_barrier, barrier_gen;
static bool last_wave_first, progress;

static void yield() { swapcontext(&fibers[thread_idx.x].ctx, &scheduler); }

static const uint32_t* meet(uint32_t v) {
  Wave& w = waves[thread_idx.x / 64];
  const unsigned g = w.gen;
  w.val[g & 1][thread_idx.x % 64] = v;
  progress = true;
  if (++w.arrived == 64) {
    w.arrived = 0;
    ++w.gen;
  }
  while (w.gen == g) yield();
  return w.val[g & 1];
}

static void barrier() {
  const unsigned g = barrier_gen;
  progress = true;
  ++at_barrier;  // (it opens when every wavefront has run as far as it gets)
  while (barrier_gen == g) yield();
}

static void entry() {
  body();
  fibers[thread_idx.x].done = true;
  progress = true;
  yield();
}

static bool launch(unsigned blocks, unsigned n_threads, std::function<void()> f) {
  body = std::move(f);
  threads = n_threads;
  grid_dim.x = blocks;
  if (fibers.size() < threads) fibers.resize(threads);
  const unsigned n_waves = threads / 64;
  for (unsigned b = 0; b < blocks; ++b) {
    block_idx.x = b;
    waves.assign(n_waves, Wave());
    at_barrier = barrier_gen = 0;
    for (unsigned t = 0; t < threads; ++t) {
      Fiber& fb = fibers[t];
      if (!fb.stack) fb.stack.reset(new char[kStack]);
      fb.done = false;
      getcontext(&fb.ctx);
      fb.ctx.uc_stack.ss_sp = fb.stack.get();
      fb.ctx.uc_stack.ss_size = kStack;
      fb.ctx.uc_link = nullptr;
      makecontext(&fb.ctx, entry, 0);
    }
    for (;;) {
      bool any = false, moved = false;
      for (unsigned k = 0; k < n_waves; ++k) {
        const unsigned w = last_wave_first ? n_waves - 1 - k : k;
        do {  // this wavefront, as far as it gets
          progress = false;
          for (unsigned l = 0; l < 64; ++l) {
            if (fibers[64 * w + l].done) continue;
            thread_idx.x = 64 * w + l;
            swapcontext(&scheduler, &fibers[64 * w + l].ctx);
          }
          moved |= progress;
        } while (progress);
        for (unsigned l = 0; l < 64; ++l) any |= !fibers[64 * w + l].done;
      }
      if (!any) break;
      if (at_barrier == threads) {
        at_barrier = 0;
        ++barrier_gen;
        continue;
      }
      if (!moved) return false;  // a barrier or a wavefront operation that some lane never reaches
    }
  }
  return true;
}

static bool all_ended;

}  // namespace emu

// ---- what gs_sample_sort.h takes from HIP and from the sources it is included in ----
#define __global__
#define __device__
#define __forceinline__ inline
#define __shared__ static
#define __launch_bounds__(...)
#define __align__(n) alignas(n)
#define threadIdx emu::thread_idx
#define blockIdx emu::block_idx
#define gridDim emu::grid_dim
#define __syncthreads emu::barrier
#define hipLaunchKernelGGL(kernel, grid, block, lds, stream, ...) \
  emu::all_ended &= emu::launch((grid).x, (block).x, [=] { kernel(__VA_ARGS__); })

typedef void* hipStream_t;
struct dim3 {
  unsigned x;
  explicit dim3(int64_t v) : x(static_cast<unsigned>(v)) {}
};
struct alignas(16) uint4 {
  uint32_t x, y, z, w;
};
static int __popcll(uint64_t v) { return __builtin_popcountll(v); }
static int __clz(int v) { return v ? __builtin_clz(static_cast<unsigned>(v)) : 32; }
static uint32_t __umulhi(uint32_t a, uint32_t b) { return static_cast<uint32_t>((static_cast<uint64_t>(a) * b) >> 32); }
static uint32_t atomicAdd(uint32_t* p, uint32_t v) {
  const uint32_t old = *p;
  *p = old + v;
  return old;
}
static uint64_t __ballot(int v) {
  const uint32_t* all = emu::meet(v != 0);
  uint64_t m = 0;
  for (int l = 0; l < 64; ++l) m |= static_cast<uint64_t>(all[l]) << l;
  return m;
}

namespace gs {
using std::max;
using std::min;
constexpr int kWave = 64;
constexpr int kScanThreads = 256;

static void wave_sync() { emu::meet(0); }
static uint64_t lanemask_lt(int lane) { return lane == 0 ? 0ull : ~0ull >> (64 - lane); }
template <typename F>
static uint32_t wave_scan(uint32_t v, uint32_t id, F f) {
  const uint32_t* all = emu::meet(v);
  uint32_t r = id;
  for (unsigned l = 0; l <= threadIdx.x % 64; ++l) r = f(r, all[l]);
  return r;
}
static uint32_t wave_incl_scan(uint32_t v) {
  return wave_scan(v, 0u, [](uint32_t a, uint32_t b) { return a + b; });
}
static uint32_t wave_last(uint32_t v) { return emu::meet(v)[63]; }
static uint32_t wave_excl_scan(uint32_t v, int, uint32_t& total) {
  const uint32_t incl = wave_incl_scan(v);
  total = wave_last(incl);
  return incl - v;
}
static uint32_t block_inclusive_scan(uint32_t v, uint32_t* s_wave, uint32_t& total) {
  const unsigned wave = threadIdx.x / 64;
  v = wave_incl_scan(v);
  if (threadIdx.x % 64 == 63) s_wave[wave] = v;
  __syncthreads();
  total = 0;
  for (unsigned w = 0; w < 4; ++w) {
    if (w < wave) v += s_wave[w];
    total += s_wave[w];
  }
  __syncthreads();
  return v;
}
template <int BITS>
static uint64_t match_bits(uint32_t d, bool valid) {
  uint64_t peers = __ballot(valid);
  for (int bit = 0; bit < BITS; ++bit) {
    const bool set = (d >> bit) & 1u;
    const uint64_t m = __ballot(set);
    peers &= set ? m : ~m;
  }
  return valid ? peers : 0ull;
}
static int xcd_tile(int b, int) { return b; }
static void rs_rowscan_kernel(uint32_t* hist, int n_tiles, uint32_t* totals) {
  if (threadIdx.x != 0) return;
  uint32_t* row = hist + static_cast<int64_t>(blockIdx.x) * n_tiles;
  uint32_t run = 0;
  for (int t = 0; t < n_tiles; ++t) {
    const uint32_t c = row[t];
    row[t] = run;
    run += c;
  }
  totals[blockIdx.x] = run;
}
}  // namespace gs

#include "gs_sample_sort.h"

// order [n] and (may be NULL) offsets [n + 1] of the stable sort of keys; false: some thread waited
// for ever. last_first: the last wavefront runs first after every barrier, else the first.
extern "C" int emulate_sample_sort(const uint32_t* keys, const uint32_t* counts, int64_t n, int last_first,
                                   uint32_t* order, uint32_t* offsets) {
  emu::last_wave_first = last_first != 0;
  emu::all_ended = true;
  std::vector<uint64_t> ws(gs::ss_layout(n).end / 8 + 1, 0xababababababababull);
  gs::sample_sort(keys, counts, n, order, offsets, reinterpret_cast<char*>(ws.data()), nullptr);
  return emu::all_ended ? 1 : 0;
}

// The sampled positions of n keys (pos: NULL, or room for them); returns their number.
extern "C" int64_t sample_positions(int64_t n, uint32_t* pos) {
  if (n <= gs::kSsSmall) return 0;
  const uint32_t S = static_cast<uint32_t>(gs::ss_layout(n).B) * gs::kSsOver;
  for (uint32_t i = 0; pos && i < S; ++i) pos[i] = gs::ss_sample_pos(i, (static_cast<uint64_t>(n) << 32) / S);
  return S;
}

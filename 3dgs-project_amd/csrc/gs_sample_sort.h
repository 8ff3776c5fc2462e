// Stable order of n 32-bit keys (with the values 0 .. n - 1) and the exclusive scan of a count per
// value in that order, by one level of buckets: the depth ordering of the binning. Included by
// binning.hip (it uses its wavefront ranking and row scan).
//
// An LSD radix sort of the depth keys takes 3 launches per 9-bit digit, each as long as one
// workgroup's chain of loads, ranking rounds and staged writes, and the scan of the counts two
// more: 11 launches and 77 us at 1M keys, of which the bytes need about 8. Here every key is moved
// once to its bucket and sorted there in LDS:
//
//   splitters  kSsOver samples per bucket, one at a hashed position in each of S equal ranges of
//              the input; a thread ranks its sample among all of them (all pairs) and writes it if
//              it is a bucket boundary. Keys compare as (key, position), so equal keys are split
//              too and no bucket depends on the keys' distribution.
//   count      2048 keys per workgroup: bucket by binary search over the boundaries in LDS, bucket
//              histogram -> tile_hist[bucket][tile]
//   rowscan    (rs_rowscan_kernel) a workgroup per bucket
//   scatter    the workgroup's keys ranked stably by bucket and written in runs; counts summed per
//              bucket
//   local      a workgroup per bucket: order and counts' scan of its keys, in LDS
//
// Up to kSsSmall keys the last kernel alone sorts everything: one launch. Depth order and offsets
// against the radix sort and scan (view depths, a third culled): 2k keys 36 -> 12 us, 4k 42 -> 16,
// 100k 47 -> 32, 300k 55 -> 39, 1M 77 -> 67; at 3M the radix sort is faster (153 against 157, and 134
// against 169 without equal keys), so it is taken beyond kSsMaxKeys. Reserving bucket space
// by atomics instead of count and rowscan was slower (one kernel of 46 us for count, rowscan and
// scatter together at 1M: a returning atomic per workgroup and bucket). No workgroup waits on
// another. Over other distributions (a third culled, 37 or 1000 distinct depths, tight clusters,
// sorted; 2k to 1M keys) it is between 0.14 and 1.05 times the radix sort's time.
#pragma once

namespace gs {

constexpr int kSsThreads = 256;
constexpr int kSsRounds = 8;
constexpr int kSsTile = kSsThreads * kSsRounds;  // keys per workgroup of count and scatter
constexpr int kSsBits = 9;
constexpr int kSsMaxBuckets = 1 << kSsBits;
constexpr int kSsOver = 8;      // samples per bucket
constexpr int kSsSmall = 4096;  // keys sorted by one workgroup
// Keys per bucket aimed at: a quarter of the LDS capacity of its workgroup. Larger buckets cost less
// per key, but fewer workgroups than CUs would leave the chip idle. A bucket beyond the capacity is
// sorted by its workgroup through global memory, at about 10 us per 1000 keys. The sampled positions
// are hashed from n alone: an input that does not follow them (whatever its order and its values'
// distribution) has such a bucket, slightly beyond the capacity, once in 1e4 inputs, but then on every
// sort of that input; one made against the positions can bring nearly all keys into one bucket (30k
// keys 0.35 ms, 100k 1.1, 1M 10.7; the radix sort takes 0.05 to 0.08).
constexpr int64_t kSsLargeFrom = int64_t(512) << 10;
static int ss_mean(int64_t n) { return n < kSsLargeFrom ? 1024 : 2048; }
constexpr int64_t kSsMaxKeys = int64_t(1) << 20;

// The published integer mixer lowbias32 (C. Wellons); any mixing of the bits would serve.
__device__ __forceinline__ uint32_t ss_hash(uint32_t x) {
  x ^= x >> 16;
  x *= 0x7feb352du;
  x ^= x >> 15;
  x *= 0x846ca68bu;
  return x ^ (x >> 16);
}

// Position of sample i: a hashed place in [i step, (i + 1) step), step = n / S in 32.32 fixed point.
__device__ __forceinline__ uint32_t ss_sample_pos(uint32_t i, uint64_t step) {
  const uint32_t lo = static_cast<uint32_t>((i * step) >> 32), hi = static_cast<uint32_t>(((i + 1) * step) >> 32);
  return lo + __umulhi(ss_hash(i), hi - lo);
}

// 32 samples per workgroup of 1024 threads, 32 comparing threads to a sample. The samples'
// positions increase with their index, so a sample before the thread's own counts when its key is
// not greater, one after it when its key is less.
__global__ __launch_bounds__(1024) void ss_splitters_kernel(const uint32_t* __restrict__ keys, uint64_t step, uint32_t S,
                                                            uint64_t* __restrict__ spl, uint32_t* __restrict__ sums) {
  __shared__ __align__(16) uint32_t s_key[kSsMaxBuckets * kSsOver];
  __shared__ uint32_t s_rank[32];
  const uint32_t tid = threadIdx.x, mine = tid & 31;
  if (blockIdx.x == 0) {
    for (uint32_t k = tid; k < S / kSsOver; k += 1024) sums[k] = 0u;
  }
  if (tid < 32) s_rank[tid] = 0u;
  const uint32_t S32 = (S + 31) & ~31u;
  for (uint32_t i = tid; i < S32; i += 1024) s_key[i] = i < S ? keys[ss_sample_pos(i, step)] : 0xffffffffu;
  __syncthreads();
  const uint32_t own = blockIdx.x * 32 + mine;
  const uint32_t key = own < S ? s_key[own] : 0u;
  uint32_t rank = 0;
  for (uint32_t b = tid >> 5; b < S32 / 32; b += 32) {
    const uint4* s4 = reinterpret_cast<const uint4*>(s_key + 32 * b);
    if (b == blockIdx.x) {
      for (uint32_t q = 0; q < 32; ++q) {
        const uint32_t v = s_key[32 * b + q];
        rank += (v < key || (v == key && q < mine)) ? 1u : 0u;
      }
    } else {
      const uint32_t top = b < blockIdx.x ? key : key - 1u;  // counts v <= top
      uint32_t c = 0;
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        const uint4 v = s4[q];
        c += (v.x <= top) + (v.y <= top) + (v.z <= top) + (v.w <= top);
      }
      rank += (b < blockIdx.x || key != 0u) ? c : 0u;
    }
  }
  atomicAdd(&s_rank[mine], rank);
  __syncthreads();
  if (tid < 32 && own < S) {
    const uint32_t r = s_rank[tid];
    if (r != 0u && r % kSsOver == 0u)
      spl[r / kSsOver - 1u] = (static_cast<uint64_t>(key) << 32) | ss_sample_pos(own, step);
  }
}

// Workgroup `tile` of count: the bucket of each of its keys (the number of boundaries not above
// it) into bucket_of, and their histogram.
__global__ __launch_bounds__(kSsThreads) void ss_count_kernel(const uint32_t* __restrict__ keys, uint32_t n,
                                                              const uint64_t* __restrict__ spl, int B,
                                                              uint16_t* __restrict__ bucket_of,
                                                              uint32_t* __restrict__ tile_hist, int n_tiles) {
  __shared__ uint64_t s_spl[kSsMaxBuckets];
  __shared__ uint32_t s_h[kSsMaxBuckets];
  const int tile = xcd_tile(blockIdx.x, gridDim.x);
  const uint32_t base = static_cast<uint32_t>(tile) * kSsTile + threadIdx.x;
  uint32_t key[kSsRounds];
#pragma unroll
  for (int r = 0; r < kSsRounds; ++r) {
    const uint32_t i = base + r * kSsThreads;
    key[r] = i < n ? keys[i] : 0u;
  }
  for (int k = threadIdx.x; k < kSsMaxBuckets; k += kSsThreads) {
    s_spl[k] = k < B - 1 ? spl[k] : ~0ull;
    s_h[k] = 0u;
  }
  __syncthreads();
  int pos[kSsRounds];
#pragma unroll
  for (int r = 0; r < kSsRounds; ++r) pos[r] = 0;
#pragma unroll
  for (int s = kSsBits - 1; s >= 0; --s) {
    const int step = 1 << s;
#pragma unroll
    for (int r = 0; r < kSsRounds; ++r) {
      const uint64_t x = (static_cast<uint64_t>(key[r]) << 32) | (base + r * kSsThreads);
      if (s_spl[pos[r] + step - 1] <= x) pos[r] += step;
    }
  }
#pragma unroll
  for (int r = 0; r < kSsRounds; ++r) {
    const uint32_t i = base + r * kSsThreads;
    if (i < n) {
      bucket_of[i] = static_cast<uint16_t>(pos[r]);
      atomicAdd(&s_h[pos[r]], 1u);
    }
  }
  __syncthreads();
  for (int k = threadIdx.x; k < B; k += kSsThreads) tile_hist[static_cast<int64_t>(k) * n_tiles + tile] = s_h[k];
}

// Scatter of a tile into the buckets: stable ranks by bucket (a wavefront owns 512 consecutive
// keys), the tile staged in LDS in bucket order, written as one run per bucket. counts (may be
// NULL) go along, their per-bucket sums into `sums`. Tile 0 writes the buckets' starts.
__global__ __launch_bounds__(kSsThreads) void ss_scatter_kernel(
    const uint32_t* __restrict__ keys, const uint16_t* __restrict__ bucket_of, const uint32_t* __restrict__ counts,
    uint32_t n, int B, const uint32_t* __restrict__ tile_offs, int n_tiles, const uint32_t* __restrict__ totals,
    uint32_t* __restrict__ seg_key, uint32_t* __restrict__ seg_val, uint32_t* __restrict__ seg_cnt,
    uint32_t* __restrict__ starts, uint32_t* __restrict__ sums) {
  constexpr int NBK = kSsMaxBuckets;
  constexpr int kWaves = kSsThreads / kWave;
  constexpr int DPT = NBK / kSsThreads;  // consecutive buckets per thread
  __shared__ uint32_t s_cnt[kWaves][NBK];
  __shared__ uint32_t s_excl[NBK], s_goff[NBK], s_sum[NBK];
  __shared__ uint32_t s_key[kSsTile], s_val[kSsTile], s_c[kSsTile];
  __shared__ uint16_t s_b[kSsTile];
  __shared__ uint32_t s_wave[4];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int tile = xcd_tile(blockIdx.x, gridDim.x);
  const uint32_t tile_base = static_cast<uint32_t>(tile) * kSsTile;
  const uint32_t base = tile_base + wave * (kWave * kSsRounds) + lane;
  uint32_t key[kSsRounds], cnt[kSsRounds], rank[kSsRounds], bkt[kSsRounds];
#pragma unroll
  for (int r = 0; r < kSsRounds; ++r) {
    const uint32_t i = base + r * kWave;
    const bool ok = i < n;
    key[r] = ok ? keys[i] : 0u;
    bkt[r] = ok ? bucket_of[i] : 0u;
    cnt[r] = (ok && counts) ? counts[i] : 0u;
  }
  for (int k = threadIdx.x; k < kWaves * NBK; k += kSsThreads) (&s_cnt[0][0])[k] = 0u;
  for (int k = threadIdx.x; k < NBK; k += kSsThreads) s_sum[k] = 0u;
  {
    uint32_t t[DPT], tsum = 0;
#pragma unroll
    for (int e = 0; e < DPT; ++e) {
      const int d = static_cast<int>(threadIdx.x) * DPT + e;
      t[e] = d < B ? totals[d] : 0u;
      tsum += t[e];
    }
    uint32_t all;
    uint32_t run = block_inclusive_scan(tsum, s_wave, all) - tsum;
#pragma unroll
    for (int e = 0; e < DPT; ++e) {
      const int d = static_cast<int>(threadIdx.x) * DPT + e;
      if (d < B) {
        s_goff[d] = run + tile_offs[static_cast<int64_t>(d) * n_tiles + tile];
        if (tile == 0) starts[d] = run;
      }
      run += t[e];
    }
    if (tile == 0 && threadIdx.x == 0) starts[B] = n;
  }
  __syncthreads();
  const uint64_t lt = lanemask_lt(lane);
#pragma unroll
  for (int r = 0; r < kSsRounds; ++r) {
    const bool valid = base + r * kWave < n;
    const uint32_t d = bkt[r];
    const uint64_t peers = match_bits<kSsBits>(d, valid);
    rank[r] = valid ? s_cnt[wave][d] + static_cast<uint32_t>(__popcll(peers & lt)) : 0u;
    wave_sync();
    if (valid && (peers & lt) == 0ull) s_cnt[wave][d] += static_cast<uint32_t>(__popcll(peers));
    wave_sync();
    if (cnt[r]) atomicAdd(&s_sum[d], cnt[r]);
  }
  __syncthreads();
  {
    uint32_t dt[DPT], tsum = 0;
#pragma unroll
    for (int e = 0; e < DPT; ++e) {
      const int d = static_cast<int>(threadIdx.x) * DPT + e;
      uint32_t acc = 0;
#pragma unroll
      for (int w = 0; w < kWaves; ++w) {
        const uint32_t c = s_cnt[w][d];
        s_cnt[w][d] = acc;
        acc += c;
      }
      dt[e] = acc;
      tsum += acc;
    }
    uint32_t all;
    uint32_t run = block_inclusive_scan(tsum, s_wave, all) - tsum;
#pragma unroll
    for (int e = 0; e < DPT; ++e) {
      s_excl[static_cast<int>(threadIdx.x) * DPT + e] = run;
      run += dt[e];
    }
  }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < kSsRounds; ++r) {
    const uint32_t i = base + r * kWave;
    if (i < n) {
      const uint32_t p = s_excl[bkt[r]] + s_cnt[wave][bkt[r]] + rank[r];
      s_key[p] = key[r];
      s_val[p] = i;
      s_c[p] = cnt[r];
      s_b[p] = static_cast<uint16_t>(bkt[r]);
    }
  }
  __syncthreads();
  const uint32_t have = min(static_cast<uint32_t>(kSsTile), n - tile_base);
  for (uint32_t p = threadIdx.x; p < have; p += kSsThreads) {
    const uint32_t d = s_b[p], g = s_goff[d] + (p - s_excl[d]);
    seg_key[g] = s_key[p];
    seg_val[g] = s_val[p];
    if (counts) seg_cnt[g] = s_c[p];
  }
  if (counts) {
    for (int d = threadIdx.x; d < B; d += kSsThreads)
      if (s_sum[d]) atomicAdd(&sums[d], s_sum[d]);
  }
}

// Fold of v over the workgroup of NT threads by f, to every thread. As in the two functions below, the
// words s_w are still being read by other wavefronts when it returns: nothing may be stored there
// before the next barrier (each of the three begins its own stores with one).
template <int NT, typename F>
__device__ __forceinline__ uint32_t block_fold(uint32_t v, uint32_t* s_w, F f) {  // (0 is f's identity)
  v = wave_last(wave_scan(v, 0u, f));
  __syncthreads();
  if ((threadIdx.x & 63) == 0) s_w[threadIdx.x >> 6] = v;
  __syncthreads();
  v = s_w[0];
  for (int w = 1; w < NT / kWave; ++w) v = f(v, s_w[w]);
  return v;
}

// Minimum of lo and maximum of hi over the workgroup, to every thread.
template <int NT>
__device__ __forceinline__ void block_min_max(uint32_t& lo, uint32_t& hi, uint32_t* s_w, uint32_t* s_w2) {
  lo = wave_last(wave_scan(lo, ~0u, [](uint32_t x, uint32_t y) { return min(x, y); }));
  hi = wave_last(wave_scan(hi, 0u, [](uint32_t x, uint32_t y) { return max(x, y); }));
  __syncthreads();
  if ((threadIdx.x & 63) == 0) {
    s_w[threadIdx.x >> 6] = lo;
    s_w2[threadIdx.x >> 6] = hi;
  }
  __syncthreads();
  for (int w = 0; w < NT / kWave; ++w) {
    lo = min(lo, s_w[w]);
    hi = max(hi, s_w2[w]);
  }
}

// Exclusive scan of one value per thread over the workgroup of NT threads; `total` the sum.
template <int NT>
__device__ __forceinline__ uint32_t block_excl_scan(uint32_t v, uint32_t* s_w, uint32_t& total) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const uint32_t incl = wave_incl_scan(v);
  __syncthreads();
  if (lane == 63) s_w[wave] = incl;
  __syncthreads();
  uint32_t before = 0, all = 0;
#pragma unroll
  for (int w = 0; w < NT / kWave; ++w) {
    const uint32_t t = s_w[w];
    before += w < wave ? t : 0u;
    all += t;
  }
  total = all;
  return before + incl - v;
}

struct SsLocalArgs {
  const uint32_t* key;  // bucket-ordered keys (the input keys for the single-workgroup sort)
  const uint32_t* val;  // their values; NULL: position
  const uint32_t* cnt;  // their counts (may be NULL: no offsets)
  // two sets of scratch of the same sizes, for buckets beyond the LDS capacity
  uint32_t *key1, *val1, *cnt1, *key2, *val2, *cnt2;
  const uint32_t* starts;  // [B + 1]; NULL: one bucket of n keys
  const uint32_t* sums;    // [B] counts per bucket
  uint32_t n;
  uint32_t* order;
  uint32_t* offsets;  // [n + 1] (may be NULL)
};

// A bucket beyond the LDS: stable 8-bit digit passes through global memory, NT keys at a time.
template <int NT>
__device__ __forceinline__ void ss_local_global(const SsLocalArgs& a, uint32_t b0, uint32_t len, uint32_t kmin, int bits,
                                             uint32_t sum_before, uint32_t* s_count, uint32_t* s_start,
                                             uint32_t* s_w) {
  constexpr int kWaves = NT / kWave;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const uint64_t lt = lanemask_lt(lane);
  const uint32_t *k1 = a.key + b0, *v1 = a.val + b0, *c1 = a.cnt ? a.cnt + b0 : nullptr;
  for (int p = 0; p < (bits + 7) / 8; ++p) {
    uint32_t* k2 = (p & 1 ? a.key2 : a.key1) + b0;
    uint32_t* v2 = (p & 1 ? a.val2 : a.val1) + b0;
    uint32_t* c2 = (p & 1 ? a.cnt2 : a.cnt1) + b0;
    __syncthreads();
    if (tid < 256) s_start[tid] = 0u;
    __syncthreads();
    for (uint32_t i = tid; i < len; i += NT) atomicAdd(&s_start[((k1[i] - kmin) >> (8 * p)) & 255u], 1u);
    __syncthreads();
    uint32_t all;
    const uint32_t ex = block_excl_scan<NT>(tid < 256 ? s_start[tid] : 0u, s_w, all);
    if (tid < 256) s_start[tid] = ex;  // (own entry only: read above by this thread)
    for (uint32_t i0 = 0; i0 < len; i0 += NT) {
      for (int k = tid; k < kWaves * 256; k += NT) s_count[k] = 0u;
      __syncthreads();
      const uint32_t i = i0 + tid;
      const bool valid = i < len;
      const uint32_t k = valid ? k1[i] : kmin, d = ((k - kmin) >> (8 * p)) & 255u;
      const uint64_t peers = match_bits<8>(d, valid);
      const uint32_t before = static_cast<uint32_t>(__popcll(peers & lt));
      if (valid && before == 0u) s_count[wave * 256 + d] = static_cast<uint32_t>(__popcll(peers));
      __syncthreads();
      uint32_t acc = 0;
      if (tid < 256) {
        for (int w = 0; w < kWaves; ++w) {
          const uint32_t c = s_count[w * 256 + tid];
          s_count[w * 256 + tid] = acc;
          acc += c;
        }
      }
      __syncthreads();
      if (valid) {
        const uint32_t q = s_start[d] + s_count[wave * 256 + d] + before;
        k2[q] = k;
        v2[q] = v1[i];
        if (c1) c2[q] = c1[i];
      }
      __syncthreads();
      if (tid < 256) s_start[tid] += acc;
    }
    k1 = k2;
    v1 = v2;
    if (c1) c1 = c2;
  }
  __syncthreads();
  uint32_t run = sum_before;
  for (uint32_t i0 = 0; i0 < len; i0 += NT) {
    const uint32_t i = i0 + tid;
    if (i < len) a.order[b0 + i] = v1[i];
    if (a.offsets) {
      uint32_t all;
      const uint32_t ex = block_excl_scan<NT>(i < len ? c1[i] : 0u, s_w, all);
      if (i < len) a.offsets[b0 + i] = run + ex;
      run += all;
    }
  }
  if (a.offsets && b0 + len == a.n && tid == 0) a.offsets[a.n] = run;
}

// A workgroup per bucket of at most CAP keys in LDS. The keys equal to the bucket's largest (the
// culled Gaussians) keep their order behind the others; the others are spread over CAP / 2 bins
// by interpolation between their smallest and largest, and each is ranked among the keys of its
// bin by (key, position): about two bins per key, no ranking rounds. Where one bin holds more than
// kSsHeavy keys (few distinct depths), 8-bit digit passes in LDS sort the bucket instead.
constexpr uint32_t kSsHeavy = 48;

template <int NT, int CAP>
__global__ __launch_bounds__(NT) void ss_local_kernel(SsLocalArgs a) {
  constexpr int kWaves = NT / kWave;
  constexpr int R = CAP / NT;  // keys per thread
  constexpr int NB = CAP / 2;
  constexpr int BPT = NB / NT;  // consecutive bins per thread
  static_assert(NB >= kWaves * 256 / 2 && NB >= R * kWaves, "the bins' words also hold the digit counters");
  __shared__ uint32_t s_key[CAP];
  __shared__ uint32_t s_alt[CAP];  // the second key buffer of the digit passes; then the counts
  __shared__ uint16_t s_pos[CAP], s_pos2[CAP];
  __shared__ uint32_t s_bin[(NB > kWaves * 256 ? NB : kWaves * 256) + 1];
  __shared__ uint32_t s_start[256];
  __shared__ uint32_t s_w[kWaves];
  __shared__ uint32_t s_top;  // number of keys equal to the largest
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const auto hi = [](uint32_t x, uint32_t y) { return max(x, y); };
  const uint32_t b0 = a.starts ? a.starts[blockIdx.x] : 0u;
  const uint32_t len = (a.starts ? a.starts[blockIdx.x + 1] : a.n) - b0;
  const uint32_t* key = a.key + b0;
  const uint32_t* val = a.val ? a.val + b0 : nullptr;
  const uint32_t* cnt = a.cnt ? a.cnt + b0 : nullptr;
  uint32_t sum_before = 0;
  if (a.offsets && a.starts) {
    uint32_t s = 0;
    for (uint32_t k = tid; k < blockIdx.x; k += NT) s += a.sums[k];
    sum_before = block_fold<NT>(s, s_w, [](uint32_t x, uint32_t y) { return x + y; });
  }
  uint32_t kmin = 0xffffffffu, kmax = 0u;
  if (len > static_cast<uint32_t>(CAP)) {  // (uniform)
    for (uint32_t i = tid; i < len; i += NT) {
      const uint32_t k = key[i];
      kmin = min(kmin, k);
      kmax = max(kmax, k);
    }
    block_min_max<NT>(kmin, kmax, s_w, s_start);
    ss_local_global<NT>(a, b0, len, kmin, kmax != kmin ? 32 - __clz(static_cast<int>(kmax - kmin)) : 0, sum_before,
                        s_bin, s_start, s_w);
    return;
  }
  const int used = static_cast<int>((len + NT - 1) / NT);  // rounds with keys
  // key r of the thread is the bucket's r NT + tid
  uint32_t k_[R], v_[R], c_[R];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    if (r >= used) break;  // (uniform)
    const uint32_t i = static_cast<uint32_t>(r * NT + tid);
    k_[r] = 0u;
    if (i < len) {
      k_[r] = key[i];
      v_[r] = val ? val[i] : i;
      c_[r] = cnt ? cnt[i] : 0u;
      kmin = min(kmin, k_[r]);
      kmax = max(kmax, k_[r]);
    }
  }
  block_min_max<NT>(kmin, kmax, s_w, s_start);
  const uint64_t lt = lanemask_lt(lane);
  // the keys equal to the largest, in order: counts per (r, wavefront), scanned by one wavefront
  uint32_t kmax2 = kmin;
  uint32_t p_[R];  // position in the bucket's order
#pragma unroll
  for (int r = 0; r < R; ++r) {
    if (r >= used) break;  // (uniform)
    const bool ok = static_cast<uint32_t>(r * NT + tid) < len;
    const bool top = ok && k_[r] == kmax;
    const uint64_t m = __ballot(top ? 1 : 0);
    p_[r] = static_cast<uint32_t>(__popcll(m & lt));
    if (lane == 0) s_bin[r * kWaves + wave] = static_cast<uint32_t>(__popcll(m));
    if (ok && !top) kmax2 = max(kmax2, k_[r]);
  }
  kmax2 = block_fold<NT>(kmax2, s_w, hi);
  if (wave == 0) {
    uint32_t run = 0;
    for (int k0 = 0; k0 < used * kWaves; k0 += 64) {
      const uint32_t v = k0 + lane < used * kWaves ? s_bin[k0 + lane] : 0u;
      uint32_t total;
      const uint32_t ex = wave_excl_scan(v, lane, total);
      if (k0 + lane < used * kWaves) s_start[k0 + lane] = run + ex;
      run += total;
    }
    if (lane == 0) s_top = run;  // (not to s_w: block_fold's readers may still be at it)
  }
  __syncthreads();
  const uint32_t n_top = s_top, n_low = len - n_top;
#pragma unroll
  for (int r = 0; r < R; ++r) {
    if (r >= used) break;  // (uniform)
    p_[r] += n_low + s_start[r * kWaves + wave];  // (right for the largest keys)
  }
  const uint32_t range = kmax2 - kmin;
  const float scale = static_cast<float>(NB) / (static_cast<float>(range) + 1.0f);
  for (int k = tid; k <= NB; k += NT) s_bin[k] = 0u;
  __syncthreads();
  uint32_t most = 0;
  uint32_t bin[R], rank[R];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    if (r >= used) break;  // (uniform)
    bin[r] = 0;
    rank[r] = 0;
    if (static_cast<uint32_t>(r * NT + tid) < len && k_[r] != kmax) {
      bin[r] = min(static_cast<uint32_t>(static_cast<float>(k_[r] - kmin) * scale), static_cast<uint32_t>(NB - 1));
      rank[r] = atomicAdd(&s_bin[bin[r]], 1u);
      most = max(most, rank[r]);
    }
  }
  if (block_fold<NT>(most, s_w, hi) < kSsHeavy) {  // (uniform)
    {
      uint32_t c[BPT], sum = 0;
#pragma unroll
      for (int e = 0; e < BPT; ++e) {
        c[e] = s_bin[tid * BPT + e];
        sum += c[e];
      }
      uint32_t all;
      uint32_t run = block_excl_scan<NT>(sum, s_w, all);
#pragma unroll
      for (int e = 0; e < BPT; ++e) {
        s_bin[tid * BPT + e] = run;
        run += c[e];
      }
      if (tid == NT - 1) s_bin[NB] = all;
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < R; ++r) {
      if (r >= used) break;  // (uniform)
      const uint32_t i = static_cast<uint32_t>(r * NT + tid);
      if (i < len && k_[r] != kmax) {
        const uint32_t q = s_bin[bin[r]] + rank[r];
        s_key[q] = k_[r];
        s_pos[q] = static_cast<uint16_t>(i);
      }
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < R; ++r) {
      if (r >= used) break;  // (uniform)
      const uint32_t i = static_cast<uint32_t>(r * NT + tid);
      if (i < len && k_[r] != kmax) {
        const uint32_t q0 = s_bin[bin[r]], q1 = s_bin[bin[r] + 1];
        uint32_t p = q0;
        if (q1 - q0 > 1) {
          for (uint32_t q = q0; q < q1; ++q) {
            const uint32_t k = s_key[q];
            p += (k < k_[r] || (k == k_[r] && s_pos[q] < i)) ? 1u : 0u;
          }
        }
        p_[r] = p;
      }
    }
  } else {
    // digit passes: a wavefront owns 64 rounds consecutive keys
    const int bits = range ? 32 - __clz(static_cast<int>(kmax - kmin)) : 32 - __clz(static_cast<int>(kmax - kmin) | 1);
    const int rounds = static_cast<int>((len + NT - 1) / NT);
    const uint32_t wbase = static_cast<uint32_t>(wave * kWave * rounds + lane);
    uint32_t *kc = s_key, *kn = s_alt;
    uint16_t *pc = s_pos, *pn = s_pos2;
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const uint32_t i = static_cast<uint32_t>(r * NT + tid);
      if (i < len) {
        kc[i] = k_[r];
        pc[i] = static_cast<uint16_t>(i);
      }
    }
    for (int p = 0; p < (bits + 7) / 8; ++p) {
      __syncthreads();
      for (int k = tid; k < kWaves * 256; k += NT) s_bin[k] = 0u;
      __syncthreads();
      uint32_t dk[R], dr[R];
#pragma unroll
      for (int r = 0; r < R; ++r) {
        if (r >= rounds) break;  // (uniform)
        const uint32_t i = wbase + r * kWave;
        const bool valid = i < len;
        dk[r] = valid ? kc[i] : kmin;
        const uint32_t d = ((dk[r] - kmin) >> (8 * p)) & 255u;
        const uint64_t peers = match_bits<8>(d, valid);
        dr[r] = valid ? s_bin[wave * 256 + d] + static_cast<uint32_t>(__popcll(peers & lt)) : 0u;
        wave_sync();
        if (valid && (peers & lt) == 0ull) s_bin[wave * 256 + d] += static_cast<uint32_t>(__popcll(peers));
        wave_sync();
      }
      __syncthreads();
      uint32_t acc = 0;
      if (tid < 256) {
#pragma unroll
        for (int w = 0; w < kWaves; ++w) {
          const uint32_t c = s_bin[w * 256 + tid];
          s_bin[w * 256 + tid] = acc;
          acc += c;
        }
      }
      uint32_t all;
      const uint32_t ex = block_excl_scan<NT>(acc, s_w, all);
      if (tid < 256) s_start[tid] = ex;
      __syncthreads();
#pragma unroll
      for (int r = 0; r < R; ++r) {
        if (r >= rounds) break;
        const uint32_t i = wbase + r * kWave;
        if (i < len) {
          const uint32_t d = ((dk[r] - kmin) >> (8 * p)) & 255u;
          const uint32_t q = s_start[d] + s_bin[wave * 256 + d] + dr[r];
          kn[q] = dk[r];
          pn[q] = pc[i];
        }
      }
      uint32_t* t = kc; kc = kn; kn = t;
      uint16_t* u = pc; pc = pn; pn = u;
    }
    __syncthreads();
    // back to the threads' own keys: the position of each in the order
    for (uint32_t q = tid; q < len; q += NT) kn[pc[q]] = q;
    __syncthreads();
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const uint32_t i = static_cast<uint32_t>(r * NT + tid);
      if (i < len) p_[r] = kn[i];
    }
    __syncthreads();
  }
#pragma unroll
  for (int r = 0; r < R; ++r) {
    if (r >= used) break;  // (uniform)
    if (static_cast<uint32_t>(r * NT + tid) < len) {
      a.order[b0 + p_[r]] = v_[r];
      s_alt[p_[r]] = c_[r];
    }
  }
  if (a.offsets) {
    __syncthreads();
    uint32_t sum = 0, c[R];
#pragma unroll
    for (int e = 0; e < R; ++e) {
      const uint32_t i = static_cast<uint32_t>(tid * R + e);
      c[e] = i < len ? s_alt[i] : 0u;
      sum += c[e];
    }
    uint32_t all;
    uint32_t run = sum_before + block_excl_scan<NT>(sum, s_w, all);
#pragma unroll
    for (int e = 0; e < R; ++e) {
      const uint32_t i = static_cast<uint32_t>(tid * R + e);
      if (i < len) s_alt[i] = run;
      run += c[e];
    }
    __syncthreads();
    for (uint32_t i = tid; i < len; i += NT) a.offsets[b0 + i] = s_alt[i];
    if (b0 + len == a.n && tid == 0) a.offsets[a.n] = sum_before + all;
  }
}

// ---- host side ------------------------------------------------------------------------
struct SsLayout {
  size_t spl, bucket_of, hist, totals, starts, sums, arr[9], end;
  int B, n_tiles;
};

static bool ss_takes(int64_t n) { return n > 0 && n <= kSsMaxKeys; }

static SsLayout ss_layout(int64_t n) {
  SsLayout L{};
  if (!ss_takes(n) || n <= kSsSmall) return L;
  L.B = static_cast<int>((n + ss_mean(n) - 1) / ss_mean(n));
  L.n_tiles = static_cast<int>((n + kSsTile - 1) / kSsTile);
  const auto up = [](size_t v) { return (v + 255) & ~static_cast<size_t>(255); };
  size_t o = 0;
  L.spl = o; o += up(static_cast<size_t>(L.B) * 8);
  L.bucket_of = o; o += up(static_cast<size_t>(n) * 2);
  L.hist = o; o += up(static_cast<size_t>(L.B) * L.n_tiles * 4);
  L.totals = o; o += up(static_cast<size_t>(L.B) * 4);
  L.starts = o; o += up((static_cast<size_t>(L.B) + 1) * 4);
  L.sums = o; o += up(static_cast<size_t>(L.B) * 4);
  for (size_t& s : L.arr) {
    s = o;
    o += up(static_cast<size_t>(n) * 4);
  }
  L.end = o;
  return L;
}

// order [n] = the stable argsort of keys; offsets (may be NULL) [n + 1] = the exclusive scan of
// counts[order[j]].
static void sample_sort(const uint32_t* keys, const uint32_t* counts, int64_t n, uint32_t* order, uint32_t* offsets,
                        char* ws, hipStream_t st) {
  SsLocalArgs a{};
  a.n = static_cast<uint32_t>(n);
  a.order = order;
  a.offsets = offsets;
  if (!offsets) counts = nullptr;
  if (n <= kSsSmall) {
    a.key = keys;
    a.cnt = counts;
    if (n <= 2048) hipLaunchKernelGGL((ss_local_kernel<512, 2048>), dim3(1), dim3(512), 0, st, a);
    else hipLaunchKernelGGL((ss_local_kernel<1024, kSsSmall>), dim3(1), dim3(1024), 0, st, a);
    return;
  }
  const SsLayout L = ss_layout(n);
  const uint32_t S = static_cast<uint32_t>(L.B) * kSsOver;
  const auto at = [ws](size_t o) { return reinterpret_cast<uint32_t*>(ws + o); };
  uint64_t* spl = reinterpret_cast<uint64_t*>(ws + L.spl);
  uint16_t* bucket_of = reinterpret_cast<uint16_t*>(ws + L.bucket_of);
  uint32_t *key = at(L.arr[0]), *val = at(L.arr[1]), *cnt = at(L.arr[2]);
  a.key = key;
  a.val = val;
  a.cnt = counts ? cnt : nullptr;
  a.key1 = at(L.arr[3]);
  a.val1 = at(L.arr[4]);
  a.cnt1 = at(L.arr[5]);
  a.key2 = at(L.arr[6]);
  a.val2 = at(L.arr[7]);
  a.cnt2 = at(L.arr[8]);
  a.starts = at(L.starts);
  a.sums = at(L.sums);
  hipLaunchKernelGGL(ss_splitters_kernel, dim3((S + 31) / 32), dim3(1024), 0, st, keys,
                     (static_cast<uint64_t>(n) << 32) / S, S, spl, at(L.sums));
  hipLaunchKernelGGL(ss_count_kernel, dim3(L.n_tiles), dim3(kSsThreads), 0, st, keys, a.n, spl, L.B, bucket_of,
                     at(L.hist), L.n_tiles);
  hipLaunchKernelGGL(rs_rowscan_kernel, dim3(L.B), dim3(kScanThreads), 0, st, at(L.hist), L.n_tiles, at(L.totals));
  hipLaunchKernelGGL(ss_scatter_kernel, dim3(L.n_tiles), dim3(kSsThreads), 0, st, keys, bucket_of, counts, a.n, L.B,
                     at(L.hist), L.n_tiles, at(L.totals), key, val, cnt, at(L.starts), at(L.sums));
  if (ss_mean(n) == 1024)
    hipLaunchKernelGGL((ss_local_kernel<512, 4096>), dim3(L.B), dim3(512), 0, st, a);
  else
    hipLaunchKernelGGL((ss_local_kernel<1024, 8192>), dim3(L.B), dim3(1024), 0, st, a);
}

}  // namespace gs

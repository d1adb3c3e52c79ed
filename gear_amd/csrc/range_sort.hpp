// One-launch stable sort of a batch of keys, gfx950: between the ranking sort (at most
// radix::kRankMax keys) and the radix sort.
//
// A radix sort of 20 000 keys is bound by its launches: two per digit of 8 bits, 8 us a digit of
// which the work is a fraction.  Here every workgroup works alone.  It reads ALL keys (held in
// registers, so one pass over L2), finds the two keys between which its share of the sorted batch
// lies -- a histogram of the keys over 4096 equal ranges, refined where one range holds too many
// -- collects the keys in between in LDS, ranks them there by counting, and writes them out.
// Nothing passes between workgroups: no scratch, no second launch, and the cuts come out the same
// everywhere because they depend on the keys alone.  The price is that 256 workgroups each count
// the whole batch (an LDS atomic a key), which is why larger batches keep the radix sort.
// us a call, back to back, here / radix sort (63-bit keys need 40 registers a thread more):
//     keys     20 bits       63 bits     63 bits, in order
//      4097   7.6 / 20.7    9.7 / 55.1      5.4 / 55.5
//     20000  12.1 / 21.6   15.9 / 58.0      8.4 / 58.2
//     32768  16.4 / 22.2   26.9 / 59.2     16.7 / 59.6
// At 40 000 keys of 20 bits the two meet (64 registers of keys a thread spill: 64 us).
#pragma once
#include "radix_sort.hpp"

namespace gearhip {
namespace ranges {
namespace {  // every translation unit gets its own copy of the kernels

constexpr int kThreads = 1024;
constexpr int kWaves = kThreads / kWave;
constexpr int kGroups = 256;           // workgroups: one a CU, whatever the batch
constexpr int kBinBits = 12;
constexpr int kBins = 1 << kBinBits;
constexpr int kPerThread = kBins / kThreads;
static_assert(kPerThread == 4, "a thread's bins are one 16-byte word");
constexpr int kCap = 1024;             // keys ranked at once in LDS
constexpr int kTol = 512;              // a cut may leave its place by so many keys
constexpr int kMax = 32 * kThreads;    // largest batch: the keys of a thread stay in registers
static_assert(kMax / kGroups + kTol <= kCap, "a share without repeated keys fits in LDS");

// the keys collected in LDS, in the order (key, position)
template <typename C>
struct List;
template <>
struct List<uint32_t> {
  __align__(16) uint64_t e[kCap];
  __device__ __forceinline__ void put(int i, uint32_t key, int pos) {
    e[i] = ((uint64_t)key << 32) | (uint32_t)pos;
  }
  __device__ __forceinline__ int pos(int i) const { return (int)(uint32_t)e[i]; }
  struct Mine {
    uint64_t e;
  };
  __device__ __forceinline__ Mine mine(int i) const { return Mine{e[i]}; }
  __device__ __forceinline__ bool before(int i, const Mine &m) const { return e[i] < m.e; }
};
template <>
struct List<uint64_t> {
  __align__(16) uint64_t k[kCap];
  int p[kCap];
  __device__ __forceinline__ void put(int i, uint64_t key, int pos) {
    k[i] = key;
    p[i] = pos;
  }
  __device__ __forceinline__ int pos(int i) const { return p[i]; }
  struct Mine {
    uint64_t k;
    int p;
  };
  __device__ __forceinline__ Mine mine(int i) const { return Mine{k[i], p[i]}; }
  __device__ __forceinline__ bool before(int i, const Mine &m) const {
    return k[i] < m.k || (k[i] == m.k && p[i] < m.p);
  }
};

__device__ __forceinline__ uint32_t lane_before(uint32_t k) { return (uint32_t)wave_shift_up1((int)k); }
__device__ __forceinline__ uint64_t lane_before(uint64_t k) {
  return (uint64_t)wave_shift_up1((int64_t)k);
}
__device__ __forceinline__ uint32_t last_lane(uint32_t k) {
  return (uint32_t)wave_read_lane((int)k, kWave - 1);
}
__device__ __forceinline__ uint64_t last_lane(uint64_t k) {
  return (uint64_t)wave_read_lane((int64_t)k, kWave - 1);
}

// A place between two keys: the keys below lo are the `below` smallest ones.
template <typename C>
struct Cut {
  C lo;
  uint32_t below, count;  // count: keys in the range [lo, lo + (1 << s))
  int s;
};

template <typename C>
struct Smem {
  __align__(16) uint32_t hist[kBins + 1];  // counts, then exclusive sums; the last entry is the total
  uint32_t wsum[kWaves];
  C wmin[kWaves], wmax[kWaves], wfirst[kWaves];
  Cut<C> cut[2];
  int sorted, found, n;
  List<C> list;
  uint32_t rank[kCap];
};

// smallest shift that leaves fewer than kBins ranges of a stretch of last + 1 keys
__device__ __forceinline__ int shift_of(uint32_t last) {
  const int bits = 32 - __builtin_clz(last | 1u);
  return bits > kBinBits ? bits - kBinBits : 0;
}
__device__ __forceinline__ int shift_of(uint64_t last) {
  const int bits = 64 - __builtin_clzll(last | 1ull);
  return bits > kBinBits ? bits - kBinBits : 0;
}

// A thread's elements: wave w holds the elements [w, w + 1) * per * 64, round i of them the elements
// 64 * i + lane; so elements in order are (wave, round, lane) in order.  The keys (less the smallest
// one) are in registers for the passes that every batch takes; the passes that only batches with
// crowded keys take ask the source again (each(), a rolled loop: unrolled ones made the kernel spill).
template <typename C, int kRounds, typename Src>
struct Keys {
  const Src &src;
  C k[kRounds];
  C mn;
  int first;   // element of round 0
  int per;     // rounds in use
  int rounds;  // of them, this thread's
  // the rounds again, unknown to the compiler: comparisons with it are not kept from pass to pass
  __device__ __forceinline__ int own_rounds() const {
    int r = rounds;
    asm volatile("" : "+v"(r));
    return r;
  }
  __device__ __forceinline__ int element(int i) const { return first + i * kWave; }
  // f(round is this thread's, element, key): as often in every lane of a wave
  template <typename F>
  __device__ __forceinline__ void each(const F &f) const {
#pragma unroll 1
    for (int i = 0; i < per; ++i) {
      const bool ok = i < rounds;
      f(ok, element(i), ok ? (C)(src.key(element(i)) - mn) : (C)0);
    }
  }
  template <typename F>
  __device__ __forceinline__ void each_held(const F &f) const {
    const int r = own_rounds();
#pragma unroll
    for (int i = 0; i < kRounds; ++i)
      if (i < r) f(element(i), k[i]);
  }
};

template <typename C>
__device__ __forceinline__ void clear_counts(Smem<C> &sm) {
  reinterpret_cast<u32x4 *>(sm.hist)[threadIdx.x] = u32x4{0, 0, 0, 0};
}

// The counts of this thread's bins, and the sum of those before them.
template <typename C>
__device__ __forceinline__ uint32_t sum_counts(Smem<C> &sm, u32x4 &c) {
  const int tid = threadIdx.x;
  __syncthreads();
  c = reinterpret_cast<const u32x4 *>(sm.hist)[tid];
  const int total = (int)(c[0] + c[1] + c[2] + c[3]);
  const int inc = wave_inclusive_sum(total);
  if ((tid & (kWave - 1)) == kWave - 1) sm.wsum[tid / kWave] = (uint32_t)inc;
  __syncthreads();
  uint32_t run = (uint32_t)(inc - total);
#pragma unroll
  for (int w = 0; w < kWaves; ++w) run += w < tid / kWave ? sm.wsum[w] : 0u;
  return run;
}

// The sums for the keys in [lo, last] over ranges of 1 << s keys.
template <typename C, typename K>
__device__ __forceinline__ void count_ranges(Smem<C> &sm, const K &keys, C lo, C last, int s) {
  clear_counts(sm);
  __syncthreads();
  keys.each([&](bool ok, int, C k) {
    if (ok && k >= lo && k <= last) atomicAdd(&sm.hist[(uint32_t)((k - lo) >> s) & (kBins - 1)], 1u);
  });
  u32x4 c;
  const uint32_t run = sum_counts(sm, c);
  reinterpret_cast<u32x4 *>(sm.hist)[threadIdx.x] =
      u32x4{run, run + c[0], run + c[0] + c[1], run + c[0] + c[1] + c[2]};
  if (threadIdx.x == kThreads - 1) sm.hist[kBins] = run + c[0] + c[1] + c[2] + c[3];
  __syncthreads();
}

// The range f with hist[f] <= at < hist[f + 1]; at is below the total, so there is exactly one.
template <typename C>
__device__ __forceinline__ int range_at(Smem<C> &sm, uint32_t at) {
  const int b0 = (int)threadIdx.x * kPerThread;
#pragma unroll
  for (int i = 0; i < kPerThread; ++i)
    if (sm.hist[b0 + i] <= at && at < sm.hist[b0 + i + 1]) sm.found = b0 + i;
  __syncthreads();
  const int f = sm.found;
  __syncthreads();
  return f;
}

// Moves a cut up towards its place while the range that holds it has too many keys.
template <typename C, typename K>
__device__ __forceinline__ void refine(Smem<C> &sm, const K &keys, Cut<C> &cut, uint32_t at) {
  while (cut.count > (uint32_t)kTol && cut.s > 0) {
    const int s = cut.s > kBinBits ? cut.s - kBinBits : 0;
    count_ranges(sm, keys, cut.lo, (C)(cut.lo + (((C)1 << cut.s) - 1)), s);
    const int f = range_at(sm, at - cut.below);
    cut.lo += (C)((C)f << s);
    cut.count = sm.hist[f + 1] - sm.hist[f];
    cut.below += sm.hist[f];
    cut.s = s;
    __syncthreads();
  }
}

// The keys in [lo, last], at most kCap, ranked and handed to emit.list as the places from `base`.
template <bool kHeld, typename C, typename K, typename Emit>
__device__ __forceinline__ void emit_window(Smem<C> &sm, const K &keys, C lo, C last, uint32_t base,
                                            uint32_t room, const Emit &emit) {
  const int tid = threadIdx.x;
  if (tid == 0) sm.n = 0;
  sm.rank[tid] = 0;
  __syncthreads();
  auto collect = [&](int j, C k) {
    if ((C)(k - lo) <= (C)(last - lo)) {
      const int slot = atomicAdd(&sm.n, 1);
      if (slot < kCap) sm.list.put(slot, k, j);
    }
  };
  if constexpr (kHeld)
    keys.each_held(collect);
  else
    keys.each([&](bool ok, int j, C k) {
      if (ok) collect(j, k);
    });
  __syncthreads();
  const int limit = room < (uint32_t)kCap ? (int)room : kCap, n = sm.n < limit ? sm.n : limit;
  // thread = (part of the list, key of it)
  const int padded = (n + kWave - 1) & ~(kWave - 1);
  const int parts = padded > 0 ? kThreads / padded : 0;
  const int part = padded > 0 ? tid / padded : 0, e = tid - part * padded;
  if (part < parts && e < n) {
    const auto mine = sm.list.mine(e);
    const int b0 = part * n / parts, b1 = (part + 1) * n / parts;
    uint32_t c = 0;
#pragma unroll 8
    for (int b = b0; b < b1; ++b) c += sm.list.before(b, mine) ? 1u : 0u;
    if (parts > 1)
      atomicAdd(&sm.rank[e], c);
    else
      sm.rank[e] = c;
  }
  __syncthreads();
  emit.list(sm.list, sm.rank, n, base);
  __syncthreads();
}

// All elements whose key is v, in their order, as the places from `base`.
template <typename C, typename K, typename Emit>
__device__ __forceinline__ void emit_equal(Smem<C> &sm, const K &keys, C v, uint32_t base,
                                           uint32_t room, const Emit &emit) {
  const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
  uint32_t mine = 0;
  keys.each([&](bool ok, int j, C k) {
    const bool hit = ok && k == v;
    mine += (uint32_t)__popcll(wave_ballot(hit));
    if (hit) sm.found = j;  // any of them: equal keys find the same
  });
  if (lane == 0) sm.wsum[wave] = mine;
  __syncthreads();
  const auto what = emit.find(sm.found);
  const uint32_t end = base + room;
  for (int w = 0; w < wave; ++w) base += sm.wsum[w];
  keys.each([&](bool ok, int j, C k) {
    const bool hit = ok && k == v;
    const uint64_t hits = wave_ballot(hit);
    const uint32_t place = base + (uint32_t)__popcll(hits & ((1ull << lane) - 1));
    if (hit && place < end) emit.put(place, j, what);
    base += (uint32_t)__popcll(hits);
  });
  __syncthreads();
}

// Src: C key(j), the key of element j.  Emit: list(list, rank, n, base) stores n collected elements
// at base + rank, by all threads; find(j) + put(place, j, found) store one of many equal keys.
// kLook: a batch that is in order already is passed on without a histogram.
template <typename C, int kRounds, bool kLook, typename Src, typename Emit>
__global__ __launch_bounds__(kThreads) void range_sort_kernel(Src src, int num, Emit emit) {
  __shared__ Smem<C> sm;
  const int tid = threadIdx.x, lane = tid & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int per = (num + kThreads - 1) / kThreads;
  const int first = wave * per * kWave + lane;
  const int left_here = num - first + kWave - 1;
  Keys<C, kRounds, Src> keys{src, {}, (C)0, first, per,
                             left_here <= 0 ? 0 : left_here / kWave < per ? left_here / kWave : per};
  const int own0 = (int)((int64_t)blockIdx.x * num / kGroups);
  const int own1 = (int)((int64_t)(blockIdx.x + 1) * num / kGroups);
  src.begin();
  C mn = ~(C)0, mx = 0;
#pragma unroll
  for (int i = 0; i < kRounds; ++i) {  // (no branch between the loads; places past the end: the last)
    const int j = keys.element(i);
    keys.k[i] = 0;
    if (i < per) keys.k[i] = src.key(j < num ? j : num - 1);
  }
  clear_counts(sm);  // (before the first barrier)
  bool ordered = true;
  C edge = 0;  // the last key of the round before
  {
    const int r = keys.own_rounds();
#pragma unroll
    for (int i = 0; i < kRounds; ++i) {
      const C k = keys.k[i];
      if (kLook) {
        C before = lane_before(k);
        if (lane == 0) before = edge;
        ordered = ordered && (i >= r || before <= k);
        edge = last_lane(k);
      }
      if (i < r) {
        mn = k < mn ? k : mn;
        mx = k > mx ? k : mx;
      }
    }
  }
#pragma unroll
  for (int off = kWave / 2; off > 0; off >>= 1) {
    const C a = __shfl_xor(mn, off, kWave), b = __shfl_xor(mx, off, kWave);
    mn = a < mn ? a : mn;
    mx = b > mx ? b : mx;
  }
  if (tid == 0) sm.sorted = 1;
  if (lane == 0) {
    sm.wmin[wave] = mn;
    sm.wmax[wave] = mx;
  }
  __syncthreads();
  if (kLook) {
    // inside the waves, and from wave to wave (a wave without elements has mn above mx)
    if (wave_ballot(!ordered) != 0 && lane == 0) sm.sorted = 0;
    if (tid > 0 && tid < kWaves && sm.wmin[tid] <= sm.wmax[tid] && sm.wmax[tid - 1] > sm.wmin[tid])
      sm.sorted = 0;
  }
#pragma unroll
  for (int w = 0; w < kWaves; ++w) {
    mn = sm.wmin[w] < mn ? sm.wmin[w] : mn;
    mx = sm.wmax[w] > mx ? sm.wmax[w] : mx;
  }
  __syncthreads();
  if (kLook && sm.sorted) {
    for (int j = own0 + tid; j < own1; j += kThreads) emit.put((uint32_t)j, j, emit.find(j));
    return;
  }
  keys.mn = mn;
#pragma unroll
  for (int i = 0; i < kRounds; ++i) keys.k[i] -= mn;
  const C all = mx - mn;
  const int s = shift_of(all);
  keys.each_held([&](int, C k) { atomicAdd(&sm.hist[(uint32_t)(k >> s)], 1u); });
  {
    u32x4 c;
    uint32_t run = sum_counts(sm, c);
#pragma unroll
    for (int i = 0; i < kPerThread; ++i) {
      const C lo = (C)((C)(tid * kPerThread + i) << s);
      if (run <= (uint32_t)own0 && (uint32_t)own0 < run + c[i]) sm.cut[0] = Cut<C>{lo, run, c[i], s};
      if (run <= (uint32_t)own1 && (uint32_t)own1 < run + c[i]) sm.cut[1] = Cut<C>{lo, run, c[i], s};
      run += c[i];
    }
  }
  __syncthreads();
  Cut<C> from = sm.cut[0], to = {0, (uint32_t)num, 0, 0};
  if (own1 < num) to = sm.cut[1];
  refine(sm, keys, from, (uint32_t)own0);
  refine(sm, keys, to, (uint32_t)own1);
  uint32_t left = to.below - from.below, base = from.below;
  // (a share is empty where its neighbour's cut is the same; the limits here and below keep every
  // place inside the batch and every loop finite even if the source changes while it is read)
  if (to.below <= from.below || to.below > (uint32_t)num) return;
  const C last = own1 < num ? (C)(to.lo - 1) : all;
  C cur = from.lo;
  if (left <= (uint32_t)kCap) {
    emit_window<true>(sm, keys, cur, last, base, left, emit);
    return;
  }
  // keys that are repeated many times are among the share
  while (left > 0) {
    C end = last;
    int t = shift_of((C)(end - cur));
    for (;;) {
      count_ranges(sm, keys, cur, end, t);
      const uint32_t total = sm.hist[kBins];
      if (total == 0) return;
      // the ranges before f together fit in LDS, the one at f no more
      const int f = total <= (uint32_t)kCap ? kBins : range_at(sm, (uint32_t)kCap);
      const uint32_t fit = sm.hist[f], next = f < kBins ? sm.hist[f + 1] : 0;
      __syncthreads();
      if (fit > 0) {
        const C stop = (C)(cur + ((C)f << t));
        emit_window<false>(sm, keys, cur, f < kBins ? (C)(stop - 1) : end, base, left, emit);
        cur = stop;  // (not used again after the last range)
        base += fit;
        left -= fit < left ? fit : left;
        break;
      }
      cur = (C)(cur + ((C)f << t));
      if (t == 0) {  // one key
        emit_equal(sm, keys, cur, base, left, emit);
        base += next;
        left -= next < left ? next : left;
        cur = (C)(cur + 1);  // (past the largest key only when nothing is left)
        break;
      }
      const C stop = (C)(cur + (((C)1 << t) - 1));
      end = stop < end ? stop : end;
      t = t > kBinBits ? t - kBinBits : 0;
    }
  }
}

inline bool fits(int64_t num) { return num > 0 && num <= kMax; }

template <typename C, bool kLook, typename Src, typename Emit>
int sort(const Src &src, int64_t num, const Emit &emit, hipStream_t st) {
  const dim3 grid(kGroups), block(kThreads);
  // (rounds beyond the batch's own cost registers and a skipped branch each)
  const int n = (int)num, per = (int)ceil_div64(num, kThreads);
  if (per <= 8)
    range_sort_kernel<C, 8, kLook, Src, Emit><<<grid, block, 0, st>>>(src, n, emit);
  else if (per <= 20)
    range_sort_kernel<C, 20, kLook, Src, Emit><<<grid, block, 0, st>>>(src, n, emit);
  else if (per <= 32)
    range_sort_kernel<C, 32, kLook, Src, Emit><<<grid, block, 0, st>>>(src, n, emit);
  else
    return GEAR_HIP_ERANGE;
  GEARHIP_RETURN_IF_LAUNCH_FAILED();
  return 0;
}

// Whether what a launch of many workgroups writes could be read by another of its workgroups.
inline bool overlap(const void *a, int64_t a_bytes, const void *b, int64_t b_bytes) {
  const uintptr_t x = reinterpret_cast<uintptr_t>(a), y = reinterpret_cast<uintptr_t>(b);
  return a && b && x < y + (uintptr_t)b_bytes && y < x + (uintptr_t)a_bytes;
}

}  // namespace
}  // namespace ranges
}  // namespace gearhip

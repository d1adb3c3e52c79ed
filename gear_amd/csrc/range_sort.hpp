// One-launch stable sort of a batch of keys, gfx950: between the ranking sort (at most
// radix::kRankMax keys) and the radix sort.
//
// A radix sort of 20 000 keys is bound by its launches: two per digit of 8 bits, 8 us a digit of
// which the work is a fraction.  Here every workgroup works alone.  It reads ALL keys (held in
// registers, so one pass over L2), finds the two keys between which its share of the sorted batch
// lies -- a histogram of the keys over 4096 equal ranges, refined where one range holds too many
// -- collects the keys in between in LDS, ranks them there by counting, and writes them out.  Keys
// that are repeated more often than a list holds are not ranked: their order is that of the batch.
// Nothing passes between workgroups: no scratch, no second launch, and the cuts come out the same
// everywhere because they depend on the keys alone.  The price is that 256 workgroups each count
// the whole batch (an LDS atomic a key), which is why larger batches keep the radix sort.
// us a call, back to back, here / radix sort (63-bit keys need 40 registers a thread more):
//     keys     20 bits      63 bits      63 bits, in order
//      4097   7.7 / 20.0    9.1 / 53.6      5.4 / 55.5
//     20000  12.4 / 21.4   15.3 / 57.5      8.4 / 58.2
//     32768  16.6 / 22.0   24.2 / 59.1     13.5 / 59.6
// A batch of a few keys, each many times over, takes longer, for the passes that find its runs: 19.6 /
// 21.9 for 20000 keys of two values, 26.3 / 22.4 for 32768 of them, 38.5 / 59.8 where they are 63 bits
// wide, 37.0 / 59.4 for 5000 values and one far away.
// At 40 000 keys of 20 bits the two meet (64 registers of keys a thread spill: 64 us); for 63-bit keys the
// registers are the limit: 32 rounds fill all 128 of them.
#pragma once
#include <type_traits>

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
constexpr int kBanks = 64;
// copies of the counts, where many lanes count in the same bank: 32768 keys of two values take 26.4 us,
// 29.2 with four, 42.3 with one
constexpr int kCopies = 8;
constexpr int kCopy = kBins + 4;       // (in different banks)
constexpr int kCap = 1024;             // keys ranked at once in LDS
// A cut may leave its place by so many keys: more are slow to rank, fewer take another pass (64 values,
// 24576 keys / 32768 keys: 23.5 / 27.4 us; with 384 27.3 / 27.4, with 512 23.4 / 33.3).
constexpr int kTol = 448;
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
  __align__(16) uint32_t hist[kCopies * kCopy];
  uint32_t wsum[kWaves];
  C wmin[kWaves], wmax[kWaves], wfirst[kWaves];
  Cut<C> cut[2];
  int sorted, crowd, n;
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
// one) stay in registers for all passes: reading them again is a round trip to L2 a round.
template <typename C, int kRounds>
struct Keys {
  static constexpr int kHeld = kRounds;
  C k[kRounds];
  int first;   // element of round 0
  int rounds;  // this thread's
  // the rounds again, unknown to the compiler: comparisons with it are not kept from pass to pass
  __device__ __forceinline__ int own_rounds() const {
    int r = rounds;
    asm volatile("" : "+v"(r));
    return r;
  }
  __device__ __forceinline__ int element(int i) const { return first + i * kWave; }
};

template <typename C>
__device__ __forceinline__ void wave_min_max(C &mn, C &mx) {
#pragma unroll
  for (int off = kWave / 2; off > 0; off >>= 1) {
    const C a = __shfl_xor(mn, off, kWave), b = __shfl_xor(mx, off, kWave);
    mn = a < mn ? a : mn;
    mx = b > mx ? b : mx;
  }
}

// A thread's four bins of every copy.
template <typename C>
__device__ __forceinline__ void clear_counts(Smem<C> &sm, int first, int copies) {
  for (int i = first; i < copies; ++i)
    reinterpret_cast<u32x4 *>(sm.hist + i * kCopy)[threadIdx.x] = u32x4{0, 0, 0, 0};
}

// The keys (kAll), or those in [lo, last], counted over ranges of 1 << s keys.  Lanes that count in the
// same bank are served one after the other; in a crowd neighbours count in different copies.
template <bool kAll, typename C, typename K>
__device__ __forceinline__ void count_ranges(Smem<C> &sm, const K &keys, C lo, C last, int s, bool crowd) {
  const int r = keys.own_rounds();
  uint32_t *hist = sm.hist + (crowd ? (int)(threadIdx.x & (kCopies - 1)) * kCopy : 0);
  const C width = (C)(last - lo);
#pragma unroll
  for (int i = 0; i < K::kHeld; ++i) {
    const C at = kAll ? keys.k[i] : (C)(keys.k[i] - lo);
    if (i < r && (kAll || at <= width)) atomicAdd(&hist[(uint32_t)(at >> s)], 1u);
  }
}

// The counts of this thread's bins, and the sum of those before them; the counts are clear again after
// the next barrier.
template <typename C>
__device__ __forceinline__ uint32_t sum_counts(Smem<C> &sm, bool crowd, u32x4 &c) {
  const int tid = threadIdx.x;
  __syncthreads();
  c = reinterpret_cast<const u32x4 *>(sm.hist)[tid];
  if (__builtin_expect(crowd, 0))
    for (int i = 1; i < kCopies; ++i) c += reinterpret_cast<const u32x4 *>(sm.hist + i * kCopy)[tid];
  clear_counts(sm, 0, crowd ? kCopies : 1);
  const int total = (int)(c[0] + c[1] + c[2] + c[3]);
  const int inc = wave_inclusive_sum(total);
  if ((tid & (kWave - 1)) == kWave - 1) sm.wsum[tid / kWave] = (uint32_t)inc;
  __syncthreads();
  uint32_t run = (uint32_t)(inc - total);
#pragma unroll
  for (int w = 0; w < kWaves; ++w) run += w < tid / kWave ? sm.wsum[w] : 0u;
  return run;
}

// The smallest and the largest key in [lo, last].
template <typename C, typename K>
__device__ __forceinline__ void tighten(Smem<C> &sm, const K &keys, C &lo, C &last) {
  const int r = keys.own_rounds();
  const C width = (C)(last - lo);
  C mn = width, mx = 0;
#pragma unroll
  for (int i = 0; i < K::kHeld; ++i) {
    const C at = (C)(keys.k[i] - lo);
    const bool takes = i < r && at <= width;
    mn = takes && at < mn ? at : mn;
    mx = takes && at > mx ? at : mx;
  }
  wave_min_max(mn, mx);
  if ((threadIdx.x & (kWave - 1)) == 0) {
    sm.wmin[threadIdx.x / kWave] = mn;
    sm.wmax[threadIdx.x / kWave] = mx;
  }
  __syncthreads();
#pragma unroll
  for (int w = 0; w < kWaves; ++w) {
    mn = sm.wmin[w] < mn ? sm.wmin[w] : mn;
    mx = sm.wmax[w] > mx ? sm.wmax[w] : mx;
  }
  last = (C)(lo + mx);
  lo = (C)(lo + mn);
  __syncthreads();
}

template <typename C>
__device__ __forceinline__ bool too_many(const Cut<C> &c) { return c.count > (uint32_t)kTol && c.s > 0; }

// The cuts for the places at0 and at1 (num: none) of a batch with keys up to `all`: each moves towards
// its place until the range that holds it has few keys, or is one key.  A range that holds both is
// counted once.  When it begins the first copy of the counts is clear; crowd: neighbours' keys share
// ranges, all copies are clear.
template <typename C, typename K>
__device__ __forceinline__ void find_cuts(Smem<C> &sm, const K &keys, C all, uint32_t num, uint32_t at0,
                                          uint32_t at1, bool crowd, Cut<C> &from, Cut<C> &to) {
  from = Cut<C>{0, 0u, num, 0};
  to = at1 < num ? from : Cut<C>{0, num, 0u, 0};
  if (all == 0) return;
  const bool split = at1 < num;
  auto place = [&](C lo, int s, bool crowd, bool mine0, bool mine1) {
    u32x4 c;
    uint32_t run = sum_counts(sm, crowd, c);
#pragma unroll
    for (int i = 0; i < kPerThread; ++i) {
      const C low = (C)(lo + ((C)(threadIdx.x * kPerThread + i) << s));
      const uint32_t p0 = at0 - from.below, p1 = at1 - to.below;
      if (mine0 && run <= p0 && p0 < run + c[i]) sm.cut[0] = Cut<C>{low, from.below + run, c[i], s};
      if (mine1 && run <= p1 && p1 < run + c[i]) sm.cut[1] = Cut<C>{low, to.below + run, c[i], s};
      run += c[i];
    }
    __syncthreads();
    if (mine0) from = sm.cut[0];
    if (mine1) to = sm.cut[1];
  };
  count_ranges<true>(sm, keys, (C)0, all, shift_of(all), crowd);
  place(0, shift_of(all), crowd, true, split);
  bool clear = crowd;
  for (;;) {
    const bool mine0 = too_many(from);
    const bool mine1 = too_many(to) && (!mine0 || (to.lo == from.lo && to.s == from.s));
    if (__builtin_expect(!mine0 && !mine1, 1)) return;
    C lo = mine0 ? from.lo : to.lo;
    C last = (C)(lo + (((C)1 << (mine0 ? from.s : to.s)) - 1));
    const bool many = (mine0 ? from.count : to.count) > num / 8;
    if (many || (mine0 ? from.s : to.s) > 2 * kBinBits) {
      // a few keys in a corner of the range, or one: a pass instead of one a level
      tighten(sm, keys, lo, last);
      if (lo == last) {
        if (mine0) from.lo = lo, from.s = 0;
        if (mine1) to.lo = lo, to.s = 0;
        continue;
      }
    }
    if (many && !clear) {
      clear_counts(sm, 1, kCopies);
      __syncthreads();
      clear = true;
    }
    const int s = shift_of((C)(last - lo));
    count_ranges<false>(sm, keys, lo, last, s, many);
    place(lo, s, many, mine0, mine1);
  }
}

// The keys in [lo, last], at most kCap, ranked and handed to emit.list as the places from `base`.
template <typename C, typename K, typename Emit>
__device__ __forceinline__ void emit_window(Smem<C> &sm, const K &keys, C lo, C last, uint32_t base,
                                            uint32_t room, const Emit &emit) {
  const int tid = threadIdx.x;
  if (tid == 0) sm.n = 0;
  sm.rank[tid] = 0;
  __syncthreads();
  const int r = keys.own_rounds();
#pragma unroll
  for (int i = 0; i < K::kHeld; ++i)
    if (i < r && (C)(keys.k[i] - lo) <= (C)(last - lo)) {
      const int slot = atomicAdd(&sm.n, 1);
      if (slot < kCap) sm.list.put(slot, keys.k[i], keys.element(i));
    }
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
}

// The places [p0, p1) of the sorted batch, at most kCap, which hold elements of the one key v whose
// elements, in their order, take the places from `start`.
template <typename C, typename K, typename Emit>
__device__ __forceinline__ void emit_equal(Smem<C> &sm, const K &keys, C v, uint32_t start, uint32_t p0,
                                           uint32_t p1, const Emit &emit) {
  if (p0 >= p1) return;
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x / kWave);
  const int r = keys.own_rounds();
  uint32_t mine = 0;
#pragma unroll
  for (int i = 0; i < K::kHeld; ++i) mine += (uint32_t)__popcll(wave_ballot(i < r && keys.k[i] == v));
  if (lane == 0) sm.wsum[wave] = mine;
  sm.rank[threadIdx.x] = 0;
  __syncthreads();
  uint32_t place = start;  // of the wave's next element
  for (int w = 0; w < wave; ++w) place += sm.wsum[w];
  if (place < p1 && place + mine > p0) {
#pragma unroll
    for (int i = 0; i < K::kHeld; ++i) {
      const bool hit = i < r && keys.k[i] == v;
      const uint64_t hits = wave_ballot(hit);
      const uint32_t at = place + (uint32_t)__popcll(hits & ((1ull << lane) - 1));
      if (hit && at >= p0 && at < p1 && at - p0 < (uint32_t)kCap) sm.rank[at - p0] = (uint32_t)keys.element(i);
      place += (uint32_t)__popcll(hits);
    }
  }
  __syncthreads();
  emit.equal(sm.rank, (int)(p1 - p0 < (uint32_t)kCap ? p1 - p0 : kCap), p0);
}

// Src: C key(j), the key of element j.  Emit, by all threads: list(list, rank, n, base) stores n
// collected elements at base + rank; equal(at, n, base) stores the elements at[0..n) of one key at
// base, base + 1, ...  kLook: a batch that is in order already is passed on without a histogram
// (Emit::put(place, j) stores element j).
// Src::kGuarded: src.done() says, to all threads alike, that there is nothing to sort.
template <typename Src, typename = void>
struct Guarded : std::false_type {};
template <typename Src>
struct Guarded<Src, std::enable_if_t<Src::kGuarded>> : std::true_type {};

template <typename C, int kRounds, bool kLook, typename Src, typename Emit>
__global__ __launch_bounds__(kThreads) void range_sort_kernel(Src src, int num, Emit emit) {
  __shared__ Smem<C> sm;
  if constexpr (Guarded<Src>::value) {
    if (src.done()) return;
  }
  const int tid = threadIdx.x, lane = tid & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int per = (num + kThreads - 1) / kThreads;
  const int first = wave * per * kWave + lane;
  const int left_here = num - first + kWave - 1;
  Keys<C, kRounds> keys{
      {}, first, left_here <= 0 ? 0 : left_here / kWave < per ? left_here / kWave : per};
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
  clear_counts(sm, 0, 1);  // (before the first barrier)
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
  wave_min_max(mn, mx);
  if (tid == 0) {
    sm.sorted = 1;
    sm.crowd = 0;
  }
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
  // neighbours of a wave's first round that count in one bank of LDS tell whether many keys do
  const C all = mx - mn;
  const C before = (C)(lane_before(keys.k[0]) - mn);
  const bool shared = 0 < keys.own_rounds() && lane > 0 &&
                      (((before ^ (C)(keys.k[0] - mn)) >> shift_of(all)) & (kBanks - 1)) == 0;
  if (__popcll(wave_ballot(shared)) >= kWave / 8 && lane == 0) sm.crowd = 1;
  __syncthreads();
  if constexpr (kLook) {
    if (sm.sorted) {
      for (int j = own0 + tid; j < own1; j += kThreads) emit.put((uint32_t)j, j);
      return;
    }
  }
  const bool crowd = sm.crowd != 0;
  if (__builtin_expect(crowd, 0)) {
    clear_counts(sm, 1, kCopies);
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < kRounds; ++i) keys.k[i] -= mn;
  Cut<C> from, to;
  find_cuts(sm, keys, all, (uint32_t)num, (uint32_t)own0, (uint32_t)own1, crowd, from, to);
  // A cut lies before the first key of its range, unless the range is one key that is repeated too
  // often: then it lies at its place among the equal ones.  So a share has at most
  // num / kGroups + kTol keys that have to be ranked, and the workgroups that a run of equal keys
  // covers take a part of it each.  (The limits here and above keep every place inside the batch and
  // every loop finite even if the source changes while it is read.)
  if (to.below > (uint32_t)num) return;
  const bool from_run = from.count > (uint32_t)kTol, to_run = to.count > (uint32_t)kTol;
  const uint32_t base = from.below + (from_run ? from.count : 0u);
  if (base < to.below)
    emit_window(sm, keys, from_run ? (C)(from.lo + 1) : from.lo, own1 < num ? (C)(to.lo - 1) : all, base,
                to.below - base, emit);
  if (__builtin_expect(!from_run && !to_run, 1)) return;
#pragma unroll 1
  for (int end = 0; end < 2; ++end) {
    if (!(end == 0 ? from_run : to_run && !(from_run && from.lo == to.lo))) continue;
    __syncthreads();  // (the lists and sums of the part before)
    const C key = end == 0 ? from.lo : to.lo;
    const uint32_t p0 = end == 0 ? from.below : to.below, p1 = p0 + (end == 0 ? from.count : to.count);
    emit_equal(sm, keys, key, p0, p0 > (uint32_t)own0 ? p0 : (uint32_t)own0,
               p1 < (uint32_t)own1 ? p1 : (uint32_t)own1, emit);
  }
}

inline bool fits(int64_t num) { return num > 0 && num <= kMax; }

// Up to how many keys this sort is the faster one: a radix sort of one digit takes 9 us, of two 14.4.
inline int64_t worth(int key_bits) { return key_bits <= 8 ? 0 : key_bits <= 16 ? 20480 : kMax; }

template <typename C, bool kLook, typename Src, typename Emit>
int sort(const Src &src, int64_t num, const Emit &emit, hipStream_t st) {
  const dim3 grid(kGroups), block(kThreads);
  // Rounds beyond the batch's own cost registers and a skipped branch each: 8192 keys take 8.5 / 10.1 /
  // 11.8 us in kernels of 8 / 20 / 32 rounds (20 bits; 10.0 / 12.2 / 17.3 with 63), 20 000 keys 12.3 / 14.1
  // in 20 / 32 (15.3 / 20.4).  A batch just beyond a step pays for it: 20 480 / 20 481 keys 12.4 / 14.4 us.
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

// Batched upper_bound of draws in an inclusive prefix array (+ importance weights), and the
// one-call batch sampler (search + ranking sort + split into window arguments), gfx950.
//
// The search is latency-bound (a chain of dependent loads), so the lanes of a group look for one
// draw together and a batch spreads over many CUs.
#include <math.h>

#include <atomic>
#include <type_traits>

#include "philox.hpp"
#include "range_sort.hpp"

namespace gearhip {
namespace {

constexpr int kBlock = 256;

// ---- search -------------------------------------------------------------------------------------
// First index with p[i] > t (n when there is none), worked out by kLanes neighbouring lanes
// together.  What a batch of draws waits for is the chain of dependent loads, so a step cuts the
// remaining range [lo, hi) into kLanes parts with one probe per lane: part j ends before
// lo + (range * (j + 1) >> log2(kLanes)), and the answer lies behind as many parts as have a last
// entry <= t -- counted, so that a larger t never gives a smaller answer, whatever the array holds.
// More lanes make the chain shorter (log_kLanes(n) steps) and the loads more: kLanes cache lines a
// draw and step, and a CU asks for one a clock.  us per batch of draws in a prefix of 1e6 / 1e7
// entries (back to back; a launch alone takes 3.1), by lanes; 1 = seven probes by one lane:
//     draws        1              8             16             32
//       512   4.5 / 5.9     3.7 / 4.5      3.3 / 3.9      3.3 / 3.6
//      4096   4.9 / 6.2     4.1 / 4.9      3.7 / 4.6      3.9 / 5.3
//     16384   5.3 / 8.9     4.9 / 7.9      6.2 / 9.9      7.6 / 13
//     65536  10.1 / 20.6   11.2 / 21.2    16.3 / 28.5    22.7 / 41
// hence 16 lanes up to 4096 draws, 8 up to 32768, 1 beyond; with importance weights, which each lane of
// a group works out, 8 up to 24576 (32768 draws: 12.6 / 18.6 with 8, 11.2 / 17.1 with 1).  With one lane
// a draw, workgroups of one wave spread fewer draws over more CUs (40000: 7.9 / 14.5, 8.9 / 15.2 in
// workgroups of four), and are too many for a hundred thousand (15.8 / 32.2, 17.0 / 29.5; with weights
// 22.1 / 39.0, 22.2 / 35.2; the two meet at 65536).
struct SearchShape {
  int lanes, threads;
};
constexpr int64_t kMost16 = 4096, kMost8 = 32768, kMost8Weights = 24576, kMostWaves = 49152;
inline SearchShape search_shape(int64_t num, bool weights) {
  if (num <= kMost16) return {16, kBlock};
  if (num <= (weights ? kMost8Weights : kMost8)) return {8, kBlock};
  return {1, num <= kMostWaves ? kWave : kBlock};
}

template <int kLanes>
struct Probe {
  int64_t lo, range;
  static constexpr int kShift = kLanes == 16 ? 4 : 3;
  static_assert(1 << kShift == kLanes, "a power of two");
  __device__ __forceinline__ int64_t parts_end(int j) const { return (range * (j + 1)) >> kShift; }
  // the entry that lane `sub` of the group looks at (empty parts at the front look at the first one)
  template <typename T>
  __device__ __forceinline__ T load(const T *__restrict__ p, int sub) const {
    const int64_t e = parts_end(sub);
    return p[lo + (e > 0 ? e - 1 : 0)];
  }
  template <typename T>
  __device__ __forceinline__ void narrow(T v, T t, int sub) {
    const uint64_t le = wave_ballot(parts_end(sub) == 0 || v <= t);
    const int first_lane = (int)(threadIdx.x & (kWave - 1)) & ~(kLanes - 1);
    const int c = __popc((uint32_t)(le >> first_lane) & ((1u << kLanes) - 1u));
    const int64_t begin = c > 0 ? parts_end(c - 1) : 0;
    range = c < kLanes ? parts_end(c) - 1 - begin : 0;
    lo += begin;
  }
};

// One lane alone: seven independent probes per step, and the last step reads the whole remaining
// stretch at once.
template <typename T>
__device__ __forceinline__ int64_t lane_search(const T *__restrict__ p, int64_t n, T t) {
  constexpr int kArity = 8, kArityShift = 3;
  int64_t lo = 0, hi = n;  // the answer lies in [lo, hi]
  while (hi - lo >= kArity) {
    const int64_t step = (hi - lo) >> kArityShift;
    T v[kArity - 1];
#pragma unroll
    for (int j = 0; j < kArity - 1; ++j) v[j] = p[lo + step * (j + 1) - 1];
    int c = 0;
#pragma unroll
    for (int j = 0; j < kArity - 1; ++j) c += (v[j] <= t) ? 1 : 0;
    const int64_t base = lo + step * c;
    if (c < kArity - 1) hi = lo + step * (c + 1) - 1;
    lo = base;
  }
  T v[kArity - 1];
#pragma unroll
  for (int j = 0; j < kArity - 1; ++j) v[j] = lo + j < hi ? p[lo + j] : t;
  int c = 0;
#pragma unroll
  for (int j = 0; j < kArity - 1; ++j) c += (lo + j < hi && v[j] <= t) ? 1 : 0;
  return lo + c;
}

// The whole search, by kLanes lanes, for a target that depends on the array's last entry, the
// total (it is what the group's last lane looks at in the first step).
template <int kLanes, typename T, typename Target>
__device__ __forceinline__ int64_t group_search(const T *__restrict__ p, int64_t n, int sub,
                                                const Target &target) {
  int64_t at;
  if constexpr (kLanes == 1) {
    at = lane_search(p, n, target(p[n - 1]));
  } else {
    Probe<kLanes> s{0, n};
    T v = s.load(p, sub);
    const T t = target(__shfl(v, kLanes - 1, kLanes));
    s.narrow(v, t, sub);
    while (s.range > 0) {
      v = s.load(p, sub);
      s.narrow(v, t, sub);
    }
    at = s.lo;
  }
  return at < n ? at : n - 1;
}

// The targets of a batch of draws, and keys of the same order to rank the draws by.
// fp64 prefix: fp32 draws, in [0, 1) (unit) or targets already.  A target that is not a number -- the
// draw or the total is none, or infinite where the other is 0 -- compares with nothing and finds
// entry 0, so it has the lowest key.
struct PhiloxU {  // draws that are worked out where they are asked for
  Philox rng;
  __device__ __forceinline__ float operator[](int64_t j) const { return rng.uniform((uint64_t)j); }
};
template <typename U>
struct DrawF64From {
  typedef double type;
  typedef uint32_t key_type;
  const double *prefix;
  int64_t n;
  U u;
  int unit;
  __device__ __forceinline__ double target(int64_t j, double total) const {
    const float f = u[j];
    return unit ? (double)f * total : (double)f;
  }
  __device__ __forceinline__ uint32_t key(int64_t j, double total) const {
    const float f = u[j];
    const uint32_t b = __float_as_uint(f);
    uint32_t k = b ^ ((uint32_t)((int32_t)b >> 31) | 0x80000000u);
    if (unit && total < 0.0) k = ~k;  // (priorities are not negative; the order holds all the same)
    // (no number where the target is none; as one multiplication in fp32)
    const float t = f * (unit && (total == 0.0 || __builtin_isinf(total)) ? (float)total : 1.0f);
    return t == t ? k : 0u;
  }
};
typedef DrawF64From<const float *> DrawF64;
// int64 prefix (a sampler over lengths): doubles in [0, 1) (unit) or int64 targets.
struct DrawI64 {
  typedef int64_t type;
  typedef int64_t key_type;
  const int64_t *prefix;
  int64_t n;
  const void *u;
  int unit;
  __device__ __forceinline__ int64_t target(int64_t j, int64_t total) const {
    return unit ? (int64_t)floor(static_cast<const double *>(u)[j] * (double)total)
                : static_cast<const int64_t *>(u)[j];
  }
  __device__ __forceinline__ int64_t key(int64_t j, int64_t total) const { return target(j, total); }
};

template <int kLanes, int kThreads, typename Draw>
__global__ __launch_bounds__(kThreads) void search_kernel(Draw draw, int64_t num,
                                                          int64_t *__restrict__ idx_out) {
  const int64_t j = ((int64_t)blockIdx.x * kThreads + threadIdx.x) / kLanes;
  const int sub = threadIdx.x & (kLanes - 1);
  if (j >= num) return;
  const int64_t i = group_search<kLanes>(
      draw.prefix, draw.n, sub, [&](typename Draw::type total) { return draw.target(j, total); });
  if (sub == 0) idx_out[j] = i;
}

// The same with the raw importance weights (N * p / total) ** -beta of the found entries and their
// maximum per workgroup.
template <int kLanes, int kThreads>
__global__ __launch_bounds__(kThreads) void search_weights_kernel(
    DrawF64 draw, int64_t num, int64_t *__restrict__ idx_out, const float *__restrict__ priorities,
    double beta, double *__restrict__ wraw, double *__restrict__ block_max) {
  __shared__ double wmax[kThreads / kWave];
  const int64_t j = ((int64_t)blockIdx.x * kThreads + threadIdx.x) / kLanes;
  const int sub = threadIdx.x & (kLanes - 1);
  double w = 0.0;
  if (j < num) {
    double total = 0.0;
    const int64_t i = group_search<kLanes>(draw.prefix, draw.n, sub, [&](double last) {
      total = last;
      return draw.target(j, last);
    });
    w = pow((double)draw.n * (double)priorities[i] / total, -beta);
    if (sub == 0) {
      idx_out[j] = i;
      wraw[j] = w;
    }
  }
  // (weights are positive, lanes without a draw hold 0)
  for (int off = 32; off >= kLanes; off >>= 1) w = fmax(w, __shfl_xor(w, off, kWave));
  if (kThreads == kWave) {
    if (threadIdx.x == 0) block_max[blockIdx.x] = w;
    return;
  }
  if ((threadIdx.x & (kWave - 1)) == 0) wmax[threadIdx.x / kWave] = w;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int i = 1; i < kThreads / kWave; ++i) w = fmax(w, wmax[i]);
    block_max[blockIdx.x] = w;
  }
}

__global__ __launch_bounds__(kBlock) void normalise_kernel(const double *__restrict__ wraw,
                                                           const double *__restrict__ block_max,
                                                           int nblocks, int64_t num,
                                                           float *__restrict__ out) {
  __shared__ double wmax[kBlock / kWave];
  double m = 0.0;
  for (int i = threadIdx.x; i < nblocks; i += kBlock) m = fmax(m, block_max[i]);
  for (int off = 32; off > 0; off >>= 1) m = fmax(m, __shfl_xor(m, off, kWave));
  if ((threadIdx.x & 63) == 0) wmax[threadIdx.x >> 6] = m;
  __syncthreads();
  m = fmax(fmax(wmax[0], wmax[1]), fmax(wmax[2], wmax[3]));
  const int64_t j = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (j < num) out[j] = (float)(wraw[j] / m);
}

__global__ __launch_bounds__(kBlock) void split_sorted_kernel(const int64_t *__restrict__ flat,
                                                              int64_t num, int64_t T,
                                                              int64_t modulo,
                                                              int64_t *__restrict__ idxs,
                                                              int64_t *__restrict__ tss,
                                                              int64_t *__restrict__ lens) {
  const int64_t j = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (j >= num) return;
  int64_t f = flat[j];
  if (modulo > 0) f %= modulo;
  const int64_t traj = f / T;
  const int64_t ts = f - traj * T;
  idxs[j] = traj;
  tss[j] = ts;
  if (lens) lens[j] = ts + 1;
}

// What happens with the entry that takes place r of the sorted batch.  resolve() needs the entry
// only and runs while the place is still being worked out; store() writes the results.

// Split of a flat step index into window arguments.
struct Split {
  int64_t *sorted_out;
  int64_t T, modulo;
  int64_t *idxs, *tss, *lens;
  struct Resolved {
    int64_t flat, traj, ts;
  };
  __device__ __forceinline__ Resolved resolve(int64_t f) const {
    Resolved r{f, 0, 0};
    if (T > 0) {
      if (f <= 0xffffffffll && T <= 0xffffffffll && modulo <= 0xffffffffll) {
        uint32_t f32 = (uint32_t)f;  // 32-bit division is a fraction of the 64-bit one
        if (modulo > 0) f32 %= (uint32_t)modulo;
        const uint32_t q = f32 / (uint32_t)T;
        r.traj = q;
        r.ts = f32 - q * (uint32_t)T;
      } else {
        if (modulo > 0) f %= modulo;
        r.traj = f / T;
        r.ts = f - r.traj * T;
      }
    }
    return r;
  }
  __device__ __forceinline__ void store(int64_t rank, const Resolved &r) const {
    if (sorted_out) sorted_out[rank] = r.flat;
    if (T > 0) {
      idxs[rank] = r.traj;
      tss[rank] = r.ts;
      if (lens) lens[rank] = r.ts + 1;
    }
  }
};

// What the loader does with a sorted batch of positions before it can gather
// (gear/loader/offline_loader.py:168-177 and the samplers' concat_indices[draws],
// gear/sampler/global_sampler.py:131,172,196), for the entry at sorted place r with position p:
//     sampled[r] = index_table ? index_table[p] : p        the batch's global trajectory index
//     local[r]   = sampled[r] - index_offset               its index in this shard's table
//     lens[r]    = lengths_table[local[r]]                  its recorded length (0 outside the table)
struct Lookup {
  const int64_t *index_table;
  int64_t index_n, index_offset;
  const int64_t *lengths_table;
  int64_t lengths_n;
  int64_t *sampled, *local, *lens;
  // a window of `window` steps inside the entry's recorded length, placed by a uniform:
  // starts[r] = floor(start_u[r] * (length - window + 1)), 0 for a length below the window
  const double *start_u = nullptr;
  int64_t window = 0;
  int64_t *starts = nullptr;
  struct Resolved {
    int64_t global, len;
  };
  __device__ __forceinline__ Resolved resolve(int64_t p) const {
    Resolved v;
    v.global = p;
    if (index_table) v.global = (p >= 0 && p < index_n) ? index_table[p] : 0;
    const int64_t l = v.global - index_offset;
    v.len = (lengths_table && l >= 0 && l < lengths_n) ? lengths_table[l] : 0;
    return v;
  }
  __device__ __forceinline__ void store(int64_t r, const Resolved &v) const {
    if (sampled) sampled[r] = v.global;
    if (local) local[r] = v.global - index_offset;
    if (lens) lens[r] = v.len;
    if (starts) {
      const int64_t room = v.len - (window - 1);
      starts[r] = room > 0 ? (int64_t)floor(start_u[r] * (double)room) : 0;
    }
  }
};

// ---- a sorted batch in one launch ---------------------------------------------------------------
// Draws are searched and put in order at the same time: a larger target never finds a smaller
// entry, so the place of a draw in the sorted batch is the place of its TARGET among the targets,
// and nothing has to be found before the sort can begin.  A workgroup takes kPlaced draws.  Its
// first waves search them (kLanes lanes each) and do the look-ups; the other waves keep the keys
// of ALL draws of the batch (at most kRankMax) in LDS and count the smaller ones, and the equal
// ones at smaller positions (the place after a stable sort); both meet in LDS at the end.
// 2048 draws in 1e6 / 1e7 entries: 4.3 / 4.9 us (a launch alone 3.1), where a search launch and a
// ranking launch took 6.8 + 6.3 in the same stream; 8 or 32 lanes a draw: 4.6 / 5.2, 4.4 / 5.0.
// At 4096 draws (5.1 us) the counting -- kPlaced * num compares a CU -- begins to be what bounds it.
constexpr int kPlaced = 16;
constexpr int kPlaceThreads = 1024;
constexpr int kPlaceWaves = kPlaceThreads / kWave;

template <typename K>
struct PlaceSmem {
  __align__(16) K keys[radix::kRankMax];
  uint32_t part[kPlaceWaves][kPlaced];
};

// Fills sm.keys, padded to a multiple of kPlaced with the largest key there is: it lies behind
// every draw and no key exceeds it, so it is never counted.
template <typename K, typename Key>
__device__ __forceinline__ void fill_keys(PlaceSmem<K> &sm, int num, const Key &key) {
  constexpr K kTop = (K)-1 > (K)0 ? ~(K)0 : (K)(((uint64_t)1 << (8 * sizeof(K) - 1)) - 1);
  const int padded = (num + kPlaced - 1) & ~(kPlaced - 1);
  for (int j = threadIdx.x; j < padded; j += kPlaceThreads) sm.keys[j] = j < num ? key(j) : kTop;
}

// The share of rank wave `rw` (of `rws`) in the places of the workgroup's draws: lane = (slice of
// the keys, draw).  A chunk of kPlaced keys lies before, behind or exactly at the workgroup's own.
template <typename K>
__device__ __forceinline__ void count_before(PlaceSmem<K> &sm, int num, int rw, int rws) {
  typedef K K4 __attribute__((ext_vector_type(4)));
  const int lane = threadIdx.x & (kWave - 1);
  const int d = lane & (kPlaced - 1), slice = lane / kPlaced;
  const int own = blockIdx.x, chunks = (num + kPlaced - 1) / kPlaced;
  const K mine = sm.keys[own * kPlaced + d];
  const K4 *keys4 = reinterpret_cast<const K4 *>(sm.keys) + slice;
  uint32_t c = 0;
  int ch = rw;
#pragma unroll 4
  for (; ch < own; ch += rws) {
    const K4 k = keys4[ch * (kPlaced / 4)];
    c += (k[0] <= mine) + (k[1] <= mine) + (k[2] <= mine) + (k[3] <= mine);
  }
  if (ch == own) {
    const K4 k = keys4[ch * (kPlaced / 4)];
#pragma unroll
    for (int i = 0; i < 4; ++i) c += k[i] < mine || (k[i] == mine && slice * 4 + i < d);
    ch += rws;
  }
#pragma unroll 4
  for (; ch < chunks; ch += rws) {
    const K4 k = keys4[ch * (kPlaced / 4)];
    c += (k[0] < mine) + (k[1] < mine) + (k[2] < mine) + (k[3] < mine);
  }
  c += (uint32_t)__shfl_xor((int)c, kPlaced, kWave);
  c += (uint32_t)__shfl_xor((int)c, 2 * kPlaced, kWave);
  if (lane < kPlaced) sm.part[rw][d] = c;
}

template <int kLanes, typename Draw, typename Emit>
__global__ __launch_bounds__(kPlaceThreads) void place_draws_kernel(Draw draw, int num, Emit emit) {
  typedef typename Draw::type T;
  constexpr int kFindWaves = kPlaced * kLanes / kWave;
  constexpr int kRankWaves = kPlaceWaves - kFindWaves;
  static_assert(kRankWaves > 0, "somebody ranks");
  __shared__ PlaceSmem<typename Draw::key_type> sm;
  __shared__ typename Emit::Resolved found[kPlaced];
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int sub = tid & (kLanes - 1), d = tid / kLanes;  // of the search
  // the first probes go out together with the loads of the draws
  Probe<kLanes> s{0, draw.n};
  T v = T(0);
  if (wave < kFindWaves) v = s.load(draw.prefix, sub);
  const T total = draw.prefix[draw.n - 1];
  fill_keys(sm, num, [&](int j) { return draw.key(j, total); });
  if (wave < kFindWaves) {
    const int e = (int)blockIdx.x * kPlaced + d;
    const T t = draw.target(e < num ? e : num - 1, total);
    __syncthreads();
    s.narrow(v, t, sub);
    while (s.range > 0) {
      v = s.load(draw.prefix, sub);
      s.narrow(v, t, sub);
    }
    if (sub == 0) found[d] = emit.resolve(s.lo < draw.n ? s.lo : draw.n - 1);
  } else {
    __syncthreads();
    count_before(sm, num, wave - kFindWaves, kRankWaves);
  }
  __syncthreads();
  if (tid < kPlaced && (int)blockIdx.x * kPlaced + tid < num) {
    uint32_t rank = 0;
#pragma unroll
    for (int w = 0; w < kRankWaves; ++w) rank += sm.part[w][tid];
    emit.store((int64_t)rank, found[tid]);
  }
}

// The same for positions that are given (no search): sorted and looked up.  raw[j]: from memory, or drawn.
struct PhiloxPositions {
  Philox rng;
  uint32_t range;
  __device__ __forceinline__ int64_t operator[](int j) const { return rng.below(range, (uint64_t)j); }
};
template <typename Raw, typename Emit>
__global__ __launch_bounds__(kPlaceThreads) void place_positions_kernel(Raw raw, int num, Emit emit) {
  __shared__ PlaceSmem<int64_t> sm;
  const int tid = threadIdx.x;
  const int e = (int)blockIdx.x * kPlaced + tid;
  const bool mine = tid < kPlaced && e < num;
  typename Emit::Resolved found = {};
  if (mine) found = emit.resolve(raw[e]);
  fill_keys(sm, num, [&](int j) { return raw[j]; });
  __syncthreads();
  count_before(sm, num, __builtin_amdgcn_readfirstlane(tid / kWave), kPlaceWaves);
  __syncthreads();
  if (mine) {
    uint32_t rank = 0;
#pragma unroll
    for (int w = 0; w < kPlaceWaves; ++w) rank += sm.part[w][tid];
    emit.store((int64_t)rank, found);
  }
}

template <typename Draw, typename Emit>
int place_draws(const Draw &draw, int64_t num, const Emit &emit, hipStream_t st) {
  place_draws_kernel<16>
      <<<dim3((unsigned)ceil_div64(num, kPlaced)), dim3(kPlaceThreads), 0, st>>>(draw, (int)num, emit);
  GEARHIP_RETURN_IF_LAUNCH_FAILED();
  return 0;
}
template <typename Raw, typename Emit>
int place_positions(const Raw &raw, int64_t num, const Emit &emit, hipStream_t st) {
  place_positions_kernel<<<dim3((unsigned)ceil_div64(num, kPlaced)), dim3(kPlaceThreads), 0, st>>>(
      raw, (int)num, emit);
  GEARHIP_RETURN_IF_LAUNCH_FAILED();
  return 0;
}

// ---- larger batches: the one-launch sort ----------------------------------------------------------
// The same idea beyond kRankMax draws: the draws are put in order by their keys, and the workgroup
// that places a draw searches it too -- the search, two launches a digit of the radix sort and the
// look-ups are one launch: 20 000 draws in 1e6 entries 14.9 us (27.5 with a launch for the search
// and six for the sort), 20 000 integer draws in 1e5 entries 17.8 (29.5), positions 11.3 (23.9).
inline __device__ uint32_t sort_key(uint32_t k) { return k; }
inline __device__ uint64_t sort_key(int64_t k) { return (uint64_t)k ^ (1ull << 63); }

template <typename Draw>
struct DrawSrc {
  typedef decltype(sort_key(typename Draw::key_type())) key_type;
  Draw draw;
  typename Draw::type total;
  __device__ __forceinline__ void begin() { total = draw.prefix[draw.n - 1]; }
  __device__ __forceinline__ key_type key(int j) const { return sort_key(draw.key(j, total)); }
};

template <typename Draw, typename Emit>
struct DrawEmit {
  Draw draw;
  Emit emit;
  int lanes;  // per draw: the same everywhere, so that a larger target never finds a smaller entry
              // whatever the prefix holds (an ulp less behind a zero priority)
  template <int kLanes>
  __device__ __forceinline__ int64_t search(int j) const {
    return group_search<kLanes>(draw.prefix, draw.n, (int)threadIdx.x & (kLanes - 1),
                                [&](typename Draw::type total) { return draw.target(j, total); });
  }
  // (equal keys find the same entry: one search)
  __device__ __forceinline__ void equal(const uint32_t *at, int n, uint32_t base) const {
    const int j = (int)at[0], e = threadIdx.x;
    const auto r = emit.resolve(lanes == 16 ? search<16>(j) : lanes == 8 ? search<8>(j) : search<1>(j));
    if (e < n) emit.store((int64_t)base + e, r);
  }
  template <int kLanes, typename L>
  __device__ __forceinline__ void list_by(const L &list, const uint32_t *rank, int n,
                                          uint32_t base) const {
    for (int e = (int)threadIdx.x / kLanes; e < n; e += ranges::kThreads / kLanes) {
      const auto r = emit.resolve(search<kLanes>(list.pos(e)));
      if ((threadIdx.x & (kLanes - 1)) == 0) emit.store((int64_t)(base + rank[e]), r);
    }
  }
  template <typename L>
  __device__ __forceinline__ void list(const L &list, const uint32_t *rank, int n,
                                       uint32_t base) const {
    if (lanes == 16)
      list_by<16>(list, rank, n, base);
    else if (lanes == 8)
      list_by<8>(list, rank, n, base);
    else
      list_by<1>(list, rank, n, base);
  }
};

struct PositionSrc {
  const int64_t *raw;
  uint32_t mask;
  __device__ __forceinline__ void begin() {}
  __device__ __forceinline__ uint32_t key(int j) const { return (uint32_t)raw[j] & mask; }
};

struct PositionEmit {
  const int64_t *raw;
  Lookup look;
  template <typename L>
  __device__ __forceinline__ void list(const L &list, const uint32_t *rank, int n,
                                       uint32_t base) const {
    const int e = threadIdx.x;
    if (e < n) look.store((int64_t)(base + rank[e]), look.resolve(raw[list.pos(e)]));
  }
  __device__ __forceinline__ void equal(const uint32_t *at, int n, uint32_t base) const {
    const int e = threadIdx.x;
    if (e < n) look.store((int64_t)base + e, look.resolve(raw[at[e]]));
  }
};

inline bool writes_over(const Split &s, const void *p, int64_t bytes, int64_t num) {
  return ranges::overlap(s.sorted_out, num * 8, p, bytes) ||
         (s.T > 0 && (ranges::overlap(s.idxs, num * 8, p, bytes) ||
                      ranges::overlap(s.tss, num * 8, p, bytes) ||
                      ranges::overlap(s.lens, num * 8, p, bytes)));
}
inline bool writes_over(const Lookup &l, const void *p, int64_t bytes, int64_t num) {
  return ranges::overlap(l.sampled, num * 8, p, bytes) || ranges::overlap(l.local, num * 8, p, bytes) ||
         ranges::overlap(l.lens, num * 8, p, bytes) || ranges::overlap(l.starts, num * 8, p, bytes);
}

// Whether a batch can be searched and stored by one launch: nothing that one workgroup stores is
// still to be read by another.  Outputs on top of the draws or the prefix take separate launches,
// where reading ends before writing begins.
template <typename Draw, typename Emit>
bool apart(const Draw &draw, int64_t num, const Emit &emit) {
  const int64_t u_bytes = num * (sizeof(typename Draw::type) == 8 && sizeof(typename Draw::key_type) == 8 ? 8 : 4);
  return !writes_over(emit, draw.u, u_bytes, num) && !writes_over(emit, draw.prefix, draw.n * 8, num);
}

template <typename Draw, typename Emit>
int sort_draws(const Draw &draw, int64_t num, const Emit &emit, hipStream_t st) {
  typedef DrawSrc<Draw> Src;
  // Lanes a draw: a workgroup searches num / 256 draws, a few more where keys crowd, and 16 lanes each
  // let it search 64 at once.  us a batch in 1e5 / 1e7 entries by lanes:
  //     draws         16             8              1
  //      4097    9.5 /  9.7     9.6 / 10.1    10.0 / 10.6
  //      8192   10.3 / 11.0    10.5 / 11.1    10.6 / 11.3
  //     12288   13.5 / 15.7    12.8 / 13.4    12.9 / 13.8
  //     20000   16.8 / 20.4    15.2 / 17.9    15.1 / 19.2
  //     24576   19.7 / 25.5    18.4 / 23.9    17.5 / 22.2
  //     32768   23.1 / 31.4    20.6 / 28.7    19.3 / 27.5
  const int lanes = num <= 8192 ? 16 : num <= 20480 ? 8 : 1;
  return ranges::sort<typename Src::key_type, false>(
      Src{draw, {}}, num, DrawEmit<Draw, Emit>{draw, emit, lanes}, st);
}

// Draws of a batch that other launches read.
__global__ __launch_bounds__(kBlock) void draw_uniform_kernel(Philox rng, int64_t num, float *__restrict__ out) {
  const int64_t j = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (j < num) out[j] = rng.uniform((uint64_t)j);
}
__global__ __launch_bounds__(kBlock) void draw_positions_kernel(PhiloxPositions raw, int64_t num,
                                                                int64_t *__restrict__ out) {
  const int64_t j = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (j < num) out[j] = raw[(int)j];
}
// Up to so many draws -- all that are placed by one launch -- every workgroup works out the draws of the whole
// batch itself, four a thread at most.  us a batch of uniforms in 1e6 entries / of positions, so and with a
// launch for the draws: 256 3.8 / 2.9 and 5.3 / 4.6, 1024 4.2 / 3.5 and 5.5 / 5.1, 4096 6.4 / 6.3 and 7.0 / 7.1.
constexpr int64_t kDrawnInPlace = radix::kRankMax;

__global__ __launch_bounds__(kBlock) void lookup_kernel(const int64_t *__restrict__ positions,
                                                        int64_t num, Lookup look) {
  const int64_t j = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (j < num) look.store(j, look.resolve(positions[j]));
}

struct SampleWs {
  size_t raw, ktmp, sorted, hist, total;
};
SampleWs sample_ws(int64_t num) {
  SampleWs w;
  const size_t m = align_up((size_t)(num > 0 ? num : 1) * 8, 256);
  w.raw = 0;
  w.ktmp = m;
  w.sorted = 2 * m;
  w.hist = 3 * m;
  w.total = 3 * m + radix::hist_bytes(num);
  return w;
}

int64_t search_blocks(int64_t num, bool weights) {
  const SearchShape s = search_shape(num, weights);
  return ceil_div64(num * s.lanes, s.threads);
}

// calls f(lanes per draw, threads per workgroup), both as std::integral_constant
template <typename F>
void with_search_shape(int64_t num, bool weights, const F &f) {
  const SearchShape s = search_shape(num, weights);
  const std::integral_constant<int, kBlock> block;
  if (s.lanes == 16)
    f(std::integral_constant<int, 16>{}, block);
  else if (s.lanes == 8)
    f(std::integral_constant<int, 8>{}, block);
  else if (s.threads == kWave)
    f(std::integral_constant<int, 1>{}, std::integral_constant<int, kWave>{});
  else
    f(std::integral_constant<int, 1>{}, block);
}
template <typename Draw>
int launch_search(const Draw &draw, int64_t num, int64_t *idx_out, hipStream_t st) {
  const int64_t blocks = search_blocks(num, false);
  if (blocks >= 0x7fffffffll) return GEAR_HIP_ERANGE;
  with_search_shape(num, false, [&](auto lanes, auto threads) {
    constexpr int kThreads = decltype(threads)::value;
    search_kernel<decltype(lanes)::value, kThreads>
        <<<dim3((unsigned)blocks), dim3(kThreads), 0, st>>>(draw, num, idx_out);
  });
  GEARHIP_RETURN_IF_LAUNCH_FAILED();
  return 0;
}

// (More draws may take fewer lanes each and so fewer workgroups: what is asked for is enough for every
// smaller batch as well.)
size_t search_ws_bytes(int64_t num) {
  if (num <= 0) return 256;
  int64_t blocks = search_blocks(num, true);
  for (const int64_t most : {kMost16, kMost8Weights, kMostWaves})
    if (most < num && search_blocks(most, true) > blocks) blocks = search_blocks(most, true);
  return align_up((size_t)num * 8, 256) + align_up((size_t)blocks * 8, 256);
}

}  // namespace
}  // namespace gearhip

using namespace gearhip;

extern "C" size_t gear_hip_search_workspace_bytes(int64_t num) { return search_ws_bytes(num); }

extern "C" int gear_hip_upper_bound_f64(const double *prefix, int64_t n, const float *u,
                                        int64_t num, int unit_uniforms, int64_t *idx_out,
                                        const float *priorities, double beta, float *weights_out,
                                        void *workspace, size_t workspace_bytes, void *stream) {
  if (n < 0 || num < 0) return GEAR_HIP_EINVAL;
  if (num == 0) return 0;
  if (n == 0 || !prefix || !u || !idx_out) return GEAR_HIP_EINVAL;
  if ((priorities == nullptr) != (weights_out == nullptr)) return GEAR_HIP_EINVAL;
  const int64_t blocks = search_blocks(num, priorities != nullptr);
  const int64_t nblocks = ceil_div64(num, kBlock);
  if (blocks >= 0x7fffffffll) return GEAR_HIP_ERANGE;
  double *wraw = nullptr, *bmax = nullptr;
  if (priorities) {
    if (!workspace || workspace_bytes < search_ws_bytes(num) ||
        (reinterpret_cast<uintptr_t>(workspace) & 7))
      return GEAR_HIP_EWORKSPACE;
    wraw = static_cast<double *>(workspace);
    bmax = reinterpret_cast<double *>(static_cast<char *>(workspace) +
                                      align_up((size_t)num * 8, 256));
  }
  hipStream_t st = as_stream(stream);
  const DrawF64 draw{prefix, n, u, unit_uniforms ? 1 : 0};
  if (!priorities) return launch_search(draw, num, idx_out, st);
  with_search_shape(num, true, [&](auto lanes, auto threads) {
    constexpr int kThreads = decltype(threads)::value;
    search_weights_kernel<decltype(lanes)::value, kThreads>
        <<<dim3((unsigned)blocks), dim3(kThreads), 0, st>>>(draw, num, idx_out, priorities, beta, wraw, bmax);
  });
  GEARHIP_RETURN_IF_LAUNCH_FAILED();
  normalise_kernel<<<dim3((unsigned)nblocks), dim3(kBlock), 0, st>>>(wraw, bmax, (int)blocks, num,
                                                                    weights_out);
  GEARHIP_RETURN_IF_LAUNCH_FAILED();
  return 0;
}

extern "C" int gear_hip_upper_bound_i64(const int64_t *prefix, int64_t n, const void *u,
                                        int64_t num, int unit_uniforms, int64_t *idx_out,
                                        void *stream) {
  if (n < 0 || num < 0) return GEAR_HIP_EINVAL;
  if (num == 0) return 0;
  if (n == 0 || !prefix || !u || !idx_out) return GEAR_HIP_EINVAL;
  return launch_search(DrawI64{prefix, n, u, unit_uniforms ? 1 : 0}, num, idx_out, as_stream(stream));
}

extern "C" size_t gear_hip_sample_workspace_bytes(int64_t num) { return sample_ws(num).total; }

extern "C" int gear_hip_sample_sorted_f64(const double *prefix, int64_t n, const float *u,
                                          int64_t num, int unit_uniforms, int64_t *sorted_out,
                                          int64_t trajectory_length, int64_t modulo,
                                          int64_t *idxs, int64_t *tss, int64_t *lens,
                                          void *workspace, size_t workspace_bytes, void *stream) {
  if (n < 0 || num < 0 || trajectory_length < 0 || modulo < 0) return GEAR_HIP_EINVAL;
  if (num == 0) return 0;
  if (n == 0 || !prefix || !u) return GEAR_HIP_EINVAL;
  if (trajectory_length > 0 && (!idxs || !tss)) return GEAR_HIP_EINVAL;
  if (trajectory_length == 0 && !sorted_out) return GEAR_HIP_EINVAL;
  int key_bits = 0;
  while (key_bits < 63 && ((uint64_t)(n - 1) >> key_bits) != 0) ++key_bits;
  hipStream_t st = as_stream(stream);
  const SampleWs w = sample_ws(num);
  if (!workspace || workspace_bytes < w.total || (reinterpret_cast<uintptr_t>(workspace) & 7))
    return GEAR_HIP_EWORKSPACE;
  char *ws = static_cast<char *>(workspace);
  int64_t *raw = reinterpret_cast<int64_t *>(ws + w.raw);
  const int64_t blocks = ceil_div64(num, kBlock);
  const Split split{sorted_out, trajectory_length, modulo, idxs, tss, lens};
  const DrawF64 draw{prefix, n, u, unit_uniforms ? 1 : 0};
  if (apart(draw, num, split)) {
    if (num <= radix::kRankMax) return place_draws(draw, num, split, st);
    if (ranges::fits(num)) return sort_draws(draw, num, split, st);
  }
  int rc = launch_search(draw, num, raw, st);
  if (rc) return rc;
  if (num <= radix::kRankMax) return place_positions(raw, num, split, st);
  int64_t *sorted = sorted_out ? sorted_out : reinterpret_cast<int64_t *>(ws + w.sorted);
  rc = radix::sort_pairs<uint64_t, uint64_t>(
      reinterpret_cast<const uint64_t *>(raw), reinterpret_cast<uint64_t *>(sorted), nullptr,
      nullptr, reinterpret_cast<uint64_t *>(ws + w.ktmp), nullptr, num, 0, key_bits,
      reinterpret_cast<uint32_t *>(ws + w.hist), st);
  if (rc) return rc;
  if (trajectory_length > 0) {
    split_sorted_kernel<<<dim3((unsigned)blocks), dim3(kBlock), 0, st>>>(
        sorted, num, trajectory_length, modulo, idxs, tss, lens);
    GEARHIP_RETURN_IF_LAUNCH_FAILED();
  }
  return 0;
}

namespace gearhip {
namespace {

int check_lookup(const Lookup &look) {
  if (look.index_n < 0 || look.lengths_n < 0) return GEAR_HIP_EINVAL;
  if ((look.lens || look.starts) && !look.lengths_table) return GEAR_HIP_EINVAL;
  if (look.starts && (!look.start_u || look.window < 1)) return GEAR_HIP_EINVAL;
  if (!look.sampled && !look.local && !look.lens && !look.starts) return GEAR_HIP_EINVAL;
  return 0;
}

// Beyond this many positions among at most 256 entries -- one digit of a radix sort, which with the
// look-ups takes 12.1 us whatever the positions are -- the one-launch sort is the slower one: 10.7 us at
// 12 288, 12.9 at 20 480, 17.5 at 32 768, a few more where they are the same few entries.  Integer draws
// take 15.1 us that way, in one launch 15.0 / 17.6 / 25.8.
constexpr int64_t kFewEntries = 12288;

// raw: num positions on the device (each in [0, bound)); sorted ascending, then looked up.
int sort_and_look_up(const int64_t *raw, int64_t num, int64_t bound, const Lookup &look, char *ws,
                     const SampleWs &w, hipStream_t st) {
  const bool over = writes_over(look, raw, num * 8, num);  // (then reading ends before writing begins)
  if (num <= radix::kRankMax && !over) return place_positions(raw, num, look, st);
  int key_bits = 1;
  while (key_bits < 63 && ((uint64_t)(bound - 1) >> key_bits) != 0) ++key_bits;
  if (key_bits <= 32 && ranges::fits(num) && (key_bits > 8 || num <= kFewEntries) && !over)
    return ranges::sort<uint32_t, false>(PositionSrc{raw, (uint32_t)(((uint64_t)1 << key_bits) - 1)},
                                         num, PositionEmit{raw, look}, st);
  int64_t *sorted = reinterpret_cast<int64_t *>(ws + w.sorted);
  const int rc = radix::sort_pairs<uint64_t, uint64_t>(
      reinterpret_cast<const uint64_t *>(raw), reinterpret_cast<uint64_t *>(sorted), nullptr,
      nullptr, reinterpret_cast<uint64_t *>(ws + w.ktmp), nullptr, num, 0, key_bits,
      reinterpret_cast<uint32_t *>(ws + w.hist), st);
  if (rc) return rc;
  lookup_kernel<<<dim3((unsigned)ceil_div64(num, kBlock)), dim3(kBlock), 0, st>>>(sorted, num, look);
  GEARHIP_RETURN_IF_LAUNCH_FAILED();
  return 0;
}

// draws: searched, sorted ascending, looked up
template <typename Draw>
int draw_and_look_up(const Draw &draw, int64_t num, const Lookup &look, char *ws, const SampleWs &w,
                     hipStream_t st) {
  if (apart(draw, num, look)) {
    if (num <= radix::kRankMax) return place_draws(draw, num, look, st);
    if (ranges::fits(num) && (sizeof(typename Draw::key_type) < 8 || draw.n > 256 || num <= kFewEntries))
      return sort_draws(draw, num, look, st);
  }
  int64_t *raw = reinterpret_cast<int64_t *>(ws + w.raw);
  const int rc = launch_search(draw, num, raw, st);
  if (rc) return rc;
  return sort_and_look_up(raw, num, draw.n, look, ws, w, st);
}

}  // namespace
}  // namespace gearhip

extern "C" int gear_hip_sample_lookup_f64(const double *prefix, int64_t n, const float *u,
                                          int64_t num, int unit_uniforms,
                                          const int64_t *index_table, int64_t index_offset,
                                          const int64_t *lengths_table, int64_t lengths_n,
                                          int64_t *sampled_out, int64_t *local_out,
                                          int64_t *lens_out, void *workspace,
                                          size_t workspace_bytes, void *stream) {
  if (n < 0 || num < 0) return GEAR_HIP_EINVAL;
  if (num == 0) return 0;
  if (n == 0 || !prefix || !u) return GEAR_HIP_EINVAL;
  const Lookup look{index_table, n, index_offset, lengths_table, lengths_n, sampled_out, local_out,
                    lens_out};
  int rc = check_lookup(look);
  if (rc) return rc;
  const SampleWs w = sample_ws(num);
  if (!workspace || workspace_bytes < w.total || (reinterpret_cast<uintptr_t>(workspace) & 7))
    return GEAR_HIP_EWORKSPACE;
  return draw_and_look_up(DrawF64{prefix, n, u, unit_uniforms ? 1 : 0}, num, look,
                          static_cast<char *>(workspace), w, as_stream(stream));
}

extern "C" int64_t gear_hip_draw_max_of(int compute_units, int threads_per_unit) {
  return most_draws(compute_units, threads_per_unit);
}
extern "C" int64_t gear_hip_draw_max(void) {
  static std::atomic<int64_t> known[64];  // per device; 0: not asked yet
  int dev = 0, units = 0, threads = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0) {
    (void)hipGetLastError();
    return 0;
  }
  const bool keep = dev < 64;
  if (keep && known[dev].load(std::memory_order_relaxed) != 0) return known[dev].load(std::memory_order_relaxed);
  if (hipDeviceGetAttribute(&units, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
      hipDeviceGetAttribute(&threads, hipDeviceAttributeMaxThreadsPerMultiProcessor, dev) != hipSuccess) {
    (void)hipGetLastError();
    return 0;
  }
  const int64_t most = most_draws(units, threads);
  if (keep) known[dev].store(most, std::memory_order_relaxed);
  return most;
}
extern "C" int64_t gear_hip_draw_max_bound(void) { return kMaxBound; }

extern "C" int gear_hip_draw_lookup_f64(const double *prefix, int64_t n, uint64_t seed, uint64_t offset,
                                        int64_t num, const int64_t *index_table, int64_t index_offset,
                                        const int64_t *lengths_table, int64_t lengths_n,
                                        int64_t *sampled_out, int64_t *local_out, int64_t *lens_out,
                                        void *workspace, size_t workspace_bytes, void *stream) {
  if (n < 0 || num < 0) return GEAR_HIP_EINVAL;
  if (num == 0) return 0;
  if (n == 0 || !prefix) return GEAR_HIP_EINVAL;
  const Lookup look{index_table, n, index_offset, lengths_table, lengths_n, sampled_out, local_out,
                    lens_out};
  int rc = check_lookup(look);
  if (rc) return rc;
  if (num > gear_hip_draw_max()) return GEAR_HIP_ERANGE;
  const SampleWs w = sample_ws(num);
  if (!workspace || workspace_bytes < w.total || (reinterpret_cast<uintptr_t>(workspace) & 7))
    return GEAR_HIP_EWORKSPACE;
  hipStream_t st = as_stream(stream);
  const Philox rng{seed, offset};
  if (num <= kDrawnInPlace && !writes_over(look, prefix, n * 8, num))
    return place_draws(DrawF64From<PhiloxU>{prefix, n, {rng}, 1}, num, look, st);
  char *ws = static_cast<char *>(workspace);
  float *u = reinterpret_cast<float *>(ws + w.ktmp);  // (free until the draws have been searched)
  draw_uniform_kernel<<<dim3((unsigned)ceil_div64(num, kBlock)), dim3(kBlock), 0, st>>>(rng, num, u);
  GEARHIP_RETURN_IF_LAUNCH_FAILED();
  return draw_and_look_up(DrawF64{prefix, n, u, 1}, num, look, ws, w, st);
}

extern "C" int gear_hip_draw_sort_lookup_i64(uint64_t seed, uint64_t offset, int64_t num, int64_t bound,
                                             const int64_t *index_table, int64_t index_n,
                                             int64_t index_offset, const int64_t *lengths_table,
                                             int64_t lengths_n, int64_t *sampled_out, int64_t *local_out,
                                             int64_t *lens_out, void *workspace, size_t workspace_bytes,
                                             void *stream) {
  if (num < 0 || bound <= 0) return GEAR_HIP_EINVAL;
  if (num == 0) return 0;
  if (bound > kMaxBound) return GEAR_HIP_ERANGE;
  const Lookup look{index_table, index_n, index_offset, lengths_table, lengths_n, sampled_out,
                    local_out, lens_out};
  int rc = check_lookup(look);
  if (rc) return rc;
  if (num > gear_hip_draw_max()) return GEAR_HIP_ERANGE;
  const SampleWs w = sample_ws(num);
  if (!workspace || workspace_bytes < w.total || (reinterpret_cast<uintptr_t>(workspace) & 7))
    return GEAR_HIP_EWORKSPACE;
  hipStream_t st = as_stream(stream);
  const PhiloxPositions drawn{{seed, offset}, (uint32_t)bound};
  if (num <= kDrawnInPlace) return place_positions(drawn, num, look, st);
  char *ws = static_cast<char *>(workspace);
  int64_t *raw = reinterpret_cast<int64_t *>(ws + w.raw);
  draw_positions_kernel<<<dim3((unsigned)ceil_div64(num, kBlock)), dim3(kBlock), 0, st>>>(drawn, num, raw);
  GEARHIP_RETURN_IF_LAUNCH_FAILED();
  return sort_and_look_up(raw, num, bound, look, ws, w, st);
}

extern "C" int gear_hip_sample_lookup_i64(const int64_t *prefix, int64_t n, const void *u,
                                          int64_t num, int unit_uniforms,
                                          const int64_t *index_table, int64_t index_offset,
                                          const int64_t *lengths_table, int64_t lengths_n,
                                          int64_t *sampled_out, int64_t *local_out,
                                          int64_t *lens_out, const double *start_uniforms,
                                          int64_t window, int64_t *starts_out, void *workspace,
                                          size_t workspace_bytes, void *stream) {
  if (n < 0 || num < 0) return GEAR_HIP_EINVAL;
  if (num == 0) return 0;
  if (n == 0 || !prefix || !u) return GEAR_HIP_EINVAL;
  Lookup look{index_table, n, index_offset, lengths_table, lengths_n, sampled_out, local_out,
              lens_out};
  look.start_u = start_uniforms;
  look.window = window;
  look.starts = starts_out;
  int rc = check_lookup(look);
  if (rc) return rc;
  const SampleWs w = sample_ws(num);
  if (!workspace || workspace_bytes < w.total || (reinterpret_cast<uintptr_t>(workspace) & 7))
    return GEAR_HIP_EWORKSPACE;
  return draw_and_look_up(DrawI64{prefix, n, u, unit_uniforms ? 1 : 0}, num, look,
                          static_cast<char *>(workspace), w, as_stream(stream));
}

extern "C" int gear_hip_sort_lookup_i64(const int64_t *positions, int64_t num, int64_t bound,
                                        const int64_t *index_table, int64_t index_n,
                                        int64_t index_offset, const int64_t *lengths_table,
                                        int64_t lengths_n, int64_t *sampled_out,
                                        int64_t *local_out, int64_t *lens_out, void *workspace,
                                        size_t workspace_bytes, void *stream) {
  if (num < 0 || bound <= 0) return GEAR_HIP_EINVAL;
  if (num == 0) return 0;
  if (!positions) return GEAR_HIP_EINVAL;
  const Lookup look{index_table, index_n, index_offset, lengths_table, lengths_n, sampled_out,
                    local_out, lens_out};
  int rc = check_lookup(look);
  if (rc) return rc;
  const SampleWs w = sample_ws(num);
  if (!workspace || workspace_bytes < w.total || (reinterpret_cast<uintptr_t>(workspace) & 7))
    return GEAR_HIP_EWORKSPACE;
  return sort_and_look_up(positions, num, bound, look, static_cast<char *>(workspace), w,
                          as_stream(stream));
}

extern "C" int gear_hip_lookup_i64(const int64_t *positions, int64_t num,
                                   const int64_t *index_table, int64_t index_n,
                                   int64_t index_offset, const int64_t *lengths_table,
                                   int64_t lengths_n, int64_t *sampled_out, int64_t *local_out,
                                   int64_t *lens_out, void *stream) {
  if (num < 0) return GEAR_HIP_EINVAL;
  if (num == 0) return 0;
  if (!positions) return GEAR_HIP_EINVAL;
  const Lookup look{index_table, index_n, index_offset, lengths_table, lengths_n, sampled_out,
                    local_out, lens_out};
  int rc = check_lookup(look);
  if (rc) return rc;
  const int64_t blocks = ceil_div64(num, kBlock);
  if (blocks >= 0x7fffffffll) return GEAR_HIP_ERANGE;
  lookup_kernel<<<dim3((unsigned)blocks), dim3(kBlock), 0, as_stream(stream)>>>(positions, num,
                                                                               look);
  GEARHIP_RETURN_IF_LAUNCH_FAILED();
  return 0;
}

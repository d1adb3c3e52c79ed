// Priority update weights[idx[j]] = values[j] with "last occurrence wins" for repeated indices.
//
// With unique indices this is one scatter.  Otherwise only the last update of an index is written:
//  * up to kClassMax updates (kClassMaxDigit in a short table): one launch, a hash table in LDS a
//    workgroup.
//  * beyond that, and where a buffer overlaps another or a table has more entries than 32 bits
//    count: the (index, position) pairs go through the stable LSD radix sort on the index, and the
//    last element of each run is written.
#include "range_sort.hpp"

namespace gearhip {
namespace {

constexpr int kBlock = 256;

template <typename T>
__global__ __launch_bounds__(kBlock) void scatter_unique_kernel(T *__restrict__ w, int64_t n,
                                                                const int64_t *__restrict__ idx,
                                                                const T *__restrict__ v,
                                                                int64_t num) {
  const int64_t j = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (j >= num) return;
  const int64_t i = idx[j];
  if (i >= 0 && i < n) w[i] = v[j];
}

__global__ __launch_bounds__(kBlock) void scatter_prepare_kernel(const int64_t *__restrict__ idx,
                                                                 int64_t n, int64_t num,
                                                                 uint64_t *__restrict__ keys,
                                                                 uint32_t *__restrict__ pos) {
  const int64_t j = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (j >= num) return;
  const int64_t i = idx[j];
  keys[j] = (i >= 0 && i < n) ? (uint64_t)i : (uint64_t)n;  // n = "ignore", sorts last
  pos[j] = (uint32_t)j;
}

template <typename T>
__global__ __launch_bounds__(kBlock) void scatter_winners_kernel(T *__restrict__ w, int64_t n,
                                                                 const uint64_t *__restrict__ keys,
                                                                 const uint32_t *__restrict__ pos,
                                                                 const T *__restrict__ v,
                                                                 int64_t num) {
  const int64_t j = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (j >= num) return;
  const uint64_t key = keys[j];
  if (key >= (uint64_t)n) return;
  if (j + 1 < num && keys[j + 1] == key) return;  // a later update of the same index exists
  w[key] = v[pos[j]];
}

// ---- the last of every index, in one launch -----------------------------------------------------------
// Workgroup c takes the indices of class c (a few bits of a cheap mix): it reads ALL indices (out
// of L2) and keeps the largest position of each of its own in a hash table in LDS, whose words hold
// index << 32 | position.  What bounds it is issuing that look at every index, 256 times over, so
// the look is seven instructions, and what passes it waits in a queue of the wave until there is a
// wave's worth to insert.  Later positions go first and a word is looked at before it is changed,
// so most updates of an index that repeats find a larger position and are done.  Should the table
// overflow (indices that crowd in one class), the class is taken in 2, 4, ... parts by further bits
// of the hash; part and slot together are at last the whole hash, which no two indices share.
// us a call, back to back, here / by sorting the pairs (a ranking sort up to 4096):
//     updates of   5 entries    255 entries    1e4 entries    1e7 entries   5 of 1e4 entries
//         64        4.3 / 11.9                   4.2 / 11.9     4.1 / 11.9
//       4096        5.7 / 13.1                   4.7 / 13.4     4.6 / 13.4
//     32 768       11.9 / 12.0    8.8 / 12.9     8.4 / 20.3     8.6 / 29.0    11.0 / 19.7
//     40 960       13.5 / 12.4   10.0 / 12.9     9.5 / 20.6     9.9 / 30.0    12.5 / 19.8
//     65 536       18.8 / 12.7   13.6 / 13.4    12.6 / 21.5    13.5 / 31.1    17.9 / 20.6
//    131 072       32.4 / 14.2   23.3 / 15.6    21.0 / 25.8    22.6 / 38.3    31.7 / 24.0
//    196 608       46.0 / 15.6   33.1 / 17.3    29.5 / 28.8    32.7 / 43.3    45.7 / 26.2
// Tables below 256 entries are one digit for the sort, which is the faster one from 40 960 updates on;
// for others the limit is the last size at which updates spread over the table win at every length of
// it.  (Indices that repeat thousands of times while the table is long lose a third there, and win
// below 90 000.)
constexpr int kClassThreads = 1024;
constexpr int kClassWaves = kClassThreads / kWave;
constexpr int kClassBits = 8, kSlotBits = 11, kPartBits = 32 - kSlotBits;
constexpr int kClasses = 1 << kClassBits, kSlots = 1 << kSlotBits;
constexpr int kMaxProbes = 128;
constexpr int kQueue = 2 * kWave;
constexpr int64_t kClassMax = 131072;  // a quarter of the slots when no index repeats
constexpr int64_t kClassMaxDigit = 40960;  // tables below 256 entries
constexpr uint64_t kEmpty = ~0ull;

__device__ __forceinline__ uint32_t class_of(uint32_t x) {
  return (uint32_t)__umul24(x ^ (x >> 15), 0x9E3779u) >> (32 - kClassBits);
}
__device__ __forceinline__ uint32_t hash_of(uint32_t x) {  // one to one (multipliers: xxHash32's primes)
  x ^= x >> 16;
  x *= 0x9E3779B1u;
  x ^= x >> 15;
  x *= 0x85EBCA77u;
  return x ^ (x >> 13);
}

// false: no room
__device__ __forceinline__ bool keep_last(uint64_t *slot, uint32_t at, uint64_t word) {
#pragma unroll 1
  for (int probe = 0; probe < kMaxProbes; ++probe) {
    uint64_t cur = __hip_atomic_load(slot + at, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    if (cur == kEmpty)
      cur = (uint64_t)atomicCAS(reinterpret_cast<unsigned long long *>(slot + at), kEmpty, word);
    if (cur == kEmpty) return true;
    if ((cur >> 32) == (word >> 32)) {
      if (cur < word) atomicMax(reinterpret_cast<unsigned long long *>(slot + at), word);
      return true;
    }
    at = (at + 1) & (kSlots - 1);
  }
  return false;
}

template <typename T>
__global__ __launch_bounds__(kClassThreads) void scatter_class_kernel(
    T *__restrict__ w, uint32_t n, const int64_t *__restrict__ idx, const T *__restrict__ v, int num) {
  __shared__ uint64_t slot[kSlots];
  __shared__ uint64_t queue_all[kClassWaves][kQueue];
  constexpr int kAhead = 8;
  const int tid = threadIdx.x, lane = tid & (kWave - 1);
  uint64_t *queue = queue_all[__builtin_amdgcn_readfirstlane(tid / kWave)];
  const uint32_t own = blockIdx.x;
  const int top = (num - 1) / kClassThreads * kClassThreads;
  for (int parts = 1;; parts *= 2) {
    bool full = false;
    for (int part = 0; part < parts && !full; ++part) {
#pragma unroll
      for (int q = 0; q < kSlots / kClassThreads; ++q) slot[q * kClassThreads + tid] = kEmpty;
      __syncthreads();
      bool room = true;
      int waiting = 0;  // in the wave's queue, at most kQueue
      int64_t seen = -1, seen2 = -1;  // what this lane queued last, at later positions
      auto insert = [&] {
        wave_lds_sync();
        for (int e = lane; e < waiting; e += kWave) {
          const uint64_t word = queue[e];
          const uint32_t h = hash_of((uint32_t)(word >> 32));
          if (((h >> kSlotBits) & (uint32_t)(parts - 1)) == (uint32_t)part)
            room = keep_last(slot, h & (kSlots - 1), word) && room;
        }
        wave_lds_sync();
        waiting = 0;
      };
#pragma unroll 1
      for (int base = top; base >= 0; base -= kAhead * kClassThreads) {
        int64_t i[kAhead];
#pragma unroll
        for (int q = 0; q < kAhead; ++q) {
          const int j = base - q * kClassThreads + tid;
          i[q] = idx[j < 0 ? 0 : j < num ? j : num - 1];  // (no branch between the loads)
        }
#pragma unroll
        for (int q = 0; q < kAhead; ++q) {
          const bool mine = class_of((uint32_t)i[q]) == own;
          if (wave_ballot(mine) == 0) continue;
          const int j = base - q * kClassThreads + tid;
          const bool take = mine && (uint64_t)i[q] < (uint64_t)n && j >= 0 && j < num &&
                            i[q] != seen && i[q] != seen2;
          const uint64_t takes = wave_ballot(take);
          seen2 = take ? seen : seen2;
          seen = take ? i[q] : seen;
          if (take)
            queue[waiting + __popcll(takes & ((1ull << lane) - 1))] =
                ((uint64_t)i[q] << 32) | (uint32_t)j;
          waiting += __popcll(takes);
          if (waiting > kQueue - kWave) insert();
        }
      }
      insert();
      full = __syncthreads_or(!room) && parts < (1 << kPartBits);
      if (!full) {
#pragma unroll
        for (int q = 0; q < kSlots / kClassThreads; ++q) {
          const uint64_t word = slot[q * kClassThreads + tid];
          if (word != kEmpty) w[word >> 32] = v[(uint32_t)word];
        }
      }
      __syncthreads();
    }
    if (!full) return;
  }
}

struct Layout {
  size_t kin, vin, kout, vout, ktmp, vtmp, hist, total;
};
Layout layout(int64_t num) {
  Layout l;
  const size_t m = num > 0 ? (size_t)num : 1;
  const size_t k8 = align_up(m * 8, 256), v4 = align_up(m * 4, 256);
  size_t o = 0;
  l.kin = o;  o += k8;
  l.kout = o; o += k8;
  l.ktmp = o; o += k8;
  l.vin = o;  o += v4;
  l.vout = o; o += v4;
  l.vtmp = o; o += v4;
  l.hist = o; o += radix::hist_bytes(num);
  l.total = o;
  return l;
}

}  // namespace
}  // namespace gearhip

using namespace gearhip;

extern "C" size_t gear_hip_scatter_workspace_bytes(int64_t num) { return layout(num).total; }

namespace {
template <typename T>
int scatter_any(T *weights, int64_t n, const int64_t *idx, const T *values, int64_t num,
                int unique_indices, void *workspace, size_t workspace_bytes, void *stream) {
  if (n < 0 || num < 0) return GEAR_HIP_EINVAL;
  if (num == 0 || n == 0) return 0;
  if (!weights || !idx || !values) return GEAR_HIP_EINVAL;
  if (num >= (1ll << 32)) return GEAR_HIP_ERANGE;
  hipStream_t st = as_stream(stream);
  const dim3 grid((unsigned)ceil_div64(num, kBlock)), block(kBlock);
  if (unique_indices) {
    scatter_unique_kernel<T><<<grid, block, 0, st>>>(weights, n, idx, values, num);
    GEARHIP_RETURN_IF_LAUNCH_FAILED();
    return 0;
  }
  const Layout l = layout(num);
  if (!workspace || workspace_bytes < l.total || (reinterpret_cast<uintptr_t>(workspace) & 7))
    return GEAR_HIP_EWORKSPACE;
  const int64_t bytes = num * (int64_t)sizeof(T), wbytes = n * (int64_t)sizeof(T);
  if (!ranges::overlap(weights, wbytes, idx, num * 8) && !ranges::overlap(weights, wbytes, values, bytes)) {
    if (num <= (n < 256 ? kClassMaxDigit : kClassMax) && n < (1ll << 32)) {
      scatter_class_kernel<T><<<dim3(kClasses), dim3(kClassThreads), 0, st>>>(weights, (uint32_t)n, idx,
                                                                            values, (int)num);
      GEARHIP_RETURN_IF_LAUNCH_FAILED();
      return 0;
    }
  }
  char *ws = static_cast<char *>(workspace);
  uint64_t *kin = reinterpret_cast<uint64_t *>(ws + l.kin);
  uint64_t *kout = reinterpret_cast<uint64_t *>(ws + l.kout);
  uint32_t *vin = reinterpret_cast<uint32_t *>(ws + l.vin);
  uint32_t *vout = reinterpret_cast<uint32_t *>(ws + l.vout);
  scatter_prepare_kernel<<<grid, block, 0, st>>>(idx, n, num, kin, vin);
  GEARHIP_RETURN_IF_LAUNCH_FAILED();
  int bits = 0;
  while (bits < 64 && ((uint64_t)n >> bits) != 0) ++bits;  // keys are in [0, n]
  int rc = radix::sort_pairs<uint64_t, uint32_t>(
      kin, kout, vin, vout, reinterpret_cast<uint64_t *>(ws + l.ktmp),
      reinterpret_cast<uint32_t *>(ws + l.vtmp), num, 0, bits,
      reinterpret_cast<uint32_t *>(ws + l.hist), st);
  if (rc) return rc;
  scatter_winners_kernel<T><<<grid, block, 0, st>>>(weights, n, kout, vout, values, num);
  GEARHIP_RETURN_IF_LAUNCH_FAILED();
  return 0;
}
}  // namespace

extern "C" int gear_hip_scatter_f32(float *weights, int64_t n, const int64_t *idx,
                                    const float *values, int64_t num, int unique_indices,
                                    void *workspace, size_t workspace_bytes, void *stream) {
  return scatter_any<float>(weights, n, idx, values, num, unique_indices, workspace,
                            workspace_bytes, stream);
}

extern "C" int gear_hip_scatter_i64(int64_t *table, int64_t n, const int64_t *idx,
                                    const int64_t *values, int64_t num, int unique_indices,
                                    void *workspace, size_t workspace_bytes, void *stream) {
  return scatter_any<int64_t>(table, n, idx, values, num, unique_indices, workspace,
                              workspace_bytes, stream);
}

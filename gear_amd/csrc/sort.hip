// gear_hip_sort_i64: ascending stable sort of non-negative int64 keys with optional payload.
#include "range_sort.hpp"

using namespace gearhip;

namespace {
struct SortWs {
  size_t ktmp, vtmp, hist, total;
};
SortWs sort_ws(int64_t num) {
  SortWs w;
  const size_t n = num > 0 ? (size_t)num : 1;
  w.ktmp = 0;
  w.vtmp = align_up(n * 8, 256);
  w.hist = w.vtmp + align_up(n * 8, 256);
  w.total = w.hist + radix::hist_bytes(num);
  return w;
}

template <typename C>
struct Src {
  const int64_t *keys;
  uint64_t mask;
  __device__ __forceinline__ void begin() {}
  __device__ __forceinline__ C key(int j) const { return (C)((uint64_t)keys[j] & mask); }
};

struct Emit {
  const int64_t *kin, *vin;
  int64_t *kout, *vout;
  __device__ __forceinline__ void put(uint32_t place, int j) const {
    kout[place] = kin[j];
    if (vin) vout[place] = vin[j];
  }
  template <typename L>
  __device__ __forceinline__ void list(const L &list, const uint32_t *rank, int n,
                                       uint32_t base) const {
    const int e = threadIdx.x;
    if (e < n) put(base + rank[e], list.pos(e));
  }
  __device__ __forceinline__ void equal(const uint32_t *at, int n, uint32_t base) const {
    const int e = threadIdx.x;
    if (e < n) put(base + (uint32_t)e, (int)at[e]);
  }
};

// Up to kRankMax keys the ranking sort is the faster one, for a digit or two the radix sort; outputs
// on top of inputs need launches that end reading before they write.
bool one_launch(const int64_t *kin, int64_t *kout, const int64_t *vin, int64_t *vout, int64_t num,
                int key_bits) {
  const int64_t b = num * 8;
  return num > radix::kRankMax && ranges::fits(num) && num <= ranges::worth(key_bits) &&
         !ranges::overlap(kin, b, kout, b) && !ranges::overlap(kin, b, vout, b) &&
         !ranges::overlap(vin, b, kout, b) && !ranges::overlap(vin, b, vout, b);
}

// ---- entries of a table, in order ---------------------------------------------------------------------
// Entries that are in order as they come need no sort, but a sort does not know it before it has read all
// of them in every workgroup (20 000 in order: 12.4 us behind 4.7 for the look-up).  The look-up sees a
// neighbour for the price of another load, so it says so, workgroup by workgroup, and stores its
// entries where they belong if all of them say so; the sort looks at those words and ends (4.0 + 2.8 us).
// Entries in no order pay for the look: 4096 / 5000 / 20 000 in 14.1 / 12.7 / 21.6 us by look-up and sort, 15.0 / 13.9 /
// 22.2 so, where those in order take 14.1 / 12.7 / 14.3 and 10.4 / 9.4 / 9.6.
// Beyond what one launch sorts nobody looks at such words: an ordinary look-up then, and the sort.
constexpr int kTakeBlock = 256;
struct Taken : Src<uint64_t> {
  static constexpr bool kGuarded = true;
  radix::InOrder in_order;
  __device__ __forceinline__ bool done() const { return in_order.holds(); }
};
constexpr uint64_t kTakenMask = ~(1ull << 63);

__global__ __launch_bounds__(kTakeBlock) void take_in_order_kernel(
    const int64_t *__restrict__ table, int64_t n, const int64_t *__restrict__ idx, int64_t num,
    int64_t *__restrict__ taken, int64_t *__restrict__ out, uint32_t *__restrict__ in_order) {
  const int64_t j = (int64_t)blockIdx.x * kTakeBlock + threadIdx.x;
  const int64_t at = j < num ? j : num - 1, next = at + 1 < num ? at + 1 : at;
  const int64_t i0 = idx[at], i1 = idx[next];
  const int64_t v0 = i0 >= 0 && i0 < n ? table[i0] : 0, v1 = i1 >= 0 && i1 < n ? table[i1] : 0;
  if (j < num) taken[j] = out[j] = v0;
  const int ordered = __syncthreads_and(((uint64_t)v0 & kTakenMask) <= ((uint64_t)v1 & kTakenMask));
  if (threadIdx.x == 0) in_order[blockIdx.x] = ordered ? 1u : 0u;
}

bool guarded(int64_t num) { return num <= radix::kRankMax || ranges::fits(num); }

struct TakeWs {
  size_t sort, taken, words, total;
};
TakeWs take_ws(int64_t num) {
  TakeWs w;
  const size_t n = num > 0 ? (size_t)num : 1;
  w.sort = 0;
  w.taken = align_up(sort_ws(num).total, 256);
  w.words = w.taken + align_up(n * 8, 256);
  w.total = w.words + (guarded(num) ? align_up((size_t)ceil_div64((int64_t)n, kTakeBlock) * 4, 256) : 0);
  return w;
}
}  // namespace

extern "C" size_t gear_hip_take_sorted_workspace_bytes(int64_t num) { return take_ws(num).total; }

extern "C" int gear_hip_take_sorted_i64(const int64_t *table, int64_t n, const int64_t *idx, int64_t num,
                                        int64_t *out, void *workspace, size_t workspace_bytes, void *stream) {
  if (num < 0 || n < 0) return GEAR_HIP_EINVAL;
  if (num == 0) return 0;
  if (!idx || !out || (n > 0 && !table)) return GEAR_HIP_EINVAL;
  if (ranges::overlap(out, num * 8, idx, num * 8) || ranges::overlap(out, num * 8, table, n * 8))
    return GEAR_HIP_EINVAL;
  const TakeWs w = take_ws(num);
  if (!workspace || workspace_bytes < w.total || (reinterpret_cast<uintptr_t>(workspace) & 7))
    return GEAR_HIP_EWORKSPACE;
  char *ws = static_cast<char *>(workspace);
  hipStream_t st = as_stream(stream);
  int64_t *taken = reinterpret_cast<int64_t *>(ws + w.taken);
  radix::InOrder in_order;
  if (guarded(num)) {
    const int64_t blocks = ceil_div64(num, kTakeBlock);
    uint32_t *words = reinterpret_cast<uint32_t *>(ws + w.words);
    take_in_order_kernel<<<dim3((unsigned)blocks), dim3(kTakeBlock), 0, st>>>(table, n, idx, num, taken, out, words);
    GEARHIP_RETURN_IF_LAUNCH_FAILED();
    in_order = radix::InOrder{words, (int)blocks};
  } else {
    // (no entries: every index is outside, nothing is read)
    const int rc = gear_hip_take_i64(n > 0 ? table : idx, n, idx, num, 0, taken, stream);
    if (rc) return rc;
  }
  if (num > radix::kRankMax && ranges::fits(num)) {
    Taken src{};
    src.keys = taken;
    src.mask = kTakenMask;
    src.in_order = in_order;
    return ranges::sort<uint64_t, false>(src, num, Emit{taken, nullptr, out, nullptr}, st);
  }
  const SortWs s = sort_ws(num);
  return radix::sort_pairs<uint64_t, uint64_t>(
      reinterpret_cast<const uint64_t *>(taken), reinterpret_cast<uint64_t *>(out), nullptr, nullptr,
      reinterpret_cast<uint64_t *>(ws + s.ktmp), nullptr, num, 0, 63, reinterpret_cast<uint32_t *>(ws + s.hist), st,
      radix::StoreSorted(), in_order);
}

extern "C" size_t gear_hip_sort_workspace_bytes(int64_t num) { return sort_ws(num).total; }

extern "C" int gear_hip_sort_i64(const int64_t *keys_in, int64_t *keys_out, const int64_t *vals_in,
                                 int64_t *vals_out, int64_t num, int key_bits, void *workspace,
                                 size_t workspace_bytes, void *stream) {
  if (num < 0 || key_bits < 0 || key_bits > 64) return GEAR_HIP_EINVAL;
  if (num == 0) return 0;
  if (!keys_in || !keys_out || ((vals_in == nullptr) != (vals_out == nullptr)))
    return GEAR_HIP_EINVAL;
  if (keys_in == keys_out || (vals_in && vals_in == vals_out)) return GEAR_HIP_EINVAL;
  const SortWs w = sort_ws(num);
  if (!workspace || workspace_bytes < w.total || (reinterpret_cast<uintptr_t>(workspace) & 7))
    return GEAR_HIP_EWORKSPACE;
  if (one_launch(keys_in, keys_out, vals_in, vals_out, num, key_bits)) {
    const uint64_t mask = key_bits >= 64 ? ~0ull : ((uint64_t)1 << key_bits) - 1;
    const Emit emit{keys_in, vals_in, keys_out, vals_out};
    if (key_bits <= 32)
      return ranges::sort<uint32_t, true>(Src<uint32_t>{keys_in, mask}, num, emit, as_stream(stream));
    return ranges::sort<uint64_t, true>(Src<uint64_t>{keys_in, mask}, num, emit, as_stream(stream));
  }
  char *ws = static_cast<char *>(workspace);
  return radix::sort_pairs<uint64_t, uint64_t>(
      reinterpret_cast<const uint64_t *>(keys_in), reinterpret_cast<uint64_t *>(keys_out),
      reinterpret_cast<const uint64_t *>(vals_in), reinterpret_cast<uint64_t *>(vals_out),
      reinterpret_cast<uint64_t *>(ws + w.ktmp), reinterpret_cast<uint64_t *>(ws + w.vtmp), num, 0,
      key_bits, reinterpret_cast<uint32_t *>(ws + w.hist), as_stream(stream));
}

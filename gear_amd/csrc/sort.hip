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
}  // namespace

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

// The random numbers of a batch where they are used: Philox4x32-10 (Salmon, Moraes, Dror, Shaw: "Parallel
// random numbers: as easy as 1, 2, 3", 2011), one block of the generator's stream per draw.
//
// A draw of a batch is the first word of the block with counter (offset / 4, number of the draw) under the
// seed as the key, which is how torch's GPU generator numbers the elements of one rand or randint call of up
// to most_draws() elements; a call takes 4 of the generator's offset.  So a batch drawn here is the
// batch that torch would have drawn from the same generator, bit for bit.
#pragma once
#include "common.hpp"

namespace gearhip {

// torch gives a thread to every element up to the threads that the GPU holds at once, in workgroups of 256;
// beyond, a thread takes further words of its block.  (256 compute units of 2048 threads: 524 288.)
inline int64_t most_draws(int64_t compute_units, int64_t threads_per_unit) {
  return compute_units > 0 && threads_per_unit > 0 ? compute_units * (threads_per_unit / 256 * 256) : 0;
}
// Ranges from 2^28 on take two words a draw in torch's randint (of one word, taken modulo such a range, some
// entries would come up visibly more often): those are left to torch.
constexpr int64_t kMaxBound = (1ll << 28) - 1;

struct Philox {
  uint64_t seed, offset;
  __device__ __forceinline__ uint32_t word(uint64_t j) const {
    const uint64_t block = offset >> 2;
    uint32_t c0 = (uint32_t)block, c1 = (uint32_t)(block >> 32), c2 = (uint32_t)j, c3 = (uint32_t)(j >> 32);
    uint32_t k0 = (uint32_t)seed, k1 = (uint32_t)(seed >> 32);
#pragma unroll
    for (int r = 0; r < 10; ++r) {
      const uint32_t h0 = __umulhi(0xd2511f53u, c0), l0 = 0xd2511f53u * c0;
      const uint32_t h1 = __umulhi(0xcd9e8d57u, c2), l1 = 0xcd9e8d57u * c2;
      c0 = h1 ^ c1 ^ k0;
      c1 = l1;
      c2 = h0 ^ c3 ^ k1;
      c3 = l0;
      k0 += 0x9e3779b9u;
      k1 += 0xbb67ae85u;
    }
    return c0;
  }
  // in [0, 1): (word + 1) / 2^32 as fp32 rounds it, 0 for 1
  __device__ __forceinline__ float uniform(uint64_t j) const {
    const float scale = 1.0f / 4294967296.0f, u = scale + (float)word(j) * scale;
    return u == 1.0f ? 0.0f : u;
  }
  // in [0, range), range <= kMaxBound
  __device__ __forceinline__ int64_t below(uint32_t range, uint64_t j) const { return (int64_t)(word(j) % range); }
};

}  // namespace gearhip

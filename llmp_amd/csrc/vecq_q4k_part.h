// A lane's operands of a Q4_K row and of its tokens' sums for the matrix instructions (vecq_mma.hip, vecq_sorted.hip,
// vecq_tile16.hip).
#ifndef LLMP_AMD_CSRC_VECQ_Q4K_PART_H_
#define LLMP_AMD_CSRC_VECQ_Q4K_PART_H_

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "common.h"
#include "vecq_common.h"

namespace llmp_hip {

// A lane's part of one super-block of its weight row: the header and, for each pair of
// sub-blocks, the eight code bytes of its K group (low nibbles sub-block 2 p, high 2 p + 1).
// As loaded, lane (row, j) holds the whole 32 bytes of pair j instead (two 16-byte loads
// where four 8-byte ones would be needed: these scattered reads cost by the instruction), K
// group g's eight bytes in q[g]; Transpose exchanges them among the row's four lanes.
struct RowPart {
  U32x4 header;  // d, dmin, scales[12]
  uint2 q[4];
};

typedef unsigned Swapped __attribute__((ext_vector_type(2)));

__device__ __forceinline__ RowPart LoadRowPart(const uint8_t* row, int sb, int kg) {
  RowPart part;
  const uint8_t* at = row + static_cast<int64_t>(sb) * 144;
  part.header = *reinterpret_cast<const U32x4*>(at);
  const U32x4 lo = *reinterpret_cast<const U32x4*>(at + 16 + 32 * kg);
  const U32x4 hi = *reinterpret_cast<const U32x4*>(at + 32 + 32 * kg);
  part.q[0] = make_uint2(lo.x, lo.y);
  part.q[1] = make_uint2(lo.z, lo.w);
  part.q[2] = make_uint2(hi.x, hi.y);
  part.q[3] = make_uint2(hi.z, hi.w);
  return part;
}

// q[g] of the row's lane j becomes q[j] of its lane g (the lanes of a row are 16 apart): a
// 4 x 4 transpose in two rounds of row swaps, lanes 32 apart then lanes 16 apart. Every lane
// of the wave takes part.
__device__ __forceinline__ void Transpose(RowPart& part) {
  uint32_t* w = reinterpret_cast<uint32_t*>(part.q);  // q[g] = w[2 g], w[2 g + 1]
#pragma unroll
  for (int half = 0; half < 2; ++half) {
    uint32_t x0 = w[half], x1 = w[2 + half], x2 = w[4 + half], x3 = w[6 + half];
    const Swapped a = __builtin_amdgcn_permlane32_swap(x0, x2, false, false);
    const Swapped b = __builtin_amdgcn_permlane32_swap(x1, x3, false, false);
    x0 = a.x, x2 = a.y, x1 = b.x, x3 = b.y;
    const Swapped c = __builtin_amdgcn_permlane16_swap(x0, x1, false, false);
    const Swapped e = __builtin_amdgcn_permlane16_swap(x2, x3, false, false);
    w[half] = c.x, w[2 + half] = c.y, w[4 + half] = e.x, w[6 + half] = e.y;
  }
}

typedef __bf16 B8 __attribute__((ext_vector_type(8)));

// The eight minimums as bf16.
__device__ __forceinline__ B8 Minimums(const Q4KHeader& h) {
  U32x4 m;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const uint32_t word = h.mn[i >> 1] >> (16 * (i & 1));
    const float m0 = static_cast<float>(word & 0xFFu), m1 = static_cast<float>((word >> 8) & 0xFFu);
    m[i] = __builtin_amdgcn_perm(__builtin_bit_cast(uint32_t, m1), __builtin_bit_cast(uint32_t, m0), 0x07060302u);
  }
  return __builtin_bit_cast(B8, m);
}

// d8 * sum in three groups of eight bits, each in the high half of its word: 11 bits times 12, nothing of a finite product
// is left over (one that is not finite is its leading group alone).
struct SumParts {
  uint32_t lead, middle, last;
};
__device__ __forceinline__ SumParts SplitSum(float d8, int sum) {
  const float product = d8 * static_cast<float>(sum);
  SumParts parts;
  parts.lead = __builtin_bit_cast(uint32_t, product) & 0xFFFF0000u;
  const float rest = __builtin_isfinite(product) ? product - __builtin_bit_cast(float, parts.lead) : 0.0f;
  parts.middle = __builtin_bit_cast(uint32_t, rest) & 0xFFFF0000u;
  parts.last = __builtin_bit_cast(uint32_t, rest - __builtin_bit_cast(float, parts.middle));
  return parts;
}

}  // namespace llmp_hip

#endif  // LLMP_AMD_CSRC_VECQ_Q4K_PART_H_

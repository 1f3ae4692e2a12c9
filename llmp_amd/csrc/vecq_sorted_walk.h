// How the workgroups of a product over rows sorted by expert share its work (vecq_mma.hip, vecq_sorted.hip).
#ifndef LLMP_AMD_CSRC_VECQ_SORTED_WALK_H_
#define LLMP_AMD_CSRC_VECQ_SORTED_WALK_H_

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "common.h"

namespace llmp_hip {

// A value that every lane of the wave holds, as one the compiler knows to be such.
__device__ __forceinline__ int64_t Uniform(int64_t v) {
  const uint32_t low = __builtin_amdgcn_readfirstlane(static_cast<int>(v));
  const uint32_t high = __builtin_amdgcn_readfirstlane(static_cast<int>(v >> 32));
  return static_cast<int64_t>((static_cast<uint64_t>(high) << 32) | low);
}

// Consecutive groups of row tiles of one expert against up to a pass's rows of its tokens: the sorted rows
// rows_first + first .. rows_first + first + m - 1, the groups group_first .. group_first + group_count - 1.
struct SortedSegment {
  int expert, rows_first, first, m, group_first, group_count;
};

// Expert e brings ceil(rows / pass) passes; a pass costs `fixed_of(its rows)` (its tokens' staging) and then, each of its
// `groups` groups of tiles, `cost_of(its rows)`. The passes in expert order lie end to end on a line of cost, and workgroup
// w takes the groups that start within its w-th of the line: a few segments of consecutive groups, `run` called on each
// by every thread. Every wave works its workgroup's part out for itself, without barriers: a lane sums a run of consecutive
// experts, and from the first expert of the lane whose run reaches into the part on, the wave looks at 64 experts at a time,
// one a lane. So its start is one trip to memory up to 64 experts and few for thousands. (With a load after the other until
// the part's first expert: 2048 -> 512, 128 rows of 512 experts 37.6 us.)
// With kWhole every pass has workgroups of its own: a part that ends within an expert is two starts, and with few groups a
// second start costs more than the groups it evens out (2048 -> 256 of 128 experts, about 1, 4 and 16 rows each, that is 85,
// 125 and 128 passes: 20.6 / 29.5 / 22.5 us by the line, 16.0 / 17.0 / 18.8 so; 2048 -> 512 29.9 / 33.8 / 27.8 and 21.0 / 22.1 /
// 23.4). So up to half as many passes as workgroups. Beyond, a pass may have one workgroup alone: still so up to eight groups, a
// wave's one (2048 -> 256, 160 passes 30.3 -> 21.7 us), and where more than four fifths of the workgroups have work (2048 -> 512,
// 243 passes 45.0 -> 35.0; with 160 the line takes 33 and this about 38).
template <bool kWhole, typename FixedOf, typename CostOf, typename Run>
__device__ __forceinline__ void WalkSortedRows(const int32_t* __restrict__ offsets, int experts, int groups, int pass,
                                               FixedOf fixed_of, CostOf cost_of, Run run) {
  const int lane = threadIdx.x & (kWave - 1);
  auto pass_cost = [&](int rows) { return static_cast<int64_t>(fixed_of(rows)) + static_cast<int64_t>(groups) * cost_of(rows); };
  auto expert_cost = [&](int rows) -> int64_t {
    if (rows <= 0) return 0;
    const int passes = (rows + pass - 1) / pass;
    return (passes - 1) * pass_cost(pass) + pass_cost(rows - (passes - 1) * pass);
  };
  auto passes_of = [&](int rows) { return (max(rows, 0) + pass - 1) / pass; };
  const int per = (experts + kWave - 1) / kWave;
  const int mine = min(lane * per, experts), after = min(mine + per, experts);
  int64_t cost = 0;
  int passes = 0;
  int my_first = offsets[mine], my_rows = 0, begin = my_first;
  if (per <= 2) {
    const int end = offsets[min(mine + 1, after)], end2 = per == 2 ? offsets[after] : end;
    my_rows = end - begin;
    cost = expert_cost(my_rows) + expert_cost(end2 - end);
    if constexpr (kWhole) passes = passes_of(my_rows) + passes_of(end2 - end);
  } else {
    constexpr int kAtOnce = 8;  // offsets on their way at a time
    for (int i0 = 0; i0 < per; i0 += kAtOnce) {
      int end[kAtOnce];
#pragma unroll
      for (int u = 0; u < kAtOnce; ++u) end[u] = offsets[min(mine + i0 + u + 1, after)];
#pragma unroll
      for (int u = 0; u < kAtOnce; ++u) {  // (past the run's end: no rows)
        cost += expert_cost(end[u] - begin);
        if constexpr (kWhole) passes += passes_of(end[u] - begin);
        begin = end[u];
      }
    }
  }
  if constexpr (kWhole) {
    int through = passes;
#pragma unroll
    for (int delta = 1; delta < kWave; delta <<= 1) {
      const int other = __shfl_up(through, delta, kWave);
      if (lane >= delta) through += other;
    }
    const int all = __builtin_amdgcn_readlane(through, kWave - 1), workgroups = gridDim.x;
    if (all <= workgroups / 2 || (all <= workgroups && (groups <= 8 || all > workgroups / 5 * 4))) {
      if (all == 0) return;
      // Pass p has the workgroups w with floor(w all / workgroups) = p.
      const int p = static_cast<int>(blockIdx.x) * all / workgroups;
      const int first = (p * workgroups + all - 1) / all, count = ((p + 1) * workgroups + all - 1) / all - first;
      const int first_lane = __ffsll(__ballot(through > p)) - 1;
      int rest = p - __builtin_amdgcn_readlane(through - passes, first_lane);  // passes of its experts ahead of p
      for (int e = first_lane * per; e < experts; ++e) {
        const int rows_first = __builtin_amdgcn_readfirstlane(offsets[e]);
        const int rows = __builtin_amdgcn_readfirstlane(offsets[e + 1]) - rows_first;
        if (rest < passes_of(rows)) {
          const int at = static_cast<int>(blockIdx.x) - first;
          const int g_first = groups * at / count, g_end = groups * (at + 1) / count;
          if (g_first < g_end) run(SortedSegment{e, rows_first, rest * pass, min(pass, rows - rest * pass), g_first, g_end - g_first});
          return;
        }
        rest -= passes_of(rows);
      }
      return;
    }
  }
  int64_t inclusive = cost;
#pragma unroll
  for (int delta = 1; delta < kWave; delta <<= 1) {
    const int64_t other = __shfl_up(inclusive, delta, kWave);
    if (lane >= delta) inclusive += other;
  }
  const int64_t line = Uniform(__shfl(inclusive, kWave - 1, kWave));
  const int64_t from = line * blockIdx.x / gridDim.x, to = line * (blockIdx.x + 1) / gridDim.x;
  // The lane whose experts hold `from`.
  const unsigned long long past = __ballot(inclusive > from);
  if (past == 0) return;  // an empty line
  const int first_lane = __ffsll(past) - 1;
  int64_t before = Uniform(__shfl(inclusive - cost, first_lane, kWave));
  // Its experts in turn, each the first one with rows among the 64 from `base` on, and at first the first that reaches past
  // `from`. (Read again after every `run`: held through it, they would take registers that it has not to spare.)
  int base = first_lane * per;
  auto read = [&]() {
    int place = base + lane;
    asm volatile("" : "+v"(place));  // here: worked out ahead of the loop it would be held through `run` too
    my_first = offsets[min(place, experts)];
    my_rows = offsets[min(place + 1, experts)] - my_first;
  };
  if (per == 1) {  // one expert a lane already
    base = 0;
    my_rows = lane < first_lane ? 0 : my_rows;
  } else {
    read();
  }
  while (true) {
    int at = kWave;
    for (unsigned long long with = __ballot(my_rows > 0); with != 0; with &= with - 1) {
      const int64_t all = expert_cost(__builtin_amdgcn_readlane(my_rows, __ffsll(with) - 1));
      if (before + all > from) {
        at = __ffsll(with) - 1;
        break;
      }
      before += all;
    }
    base += at;
    if (at < kWave) {
      const int rows_first = __builtin_amdgcn_readlane(my_first, at), rows = __builtin_amdgcn_readlane(my_rows, at);
      for (int p0 = 0; p0 < rows; p0 += pass) {
        const int m = min(pass, rows - p0);
        const int each = cost_of(m);
        // The pass's groups start at start, start + each, ...: those within [from, to).
        const int64_t start = before + fixed_of(m);
        const int g_first = from <= start ? 0 : static_cast<int>(min<int64_t>((from - start + each - 1) / each, groups));
        const int g_end = to <= start ? 0 : static_cast<int>(min<int64_t>((to - start + each - 1) / each, groups));
        if (g_first < g_end) run(SortedSegment{base, rows_first, p0, m, g_first, g_end - g_first});
        before += pass_cost(m);
      }
      ++base;
    }
    if (base >= experts || before >= to) return;
    read();
  }
}

}  // namespace llmp_hip

#endif  // LLMP_AMD_CSRC_VECQ_SORTED_WALK_H_

// llmp.vecq over Q4_K rows sorted by expert (a routed-expert layer over a prompt chunk): the sub-blocks' dot products
// on v_mfma_f32_32x32x16_f16, rows of up to eight super-blocks.
//
// The arithmetic is that of vecq_mma.hip's Q4_K form: sc_g * q and the tokens' codes are exact in F16, a sub-block's
// sum of their products is an integer below 2^24, exact in F32, and what is left a (token, row, sub-block) is one fma by
// the token's block scale d8:
//   main = P_0 * d8_0, then fma(P_g, d8_g, main);  out = fma(minimums, -dmin, fma(main, d, out)), super-blocks in order.
// The minimums, the sum over g of m_g * (d8_g * sum of the token's codes), come from two v_mfma_f32_32x32x16_bf16 a
// super-block: m_g is exact in bf16, and the F32 factor (11 bits of d8 times 12 of the sum) is the sum of its three
// leading groups of eight bits, each a bf16, so the products are exact and only their sum rounds, in F32.
//
// What bounds the form is vector instructions (a wave's matrix instruction occupies the vector unit for a quarter to a
// half of its own time, the rest overlaps), so the tile is chosen for few of them a weight:
//   - 32 rows (with a GLU 16 of the up matrix and the same 16 of the gate, which meet in a lane's registers r and
//     r + 8) by 32 tokens: two lanes share a row, so they decode its header twice, not four times;
//   - the two halves of K of an instruction are the low and the high 16 bytes of each 32-byte pair of sub-blocks, so a
//     lane's loads (16 bytes a pair) are its operands as they lie and the row's lanes exchange nothing;
//   - a nibble is never made a float: under a mask, bits 0 .. 3 or 4 .. 7 of a half are the F16 subnormals q * 2^-24 and
//     q * 2^-20, and one packed product by sc * 2^5 (2^1 for the high nibbles) gives sc * q * 2^-19, exact (the
//     matrix cores take subnormal operands as they are); the 2^19 is in the row's scale d;
//   - the row scales reach the result's layout (rows 8 (i / 4) + 4 (lane / 32) + i % 4) through LDS, not by F32 matrix
//     instructions, which overlap with nothing.
// About 375 vector instructions for 32 rows x 256 values x 32 tokens, 560 for 64 tokens: a pass takes up to 64 tokens where
// their operands fit LDS (rows of up to four super-blocks), else 32. Three waves a SIMD at 32 tokens, two at 64, by their
// registers; a wave takes the workgroup's next tile when it is done with one, since of a SIMD's waves the older get more.
//
// Measured, 512 tokens of top 8 of 128 experts (about 32 rows an expert, 46 % of the experts a second pass), against the
// 16 x 16 form of vecq_mma.hip: gate/up 2048 -> 2 x 768 with SwiGLU 125 -> 95 us, down 768 -> 2048 68 -> 48 us; 2 rows an
// expert 66 -> 59 us (226 MB of weights); against F64 the error of gate/up 2.5e-7 -> 1.7e-7, of down 1.2e-7 -> 9.3e-8. A
// super-block's step takes 1.0 us of a SIMD at the 1.95 GHz that it runs at under this load (2000 cycles of which the
// vector instructions are 1600), so gate/up is 72 us of steps, 7 us before the first one and the waits at a segment's end
// for its last tiles. Weights from L2 (one expert's for all) take 13 us off.
// Measured and not kept: a wave a super-block of a tile with its tokens in registers, the eight meeting in LDS (at a barrier
// a round 97.6 us, by counters a round ahead of each other 95.5-99, with loads two rounds ahead 100: the meeting costs what
// the segments' ends do here).

#include <hip/hip_runtime.h>

#include "common.h"
#include "llmp_hip.h"
#include "vecq_common.h"
#include "vecq_q4k_part.h"
#include "vecq_sorted_walk.h"

namespace llmp_hip {
namespace {

constexpr int kTokens = 32;  // a token group: the instruction's columns
constexpr size_t kLdsMost = 160 * 1024 - 2048;
constexpr float kLift = 524288.0f;  // 2^19

typedef float V16f __attribute__((ext_vector_type(16)));
typedef _Float16 H2 __attribute__((ext_vector_type(2)));
typedef _Float16 H8 __attribute__((ext_vector_type(8)));

// The staged tokens: TG groups of 32, in operand layout, a super-block after the other.
//   codes   [sub-block][half of its K steps][K half][token] 16 bytes: eight codes as F16, a dword's in the order 0, 2, 1, 3;
//   d8      [four sub-blocks][token] 16 bytes;
//   sums    [leading, middle, last eight bits, zeros][token] 16 bytes: d8_g * sum(codes) of the eight sub-blocks as bf16.
template <int TG>
struct Staged {
  static constexpr int kWaves = TG == 1 ? 12 : 8;  // a workgroup's: what the registers of a SIMD hold
  static constexpr int kGroup = kWaves * kWave;
  static constexpr int T = TG * kTokens;
  static constexpr int kStep = 2 * T * 16;       // a K step of 16 values
  static constexpr int kBlock = 2 * kStep;       // a sub-block
  static constexpr int kCodes = 8 * kBlock;      // a super-block's codes
  static constexpr int kScales = 2 * T * 16;
  static constexpr int kSums = 4 * T * 16;
  static constexpr int kAll = kCodes + kScales + kSums;
  static constexpr size_t Bytes(int nsb) { return static_cast<size_t>(nsb) * kAll + kWaves * kWave * 4; }
};

// A lane's part of one super-block of its row: the header and its 16 bytes of each pair of sub-blocks.
struct HalfPart {
  U32x4 header;
  U32x4 q[4];
};

// The sums exist from here on: the compiler would otherwise put their additions off to the tile's end and hold every
// product's result until then.
__device__ __forceinline__ void Here(V16f& v) { asm volatile("" : "+v"(v)); }

__device__ __forceinline__ H2 Both(float v) {
  const _Float16 h = static_cast<_Float16>(v);
  return H2{h, h};
}

// Two F16 from two bytes of `word`, each 1024 + the byte.
__device__ __forceinline__ H2 Biased(uint32_t word, uint32_t places) {
  return __builtin_bit_cast(H2, __builtin_amdgcn_perm(0x64646464u, word, places));
}

// The operand of one K step: two dwords' low or high nibbles, times the sub-block's scale.
__device__ __forceinline__ H8 Weights(uint32_t w0, uint32_t w1, uint32_t mask, H2 scale) {
  auto half = [&](uint32_t bits) { return __builtin_bit_cast(H2, bits & mask) * scale; };
  const H2 a = half(w0), b = half(w0 >> 8), c = half(w1), d = half(w1 >> 8);
  return __builtin_shufflevector(__builtin_shufflevector(a, b, 0, 1, 2, 3), __builtin_shufflevector(c, d, 0, 1, 2, 3), 0, 1, 2, 3,
                                 4, 5, 6, 7);
}

// The scale of sub-block g in both halves: 1024 + sc, less 1024, times 2^5 (2 for the high nibbles, 16 q in place).
__device__ __forceinline__ H2 Scale(const Q4KHeader& h, int g) {
  const uint32_t at = g & 3;
  const H2 biased = Biased(h.sc[g >> 2], 0x04000400u | at | (at << 16));
  return g % 2 == 0 ? __builtin_elementwise_fma(biased, Both(32.0f), Both(-32768.0f))
                    : __builtin_elementwise_fma(biased, Both(2.0f), Both(-2048.0f));
}

// Eight codes (two dwords) as F16, a dword's in the order 0, 2, 1, 3: a code plus 128 is a byte, 1024 + 128 + code less 1152.
__device__ __forceinline__ U32x4 TokenCodes(uint32_t w0, uint32_t w1) {
  const uint32_t a = w0 ^ 0x80808080u, c = w1 ^ 0x80808080u;
  constexpr uint32_t k02 = 0x04020400u, k13 = 0x04030401u;
  U32x4 packed;
  packed.x = __builtin_bit_cast(uint32_t, Biased(a, k02) - Both(1152.0f));
  packed.y = __builtin_bit_cast(uint32_t, Biased(a, k13) - Both(1152.0f));
  packed.z = __builtin_bit_cast(uint32_t, Biased(c, k02) - Both(1152.0f));
  packed.w = __builtin_bit_cast(uint32_t, Biased(c, k13) - Both(1152.0f));
  return packed;
}

// One Q8_1 block (sub-block g of super-block sb) of token t into the staged layout.
template <int TG>
__device__ __forceinline__ void StageBlock(const uint32_t (&w)[9], int t, int sb, int g, uint8_t* staged) {
  using L = Staged<TG>;
  uint8_t* to = staged + sb * L::kAll;
#pragma unroll
  for (int kg = 0; kg < 2; ++kg)
#pragma unroll
    for (int s = 0; s < 2; ++s)
      *reinterpret_cast<U32x4*>(to + g * L::kBlock + s * L::kStep + (kg * L::T + t) * 16) =
          TokenCodes(w[1 + 4 * kg + 2 * s], w[2 + 4 * kg + 2 * s]);
  int sum = 0;
#pragma unroll
  for (int i = 0; i < 8; ++i) sum = Dot4(0x01010101, static_cast<int>(w[1 + i]), sum);
  const float scale = HalfBitsToFloat(w[0] & 0xFFFFu);
  *reinterpret_cast<float*>(to + L::kCodes + ((g >> 2) * L::T + t) * 16 + (g & 3) * 4) = scale;
  const SumParts parts = SplitSum(scale, sum);
  uint16_t* sums = reinterpret_cast<uint16_t*>(to + L::kCodes + L::kScales + t * 16 + g * 2);
  sums[0] = static_cast<uint16_t>(parts.lead >> 16);
  sums[L::T * 8] = static_cast<uint16_t>(parts.middle >> 16);
  sums[2 * L::T * 8] = static_cast<uint16_t>(parts.last >> 16);
  sums[3 * L::T * 8] = 0;
}

// One super-block of a tile times the staged tokens of LIVE groups. `staged`: the super-block's; `lane_at`: 16 (lane % 32),
// this lane's token, `rows`: 64 floats of LDS, the wave's own.
template <int TG, int LIVE>
__device__ __forceinline__ void DotStep(const HalfPart& part, int kg, const uint8_t* staged, int lane_at, float* rows, int lane,
                                        V16f (&out)[TG]) {
  using L = Staged<TG>;
  const Q4KHeader h = DecodeQ4KHeader(part.header);
  // Row lane % 32's d and -dmin, at its place among 32 of each: the writes and reads of a wave's own LDS keep their order.
  rows[lane] = kg == 0 ? h.d * kLift : -h.dmin;
  {
    const B8 minimums = Minimums(h);
    const uint8_t* sums = staged + L::kCodes + L::kScales + kg * L::T * 16 + lane_at;
    const V16f zero = {};
    V16f low[LIVE];
#pragma unroll
    for (int tg = 0; tg < LIVE; ++tg) {
      const B8 lead = *reinterpret_cast<const B8*>(sums + tg * kTokens * 16);
      const B8 rest = *reinterpret_cast<const B8*>(sums + 2 * L::T * 16 + tg * kTokens * 16);
      low[tg] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(minimums, lead, zero, 0, 0, 0);
      low[tg] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(minimums, rest, low[tg], 0, 0, 0);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float4 s = *reinterpret_cast<const float4*>(rows + 32 + 8 * i + 4 * kg);
#pragma unroll
      for (int tg = 0; tg < LIVE; ++tg) {
        out[tg][4 * i] = fmaf(low[tg][4 * i], s.x, out[tg][4 * i]);
        out[tg][4 * i + 1] = fmaf(low[tg][4 * i + 1], s.y, out[tg][4 * i + 1]);
        out[tg][4 * i + 2] = fmaf(low[tg][4 * i + 2], s.z, out[tg][4 * i + 2]);
        out[tg][4 * i + 3] = fmaf(low[tg][4 * i + 3], s.w, out[tg][4 * i + 3]);
      }
    }
  }
#pragma unroll
  for (int tg = 0; tg < LIVE; ++tg) Here(out[tg]);
  __builtin_amdgcn_sched_barrier(0);
  V16f main[LIVE];
  float4 d8[LIVE];
#pragma unroll
  for (int p = 0; p < 4; ++p) {
    const H2 sc_lo = Scale(h, 2 * p), sc_hi = Scale(h, 2 * p + 1);
    const U32x4 q = part.q[p];
    const H8 lo0 = Weights(q.x, q.y, 0x000F000Fu, sc_lo), lo1 = Weights(q.z, q.w, 0x000F000Fu, sc_lo);
    const H8 hi0 = Weights(q.x, q.y, 0x00F000F0u, sc_hi), hi1 = Weights(q.z, q.w, 0x00F000F0u, sc_hi);
    const uint8_t* codes = staged + 2 * p * L::kBlock + kg * L::T * 16 + lane_at;
    const V16f zero = {};
#pragma unroll
    for (int tg = 0; tg < LIVE; ++tg) {
      const uint8_t* c = codes + tg * kTokens * 16;
      if (p % 2 == 0) d8[tg] = *reinterpret_cast<const float4*>(staged + L::kCodes + (p / 2) * L::T * 16 + tg * kTokens * 16 + lane_at);
      V16f a = __builtin_amdgcn_mfma_f32_32x32x16_f16(lo0, *reinterpret_cast<const H8*>(c), zero, 0, 0, 0);
      a = __builtin_amdgcn_mfma_f32_32x32x16_f16(lo1, *reinterpret_cast<const H8*>(c + L::kStep), a, 0, 0, 0);
      V16f b = __builtin_amdgcn_mfma_f32_32x32x16_f16(hi0, *reinterpret_cast<const H8*>(c + L::kBlock), zero, 0, 0, 0);
      b = __builtin_amdgcn_mfma_f32_32x32x16_f16(hi1, *reinterpret_cast<const H8*>(c + L::kBlock + L::kStep), b, 0, 0, 0);
      const float s0 = p % 2 == 0 ? d8[tg].x : d8[tg].z, s1 = p % 2 == 0 ? d8[tg].y : d8[tg].w;
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        main[tg][i] = p == 0 ? a[i] * s0 : fmaf(a[i], s0, main[tg][i]);
        main[tg][i] = fmaf(b[i], s1, main[tg][i]);
      }
      Here(main[tg]);
      if (LIVE > 1) __builtin_amdgcn_sched_barrier(0);
    }
    __builtin_amdgcn_sched_barrier(0);
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float4 s = *reinterpret_cast<const float4*>(rows + 8 * i + 4 * kg);
#pragma unroll
    for (int tg = 0; tg < LIVE; ++tg) {
      out[tg][4 * i] = fmaf(main[tg][4 * i], s.x, out[tg][4 * i]);
      out[tg][4 * i + 1] = fmaf(main[tg][4 * i + 1], s.y, out[tg][4 * i + 1]);
      out[tg][4 * i + 2] = fmaf(main[tg][4 * i + 2], s.z, out[tg][4 * i + 2]);
      out[tg][4 * i + 3] = fmaf(main[tg][4 * i + 3], s.w, out[tg][4 * i + 3]);
    }
  }
}

// grid: a workgroup a compute unit, sharing the passes of all experts (WalkSortedRows, kWhole too); a wave a tile of 32 rows (with a
// GLU 16 of each matrix) and all of K, the workgroup's waves consecutive tiles. LDS: the staged tokens, the waves' row scales.
template <bool kGlu, int TG, bool kWhole>
__global__ __launch_bounds__(Staged<TG>::kGroup, 1) void VecQSorted(const VecQArgs a) {
  using L = Staged<TG>;
  constexpr int kWaves = L::kWaves, kGroup = L::kGroup;
  constexpr int kRows = kGlu ? 16 : 32;
  constexpr int kAhead = TG == 1 ? 3 : 4;  // blocks a thread holds in registers between their loads and their staging
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
  __shared__ int next_tile;

  const llmp_vecq_desc& d = a.d;
  const int tid = threadIdx.x;
  const int lane = tid & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int nsb = d.ncols_x / 256;
  float* rows = reinterpret_cast<float*>(lds + nsb * L::kAll) + wave * kWave;
  const int kg = lane >> 5, row_in_tile = lane & 31;
  const int lane_at = row_in_tile * 16;
  const int tiles = (d.nrows + kRows - 1) / kRows;
  const uint8_t* matrix = static_cast<const uint8_t*>(kGlu && row_in_tile >= 16 ? d.g : d.w);
  const bool wide = reinterpret_cast<uintptr_t>(d.dst) % 16 == 0 && d.dst_token % 4 == 0;
  bool staged_before = false;

  auto run = [&](const SortedSegment& seg) {
    const int live = seg.m <= kTokens ? 1 : TG;
    const int last_tile = seg.group_first + seg.group_count - 1;
    const int first_row = seg.rows_first + seg.first;
    if (staged_before) __syncthreads();  // the last segment's readers of the staged tokens
    staged_before = true;
    if (tid == 0) next_tile = seg.group_first + kWaves;

    // The tokens' blocks are asked for before the weights (loads return in order, and the tokens are needed whole before
    // the first step), staged after the first weights are. Eight consecutive threads hold the same block of eight
    // consecutive tokens, whose 16-byte pieces lie side by side in LDS. Where a wave has no second tile the staging is much
    // of the segment, and only eights of tokens that hold rows are staged (1536 -> 512, four rows of each of 64 experts 17.6
    // -> 16.6 us; with more tiles nothing gained: 1536 -> 2 x 4096, two rows of 128, 190 us, 195 so); the columns past those
    // are what LDS held: a result's column is its own operand column's, and theirs are dropped.
    const bool few = seg.group_count <= kWaves;
    const int eights_log = few && seg.m <= 8 ? 0 : few && seg.m <= 16 ? 1 : live == 1 ? 2 : 3;
    const int staged = nsb << (6 + eights_log);
    auto place = [&](int index, int* t, int* b) {
      const int rest = index >> 6;
      const int sb = rest >> eights_log;
      *t = (rest - (sb << eights_log)) * 8 + (index & 7);
      *b = sb * 8 + ((index >> 3) & 7);
    };
    auto fetch_block = [&](int t, int b, uint32_t(&w)[9]) {
      // Tokens past m repeat the last: computed and dropped.
      const int r = first_row + min(t, seg.m - 1);
      const int64_t y_row = a.rows != nullptr ? a.rows[r] : r;
      const uint32_t* src = reinterpret_cast<const uint32_t*>(static_cast<const uint8_t*>(d.y) + (y_row * d.y_token + b) * kQ8Block);
#pragma unroll
      for (int i = 0; i < 9; ++i) w[i] = src[i];
    };
    uint32_t held[kAhead][9];
#pragma unroll
    for (int it = 0; it < kAhead; ++it) {
      const int index = tid + it * kGroup;
      if (index < staged) {
        int t, b;
        place(index, &t, &b);
        fetch_block(t, b, held[it]);
      }
    }
    __builtin_amdgcn_sched_barrier(0);

    const uint8_t* expert = matrix + static_cast<int64_t>(seg.expert) * d.stride_expert * 144 + 16 * kg;
    const uint8_t* row = nullptr;
    int fetch_tile = seg.group_first + wave, fetch_sb = 0;
    auto aim = [&]() {
      const int r = min(min(fetch_tile, last_tile) * kRows + (row_in_tile & (kRows - 1)), d.nrows - 1);
      row = expert + static_cast<int64_t>(r) * d.stride_row * 144;
    };
    // Queued here and no later. A wave's next tile is the next that no wave has begun: of a SIMD's waves the older get
    // more of it. Past the segment's end its last tile again: a load under a branch would make every wait for loads a
    // wait for all of them.
    auto fetch = [&](HalfPart& part) {
      if (fetch_sb == nsb) {
        fetch_sb = 0;
        int taken = 0;
        if (lane == 0) taken = atomicAdd(&next_tile, 1);
        fetch_tile = __builtin_amdgcn_readfirstlane(taken);
        aim();
      }
      const uint8_t* at = row + fetch_sb * 144;
      part.header = *reinterpret_cast<const U32x4*>(at - 16 * kg);
#pragma unroll
      for (int p = 0; p < 4; ++p) part.q[p] = *reinterpret_cast<const U32x4*>(at + 16 + 32 * p);
      __builtin_amdgcn_sched_barrier(0);
      ++fetch_sb;
    };
    HalfPart even, odd;
    aim();
    fetch(even);

#pragma unroll
    for (int it = 0; it < kAhead; ++it) {
      const int index = tid + it * kGroup;
      if (index < staged) {
        int t, b;
        place(index, &t, &b);
        StageBlock<TG>(held[it], t, b >> 3, b & 7, lds);
      }
    }
    for (int index = tid + kAhead * kGroup; index < staged; index += kGroup) {
      int t, b;
      place(index, &t, &b);
      uint32_t w[9];
      fetch_block(t, b, w);
      StageBlock<TG>(w, t, b >> 3, b & 7, lds);
    }
    __syncthreads();

    V16f out[TG];
#pragma unroll
    for (int tg = 0; tg < TG; ++tg) out[tg] = V16f{};
    int tile = seg.group_first + wave, sb = 0;
    auto finish = [&]() {
      const int row0 = tile * kRows;
#pragma unroll
      for (int tg = 0; tg < TG; ++tg) {
        const int t = tg * kTokens + row_in_tile;
        if (t < seg.m) {
          float* dst = d.dst + static_cast<int64_t>(first_row + t) * d.dst_token;
#pragma unroll
          for (int i = 0; i < kRows / 2; i += 4) {
            const int r = row0 + 2 * i + 4 * kg;  // four consecutive rows
            float v[4];
#pragma unroll
            for (int q = 0; q < 4; ++q)
              v[q] = kGlu ? Glu(d.glu, out[tg][i + q + (kGlu ? 8 : 0)], out[tg][i + q], d.limit) : out[tg][i + q];
            if (wide && r + 4 <= d.nrows) {
              *reinterpret_cast<float4*>(dst + r) = make_float4(v[0], v[1], v[2], v[3]);
            } else {
#pragma unroll
              for (int q = 0; q < 4; ++q)
                if (r + q < d.nrows) dst[r + q] = v[q];
            }
          }
        }
        out[tg] = V16f{};
      }
    };
    auto step = [&](const HalfPart& part) {
      const uint8_t* at = lds + sb * L::kAll;
      if (TG == 1 || live == TG) {
        DotStep<TG, TG>(part, kg, at, lane_at, rows, lane, out);
      } else {
        DotStep<TG, 1>(part, kg, at, lane_at, rows, lane, out);
      }
      if (++sb == nsb) {
        finish();
        sb = 0;
        tile = fetch_tile;  // that of the next step, asked for before this one
      }
    };
    while (tile <= last_tile) {
      fetch(odd);
      step(even);
      if (tile > last_tile) break;
      fetch(even);
      step(odd);
    }
  };

  // A step of one and of two live token groups takes 1.0 and 1.6 us of a SIMD, a staging 4 to 5 us of the workgroup and the
  // wait for the last segment's tiles before it as much again: in units of a fifth of a step, four SIMDs' of which pass at a
  // time. (With the staging alone, half of it: 1024 -> 2 x 768 of 64 experts 46 -> 42.5 us, 1536 -> 2 x 768 60 -> 57.4, 768 ->
  // 2048 of 128 experts 49.6 -> 48.3; half as much again is no better.)
  auto cost_of = [nsb](int m) { return nsb * (m <= kTokens ? 5 : 8); };
  auto fixed_of = [nsb](int m) { return 110 + 10 * nsb * (m <= kTokens ? 1 : TG); };
  WalkSortedRows<kWhole>(a.offsets, d.used, tiles, TG * kTokens, fixed_of, cost_of, run);
}

template <bool kGlu, int TG, bool kWhole>
void LaunchOne(const VecQArgs& a, int workgroups, hipStream_t stream) {
  static bool sized = false;
  if (!AllowLds(reinterpret_cast<const void*>(&VecQSorted<kGlu, TG, kWhole>), static_cast<int>(kLdsMost), &sized)) return;
  hipLaunchKernelGGL((VecQSorted<kGlu, TG, kWhole>), dim3(static_cast<unsigned>(workgroups)), dim3(Staged<TG>::kGroup),
                     Staged<TG>::Bytes(a.d.ncols_x / 256), stream, a);
}

}  // namespace

bool SortedTakes(int type, const llmp_vecq_desc& d) {
  return type == LLMP_TYPE_Q4_K && Staged<1>::Bytes(d.ncols_x / 256) <= kLdsMost;
}

template <bool kWhole>
void LaunchShape(const VecQArgs& a, int workgroups, hipStream_t stream) {
  const bool wide = Staged<2>::Bytes(a.d.ncols_x / 256) <= kLdsMost;
  if (a.d.g != nullptr) {
    wide ? LaunchOne<true, 2, kWhole>(a, workgroups, stream) : LaunchOne<true, 1, kWhole>(a, workgroups, stream);
  } else {
    wide ? LaunchOne<false, 2, kWhole>(a, workgroups, stream) : LaunchOne<false, 1, kWhole>(a, workgroups, stream);
  }
}

void LaunchSorted(const VecQArgs& a, int workgroups, hipStream_t stream) {
  // Up to sixteen tiles, a wave's one or two, the passes may have workgroups of their own (WalkSortedRows); with more that
  // evens out too little, and to look for it cost every launch 0.7 to 0.9 us.
  const int tiles = a.d.g != nullptr ? (a.d.nrows + 15) / 16 : (a.d.nrows + 31) / 32;
  tiles <= 16 ? LaunchShape<true>(a, workgroups, stream) : LaunchShape<false>(a, workgroups, stream);
}

}  // namespace llmp_hip

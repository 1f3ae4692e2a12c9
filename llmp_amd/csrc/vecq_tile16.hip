// llmp.vecq over Q4_K rows for 9 to 16 tokens of a dense or grouped product: sub-blocks' dot products on
// v_mfma_i32_16x16x32_i8, a super-block of 16 rows a wave.
//
// The token operand is a sub-block's Q8_1 codes as they are, the weight operand its nibbles under a mask: an instruction's
// result is the exact int32 sum of a sub-block for 16 rows and 16 tokens. The tokens are the instruction's first operand, so
// a lane keeps row lane % 16 and tokens 4 (lane / 16) + q: its row's 6-bit scales and d are its own registers, and what is
// left a (token, row, sub-block) is a conversion, the exact product sc * d8 and one fma:
//   main = P_0 * (sc_0 d8_0), then fma(P_g, sc_g d8_g, main);  out = fma(main, d, fma(minimums, -dmin, out)).
// The minimums come from one v_mfma_f32_16x16x32_bf16 a super-block: m_g is exact in bf16, d8_g * sum(codes) is the sum of
// three of them, one a K group (SplitSum). About 175 vector instructions for 16 rows x 256 values, whatever the tokens.
//
// A workgroup takes 1, 2, 4 or 8 tiles of 16 rows at a time, its sixteen waves the tiles' super-blocks (and, with a GLU,
// both matrices') in turn; a tile's waves meet in LDS. So a matrix of few long rows still gives every SIMD four waves, each
// with two super-blocks on their way while it multiplies a third. The tokens are staged once a workgroup (a span of the
// super-blocks at a time where they do not fit LDS whole).
//
// What bounds it is the vector unit and the loads' issue: with the weights in the Infinity Cache the gate/up pair below
// takes two microseconds less. HBM traffic is 1.01 of the weights. Measured, 9 and 16 tokens, against what was the default:
// 3840 -> 2 x 15360 with GeGLU 27.2 / 28.1 -> 22.3 / 23.2 us, 15360 -> 3840 28.5 / 35.2 -> 16.8 / 22.1, 4096 -> 4096
// 15.4 / 15.9 -> 8.2 / 9.6, 2048 -> 2 x 8192 22.8 / 22.7 -> 10.1 / 10.4, 1024 -> 4096 8.4 / 8.6 -> 5.4 / 5.5. Error against
// F64 1.2e-7 (1.4e-7 in the row-a-lane form, 2.4e-7 in the 16 x 16 form).
// Measured and not kept: up to eight tokens with a pair of sub-blocks in one v_mfma_i32_16x16x64_i8, a token's first and
// second sub-blocks in rows 0 to 7 and 8 to 15 (134 vector instructions; 15360 -> 3840 at 6 tokens 18.3 -> 14.3 us, but at 4
// 11.4 -> 13.4, and a token's bits are the same from two to eight); the tokens' rows through LDS as they lie and out of it
// again (whole lines a load, but two more meetings of sixteen waves: 3 us more).

#include <hip/hip_runtime.h>

#include "common.h"
#include "llmp_hip.h"
#include "vecq_common.h"
#include "vecq_q4k_part.h"

namespace llmp_hip {
namespace {

constexpr int kWaves = 16;
constexpr int kGroup = kWaves * kWave;
constexpr int kRows = 16;
constexpr int kMostTiles = 8;                     // of a workgroup at a time
constexpr int kPartBytes = kWaves * kWave * 16;   // the waves' sums
constexpr int64_t kLdsMost = 160 * 1024 - 2048;
constexpr int kDepth = 3;                         // weight buffers

typedef int V4i __attribute__((ext_vector_type(4)));
typedef float V4f __attribute__((ext_vector_type(4)));

struct Tile16Plan {
  int tiles;  // a workgroup's at a time
  int span;   // steps whose tokens are staged at a time
  int parts;  // buffers of the waves' sums: two where a workgroup takes tiles more than once
};

// The staged tokens of a super-block: codes [sub-block][K group][token] 8 bytes; d8 [sub-block][tokens rounded up to fours]
// floats; the bf16 parts of d8 * sum(codes) [leading, middle, last, zeros][token] 16 bytes, sub-block g at 2 g.
__host__ __device__ inline int TokensInFours(int tokens) { return (tokens + 3) & ~3; }
__host__ __device__ inline int StagedBytes(int tokens) { return 320 * tokens + 32 * TokensInFours(tokens); }

// Sub-blocks g and g + 1 (g even) of token t.
__device__ __forceinline__ void StageBlocks(const uint32_t (&w)[18], int t, int g, int tokens, uint8_t* to) {
  const int fours = TokensInFours(tokens);
  uint32_t sums[2][3];
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    // (A sub-block's K groups are rotated by its pair's number: consecutive threads' writes then lie in different banks.)
#pragma unroll
    for (int kg = 0; kg < 4; ++kg)
      *reinterpret_cast<uint2*>(to + (((g + j) * 4 + ((kg + (g >> 1)) & 3)) * tokens + t) * 8) =
          make_uint2(w[9 * j + 1 + 2 * kg], w[9 * j + 2 + 2 * kg]);
    int sum = 0;
#pragma unroll
    for (int i = 0; i < 8; ++i) sum = Dot4(0x01010101, static_cast<int>(w[9 * j + 1 + i]), sum);
    const float scale = HalfBitsToFloat(w[9 * j] & 0xFFFFu);
    *reinterpret_cast<float*>(to + 256 * tokens + ((g + j) * fours + t) * 4) = scale;
    const SumParts parts = SplitSum(scale, sum);
    sums[j][0] = parts.lead, sums[j][1] = parts.middle, sums[j][2] = parts.last;
  }
  uint8_t* at = to + 256 * tokens + 32 * fours + t * 16 + g * 2;
#pragma unroll
  for (int i = 0; i < 3; ++i)
    *reinterpret_cast<uint32_t*>(at + i * tokens * 16) = __builtin_amdgcn_perm(sums[1][i], sums[0][i], 0x07060302u);
  *reinterpret_cast<uint32_t*>(at + 3 * tokens * 16) = 0;
}

// A lane's places in a super-block's staged tokens.
struct Places {
  int codes[4], d8, sums;  // codes: by the pair of sub-blocks
};

// A super-block of 16 rows times the staged tokens.
__device__ __forceinline__ void DotStep(const RowPart& loaded, const uint8_t* staged, const Places& at, int tokens, V4f& out) {
  RowPart part = loaded;
  Transpose(part);
  const Q4KHeader h = DecodeQ4KHeader(part.header);
  const V4f zero = {0.0f, 0.0f, 0.0f, 0.0f};
  const V4i none = {0, 0, 0, 0};
  const V4f low = __builtin_amdgcn_mfma_f32_16x16x32_bf16(*reinterpret_cast<const B8*>(staged + at.sums), Minimums(h), zero, 0, 0, 0);
  const int fours = TokensInFours(tokens);
  V4f main = zero;
#pragma unroll
  for (int g = 0; g < 8; ++g) {
    const uint2 q = part.q[g >> 1];
    const uint32_t w0 = (g % 2 == 0 ? q.x : q.x >> 4) & 0x0F0F0F0Fu, w1 = (g % 2 == 0 ? q.y : q.y >> 4) & 0x0F0F0F0Fu;
    const int64_t weights = static_cast<int64_t>((static_cast<uint64_t>(w1) << 32) | w0);
    const int64_t codes = *reinterpret_cast<const int64_t*>(staged + g * 32 * tokens + at.codes[g >> 1]);
    const V4i sums = __builtin_amdgcn_mfma_i32_16x16x32_i8(codes, weights, none, 0, 0, 0);
    const float4 d8 = *reinterpret_cast<const float4*>(staged + g * fours * 4 + at.d8);
    const float sc = static_cast<float>((h.sc[g >> 2] >> (8 * (g & 3))) & 0xFFu);
    main[0] = fmaf(static_cast<float>(sums[0]), sc * d8.x, main[0]);
    main[1] = fmaf(static_cast<float>(sums[1]), sc * d8.y, main[1]);
    main[2] = fmaf(static_cast<float>(sums[2]), sc * d8.z, main[2]);
    main[3] = fmaf(static_cast<float>(sums[3]), sc * d8.w, main[3]);
  }
#pragma unroll
  for (int q = 0; q < 4; ++q) out[q] = fmaf(main[q], h.d, fmaf(low[q], -h.dmin, out[q]));
  asm volatile("" : "+v"(out));  // here, not at the tile's end with every operand kept until then
}

// grid (workgroups, slots).
template <bool kGlu>
__global__ __launch_bounds__(kGroup, 1) void VecQTile16(const VecQArgs a, const Tile16Plan plan) {
  constexpr int kMatrices = kGlu ? 2 : 1;
  constexpr int kAhead = 2;  // pairs of blocks a thread holds in registers between their loads and their staging
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
  const llmp_vecq_desc& d = a.d;
  const int tid = threadIdx.x;
  const int lane = tid & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int nsb = d.ncols_x / 256, tokens = d.tokens, slot = blockIdx.y;
  const int staged_bytes = StagedBytes(tokens), fours = TokensInFours(tokens);
  float* const parts = reinterpret_cast<float*>(lds);
  uint8_t* const staged = lds + plan.parts * kPartBytes;

  const int tile_waves = kWaves / plan.tiles;        // of a tile
  const int step_blocks = tile_waves / kMatrices;    // super-blocks of a row a step
  const int tile_in_round = wave / tile_waves, unit = wave - tile_in_round * tile_waves;
  const int sb_first = unit / kMatrices;
  const int steps = (nsb + step_blocks - 1) / step_blocks;  // a tile's
  const int tiles = (d.nrows + kRows - 1) / kRows;
  const int rounds = (tiles + plan.tiles - 1) / plan.tiles;
  const int mine = (rounds - static_cast<int>(blockIdx.x) + static_cast<int>(gridDim.x) - 1) / static_cast<int>(gridDim.x);
  const int total = mine * steps;
  const int row_in_tile = lane & 15, kg = lane >> 4;

  // Tokens past the last repeat it: computed and dropped.
  Places at;
  const int token = min(row_in_tile, tokens - 1);
#pragma unroll
  for (int p = 0; p < 4; ++p) at.codes[p] = (((kg + p) & 3) * tokens + token) * 8;
  at.d8 = 256 * tokens + min(kg, fours / 4 - 1) * 16;
  at.sums = 256 * tokens + 32 * fours + (kg * tokens + token) * 16;
  const uint8_t* const y = static_cast<const uint8_t*>(d.y) + static_cast<int64_t>(slot) * d.y_slot * kQ8Block;

  // Pair of blocks `index` of a span: consecutive threads take the tokens of one pair, then the next pair.
  auto fetch_blocks = [&](int index, int span_first, uint32_t(&words)[18]) {
    const int b = index / tokens, t = index - b * tokens;
    const uint32_t* src = reinterpret_cast<const uint32_t*>(y + (static_cast<int64_t>(t) * d.y_token + span_first * 8 + 2 * b) * kQ8Block);
#pragma unroll
    for (int i = 0; i < 18; ++i) words[i] = src[i];
  };
  auto stage_blocks = [&](int index, const uint32_t(&words)[18]) {
    const int b = index / tokens, t = index - b * tokens;
    StageBlocks(words, t, 2 * (b & 3), tokens, staged + (b >> 2) * staged_bytes);
  };
  const int span_blocks = plan.span * step_blocks;  // super-blocks of a span
  uint32_t held[kAhead][18];
  const int first_staged = min(span_blocks, nsb) * 4 * tokens;
#pragma unroll
  for (int it = 0; it < kAhead; ++it)
    if (tid + it * kGroup < first_staged) fetch_blocks(tid + it * kGroup, 0, held[it]);
  __builtin_amdgcn_sched_barrier(0);

  const uint8_t* const matrix = static_cast<const uint8_t*>(kGlu && (unit & 1) ? d.g : d.w) +
                                static_cast<int64_t>(slot) * d.stride_expert * 144;
  const uint8_t* row = nullptr;
  int fetch_round = blockIdx.x, fetch_step = 0, fetched = 0;
  auto aim = [&]() {
    const int r = min((fetch_round * plan.tiles + tile_in_round) * kRows + row_in_tile, d.nrows - 1);
    row = matrix + static_cast<int64_t>(r) * d.stride_row * 144;
  };
  // Queued here and no later. Past the row's and the workgroup's end the last again: a load under a branch would make every
  // wait for loads a wait for all of them.
  auto fetch = [&](RowPart& part) {
    part = LoadRowPart(row, min(sb_first + fetch_step * step_blocks, nsb - 1), kg);
    __builtin_amdgcn_sched_barrier(0);
    if (++fetched < total && ++fetch_step == steps) {
      fetch_step = 0;
      fetch_round += gridDim.x;
      aim();
    }
  };
  RowPart buffer[kDepth];
  aim();
#pragma unroll
  for (int j = 0; j < kDepth - 1; ++j) fetch(buffer[j]);

#pragma unroll
  for (int it = 0; it < kAhead; ++it)
    if (tid + it * kGroup < first_staged) stage_blocks(tid + it * kGroup, held[it]);
  auto stage = [&](int from, int span_first) {
    const int count = min(span_blocks, nsb - span_first) * 4 * tokens;
    for (int index = from; index < count; index += kGroup) {
      uint32_t words[18];
      fetch_blocks(index, span_first, words);
      stage_blocks(index, words);
    }
  };
  stage(tid + kAhead * kGroup, 0);
  __syncthreads();

  V4f out = {0.0f, 0.0f, 0.0f, 0.0f};
  int round = blockIdx.x, step = 0, part_at = 0;
  auto finish = [&]() {
    *reinterpret_cast<V4f*>(parts + part_at + (wave * kWave + lane) * 4) = out;
    out = V4f{0.0f, 0.0f, 0.0f, 0.0f};
    __syncthreads();
    for (int i = tid; i < plan.tiles * kRows * 16; i += kGroup) {
      const int r = i & 15, t = (i >> 4) & 15, tile = i >> 8;
      const int to = (round * plan.tiles + tile) * kRows + r;
      if (t < tokens && to < d.nrows) {
        const float* from = parts + part_at + ((tile * tile_waves * kWave) + 16 * (t >> 2) + r) * 4 + (t & 3);
        float up = from[0], gate = kGlu ? from[kWave * 4] : 0.0f;
        for (int w = kMatrices; w < tile_waves; w += kMatrices) {
          up += from[w * kWave * 4];
          if constexpr (kGlu) gate += from[(w + 1) * kWave * 4];
        }
        d.dst[static_cast<int64_t>(t) * d.dst_token + static_cast<int64_t>(slot) * d.dst_slot + to] =
            kGlu ? Glu(d.glu, gate, up, d.limit) : up;
      }
    }
    // With two buffers whoever writes this one again has passed the other's barrier, after its readers.
    if (plan.parts == 2) part_at = kPartBytes / 4 - part_at;
  };
  auto advance = [&](const RowPart& part) {
    if (plan.span < steps && step % plan.span == 0 && step > 0) {
      __syncthreads();  // the last span's readers
      stage(tid, step * step_blocks);
      __syncthreads();
    }
    const int sb = sb_first + step * step_blocks;
    if (sb < nsb) DotStep(part, staged + (sb - step / plan.span * span_blocks) * staged_bytes, at, tokens, out);
    if (++step == steps) {
      finish();
      step = 0;
      round += gridDim.x;
    }
  };
  for (int s = 0; s < total; s += kDepth) {
#pragma unroll
    for (int j = 0; j < kDepth; ++j) {
      if (j == 0 || s + j < total) {
        fetch(buffer[(j + kDepth - 1) % kDepth]);
        advance(buffer[j]);
      }
    }
  }
}

int ComputeUnits() {
  static const int units = [] {
    const int cus = llmp_hip_compute_units();
    return cus > 0 ? cus : 256;
  }();
  return units;
}

// The super-blocks whose tokens fit LDS beside the sums.
int64_t Room(int tokens, int parts) { return (kLdsMost - parts * kPartBytes) / StagedBytes(tokens); }

// The tiles a workgroup takes at a time: those with the fewest steps of a wave, then the fewest. By the shape alone, as if
// there were sixteen tokens: the order of a row's sums, and so a token's bits, do not depend on the count. False: the tokens
// of a row fit LDS only a span at a time and a workgroup would stage them again for every tile.
bool PlanTile16(const llmp_vecq_desc& d, int cus, Tile16Plan* plan, int* workgroups) {
  const int nsb = d.ncols_x / 256, matrices = d.g != nullptr ? 2 : 1;
  const int tiles = (d.nrows + kRows - 1) / kRows;
  const int most = cus / d.used < 1 ? 1 : cus / d.used;
  int64_t best = 0;
  for (int at_once = 1; at_once <= kMostTiles; at_once *= 2) {
    const int step_blocks = kWaves / at_once / matrices;
    const int steps = (nsb + step_blocks - 1) / step_blocks;
    const int rounds = (tiles + at_once - 1) / at_once;
    const int groups = rounds < most ? rounds : most;
    const int64_t cost = static_cast<int64_t>((rounds + groups - 1) / groups) * steps;
    const int parts = rounds > groups ? 2 : 1;
    if (Room(16, parts) < nsb && rounds > groups) continue;
    if (best == 0 || cost < best) {
      best = cost;
      const int64_t room = Room(d.tokens, parts);  // 22 super-blocks at least, a step at most sixteen
      *plan = Tile16Plan{at_once, room >= nsb ? steps : static_cast<int>(room / step_blocks), parts};
      *workgroups = groups;
    }
  }
  return best != 0;
}

template <bool kGlu>
void LaunchOne(const VecQArgs& a, const Tile16Plan& plan, dim3 grid, hipStream_t stream) {
  static bool sized = false;
  if (!AllowLds(reinterpret_cast<const void*>(&VecQTile16<kGlu>), static_cast<int>(kLdsMost), &sized)) return;
  const int nsb = a.d.ncols_x / 256, step_blocks = kWaves / plan.tiles / (kGlu ? 2 : 1);
  const int held = plan.span * step_blocks < nsb ? plan.span * step_blocks : nsb;
  const size_t lds = static_cast<size_t>(plan.parts) * kPartBytes + static_cast<size_t>(held) * StagedBytes(a.d.tokens);
  hipLaunchKernelGGL((VecQTile16<kGlu>), grid, dim3(kGroup), lds, stream, a, plan);
}

}  // namespace

bool Tile16Takes(const llmp_vecq_desc& d) {
  Tile16Plan plan;
  int workgroups;
  return PlanTile16(d, ComputeUnits(), &plan, &workgroups);
}

void LaunchTile16(const VecQArgs& a, hipStream_t stream) {
  const llmp_vecq_desc& d = a.d;
  Tile16Plan plan;
  int workgroups;
  if (!PlanTile16(d, ComputeUnits(), &plan, &workgroups)) return;
  const dim3 grid(static_cast<unsigned>(workgroups), static_cast<unsigned>(d.used));
  d.g != nullptr ? LaunchOne<true>(a, plan, grid, stream) : LaunchOne<false>(a, plan, grid, stream);
}

}  // namespace llmp_hip

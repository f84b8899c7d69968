// MI355X (gfx950) construction of the resident ternary sketch.
//
// The reader's screen reads a sketch of every expert's gate/up rows: each
// rotated 128-coordinate block of a row is ternarised by the TWN rule and five
// rows' trits at one coordinate share a byte. The reference builds it with a
// torch loop over experts (calibration_free_moe/reader/sketch.py:84-150 of
// AidenGeunGeun/calibration-free-moe); this kernel builds the same format on
// the device in one launch per layer (cfmoe_build_sketch).
//
// Per (expert, row, block), in FP32:
//   v = blockdiag(H128)/sqrt(128) diag(signs) w   (sketch.py:38-50; the seven
//       butterfly stages pair coordinates c, c + w into (l + r, l - r), then
//       one multiply by fp32(1/sqrt(128)): the same operations in the same
//       order as the reference, so the rotated values are bit-identical)
//   keep = |v| > 0.7 * mean|v|, t = keep ? sign(v) : 0
//   scale = sum of kept |v| / max(kept, 1), residual = mean (v - t scale)^2
// Byte j = 2 g + plane of coordinate c packs channels 5 g .. 5 g + 4 of the
// gate (plane 0) or up (plane 1) rows as sum_d (t_d + 1) 3^d (= 121 +
// sum_d t_d 3^d; channels past the width count as zero trits). Bytes [0,
// body) of a coordinate sit at (b 128 + c) body, bytes [body, stride) at
// blocks 128 body + ((b / 2) 128 + c) 32 + (b % 2) 16. The FP16 statistics
// go to the physical [E, blocks, 2, 2 I] layout (scale plane, residual plane).
//
// The sums behind mean|v|, the scale and the residual are xor trees, not
// torch's reduction order: the threshold test can differ from a torch build
// only for |v| within an FP32 rounding of 0.7 mean|v|, and the FP16
// statistics only by a rounding.

#include <hip/hip_fp16.h>
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>
#include <type_traits>

#include "cfmoe_reader.h"

namespace cfmoe {

int fail(int code, const char *message);
int check_launch(const char *stage);
int code_stride(int rows);

namespace {

constexpr float kRotationScale = 0.08838834764831845f;  // fp32(1 / sqrt(128))

struct SketchArgs {
  const uint16_t *weights;  // [E, 2 I, H] bf16
  const int8_t *signs;      // [H] +-1, or NULL (unrotated blocks)
  uint8_t *codes;           // [E, storage]
  __half *stats;            // physical [E, blocks, 2, 2 I]
  long storage;
  int rows, width, hidden, blocks, groups, stride, body;
  int tiles;  // column tiles of a coordinate's code run
  int packs;  // workgroups over the blocks
};

// Loads and stores at the element's own alignment: callers' tensors may be
// views at any element offset (one wide access each all the same).
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef u32x4 row_words __attribute__((aligned(2)));
typedef u32x2 sign_words __attribute__((aligned(1)));
typedef uint32_t code_word __attribute__((aligned(1)));

// Eight lanes of a wave share one row's block: lane i of the eight holds the
// coordinates 8 y .. 8 y + 7 and 64 + 8 y .. 64 + 8 y + 7 with y = (i & 3) ^
// (i & 4 ? 7 : 0), so that the lanes whose y differ in bit 0, 1 or 2 are i ^ 1,
// i ^ 2 and i ^ 7: one DPP move each (two quad permutes, the half-row mirror).
constexpr int kRowLanes = 8;
constexpr int kLaneValues = 16;
constexpr int kExchange[3] = {0xb1, 0x4e, 0x141};

template <int kControl>
__device__ __forceinline__ float partner(float v) {
  // (bound_ctrl set: the move folds into the add that uses it)
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), kControl, 0xf, 0xf, true));
}

// Sum of a block's 128 values, every lane of the eight gets it: coordinates c
// and c + 64 first, then the xor tree over c's bits 0 .. 5 (the order of a
// 64-lane wave tree over lanes c that each hold c and c + 64).
__device__ __forceinline__ float block_total(const float (&v)[kLaneValues]) {
  float t[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) t[i] = v[i] + v[8 + i];
  float sum = ((t[0] + t[1]) + (t[2] + t[3])) + ((t[4] + t[5]) + (t[6] + t[7]));
  sum = sum + partner<kExchange[0]>(sum);
  sum = sum + partner<kExchange[1]>(sum);
  return sum + partner<kExchange[2]>(sum);
}

constexpr int kTileUnits = 64;  // code byte columns per workgroup, eight lanes each
constexpr int kTileThreads = kTileUnits * kRowLanes;
constexpr int kNarrowColumns = 16;

// Workgroup = (expert e, kColumns code byte columns, 64 / kColumns blocks),
// eight lanes per column of a block: the column's five rows (channels 5 g ..
// 5 g + 4 of one plane) are loaded together, each lane keeps the codes of its
// 16 coordinates in registers, and the tile's bytes and statistics leave
// through LDS as whole words. Every byte of the blocks' code rows is written
// (padding columns, and the missing half of an odd block count's last tail
// rows, hold 121).
//
// Bound by the vector unit (about 470 instructions per eight row blocks: 176
// of them the butterflies): a 128-expert layer of 1536 x 2048 rows takes 262
// us, 3.4 TB/s of its 898 MB, where the instructions alone take about 250. A
// wave per column with two coordinates per lane took 990 us, in single-byte
// stores `body` bytes apart, LDS exchanges for every butterfly and three
// 64-lane trees per row. A tile is 64 bytes of one block's columns because a
// coordinate's run then leaves as one 64-byte piece. Widths up to 40, whose
// runs are 16 bytes, take four blocks to a workgroup and number the columns
// that hold channels through them, so that waves are full down to a width of
// five (128 experts of H = 2048 at width 16: 13.9 us, 55 with one block's 64
// columns; 512 of H = 4096 at width 5: 59 and 405).
template <bool kRotate, int kColumns>
__global__ __launch_bounds__(kTileThreads) void build_sketch_kernel(SketchArgs a) {
  constexpr int kPack = kTileUnits / kColumns;  // blocks
  constexpr int kTileStride = kColumns + 4;     // LDS bytes per coordinate (bank spread)
  constexpr int kTileChannels = 5 * kColumns / 2;
  __shared__ __align__(16) uint8_t tile[kPack][128 * kTileStride];
  __shared__ __half tile_stats[kPack][2][2][kTileChannels];  // [block][plane][scale, residual][channel]
  const int tid = threadIdx.x;
  int item = blockIdx.x;
  const int block0 = item % a.packs * kPack;
  item /= a.packs;
  const int column0 = item % a.tiles * kColumns;
  const int e = item / a.tiles;
  // columns that hold channels (at least one: the run is 2 `groups` bytes
  // rounded up to 16); unit i of eight lanes is column i % columns of block i / columns
  const int columns = min(kColumns, 2 * a.groups - column0);
  const int unit = tid / kRowLanes;
  const int pack = kPack == 1 ? 0 : unit / columns, local = unit - pack * columns;
  const int b = min(block0 + pack, a.blocks - 1);
  const int j = column0 + local;
  const int plane = j & 1, g = j >> 1;
  const int i8 = tid % kRowLanes, y = (i8 & 3) ^ (i8 & 4 ? 7 : 0);
  const int base = b * 128;
  const bool live = unit < kPack * columns && block0 + pack < a.blocks;

  if (__ballot(live) != 0) {  // (waves past the last column's only store)
    u32x4 words[5][2];
    const uint16_t *rows = a.weights + (static_cast<long>(e) * a.rows + plane * a.width) * a.hidden + base + 8 * y;
#pragma unroll
    for (int d = 0; d < 5; ++d) {
      // (a channel past the width reads the last one; its trits stay zero)
      const long row = static_cast<long>(min(5 * g + d, a.width - 1)) * a.hidden;
      words[d][0] = *reinterpret_cast<const row_words *>(rows + row);
      words[d][1] = *reinterpret_cast<const row_words *>(rows + row + 64);
    }
    float sign[kLaneValues];
    if (kRotate) {
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const u32x2 s = *reinterpret_cast<const sign_words *>(a.signs + base + 64 * h + 8 * y);
#pragma unroll
        for (int i = 0; i < 8; ++i)
          sign[8 * h + i] = static_cast<float>(static_cast<int8_t>((i < 4 ? s.x : s.y) >> (8 * (i & 3))));
      }
    }
    // the upper half of a cross-lane butterfly subtracts: its own value negated
    uint32_t negate[3];
#pragma unroll
    for (int s = 0; s < 3; ++s) negate[s] = (y >> s) & 1 ? 0x80000000u : 0u;

    float code[kLaneValues];  // 121 + sum_d t_d 3^d
#pragma unroll
    for (int i = 0; i < kLaneValues; ++i) code[i] = 121.0f;
    float power = 1.0f;
#pragma unroll
    for (int d = 0; d < 5; ++d, power *= 3.0f) {
      float v[kLaneValues];
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          v[8 * h + 2 * i] = __uint_as_float(words[d][h][i] << 16);
          v[8 * h + 2 * i + 1] = __uint_as_float(words[d][h][i] & 0xffff0000u);
        }
      if (kRotate) {
#pragma unroll
        for (int i = 0; i < kLaneValues; ++i) v[i] = v[i] * sign[i];
        auto within = [&](int width) {  // coordinates of the lane's own registers
#pragma unroll
          for (int i = 0; i < kLaneValues; ++i) {
            if (i & width) continue;
            const float low = v[i], high = v[i + width];
            v[i] = low + high;
            v[i + width] = low - high;
          }
        };
        auto across = [&](auto stage) {  // the partner lane's
          constexpr int kStage = decltype(stage)::value;
#pragma unroll
          for (int i = 0; i < kLaneValues; ++i)
            v[i] = __uint_as_float(__float_as_uint(v[i]) ^ negate[kStage]) + partner<kExchange[kStage]>(v[i]);
        };
        within(1);
        within(2);
        within(4);
        across(std::integral_constant<int, 0>());
        across(std::integral_constant<int, 1>());
        across(std::integral_constant<int, 2>());
        within(8);  // coordinates 64 apart
#pragma unroll
        for (int i = 0; i < kLaneValues; ++i) v[i] = v[i] * kRotationScale;
      }
      float m[kLaneValues];
#pragma unroll
      for (int i = 0; i < kLaneValues; ++i) m[i] = fabsf(v[i]);
      const float threshold = 0.7f * (block_total(m) / 128.0f);
      int kept = 0;
      float kept_m[kLaneValues];
#pragma unroll
      for (int i = 0; i < kLaneValues; ++i) {
        kept += m[i] > threshold;
        kept_m[i] = m[i] > threshold ? m[i] : 0.0f;
      }
      kept += __builtin_amdgcn_mov_dpp(kept, kExchange[0], 0xf, 0xf, false);
      kept += __builtin_amdgcn_mov_dpp(kept, kExchange[1], 0xf, 0xf, false);
      kept += __builtin_amdgcn_mov_dpp(kept, kExchange[2], 0xf, 0xf, false);
      const float scale = block_total(kept_m) / static_cast<float>(max(kept, 1));
      // (v - t scale)^2 = (|v| - [kept] scale)^2
      float square[kLaneValues];
#pragma unroll
      for (int i = 0; i < kLaneValues; ++i) {
        const float r = m[i] - (m[i] > threshold ? scale : 0.0f);
        square[i] = r * r;
      }
      const float residual = block_total(square) / 128.0f;
      const bool inside = live && 5 * g + d < a.width;
      const float trit = inside ? power : 0.0f;
#pragma unroll
      for (int i = 0; i < kLaneValues; ++i)
        code[i] = code[i] + (m[i] > threshold ? copysignf(trit, v[i]) : 0.0f);
      if (i8 == 0 && live) {
        const int channel = 5 * (local >> 1) + d;
        tile_stats[pack][plane][0][channel] = __float2half_rn(scale);
        tile_stats[pack][plane][1][channel] = __float2half_rn(residual);
      }
      // (each row's codes are done before the next row begins: left to the end,
      // the five rows' kept masks would not fit the scalar registers)
#pragma unroll
      for (int i = 0; i < kLaneValues; ++i) asm volatile("" : "+v"(code[i]));
      __builtin_amdgcn_sched_barrier(0);
    }
    if (live)
#pragma unroll
      for (int i = 0; i < kLaneValues; ++i)
        tile[pack][(64 * (i >> 3) + 8 * y + (i & 7)) * kTileStride + local] =
            static_cast<uint8_t>(static_cast<int>(code[i]));
  }
  __syncthreads();

  // the tile's code words: bytes [0, body) of a coordinate in the block's
  // body, [body, stride) in its half of the block pair's tail row
  uint8_t *codes = a.codes + static_cast<long>(e) * a.storage;
  const long tails = static_cast<long>(a.blocks) * 128 * a.body;
  constexpr int kRunWords = kColumns / 4;
#pragma unroll
  for (int n = 0; n < kPack * 128 * kRunWords / kTileThreads; ++n) {
    const int at = tid + n * kTileThreads;
    const int p = at / (128 * kRunWords), block = block0 + p;
    const int c = at / kRunWords % 128, byte = 4 * (at % kRunWords), column = column0 + byte;
    if (column >= a.stride || block >= a.blocks) continue;
    uint32_t word = *reinterpret_cast<const uint32_t *>(&tile[p][c * kTileStride + byte]);
    // (columns past the last that holds channels: no unit wrote them)
    const int held = columns - byte;
    const uint32_t mask = held >= 4 ? 0xffffffffu : held <= 0 ? 0u : (1u << (8 * held)) - 1u;
    word = (word & mask) | (0x79797979u & ~mask);
    if (column < a.body) {
      *reinterpret_cast<code_word *>(codes + (static_cast<long>(block) * 128 + c) * a.body + column) = word;
    } else {
      const long row = tails + ((block / 2) * 128 + c) * 32 + (column - a.body);
      *reinterpret_cast<code_word *>(codes + row + (block % 2) * 16) = word;
      // (an odd block count's last tail rows have no second block)
      if (block % 2 == 0 && block + 1 == a.blocks) *reinterpret_cast<code_word *>(codes + row + 16) = 0x79797979u;
    }
  }
  __half *stats = a.stats + static_cast<long>(e) * a.blocks * 2 * a.rows;
  for (int at = tid; at < kPack * 4 * kTileChannels; at += kTileThreads) {
    const int p = at / (4 * kTileChannels), which = at / kTileChannels % 2, within = at % kTileChannels;
    const int channel_plane = at / (2 * kTileChannels) % 2;
    const int channel = 5 * (column0 / 2) + within;
    if (channel < a.width && block0 + p < a.blocks)
      stats[(static_cast<long>(block0 + p) * 2 + which) * a.rows + channel_plane * a.width + channel] =
          tile_stats[p][channel_plane][which][within];
  }
}

}  // namespace
}  // namespace cfmoe

extern "C" {

using namespace cfmoe;

CFMOE_API int cfmoe_build_sketch(int32_t experts, int32_t width, int32_t hidden,
                                 const void *gate_up, const int8_t *signs, uint8_t *codes,
                                 void *statistics, cfmoe_stream stream) {
  if (experts <= 0 || width <= 0 || hidden <= 0 || hidden % 128)
    return fail(CFMOE_EINVAL, "sketch needs experts, width > 0 and hidden a multiple of 128");
  if (!gate_up || !codes || !statistics) return fail(CFMOE_EINVAL, "NULL argument");
  SketchArgs a;
  a.weights = static_cast<const uint16_t *>(gate_up);
  a.signs = signs;
  a.codes = codes;
  a.stats = static_cast<__half *>(statistics);
  a.rows = 2 * width;
  a.width = width;
  a.hidden = hidden;
  a.blocks = hidden / 128;
  a.groups = (width + 4) / 5;
  a.stride = code_stride(a.rows);
  a.body = a.stride - a.stride % 32;
  const long tail = a.stride % 32 ? static_cast<long>((a.blocks + 1) / 2) * 128 * 32 : 0;
  a.storage = static_cast<long>(a.blocks) * 128 * a.body + tail;
  const bool narrow = a.stride <= kNarrowColumns;
  const int columns = narrow ? kNarrowColumns : kTileUnits, pack = kTileUnits / columns;
  a.tiles = (a.stride + columns - 1) / columns;
  a.packs = (a.blocks + pack - 1) / pack;
  // (a launch holds fewer than 2^32 threads: more experts than that take several)
  const long per_expert = static_cast<long>(a.tiles) * a.packs;
  const long most = 0xffffffffL / kTileThreads / per_expert;
  if (most < 1) return fail(CFMOE_EINVAL, "sketch has too many blocks for one launch");
  for (long first = 0; first < experts; first += most) {
    const unsigned items = static_cast<unsigned>(std::min<long>(most, experts - first) * per_expert);
    auto launch = [&](auto kernel) {
      hipLaunchKernelGGL(kernel, dim3(items), dim3(kTileThreads), 0, stream, a);
    };
    if (narrow) launch(a.signs ? build_sketch_kernel<true, kNarrowColumns> : build_sketch_kernel<false, kNarrowColumns>);
    else launch(a.signs ? build_sketch_kernel<true, kTileUnits> : build_sketch_kernel<false, kTileUnits>);
    if (int rc = check_launch("build_sketch")) return rc;
    a.weights += most * a.rows * a.hidden;
    a.codes += most * a.storage;
    a.stats += most * a.blocks * 2 * a.rows;
  }
  return 0;
}

}  // extern "C"

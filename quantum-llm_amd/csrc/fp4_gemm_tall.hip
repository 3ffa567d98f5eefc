// FP4 (E2M1, block-scaled) weight GEMM for tall batches (prompt prefill,
// M >> 8 rows).
//
// Replaces fp4_gemm_block32_kernel of the reference
// (runtime/src/cuda/transformer_kernels.cu:1284-1430: weights expanded to
// bf16 with their block scale, bf16 activations, 16x16x16 tensor-core tiles,
// F32 accumulation).  Here the contraction is compute-bound, so it is laid out
// for the matrix cores: a workgroup of four waves owns 128 activation rows x
// 256 weight rows (or fewer); every wave keeps the 128 x 64 accumulator of its
// two 32-row weight tiles in registers (8 x 4 tiles of v_mfma_f32_16x16x32), takes
// its weights straight from the provider's streaming layout - the 16-byte
// piece a lane loads per (tile, chunk) is its B operand for the chunk's four
// instructions, no LDS and no shuffle - and shares the activation tile of the
// chunk through LDS (one barrier per 64 columns of K).  Batches whose tiles are
// too few for the GPU - short prompts, and long ones against matrices of few
// rows - are cut along K and use lower workgroups (plan_tall).
//
// Scale schemes:
//  * UE8M0 per 32: the power-of-two scale is folded into the nibble -> bf16
//    conversion, which stays exact; bf16 matrix instructions.
//  * binary16 per 16: weight x scale has up to 13 significant bits (a 3-bit
//    weight times an 11-bit scale).  It is split into two binary16 values,
//    hi = the product rounded to binary16 and lo = its rounding error, which
//    a fused multiply-add returns exactly; they go through the matrix cores
//    one after the other into the same F32 accumulator; the bf16 activations
//    are converted to binary16 (exact between 6.1e-5 and 65504 in magnitude -
//    the range of a decoder's normalised activations; beyond it they saturate
//    or lose low bits).  The products are the exact ones, as in the small-batch
//    kernel, at twice the matrix instructions - for block scales between 2^-13
//    (1.22e-4) and 10917 in magnitude: both halves are formed in binary16, so
//    a weight of 6 under a larger scale overflows it (the small-batch kernel
//    multiplies in F32 and stays finite), and under a smaller scale the low
//    half has bits below 2^-24 and is cut short (a relative error of up to
//    2^-11 in that weight).  Checkpoint scales lie well inside.
#include "common.hpp"

#include <algorithm>
#include <iterator>
#include <type_traits>
#include <utility>

namespace qllm {
namespace {

constexpr int kSchemeUe8m0 = QLLM_SCALE_UE8M0_BLOCK32;
constexpr int kSchemeF16 = QLLM_SCALE_F16_BLOCK16;

constexpr uint32_t kChunk = 64;          // K columns per step
constexpr uint32_t kRowsM = 128;         // activation rows per workgroup
constexpr uint32_t kTilesM = kRowsM / 16;
constexpr uint32_t kWaves = 4;
constexpr uint32_t kTilesPerWave = 2;    // 32-row weight tiles per wave
constexpr uint32_t kTilesN = kWaves * kTilesPerWave;   // per workgroup
constexpr uint32_t kTileRows = 32;
constexpr uint32_t kBand = 8;            // activation tiles per band of the grid
constexpr uint32_t kLowestTail = 5;      // height from which on tiles may be cut alone
// LDS row of the activation tile: 64 values of 16 bits in eight pieces, piece p of
// row r at p ^ (r % 8), so that a fragment load meets no bank conflict (with rows
// 16 bytes longer instead, every one of them cost four more cycles)
constexpr uint32_t kLdsRow = kChunk * 2u;
__device__ __forceinline__ uint32_t swizzled(uint32_t piece, uint32_t row) {
  return (piece ^ (row % 8u)) * 16u;
}

typedef __attribute__((ext_vector_type(8))) _Float16 f16x8;
typedef __attribute__((ext_vector_type(2))) _Float16 f16x2;

struct TallArgs {
  const uint8_t* weights;        // streaming layout, 32-row tiles
  const uint8_t* scales;
  // SWIGLU form: `weights` / `scales` are the gate matrix, these the up matrix
  // of the same shape; output = bf16(bf16(silu(gate . x)) * (up . x))
  const uint8_t* up_weights;
  const uint8_t* up_scales;
  const uint16_t* activations;   // bf16 [batch, padded_columns]
  uint32_t rows;                 // weight rows = output columns
  uint32_t padded_columns;
  uint32_t batch;
  uint32_t m_tiles;
  uint32_t n_tiles;
  // K cut over `splits` workgroups per tile: part p of a tile sums its share of
  // the chunks into partials[p][batch][rows] (SWIGLU: partials[p][2][batch]
  // [rows], gate before up), and whoever reads them adds the parts in order
  uint32_t splits;
  // With `cut` only the last tiles are cut: the first `whole` run whole, each of the
  // others is `cut` pieces, whose accumulators go to partials as they stand in the
  // registers ([piece][vector of a thread][thread]), for tall_tail_kernel
  uint32_t whole;
  uint32_t cut;
  float* partials;
  void* output;                  // [batch, rows]
  uint32_t output_kind;
  const float* residual;
  // optional split of the output columns over up to three buffers
  uint32_t segments;
  uint32_t segment_rows[3];
  uint32_t segment_kind[3];
  void* segment_output[3];
};

// Workgroups are dealt to the eight XCDs in turn, so XCD x runs the ids x,
// x + 8, ...: the position that gives each XCD a contiguous range instead.
__device__ __forceinline__ uint32_t xcd_contiguous(uint32_t id, uint32_t total) {
  const uint32_t xcd = id % 8u;
  return xcd * (total / 8u) + min(xcd, total % 8u) + id / 8u;
}

// What a workgroup does: chunks [first_chunk, end_chunk) of tile (m_tile, n_tile), as
// part `part` of the launch or piece `piece` of a cut tile.
struct Work {
  uint32_t m_tile, n_tile;
  uint32_t first_chunk, end_chunk;
  uint32_t part, piece;
  bool is_piece;
};

// Tiles go band by band (kBand activation tiles high), column by column: the 64
// workgroups an XCD runs at a time then cover about 8 x 8 tiles and fetch 8 + 8
// operand tiles per K step into its L2 rather than 64 + 1.
__device__ __forceinline__ void place_tile(const TallArgs& args, uint32_t id,
                                           uint32_t& m_tile, uint32_t& n_tile) {
  const uint32_t band_tiles = kBand * args.n_tiles;
  const uint32_t band = id / band_tiles;
  const uint32_t in_band = id - band * band_tiles;
  const uint32_t height = min(kBand, args.m_tiles - band * kBand);
  m_tile = band * kBand + in_band % height;
  n_tile = in_band / height;
}

// An XCD gets a contiguous range of a part's tiles, or - launches that may be TAILED -
// of the whole tiles and then of the pieces.
template <bool TAILED>
__device__ __forceinline__ Work work_of(const TallArgs& args, uint32_t chunks) {
  const uint32_t tiles = args.m_tiles * args.n_tiles;
  Work work{};
  uint32_t id, share = 0u, shares = 1u;
  if constexpr (!TAILED) {
    // (the low workgroups of short launches: no band is higher than the batch)
    const uint32_t position = xcd_contiguous(blockIdx.x, tiles * args.splits);
    work.part = position / tiles;
    id = position - work.part * tiles;
    work.n_tile = id / args.m_tiles;
    work.m_tile = id - work.n_tile * args.m_tiles;
    work.first_chunk = chunks * work.part / args.splits;
    work.end_chunk = chunks * (work.part + 1u) / args.splits;
    return work;
  }
  if (args.cut && blockIdx.x >= args.whole) {
    work.is_piece = true;
    work.piece = xcd_contiguous(blockIdx.x - args.whole, (tiles - args.whole) * args.cut);
    id = args.whole + work.piece / args.cut;
    share = work.piece % args.cut;
    shares = args.cut;
  } else if (args.cut) {
    id = xcd_contiguous(blockIdx.x, args.whole);
  } else {
    const uint32_t position = xcd_contiguous(blockIdx.x, tiles * args.splits);
    work.part = share = position / tiles;
    id = position - share * tiles;
    shares = args.splits;
  }
  work.first_chunk = chunks * share / shares;
  work.end_chunk = chunks * (share + 1u) / shares;
  place_tile(args, id, work.m_tile, work.n_tile);
  return work;
}

__device__ __forceinline__ void store_value(void* output, uint32_t kind,
                                            size_t index, float value) {
  if (kind == QLLM_OUT_BF16)
    static_cast<uint16_t*>(output)[index] =
        static_cast<uint16_t>(f32_to_bf16_bits(value));
  else if (kind == QLLM_OUT_F32_BF16_ROUNDED)
    static_cast<float*>(output)[index] = bf16_round(value);
  else
    static_cast<float*>(output)[index] = value;
}

// Two bf16 values (one dword) -> two binary16 values.  Round toward zero only
// matters outside binary16's normal range, where it saturates instead of
// producing infinities.
__device__ __forceinline__ uint32_t bf16x2_to_f16x2(uint32_t pair) {
  const float low = __uint_as_float(pair << 16);
  const float high = __uint_as_float(pair & 0xffff0000u);
  return __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_pkrtz(low, high));
}

template <int SCHEME>
struct Operand;

template <>
struct Operand<kSchemeUe8m0> {
  using Vector = bf16x8;
  static constexpr int kParts = 1;
  // `scale` = the block's power of two
  static __device__ __forceinline__ void weights(uint32_t packed, float scale,
                                                 uint32_t, Vector (&out)[1]) {
    const bf16x2 p0 = fp4x2_to_bf16<0>(packed, scale);
    const bf16x2 p1 = fp4x2_to_bf16<1>(packed, scale);
    const bf16x2 p2 = fp4x2_to_bf16<2>(packed, scale);
    const bf16x2 p3 = fp4x2_to_bf16<3>(packed, scale);
    Vector w;
    w[0] = p0[0]; w[1] = p0[1]; w[2] = p1[0]; w[3] = p1[1];
    w[4] = p2[0]; w[5] = p2[1]; w[6] = p3[0]; w[7] = p3[1];
    out[0] = w;
  }
  static __device__ __forceinline__ f32x4 mfma(Vector a, Vector b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ uint32_t stage(uint32_t pair) { return pair; }
};

typedef __attribute__((ext_vector_type(2))) float f32x2;

template <>
struct Operand<kSchemeF16> {
  using Vector = f16x8;
  static constexpr int kParts = 2;
  // `scale_bits` = the block's binary16 scale; out[0] = hi, out[1] = lo with
  // hi + lo = weight x scale exactly
  // hi = the product rounded to binary16, lo = the rounding error, which a
  // fused multiply-add returns exactly (it has at most two significant bits):
  // three packed instructions per pair of weights.
  static __device__ __forceinline__ void weights(uint32_t packed, float,
                                                 uint32_t scale_bits,
                                                 Vector (&out)[2]) {
    const f16x2 scale =
        __builtin_bit_cast(f16x2, scale_bits | (scale_bits << 16));
    Vector hi, lo;
#pragma unroll
    for (int pair = 0; pair < 4; ++pair) {
      f16x2 w;
      switch (pair) {
        case 0: w = __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(packed, 1.0f, 0); break;
        case 1: w = __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(packed, 1.0f, 1); break;
        case 2: w = __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(packed, 1.0f, 2); break;
        default: w = __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(packed, 1.0f, 3); break;
      }
      const f16x2 top = w * scale;
      const f16x2 rest = __builtin_elementwise_fma(w, scale, -top);
      hi[2 * pair] = top[0]; hi[2 * pair + 1] = top[1];
      lo[2 * pair] = rest[0]; lo[2 * pair + 1] = rest[1];
    }
    out[0] = hi;
    out[1] = lo;
  }
  static __device__ __forceinline__ f32x4 mfma(Vector a, Vector b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ uint32_t stage(uint32_t pair) {
    return bf16x2_to_f16x2(pair);
  }
};

// Where the output columns from `column` on go: the matrix's output, or the
// segment that holds them (segments are multiples of 32 rows).
struct Destination {
  void* output;
  uint32_t kind;
  uint32_t width;
  uint32_t first;   // the destination's first column in the matrix
};
__device__ __forceinline__ Destination destination_of(const TallArgs& args,
                                                      uint32_t column) {
  if (!args.segments) return {args.output, args.output_kind, args.rows, 0u};
  uint32_t segment = 0, first = 0;
  while (segment + 1u < args.segments &&
         column >= first + args.segment_rows[segment]) {
    first += args.segment_rows[segment];
    ++segment;
  }
  return {args.segment_output[segment], args.segment_kind[segment],
          args.segment_rows[segment], first};
}

// bf16(bf16(silu(gate)) * up), the rounding points of the SiLU-product launch
__device__ __forceinline__ uint16_t swiglu_bits(float gate, float up) {
  const float activated = bf16_round(gate / (1.0f + expf(-gate)));
  return static_cast<uint16_t>(f32_to_bf16_bits(activated * up));
}

// A piece's accumulators, vector q of thread i at ((piece Q + q) 256 + i) of
// args.partials (Q vectors a thread).
template <int MT, int T>
__device__ __forceinline__ void store_piece(const TallArgs& args, uint32_t piece,
                                            const f32x4 (&acc)[MT][T][2]) {
  f32x4* target = reinterpret_cast<f32x4*>(args.partials) +
                  static_cast<size_t>(piece) * (MT * T * 2u * kWaves * 64u) + threadIdx.x;
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int t = 0; t < T; ++t)
#pragma unroll
      for (int j = 0; j < 2; ++j)
        target[((mt * T + t) * 2 + j) * (kWaves * 64u)] = acc[mt][t][j];
}

// The weight tiles of a wave: 32 rows of the gate matrix and the same of the up
// matrix, or T tiles side by side.
template <int T, bool SWIGLU>
__device__ __forceinline__ uint32_t weight_tile(uint32_t n_tile, uint32_t wave, uint32_t t) {
  return SWIGLU ? n_tile * kWaves + wave : (n_tile * kWaves + wave) * T + t;
}

// Stores a wave's accumulators.  D register i of lane (n, g): activation row
// first_m + 16 mt + 4 g + i, weight row 32 tile + 16 j + n.
template <int MT, int T, bool SWIGLU>
__device__ __forceinline__ void store_tiles(const TallArgs& args, uint32_t part,
                                            uint32_t first_m,
                                            const uint32_t (&tile_index)[T],
                                            uint32_t tile_count,
                                            const f32x4 (&acc)[MT][T][2]) {
  const uint32_t n = threadIdx.x & 15u;
  const uint32_t g = (threadIdx.x & 63u) >> 4;
  if (args.splits > 1u) {
#pragma unroll
    for (int t = 0; t < T; ++t) {
      if (tile_index[t] >= tile_count) continue;
      const uint32_t plane = SWIGLU ? part * 2u + t : part;
#pragma unroll
      for (uint32_t j = 0; j < 2u; ++j) {
        const uint32_t column = tile_index[t] * kTileRows + 16u * j + n;
        if (column >= args.rows) continue;
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
          for (uint32_t i = 0; i < 4u; ++i) {
            const uint32_t row = first_m + 16u * mt + 4u * g + i;
            if (row >= args.batch) continue;
            args.partials[(static_cast<size_t>(plane) * args.batch + row) *
                              args.rows + column] = acc[mt][t][j][i];
          }
      }
    }
    return;
  }
  if constexpr (SWIGLU) {
    if (tile_index[0] >= tile_count) return;
#pragma unroll
    for (uint32_t j = 0; j < 2u; ++j) {
      const uint32_t column = tile_index[0] * kTileRows + 16u * j + n;
      if (column >= args.rows) continue;
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (uint32_t i = 0; i < 4u; ++i) {
          const uint32_t row = first_m + 16u * mt + 4u * g + i;
          if (row >= args.batch) continue;
          static_cast<uint16_t*>(args.output)[static_cast<size_t>(row) * args.rows +
                                              column] =
              swiglu_bits(acc[mt][0][j][i], acc[mt][1][j][i]);
        }
    }
    return;
  }
#pragma unroll
  for (int t = 0; t < T; ++t) {
    if (tile_index[t] >= tile_count) continue;
    const uint32_t tile_first = tile_index[t] * kTileRows;
    const Destination to = destination_of(args, tile_first);
    const bool add = args.residual && !args.segments;
#pragma unroll
    for (uint32_t j = 0; j < 2u; ++j) {
      const uint32_t column = tile_first + 16u * j + n;
      if (column >= args.rows) continue;
      // the residual's values are fetched together: it may be the output itself,
      // and a load after a store would wait for every one before it
      float rest[MT][4];
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (uint32_t i = 0; i < 4u; ++i) {
          const uint32_t row = min(first_m + 16u * mt + 4u * g + i, args.batch - 1u);
          rest[mt][i] =
              add ? args.residual[static_cast<size_t>(row) * args.rows + column] : 0.0f;
        }
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (uint32_t i = 0; i < 4u; ++i) {
          const uint32_t row = first_m + 16u * mt + 4u * g + i;
          if (row >= args.batch) continue;
          store_value(to.output, to.kind,
                      static_cast<size_t>(row) * to.width + (column - to.first),
                      add ? acc[mt][t][j][i] + rest[mt][i] : acc[mt][t][j][i]);
        }
    }
  }
}

constexpr uint32_t kPastTheEnd = 0x80000000u;   // an offset that fetches nothing

// A workgroup of 16 MT activation rows by 128 T weight rows and the chunks of its part or
// piece.  SWIGLU: 128 rows of the gate and of the up matrix each, a wave's two tiles are
// the same 32 rows of both, and the epilogue writes silu(gate) * up in bf16 with the
// rounding points of the separate SiLU-product launch - no F32 round trip of the two.
//
// Up to 64 rows the weights' way from memory is what there is to hide, not the matrix
// cores' time: a wave keeps its weights of the next four chunks on their way in registers
// (two where accumulators leave no room), activations are two or three steps ahead, and
// a step covers so many chunks that its barrier costs about the same whatever the height.
// With 128 rows it is the matrix cores, as far as the card's power lets them: gate and up
// of [17408, 5120] with binary16 scales over 8192 rows kept them busy 73 % of the time at
// 2.10 GHz when a unit's weights were converted before its products and a half chunk's
// activations waited for; with both done in between the products 80 % at 2.00 GHz, 3750 ->
// 3650 us.  UE8M0 scales, whose activations need no conversion and are copied to the LDS
// without passing through registers: 63 -> 75 %, 2245 -> 2037 us; 300 rows by [10240, 5120]
// 50.9 -> 42.4 (binary16: 80 -> 71), 64 by [32000, 2048] 21.7 -> 19.5 (28.7 -> 26.8); 48 rows
// by [10240, 5120] stay within 3 % of 20 (25).  80 and 112 rows
// stand between so that fewer rows of a batch's last workgroups are padding; a weight's
// conversion, three vector instructions a pair of binary16 scaled ones, serves that many
// more rows.
//
// FAR: matrices of 2^24 columns and more, whose activation rows and weight tiles lie past
// 32-bit offsets: 64-bit addresses of every lane's own and a range a chunk.
template <int SCHEME, int MT, int T, bool SWIGLU, bool FAR = false>
__global__ __launch_bounds__(kWaves * 64, 2) void fp4_gemm_rows_kernel(const TallArgs args) {
  using Op = Operand<SCHEME>;
  using Vector = typename Op::Vector;
  constexpr bool F16 = SCHEME == kSchemeF16;
  static_assert(!SWIGLU || T == 2);
  constexpr int kAhead = MT > 4 ? 2 : 4;            // chunks of weights in flight
  constexpr int kSpan = MT > 4 ? 1 : MT == 3 ? 2 : 4 / MT;   // chunks per step
  // Activations that stay bf16 are copied straight to the LDS, into one of four tiles;
  // those converted on the way pass through registers and two tiles.  (Tiles are arrays of
  // their own: of one array's parts the compiler would have every read wait for all copies.)
  constexpr bool kCopied = !F16;
  constexpr int kTiles = kCopied ? 4 : 2;
  constexpr int kStages = MT > 7 ? 1 : 2;           // steps of activations in registers
  constexpr uint32_t kRow = kSpan * kLdsRow;
  constexpr uint32_t kTileBytes = 16u * MT * kRow;
  // 16-byte pieces of a step's activations, of the workgroup and of a thread (an odd
  // height's last ones are the same pieces for half of the waves)
  constexpr uint32_t kAllPieces = kTileBytes / 16u;
  constexpr uint32_t kPieces = (kAllPieces + kWaves * 64u - 1u) / (kWaves * 64u);
  constexpr uint32_t kStepLoads = kPieces + 2u * T * kSpan;
  __shared__ __attribute__((aligned(16))) uint8_t tile0[kTileBytes];
  __shared__ __attribute__((aligned(16))) uint8_t tile1[kTileBytes];
  __shared__ __attribute__((aligned(16))) uint8_t tile2[kTiles > 2 ? kTileBytes : 16u];
  __shared__ __attribute__((aligned(16))) uint8_t tile3[kTiles > 2 ? kTileBytes : 16u];
  const auto tile_of = [&](int position) {
    position %= kTiles;
    return position == 0 ? tile0 : position == 1 ? tile1 : position == 2 ? tile2 : tile3;
  };

  const uint32_t lane = threadIdx.x & 63u;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t n = lane & 15u;
  const uint32_t g = lane >> 4;
  const uint32_t K = args.padded_columns;
  const uint32_t chunks = K / kChunk;

  // activation tiles of one weight tile run side by side on an XCD, then the weight
  // tiles of a part: weights and activations come from its L2
  constexpr bool kTailed = MT >= static_cast<int>(kLowestTail);
  const Work work = work_of<kTailed>(args, chunks);
  const uint32_t first_m = work.m_tile * (16u * MT);
  const uint32_t first_chunk = work.first_chunk;
  const uint32_t end_chunk = work.end_chunk;

  // weight streams of this wave's tiles (tiles past the matrix repeat the last
  // one and are not stored)
  constexpr uint32_t kCodes = kTileRows * 32u, kScales = kTileRows * (F16 ? 8u : 2u);
  const uint32_t tile_count = (args.rows + kTileRows - 1u) / kTileRows;
  __amdgpu_buffer_rsrc_t code_stream[T], scale_stream[T];
  uint32_t tile_index[T];
  const auto codes_of = [&](int t) { return SWIGLU && t ? args.up_weights : args.weights; };
  const auto scales_of = [&](int t) { return SWIGLU && t ? args.up_scales : args.scales; };
  // `count` chunks of tile t from chunk `at` on, `bytes` each
  const auto stream_of = [&](const uint8_t* first, int t, uint32_t at, uint32_t count,
                             uint32_t bytes) __attribute__((always_inline)) {
    const size_t stream = static_cast<size_t>(min(tile_index[t], tile_count - 1u)) * chunks;
    return memory_range(first + (stream + at) * bytes, size_t{count} * bytes);
  };
#pragma unroll
  for (int t = 0; t < T; ++t) {
    tile_index[t] = weight_tile<T, SWIGLU>(work.n_tile, wave, t);
    if constexpr (!FAR) {
      code_stream[t] = stream_of(codes_of(t), t, 0u, chunks, kCodes);
      scale_stream[t] = stream_of(scales_of(t), t, 0u, chunks, kScales);
    }
  }
  const uint32_t code_offset = lane * 16u;
  const uint32_t scale_offset = F16 ? ((g >> 1) * 16u + n) * 8u : n * 4u;

  // Piece p of a step's tile: row p / (8 kSpan) and, of its chunk p / 8 % kSpan, the eight
  // columns that the swizzle puts there.  Rows past the batch read as zero and are not
  // stored; columns past K read what follows, or zero, and meet no weights.
  const auto activations = memory_range(args.activations + static_cast<size_t>(first_m) * K,
                                        static_cast<size_t>(args.batch - first_m) * K * 2u);
  uint32_t source[kPieces], target[kPieces];
#pragma unroll
  for (uint32_t p = 0; p < kPieces; ++p) {
    const uint32_t wave_piece = min(p * kWaves + wave, kAllPieces / 64u - 1u) * 64u;
    const uint32_t piece = wave_piece + lane;
    const uint32_t row = piece / (8u * kSpan);
    source[p] = row * K * 2u + (piece / 8u % kSpan * 8u + ((piece ^ row) % 8u)) * 16u;
    target[p] = (kCopied ? wave_piece : piece) * 16u;
  }
  const uint32_t fragment_offset[2] = {n * kRow + swizzled(g, n),
                                       n * kRow + swizzled(g + 4u, n)};

  f32x4 acc[MT][T][2];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int t = 0; t < T; ++t)
#pragma unroll
      for (uint32_t j = 0; j < 2u; ++j) acc[mt][t][j] = f32x4{0.f, 0.f, 0.f, 0.f};

  const auto source_at = [&](uint32_t p, uint32_t chunk) {
    return source[p] + min(chunk, end_chunk - 1u) * (kChunk * 2u);
  };
  // (rows past the batch are its last one here)
  const auto far_source = [&](uint32_t p, uint32_t chunk) {
    const uint32_t piece = min(p * kWaves + wave, kAllPieces / 64u - 1u) * 64u + lane;
    const uint32_t row = piece / (8u * kSpan);
    const size_t at = min(chunk + piece / 8u % kSpan, end_chunk - 1u);
    return reinterpret_cast<const uint8_t*>(
               args.activations + static_cast<size_t>(min(first_m + row, args.batch - 1u)) * K) +
           at * (kChunk * 2u) + (piece ^ row) % 8u * 16u;
  };
  const auto copy_activations = [&](uint8_t* tile, uint32_t chunk) {
#pragma unroll
    for (uint32_t p = 0; p < kPieces; ++p)
      if constexpr (FAR)
        copy16_to_lds(far_source(p, chunk), tile + target[p]);
      else
        copy16_to_lds(activations, source_at(p, chunk), 0u, tile + target[p]);
  };
  i32x4 staged[kStages][kPieces];
  const auto fetch_activations = [&](int slot, uint32_t chunk) {
#pragma unroll
    for (uint32_t p = 0; p < kPieces; ++p)
      if constexpr (FAR)
        staged[slot][p] = *reinterpret_cast<const i32x4*>(far_source(p, chunk));
      else
        staged[slot][p] = __builtin_bit_cast(
            i32x4,
            __builtin_amdgcn_raw_buffer_load_b128(activations, source_at(p, chunk), 0, 0));
  };
  const auto store_activations = [&](int slot, uint8_t* tile) {
#pragma unroll
    for (uint32_t p = 0; p < kPieces; ++p) {
      i32x4 v = staged[slot][p];
#pragma unroll
      for (int i = 0; i < 4; ++i)
        v[i] = static_cast<int>(Op::stage(static_cast<uint32_t>(v[i])));
      *reinterpret_cast<i32x4*>(tile + target[p]) = v;
    }
  };
  i32x4 codes[kAhead][T];
  i32x2 scales[kAhead][T];
  const auto fetch_weights = [&](int slot, uint32_t chunk) {
    // nothing is fetched past the part's end
    const uint32_t at = min(chunk, end_chunk - 1u);
    const uint32_t past = chunk < end_chunk ? 0u : kPastTheEnd;
#pragma unroll
    for (int t = 0; t < T; ++t) {
      const auto code = FAR ? stream_of(codes_of(t), t, at, 1u, kCodes) : code_stream[t];
      const auto scale = FAR ? stream_of(scales_of(t), t, at, 1u, kScales) : scale_stream[t];
      codes[slot][t] = __builtin_bit_cast(
          i32x4, __builtin_amdgcn_raw_buffer_load_b128(code, code_offset | past,
                                                       FAR ? 0u : at * kCodes, 0));
      if constexpr (F16)
        scales[slot][t] = __builtin_bit_cast(
            i32x2, __builtin_amdgcn_raw_buffer_load_b64(scale, scale_offset | past,
                                                        FAR ? 0u : at * kScales, 0));
      else
        scales[slot][t][0] = static_cast<int>(__builtin_amdgcn_raw_buffer_load_b32(
            scale, scale_offset | past, FAR ? 0u : at * kScales, 0));
    }
  };

  // Unit u of a chunk: 16 weight rows by 32 columns, u = 2 T s + 2 t + j.
  constexpr int kUnits = 4 * T;
  const auto convert = [&](int slot, int unit, Vector (&w)[Op::kParts]) {
    const int s = unit / (2 * T), t = unit / 2 % T, j = unit % 2;
    const uint32_t packed = static_cast<uint32_t>(codes[slot][t][2 * j + s]);
    // scale of (j, s): binary16 halves of the two words, or UE8M0 bytes
    const uint32_t word = static_cast<uint32_t>(scales[slot][t][F16 ? j : 0]);
    const uint32_t f16_bits = s ? word >> 16 : word & 0xffffu;
    const float fold = F16 ? 1.0f : ue8m0_to_f32(word >> (8 * (2 * j + s)) & 0xffu);
    Op::weights(packed, fold, f16_bits, w);
  };
  Vector w[2][Op::kParts];   // of this unit and of the next
  // activations of this half chunk and of the next, or - heights whose accumulators
  // leave no room for two - each of the next in the place of the one just used
  constexpr int kHalves = MT > 5 ? 1 : 2;
  Vector a[kHalves][MT];
  const auto fragment = [&](const uint8_t* tile, int c, int s, int mt) {
    return __builtin_bit_cast(Vector,
                              *reinterpret_cast<const i32x4*>(
                                  tile + mt * 16u * kRow + fragment_offset[s] + c * kLdsRow));
  };
  // Matrix instructions of a chunk with what the next ones need in between: an
  // instruction keeps the matrix cores for sixteen cycles and the wave's issue for four.
  // Told where to put them only where the products outweigh them: heights of up to 64 rows
  // (binary16 scales: 48) are up to 6 % faster as the compiler orders them.
  constexpr bool kPaced = MT > (F16 ? 3 : 4);
  // Whether a chunk's last unit converts the next chunk's first: that waits for its weights
  // before those of four chunks on are asked for.  Low workgroups, which wait for weights
  // and nothing else, ask first (16 rows, UE8M0 scales: [32000, 2048] 12.3 -> 11.4 us,
  // [5120, 17408] 20.9 -> 19.1, where one unit at a time had taken 11.4 and 19.3; with 32
  // rows and binary16 scales it gains nothing).
  constexpr bool kAcross = MT > (F16 ? 1 : 2);
  constexpr int kProducts = MT * Op::kParts;               // of a unit
  constexpr int kConversion = F16 ? 13 : 6;                // vector instructions of a unit
  const auto multiply = [&](int slot, const uint8_t* tile,
                            int c) __attribute__((always_inline)) {
    const bool last_of_step = c + 1 == kSpan;
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (!kAcross) convert(slot, 0, w[0]);
    if (c == 0)
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) a[0][mt] = fragment(tile, 0, 0, mt);
#pragma unroll
    for (int unit = 0; unit < kUnits; ++unit) {
      const int s = unit / (2 * T), t = unit / 2 % T, j = unit % 2;
      const bool reads =
          unit % (2 * T) == (kHalves > 1 ? 0 : 2 * T - 1) && !(last_of_step && s == 1);
      const auto read = [&](int mt) {
        if (reads)
          a[(1 - s) % kHalves][mt] = fragment(tile, s ? c + 1 : c, s ? 0 : 1, mt);
      };
      if constexpr (kHalves > 1)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) read(mt);
      if (unit + 1 < kUnits)
        convert(slot, unit + 1, w[(unit + 1) % 2]);
      else if constexpr (kAcross)
        convert((slot + 1) % kAhead, 0, w[(unit + 1) % 2]);
#pragma unroll
      for (int part = 0; part < Op::kParts; ++part)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
          acc[mt][t][j] = Op::mfma(a[s % kHalves][mt], w[unit % 2][part], acc[mt][t][j]);
          if (kHalves == 1 && part + 1 == Op::kParts) read(mt);
        }
      if constexpr (!kPaced) continue;
#pragma unroll
      for (int i = 0; i < kProducts; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        if (reads && (kHalves > 1 ? i < MT : i >= kProducts - MT))
          __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x002, (kConversion + kProducts - 1) / kProducts,
                                             0);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };

  // About in the order in which the loop waits for them, and in just this order: the
  // copies' waits count on all weights behind the first tile, and on a step's at least
  // behind the second.
  static_assert(kAhead >= kSpan && kAhead <= 4);
  constexpr int kWeightsFirst = kAhead > kSpan ? 0 : kTiles - 2;
#pragma unroll
  for (int ahead = 0; ahead < std::max(kTiles - 1, kAhead + kWeightsFirst); ++ahead) {
    if constexpr (kCopied) {
      if (ahead + 1 < kTiles) copy_activations(tile_of(ahead), first_chunk + ahead * kSpan);
      __builtin_amdgcn_sched_barrier(0);
    } else {
      if (ahead < kStages) fetch_activations(ahead, first_chunk + ahead * kSpan);
    }
    if (ahead >= kWeightsFirst && ahead < kAhead + kWeightsFirst)
      fetch_weights(ahead - kWeightsFirst, first_chunk + ahead - kWeightsFirst);
    __builtin_amdgcn_sched_barrier(0);
  }
  if constexpr (kCopied)
    wait_for_loads<(kTiles - 2) * kPieces + 2u * T * kAhead>();
  else
    store_activations(0, tile0);
  if constexpr (kAcross) convert(0, 0, w[0]);

  // Step P of a round.  A chunk's weights are refilled as soon as they have been
  // multiplied; one past the part's end makes its loads, which fetch nothing, and
  // multiplies nothing, so that every wait can count on the same loads having been made.
  const auto step_at = [&]<int P, bool WHOLE>(std::integral_constant<int, P>,
                                              std::bool_constant<WHOLE>,
                                              uint32_t chunk) __attribute__((always_inline)) {
    if constexpr (kCopied) {
      // this step's tile is there: what later steps asked for may be on its way
      wait_for_loads<(kTiles - 2) * kStepLoads>();
      barrier_beside_copies();   // everybody's is, and the tile before has been read
      copy_activations(tile_of(P + kTiles - 1), chunk + (kTiles - 1) * kSpan);
    } else {
      __syncthreads();   // this step's tile is complete; the other one is free
      fetch_activations(P % kStages, chunk + kStages * kSpan);
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int c = 0; c < kSpan; ++c) {
      const int slot = (P * kSpan + c) % kAhead;
      if (WHOLE || chunk + c < end_chunk) multiply(slot, tile_of(P), c);
      // the loads stay here: moved up they would need registers of their own and
      // copies at the loop's end, which wait for them, moved down they come late
      __builtin_amdgcn_sched_barrier(0);
      fetch_weights(slot, chunk + c + kAhead);
      __builtin_amdgcn_sched_barrier(0);
    }
    if constexpr (!kCopied) store_activations((P + 1) % kStages, tile_of(P + 1));
  };
  // Rounds of steps, after which every tile, stage and slot has had its turn.  Of copied
  // activations whole ones and what is left (of a loop that is left within a round the
  // compiler takes every step for the one before the next round, which then starts with a
  // wait for copies and weights just asked for); of two stages whole ones alone, steps past
  // the end among them (the same, for what passes through registers).
  constexpr int kRound = std::max(kTiles, (kAhead + kSpan - 1) / kSpan);
  uint32_t chunk = first_chunk;
  for (; kCopied ? chunk + kRound * kSpan <= end_chunk : chunk < end_chunk;
       chunk += kRound * kSpan)
    [&]<int... P>(std::integer_sequence<int, P...>) {
      (step_at(std::integral_constant<int, P>{}, std::bool_constant<kCopied>{},
               chunk + P * kSpan),
       ...);
    }(std::make_integer_sequence<int, kRound>{});
  if (kCopied && chunk < end_chunk)
    [&]<int... P>(std::integer_sequence<int, P...>) {
      (void)((step_at(std::integral_constant<int, P>{}, std::false_type{}, chunk + P * kSpan),
              chunk + (P + 1) * kSpan < end_chunk) &&
             ...);
    }(std::make_integer_sequence<int, kRound>{});
  if constexpr (kCopied) wait_for_loads<0>();   // no copy outlives its workgroup
  if (kTailed && work.is_piece)
    store_piece<MT, T>(args, work.piece, acc);
  else
    store_tiles<MT, T, SWIGLU>(args, work.part, first_m, tile_index, tile_count, acc);
}

// Adds the pieces of a cut tile in their order and stores the tile as a whole one's
// workgroup would have, sixteen activation rows a workgroup (grid: tiles, MT).
template <int MT, int T, bool SWIGLU>
__global__ __launch_bounds__(kWaves * 64) void tall_tail_kernel(const TallArgs args) {
  constexpr uint32_t kVectors = MT * T * 2u;
  const uint32_t mt = blockIdx.y;
  const f32x4* source = reinterpret_cast<const f32x4*>(args.partials) +
                        (static_cast<size_t>(blockIdx.x) * args.cut * kVectors +
                         mt * (T * 2u)) * (kWaves * 64u) + threadIdx.x;
  f32x4 acc[1][T][2] = {};
  for (uint32_t piece = 0; piece < args.cut; ++piece) {
#pragma unroll
    for (int t = 0; t < T; ++t)
#pragma unroll
      for (int j = 0; j < 2; ++j)
        acc[0][t][j] += source[static_cast<size_t>(t * 2 + j) * (kWaves * 64u)];
    source += static_cast<size_t>(kVectors) * (kWaves * 64u);
  }
  uint32_t m_tile, n_tile, tile_index[T];
  place_tile(args, args.whole + blockIdx.x, m_tile, n_tile);
#pragma unroll
  for (int t = 0; t < T; ++t)
    tile_index[t] = weight_tile<T, SWIGLU>(n_tile, threadIdx.x / 64u, t);
  store_tiles<1, T, SWIGLU>(args, 0u, m_tile * (16u * MT) + 16u * mt, tile_index,
                            (args.rows + kTileRows - 1u) / kTileRows, acc);
}

// Adds the parts of a launch whose K was cut, four columns per thread, and
// stores what its epilogue would have stored.
template <bool SWIGLU>
__global__ __launch_bounds__(256) void tall_parts_kernel(const TallArgs args) {
  const uint32_t column = (blockIdx.x * 256u + threadIdx.x) * 4u;
  const uint32_t row = blockIdx.y;
  if (column >= args.rows) return;
  const size_t plane = static_cast<size_t>(args.batch) * args.rows;
  const float* source =
      args.partials + static_cast<size_t>(row) * args.rows + column;
  const size_t step = SWIGLU ? 2u * plane : plane;
  f32x4 sum = *reinterpret_cast<const f32x4*>(source);
  f32x4 up{};
  if constexpr (SWIGLU) up = *reinterpret_cast<const f32x4*>(source + plane);
  for (uint32_t part = 1; part < args.splits; ++part) {
    source += step;
    sum += *reinterpret_cast<const f32x4*>(source);
    if constexpr (SWIGLU) up += *reinterpret_cast<const f32x4*>(source + plane);
  }
  if constexpr (SWIGLU) {
    uint16_t* out = static_cast<uint16_t*>(args.output) +
                    static_cast<size_t>(row) * args.rows + column;
#pragma unroll
    for (int i = 0; i < 4; ++i) out[i] = swiglu_bits(sum[i], up[i]);
    return;
  }
  const Destination to = destination_of(args, column);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    float value = sum[i];
    if (args.residual && !args.segments)
      value += args.residual[static_cast<size_t>(row) * args.rows + column + i];
    store_value(to.output, to.kind,
                static_cast<size_t>(row) * to.width + (column + i - to.first), value);
  }
}

// Columns from which on a lane's 32-bit offset does not reach over 128 activation rows:
// such matrices take the kernel's FAR form.
constexpr uint32_t kFarColumns = 1u << 24;

bool tall_matrix_ok(const qllm_fp4_matrix* m) {
  return m && m->weights && m->scales && m->rows && m->columns &&
         m->padded_columns >= m->columns && m->padded_columns % kChunk == 0u &&
         (m->scale_scheme == QLLM_SCALE_UE8M0_BLOCK32 ||
          m->scale_scheme == QLLM_SCALE_F16_BLOCK16) &&
         m->layout == QLLM_LAYOUT_TILED &&
         (m->tile_rows == 0u || m->tile_rows == kTileRows);
}

// How a launch is laid out: 16 `height` rows of activations per workgroup (height 1,
// 2, 3, 4, 5, 7 or 8) and `splits` parts of K.
//
// Chosen by what the busiest CU will take.  With W workgroups per part it runs
// n = ceil(W splits / 256) of them, each over ceil(chunks / splits) chunks; a
// chunk costs `alone` ns where n = 1 (its round trips and barriers show) and
// n * `shared` where workgroups hide each other's.  Parts are written and read
// once more, at 6.2 TB/s, and take a launch of their own where no norm adds
// them.  The constants are a fit to 1300 timed launches over weights that come
// from memory (nine matrices of [2048, 2048] to [17408, 5120], 8 to 3000 rows,
// heights 1, 2, 4 and 8; 7 % root mean square error) of the kernels that converted a unit's
// weights before its products; the chosen layout was 1.5 % slower than the best of those
// timed on average, and of the present kernel 4 % (20000 layouts of twelve matrices, 8 to
// 3001 rows; most with 40 to 80 rows, whose K is cut into more parts than pay).  What the
// rule gives over one workgroup per 128 rows and tile: [5120, 17408] with binary16 scales,
// 48 rows 400 -> 27 us, 300 rows 404 -> 97, 1000 rows 405 -> 254, 2000 rows 668 -> 498;
// [10240, 5120] 127 -> 25, 135 -> 73, 211 -> 190, 333 -> 327; gate and up of [17408, 5120]
// 129 -> 54, 221 -> 195, then unchanged.
//
// Where parts are added by a launch of their own, the tiles past the last full round of
// the CUs may be cut instead of all of them: `cut` pieces each, the others run whole, as
// where 500 rows by gate and up of [17408, 5120] are 544 tiles, of which the last 32 took
// a CU's time for two again.  With that and the heights of 80 and 112 rows the four
// linears of a layer of the 27B widths, binary16 scales, take 0.87 of the time for 80
// rows, 0.92 for 300, 0.91 for 500, 0.93 for 1000, 0.98 for 1500 and 0.91 for 5000 (300
// rows: 417 -> 382 us; 1000: 1102 -> 1021), with UE8M0 scales 0.92, 0.97, 0.95, 0.96, 0.94
// and 0.91.
struct TallPlan {
  uint32_t height;
  uint32_t splits;
  uint32_t cut;   // 0: no tile is cut by itself
};

constexpr uint32_t kMaximumParts = 16;
constexpr uint32_t kComputeUnits = 256;
constexpr size_t kPartsBytes = size_t{128} << 20;
constexpr uint32_t kMostPieces = 2u * kComputeUnits;   // of cut tiles

struct ChunkCost {
  float alone, shared;   // ns
};
// Workgroups of 80 and 112 rows and cut tiles are for matrices of these rows: with fewer
// they were not timed, and of 32000 rows by 2048, where the estimate errs most, 224 rows
// of a batch took 48 us instead of 41.  Thirteen matrices in between, 2048 to 17408
// columns (the widths of 2048, 3072, 4096 and 5120), 40 to 3000 rows of a batch, both
// scale schemes: the launches for which they are chosen take 0.92 of the time on average
// and at most 1.04 (one in 300 1.09: 1300 rows by [5120, 3072], UE8M0 scales, 59 us for
// 54).  A launch whose parts the next norm adds takes those heights only where they
// gain clearly, since the norm pays for more parts.
constexpr uint32_t kFewestTimedRows = 3072, kMostTimedRows = 17408;
constexpr double kClearly = 1.025;
constexpr uint32_t kHeights[] = {1u, 2u, 3u, 4u, 5u, 7u, 8u};
// [scheme][SwiGLU][height].  Those of 80 and 112 rows are a fit of their own, to 410
// launches of the 27B widths over 80 to 784 rows (4 to 8 % root mean square error), brought
// to the scale of the others by the heights of 64 and 128 rows in it.  Those of 48 rows are
// no part of a fit: 86 % of the 64-row workgroup's, the share that 48 rows of the 27B
// widths took; other widths were not timed at that height.
constexpr ChunkCost kChunkCost[2][2][7] = {
    {{{160.f, 150.f}, {195.f, 180.f}, {315.f, 215.f}, {365.f, 250.f}, {770.f, 530.f},
      {980.f, 690.f}, {1160.f, 780.f}},
     {{250.f, 325.f}, {335.f, 345.f}, {520.f, 360.f}, {605.f, 420.f}, {790.f, 535.f},
      {1000.f, 705.f}, {1215.f, 780.f}}},
    {{{220.f, 230.f}, {300.f, 280.f}, {470.f, 335.f}, {545.f, 390.f}, {1150.f, 875.f},
      {1440.f, 1120.f}, {1690.f, 1265.f}},
     {{380.f, 440.f}, {515.f, 500.f}, {845.f, 615.f}, {985.f, 715.f}, {1150.f, 860.f},
      {1440.f, 1110.f}, {1710.f, 1230.f}}}};

uint32_t weight_rows_of(uint32_t height, bool swiglu) {
  return (height >= 5u && !swiglu ? kTilesN : kWaves) * kTileRows;
}

uint32_t workgroups_of(uint32_t rows, uint32_t batch, uint32_t height, bool swiglu) {
  const uint32_t weight_rows = weight_rows_of(height, swiglu);
  return (batch + 16u * height - 1u) / (16u * height) *
         ((rows + weight_rows - 1u) / weight_rows);
}

size_t parts_bytes(uint32_t rows, uint32_t batch, uint32_t splits, bool swiglu) {
  return splits > 1u ? size_t{splits} * (swiglu ? 2u : 1u) * batch * rows * 4u : 0u;
}

// Tiles that a plan with `cut` cuts: those past the last full round of the CUs.
uint32_t tail_tiles_of(uint32_t workgroups) { return workgroups % kComputeUnits; }

size_t piece_bytes(uint32_t height, bool swiglu) {
  return size_t{16u} * height * weight_rows_of(height, swiglu) * (swiglu ? 8u : 4u);
}

// Bytes of workspace that a plan takes.
size_t plan_bytes(const TallPlan& plan, uint32_t rows, uint32_t batch, bool swiglu) {
  if (!plan.cut) return parts_bytes(rows, batch, plan.splits, swiglu);
  return piece_bytes(plan.height, swiglu) * plan.cut *
         tail_tiles_of(workgroups_of(rows, batch, plan.height, swiglu));
}

// At most `workspace_bytes` of parts; `separate`: they are added by a launch of
// their own.
TallPlan plan_tall(uint32_t rows, uint32_t padded_columns, uint32_t batch,
                   uint32_t scheme, bool swiglu, bool separate,
                   size_t workspace_bytes, uint32_t fixed_splits = 0u) {
  const uint32_t chunks = padded_columns / kChunk;
  const uint32_t first = fixed_splits ? fixed_splits : 1u;
  // A part has two rounds of a workgroup's four chunks in flight at least; parts
  // are added four columns at a time, a row per grid row.  Matrices far below the
  // timed ones, which no decoder layer has, stay whole: the fit says nothing there.
  const bool whole = rows % 4u || batch > 65535u || chunks < 16u ||
                     uint64_t{rows} * padded_columns < (1u << 20);
  const uint32_t last = fixed_splits                  ? fixed_splits
                        : whole                       ? 1u
                        : chunks / 8u < kMaximumParts ? chunks / 8u
                                                      : kMaximumParts;
  TallPlan best{};
  double least = 0.0;
  const auto offer = [&](const TallPlan& plan, double time) {
    if (best.height && time >= least) return;
    best = plan;
    least = time;
  };
  const bool timed = rows >= kFewestTimedRows && rows <= kMostTimedRows;
  uint32_t lower = 0;   // the height before
  for (uint32_t index = 0; index < std::size(kHeights); ++index) {
    const uint32_t height = kHeights[index];
    const bool between = height == 5u || height == 7u;
    if (!timed && between) continue;
    // (far matrices, which no decoder has: 128 rows pay from 256 workgroups on, a hundred
    // GB of operands)
    if (padded_columns >= kFarColumns && (height == 3u || height > 4u)) continue;
    // one or two tiles of rows where they hold the batch, else the higher ones, and
    // none of which a lower one would hold the batch
    if (height < 3u ? batch > 16u * height : batch <= 32u) continue;
    if (index && batch <= 16u * lower) continue;
    lower = height;
    const ChunkCost cost = kChunkCost[scheme][swiglu][index];
    const uint32_t workgroups = workgroups_of(rows, batch, height, swiglu);
    for (uint32_t splits = first; splits <= last; ++splits) {
      const size_t bytes = parts_bytes(rows, batch, splits, swiglu);
      if (!fixed_splits && bytes > workspace_bytes) break;
      const uint64_t on_one =
          (uint64_t{workgroups} * splits + kComputeUnits - 1u) / kComputeUnits;
      const double chunk =
          on_one > 1u && on_one * cost.shared > cost.alone ? on_one * cost.shared
                                                           : cost.alone;
      const double time = (chunks + splits - 1u) / splits * chunk +
                          (separate ? 2.0 : 1.0) * bytes / 6200.0 +
                          (separate && splits > 1u ? 4300.0 : 0.0);
      offer({height, splits, 0u}, between && !separate ? time * kClearly : time);
    }
    // (whole tiles on every CU, so that two workgroups share it all the way)
    const uint32_t tail = tail_tiles_of(workgroups);
    if (!separate || whole || !timed || height < kLowestTail || tail == workgroups || !tail)
      continue;
    for (uint32_t cut = 2u; cut <= last && tail * cut <= kMostPieces; ++cut) {
      const TallPlan plan{height, 1u, cut};
      const size_t bytes = plan_bytes(plan, rows, batch, swiglu);
      if (bytes > workspace_bytes) break;
      const double rounds =
          workgroups / kComputeUnits +
          static_cast<double>((tail * cut + kComputeUnits - 1u) / kComputeUnits) / cut;
      offer(plan, chunks * std::max<double>(rounds * cost.shared, cost.alone) +
                      2.0 * bytes / 6200.0 + 4300.0);
    }
  }
  return best;
}

template <int SCHEME, int MT, int T, bool FAR>
void start_rows(const TallArgs& args, bool swiglu, uint32_t grid, hipStream_t stream) {
  constexpr uint32_t kThreads = kWaves * 64;
  if (swiglu)
    fp4_gemm_rows_kernel<SCHEME, MT, 2, true, FAR><<<grid, kThreads, 0, stream>>>(args);
  else
    fp4_gemm_rows_kernel<SCHEME, MT, T, false, FAR><<<grid, kThreads, 0, stream>>>(args);
}

template <int SCHEME>
void start_tall(const TallArgs& args, uint32_t height, bool swiglu, uint32_t grid,
                hipStream_t stream) {
  if (args.padded_columns >= kFarColumns) {
    switch (height) {
      case 1: return start_rows<SCHEME, 1, 1, true>(args, swiglu, grid, stream);
      case 2: return start_rows<SCHEME, 2, 1, true>(args, swiglu, grid, stream);
      default: return start_rows<SCHEME, 4, 1, true>(args, swiglu, grid, stream);
    }
  }
  switch (height) {
    case 1: return start_rows<SCHEME, 1, 1, false>(args, swiglu, grid, stream);
    case 2: return start_rows<SCHEME, 2, 1, false>(args, swiglu, grid, stream);
    case 3: return start_rows<SCHEME, 3, 1, false>(args, swiglu, grid, stream);
    case 4: return start_rows<SCHEME, 4, 1, false>(args, swiglu, grid, stream);
    case 5: return start_rows<SCHEME, 5, 2, false>(args, swiglu, grid, stream);
    case 7: return start_rows<SCHEME, 7, 2, false>(args, swiglu, grid, stream);
    default: return start_rows<SCHEME, 8, 2, false>(args, swiglu, grid, stream);
  }
}

void start_tail(const TallArgs& args, uint32_t height, uint32_t tail, hipStream_t stream) {
  const dim3 grid(tail, height);
  constexpr uint32_t kThreads = kWaves * 64;
  switch (height) {
    case 5:
      if (args.up_weights)
        tall_tail_kernel<5, 2, true><<<grid, kThreads, 0, stream>>>(args);
      else
        tall_tail_kernel<5, 2, false><<<grid, kThreads, 0, stream>>>(args);
      break;
    case 7:
      if (args.up_weights)
        tall_tail_kernel<7, 2, true><<<grid, kThreads, 0, stream>>>(args);
      else
        tall_tail_kernel<7, 2, false><<<grid, kThreads, 0, stream>>>(args);
      break;
    default:
      if (args.up_weights)
        tall_tail_kernel<8, 2, true><<<grid, kThreads, 0, stream>>>(args);
      else
        tall_tail_kernel<8, 2, false><<<grid, kThreads, 0, stream>>>(args);
  }
}

// The parts of a cut launch stay in args.partials.
int32_t launch_tall(TallArgs args, uint32_t scheme, const TallPlan& plan,
                    hipStream_t stream) {
  const bool swiglu = args.up_weights != nullptr;
  const uint32_t weight_rows = weight_rows_of(plan.height, swiglu);
  args.m_tiles = (args.batch + 16u * plan.height - 1u) / (16u * plan.height);
  args.n_tiles = (args.rows + weight_rows - 1u) / weight_rows;
  args.splits = plan.splits;
  args.cut = plan.cut;
  const uint32_t tiles = args.m_tiles * args.n_tiles;
  const uint32_t tail = tail_tiles_of(tiles);
  args.whole = tiles - tail;
  const uint32_t grid =
      plan.cut ? args.whole + tail * plan.cut : tiles * plan.splits;
  if (scheme == QLLM_SCALE_F16_BLOCK16)
    start_tall<kSchemeF16>(args, plan.height, swiglu, grid, stream);
  else
    start_tall<kSchemeUe8m0>(args, plan.height, swiglu, grid, stream);
  if (plan.cut) start_tail(args, plan.height, tail, stream);
  return launched("tall FP4 GEMM");
}

int32_t add_parts(const TallArgs& args, hipStream_t stream) {
  const dim3 grid((args.rows / 4u + 255u) / 256u, args.batch);
  if (args.up_weights)
    tall_parts_kernel<true><<<grid, 256, 0, stream>>>(args);
  else
    tall_parts_kernel<false><<<grid, 256, 0, stream>>>(args);
  return launched("tall FP4 GEMM parts");
}

// One launch, or - where the plan cuts K and `workspace` holds the parts - two.
int32_t run_tall(TallArgs args, uint32_t scheme, void* workspace,
                 size_t workspace_bytes, hipStream_t stream) {
  const bool swiglu = args.up_weights != nullptr;
  const TallPlan plan =
      plan_tall(args.rows, args.padded_columns, args.batch, scheme, swiglu, true,
                workspace ? workspace_bytes : 0u);
  args.partials = static_cast<float*>(workspace);
  args.splits = plan.splits;
  const int32_t status = launch_tall(args, scheme, plan, stream);
  if (status != QLLM_OK || plan.splits == 1u) return status;
  return add_parts(args, stream);
}

}  // namespace
}  // namespace qllm

using namespace qllm;

namespace {

// The arguments of a launch over `matrix` after the checks that all forms share.
bool tall_arguments(const qllm_fp4_matrix* matrix, const void* input,
                    size_t input_bytes, uint32_t batch, TallArgs& args) {
  if (!tall_matrix_ok(matrix) || !input || !batch || batch > (1u << 20) ||
      (reinterpret_cast<uintptr_t>(input) & 15u) ||
      input_bytes < static_cast<size_t>(batch) * matrix->padded_columns * 2u)
    return false;
  args.weights = matrix->weights;
  args.scales = static_cast<const uint8_t*>(matrix->scales);
  args.activations = static_cast<const uint16_t*>(input);
  args.rows = matrix->rows;
  args.padded_columns = matrix->padded_columns;
  args.batch = batch;
  return true;
}

bool workspace_ok(const void* workspace) {
  return (reinterpret_cast<uintptr_t>(workspace) & 15u) == 0u;
}

}  // namespace

extern "C" size_t qllm_fp4_tall_workspace_bytes(void) { return kPartsBytes; }

extern "C" uint32_t qllm_fp4_tall_parts(const qllm_fp4_matrix* matrix, uint32_t batch) {
  if (!tall_matrix_ok(matrix) || !batch) return 1u;
  return plan_tall(matrix->rows, matrix->padded_columns, batch, matrix->scale_scheme,
                   false, false, kPartsBytes).splits;
}

extern "C" int32_t qllm_fp4_tall_layout(const qllm_fp4_matrix* matrix, int32_t swiglu,
                                        uint32_t batch, size_t workspace_bytes,
                                        uint32_t parts, qllm_launch_layout* layout) {
  if (!tall_matrix_ok(matrix) || !batch || batch > (1u << 20) || parts > kMaximumParts ||
      parts > matrix->padded_columns / kChunk || (parts && swiglu) || !layout)
    return fail(QLLM_INVALID_ARGUMENT, "invalid tall FP4 GEMM layout");
  const TallPlan plan =
      plan_tall(matrix->rows, matrix->padded_columns, batch, matrix->scale_scheme, swiglu,
                parts == 0u, workspace_bytes, parts);
  *layout = {16u * plan.height, weight_rows_of(plan.height, swiglu), plan.splits};
  return QLLM_OK;
}

extern "C" uint32_t qllm_fp4_tall_tail_parts(const qllm_fp4_matrix* matrix, int32_t swiglu,
                                             uint32_t batch, size_t workspace_bytes) {
  if (!tall_matrix_ok(matrix) || !batch || batch > (1u << 20)) return 0u;
  return plan_tall(matrix->rows, matrix->padded_columns, batch, matrix->scale_scheme,
                   swiglu, true, workspace_bytes).cut;
}

extern "C" size_t qllm_fp4_tall_parts_bytes(const qllm_fp4_matrix* matrix, int32_t swiglu,
                                            uint32_t batch) {
  if (!tall_matrix_ok(matrix)) return 0u;
  const uint32_t rows = matrix->rows;
  size_t most = 0;
  // Within 16 batch rows the workgroups of every height stay the same in number and a
  // row makes the parts cost more, so the first row of 16 asks for the most parts.
  for (uint64_t first = 1u; first <= batch; first += 16u) {
    const uint32_t row = static_cast<uint32_t>(first);
    if (parts_bytes(rows, row, 2u, swiglu) > kPartsBytes) {
      // no launch of so many rows is cut as a whole: the room of the most pieces
      if (rows >= kFewestTimedRows && rows <= kMostTimedRows && rows % 4u == 0u &&
          matrix->padded_columns >= 16u * kChunk)
        most = std::max(most, kMostPieces * piece_bytes(kHeights[std::size(kHeights) - 1u],
                                                        swiglu));
      break;
    }
    const uint32_t last = static_cast<uint32_t>(std::min<uint64_t>(first + 15u, batch));
    for (const bool separate : {true, false}) {
      if (!separate && swiglu) continue;
      // (a cut tile's pieces are the same all along, so a plan that has them at any of
      // the rows has them at the last one)
      for (const uint32_t at : {row, last}) {
        const TallPlan plan = plan_tall(rows, matrix->padded_columns, at,
                                        matrix->scale_scheme, swiglu, separate, kPartsBytes);
        most = std::max(most, std::min(plan_bytes(plan, rows, last, swiglu), kPartsBytes));
      }
    }
  }
  return most;
}

extern "C" int32_t qllm_fp4_gemm_bf16_tall_partial(const qllm_fp4_matrix* matrix,
                                                   const void* input, size_t input_bytes,
                                                   float* partials, uint32_t parts,
                                                   uint32_t batch, void* stream) {
  TallArgs args{};
  if (!tall_arguments(matrix, input, input_bytes, batch, args) || !partials ||
      !parts || parts > kMaximumParts || parts > matrix->padded_columns / kChunk ||
      !workspace_ok(partials))
    return fail(QLLM_INVALID_ARGUMENT, "invalid partial tall FP4 GEMM");
  const TallPlan plan = plan_tall(args.rows, args.padded_columns, batch,
                                  matrix->scale_scheme, false, false, 0u, parts);
  args.partials = partials;
  args.output = partials;   // of a single part
  args.output_kind = QLLM_OUT_F32;
  return launch_tall(args, matrix->scale_scheme, plan, as_stream(stream));
}

extern "C" int32_t qllm_fp4_gemm_bf16_tall_cut(const qllm_fp4_matrix* matrix,
                                               const void* input, size_t input_bytes,
                                               void* output, uint32_t output_kind,
                                               const float* residual, uint32_t batch,
                                               void* workspace, size_t workspace_bytes,
                                               void* stream) {
  TallArgs args{};
  if (!tall_arguments(matrix, input, input_bytes, batch, args) || !output ||
      output_kind > QLLM_OUT_BF16 || !workspace_ok(workspace))
    return fail(QLLM_INVALID_ARGUMENT, "invalid tall FP4 GEMM");
  if (residual && output_kind == QLLM_OUT_BF16 &&
      static_cast<const void*>(residual) == output)
    return fail(QLLM_INVALID_ARGUMENT,
                "tall FP4 GEMM: bf16 output cannot alias the f32 residual");
  args.output = output;
  args.output_kind = output_kind;
  args.residual = residual;
  return run_tall(args, matrix->scale_scheme, workspace, workspace_bytes,
                  as_stream(stream));
}

extern "C" int32_t qllm_fp4_gemm_bf16_tall(const qllm_fp4_matrix* matrix,
                                           const void* input, size_t input_bytes,
                                           void* output, uint32_t output_kind,
                                           const float* residual, uint32_t batch,
                                           void* stream) {
  return qllm_fp4_gemm_bf16_tall_cut(matrix, input, input_bytes, output, output_kind,
                                     residual, batch, nullptr, 0u, stream);
}

extern "C" int32_t qllm_fp4_swiglu_bf16_tall_cut(const qllm_fp4_matrix* gate,
                                                 const qllm_fp4_matrix* up,
                                                 const void* input, size_t input_bytes,
                                                 void* output_bf16, uint32_t batch,
                                                 void* workspace, size_t workspace_bytes,
                                                 void* stream) {
  TallArgs args{};
  if (!tall_arguments(gate, input, input_bytes, batch, args) || !tall_matrix_ok(up) ||
      gate->rows != up->rows || gate->padded_columns != up->padded_columns ||
      gate->scale_scheme != up->scale_scheme || !output_bf16 || !workspace_ok(workspace))
    return fail(QLLM_INVALID_ARGUMENT, "invalid tall FP4 SwiGLU");
  args.up_weights = up->weights;
  args.up_scales = static_cast<const uint8_t*>(up->scales);
  args.output = output_bf16;
  args.output_kind = QLLM_OUT_BF16;
  return run_tall(args, gate->scale_scheme, workspace, workspace_bytes, as_stream(stream));
}

extern "C" int32_t qllm_fp4_swiglu_bf16_tall(const qllm_fp4_matrix* gate,
                                             const qllm_fp4_matrix* up,
                                             const void* input, size_t input_bytes,
                                             void* output_bf16, uint32_t batch,
                                             void* stream) {
  return qllm_fp4_swiglu_bf16_tall_cut(gate, up, input, input_bytes, output_bf16, batch,
                                       nullptr, 0u, stream);
}

extern "C" int32_t qllm_fp4_gemm_bf16_tall_split_cut(
    const qllm_fp4_matrix* matrix, const void* input, size_t input_bytes,
    const qllm_gemm_segment* segments, uint32_t segment_count, uint32_t batch,
    void* workspace, size_t workspace_bytes, void* stream) {
  TallArgs args{};
  if (!tall_arguments(matrix, input, input_bytes, batch, args) || !segments ||
      !segment_count || segment_count > 3u || !workspace_ok(workspace))
    return fail(QLLM_INVALID_ARGUMENT, "invalid split tall FP4 GEMM");
  uint64_t total = 0;
  for (uint32_t index = 0; index < segment_count; ++index) {
    if (!segments[index].output || !segments[index].rows ||
        segments[index].rows % kTileRows || segments[index].output_kind > QLLM_OUT_BF16)
      return fail(QLLM_INVALID_ARGUMENT,
                  "split tall FP4 GEMM: segments must be multiples of 32 rows");
    args.segment_rows[index] = segments[index].rows;
    args.segment_kind[index] = segments[index].output_kind;
    args.segment_output[index] = segments[index].output;
    total += segments[index].rows;
  }
  if (total != matrix->rows)
    return fail(QLLM_INVALID_ARGUMENT,
                "split tall FP4 GEMM: segments do not cover the matrix");
  args.segments = segment_count;
  return run_tall(args, matrix->scale_scheme, workspace, workspace_bytes,
                  as_stream(stream));
}

extern "C" int32_t qllm_fp4_gemm_bf16_tall_split(
    const qllm_fp4_matrix* matrix, const void* input, size_t input_bytes,
    const qllm_gemm_segment* segments, uint32_t segment_count, uint32_t batch,
    void* stream) {
  return qllm_fp4_gemm_bf16_tall_split_cut(matrix, input, input_bytes, segments,
                                           segment_count, batch, nullptr, 0u, stream);
}

// Linear layers with bf16 weights: several matrices per launch, each with its
// own input rows and epilogue (store, residual add, gated activation, K-split
// partial sums).
//
// The weights lie in fragment order: 16 rows x 32 columns are one contiguous
// KiB in which lane 16g + n finds row n, columns 8g .. 8g + 7 - its operand of
// v_mfma_f32_16x16x32_bf16.  Every weight load of a wave is one contiguous
// KiB and goes straight to the matrix cores, whatever the batch:
//
//  * up to 64 rows (decode): a workgroup owns one 16-row tile (two for the
//    gated epilogue), its eight waves split K and add their accumulators
//    through LDS in a fixed order.  Up to eight of a wave's loads are in flight at
//    once; a small batch costs one matrix instruction per KiB of weights.
//  * more rows (prompts): four waves side by side along the weight rows, each
//    with NT x MT accumulator tiles; the activation tile of 64 columns is
//    shared through LDS (copied there ahead of its step, one barrier per step,
//    16-byte pieces swizzled by row so that a fragment read touches every bank),
//    weights are prefetched one step ahead in registers.  An XCD gets a contiguous range
//    of the grid walked in bands of activation tiles, so operands are shared
//    in its L2.
//  * F32 mode runs on the same kernels: a 32-bit activation is the sum of three
//    bf16 values (its 24 significant bits, eight at a time), their products with
//    a bf16 weight are exact in 32 bits, and all three go into the same F32
//    accumulator.  Down to 2^-110 nothing of the activation is lost; below, where
//    the third part passes bf16's smallest step, what is lost is less than 2^-133.
//    Against 64 bits a product is 2 to 4 times closer than a chain of multiply-adds
//    over K was (of [11264, 2048] 1.9e-7 up to 64 rows and 4.9e-7 above, 8.1e-7
//    before), and it takes 13 us for one row and 73 for 333 instead of 330 and 440.
#include "common.hpp"
#include "mixed_norm.hpp"

#include <algorithm>
#include <cmath>
#include <iterator>
#include <utility>

namespace qllm {
namespace {

constexpr uint32_t kMaximumSegments = 8;
constexpr uint32_t kSmallWaves = 8;
constexpr uint32_t kBandTiles = 8;       // activation tiles per band of the grid

struct LinearArgs {
  qllm_linear_segment segment[kMaximumSegments];
  uint32_t first_unit[kMaximumSegments + 1];   // workgroups before segment s; ~0 past the last
  uint32_t count;
  uint32_t batch;
};

__device__ __forceinline__ uint32_t segment_of(const LinearArgs& args, uint32_t unit) {
  uint32_t index = 0;
#pragma unroll
  for (uint32_t i = 1; i < kMaximumSegments; ++i)   // (one trip to memory for all of them)
    index = unit >= args.first_unit[i] ? i : index;
  return index;
}

// Four consecutive output columns n .. n + 3 of batch row m.
__device__ __forceinline__ void store_four(const qllm_linear_segment& s, float* base,
                                           uint32_t m, uint32_t n, f32x4 value,
                                           bool add) {
  if (n >= s.output_columns) return;
  float* out = base + size_t{m} * s.output_stride + n;
  if (n + 4u <= s.output_columns && s.output_stride % 4u == 0u) {
    f32x4* vector = reinterpret_cast<f32x4*>(out);
    *vector = add ? *vector + value : value;
  } else {
    for (uint32_t i = 0; i < 4u && n + i < s.output_columns; ++i)
      out[i] = add ? out[i] + value[i] : value[i];
  }
}

template <typename T>
__device__ __forceinline__ void store_gated(const qllm_linear_segment& s, uint32_t m,
                                            uint32_t n, f32x4 gate, f32x4 up) {
  T* out = static_cast<T*>(s.output) + size_t{m} * s.output_stride + n;
  for (uint32_t i = 0; i < 4u && n + i < s.output_columns; ++i)
    store_element(out + i, activate(s.activation, gate[i]) * up[i]);
}

// ---- operands -----------------------------------------------------------------

// Eight consecutive input values of a row as they come from memory, and as
// operands of the matrix instructions: bf16 as it is, F32 in three bf16 parts.
template <bool F32>
struct Input;

template <>
struct Input<false> {
  static constexpr int kParts = 1;
  using Element = uint16_t;
  using Raw = i32x4;
  static __device__ __forceinline__ Raw load(const uint16_t* source) {
    return *reinterpret_cast<const i32x4*>(source);
  }
  static __device__ __forceinline__ void split(const Raw& raw, i32x4 (&out)[1]) {
    out[0] = raw;
  }
};

template <>
struct Input<true> {
  static constexpr int kParts = 3;
  using Element = float;
  struct Raw {
    f32x4 low, high;
  };
  static __device__ __forceinline__ Raw load(const float* source) {
    const f32x4* vector = reinterpret_cast<const f32x4*>(source);
    return {vector[0], vector[1]};
  }
  // The upper 16 bits of x are its first eight significant bits, x minus those
  // has sixteen left, and so on: every difference is exact, and with |x| >= 2^-110
  // the last one is a bf16.  An infinity is its first part alone; a NaN reaches the
  // second one whatever its bits are.
  static __device__ __forceinline__ void split(const Raw& raw, i32x4 (&out)[3]) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      uint32_t part[3][2];
#pragma unroll
      for (int half = 0; half < 2; ++half) {
        const int at = 2 * i + half;
        float rest = at < 4 ? raw.low[at] : raw.high[at - 4];
#pragma unroll
        for (int p = 0; p < 3; ++p) {
          part[p][half] = __float_as_uint(rest);
          const float top = __uint_as_float(part[p][half] & 0xffff0000u);
          rest = fabsf(rest) == INFINITY ? 0.0f : rest - top;
        }
      }
#pragma unroll
      for (int p = 0; p < 3; ++p)
        out[p][i] = static_cast<int>(
            __builtin_amdgcn_perm(part[p][1], part[p][0], 0x07060302u));
    }
  }
};

// Weights for the second and third part of an F32 input.  Those are often zero, and
// zero times an infinite weight would make a NaN of the infinity that the product
// is: they take the largest finite magnitude in its place, whose products have the
// same sign.  (A NaN is through with the first part as well.)
__device__ __forceinline__ i32x4 finite_weights(const i32x4& weights) {
  using u16x8 = uint16_t __attribute__((ext_vector_type(8)));
  const u16x8 bits = __builtin_bit_cast(u16x8, weights);
  const u16x8 magnitude = __builtin_elementwise_min(
      bits & static_cast<uint16_t>(0x7fff), u16x8(static_cast<uint16_t>(0x7f7f)));
  return __builtin_bit_cast(i32x4, (bits & static_cast<uint16_t>(0x8000)) | magnitude);
}

// Whether a sum has to be formed again with finite_weights.  (Changing the weights
// on the way to every product instead took the 32-bit decoder's turn from 3.28 to
// 3.68 ms; the question costs nothing measurable for a row and 0.2 us of 51 for 333
// rows of [8720, 2048].)
template <int N, int MT>
__device__ __forceinline__ bool any_nan(const f32x4 (&sum)[N][MT]) {
  bool found = false;
#pragma unroll
  for (int n = 0; n < N; ++n)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int i = 0; i < 4; ++i) found |= sum[n][mt][i] != sum[n][mt][i];
  return found;
}

// ---- up to 64 rows ------------------------------------------------------------

template <bool F32, int MT, int TILES, int UNROLL>
__device__ __forceinline__ void small_unit(const qllm_linear_segment& s, uint32_t unit,
                                           uint32_t batch, f32x4* scratch) {
  const uint32_t wave =
      MT == 1 && !F32 ? __builtin_amdgcn_readfirstlane(threadIdx.x / kWave) : threadIdx.x / kWave;
  const uint32_t lane = threadIdx.x % kWave;
  const uint32_t tiles = s.rows / (16u * TILES);
  const uint32_t parts = s.epilogue == QLLM_LINEAR_PARTIALS ? s.splits : 1u;
  const uint32_t part = unit / tiles;
  const uint32_t tile = unit % tiles;
  const uint32_t chunks = s.columns / 32u;
  const uint32_t part_begin = chunks * part / parts;
  const uint32_t span = chunks * (part + 1u) / parts - part_begin;
  const uint32_t begin = part_begin + span * wave / kSmallWaves;
  const uint32_t end = part_begin + span * (wave + 1u) / kSmallWaves;

  const i32x4* weights = static_cast<const i32x4*>(s.weights) +
                         size_t{tile} * TILES * chunks * kWave + lane;
  using In = Input<F32>;
  using Element = typename In::Element;
  const Element* input[MT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    const uint32_t row = min(mt * 16u + lane % 16u, batch - 1u);
    input[mt] = static_cast<const Element*>(s.input) + size_t{row} * s.input_stride +
                8u * (lane / 16u);
  }
  f32x4 sum[TILES][MT] = {};
  const auto multiply = [&](const i32x4 (&w)[TILES], const typename In::Raw& raw, int mt,
                            auto again) {
    i32x4 x[In::kParts];
    In::split(raw, x);
#pragma unroll
    for (int p = 0; p < In::kParts; ++p)
#pragma unroll
      for (int t = 0; t < TILES; ++t)
        sum[t][mt] =
            mfma_bf16(again() && p ? finite_weights(w[t]) : w[t], x[p], sum[t][mt]);
  };
  const auto one_by_one = [&](uint32_t from, auto again) {
    for (uint32_t chunk = from; chunk < end; ++chunk) {
      i32x4 w[TILES];
#pragma unroll
      for (int t = 0; t < TILES; ++t)
        w[t] = weights[(size_t{static_cast<uint32_t>(t)} * chunks + chunk) * kWave];
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
        multiply(w, In::load(input[mt] + chunk * 32u), mt, again);
    }
  };
  uint32_t chunk = begin;
  for (; chunk + UNROLL <= end; chunk += UNROLL) {
    i32x4 w[UNROLL][TILES];
    typename In::Raw x[UNROLL][MT];
#pragma unroll
    for (int u = 0; u < UNROLL; ++u)
#pragma unroll
      for (int t = 0; t < TILES; ++t)
        w[u][t] = __builtin_nontemporal_load(
            weights + (size_t{static_cast<uint32_t>(t)} * chunks + chunk + u) * kWave);
#pragma unroll
    for (int u = 0; u < UNROLL; ++u)
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) x[u][mt] = In::load(input[mt] + (chunk + u) * 32u);
#pragma unroll
    for (int u = 0; u < UNROLL; ++u)
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) multiply(w[u], x[u][mt], mt, std::false_type{});
  }
  if constexpr (F32 || MT > 1) {
    one_by_one(chunk, std::false_type{});
  } else {
    // What is left, its loads all in flight at once.  A wave's part is no whole number of
    // rounds in most layers (decoding one row, us, chunk by chunk and so: [2048, 7680] in
    // six parts 8.1 and 7.5, [3072, 1536] 6.2 and 4.1, [32000, 1024] 16.7 and 14.2; with
    // more registers for it 32-bit inputs would lose a workgroup a CU, 10.1 and 11.0).
    // Non-temporal like the rounds: in a decoder the launch by itself takes 7.1 and 7.4 then,
    // its weights staying in no cache, but the launches around it 0.3 - 0.7 less each, and a
    // turn of 32 tokens 6.46 and 6.24 ms (with plain loads 6.47).
    const auto rest = [&](auto count) __attribute__((always_inline)) {
      constexpr int N = count();
      // (of a single chunk, a matrix of few columns in the main, what the L2 may well hold)
      const auto stream = [](const i32x4* from) __attribute__((always_inline)) {
        return N > 1 ? __builtin_nontemporal_load(from) : *from;
      };
      if constexpr (N < UNROLL) {
        i32x4 w[N][TILES];
        typename In::Raw x[N];
#pragma unroll
        for (int u = 0; u < N; ++u)
#pragma unroll
          for (int t = 0; t < TILES; ++t)
            w[u][t] = stream(weights + (size_t{static_cast<uint32_t>(t)} * chunks + chunk + u) *
                                           kWave);
#pragma unroll
        for (int u = 0; u < N; ++u) x[u] = In::load(input[0] + (chunk + u) * 32u);
#pragma unroll
        for (int u = 0; u < N; ++u) multiply(w[u], x[u], 0, std::false_type{});
      }
    };
    switch (end - chunk) {
      case 1: rest(std::integral_constant<int, 1>{}); break;
      case 2: rest(std::integral_constant<int, 2>{}); break;
      case 3: rest(std::integral_constant<int, 3>{}); break;
      case 4: rest(std::integral_constant<int, 4>{}); break;
      case 5: rest(std::integral_constant<int, 5>{}); break;
      case 6: rest(std::integral_constant<int, 6>{}); break;
      case 7: rest(std::integral_constant<int, 7>{}); break;
      default: break;
    }
  }
  if constexpr (F32)
    if (__any(any_nan(sum))) {
#pragma unroll
      for (int t = 0; t < TILES; ++t)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) sum[t][mt] = f32x4{};
      one_by_one(begin, std::true_type{});
    }

#pragma unroll
  for (int t = 0; t < TILES; ++t)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
      scratch[((t * MT + mt) * kSmallWaves + wave) * kWave + lane] = sum[t][mt];
  __syncthreads();
  for (uint32_t index = threadIdx.x; index < MT * kWave; index += kSmallWaves * kWave) {
    const uint32_t mt = index / kWave;
    const uint32_t at = index % kWave;
    f32x4 total[TILES];
#pragma unroll
    for (int t = 0; t < TILES; ++t) {
      total[t] = scratch[(t * MT + mt) * kSmallWaves * kWave + at];
      for (uint32_t other = 1; other < kSmallWaves; ++other)
        total[t] += scratch[((t * MT + mt) * kSmallWaves + other) * kWave + at];
    }
    const uint32_t m = mt * 16u + at % 16u;
    const uint32_t n = tile * 16u + 4u * (at / 16u);
    if (m >= batch) continue;
    if constexpr (TILES == 2) {
      store_gated<Element>(s, m, n, total[0], total[1]);
    } else {
      float* base = static_cast<float*>(s.output) +
                    size_t{part} * batch * s.output_stride;
      store_four(s, base, m, n, total[0], s.epilogue == QLLM_LINEAR_ADD);
    }
  }
}

template <bool F32, int MT>
__global__ __launch_bounds__(kSmallWaves* kWave) void linear_small_kernel(LinearArgs args) {
  __shared__ f32x4 scratch[2 * MT * kSmallWaves * kWave];
  const uint32_t index = segment_of(args, blockIdx.x);
  const qllm_linear_segment& s = args.segment[index];
  const uint32_t unit = blockIdx.x - args.first_unit[index];
  // (F32 input takes twice the registers in flight)
  constexpr int kUnroll = F32 && MT > 2 ? 2 : MT > 1 ? 4 : 8;
  if (s.epilogue == QLLM_LINEAR_GATED)
    small_unit<F32, MT, 2, (kUnroll > 2 ? kUnroll / 2 : kUnroll)>(s, unit, args.batch,
                                                                  scratch);
  else
    small_unit<F32, MT, 1, kUnroll>(s, unit, args.batch, scratch);
}

// ---- one token with its norm ----------------------------------------------------
//
// A token's norm is one workgroup that everything waits for: 4 - 5 us of launch and memory
// latency, one or two of them a layer.  Here every workgroup of the projection takes
// the norm by itself instead, from the caches (up to ten rows, 80 KB at width 2048, as much
// as its weights), after its weight loads have set out, so that a token waits for one memory
// latency instead of two.  The weights stream through the registers: each is loaded for the
// next tile as soon as it has been used.  In 32-bit mode the activation is split into its
// parts once a workgroup instead of once for every matrix instruction.
// Norm of a row with six partial sums and projection, us, two launches and this one:
//   2048 columns, bf16: 545 tiles 12.2 -> 10.0, 996 15.6 -> 13.1, 2000 26.0 -> 22.9
//   2048 columns, F32: 545 tiles 14.6 -> 10.5, 996 19.1 -> 13.5, 2000 30.1 -> 23.0
//   4096 columns, bf16: 545 tiles 20.1 -> 16.5, 996 gated 56.9 -> 47.2

constexpr uint32_t kNormedThreads = kSmallWaves * kWave;
constexpr uint32_t kNormedWidth = 4u * kNormedThreads;   // values of a piece of every thread
constexpr uint32_t kNormedParts = 8;                     // most partial sums of the stream

struct NormedArgs {
  LinearArgs linear;                     // first_unit counts workgroups
  NormArgs norm;
  uint32_t source[kMaximumSegments];     // what a segment reads: weight[0 or 1], 2 + shift
};

// The norm's row `source` as operands of the matrix instructions (of 32-bit mode its three
// parts one after the other, kNormedWidth * PIECES apart), to `values`, zeros from the width
// on to `columns`: the sums, products and roundings of stream_norm_wide_kernel for one row,
// whose waves these are with PIECES == 1 and two by two with 2.  Workgroup `first` leaves
// the stream and the carried row.  `set_out` runs once all that the norm reads is asked for.
template <bool F32, int PIECES, typename SetOut>
__device__ __forceinline__ void normed_row(const NormArgs& args, uint32_t source,
                                           uint32_t columns, bool first, uint16_t* values,
                                           float* scratch, const SetOut& set_out) {
  constexpr uint32_t kRow = PIECES * kNormedWidth;
  const qllm_stream_norm_launch& l = args.launch;
  const qllm_token_shift& shift = args.shift;
  const uint32_t pieces = l.width / 4u;
  const uint32_t wave = threadIdx.x / kWave;
  const bool table = args.tokens.table != nullptr;
  const bool blended = source >= 2u;
  const auto row_of = [](const float* rows, uint32_t piece) {
    return reinterpret_cast<const f32x4*>(rows)[piece];
  };
  f32x4 held[PIECES], before[PIECES], weight[PIECES], share[PIECES];
  i32x4 part[PIECES][kNormedParts];
  // (absent partial sums lie past the end of the range: nothing is fetched)
  const auto parts =
      memory_range(l.partials, size_t{l.partial_count} * l.partial_stride * 4u);
#pragma unroll
  for (int i = 0; i < PIECES; ++i) {
    const uint32_t piece = min(threadIdx.x + i * kNormedThreads, pieces - 1u);
    held[i] = f32x4{};
    if (table) {
      if (const uint16_t* values16 = table_row(args, 0u)) {
        const i32x2 bits = reinterpret_cast<const i32x2*>(values16)[piece];
        held[i][0] = __int_as_float(bits[0]);
        held[i][1] = __int_as_float(bits[1]);
      }
    } else if (!l.branch_weight) {
      held[i] = row_of(l.input, piece);
    }
#pragma unroll
    for (uint32_t p = 0; p < kNormedParts; ++p)
      part[i][p] = __builtin_bit_cast(
          i32x4, __builtin_amdgcn_raw_buffer_load_b128(
                     parts, piece * 16u + p * l.partial_stride * 4u, 0, 0));
    if (l.branch_weight) {
      before[i] = row_of(l.input, piece);
      share[i] = row_of(l.branch_weight, piece);
    }
    if (blended) {
      before[i] = row_of(shift.previous + l.step[kStepSlot] * shift.slot_stride, piece);
      share[i] = row_of(shift.mu[source - 2u], piece);
    }
    weight[i] = row_of(l.weight[source == 1u ? 1 : 0], piece);
  }
  set_out();
#pragma unroll
  for (int i = 0; i < PIECES; ++i) {
    if (table)
      held[i] = bf16_values4(i32x2{__float_as_int(held[i][0]), __float_as_int(held[i][1])},
                             args.tokens.scale);
    if (l.partial_count)
#pragma unroll
      for (uint32_t p = 0; p < kNormedParts; ++p)
        held[i] += __builtin_bit_cast(f32x4, part[i][p]);
  }
  const auto inside = [&](int i) { return threadIdx.x + i * kNormedThreads < pieces; };
  const auto inverse_of = [&](float epsilon) __attribute__((always_inline)) {
    __syncthreads();
#pragma unroll
    for (int i = 0; i < PIECES; ++i) {
      float squares = 0.0f;
#pragma unroll
      for (int c = 0; c < 4; ++c) squares = fmaf(held[i][c], held[i][c], squares);
      squares = wave_sum(inside(i) ? squares : 0.0f);
      if (threadIdx.x % kWave == 0u) scratch[i * kSmallWaves + wave] = squares;
    }
    __syncthreads();
    float total = 0.0f;
#pragma unroll
    for (uint32_t w = 0; w < PIECES * kSmallWaves; ++w) total += scratch[w];
    return inverse_rms(total, l.width, epsilon);
  };
  if (l.branch_weight) {
    const float unit = inverse_of(l.branch_epsilon);
#pragma unroll
    for (int i = 0; i < PIECES; ++i)
#pragma unroll
      for (int c = 0; c < 4; ++c)
        held[i][c] = fmaf(held[i][c] * unit * share[i][c], l.branch_scale, before[i][c]);
  }
  if (first && (table || l.partial_count))
#pragma unroll
    for (int i = 0; i < PIECES; ++i)
      if (inside(i))
        reinterpret_cast<f32x4*>(l.stream_out)[threadIdx.x + i * kNormedThreads] = held[i];
  const float inverse = inverse_of(l.epsilon);
#pragma unroll
  for (int i = 0; i < PIECES; ++i) {
    if (!inside(i)) continue;
    const uint32_t piece = threadIdx.x + i * kNormedThreads;
    const f32x4 unit = held[i] * inverse;
    const f32x4 here = unit * weight[i];
    f32x4 value = here;
    if (blended)   // (rounded as the compiler does it there)
#pragma unroll
      for (int c = 0; c < 4; ++c)
        value[c] = fmaf(fmaf(-unit[c], weight[i][c], before[i][c]), share[i][c], here[c]);
    if constexpr (F32) {
      i32x4 split[3];
      Input<true>::split({value, f32x4{}}, split);
#pragma unroll
      for (int p = 0; p < 3; ++p)
        *reinterpret_cast<i32x2*>(values + p * kRow + piece * 4u) =
            i32x2{split[p][0], split[p][1]};
    } else {
      put4<uint16_t>(values, piece * 4u, value);
    }
    if (first && blended) reinterpret_cast<f32x4*>(shift.last)[piece] = here;
  }
  for (uint32_t c = l.width + threadIdx.x; c < columns; c += kNormedThreads)
#pragma unroll
    for (int p = 0; p < Input<F32>::kParts; ++p) values[p * kRow + c] = 0;
  __syncthreads();
}

// What a wave reads of a unit of TILES weight tiles: its eighth of the columns.
struct NormedPart {
  const i32x4* weights;
  uint32_t chunks, begin, end;   // of 32 columns: of the tile, of the wave
};

// A lane's 16 bytes of a chunk of a unit's tile `tile` of `tiles`.  Past the wave's part
// nothing is fetched, but there is a load all the same: the compiler knows how many are on
// their way.
__device__ __forceinline__ i32x4 load_weights(const NormedPart& part, uint32_t tiles,
                                              uint32_t unit, uint32_t chunk,
                                              uint32_t tile) {
  const uint32_t tile_bytes = part.chunks * kWave * 16u;
  const auto range = memory_range(part.weights + size_t{unit} * tiles * part.chunks * kWave,
                                  size_t{tiles} * tile_bytes);
  const uint32_t from =
      chunk < part.end ? chunk * (kWave * 16u) + tile * tile_bytes : 0x80000000u;
  return __builtin_bit_cast(
      i32x4, __builtin_amdgcn_raw_buffer_load_b128(range, threadIdx.x % kWave * 16u + from, 0,
                                                   2 /* non-temporal */));
}

// The units unit, unit + step, ... of a segment.  The first one's loads are in flight when
// this begins; afterwards every register is loaded again as soon as it has been used.
template <bool F32, int TILES, int PIECES>
__device__ __forceinline__ void normed_units(const qllm_linear_segment& s,
                                             const NormedPart& part, uint32_t unit,
                                             uint32_t step, const uint16_t* values,
                                             f32x4* scratch, i32x4 (&w)[8 * PIECES]) {
  constexpr uint32_t kRow = PIECES * kNormedWidth;
  constexpr uint32_t kUnroll = 8u * PIECES / TILES;
  constexpr int kParts = Input<F32>::kParts;
  const uint32_t wave = threadIdx.x / kWave;
  const uint32_t lane = threadIdx.x % kWave;
  const uint32_t units = s.rows / (16u * TILES);
  const uint16_t* input = values + 8u * (lane / 16u);
  const auto operand = [&](int p, uint32_t chunk) __attribute__((always_inline)) {
    return *reinterpret_cast<const i32x4*>(input + p * kRow + chunk * 32u);
  };
  for (; unit < units; unit += step) {
    const bool more = unit + step < units;
    f32x4 sum[TILES][1] = {};
    uint32_t chunk = part.begin;
    const auto multiply = [&](auto again, uint32_t next, uint32_t from)
                              __attribute__((always_inline)) {
#pragma unroll
      for (uint32_t u = 0; u < kUnroll; ++u) {
        if (chunk + u < part.end) {
#pragma unroll
          for (int p = 0; p < kParts; ++p)
#pragma unroll
            for (int t = 0; t < TILES; ++t)
              sum[t][0] = mfma_bf16(w[u * TILES + t], operand(p, chunk + u), sum[t][0]);
        }
        if constexpr (again())
#pragma unroll
          for (int t = 0; t < TILES; ++t)
            w[u * TILES + t] = load_weights(part, TILES, next, from + u, t);
      }
    };
    for (; chunk + kUnroll < part.end; chunk += kUnroll)
      multiply(std::true_type{}, unit, chunk + kUnroll);
    if (more)
      multiply(std::true_type{}, unit + step, part.begin);
    else
      multiply(std::false_type{}, 0u, 0u);
    if constexpr (F32)
      if (__any(any_nan(sum))) {
#pragma unroll
        for (int t = 0; t < TILES; ++t) sum[t][0] = f32x4{};
        for (uint32_t chunk = part.begin; chunk < part.end; ++chunk)
#pragma unroll
          for (int t = 0; t < TILES; ++t) {
            const i32x4 tile = load_weights(part, TILES, unit, chunk, t);
#pragma unroll
            for (int p = 0; p < kParts; ++p)
              sum[t][0] = mfma_bf16(p ? finite_weights(tile) : tile, operand(p, chunk),
                                    sum[t][0]);
          }
      }
#pragma unroll
    for (int t = 0; t < TILES; ++t)
      scratch[(t * kSmallWaves + wave) * kWave + lane] = sum[t][0];
    __syncthreads();
    if (wave == 0u) {
      f32x4 total[TILES];
#pragma unroll
      for (int t = 0; t < TILES; ++t) {
        total[t] = scratch[t * kSmallWaves * kWave + lane];
#pragma unroll
        for (uint32_t other = 1; other < kSmallWaves; ++other)
          total[t] += scratch[(t * kSmallWaves + other) * kWave + lane];
      }
      const uint32_t n = unit * 16u + 4u * (lane / 16u);
      if (lane % 16u == 0u) {
        if constexpr (TILES == 2)
          store_gated<typename Input<F32>::Element>(s, 0u, n, total[0], total[1]);
        else
          store_four(s, static_cast<float*>(s.output), 0u, n, total[0], false);
      }
    }
    if (more) __syncthreads();
  }
}

template <bool F32, int PIECES>
__global__ __launch_bounds__(kNormedThreads, PIECES == 1 ? 4 : 2) void linear_normed_kernel(
    NormedArgs args) {
  __shared__ f32x4 scratch[2 * kNormedThreads];
  __shared__ __attribute__((aligned(16))) uint16_t values[Input<F32>::kParts * PIECES *
                                                           kNormedWidth];
  __shared__ __attribute__((aligned(16))) float sums[PIECES * kSmallWaves];
  const uint32_t index = segment_of(args.linear, blockIdx.x);
  const qllm_linear_segment& s = args.linear.segment[index];
  const uint32_t first = args.linear.first_unit[index];
  const uint32_t step = args.linear.first_unit[index + 1u] - first;
  const uint32_t unit = blockIdx.x - first;
  const bool gated = s.epilogue == QLLM_LINEAR_GATED;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const uint32_t chunks = s.columns / 32u;
  const NormedPart part{static_cast<const i32x4*>(s.weights), chunks,
                        chunks * wave / kSmallWaves, chunks * (wave + 1u) / kSmallWaves};
  const uint32_t tiles = __builtin_amdgcn_readfirstlane(gated ? 2u : 1u);
  i32x4 w[8 * PIECES];
  normed_row<F32, PIECES>(
      args.norm, args.source[index], s.columns, blockIdx.x == 0u, values, sums,
      [&]() __attribute__((always_inline)) {
#pragma unroll
        for (uint32_t j = 0; j < 8u * PIECES; ++j)
          w[j] = gated ? load_weights(part, tiles, unit, part.begin + j / 2u, j % 2u)
                       : load_weights(part, tiles, unit, part.begin + j, 0u);
        __builtin_amdgcn_sched_barrier(0);
      });
  if (gated)
    normed_units<F32, 2, PIECES>(s, part, unit, step, values, scratch, w);
  else
    normed_units<F32, 1, PIECES>(s, part, unit, step, values, scratch, w);
}

// ---- tall batches --------------------------------------------------------------

// What a workgroup of 64 NT weight rows by 16 MT batch rows works on.
struct TallPlace {
  uint32_t segment, part, m_tile, n_tile;
};

template <int NT, int MT>
__device__ __forceinline__ TallPlace tall_place(const LinearArgs& args) {
  constexpr uint32_t kRowsM = MT * 16u;
  const uint32_t m_tiles = (args.batch + kRowsM - 1u) / kRowsM;
  // contiguous ranges of workgroups per XCD (consecutive ids go round the XCDs)
  uint32_t work = blockIdx.x;
  {
    const uint32_t per_xcd = gridDim.x / 8u;
    if (work < per_xcd * 8u) work = (work % 8u) * per_xcd + work / 8u;
  }
  const uint32_t index = segment_of(args, work);
  const qllm_linear_segment& s = args.segment[index];
  const uint32_t n_tiles = (s.rows + 64u * NT - 1u) / (64u * NT);
  const uint32_t part = (work - args.first_unit[index]) / (n_tiles * m_tiles);
  const uint32_t unit = (work - args.first_unit[index]) % (n_tiles * m_tiles);
  // bands of kBandTiles activation tiles, walked column by column
  const uint32_t band = unit / (kBandTiles * n_tiles);
  const uint32_t band_rows = min(kBandTiles, m_tiles - band * kBandTiles);
  const uint32_t in_band = unit - band * kBandTiles * n_tiles;
  return {index, part, band * kBandTiles + in_band % band_rows, in_band / band_rows};
}

// Stores a wave's sums: weight tiles first_tile + t, batch rows m_tile 16 MT + 16 mt.
template <bool F32, int NT, int MT>
__device__ __forceinline__ void store_tall(const LinearArgs& args, const TallPlace& place,
                                           uint32_t first_tile, f32x4 (&sum)[NT][MT]) {
  using Element = typename Input<F32>::Element;
  constexpr uint32_t kRowsM = MT * 16u;
  const qllm_linear_segment& s = args.segment[place.segment];
  const uint32_t m_tile = place.m_tile;
  const uint32_t part = place.part;
  const uint32_t lane = threadIdx.x % kWave;
  const uint32_t weight_tiles = s.rows / 16u;
  // What the sums are added to is fetched before anything is stored, and - where
  // the wave's tiles are whole - all of it at once: every load after a store would
  // wait for all before it.
  if (s.epilogue == QLLM_LINEAR_ADD) {
    const bool whole =
        s.output_stride % 4u == 0u && (first_tile + NT) * 16u <= s.output_columns;
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      const uint32_t m = min(m_tile * kRowsM + mt * 16u + lane % 16u, args.batch - 1u);
      const float* out = static_cast<const float*>(s.output) + size_t{m} * s.output_stride +
                         first_tile * 16u + 4u * (lane / 16u);
      if (whole) {
#pragma unroll
        for (int t = 0; t < NT; ++t)
          sum[t][mt] += *reinterpret_cast<const f32x4*>(out + t * 16);
        continue;
      }
      for (int t = 0; t < NT; ++t)
        for (uint32_t i = 0; i < 4u; ++i)
          if (first_tile * 16u + 4u * (lane / 16u) + t * 16u + i < s.output_columns)
            sum[t][mt][i] += out[t * 16 + i];
    }
  }
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    const uint32_t m = m_tile * kRowsM + mt * 16u + lane % 16u;
    if (m >= args.batch) continue;
    if (s.epilogue == QLLM_LINEAR_GATED) {
      if constexpr (NT % 2 == 0) {
#pragma unroll
        for (int t = 0; t < NT; t += 2) {
          const uint32_t at = first_tile + t;
          if (at >= weight_tiles) continue;
          const uint32_t n = at / 2u * 16u + 4u * (lane / 16u);
          if (!F32 && n + 4u <= s.output_columns && s.output_stride % 4u == 0u) {
            const f32x4 gate = sum[t][mt];
            const f32x4 up = sum[t + 1][mt];
            uint32_t bits[4];
#pragma unroll
            for (int i = 0; i < 4; ++i)
              bits[i] = f32_to_bf16_bits(activate(s.activation, gate[i]) * up[i]);
            *reinterpret_cast<i32x2*>(static_cast<uint16_t*>(s.output) +
                                      size_t{m} * s.output_stride + n) =
                i32x2{static_cast<int>(bits[0] | bits[1] << 16),
                      static_cast<int>(bits[2] | bits[3] << 16)};
          } else {
            store_gated<Element>(s, m, n, sum[t][mt], sum[t + 1][mt]);
          }
        }
      }
    } else {
#pragma unroll
      for (int t = 0; t < NT; ++t)
        if (first_tile + t < weight_tiles)
          store_four(s,
                     static_cast<float*>(s.output) +
                         size_t{part} * args.batch * s.output_stride,
                     m, (first_tile + t) * 16u + 4u * (lane / 16u), sum[t][mt], false);
    }
  }
}

// bf16 input.  Bound by the matrix cores and by what their waves wait for: with the
// activation tile staged through registers a step ahead they were busy 63 % of the time
// over thousands of rows.  Here the tile goes from memory straight to the LDS two or three
// steps ahead, without a register, an address or a store of the wave's; weights go to
// registers a step ahead, and a half's activations are read in between the products of
// the half before.  6000 rows by [28672, 4096] 1285 -> 1153 us (1097 -> 1222 TFLOP/s), by
// [4096, 18432] 833 -> 721, by [11264, 2048] 294 -> 258; 300 rows of the three 110 -> 104,
// 69.5 -> 68.2, 29.8 -> 29.2.  The tiles are arrays of their own: of one array's parts the
// compiler would have every read wait for all copies.
//
// LOADS_FIRST: a workgroup that has a CU to itself, or shares it with one other that is as
// high as wide, waits for its loads, so they go out before anything else (70 rows by [8192,
// 2048], 128 workgroups, 19.8 -> 17.8 us); where more share a CU they go out between the
// products (500 rows by the same, 512 workgroups, 28.2 us, and 29.8 the other way).
//
// FAR: input rows 2^24 values apart and more, past a 32-bit offset over 128 of them; every
// lane has a 64-bit address of its own.
template <int NT, int MT, bool LOADS_FIRST, bool FAR = false>
__global__ __launch_bounds__(256, 2) void linear_tall_kernel(LinearArgs args) {
  constexpr uint32_t kRowsM = MT * 16u;
  constexpr uint32_t kPieces = kRowsM * 8u;           // 16-byte pieces of a tile
  constexpr uint32_t kLoads = kPieces / 256u;
  static_assert(kPieces % 256u == 0u);
  // (three workgroups of 128 weight rows fit a CU, with a fourth tile two)
  constexpr int kTiles = NT > 2 ? 4 : 3;
  constexpr uint32_t kStepLoads = kLoads + 2u * NT;
  __shared__ i32x4 tile0[kPieces];
  __shared__ i32x4 tile1[kPieces];
  __shared__ i32x4 tile2[kPieces];
  __shared__ i32x4 tile3[kTiles > 3 ? kPieces : 1u];

  const TallPlace place = tall_place<NT, MT>(args);
  const qllm_linear_segment& s = args.segment[place.segment];
  const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const uint32_t lane = threadIdx.x % kWave;
  const uint32_t chunks = s.columns / 32u;
  const uint32_t steps = s.columns / 64u;
  const uint32_t parts = s.epilogue == QLLM_LINEAR_PARTIALS ? s.splits : 1u;
  const uint32_t first_step = steps * place.part / parts;
  const uint32_t end_step = steps * (place.part + 1u) / parts;
  const uint32_t weight_tiles = s.rows / 16u;
  const uint32_t first_tile = (place.n_tile * 4u + wave) * NT;

  const i32x4* weights[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t)
    weights[t] = static_cast<const i32x4*>(s.weights) +
                 size_t{min(first_tile + t, weight_tiles - 1u)} * chunks * kWave;

  // piece p of the tile: row p / 8, swizzled slot p % 8; rows past the batch are not read
  const size_t first_row = size_t{place.m_tile} * kRowsM;
  const auto input = memory_range(
      static_cast<const uint16_t*>(s.input) + first_row * s.input_stride,
      (args.batch - first_row) * s.input_stride * 2u);
  uint32_t source[kLoads];
#pragma unroll
  for (uint32_t i = 0; i < kLoads; ++i) {
    const uint32_t piece = i * 256u + threadIdx.x;
    const uint32_t row = piece / 8u;
    source[i] = (row * s.input_stride + ((piece % 8u) ^ (row % 8u)) * 8u) * 2u;
  }
  const uint32_t fragment[2] = {(lane % 16u) * 8u + ((lane / 16u) ^ (lane % 8u)),
                                (lane % 16u) * 8u + ((4u + lane / 16u) ^ (lane % 8u))};

  f32x4 sum[NT][MT] = {};
  i32x4 held[2][2][NT];   // [step parity][half of 32 columns][tile]
  const auto copy_input = [&](i32x4* to, uint32_t step) {
#pragma unroll
    for (uint32_t i = 0; i < kLoads; ++i)
      if constexpr (FAR) {   // (rows past the batch are its last one here)
        const uint32_t piece = i * 256u + threadIdx.x;
        const size_t row = min(first_row + piece / 8u, size_t{args.batch - 1u});
        copy16_to_lds(static_cast<const uint16_t*>(s.input) + row * s.input_stride +
                          step * 64u + ((piece ^ piece / 8u) % 8u) * 8u,
                      to + i * 256u + wave * kWave);
      } else {
        copy16_to_lds(input, source[i], step * 128u, to + i * 256u + wave * kWave);
      }
  };
  const auto fetch_weights = [&](uint32_t slot, uint32_t step) {
#pragma unroll
    for (int half = 0; half < 2; ++half)
#pragma unroll
      for (int t = 0; t < NT; ++t)
        held[slot][half][t] = weights[t][(step * 2u + half) * kWave + lane];
  };
  // (a part without steps, of more parts than steps, loads the last one for nothing)
  const uint32_t last = end_step > first_step ? end_step - 1u : min(first_step, steps - 1u);
  const auto tile_of = [&](int position) {
    position %= kTiles;
    return position == 0 ? tile0 : position == 1 ? tile1 : position == 2 ? tile2 : tile3;
  };
  // (in this order: the waits count on the tiles one after the other, weights behind them)
#pragma unroll
  for (int ahead = 0; ahead + 1 < kTiles; ++ahead) {
    copy_input(tile_of(ahead), min(first_step + ahead, last));
    __builtin_amdgcn_sched_barrier(0);
  }
  fetch_weights(0u, min(first_step, last));
  __builtin_amdgcn_sched_barrier(0);
  wait_for_loads<(kTiles - 2u) * kLoads + 2u * NT>();

  const auto step_at = [&]<int P>(std::integral_constant<int, P>, uint32_t step) {
    const i32x4* current = tile_of(P);
    // this step's copies are there: what later steps asked for may be on its way
    wait_for_loads<(kTiles - 2u) * kStepLoads>();
    barrier_beside_copies();   // everybody's are, and the tile before has been read
    i32x4 x[MT];
    const auto read_first_half = [&] {
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) x[mt] = current[mt * 128 + fragment[0]];
    };
    if constexpr (!LOADS_FIRST) read_first_half();
    fetch_weights((P + 1) % 2, min(step + 1u, last));
    copy_input(tile_of(P + kTiles - 1), min(step + kTiles - 1u, last));
    if constexpr (LOADS_FIRST) {
      __builtin_amdgcn_sched_barrier(0);
      read_first_half();
    }
#pragma unroll
    for (int half = 0; half < 2; ++half)
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) {
#pragma unroll
        for (int t = 0; t < NT; ++t)
          sum[t][mt] = mfma_bf16(held[P % 2][half][t], x[mt], sum[t][mt]);
        if (half == 0) x[mt] = current[mt * 128 + fragment[1]];
      }
    // loads and the second half's reads go between the products
    __builtin_amdgcn_sched_group_barrier(0x100, MT, 0);
#pragma unroll
    for (int half = 0; half < 2; ++half)
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) {
        __builtin_amdgcn_sched_group_barrier(0x008, NT, 0);
        if (!LOADS_FIRST) __builtin_amdgcn_sched_group_barrier(0x020, 2, 0);
        if (half == 0) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
      }
    __builtin_amdgcn_sched_barrier(0);
  };
  constexpr int kRound = kTiles % 2 ? 2 * kTiles : kTiles;
  // Rounds of steps, after which every tile and slot has had its turn, and what is left.
  // (Of a loop that is left within a round the compiler takes every step for the one before
  // the next round, which then starts with a wait for copies and weights just asked for.)
  uint32_t step = first_step;
  for (; step + kRound <= end_step; step += kRound)
    [&]<int... P>(std::integer_sequence<int, P...>) {
      (step_at(std::integral_constant<int, P>{}, step + P), ...);
    }(std::make_integer_sequence<int, kRound>{});
  if (step < end_step)
    [&]<int... P>(std::integer_sequence<int, P...>) {
      (void)((step_at(std::integral_constant<int, P>{}, step + P), step + P + 1u < end_step) &&
             ...);
    }(std::make_integer_sequence<int, kRound - 1>{});
  wait_for_loads<0>();   // no copy outlives its workgroup
  store_tall<false, NT, MT>(args, place, first_tile, sum);
}

// 32-bit input, which is cut into its three parts on its way to the LDS.
template <int NT, int MT>
__global__ __launch_bounds__(256, 2) void linear_tall_f32_kernel(LinearArgs args) {
  using In = Input<true>;
  using Element = float;
  constexpr int kParts = In::kParts;
  constexpr uint32_t kRowsM = MT * 16u;
  constexpr uint32_t kPieces = kRowsM * 8u;           // 16-byte pieces of a tile
  constexpr uint32_t kLoads = kPieces / 256u;
  static_assert(kPieces % 256u == 0u);
  __shared__ i32x4 tile[2][kParts][kPieces];

  const TallPlace place = tall_place<NT, MT>(args);
  const qllm_linear_segment& s = args.segment[place.segment];
  const uint32_t wave = threadIdx.x / kWave;
  const uint32_t lane = threadIdx.x % kWave;
  const uint32_t chunks = s.columns / 32u;
  const uint32_t steps = s.columns / 64u;
  const uint32_t parts = s.epilogue == QLLM_LINEAR_PARTIALS ? s.splits : 1u;
  const uint32_t first_step = steps * place.part / parts;
  const uint32_t end_step = steps * (place.part + 1u) / parts;
  const uint32_t weight_tiles = s.rows / 16u;
  const uint32_t first_tile = (place.n_tile * 4u + wave) * NT;

  const i32x4* weights[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t)
    weights[t] = static_cast<const i32x4*>(s.weights) +
                 size_t{min(first_tile + t, weight_tiles - 1u)} * chunks * kWave + lane;

  // piece p of the tile: row p / 8, swizzled slot p % 8
  const Element* source[kLoads];
#pragma unroll
  for (uint32_t i = 0; i < kLoads; ++i) {
    const uint32_t piece = i * 256u + threadIdx.x;
    const uint32_t row = piece / 8u;
    const uint32_t column = (piece % 8u) ^ (row % 8u);
    const uint32_t batch_row = min(place.m_tile * kRowsM + row, args.batch - 1u);
    source[i] = static_cast<const Element*>(s.input) +
                size_t{batch_row} * s.input_stride + column * 8u;
  }

  f32x4 sum[NT][MT] = {};
  typename In::Raw staged[kLoads];
  i32x4 held[2][2][NT];   // [step parity][half of 32 columns][tile]
  const auto fetch_input = [&](uint32_t step) {
#pragma unroll
    for (uint32_t i = 0; i < kLoads; ++i) staged[i] = In::load(source[i] + step * 64u);
  };
  const auto store_input = [&](uint32_t buffer) {
#pragma unroll
    for (uint32_t i = 0; i < kLoads; ++i) {
      i32x4 split[kParts];
      In::split(staged[i], split);
#pragma unroll
      for (int p = 0; p < kParts; ++p) tile[buffer][p][i * 256u + threadIdx.x] = split[p];
    }
  };
  const auto fetch_weights = [&](auto slot, uint32_t step) {
#pragma unroll
    for (int half = 0; half < 2; ++half)
#pragma unroll
      for (int t = 0; t < NT; ++t)
        held[slot][half][t] = weights[t][(step * 2u + half) * kWave];
  };
  constexpr std::integral_constant<int, 0> even;
  constexpr std::integral_constant<int, 1> odd;
  // (a part without steps, of more parts than steps, loads the last one for nothing)
  fetch_input(min(first_step, steps - 1u));
  fetch_weights(even, min(first_step, steps - 1u));
  store_input(0u);
  __syncthreads();

  const auto step_at = [&](uint32_t step, auto parity) {
    constexpr int P = decltype(parity)::value;
    const uint32_t next = min(step + 1u, end_step - 1u);   // the last one re-reads itself
    fetch_input(next);
    fetch_weights(std::integral_constant<int, 1 - P>{}, next);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int half = 0; half < 2; ++half)
#pragma unroll
      for (int p = 0; p < kParts; ++p) {
        i32x4 x[MT];
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
          const uint32_t row = mt * 16u + lane % 16u;
          const uint32_t column = half * 4u + lane / 16u;
          x[mt] = tile[P][p][row * 8u + (column ^ (row % 8u))];
        }
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
          for (int t = 0; t < NT; ++t)
            sum[t][mt] = mfma_bf16(held[P][half][t], x[mt], sum[t][mt]);
      }
    store_input(1 - P);
    __syncthreads();
  };
  uint32_t step = first_step;
  for (; step + 2u <= end_step; step += 2u) {
    step_at(step, even);
    step_at(step + 1u, odd);
  }
  if (step < end_step) step_at(step, even);
  if (__any(any_nan(sum))) {   // this wave's alone, its inputs past the LDS
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) sum[t][mt] = f32x4{};
    for (uint32_t chunk = 2u * first_step; chunk < 2u * end_step; ++chunk)
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) {
        const uint32_t row = min(place.m_tile * kRowsM + mt * 16u + lane % 16u, args.batch - 1u);
        i32x4 x[kParts];
        In::split(In::load(static_cast<const Element*>(s.input) +
                           size_t{row} * s.input_stride + chunk * 32u + 8u * (lane / 16u)),
                  x);
#pragma unroll
        for (int t = 0; t < NT; ++t) {
          const i32x4 w = weights[t][chunk * kWave];
#pragma unroll
          for (int p = 0; p < kParts; ++p)
            sum[t][mt] = mfma_bf16(p ? finite_weights(w) : w, x[p], sum[t][mt]);
        }
      }
  }

  store_tall<true, NT, MT>(args, place, first_tile, sum);
}

__global__ void linear_pack_kernel(const uint16_t* source, uint32_t rows, uint32_t columns,
                                   uint64_t row_stride, uint64_t column_stride,
                                   uint16_t* packed, uint32_t packed_chunks,
                                   uint32_t first_tile, uint32_t tile_stride,
                                   uint32_t first_chunk, uint32_t chunks,
                                   uint64_t elements) {
  for (uint64_t i = uint64_t{blockIdx.x} * blockDim.x + threadIdx.x; i < elements;
       i += uint64_t{gridDim.x} * blockDim.x) {
    const uint32_t in_fragment = static_cast<uint32_t>(i % 512u);
    const uint64_t fragment = i / 512u;
    const uint32_t chunk = static_cast<uint32_t>(fragment % chunks);
    const uint32_t tile = static_cast<uint32_t>(fragment / chunks);
    const uint32_t lane = in_fragment / 8u;
    const uint32_t row = tile * 16u + lane % 16u;
    const uint32_t column = chunk * 32u + lane / 16u * 8u + in_fragment % 8u;
    const uint16_t value = row < rows && column < columns
                               ? source[row * row_stride + column * column_stride]
                               : uint16_t{0};
    packed[(uint64_t{first_tile + tile * tile_stride} * packed_chunks + first_chunk +
            chunk) * 512u + in_fragment] = value;
  }
}

uint32_t parts_of(const qllm_linear_segment& s) {
  return s.epilogue == QLLM_LINEAR_PARTIALS ? s.splits : 1u;
}

// The forms of the tall kernel: NT weight tiles of 16 rows a wave, MT activation
// tiles of 16 rows a workgroup.
//
// Which one, and how many parts of K where the caller can take parts, follows from
// what the busiest CU will take: n = ceil(workgroups / 256) workgroups over their
// steps of 64 columns, a step `alone` ns for n = 1 and n * `shared` where workgroups
// hide each other's round trips, and parts written and read at 6.5 TB/s.  The
// constants are a fit to 1150 timed launches over weights from memory (eight
// matrices of [2048, 2048] to [24576, 4096], 66 to 3000 rows; 8 % root mean square
// error) of the kernel that staged its activation tile through registers; 32-bit input
// still runs it.  What they picked there was 0.7 % slower than the best of those timed, the
// rule before it - largest tiles that give two workgroups a CU, K never cut - 68 %: [2048,
// 7680] 100 rows 62 -> 13 us, 1000 rows 60 -> 40, 3000 rows 117 -> 93; in 32 bits 100 rows
// 141 -> 20, 500 rows 143 -> 47.  With the tiles copied straight to the LDS the form they
// pick for given parts is 2.1 % slower than the best of the three (368 launches of twenty
// matrices, 65 to 3000 rows; 1.23 at worst).  A fit of those took 0.9 % and lost up to 1.2
// in launches that are at their best now.
struct TallForm {
  uint32_t nt, mt;
  float alone, shared;
};
constexpr TallForm kTallForms[] = {
    {2, 4, 435.f, 325.f}, {2, 8, 725.f, 515.f}, {4, 8, 1130.f, 895.f}};
constexpr TallForm kTallFormsF32[] = {{2, 4, 1105.f, 775.f}, {4, 4, 1525.f, 1230.f}};

uint64_t tall_units(const TallForm& form, uint32_t rows, uint32_t batch) {
  return uint64_t{(rows + 64u * form.nt - 1u) / (64u * form.nt)} *
         ((batch + 16u * form.mt - 1u) / (16u * form.mt));
}

// Time of `units` workgroups that run `steps` steps on average.
double tall_time(const TallForm& form, double units, double steps) {
  const double on_one = std::ceil(units / 256.0);
  return steps * std::max<double>(form.alone, on_one * form.shared);
}

// Calls visit(form, index) for the forms of an element type.
template <typename Visit>
void each_form(bool f32, const Visit& visit) {
  if (f32)
    for (uint32_t i = 0; i < std::size(kTallFormsF32); ++i) visit(kTallFormsF32[i], i);
  else
    for (uint32_t i = 0; i < std::size(kTallForms); ++i) visit(kTallForms[i], i);
}

// Values between input rows from which on a lane's 32-bit offset does not reach over 128.
constexpr uint32_t kFarStride = 1u << 24;

// More than two workgroups of 64 x 128 a CU share more of its cache's rate than it has: a
// step of 64 columns is 24 KB for half the products of 128 x 128 with 32.  Large matrices in
// many steps show it: 400 rows by [12288, 4096] 71.4 us and with 128 x 128 62.2, 160 rows by
// [4096, 18432] in eight parts 54.1 and 45.8, by [32000, 2048] 46.5 and 40.8, 26 others 0.87
// to 1.02.  Smaller ones, or of fewer steps, are up to 1.2 times as fast with 64 x 128 (1500
// rows by [2816, 1024] 18.2 and 21.9, by [3072, 3072] 44.7 and 47.2).
constexpr double kMostSmall = 2.0, kManySteps = 24.0, kLargeMatrix = 1 << 24;

bool rows_far_apart(const LinearArgs& args) {
  bool far = false;
  for (uint32_t i = 0; i < args.count; ++i)
    far |= args.segment[i].input_stride >= kFarStride;
  return far;
}

// The form for a launch whose parts are given.
uint32_t tall_form(const LinearArgs& args, bool f32) {
  const bool far = !f32 && rows_far_apart(args);
  uint32_t best = 0;
  double least = 0.0;
  each_form(f32, [&](const TallForm& form, uint32_t index) {
    if (far && form.nt > 2u) return;   // (no registers left for addresses)
    double units = 0.0;
    double work = 0.0;
    double weights = 0.0;
    for (uint32_t i = 0; i < args.count; ++i) {
      const auto& s = args.segment[i];
      weights += static_cast<double>(s.rows) * s.columns;
      const double own = static_cast<double>(tall_units(form, s.rows, args.batch));
      units += own * parts_of(s);
      work += own * (s.columns / 64u);
    }
    const double time = tall_time(form, units, work / units);
    if (!f32 && index == 0u && units > kMostSmall * 256.0 && work / units >= kManySteps &&
        weights >= kLargeMatrix)
      return;
    if (least == 0.0 || time < least) {
      best = index;
      least = time;
    }
  });
  return best;
}

// Workgroups up to which a launch asks for its loads first.  64 x 128: as many as CUs (128 to
// 256: 5 to 12 % faster so; 286 to 312: 2 to 5 % slower, 500 rows by [8192, 2048], 512, 6 %).
// 128 x 128: two a CU (448 to 512: 2 to 4 % faster, 65 rows by [5120, 17408] in twelve parts
// 45.4 -> 43.8 us; 752: 2 to 4 % slower).
constexpr uint32_t loads_first_up_to(int mt) { return mt == 4 ? 256u : 512u; }

template <bool F32, int NT, int MT>
int32_t launch_tall(LinearArgs& args, hipStream_t stream) {
  args.first_unit[0] = 0;
  for (uint32_t i = 0; i < args.count; ++i)
    args.first_unit[i + 1] =
        args.first_unit[i] +
        static_cast<uint32_t>(tall_units({NT, MT, 0.f, 0.f}, args.segment[i].rows,
                                         args.batch)) *
            parts_of(args.segment[i]);
  const uint32_t grid = args.first_unit[args.count];
  if constexpr (F32) {
    linear_tall_f32_kernel<NT, MT><<<grid, 256, 0, stream>>>(args);
  } else if constexpr (NT > 2) {
    linear_tall_kernel<NT, MT, false><<<grid, 256, 0, stream>>>(args);
  } else if (rows_far_apart(args)) {
    linear_tall_kernel<NT, MT, false, true><<<grid, 256, 0, stream>>>(args);
  } else if (grid <= loads_first_up_to(MT)) {
    linear_tall_kernel<NT, MT, true><<<grid, 256, 0, stream>>>(args);
  } else {
    linear_tall_kernel<NT, MT, false><<<grid, 256, 0, stream>>>(args);
  }
  return launched("tall linear");
}

template <bool F32, int MT>
void launch_small(const LinearArgs& args, hipStream_t stream) {
  linear_small_kernel<F32, MT>
      <<<args.first_unit[args.count], kSmallWaves * kWave, 0, stream>>>(args);
}

}  // namespace
}  // namespace qllm

using namespace qllm;

extern "C" size_t qllm_linear_packed_bytes(uint32_t rows, uint32_t columns) {
  return size_t{(rows + 15u) / 16u * 16u} * ((size_t{columns} + 63u) / 64u * 64u) * 2u;
}

extern "C" int32_t qllm_linear_pack(const void* source_bf16, uint32_t rows, uint32_t columns,
                                    void* packed, uint32_t packed_columns,
                                    uint32_t first_tile, uint32_t tile_stride,
                                    uint32_t first_column, void* stream) {
  return qllm_linear_pack_strided(source_bf16, rows, columns, columns, 1u, packed,
                                  packed_columns, first_tile, tile_stride, first_column,
                                  stream);
}

extern "C" int32_t qllm_linear_pack_strided(const void* source_bf16, uint32_t rows,
                                            uint32_t columns, uint64_t row_stride,
                                            uint64_t column_stride, void* packed,
                                            uint32_t packed_columns, uint32_t first_tile,
                                            uint32_t tile_stride, uint32_t first_column,
                                            void* stream) {
  const uint32_t padded = (columns + 63u) / 64u * 64u;
  if (!source_bf16 || !packed || !rows || !columns || !tile_stride ||
      packed_columns % 64u || first_column % 64u || !aligned16(packed) ||
      packed_columns < padded || first_column > packed_columns - padded)
    return fail(QLLM_INVALID_ARGUMENT, "invalid linear pack");
  const uint32_t chunks = padded / 32u;
  const uint64_t elements = uint64_t{(rows + 15u) / 16u} * chunks * 512u;
  const uint32_t blocks =
      static_cast<uint32_t>(elements / 256u < 65536u ? (elements + 255u) / 256u : 65536u);
  linear_pack_kernel<<<blocks, 256, 0, as_stream(stream)>>>(
      static_cast<const uint16_t*>(source_bf16), rows, columns, row_stride, column_stride,
      static_cast<uint16_t*>(packed), packed_columns / 32u, first_tile, tile_stride,
      first_column / 32u, chunks, elements);
  return launched("linear pack");
}

namespace {

int32_t linear_arguments(const qllm_linear_segment* segments, uint32_t count,
                         uint32_t batch, uint32_t element, LinearArgs& args) {
  if (!segments || !count || count > kMaximumSegments || !batch ||
      element > QLLM_ELEMENT_F32)
    return fail(QLLM_INVALID_ARGUMENT, "invalid linear batch");
  args.count = count;
  args.batch = batch;
  std::fill(std::begin(args.first_unit) + 1, std::end(args.first_unit), ~0u);
  for (uint32_t i = 0; i < count; ++i) {
    const qllm_linear_segment& s = segments[i];
    const bool gated = s.epilogue == QLLM_LINEAR_GATED;
    const bool partials = s.epilogue == QLLM_LINEAR_PARTIALS;
    const uint32_t outputs = gated ? s.rows / 2u : s.rows;
    if (!s.weights || !s.input || !s.output || !s.rows || !s.columns ||
        s.rows % (gated ? 32u : 16u) || s.columns % 64u || s.input_stride < s.columns ||
        s.input_stride % 8u || !s.output_columns ||
        s.output_columns > outputs || s.output_stride < s.output_columns ||
        s.epilogue > QLLM_LINEAR_PARTIALS || s.activation > QLLM_ACTIVATION_SILU ||
        (partials && (!s.splits || s.splits > 16u)) ||
        !aligned16(s.weights) || !aligned16(s.input) || !aligned16(s.output))
      return fail(QLLM_INVALID_ARGUMENT, "invalid linear segment");
    args.segment[i] = s;
  }
  return QLLM_OK;
}

// batch rows of a workgroup of the form for up to 64
uint32_t small_rows(uint32_t batch) { return batch <= 16u ? 16u : batch <= 32u ? 32u : 64u; }

// Which row of the norm every segment reads; false where the launch is not one of
// linear_normed_kernel: rows it does not hold, and where two launches are faster.  Those are
// many short tiles, which leave the workgroups too little to read at a time (256 columns,
// two launches against one: 2000 gated tiles 13.5 and 13.1 us, 3000 16.7 and 18.0, 8000 31.9
// and 38.4), and heads of a workgroup a CU that are long enough to hide a norm (4096 columns
// of bf16: 3000 tiles 66.1 and 65.1 us, 4500 94.1 and 94.3, 8000 159.4 and 161.4).
bool normed_sources(NormedArgs& args) {
  const qllm_stream_norm_launch& l = args.norm.launch;
  if (l.rows != 1u || l.gather || l.width > 2u * kNormedWidth ||
      l.partial_count > kNormedParts || l.partial_stride >= 1u << 24)
    return false;
  bool carried = !l.shift;   // the shift's last row is left by workgroup 0
  uint64_t stored = 0, gated = 0;
  uint32_t columns = ~0u;
  for (uint32_t i = 0; i < args.linear.count; ++i) {
    const qllm_linear_segment& s = args.linear.segment[i];
    const uint32_t most = l.width <= kNormedWidth ? kNormedWidth : 2u * kNormedWidth;
    uint32_t source = ~0u;
    if (l.shift)
      for (uint32_t b = 0; b < l.shift->count; ++b)
        if (l.shift->output[b] == s.input) source = 2u + b;
    for (uint32_t o = l.shift ? 1u : 0u; o < 2u && source == ~0u; ++o)
      if (l.weight[o] && l.output[o] == s.input) source = o;
    if (source == ~0u || s.columns > most ||
        s.columns > l.stride[source == 1u ? 1 : 0] || s.epilogue == QLLM_LINEAR_ADD ||
        s.epilogue == QLLM_LINEAR_PARTIALS)
      return false;
    carried |= i == 0u && source >= 2u;
    args.source[i] = source;
    (s.epilogue == QLLM_LINEAR_GATED ? gated : stored) +=
        s.rows / (s.epilogue == QLLM_LINEAR_GATED ? 32u : 16u);
    columns = std::min(columns, s.columns);
  }
  if (columns < 512u && stored + gated > 2048u) return false;
  if (l.element == QLLM_ELEMENT_BF16 && l.width > kNormedWidth && !gated && stored > 4096u)
    return false;
  return carried;
}

// Whether the launch writes nothing that it reads or writes elsewhere: a workgroup takes the
// norm whenever it starts, when others may have stored their outputs and the first one the
// stream and the carried row.  Two launches read all of it before, and leave the
// normalised rows in memory.
bool normed_apart(const NormedArgs& args) {
  struct Range {
    uintptr_t first, end;
  };
  const auto range = [](const void* first, uint64_t bytes) {
    const auto at = reinterpret_cast<uintptr_t>(first);
    return Range{at, first ? at + bytes : at};
  };
  const auto meet = [](Range a, Range b) {
    return a.first < b.end && b.first < a.end && a.first < a.end && b.first < b.end;
  };
  const qllm_stream_norm_launch& l = args.norm.launch;
  const qllm_token_shift& shift = args.norm.shift;
  const qllm_token_rows& tokens = args.norm.tokens;
  const uint64_t element = l.element == QLLM_ELEMENT_F32 ? 4u : 2u;
  const uint64_t row = uint64_t{l.width} * 4u;
  const bool leaves_stream = tokens.table || l.partial_count;
  const Range stream = range(leaves_stream ? l.stream_out : nullptr, row);
  const Range last = range(l.shift ? shift.last : nullptr, row);
  if (meet(stream, last)) return false;
  const auto output = [&](const qllm_linear_segment& s) {
    return range(s.output, s.output_columns *
                               (s.epilogue == QLLM_LINEAR_GATED ? element : uint64_t{4u}));
  };
  const auto written = [&](Range with) {
    bool any = meet(stream, with) || meet(last, with);
    for (uint32_t i = 0; i < args.linear.count; ++i)
      any |= meet(output(args.linear.segment[i]), with);
    return any;
  };
  for (uint32_t i = 0; i < args.linear.count; ++i) {
    const qllm_linear_segment& s = args.linear.segment[i];
    if (meet(output(s), stream) || meet(output(s), last) ||
        written(range(s.weights, uint64_t{s.rows} * s.columns * 2u)))
      return false;
  }
  for (int i = 0; i < 2; ++i)
    if (l.weight[i] &&
        (written(range(l.weight[i], row)) || written(range(l.output[i], l.stride[i] * element))))
      return false;
  if (l.partial_count &&
      (written(range(l.partials, (uint64_t{l.partial_count} - 1u) * l.partial_stride * 4u + row)) ||
       written(range(l.branch_weight, row))))
    return false;
  if (tokens.table) {
    if (written(range(tokens.table, uint64_t{tokens.vocabulary} * l.width * 2u)) ||
        written(range(tokens.tokens, 4u)))
      return false;
  } else if (written(range(l.input, row))) {
    return false;
  }
  if (!l.shift) return true;
  for (uint32_t b = 0; b < shift.count; ++b)
    if (written(range(shift.mu[b], row)) || written(range(shift.output[b], l.stride[0] * element)))
      return false;
  // (which slot's row is read is known on the device alone: any row may be `last`)
  const uint64_t slot = shift.slot_stride * 4u;
  const uint64_t into = last.first - reinterpret_cast<uintptr_t>(shift.previous);
  if (last.first >= reinterpret_cast<uintptr_t>(shift.previous) && slot && into % slot == 0u)
    return false;
  return !written(range(shift.previous, row)) &&
         !written(range(l.step, (kStepSlot + 1) * sizeof(uint32_t)));
}

// Workgroups of a launch: one a tile as long as `most` fit the chip at once, beyond that as
// many as fit, dealt to the segments by their tiles.
void normed_workgroups(LinearArgs& args, uint32_t most) {
  const auto units = [](const qllm_linear_segment& s) {
    return s.rows / (s.epilogue == QLLM_LINEAR_GATED ? 32u : 16u);
  };
  uint64_t total = 0;
  for (uint32_t i = 0; i < args.count; ++i) total += units(args.segment[i]);
  for (uint32_t i = 0; i < args.count; ++i) {
    const uint64_t own = units(args.segment[i]);
    const uint64_t groups = total <= most
                                ? own
                                : std::max<uint64_t>(own * most / total, 1u);
    args.first_unit[i + 1] = args.first_unit[i] + static_cast<uint32_t>(groups);
  }
}

// The arguments of qllm_linear_normed, checked and collected; `together`: one launch.
int32_t normed_arguments(const qllm_stream_norm_launch* norm, const qllm_token_rows* tokens,
                         const qllm_linear_segment* segments, uint32_t count, NormedArgs& args,
                         bool& together) {
  bool wide = false;
  if (const int32_t status = stream_norm_arguments(norm, tokens, args.norm, wide))
    return status;
  if (const int32_t status =
          linear_arguments(segments, count, norm->rows, norm->element, args.linear))
    return status;
  together = wide && normed_sources(args) && normed_apart(args);
  return QLLM_OK;
}

}  // namespace

extern "C" int32_t qllm_linear_layout(const qllm_linear_segment* segments, uint32_t count,
                                      uint32_t batch, uint32_t element,
                                      qllm_launch_layout* layout) {
  LinearArgs args{};
  if (!layout) return fail(QLLM_INVALID_ARGUMENT, "invalid linear layout");
  if (const int32_t status = linear_arguments(segments, count, batch, element, args))
    return status;
  const bool f32 = element == QLLM_ELEMENT_F32;
  if (batch <= 64u) {
    *layout = {small_rows(batch), 16u, parts_of(args.segment[0])};
    return QLLM_OK;
  }
  const uint32_t form = tall_form(args, f32);
  const TallForm& tile = f32 ? kTallFormsF32[form] : kTallForms[form];
  *layout = {16u * tile.mt, 64u * tile.nt, parts_of(args.segment[0])};
  return QLLM_OK;
}

extern "C" int32_t qllm_linear_batch(const qllm_linear_segment* segments, uint32_t count,
                                     uint32_t batch, uint32_t element, void* stream) {
  LinearArgs args{};
  if (const int32_t status = linear_arguments(segments, count, batch, element, args))
    return status;
  const auto hip_stream = as_stream(stream);
  const bool f32 = element == QLLM_ELEMENT_F32;
  if (batch <= 64u) {
    for (uint32_t i = 0; i < count; ++i) {
      const qllm_linear_segment& s = segments[i];
      const uint32_t parts = s.epilogue == QLLM_LINEAR_PARTIALS ? s.splits : 1u;
      const uint32_t tile_rows = s.epilogue == QLLM_LINEAR_GATED ? 32u : 16u;
      args.first_unit[i + 1] = args.first_unit[i] + s.rows / tile_rows * parts;
    }
    if (small_rows(batch) == 16u)
      f32 ? launch_small<true, 1>(args, hip_stream) : launch_small<false, 1>(args, hip_stream);
    else if (small_rows(batch) == 32u)
      f32 ? launch_small<true, 2>(args, hip_stream) : launch_small<false, 2>(args, hip_stream);
    else
      f32 ? launch_small<true, 4>(args, hip_stream) : launch_small<false, 4>(args, hip_stream);
    return launched("small-batch linear");
  }
  const uint32_t form = tall_form(args, f32);
  if (f32)
    return form ? launch_tall<true, 4, 4>(args, hip_stream)
                : launch_tall<true, 2, 4>(args, hip_stream);
  if (form == 2u) return launch_tall<false, 4, 8>(args, hip_stream);
  return form ? launch_tall<false, 2, 8>(args, hip_stream)
              : launch_tall<false, 2, 4>(args, hip_stream);
}

extern "C" int32_t qllm_linear_normed_launches(const qllm_stream_norm_launch* norm,
                                               const qllm_token_rows* tokens,
                                               const qllm_linear_segment* segments,
                                               uint32_t count, uint32_t* launches) {
  NormedArgs args{};
  bool together = false;
  if (!launches) return fail(QLLM_INVALID_ARGUMENT, "invalid linear of a norm");
  if (const int32_t status = normed_arguments(norm, tokens, segments, count, args, together))
    return status;
  *launches = together ? 1u : 2u;
  return QLLM_OK;
}

extern "C" int32_t qllm_linear_normed(const qllm_stream_norm_launch* norm,
                                      const qllm_token_rows* tokens,
                                      const qllm_linear_segment* segments, uint32_t count,
                                      void* stream) {
  NormedArgs args{};
  bool together = false;
  if (const int32_t status = normed_arguments(norm, tokens, segments, count, args, together))
    return status;
  if (!together) {
    if (const int32_t status = tokens ? qllm_stream_norm_tokens(norm, tokens, stream)
                                      : qllm_stream_norm(norm, stream))
      return status;
    return qllm_linear_batch(segments, count, norm->rows, norm->element, stream);
  }
  // (128 registers a lane up to kNormedWidth values, 256 beyond: two workgroups a CU, or one)
  normed_workgroups(args.linear, norm->width <= kNormedWidth ? 512u : 256u);
  const uint32_t grid = args.linear.first_unit[count];
  const auto hip_stream = as_stream(stream);
  const bool f32 = norm->element == QLLM_ELEMENT_F32;
  const auto launch = [&](auto kernel) {
    kernel<<<grid, kNormedThreads, 0, hip_stream>>>(args);
  };
  if (norm->width <= kNormedWidth)
    f32 ? launch(linear_normed_kernel<true, 1>) : launch(linear_normed_kernel<false, 1>);
  else
    f32 ? launch(linear_normed_kernel<true, 2>) : launch(linear_normed_kernel<false, 2>);
  return launched("linear of a norm");
}

extern "C" uint32_t qllm_linear_part_rows(uint32_t rows, uint32_t columns, uint32_t batch,
                                          uint32_t element) {
  uint32_t most = 0u;
  // Within 64 batch rows the workgroups of every form stay the same in number and a row
  // makes the parts cost more, so the first row of 64 asks for the most parts.
  for (uint64_t first = 65u; first <= batch && 2u * first <= QLLM_LINEAR_PART_ROWS;
       first += 64u) {
    const uint32_t parts =
        qllm_linear_parts(rows, columns, static_cast<uint32_t>(first), element);
    const uint64_t last = std::min<uint64_t>(first + 63u, batch);
    if (parts > 1u)
      most = std::max(most, static_cast<uint32_t>(std::min<uint64_t>(
                                parts * last, QLLM_LINEAR_PART_ROWS)));
  }
  return most;
}

extern "C" uint32_t qllm_linear_parts(uint32_t rows, uint32_t columns, uint32_t batch,
                                      uint32_t element) {
  const uint32_t steps = columns / 64u;
  uint32_t best = 1u;
  double least = 0.0;
  each_form(element == QLLM_ELEMENT_F32, [&](const TallForm& form, uint32_t) {
    const double units = static_cast<double>(tall_units(form, rows, batch));
    for (uint32_t parts = 1; parts <= 16u && parts <= std::max(steps, 1u); ++parts) {
      if (parts > 1u && uint64_t{parts} * batch > QLLM_LINEAR_PART_ROWS) break;
      const double time = tall_time(form, units * parts, (steps + parts - 1u) / parts) +
                          parts * 4.0 * batch * rows / 6500.0;
      if (least == 0.0 || time < least) {
        best = parts;
        least = time;
      }
    }
  });
  return best;
}

// Pieces shared by the paged decode-attention split kernels (Q4H and exact
// F16 caches): lane-group reductions, the scalar page-table fetch, and the
// merge of a workgroup's eight wave states into one split partial.
#pragma once

#include "common.hpp"

#include <initializer_list>
#include <type_traits>

namespace qllm {

typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));

constexpr int kSplitWaves = 8;
constexpr float kMaskedMax = -1.0e30f;

// max over the lanes {l, l^16, l^32, l^48}
__device__ __forceinline__ float quad_row_max(float value) {
  auto a = __builtin_amdgcn_permlane32_swap(__float_as_uint(value),
                                            __float_as_uint(value), false, false);
  value = fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
  auto b = __builtin_amdgcn_permlane16_swap(__float_as_uint(value),
                                            __float_as_uint(value), false, false);
  return fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1]));
}

// max over all 64 lanes without the LDS pipeline: four cross-lane steps inside
// each row of 16 lanes, then the rows
__device__ __forceinline__ float wave_max_in_registers(float value) {
  const auto step = [](float v, auto control) {
    const int moved = __builtin_amdgcn_update_dpp(
        __float_as_int(v), __float_as_int(v), decltype(control)::value, 0xf, 0xf,
        false);
    return fmaxf(v, __int_as_float(moved));
  };
  value = step(value, std::integral_constant<int, 0xb1>{});    // quad_perm 1,0,3,2
  value = step(value, std::integral_constant<int, 0x4e>{});    // quad_perm 2,3,0,1
  value = step(value, std::integral_constant<int, 0x141>{});   // row_half_mirror
  value = step(value, std::integral_constant<int, 0x140>{});   // row_mirror
  return quad_row_max(value);
}

__device__ __forceinline__ float quad_row_sum(float value) {
  auto a = __builtin_amdgcn_permlane32_swap(__float_as_uint(value),
                                            __float_as_uint(value), false, false);
  value = __uint_as_float(a[0]) + __uint_as_float(a[1]);
  auto b = __builtin_amdgcn_permlane16_swap(__float_as_uint(value),
                                            __float_as_uint(value), false, false);
  return __uint_as_float(b[0]) + __uint_as_float(b[1]);
}

// Page table entry at a wave-uniform index, fetched with a scalar load (the
// table is never written while attention kernels run), so everything derived
// from the page address stays in scalar registers.
__device__ __forceinline__ const void* uniform_page(
    const void* const* page_table, uint32_t index) {
  typedef const void* __attribute__((address_space(4))) const* constant_table;
  return ((constant_table)page_table)[index];
}

// Tells the compiler that a pointer every lane computes alike is wave-uniform,
// so that it can live in scalar registers.
__device__ __forceinline__ const uint8_t* uniform_pointer(const uint8_t* pointer) {
  const uint64_t bits = reinterpret_cast<uint64_t>(pointer);
  const uint32_t low =
      __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(bits));
  const uint32_t high =
      __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(bits >> 32));
  return reinterpret_cast<const uint8_t*>((static_cast<uint64_t>(high) << 32) | low);
}

// Direct global -> LDS loads (no VGPRs): lane l of the wave fetches 16 (4)
// bytes at base + offset[l] and they land at lds + 16*l (4*l).  `base` and
// `lds` are wave-uniform.  Written as assembly so that the address stays in
// the scalar-base + 32-bit-lane-offset form (one VGPR for all loads of a tile)
// and so that the compiler, which would otherwise wait for every outstanding
// load before any later LDS access, leaves the waiting to this kernel.
__device__ __forceinline__ void copy16_to_lds(const uint8_t* base,
                                              uint32_t lane_offset,
                                              uint32_t lds) {
  uint32_t saved_m0;  // M0 carries the LDS address; it is put back afterwards
  asm volatile(
      "s_mov_b32 %0, m0\n\t"
      "s_mov_b32 m0, %3\n\t"
      "s_nop 0\n\t"
      "global_load_lds_dwordx4 %1, %2\n\t"
      "s_mov_b32 m0, %0"
      : "=&s"(saved_m0) : "v"(lane_offset), "s"(base), "s"(lds) : "memory");
}
__device__ __forceinline__ void copy4_to_lds(const uint8_t* base,
                                             uint32_t lane_offset,
                                             uint32_t lds) {
  uint32_t saved_m0;  // M0 carries the LDS address; it is put back afterwards
  asm volatile(
      "s_mov_b32 %0, m0\n\t"
      "s_mov_b32 m0, %3\n\t"
      "s_nop 0\n\t"
      "global_load_lds_dword %1, %2\n\t"
      "s_mov_b32 m0, %0"
      : "=&s"(saved_m0) : "v"(lane_offset), "s"(base), "s"(lds) : "memory");
}

// at most COUNT vmem loads (direct-to-LDS loads included) still in flight
template <int COUNT>
__device__ __forceinline__ void vmem_wait() {
  asm volatile("s_waitcnt vmcnt(%0)" :: "n"(COUNT) : "memory");
}
// Lane index recomputed where it is needed (two instructions) instead of
// being kept in a register across the tile loop.
__device__ __forceinline__ uint32_t fresh_lane_index() {
  uint32_t lane;
  asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0"
               : "=v"(lane));
  return lane;
}
__device__ __forceinline__ uint32_t lds_address(const void* pointer) {
  return static_cast<uint32_t>(reinterpret_cast<uintptr_t>(
      (__attribute__((address_space(3))) const void*)pointer));
}

// (cos, sin) of a row's rotary angle for one pair of dimensions.
__device__ __forceinline__ float2 rotary_angle(uint32_t position, uint32_t pair,
                                               uint32_t rotary_dim, float theta,
                                               bool bf16_activations) {
  const float angle = static_cast<float>(position) *
                      powf(theta, -2.0f * static_cast<float>(pair) /
                                      static_cast<float>(rotary_dim));
  float sine, cosine;
  sincosf(angle, &sine, &cosine);
  if (bf16_activations) {
    cosine = bf16_round(cosine);
    sine = bf16_round(sine);
  }
  return make_float2(cosine, sine);
}

// A word of a small device-side parameter block (step positions) that no
// kernel writes: fetched with a scalar load, like the page table.
__device__ __forceinline__ uint32_t uniform_word(const uint32_t* words,
                                                 uint32_t index) {
  typedef const uint32_t __attribute__((address_space(4)))* constant_words;
  return ((constant_words)words)[index];
}

// One wave writes the K (kind 0) or V (kind 1) vector of (cache slot, kv head)
// into the proposer's Q8 layer at `layer_base` (page + the layer's offset):
// codes [kind][slot][kv head][head_dim] int8, then scales [kind][kv head]
// [page_tokens] binary16; scale = f16(max(absmax / 127, 2^-24)), code =
// clamp(rn(x / scale), -127, 127) (transformer_kernels.cu:601-625).  `source`
// may lie in LDS or in global memory.
__device__ __forceinline__ void q8_encode_record(const float* source,
                                                 uint32_t head_dim, uint8_t* layer_base,
                                                 uint32_t kind, uint32_t slot,
                                                 uint32_t kv_head, uint32_t kv_heads,
                                                 uint32_t page_tokens, uint32_t lane) {
  const size_t codes_bytes = static_cast<size_t>(page_tokens) * kv_heads * head_dim;
  const size_t record = static_cast<size_t>(slot) * kv_heads + kv_head;
  float maximum = 0.0f;
  for (uint32_t index = lane; index < head_dim; index += 64u)
    maximum = fmaxf(maximum, fabsf(source[index]));
  maximum = wave_max(maximum);
  const uint32_t scale_bits = f32_to_f16_bits(fmaxf(maximum / 127.0f, 0x1p-24f));
  const float scale = f16_bits_to_f32(scale_bits);
  int8_t* codes =
      reinterpret_cast<int8_t*>(layer_base + kind * codes_bytes) + record * head_dim;
  for (uint32_t index = lane; index < head_dim; index += 64u) {
    const int code = max(-127, min(127, __float2int_rn(source[index] / scale)));
    codes[index] = static_cast<int8_t>(code);
  }
  if (lane == 0u) {
    uint16_t* scales = reinterpret_cast<uint16_t*>(layer_base + 2u * codes_bytes) +
                       static_cast<size_t>(kind) * kv_heads * page_tokens;
    scales[static_cast<size_t>(kv_head) * page_tokens + slot] =
        static_cast<uint16_t>(scale_bits);
  }
}

// Tiles [first, last) of the context that wave `wave` of split `split` walks.
// split_tokens == 0: balanced - the context's tiles are dealt evenly over
// every wave of the grid row, whatever the context length.  Otherwise split
// s covers tokens [s*split_tokens, (s+1)*split_tokens) and its tiles are dealt
// evenly over the workgroup's waves.
// tail_work (balanced only): what the waves at the end of the context do
// besides their tiles, in tiles' worth of time - the deal is over
// context_tiles + tail_work tiles of which the last tail_work do not exist, so
// those waves walk that many fewer.  tail_alone: where the other workgroups' waves hold
// all tiles but the last one each, the last workgroup has that one alone.
template <int WAVES = kSplitWaves>
__device__ __forceinline__ void wave_tile_range(uint32_t context_tiles,
                                                uint32_t tile_tokens,
                                                uint32_t split_tokens,
                                                uint32_t split, uint32_t splits,
                                                uint32_t wave,
                                                uint32_t& tile_first,
                                                uint32_t& tile_last,
                                                uint32_t tail_work = 0u,
                                                bool tail_alone = false) {
  if (split_tokens == 0u) {
    // floor(slot * tiles / slots) in 32-bit arithmetic: with tiles = q * slots
    // + r it is slot * q + floor(slot * r / slots), and slot * r < slots^2
    const uint32_t slots = splits * WAVES;
    const uint32_t slot = split * WAVES + wave;
    const uint32_t others = slots - WAVES;   // slots of the other workgroups
    if (tail_alone && splits > 1u && context_tiles <= others + 1u) {
      const uint32_t before = context_tiles - 1u;
      // (its last wave, which has none of a few rows' records to encode: one row of 24 heads
      // on 4 of 256 dimensions after 300 tokens 13.2 us with the first wave, 12.7 so)
      tile_first = slot < others ? slot * before / others : before;
      tile_last = slot < others       ? (slot + 1u) * before / others
                  : slot + 1u == slots ? context_tiles
                                       : before;
      return;
    }
    const uint32_t dealt = context_tiles + tail_work;
    const uint32_t quotient = dealt / slots;
    const uint32_t remainder = dealt - quotient * slots;
    tile_first = min(slot * quotient + slot * remainder / slots, context_tiles);
    tile_last = min((slot + 1u) * quotient + (slot + 1u) * remainder / slots,
                    context_tiles);
  } else {
    const uint32_t split_tiles = split_tokens / tile_tokens;
    const uint32_t begin = min(split * split_tiles, context_tiles);
    const uint32_t count = min(begin + split_tiles, context_tiles) - begin;
    tile_first = begin + wave * count / WAVES;
    tile_last = begin + (wave + 1u) * count / WAVES;
  }
}

// Four neighbouring outputs of a row from their sums over the context and the row's
// probability sum: divided, gated (gate: the four values of the query's second half),
// stored in the output's type at element `index`.
__device__ __forceinline__ void store_attention_outputs(f32x4 result, float sum,
                                                        bool gated, f32x4 gate,
                                                        void* output,
                                                        uint32_t output_kind,
                                                        size_t index) {
  // (the quotients of one divisor: its correctly rounded reciprocal once, then the product
  // and its remainder - P. Markstein, "Computation of elementary functions on the IBM RISC
  // System/6000 processor", 1990: rounded as the division where the remainder does not
  // underflow, that is for outputs from some 2^-100 on; infinities have no remainder)
  const float inverse = 1.0f / sum;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float quotient = result[i] * inverse;
    const float refined = fmaf(fmaf(-quotient, sum, result[i]), inverse, quotient);
    result[i] = __builtin_isfinite(quotient) ? refined : quotient;
    if (gated) result[i] *= 1.0f / (1.0f + expf(-gate[i]));
  }
  if (output_kind == QLLM_OUT_BF16) {
    uint2 packed;
    packed.x = f32_to_bf16_bits(result[0]) | (f32_to_bf16_bits(result[1]) << 16);
    packed.y = f32_to_bf16_bits(result[2]) | (f32_to_bf16_bits(result[3]) << 16);
    *reinterpret_cast<uint2*>(static_cast<uint16_t*>(output) + index) = packed;
  } else {
    *reinterpret_cast<f32x4*>(static_cast<float*>(output) + index) = result;
  }
}

struct PartialTarget {
  float* partial_maxima;   // [rows, maximum_splits, query_heads]
  float* partial_sums;     // same
  float* partial_outputs;  // [rows, maximum_splits, query_heads, D]
  uint32_t maximum_splits;
  uint32_t query_heads;
  uint32_t kv_head;
  uint32_t split;
  uint32_t group;          // query heads per KV head
  uint32_t matrix_rows;    // rows * group
  // ONE only; gate_query: the rows whose second half gates the outputs, or null
  void* output;            // [rows, query_heads, D]
  uint32_t output_kind;
  const float* gate_query;
  uint32_t query_stride;
};

// Merges the wave states of a workgroup (of eight waves unless said otherwise) and
// writes the split partial, or the outputs themselves.
// A wave's state: per row tile rt (16 matrix rows; lane (col = lane%16, quad =
// lane/16) owns matrix row 16*rt + col) the running maximum (log2 units) and
// sum, and out[dt][rt] = O^T elements d = 16*dt + 4*quad .. +3 of that row.
//  1. every wave publishes its (max, sum) per row; all waves derive the
//     merged maximum and bring their own accumulators to it.
//  2. the accumulators are summed reduce-scatter style, eight 1 KiB register
//     vectors at a time: each wave drops the eight vectors of the group into
//     LDS, lane-linear (no bank conflicts), and wave v adds up vectors v,
//     v + WAVES, ... of all waves in a fixed order, owns them in the result and
//     writes them out.
// `pool` needs 8 KiB of LDS per wave, `summary` 512*RT bytes per wave; both may
// overlap whatever the tile loop used (the function starts with a barrier).
// ONE (a launch of one split): the outputs themselves, as the combine would leave
// them.  A parameter and not a test of `output`: with the test in every kernel
// launches of nine splits took 2 - 4 % longer.
template <int D, int RT, int WAVES = kSplitWaves, bool ONE = false>
__device__ __forceinline__ void merge_wave_states(
    float (&running_max)[RT], float (&running_sum)[RT],
    f32x4 (&out)[D / 16][RT], float* pool, float2* summary, uint32_t wave,
    uint32_t lane, const PartialTarget& target) {
  constexpr int DT = D / 16;
  constexpr int VECTORS = DT * RT;   // f32x4 accumulator vectors per wave
  constexpr int ROUND = 8;           // vectors of a round
  constexpr int OWN = ROUND / WAVES;
  static_assert(VECTORS % ROUND == 0 && ROUND % WAVES == 0, "vectors are dealt to the waves");
  const uint32_t col = lane & 15u;
  const uint32_t quad = lane >> 4;
  // (ONE: the gates of the vectors this wave will own travel during the merge)
  f32x4 gates[ONE ? VECTORS / WAVES : 1] = {};
  if (ONE && target.gate_query) {
#pragma unroll
    for (int group_index = 0; group_index < VECTORS / WAVES; ++group_index) {
      const uint32_t k = group_index * WAVES + wave;
      const uint32_t matrix_row = min(16u * (k % RT) + col, target.matrix_rows - 1u);
      const size_t record =
          static_cast<size_t>(matrix_row / target.group) * target.query_heads +
          target.kv_head * target.group + matrix_row % target.group;
      gates[group_index] = *reinterpret_cast<const f32x4*>(
          target.gate_query + record * target.query_stride + D + 16u * (k / RT) +
          4u * quad);
    }
  }
  __syncthreads();  // tiles done: the LDS they used is free
#pragma unroll
  for (int rt = 0; rt < RT; ++rt)
    summary[(wave * RT + rt) * 64 + lane] =
        make_float2(running_max[rt], running_sum[rt]);
  __syncthreads();
  float merged_max[RT], merged_sum[RT];
#pragma unroll
  for (int rt = 0; rt < RT; ++rt) {
    float2 part[WAVES];
    float maximum = kMaskedMax;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) {
      part[w] = summary[(w * RT + rt) * 64 + lane];
      maximum = fmaxf(maximum, part[w].x);
    }
    float sum = 0.0f;
#pragma unroll
    for (int w = 0; w < WAVES; ++w)
      sum = fmaf(part[w].y, __builtin_amdgcn_exp2f(part[w].x - maximum), sum);
    const float factor = __builtin_amdgcn_exp2f(running_max[rt] - maximum);
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int i = 0; i < 4; ++i) out[dt][rt][i] *= factor;
    merged_max[rt] = maximum;
    merged_sum[rt] = sum;
  }
  f32x4 merged[VECTORS / WAVES];
#pragma unroll
  for (int group_index = 0; group_index < VECTORS / ROUND; ++group_index) {
#pragma unroll
    for (int v = 0; v < ROUND; ++v) {
      const int k = group_index * ROUND + v;
      *reinterpret_cast<f32x4*>(pool + ((wave * ROUND + v) * 64 + lane) * 4u) =
          out[k / RT][k % RT];
    }
    __syncthreads();
#pragma unroll
    for (int own = 0; own < OWN; ++own) {
      f32x4 total = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int w = 0; w < WAVES; ++w)
        total += *reinterpret_cast<const f32x4*>(
            pool + ((w * ROUND + own * WAVES + wave) * 64 + lane) * 4u);
      merged[group_index * OWN + own] = total;
    }
    __syncthreads();
  }

  // partials: wave v writes the vectors it owns, wave 0 also max and sum
#pragma unroll
  for (int group_index = 0; group_index < VECTORS / WAVES; ++group_index) {
    const uint32_t k = group_index * WAVES + wave;
    const uint32_t dt = k / RT;
    const uint32_t rt = k % RT;
    const uint32_t matrix_row = 16u * rt + col;
    if (matrix_row >= target.matrix_rows) continue;
    const uint32_t row = matrix_row / target.group;
    const uint32_t head = target.kv_head * target.group + matrix_row % target.group;
    if constexpr (ONE) {
      float sum = merged_sum[0];
#pragma unroll
      for (int other = 1; other < RT; ++other)
        if (rt == static_cast<uint32_t>(other)) sum = merged_sum[other];
      const size_t record = static_cast<size_t>(row) * target.query_heads + head;
      store_attention_outputs(merged[group_index], sum, target.gate_query != nullptr,
                              gates[group_index], target.output, target.output_kind,
                              record * D + 16u * dt + 4u * quad);
      continue;
    }
    const size_t partial =
        (static_cast<size_t>(row) * target.maximum_splits + target.split) *
            target.query_heads + head;
    *reinterpret_cast<f32x4*>(target.partial_outputs + partial * D + 16u * dt +
                              4u * quad) = merged[group_index];
  }
  if (ONE || wave != 0u || quad != 0u) return;
#pragma unroll
  for (int rt = 0; rt < RT; ++rt) {
    const uint32_t matrix_row = 16u * rt + col;
    if (matrix_row >= target.matrix_rows) continue;
    const uint32_t row = matrix_row / target.group;
    const uint32_t head = target.kv_head * target.group + matrix_row % target.group;
    const size_t partial =
        (static_cast<size_t>(row) * target.maximum_splits + target.split) *
            target.query_heads + head;
    target.partial_maxima[partial] = merged_max[rt];
    target.partial_sums[partial] = merged_sum[rt];
  }
}

// What a launch reads besides the cache pages.
struct AttentionInput {
  const void* data;   // may be null
  size_t bytes;
};
// The entries of a page table that a context of `tokens` takes (with positions on the
// device: of the context that the launch's own words name).
inline AttentionInput page_table_input(const void* const* table, uint32_t tokens,
                                       uint32_t page_tokens) {
  const uint64_t pages = (uint64_t{tokens} + page_tokens - 1u) / page_tokens;
  return {table, sizeof(void*) * (pages ? pages : 1u)};
}
// Whether a launch's workgroups may write its outputs themselves: it has one split, the
// outputs can be stored four at a time, and they lie over nothing that other workgroups
// of the launch still read.  Otherwise the partials go through the combine's launch.
bool one_split_writes_output(const void* output, uint32_t output_kind,
                             uint32_t maximum_splits, uint32_t split_tokens,
                             uint32_t rows, uint32_t query_heads, uint32_t head_dim,
                             std::initializer_list<AttentionInput> inputs);

}  // namespace qllm

// What the norms of the residual stream take in, for the launches that write them and
// those that take a token's norm straight into a projection.
#pragma once

#include "mixed_common.hpp"

namespace qllm {

inline bool aligned16(const void* pointer) {
  return (reinterpret_cast<uintptr_t>(pointer) & 15u) == 0u;
}

struct NormArgs {
  qllm_stream_norm_launch launch;
  qllm_token_shift shift;
  qllm_token_rows tokens;   // TABLE: the stream's rows are these, not launch.input
};

__device__ __forceinline__ const uint16_t* table_row(const NormArgs& args, uint32_t row) {
  const uint32_t token = args.tokens.tokens[row];
  return token < args.tokens.vocabulary
             ? static_cast<const uint16_t*>(args.tokens.table) +
                   size_t{token} * args.launch.width
             : nullptr;
}

// Four bf16 values as they come from memory, times `scale`.
__device__ __forceinline__ f32x4 bf16_values4(i32x2 bits, float scale) {
  f32x4 value;
#pragma unroll
  for (int c = 0; c < 4; ++c)
    value[c] = bf16_bits_to_f32(static_cast<uint32_t>(bits[c / 2]) >> (16 * (c % 2)) & 0xffffu) *
               scale;
  return value;
}

__device__ __forceinline__ f32x4 table_value4(const NormArgs& args, uint32_t row,
                                              uint32_t piece) {
  const uint16_t* values = table_row(args, row);
  return values ? bf16_values4(reinterpret_cast<const i32x2*>(values)[piece],
                               args.tokens.scale)
                : f32x4{};
}

// The stream with the partial sums added; with a branch norm the sums alone.
__device__ __forceinline__ f32x4 stream_value4(const qllm_stream_norm_launch& l,
                                               uint32_t row, uint32_t piece) {
  f32x4 value = l.branch_weight
                    ? f32x4{}
                    : reinterpret_cast<const f32x4*>(l.input + size_t{row} * l.width)[piece];
  // eight loads in flight at a time
  for (uint32_t first = 0; first < l.partial_count; first += 8u) {
    f32x4 part[8];
#pragma unroll
    for (uint32_t i = 0; i < 8u; ++i)
      part[i] = first + i < l.partial_count
                    ? reinterpret_cast<const f32x4*>(
                          l.partials +
                          (size_t{first + i} * l.rows + row) * l.partial_stride)[piece]
                    : f32x4{};
#pragma unroll
    for (uint32_t i = 0; i < 8u; ++i) value += part[i];
  }
  return value;
}

__device__ __forceinline__ float stream_value(const qllm_stream_norm_launch& l,
                                              uint32_t row, uint32_t column) {
  float value = l.branch_weight ? 0.0f : l.input[size_t{row} * l.width + column];
  for (uint32_t p = 0; p < l.partial_count; ++p)
    value += l.partials[(size_t{p} * l.rows + row) * l.partial_stride + column];
  return value;
}

__device__ __forceinline__ float inverse_rms(float squares, uint32_t width, float epsilon) {
  return 1.0f / sqrtf(squares / static_cast<float>(width) + epsilon);
}

template <typename T>
__device__ __forceinline__ void put4(void* output, size_t index, f32x4 value) {
  if constexpr (sizeof(T) == 4) {
    *reinterpret_cast<f32x4*>(static_cast<float*>(output) + index) = value;
  } else {
    const uint32_t low = f32_to_bf16_bits(value[0]) | f32_to_bf16_bits(value[1]) << 16;
    const uint32_t high = f32_to_bf16_bits(value[2]) | f32_to_bf16_bits(value[3]) << 16;
    *reinterpret_cast<i32x2*>(static_cast<uint16_t*>(output) + index) =
        i32x2{static_cast<int>(low), static_cast<int>(high)};
  }
}

// The arguments of qllm_stream_norm and, with `tokens`, of qllm_stream_norm_tokens, checked
// and collected; `wide`: the rows can be taken 16 bytes at a time.
int32_t stream_norm_arguments(const qllm_stream_norm_launch* launch,
                              const qllm_token_rows* tokens, NormArgs& args, bool& wide);

}  // namespace qllm

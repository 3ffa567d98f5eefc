// The residual stream of mixed-layer decoders: embedding lookup (by itself or as the
// first norm's input) and the norm kernel every layer starts with - the partial sums of
// the projection before it added to the stream, the row's root mean square taken once,
// up to two normalised copies written (a parallel layer feeds its mixer and its
// feed-forward from the same row), or the token-shift blends of a mixer that reads the
// previous token's normalised input as well.
#include "mixed_norm.hpp"

namespace qllm {
namespace {

constexpr int kHeld = 4;   // most 16-byte pieces of a row a thread keeps in registers
// Rows up to which a thread per piece asks for all that it needs at first
constexpr uint32_t kFewRows = 512;

template <typename T>
__device__ __forceinline__ void pad_row(void* output, uint32_t row, uint32_t width,
                                        uint32_t stride) {
  for (uint32_t c = width + threadIdx.x; c < stride; c += blockDim.x)
    store_element(static_cast<T*>(output) + size_t{row} * stride + c, 0.0f);
}

// Rows whose width is a multiple of 4 and fits HELD pieces per thread.
//
// A row by itself is one workgroup whose time is the memory round trips it waits for one
// after the other, 0.7 to 1.5 us each (4 - 5 us: a decoded token's projections take its
// norm in where they can, linear_normed_kernel).  So all that it needs - partial sums, norm
// weights, the previous token's row and the blends - is asked for before the first sum over
// the row, with HELD = 1 (a thread per 16 bytes).  The lookup of the first layer's rows in
// the same launch (TABLE) saves the launch before it: 1 to 3000 rows 0.64 of the two.
// More pieces a thread fetch weights and blends where they use them, and none for
// pieces that the row does not have: all of it asked for first cost norms of 3000 rows of
// 5120 (plain / with blends) 38 -> 45 / 80 -> 97 us, of one row 4.0 -> 4.5, and of rows
// enough to hide each other's trips also with one piece a thread: 3000 rows of 512 with
// four partial sums 8.2 -> 9.5 us (from 800 rows on the two differ by less than 4 %).
template <typename T, int HELD, bool TABLE>
__global__ __launch_bounds__(1024) void stream_norm_wide_kernel(NormArgs args) {
  __shared__ float scratch[16];
  const qllm_stream_norm_launch& l = args.launch;
  const qllm_token_shift& shift = args.shift;
  const uint32_t row = blockIdx.x;
  const uint32_t source = !TABLE && l.gather ? l.gather[row] : row;
  const uint32_t pieces = l.width / 4u;
  const bool shifted = l.shift != nullptr;
  // (the request's slot is a load of its own that an address waits for)
  const f32x4* carried =
      shifted && row == 0u
          ? reinterpret_cast<const f32x4*>(shift.previous +
                                           l.step[kStepSlot] * shift.slot_stride)
          : nullptr;
  const bool writes = TABLE || (l.partial_count && !l.branch_weight);
  constexpr bool kFirst = HELD == 1;   // all loads set out before the first sum
  f32x4 held[HELD], before[HELD], weight[2], branch, mu[6];
  float squares = 0.0f;
  if constexpr (kFirst) {
    const uint32_t piece = min(threadIdx.x, pieces - 1u);
#pragma unroll
    for (int output = 0; output < 2; ++output)
      if (l.weight[output])
        weight[output] = reinterpret_cast<const f32x4*>(l.weight[output])[piece];
    if (l.branch_weight) {
      before[0] = reinterpret_cast<const f32x4*>(l.input + size_t{row} * l.width)[piece];
      branch = reinterpret_cast<const f32x4*>(l.branch_weight)[piece];
    }
    if (shifted) {
#pragma unroll
      for (uint32_t s = 0; s < 6u; ++s)
        if (s < shift.count) mu[s] = reinterpret_cast<const f32x4*>(shift.mu[s])[piece];
      if (carried) before[0] = carried[piece];
    }
  }
  const auto weight_at = [&](int output, uint32_t piece) {
    return kFirst ? weight[output]
                  : reinterpret_cast<const f32x4*>(l.weight[output])[piece];
  };
#pragma unroll
  for (int i = 0; i < HELD; ++i) {
    const uint32_t piece = threadIdx.x + i * blockDim.x;
    held[i] = f32x4{};
    if (piece >= pieces) continue;
    held[i] = TABLE ? table_value4(args, row, piece) : stream_value4(l, source, piece);
    if (writes)
      reinterpret_cast<f32x4*>(l.stream_out + size_t{row} * l.width)[piece] = held[i];
#pragma unroll
    for (int c = 0; c < 4; ++c) squares = fmaf(held[i][c], held[i][c], squares);
  }
  if (!TABLE && l.branch_weight) {
    f32x4 branches[HELD];
#pragma unroll
    for (int i = 0; i < HELD; ++i) {
      const uint32_t piece = threadIdx.x + i * blockDim.x;
      if (kFirst) branches[i] = branch;
      if (kFirst || piece >= pieces) continue;
      before[i] = reinterpret_cast<const f32x4*>(l.input + size_t{row} * l.width)[piece];
      branches[i] = reinterpret_cast<const f32x4*>(l.branch_weight)[piece];
    }
    const float unit =
        inverse_rms(block_sum(squares, scratch), l.width, l.branch_epsilon);
    squares = 0.0f;
#pragma unroll
    for (int i = 0; i < HELD; ++i) {
      const uint32_t piece = threadIdx.x + i * blockDim.x;
      if (piece >= pieces) continue;
      held[i] = before[i] + held[i] * unit * branches[i] * l.branch_scale;
      reinterpret_cast<f32x4*>(l.stream_out + size_t{row} * l.width)[piece] = held[i];
#pragma unroll
      for (int c = 0; c < 4; ++c) squares = fmaf(held[i][c], held[i][c], squares);
    }
  }
  const float inverse = inverse_rms(block_sum(squares, scratch), l.width, l.epsilon);
#pragma unroll
  for (int output = 0; output < 2; ++output) {
    if (!l.weight[output] || (shifted && output == 0)) continue;
#pragma unroll
    for (int i = 0; i < HELD; ++i) {
      const uint32_t piece = threadIdx.x + i * blockDim.x;
      if (piece >= pieces) continue;
      put4<T>(l.output[output], size_t{row} * l.stride[output] + piece * 4u,
              held[i] * inverse * weight_at(output, piece));
    }
    pad_row<T>(l.output[output], row, l.width, l.stride[output]);
  }
  if (!shifted) return;

  float before_inverse = 0.0f;
  if (!kFirst || row) {   // row 0 takes the norm the request carries, already weighted
    float before_squares = 0.0f;
#pragma unroll
    for (int i = 0; i < HELD; ++i) {
      const uint32_t piece = threadIdx.x + i * blockDim.x;
      before[i] = f32x4{};
      if (piece >= pieces) continue;
      before[i] = !kFirst && row == 0u ? carried[piece]
                  : TABLE              ? table_value4(args, row - 1u, piece)
                                       : stream_value4(l, row - 1u, piece);
#pragma unroll
      for (int c = 0; c < 4; ++c)
        before_squares = fmaf(before[i][c], before[i][c], before_squares);
    }
    before_inverse = inverse_rms(block_sum(before_squares, scratch), l.width, l.epsilon);
  }
#pragma unroll
  for (int i = 0; i < HELD; ++i) {
    const uint32_t piece = threadIdx.x + i * blockDim.x;
    if (piece >= pieces) continue;
    const f32x4 own = weight_at(0, piece);
    const f32x4 here = held[i] * inverse * own;
    const f32x4 there = row == 0u ? before[i] : before[i] * before_inverse * own;
    const auto blend = [&](uint32_t s, const f32x4& share) {
      put4<T>(shift.output[s], size_t{row} * l.stride[0] + piece * 4u,
              here + (there - here) * share);
    };
    if constexpr (kFirst) {
#pragma unroll
      for (uint32_t s = 0; s < 6u; ++s)
        if (s < shift.count) blend(s, mu[s]);
    } else {
      for (uint32_t s = 0; s < shift.count; ++s)
        blend(s, reinterpret_cast<const f32x4*>(shift.mu[s])[piece]);
    }
    if (row + 1u == l.rows) reinterpret_cast<f32x4*>(shift.last)[piece] = here;
  }
  for (uint32_t s = 0; s < shift.count; ++s)
    pad_row<T>(shift.output[s], row, l.width, l.stride[0]);
}

template <typename T, bool TABLE>
__global__ __launch_bounds__(256) void stream_norm_narrow_kernel(NormArgs args) {
  __shared__ float scratch[16];
  const qllm_stream_norm_launch& l = args.launch;
  const uint32_t row = blockIdx.x;
  const uint32_t source = !TABLE && l.gather ? l.gather[row] : row;
  const bool shifted = l.shift != nullptr;
  const auto own_value = [&](uint32_t at, uint32_t c) {
    if constexpr (TABLE) {
      const uint16_t* values = table_row(args, at);
      return values ? bf16_bits_to_f32(values[c]) * args.tokens.scale : 0.0f;
    } else {
      return stream_value(l, at, c);
    }
  };
  const float* carried =
      shifted && row == 0u ? args.shift.previous + l.step[kStepSlot] * args.shift.slot_stride
                           : nullptr;
  float squares = 0.0f;
  float before_squares = 0.0f;
  float unit_branch = 0.0f;
  if (l.branch_weight) {
    float branch_squares = 0.0f;
    for (uint32_t c = threadIdx.x; c < l.width; c += blockDim.x) {
      const float value = stream_value(l, source, c);
      branch_squares = fmaf(value, value, branch_squares);
    }
    unit_branch = inverse_rms(block_sum(branch_squares, scratch), l.width, l.branch_epsilon) *
                  l.branch_scale;
  }
  const auto here_value = [&](uint32_t c) {
    const float value = own_value(source, c);
    return l.branch_weight ? l.input[size_t{row} * l.width + c] +
                                 value * unit_branch * l.branch_weight[c]
                           : value;
  };
  for (uint32_t c = threadIdx.x; c < l.width; c += blockDim.x) {
    const float value = here_value(c);
    if (TABLE || l.partial_count) l.stream_out[size_t{row} * l.width + c] = value;
    squares = fmaf(value, value, squares);
    if (shifted && !carried) {
      const float before = own_value(row - 1u, c);
      before_squares = fmaf(before, before, before_squares);
    }
  }
  const float inverse = inverse_rms(block_sum(squares, scratch), l.width, l.epsilon);
  const float before_inverse =
      inverse_rms(block_sum(before_squares, scratch), l.width, l.epsilon);
  for (uint32_t c = threadIdx.x; c < l.width; c += blockDim.x) {
    const float unit = here_value(c) * inverse;
    for (int output = 0; output < 2; ++output)
      if (l.weight[output] && !(shifted && output == 0))
        store_element(static_cast<T*>(l.output[output]) +
                          size_t{row} * l.stride[output] + c,
                      unit * l.weight[output][c]);
    if (!shifted) continue;
    const float here = unit * l.weight[0][c];
    const float there =
        carried ? carried[c]
                : own_value(row - 1u, c) * before_inverse * l.weight[0][c];
    for (uint32_t s = 0; s < args.shift.count; ++s)
      store_element(static_cast<T*>(args.shift.output[s]) + size_t{row} * l.stride[0] + c,
                    here + (there - here) * args.shift.mu[s][c]);
    if (row + 1u == l.rows) args.shift.last[c] = here;
  }
  for (int output = 0; output < 2; ++output)
    if (l.weight[output] && !(shifted && output == 0))
      pad_row<T>(l.output[output], row, l.width, l.stride[output]);
  if (shifted)
    for (uint32_t s = 0; s < args.shift.count; ++s)
      pad_row<T>(args.shift.output[s], row, l.width, l.stride[0]);
}

__global__ void embedding_bf16_kernel(const uint16_t* table, uint32_t vocabulary,
                                      const uint32_t* tokens, float* output,
                                      uint32_t width, float scale) {
  const uint32_t token = tokens[blockIdx.x];
  for (uint32_t c = threadIdx.x; c < width; c += blockDim.x)
    output[size_t{blockIdx.x} * width + c] =
        token < vocabulary
            ? bf16_bits_to_f32(table[size_t{token} * width + c]) * scale
            : 0.0f;
}

}  // namespace
}  // namespace qllm

using namespace qllm;

extern "C" int32_t qllm_embedding_bf16_batch(const void* table_bf16, uint32_t vocabulary,
                                             const uint32_t* tokens, float* output,
                                             uint32_t rows, uint32_t width, float scale,
                                             void* stream) {
  if (!table_bf16 || !tokens || !output || !rows || !width || !vocabulary)
    return fail(QLLM_INVALID_ARGUMENT, "invalid bf16 embedding lookup");
  embedding_bf16_kernel<<<rows, 256, 0, as_stream(stream)>>>(
      static_cast<const uint16_t*>(table_bf16), vocabulary, tokens, output, width, scale);
  return launched("bf16 embedding lookup");
}

namespace {

template <typename T, bool TABLE>
void launch_norm(const NormArgs& args, bool wide, hipStream_t stream) {
  const qllm_stream_norm_launch& l = args.launch;
  const uint32_t pieces = l.width / 4u;
  uint32_t threads = l.rows <= 16u ? 1024u : 256u;
  while (threads > 64u && threads / 2u >= pieces) threads /= 2u;
  if (pieces > threads * kHeld) threads = 1024u;
  if (!wide || pieces > threads * kHeld)
    stream_norm_narrow_kernel<T, TABLE><<<l.rows, 256, 0, stream>>>(args);
  else if (pieces <= threads && l.rows <= kFewRows)
    stream_norm_wide_kernel<T, 1, TABLE><<<l.rows, threads, 0, stream>>>(args);
  else
    stream_norm_wide_kernel<T, kHeld, TABLE><<<l.rows, threads, 0, stream>>>(args);
}

}  // namespace

namespace qllm {

int32_t stream_norm_arguments(const qllm_stream_norm_launch* launch,
                              const qllm_token_rows* tokens, NormArgs& args, bool& wide) {
  if (tokens && (!launch || !tokens->table || !tokens->tokens || !tokens->vocabulary ||
                 !launch->stream_out || launch->gather || launch->partial_count))
    return fail(QLLM_INVALID_ARGUMENT, "invalid stream norm of tokens");
  qllm_stream_norm_launch own{};
  if (launch) own = *launch;
  if (tokens) own.input = own.stream_out;
  if (!launch || !own.input || !launch->rows || !launch->width ||
      launch->element > QLLM_ELEMENT_F32 ||
      (launch->partial_count &&
       (tokens || !launch->partials || !launch->stream_out || launch->stream_out == own.input ||
        launch->partial_stride < launch->width || launch->gather)) ||
      (launch->branch_weight && (!launch->partial_count || launch->shift)))
    return fail(QLLM_INVALID_ARGUMENT, "invalid stream norm");
  wide = launch->width % 4u == 0u && launch->partial_stride % 4u == 0u &&
         aligned16(own.input) && aligned16(launch->stream_out) &&
         aligned16(launch->partials) && aligned16(launch->branch_weight);
  for (int i = 0; i < 2; ++i) {
    if (!launch->weight[i]) continue;
    const bool blended = i == 0 && launch->shift;
    if ((!launch->output[i] && !blended) || launch->stride[i] < launch->width)
      return fail(QLLM_INVALID_ARGUMENT, "invalid stream norm output");
    wide = wide && aligned16(launch->weight[i]) && aligned16(launch->output[i]) &&
           launch->stride[i] % 4u == 0u;
  }
  args = {own, {}, {}};
  if (const auto* shift = launch->shift) {
    if (!shift->count || shift->count > 6u || !shift->previous || !shift->last ||
        !launch->step || launch->gather || !launch->weight[0])
      return fail(QLLM_INVALID_ARGUMENT, "invalid token shift");
    for (uint32_t s = 0; s < shift->count; ++s) {
      if (!shift->mu[s] || !shift->output[s])
        return fail(QLLM_INVALID_ARGUMENT, "invalid token shift");
      wide = wide && aligned16(shift->mu[s]) && aligned16(shift->output[s]);
    }
    wide = wide && aligned16(shift->previous) && aligned16(shift->last) &&
           shift->slot_stride % 4u == 0u;
    args.shift = *shift;
  }
  if (tokens) {
    args.tokens = *tokens;
    wide = wide && (reinterpret_cast<uintptr_t>(tokens->table) & 7u) == 0u;
  }
  return QLLM_OK;
}

}  // namespace qllm

namespace {

int32_t norm_rows(const qllm_stream_norm_launch* launch, const qllm_token_rows* tokens,
                  void* stream) {
  NormArgs args{};
  bool wide = false;
  if (const int32_t status = stream_norm_arguments(launch, tokens, args, wide)) return status;
  const auto hip_stream = as_stream(stream);
  if (launch->element == QLLM_ELEMENT_F32)
    tokens ? launch_norm<float, true>(args, wide, hip_stream)
           : launch_norm<float, false>(args, wide, hip_stream);
  else
    tokens ? launch_norm<uint16_t, true>(args, wide, hip_stream)
           : launch_norm<uint16_t, false>(args, wide, hip_stream);
  return launched("stream norm");
}

}  // namespace

extern "C" int32_t qllm_stream_norm(const qllm_stream_norm_launch* launch, void* stream) {
  return norm_rows(launch, nullptr, stream);
}

extern "C" int32_t qllm_stream_norm_tokens(const qllm_stream_norm_launch* launch,
                                           const qllm_token_rows* tokens, void* stream) {
  if (!tokens) return fail(QLLM_INVALID_ARGUMENT, "invalid stream norm of tokens");
  return norm_rows(launch, tokens, stream);
}

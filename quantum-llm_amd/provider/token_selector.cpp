#include "token_selector.hpp"

#include "host_support.hpp"
#include "qllm_kernels.h"

#include <hip/hip_runtime.h>

#include <algorithm>
#include <array>
#include <chrono>
#include <cmath>
#include <cstring>
#include <numeric>
#include <stdexcept>
#include <utility>

namespace qllm {

TokenSelector::TokenSelector(void* stream, std::uint32_t vocabulary, void* workspace,
                             std::size_t workspace_bytes, TopKRows top_k_rows)
    : stream_(stream), vocabulary_(vocabulary), workspace_(workspace),
      workspace_bytes_(workspace_bytes), top_k_rows_(top_k_rows) {
  void* pinned = nullptr;
  hip_check(hipHostMalloc(&pinned, sizeof(Staging), hipHostMallocDefault),
            "allocate pinned staging");
  staging_ = static_cast<Staging*>(pinned);
  *staging_ = Staging{};
}

TokenSelector::~TokenSelector() {
  if (staging_) (void)hipHostFree(staging_);
}

std::size_t TokenSelector::workspace_bytes(std::uint32_t vocabulary,
                                           std::uint32_t rows) {
  return std::max({qllm_argmax_workspace_bytes(vocabulary, rows),
                   qllm_topk_workspace_bytes(vocabulary, kMaximumTopK),
                   qllm_topk_batch_workspace_bytes(vocabulary, kMaximumTopK, rows)});
}

void TokenSelector::mark(
    std::uint8_t* emitted, std::span<const std::uint32_t> tokens) {
  if (tokens.empty()) return;
  status_check(qllm_mark_presence_values(emitted, tokens.data(),
                                         static_cast<std::uint32_t>(tokens.size()),
                                         vocabulary_, stream_));
}

std::uint32_t TokenSelector::read_token(const std::uint32_t* device_token,
                                        std::uint8_t* emitted) {
  return *read_words(device_token, 1U, emitted);
}

// A kernel writes words into pinned memory, and a sequence number that says so.  After a
// replayed graph the host watches the number: a wait for the stream takes 7.5 us longer, and
// whoever waits for it later, if anybody does, finds 10 to 15 us of it left, as many after
// 4096 replays as after one.  Launches of a pass one by one are waited for here: watching
// saves 5 us of a pass of 40 and leaves 31 to the next wait, which is the next capture's,
// copy's or the caller's.  What has not arrived after two milliseconds - a device that has
// failed - is waited for with the stream, which reports what went wrong.
template <typename Arrived>
void TokenSelector::await(const Arrived& arrived) {
  const bool watched = std::exchange(replayed_, false);
  if (watched && ++unwaited_ < kMostUnwaited) {
    const auto deadline = std::chrono::steady_clock::now() + std::chrono::milliseconds(2);
    do {
      for (int turn = 0; turn < 64; ++turn) {
        if (arrived()) return;
        __builtin_ia32_pause();
      }
    } while (std::chrono::steady_clock::now() < deadline);
  }
  hip_check(hipStreamSynchronize(static_cast<hipStream_t>(stream_)), "wait for the device");
  unwaited_ = 0U;
  if (!arrived()) throw std::runtime_error("the device's words have not arrived");
}

const std::uint32_t* TokenSelector::read_words(const std::uint32_t* device_words,
                                               std::uint32_t count, std::uint8_t* emitted) {
  if (!count || count > kMostWords) throw std::runtime_error("invalid device words to read");
  const std::uint32_t sequence = ++sequence_;
  status_check(qllm_publish_words(device_words, count, staging_->words, &staging_->sequence,
                                  sequence, emitted, vocabulary_, stream_));
  await([&] {
    return __atomic_load_n(&staging_->sequence, __ATOMIC_ACQUIRE) == sequence;
  });
  return staging_->words;
}

const std::uint32_t* TokenSelector::read_handed(std::uint32_t rows) {
  if (!rows || rows > kMostHanded) throw std::runtime_error("invalid tokens to read");
  await([&] {
    for (std::uint32_t row = 0; row < rows; ++row) {
      const std::uint64_t word = __atomic_load_n(&staging_->handed[row], __ATOMIC_ACQUIRE);
      if (word >> 32 != handed_sequence_) return false;
      handed_tokens_[row] = static_cast<std::uint32_t>(word);
    }
    return true;
  });
  return handed_tokens_;
}

bool TokenSelector::marks_handed(const er::ProgramRequestContext& request,
                                 std::uint32_t sample_position) {
  for (const char* name : {"sampling_first_output_position", "sampling_temperature_ppm",
                           "sampling_presence_penalty_biased_ppm"})
    if (!request.parameters.contains(name)) return false;   // which select() reports
  return sample_position >= request_parameter(request, "sampling_first_output_position") &&
         request_parameter(request, "sampling_temperature_ppm") == 0U &&
         request_parameter(request, "sampling_presence_penalty_biased_ppm") == 2'000'000U;
}

// The head's token for a request (run_head with a request, :8433-8517): the
// presence penalty from the first output position on, arg-max at temperature
// zero, otherwise top-k or whole-row candidates ordered on the host and one
// draw from stream 0; an output token is marked as emitted.  One row of
// logits.
std::uint32_t TokenSelector::select(float* logits, std::uint8_t* presence,
                                    std::uint32_t* argmax_tokens,
                                    const er::ProgramRequestContext& request,
                                    std::uint32_t sample_position, bool handed) {
  const auto stream = static_cast<hipStream_t>(stream_);
  const auto first_output =
      request_parameter(request, "sampling_first_output_position");
  const bool output_sampling = sample_position >= first_output;
  const auto penalty = presence_penalty_of(request);
  if (output_sampling && penalty != 0.0) {
    status_check(qllm_apply_presence_penalty(logits, presence, vocabulary_,
                                             static_cast<float>(penalty),
                                             stream_));
    status_check(qllm_argmax_batch(logits, vocabulary_, 1U, argmax_tokens,
                                   workspace_, workspace_bytes_,
                                   stream_));
  }
  const auto temperature = request_parameter(request, "sampling_temperature_ppm");
  std::uint32_t selected{};
  if (temperature == 0U) {
    selected = handed && !(output_sampling && penalty != 0.0)
                   ? *read_handed(1U)
                   : read_token(argmax_tokens, output_sampling ? presence : nullptr);
    // a row without a finite logit selects nothing (0xffffffff): reported
    // before the presence bytes or the caller's state change
    if (selected >= vocabulary_)
      throw std::runtime_error("head logits have no finite maximum");
  } else {
    // the penalty, if any, has been applied: the distribution is taken from
    // the row as it stands
    er::ProgramRequestContext unpenalised = request;
    unpenalised.parameters["sampling_presence_penalty_biased_ppm"] = 2'000'000U;
    const auto top_k = request_parameter(request, "sampling_top_k");
    if (top_k > kMaximumTopK) {
      // the scalar sampler orders that many candidates on the host
      // (sample_token, :773-799)
      std::vector<float> row(vocabulary_);
      hip_check(hipMemcpyAsync(row.data(), logits, row.size() * 4U,
                               hipMemcpyDeviceToHost, stream),
                "copy sampling logits");
      hip_check(hipStreamSynchronize(stream), "copy sampling logits");
      replayed_ = false;
      if (top_k > row.size())
        throw std::runtime_error("invalid token sampling contract");
      std::vector<std::uint32_t> candidates(row.size());
      std::iota(candidates.begin(), candidates.end(), 0U);
      const auto before = [&](std::uint32_t left, std::uint32_t right) {
        const float a = row[left];
        const float b = row[right];
        if (std::isnan(a)) return false;
        if (std::isnan(b)) return true;
        return a == b ? left < right : a > b;
      };
      std::partial_sort(candidates.begin(), candidates.begin() + top_k,
                        candidates.end(), before);
      candidates.resize(top_k);
      std::vector<float> ordered;
      for (const auto candidate : candidates) ordered.push_back(row[candidate]);
      logit_transfer_bytes_ += row.size() * 4U;
      const auto distribution = er::make_sampling_distribution(
          ordered, candidates, static_cast<std::uint32_t>(temperature),
          static_cast<std::uint32_t>(
              request_parameter(request, "sampling_top_p_ppm")),
          static_cast<std::uint32_t>(
              request_parameter(request, "sampling_min_p_ppm")));
      selected = er::sample_distribution(
          distribution,
          er::counter_uniform(request_parameter(request, "sampling_seed"),
                              sample_position, 0U));
    } else {
      const auto chosen = this->distribution(
          logits, vocabulary_, argmax_tokens, unpenalised, nullptr);
      selected = er::sample_distribution(
          chosen,
          er::counter_uniform(request_parameter(request, "sampling_seed"),
                              sample_position, 0U));
    }
  }
  if (output_sampling && temperature != 0U) {   // (the other has been marked with its word)
    const std::uint32_t token[1] = {selected};
    mark(presence, token);
  }
  return selected;
}


// distribution_from_logits, dense_fp4_provider.cpp:8331-8391.  top_k == 0
// selects the whole-vocabulary path of the scalar sampler (sample_token,
// :773-799): the row is copied to the host and ordered there.
er::SamplingDistribution TokenSelector::distribution(
    float* row_logits, std::uint32_t vocabulary, std::uint32_t* device_argmax,
    const er::ProgramRequestContext& request, const std::uint8_t* presence) {
  const auto stream = static_cast<hipStream_t>(stream_);
  const auto penalty = presence_penalty_of(request);
  const auto temperature = request_parameter(request, "sampling_temperature_ppm");
  if (penalty != 0.0) {
    if (!presence) throw std::runtime_error("sampling presence state is absent");
    status_check(qllm_apply_presence_penalty(row_logits, presence, vocabulary,
                                             static_cast<float>(penalty),
                                             stream_));
    // the arg-max the pass left behind was taken before the penalty
    if (temperature == 0U)
      status_check(qllm_argmax_batch(row_logits, vocabulary, 1U, device_argmax,
                                     workspace_, workspace_bytes_,
                                     stream_));
  }
  if (temperature == 0U) return {{{read_token(device_argmax), 1.0}}};
  const auto top_p = static_cast<std::uint32_t>(
      request_parameter(request, "sampling_top_p_ppm"));
  const auto min_p = static_cast<std::uint32_t>(
      request_parameter(request, "sampling_min_p_ppm"));
  const auto top_k = request_parameter(request, "sampling_top_k");
  if (top_k > kMaximumTopK || top_k > vocabulary)
    throw std::runtime_error(
        "sampled exact decode requires top-k of at most 64 (0 = whole row)");
  std::vector<float> host_logits;
  std::vector<std::uint32_t> host_tokens;
  if (top_k == 0U) {
    std::vector<float> full(vocabulary);
    hip_check(hipMemcpyAsync(full.data(), row_logits, full.size() * 4U,
                             hipMemcpyDeviceToHost, stream),
              "copy logit row");
    hip_check(hipStreamSynchronize(stream), "copy logit row");
    replayed_ = false;
    host_tokens.resize(vocabulary);
    std::iota(host_tokens.begin(), host_tokens.end(), 0U);
    std::sort(host_tokens.begin(), host_tokens.end(),
              [&](std::uint32_t left, std::uint32_t right) {
                const float a = full[left];
                const float b = full[right];
                if (std::isnan(a)) return false;
                if (std::isnan(b)) return true;
                return a == b ? left < right : a > b;
              });
    host_logits.reserve(vocabulary);
    for (const auto token : host_tokens) host_logits.push_back(full[token]);
    logit_transfer_bytes_ += full.size() * 4U;
  } else {
    return std::move(top_k_distributions(row_logits, vocabulary, vocabulary,
                                              1U, request)
                         .front());
  }
  return er::make_sampling_distribution(
      host_logits, host_tokens, static_cast<std::uint32_t>(temperature), top_p,
      min_p);
}

// The distributions of `rows` rows of logits (row r at logits + r * stride)
// for a sampled request with 1 <= top_k <= 64: one selection for all rows, which
// leaves them in pinned memory, then make_sampling_distribution per row
// (distribution_from_logits, dense_fp4_provider.cpp:8331-8391, which selects
// and reads back row by row).
std::vector<er::SamplingDistribution>
TokenSelector::top_k_distributions(
    const float* logits, std::uint32_t vocabulary, std::size_t stride,
    std::uint32_t rows, const er::ProgramRequestContext& request) {
  const auto temperature = request_parameter(request, "sampling_temperature_ppm");
  const auto top_p = static_cast<std::uint32_t>(
      request_parameter(request, "sampling_top_p_ppm"));
  const auto min_p = static_cast<std::uint32_t>(
      request_parameter(request, "sampling_min_p_ppm"));
  const auto top_k =
      static_cast<std::uint32_t>(request_parameter(request, "sampling_top_k"));
  if (!rows || rows > 8U || !top_k || top_k > kMaximumTopK ||
      top_k > vocabulary)
    throw std::runtime_error(
        "sampled exact decode requires top-k of at most 64 (0 = whole row)");
  // logits of all rows, then tokens of all rows
  const std::uint32_t chosen = rows * top_k;
  const std::uint32_t sequence = ++sequence_;
  std::uint32_t* const words = staging_->words;
  if (!top_k_rows_) throw std::logic_error("this selector takes no top k");
  status_check(top_k_rows_(
      logits, vocabulary, stride, top_k, rows, reinterpret_cast<float*>(words),
      words + chosen, staging_->row_sequences, sequence, workspace_, workspace_bytes_,
      stream_));
  await([&] {
    for (std::uint32_t row = 0; row < rows; ++row)
      if (__atomic_load_n(&staging_->row_sequences[row], __ATOMIC_ACQUIRE) != sequence)
        return false;
    return true;
  });
  ++gpu_calls_;
  logit_transfer_bytes_ += std::size_t{rows} * top_k * 8U;
  std::vector<er::SamplingDistribution> result;
  result.reserve(rows);
  for (std::uint32_t row = 0; row < rows; ++row) {
    std::array<float, kMaximumTopK> row_logits;
    std::memcpy(row_logits.data(), words + std::size_t{row} * top_k, top_k * sizeof(float));
    const std::span<const std::uint32_t> row_tokens(
        words + chosen + std::size_t{row} * top_k, top_k);
    result.push_back(er::make_sampling_distribution(
        std::span<const float>(row_logits.data(), top_k), row_tokens,
        static_cast<std::uint32_t>(temperature), top_p, min_p));
  }
  return result;
}

}  // namespace qllm

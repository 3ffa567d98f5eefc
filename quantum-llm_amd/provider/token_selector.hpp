// Token selection from rows of logits, shared by the providers' heads: presence
// penalty, arg-max at temperature zero, otherwise top-k on the device (or the
// whole row on the host) and the sampling rules of speculative_sampling.
#pragma once

#include "expert/runtime/program_executor.hpp"
#include "expert/runtime/speculative_sampling.hpp"

#include "host_support.hpp"

#include <cstddef>
#include <cstdint>
#include <span>
#include <vector>

namespace qllm {

class TokenSelector final {
 public:
  static constexpr std::uint32_t kMaximumTopK = 64U;  // provider.cpp:8359

  // qllm_topk_logits_batch_handed, for requests that sample from a top k (a selector of
  // arg-max tokens has no need of it).
  using TopKRows = std::int32_t (*)(const float*, std::uint32_t, std::size_t, std::uint32_t,
                                    std::uint32_t, float*, std::uint32_t*, std::uint32_t*,
                                    std::uint32_t, void*, std::size_t, void*);
  // `workspace`: device memory of at least workspace_bytes(), shared with the
  // caller's own arg-max launches on the same stream.
  TokenSelector(void* stream, std::uint32_t vocabulary, void* workspace,
                std::size_t workspace_bytes, TopKRows top_k_rows = nullptr);
  ~TokenSelector();
  TokenSelector(const TokenSelector&) = delete;
  TokenSelector& operator=(const TokenSelector&) = delete;
  [[nodiscard]] static std::size_t workspace_bytes(std::uint32_t vocabulary,
                                                   std::uint32_t rows);

  // The head's token for a request (dense_fp4_provider.cpp:8433-8517) from one
  // row of logits whose arg-max lies in `argmax_tokens`; an output token is
  // marked as emitted in `presence`.  `handed`: the launch that took the arg-max hands it
  // over, and has marked it where marks_handed() says so.
  [[nodiscard]] std::uint32_t select(float* logits, std::uint8_t* presence,
                                     std::uint32_t* argmax_tokens,
                                     const er::ProgramRequestContext& request,
                                     std::uint32_t sample_position, bool handed = false);
  // Whether select() emits the arg-max of the logits as they are.
  [[nodiscard]] static bool marks_handed(const er::ProgramRequestContext& request,
                                         std::uint32_t sample_position);
  [[nodiscard]] er::SamplingDistribution distribution(
      float* row_logits, std::uint32_t vocabulary, std::uint32_t* device_argmax,
      const er::ProgramRequestContext& request, const std::uint8_t* presence);
  [[nodiscard]] std::vector<er::SamplingDistribution> top_k_distributions(
      const float* logits, std::uint32_t vocabulary, std::size_t stride,
      std::uint32_t rows, const er::ProgramRequestContext& request);
  // A selection on the device, after everything enqueued so far; with `emitted` it is
  // marked there (if it is a token).
  [[nodiscard]] std::uint32_t read_token(const std::uint32_t* device_token,
                                         std::uint8_t* emitted = nullptr);
  // Whether the pass whose words are read next is a replayed graph.
  void replayed(bool graph = true) noexcept { replayed_ = graph; }
  // Up to kMostWords words of device memory, after everything enqueued so far: there
  // until the next call.
  static constexpr std::uint32_t kMostWords = 2U * 8U * kMaximumTopK;
  [[nodiscard]] const std::uint32_t* read_words(const std::uint32_t* device_words,
                                                std::uint32_t count,
                                                std::uint8_t* emitted = nullptr);
  // Where an arg-max of up to kMostHanded rows leaves its tokens by itself; the next
  // sequence number, for the device word that its launch reads; and the tokens handed over
  // with that number, after everything enqueued so far: there until the next call.
  static constexpr std::uint32_t kMostHanded = 8U;
  [[nodiscard]] std::uint64_t* handed_words() const noexcept { return staging_->handed; }
  [[nodiscard]] std::uint32_t next_handover() noexcept { return ++handed_sequence_; }
  [[nodiscard]] const std::uint32_t* read_handed(std::uint32_t rows);
  // emitted[token] = 1 for every token (one launch)
  void mark(std::uint8_t* emitted, std::span<const std::uint32_t> tokens);

  [[nodiscard]] std::uint64_t gpu_calls() const noexcept { return gpu_calls_; }
  [[nodiscard]] std::uint64_t logit_transfer_bytes() const noexcept {
    return logit_transfer_bytes_;
  }

 private:
  // Pinned: written by the device, the sequence number after the words it stands for.
  struct Staging final {
    std::uint32_t words[kMostWords];
    alignas(64) std::uint32_t sequence;
    alignas(64) std::uint32_t row_sequences[8];      // of a top-k launch's rows
    alignas(64) std::uint64_t handed[kMostHanded];   // sequence << 32 | token
  };
  // Waits until arrived(): the one way to read what the device writes.
  template <typename Arrived>
  void await(const Arrived& arrived);
  // hand-overs in a row without a wait for the stream, for which the runtime keeps a
  // little of every launch
  static constexpr std::uint32_t kMostUnwaited = 256U;
  void* stream_{};
  std::uint32_t vocabulary_{};
  void* workspace_{};
  std::size_t workspace_bytes_{};
  TopKRows top_k_rows_{};
  Staging* staging_{};
  std::uint32_t sequence_{};
  std::uint32_t handed_sequence_{};
  std::uint32_t handed_tokens_[kMostHanded]{};
  std::uint32_t unwaited_{};
  bool replayed_{};
  std::uint64_t gpu_calls_{};
  std::uint64_t logit_transfer_bytes_{};
};

}  // namespace qllm

// A model's program one operation at a time, with a request of its own for the embedding:
// what a host that keeps requests per operation does, and no public call of the library.
#include "model_host.hpp"

#include <cstdint>
#include <cstdio>
#include <memory>
#include <string>
#include <vector>

namespace er = expert::runtime;

// `prompt`, then `steps` tokens, each the last one selected; the last `penalised` of them
// under a presence penalty of 2.  With `bare_embedding` the embedding's request has no
// parameters.  The tokens selected are left in `selected` [1 + steps].
extern "C" int32_t qprobe_operations(const char* path, const uint32_t* prompt, uint32_t count,
                                     uint32_t steps, uint32_t penalised,
                                     int32_t bare_embedding, uint32_t* selected) try {
  qllm::ArtifactProviderOptions options;
  options.max_context = count + steps + 8U;
  options.capacity = 1U;
  options.kv_page_tokens = 32U;
  options.kv_cache_dtype = "fp32";
  std::unique_ptr<qllm::ModelHost> host;
  if (const auto status = qllm::ModelHost::open(path, options, host); !status.ok())
    throw std::runtime_error(std::string(status.message()));
  std::unique_ptr<qllm::ProgramSession> session;
  if (const auto status = host->begin(qllm::greedy_request(1U), session); !status.ok())
    throw std::runtime_error(std::string(status.message()));
  const auto& prepared = host->prepared();
  const auto& program = prepared.bound.program;
  std::uint32_t position = 0U, last = 0U;
  for (std::uint32_t step = 0; step <= steps; ++step) {
    const std::vector<std::uint32_t> tokens =
        step ? std::vector<std::uint32_t>{last}
             : std::vector<std::uint32_t>(prompt, prompt + count);
    std::vector<std::uint32_t> positions(tokens.size());
    for (std::size_t row = 0; row < tokens.size(); ++row)
      positions[row] = position + static_cast<std::uint32_t>(row);
    auto request = session->request();
    if (step > steps - penalised)
      request.parameters["sampling_presence_penalty_biased_ppm"] = 4'000'000U;
    auto bare = request;
    if (bare_embedding) bare.parameters.clear();
    std::vector<er::ExecutionValue> values(program.values.size());
    for (const auto& endpoint : program.inputs) {
      const auto& abi = program.values.at(endpoint.value_index).abi;
      auto words = std::make_shared<std::vector<std::uint32_t>>(
          endpoint.role == "token_ids" ? tokens : positions);
      const auto* bytes = reinterpret_cast<const std::byte*>(words->data());
      const std::uint64_t size = words->size() * 4U;
      values[endpoint.value_index] = {std::string(abi), "host", std::move(words), bytes, size};
    }
    for (std::size_t index = 0; index < program.operations.size(); ++index) {
      const auto& compiled = program.operations[index];
      std::vector<er::ExecutionValue> operands;
      for (const auto& binding : compiled.input_values)
        operands.push_back(values.at(binding.value_index));
      auto handle = host->provider().execute(
          *prepared.operations[index], session->state(),
          er::OperationInvocation{index ? request : bare, compiled, operands});
      auto result = handle.poll();
      if (!result) throw std::runtime_error("operation did not complete");
      if (!result->status.ok()) throw std::runtime_error(std::string(result->status.message()));
      for (std::size_t port = 0; port < compiled.output_values.size(); ++port)
        values[compiled.output_values[port].value_index] = result->outputs.at(port);
    }
    for (const auto& endpoint : program.outputs)
      if (endpoint.role == "token_ids")
        last = *reinterpret_cast<const std::uint32_t*>(values[endpoint.value_index].data);
    selected[step] = last;
    position += static_cast<std::uint32_t>(tokens.size());
  }
  return 0;
} catch (const std::exception& error) {
  std::fprintf(stderr, "qprobe_operations: %s\n", error.what());
  return 1;
}

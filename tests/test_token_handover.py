"""When a token selector waits for its stream and when it watches for the device's words:
its sources over a runtime that counts waits and runs what a stream holds only when the
stream is waited for, or at once."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PROVIDER = os.path.join(ROOT, "quantum-llm_amd", "provider")

DRIVER = r"""
#include "token_selector.hpp"
#include "qllm_kernels.h"
#include <hip/hip_runtime.h>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <stdexcept>

static int waits;
static bool lazy, lost;                 // launches run when waited for; never
static std::function<void()> pending;

extern "C" {
hipError_t hipMalloc(void** p, size_t n) { *p = std::calloc(1, n); return hipSuccess; }
hipError_t hipFree(void* p) { std::free(p); return hipSuccess; }
hipError_t hipHostMalloc(void** p, size_t n, unsigned) { *p = std::calloc(1, n); return hipSuccess; }
hipError_t hipHostFree(void* p) { std::free(p); return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "error"; }
hipError_t hipMemcpyAsync(void* to, const void* from, size_t n, hipMemcpyKind, hipStream_t) {
  std::memcpy(to, from, n);
  return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) {
  ++waits;
  if (pending) pending();
  pending = nullptr;
  return hipSuccess;
}
const char* qllm_last_error(void) { return "error"; }
int32_t qllm_publish_words(const uint32_t* words, uint32_t count, uint32_t* host,
                           uint32_t* host_sequence, uint32_t sequence, uint8_t*, uint32_t,
                           void*) {
  const auto run = [=] {
    std::memcpy(host, words, count * 4u);
    __atomic_store_n(host_sequence, sequence, __ATOMIC_RELEASE);
  };
  if (lost) return QLLM_OK;
  if (lazy) pending = run; else run();
  return QLLM_OK;
}
size_t qllm_argmax_workspace_bytes(uint32_t, uint32_t) { return 0; }
size_t qllm_topk_workspace_bytes(uint32_t, uint32_t) { return 0; }
size_t qllm_topk_batch_workspace_bytes(uint32_t, uint32_t, uint32_t) { return 0; }
int32_t qllm_mark_presence_values(uint8_t*, const uint32_t*, uint32_t, uint32_t, void*) { return QLLM_OK; }
int32_t qllm_apply_presence_penalty(float*, const uint8_t*, uint32_t, float, void*) { return QLLM_OK; }
int32_t qllm_argmax_batch(const float*, uint32_t, uint32_t, uint32_t*, void*, size_t, void*) { return QLLM_OK; }
int32_t qllm_topk_logits_batch(const float*, uint32_t, size_t, uint32_t, uint32_t, float*,
                               uint32_t*, void*, size_t, void*) { return QLLM_OK; }
}

#define EXPECT(x) do { if (!(x)) { std::printf("line %d: %s\n", __LINE__, #x); return 1; } } while (0)

int main() {
  qllm::TokenSelector selector(nullptr, 64u, nullptr, 0u);
  std::uint32_t word = 7u;
  // a pass launched one by one is waited for, every time
  for (int pass = 1; pass <= 40; ++pass) {
    word = static_cast<std::uint32_t>(pass);
    EXPECT(selector.read_token(&word) == word && waits == pass);
  }
  // a replayed graph's words are watched; one reading, and the next is waited for
  waits = 0;
  selector.replayed();
  EXPECT(selector.read_token(&word) == word && waits == 0);
  EXPECT(selector.read_token(&word) == word && waits == 1);
  // a graph that its owner waits for
  selector.replayed();
  selector.replayed(false);
  EXPECT(selector.read_token(&word) == word && waits == 2);
  // many replays in a row: one wait in 256
  waits = 0;
  for (int pass = 0; pass < 1024; ++pass) {
    selector.replayed();
    EXPECT(selector.read_token(&word) == word);
  }
  EXPECT(waits == 4);
  // words that are late arrive with the stream, words that never do are an error
  waits = 0;
  lazy = true;
  word = 9u;
  selector.replayed();
  EXPECT(selector.read_token(&word) == 9u && waits == 1);
  EXPECT(selector.read_token(&word) == 9u && waits == 2);
  lost = true;
  for (const bool graph : {false, true}) {
    selector.replayed(graph);
    bool thrown = false;
    try { (void)selector.read_token(&word); } catch (const std::runtime_error&) { thrown = true; }
    EXPECT(thrown);
  }
  std::puts("ok");
  return 0;
}
"""

HANDED = DRIVER[:DRIVER.index("int main()")] + r"""
int main() {
  qllm::TokenSelector selector(nullptr, 64u, nullptr, 0u);
  std::uint64_t* const host = selector.handed_words();
  // tokens that are there with their number are read without a launch; watched after a
  // replayed graph, waited for otherwise
  for (std::uint32_t pass = 1; pass <= 40; ++pass) {
    const std::uint32_t number = selector.next_handover();
    EXPECT(number == pass);
    for (std::uint32_t row = 0; row < 8u; ++row)
      host[row] = std::uint64_t{number} << 32 | (pass + row);
    waits = 0;
    if (pass % 2u) selector.replayed();
    const std::uint32_t* const tokens = selector.read_handed(8u);
    for (std::uint32_t row = 0; row < 8u; ++row) EXPECT(tokens[row] == pass + row);
    EXPECT(waits == (pass % 2u ? 0 : 1));
  }
  // a row that is late arrives with the stream; one that never does is an error, and so
  // is the token of an earlier pass
  const std::uint32_t number = selector.next_handover();
  host[0] = std::uint64_t{number} << 32 | 5u;
  pending = [=] { host[1] = std::uint64_t{number} << 32 | 0xffffffffu; };
  selector.replayed();
  waits = 0;
  EXPECT(selector.read_handed(2u)[1] == 0xffffffffu && waits == 1);
  (void)selector.next_handover();
  for (const bool graph : {false, true}) {
    selector.replayed(graph);
    bool thrown = false;
    try { (void)selector.read_handed(1u); } catch (const std::runtime_error&) { thrown = true; }
    EXPECT(thrown);
  }
  // which requests emit the arg-max as it is
  qllm::er::ProgramRequestContext request;
  EXPECT(!qllm::TokenSelector::marks_handed(request, 9u));
  request.parameters["sampling_first_output_position"] = 5u;
  request.parameters["sampling_temperature_ppm"] = 0u;
  request.parameters["sampling_presence_penalty_biased_ppm"] = 2'000'000u;
  EXPECT(qllm::TokenSelector::marks_handed(request, 5u));
  EXPECT(!qllm::TokenSelector::marks_handed(request, 4u));
  request.parameters["sampling_presence_penalty_biased_ppm"] = 2'000'001u;
  EXPECT(!qllm::TokenSelector::marks_handed(request, 5u));
  request.parameters["sampling_presence_penalty_biased_ppm"] = 2'000'000u;
  request.parameters["sampling_temperature_ppm"] = 1u;
  EXPECT(!qllm::TokenSelector::marks_handed(request, 5u));
  std::puts("ok");
  return 0;
}
"""


def test_only_replayed_graphs_leave_the_stream_unwaited_for(tmp_path):
    run_driver(tmp_path, DRIVER)


def test_tokens_handed_over_with_their_number(tmp_path):
    run_driver(tmp_path, HANDED)


def run_driver(tmp_path, driver):
    if not os.path.isdir("/opt/rocm/include/hip"):
        pytest.skip("the runtime's headers are not installed")
    source, binary = tmp_path / "driver.cpp", tmp_path / "driver"
    source.write_text(driver)
    done = subprocess.run(
        ["g++", "-std=c++20", "-O1", "-D__HIP_PLATFORM_AMD__", "-I" + os.path.join(ROOT, "include"),
         "-I" + os.path.join(PROVIDER, "include"), "-I" + PROVIDER, "-isystem", "/opt/rocm/include",
         str(source), *(os.path.join(PROVIDER, name) for name in
                        ("token_selector.cpp", "host_support.cpp", "operation_handles.cpp",
                         "speculative_sampling.cpp")),
         "-o", str(binary)], capture_output=True, text=True, timeout=300)
    assert done.returncode == 0, done.stderr[-4000:]
    ran = subprocess.run([str(binary)], capture_output=True, text=True, timeout=60)
    assert ran.returncode == 0 and ran.stdout == "ok\n", ran.stdout + ran.stderr

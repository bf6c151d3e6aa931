// checks.cpp -- host-side checks of the library on a HIP runtime without a
// device (fake_hip.hpp).
//
//   checks failures KIND CASE   makes the first, second, ... call of KIND (new,
//                               launch, copy) fail in a batched prompt, until
//                               one runs through.  Every call returns a status,
//                               leaves no copy of host memory in flight and
//                               frees none under one; a failed ring prompt
//                               leaves the ring as it was, and the next prompt
//                               works.
//   checks launches             one line per product read from stdin ("mode
//                               pair T N K offset", offset: bytes that W is off
//                               16-byte alignment): the kernels it launches,
//                               "name gx gy gz block lds" each, tab-separated
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include <new>

#include "fake_hip.hpp"
#include "gemma_hip.h"
#include "runtime/runtime.hpp"

gh_status gh::noalloc_setup(int) { return GH_OK; }

namespace {
gh_context* context(const char* dir) {
  gh_context* ctx = nullptr;
  if (gh_context_init(dir, &ctx) != GH_OK) {
    fprintf(stderr, "context: %s\n", gh_last_error());
    exit(2);
  }
  return ctx;
}

int bad = 0;
#define CHECK(cond, ...)          \
  do {                            \
    if (!(cond)) {                \
      bad++;                      \
      printf("FAILED: " __VA_ARGS__); \
      printf("\n");               \
    }                             \
  } while (0)

constexpr uint32_t A = 4, W = 16, R = 4, SLOTS = A + W + R, H = 256;

struct Ring {
  std::vector<uint32_t> clocks, flags;
  bool operator==(const Ring& o) const { return clocks == o.clocks && flags == o.flags; }
};
Ring device_ring(gh_model* m) {
  Ring r{std::vector<uint32_t>(SLOTS), std::vector<uint32_t>(SLOTS)};
  gh_model_read_tensor(m, -1, GH_T_RING_CLOCKS, r.clocks.data(), SLOTS * 4);
  gh_model_read_tensor(m, -1, GH_T_RING_FLAGS, r.flags.data(), SLOTS * 4);
  return r;
}
Ring host_ring(gh_model* m) {  // (no recall slot is in use: clearing them uploads the host's state)
  gh_model_ring_clear_recall(m);
  return device_ring(m);
}

// A prompt of T tokens at clock `first` on a ring that holds the tokens before
// it; `lists`: through gh_model_prefill with lists of the host's own ring.
int failures(gh_context* ctx, fake::Kind kind, uint32_t T, uint32_t first, uint32_t head_dim, bool lists, bool warm) {
  gh_model_config c{};
  c.vocab_size = 64;
  c.hidden_size = H;
  c.intermediate_size = 512;
  c.num_hidden_layers = 2;
  c.num_attention_heads = 4;
  c.num_key_value_heads = c.num_global_key_value_heads = 2;
  c.head_dim = c.global_head_dim = head_dim;
  c.max_slots = SLOTS;
  c.rms_norm_eps = 1e-6f;
  c.rope_theta = c.rope_theta_full = 1e4f;
  std::vector<float> x((size_t)std::max(T, first) * H, 0.5f);
  long n = 1;
  for (; n < 2000; n++) {
    gh_model* m = nullptr;
    if (gh_model_init_synthetic(ctx, &c, GH_QUANT_Q4, 1, &m) != GH_OK ||
        gh_model_ring_init(m, A, W, R) != GH_OK) {
      fprintf(stderr, "model: %s\n", gh_last_error());
      exit(2);
    }
    uint32_t token = 0;
    if (warm && gh_model_ring_prefill(m, x.data(), T, 0, 0, &token) != GH_OK) exit(2);
    if (warm) gh_model_ring_init(m, A, W, R);
    if (first && gh_model_ring_prefill(m, x.data(), first, 0, 0, &token) != GH_OK) exit(2);
    const Ring before = device_ring(m);
    std::vector<uint64_t> clocks(T);
    std::vector<uint32_t> slots(T), active((size_t)T * SLOTS), count(T);
    gh_ring* own = nullptr;
    gh_ring_create(1, A, W, R, &own);
    for (uint32_t t = 0; t < first; t++) gh_ring_activate_slot(own, 0, t);
    for (uint32_t t = 0; t < T; t++) {
      clocks[t] = first + t;
      slots[t] = gh_ring_activate_slot(own, 0, clocks[t]);
      count[t] = gh_ring_active_slots(own, 0, clocks[t], &active[(size_t)t * SLOTS], SLOTS);
    }
    gh_ring_destroy(own);
    fake::freed_under_copy = 0;
    gh_status st = GH_OK;
    bool escaped = false;
    fake::fail_nth(kind, n);
    try {
      st = lists ? gh_model_prefill(m, x.data(), T, clocks.data(), slots.data(), active.data(), SLOTS, count.data(),
                                    1, &token)
                 : gh_model_ring_prefill(m, x.data(), T, first, 1, &token);
    } catch (const std::bad_alloc&) {
      escaped = true;
    }
    const bool hit = fake::failed(kind);  // (the call may still succeed, for instance without its early copy)
    fake::fail_nth(kind, 0);
    CHECK(!escaped, "call %ld: an exception left the entry point", n);
    CHECK(fake::pending_host_copies() == 0, "call %ld: %zu copies of host memory in flight", n,
          fake::pending_host_copies());
    CHECK(fake::freed_under_copy == 0, "call %ld: %zu blocks freed under a copy", n, fake::freed_under_copy);
    gh_sync(ctx);
    if (!escaped && st != GH_OK) {
      CHECK(gh_last_error()[0] != 0, "call %ld: no message", n);
      if (!lists) CHECK(device_ring(m) == before, "call %ld: the device's ring changed", n);
      if (!lists || T <= SLOTS) CHECK(host_ring(m) == before, "call %ld: the host's ring changed", n);
      CHECK(gh_model_ring_prefill(m, x.data(), T, first, 1, &token) == GH_OK, "call %ld: the next prompt: %s", n,
            gh_last_error());
    }
    const Ring now = device_ring(m);
    CHECK(escaped || now.clocks[A] != 0 || T + first <= A, "call %ld: the prompt's slots are not active", n);
    CHECK(escaped || host_ring(m) == now, "call %ld: the host's ring is not the device's", n);
    gh_model_deinit(m);
    if (st == GH_OK && !escaped && !hit) break;
  }
  return (int)n;
}

void launches(gh_context* ctx) {
  char mode[8];
  unsigned pair, T, N, K, off;
  while (scanf("%7s %u %u %u %u %u", mode, &pair, &T, &N, &K, &off) == 6) {
    const gh_quant_mode q = mode[1] == '4' ? GH_QUANT_Q4 : mode[1] == '8' ? GH_QUANT_Q8 : GH_QUANT_NONE;
    fake::launches.clear();
    // (no kernel runs: the addresses only have the right alignment)
    const auto at = [](uintptr_t a) { return reinterpret_cast<float*>(a); };
    const gh_status st = pair ? gh_prefill_gate_up_geglu(ctx, q, at(4096 + off), at(8192 + off), at(4096), at(4096), T, N, K)
                              : gh_prefill_gemm(ctx, q, at(4096 + off), at(4096), at(4096), T, N, K);
    if (st != GH_OK) printf("error %s", gh_last_error());
    for (const auto& l : fake::launches)
      if (l.name != "gh_fill_u32_k")
        printf("%s %u %u %u %u %u\t", l.name.c_str(), l.grid[0], l.grid[1], l.grid[2], l.block, l.lds);
    printf("\n");
  }
}
}  // namespace

int main(int argc, char** argv) {
  if (argc < 3) return 2;
  gh_context* ctx = context(argv[1]);
  if (!strcmp(argv[2], "launches")) {
    launches(ctx);
  } else if (argc >= 9) {  // DIR failures KIND T FIRST HEAD_DIM LISTS WARM
    const fake::Kind kind = argv[3][0] == 'n' ? fake::kNew : argv[3][0] == 'l' ? fake::kLaunch : fake::kCopy;
    const int n = failures(ctx, kind, atoi(argv[4]), atoi(argv[5]), atoi(argv[6]), atoi(argv[7]), atoi(argv[8]));
    printf("%d calls failed\n", n - 1);
  }
  gh_context_deinit(ctx);
  return bad ? 1 : 0;
}

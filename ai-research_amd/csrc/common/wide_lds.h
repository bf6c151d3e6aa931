// wide_lds.h -- the LDS of the wide prefill tile (64 tm tokens by br weight
// rows), laid out by the gfx950 kernel and allocated by the host launcher:
// `stages` steps of A, `groups` groups of four blocks of W (bf16: a step's W
// beside its A), and a place for the unused part of a group's last load.
#pragma once
#include <stdint.h>

#define WIDE_LDS_MAX (160u * 1024u)  // a CU's
#define WIDE_CHUNKS_Q4 5u            // 16-byte pieces of a row's four blocks
#define WIDE_CHUNKS_Q8 9u
#define WIDE_CHUNKS_BF16 4u  // of a step's 32 values

struct WideLds {
  uint32_t a, b, pad;        // bytes of one step of A, of one group (bf16: step) of W
  uint32_t groups, stages;   // (bf16: no groups)
  uint32_t bytes;            // all of it
};

constexpr WideLds wide_lds(bool bf16, uint32_t chunks, uint32_t tm, uint32_t br) {
  WideLds l = {64 * tm * 128, br * 16 * chunks, bf16 ? 0u : 1024u, 0, 0, 0};
  l.groups = bf16 ? 0 : 3 * l.a + 3 * l.b + l.pad <= WIDE_LDS_MAX ? 3 : 2;
  const uint32_t fit = (WIDE_LDS_MAX - l.pad - l.groups * l.b) / (l.a + (bf16 ? l.b : 0));
  l.stages = fit < 5 ? fit : 5;
  l.bytes = l.stages * l.a + (bf16 ? l.stages : l.groups) * l.b + l.pad;
  return l;
}

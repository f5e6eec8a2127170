// Host build of fp8_linear's launch plans (colormlm_amd/csrc/
// s14_linear_plan.h) for the CPU test of their sizing and rules.
#include <stdint.h>

#include "s14_linear_plan.h"

extern "C" void lin_plan(uint32_t m, uint32_t n, uint32_t groups, uint32_t *cw, uint32_t *blocks) {
  const s14::LinFastPlan p = s14::lin_fast_plan(m, n, groups);
  *cw = p.cw;
  *blocks = p.blocks;
}

extern "C" uint32_t lin_chunks(uint32_t groups, uint32_t tiles, uint32_t blocks, uint32_t ntok) {
  return s14::lin_fast_chunks(groups, tiles, blocks, ntok);
}

extern "C" void lin_limits(uint64_t *part_bytes, uint32_t *counters, uint32_t *stage_bytes, uint32_t *tile) {
  *part_bytes = s14::kLinPartBytes;
  *counters = s14::kLinMaxCounters;
  *stage_bytes = s14::kLinStageBytes;
  *tile = s14::kLinTile;
}

extern "C" void lin_gemm(uint32_t m, uint32_t n, uint32_t groups, uint32_t *tokens, uint32_t *splits) {
  const s14::LinGemmPlan p = s14::lin_gemm_plan(m, n, groups);
  *tokens = p.tokens;
  *splits = p.splits;
}

extern "C" uint32_t lin_exact(uint32_t m, uint32_t n, uint32_t groups, uint32_t *tokens, uint32_t *waves) {
  const s14::LinExactPlan p = s14::lin_exact_plan(m, n, groups);
  *tokens = p.tokens;
  *waves = p.waves;
  return s14::lin_exact_first(m, n, groups);
}

extern "C" uint32_t lin_route_of(int fast, uint32_t m, uint32_t n, uint32_t k, int f32_scales, int aligned) {
  return uint32_t(s14::lin_route(fast != 0, m, n, k, f32_scales != 0, aligned != 0));
}

// Bit i: kind i of the EXACT f32-MFMA plan is launched at some size.
extern "C" uint32_t lin_exact_kinds(uint32_t *count) {
  *count = uint32_t(sizeof(s14::kLinExactKinds) / sizeof(s14::kLinExactKinds[0]));
  uint32_t seen = 0;
  for (uint32_t tiles = 1; tiles <= 600; ++tiles)
    for (uint32_t groups = 1; groups <= 1024; groups += groups < 64 ? 1 : 64)
      for (uint32_t m = 2; m <= 300; ++m) {
        if (s14::lin_route(false, m, 64 * tiles, 128 * groups, false, true) != s14::LinRoute::kExactMfma) continue;
        const uint32_t first = s14::lin_exact_first(m, 64 * tiles, groups);
        for (uint32_t part : {first, m - first}) {
          if (!part) continue;
          const s14::LinExactPlan p = s14::lin_exact_plan(part, 64 * tiles, groups);
          for (uint32_t i = 0; i < *count; ++i)
            if (s14::kLinExactKinds[i].tokens == p.tokens && s14::kLinExactKinds[i].waves == p.waves) seen |= 1u << i;
        }
      }
  return seen;
}

// Launch planning of fp8_linear: which kernel takes a call (lin_route) and its
// sizes.  FAST: how many 128-k chunks each wavefront of k_linear_fast streams
// (its K split is groups / cw) and how many 32-token blocks one launch takes,
// so that the split-K partials and the arrival counters always fit the
// context's linear workspace; the K splits of k_linear_gemm.  EXACT: the tile
// of k_linear_exact_mfma, and the tokens of a first launch where two are
// faster.  Plain C++ (no HIP types): the library and a host-only test include
// it.
#pragma once

#include <cstddef>
#include <cstdint>
#include <initializer_list>

namespace s14 {

constexpr uint32_t kLinGroup = 128;                 // k values per activation / weight scale (fp8.py:14)
constexpr uint32_t kLinTile = 32;                   // FAST: output rows (and token columns) per MFMA tile
constexpr size_t kLinPartBytes = size_t(32) << 20;  // FAST split-K partials (per context)
constexpr uint32_t kLinMaxCounters = 65536;         // FAST: one arrival counter per (row tile, token block)
// Staged activations per wavefront: ntok x cw chunks x 128 bf16, plus the
// f32 scale of every (token, chunk) when the scales are f32.
constexpr uint32_t kLinStageBytes = 40u * 1024u;
// Wavefronts a FAST launch aims for (more K splits fill the GPU for short,
// wide weights; fewer amortise the ring's prologue).
constexpr uint32_t kLinFastWaves = 1024;

constexpr uint32_t lin_stage_bytes(uint32_t ntok, uint32_t cw) { return ntok * cw * (kLinGroup * 2u + 4u); }

// Bytes of split-K partials a launch of `blocks` token blocks writes.
constexpr uint64_t lin_part_bytes(uint32_t tiles, uint32_t blocks, uint32_t splits) {
  return splits > 1u ? uint64_t(tiles) * blocks * splits * kLinTile * kLinTile * sizeof(float) : 0u;
}

// Chunks per wavefront for one launch of `blocks` token blocks: the smallest
// multiple of 4 dividing G that keeps the grid within kLinFastWaves
// wavefronts, else the largest that fits.  A width fits when its staged
// activations fit kLinStageBytes and, if it splits K, the launch's partials
// fit kLinPartBytes and its (tile, block) counters kLinMaxCounters.  0: no
// width fits.
inline uint32_t lin_fast_chunks(uint32_t G, uint32_t tiles, uint32_t blocks, uint32_t ntok) {
  const uint64_t tiles_all = uint64_t(tiles) * blocks;
  uint32_t best = 0;
  for (uint32_t cw = 4; cw <= G; cw += 4) {
    if (G % cw) continue;
    if (lin_stage_bytes(ntok, cw) > kLinStageBytes) break;
    const uint32_t splits = G / cw;
    if (splits > 1u && (tiles_all > kLinMaxCounters || lin_part_bytes(tiles, blocks, splits) > kLinPartBytes))
      continue;
    best = cw;
    if (tiles_all * splits <= kLinFastWaves) return cw;
  }
  return best;
}

struct LinFastPlan {
  uint32_t cw;      // chunks per wavefront; 0: FAST cannot take the shape
  uint32_t blocks;  // 32-token blocks per launch (the last launch may take fewer)
};

// The launch plan for m tokens: all token blocks in one launch when a chunk
// width fits them, else halved until one does.  {0, 0} when no width fits
// even one block (G not a multiple of 4, or K split so finely that one
// block's partials exceed the workspace): the caller takes the EXACT path.
inline LinFastPlan lin_fast_plan(uint32_t m, uint32_t n, uint32_t G) {
  if (m == 0 || n == 0 || G == 0 || G % 4u) return {0, 0};
  const uint32_t tiles = (n + kLinTile - 1) / kLinTile;
  const uint32_t ntok = m < kLinTile ? m : kLinTile;
  uint32_t blocks = (m + kLinTile - 1) / kLinTile;
  for (;;) {
    if (const uint32_t cw = lin_fast_chunks(G, tiles, blocks, ntok)) return {cw, blocks};
    if (blocks == 1) return {0, 0};
    blocks = (blocks + 1) / 2;
  }
}

// FAST for prompts (k_linear_gemm): 128 rows x `tokens` per workgroup, K in
// `splits` ranges whose sums go through the workspace.  The split with the
// least estimated time, in ns: a group of one workgroup takes 1,070 alone on
// its CU and 1,600 when two share it (wo_a, wo_b at 512 tokens, 64 a
// workgroup; the 32-token form a little over half); splits write and read
// their sums at about 4 TB/s and take a second launch.
struct LinGemmPlan {
  uint32_t tokens, splits;
};
inline LinGemmPlan lin_gemm_plan(uint32_t m, uint32_t n, uint32_t G) {
  const uint32_t tokens = m <= 32u ? 32u : 64u;
  const uint64_t tiles = (uint64_t(n) + 127u) / 128u * ((uint64_t(m) + tokens - 1u) / tokens);
  const uint64_t alone = tokens == 32u ? 650u : 1070u, shared = tokens == 32u ? 900u : 1600u;
  LinGemmPlan best{tokens, 1};
  uint64_t least = ~uint64_t(0);
  for (uint32_t s : {1u, 2u, 3u, 4u, 6u, 8u, 12u, 16u, 24u, 32u}) {
    const uint64_t part = uint64_t(m) * n * s * sizeof(float), per = (G + s - 1u) / s;
    // four groups a split or more (as k_linear_fast has: more partial sums
    // round more often); the last one takes what is left, at least one
    if (s > 1u && (part > kLinPartBytes || per < 4u || uint64_t(s - 1u) * per >= G)) continue;
    const uint64_t wgs = tiles * s;
    const uint64_t t = (wgs <= 256u ? alone : (wgs + 511u) / 512u * shared) * per +
                       (s > 1u ? 3000u + 2u * part / 4000u : 0u);
    if (t < least) {
      least = t;
      best.splits = s;
    }
  }
  return best;
}

// EXACT on the f32 MFMA (k_linear_exact_mfma): tokens per workgroup and
// wavefronts per workgroup, the pair with the least estimated time.  A
// workgroup is 64 rows x `tokens`; its wavefronts take ceil(G / waves) groups
// each, and whole rounds of 256 workgroups count.  ns per group of four
// wavefronts, measured at wo_a and wo_b with at most one workgroup per CU
// (alone) and with several: few wide tiles leave MFMA latency and the LDS
// reads uncovered, many small ones convert the same weights more often.
struct LinExactPlan {
  uint32_t tokens, waves;
  uint64_t ns;  // estimated
};
struct LinExactKind {
  uint32_t tokens, waves, alone_ns, shared_ns;
};
// (8 tokens on 8 wavefronts was the fastest at no size: 16 wavefronts of four
// tokens or 4 of eight are.)
constexpr LinExactKind kLinExactKinds[] = {{4, 4, 1760, 1110},  {4, 16, 1220, 1420}, {8, 4, 3000, 1900},
                                           {16, 4, 3200, 2600}, {16, 8, 2650, 2850}, {32, 4, 5300, 4660}};
inline LinExactPlan lin_exact_plan(uint32_t m, uint32_t n, uint32_t G) {
  const uint64_t tiles = (uint64_t(n) + 63u) / 64u;
  LinExactPlan best{0, 0, ~uint64_t(0)};
  for (const LinExactKind &k : kLinExactKinds) {
    const uint64_t wgs = tiles * ((uint64_t(m) + k.tokens - 1u) / k.tokens);
    const uint64_t t = (wgs + 255u) / 256u * ((G + k.waves - 1u) / k.waves) * (k.waves / 4u) *
                       (wgs <= 256u ? k.alone_ns : k.shared_ns);
    if (t < best.ns) best = {k.tokens, k.waves, t};
  }
  return best;
}
// Tokens of a first launch when two launches (whole 32-token blocks, then
// the rest) are estimated faster than one, else m: a last round of a few
// workgroups costs as much as a full one (wo_a at 333 tokens: 11 blocks of 128
// workgroups are 5.5 rounds, run as 6; 10 blocks and 13 tokens on their own
// 214 us against 224).
constexpr uint64_t kLinLaunchNs = 5000;
inline uint32_t lin_exact_first(uint32_t m, uint32_t n, uint32_t G) {
  uint64_t least = lin_exact_plan(m, n, G).ns;
  uint32_t first = m;
  for (uint32_t cut = m / 32u * 32u, i = 0; cut > 0u && i < 8u; cut -= 32u, ++i) {
    if (cut == m) continue;
    const uint64_t t = lin_exact_plan(cut, n, G).ns + lin_exact_plan(m - cut, n, G).ns + kLinLaunchNs;
    if (t < least) {
      least = t;
      first = cut;
    }
  }
  return first;
}

// Is k_linear_tile with k_linear_sum estimated faster than the f32 MFMA
// kernel?  Few rows and tokens leave that one a few workgroups whose
// wavefronts take several groups each, where the tiles have a wavefront per
// group: their time goes by rounds of 1,024 wavefronts (graph replays, us,
// tiles / f32 MFMA: [512, 4096] 8 tokens 10.0 / 11.9, 32 tokens 10.8 / 12.0, 64
// tokens 15.5 / 12.2; [2048, 4096] 8 tokens 10.7 / 12.1, 12 tokens 15.3 / 12.1;
// [1024, 8192] 16 tokens 17.1 / 21.5, 32 tokens 26.9 / 21.7; [512, 2048] 2 tokens
// 5.4 / 6.9, 5 tokens 9.1 / 7.1).  The MFMA estimate lacks the launch.
inline bool lin_exact_tiles(uint32_t m, uint32_t n, uint32_t G) {
  const uint64_t waves = (uint64_t(n) + 63u) / 64u * G * ((uint64_t(m) + 7u) / 8u);
  const uint64_t first = m <= 2u ? 5600u : m <= 4u ? 6800u : 9500u, more = m <= 2u ? 2200u : m <= 4u ? 3000u : 5200u;
  return first + (waves + 1023u) / 1024u * more - more < lin_exact_plan(m, n, G).ns + 2000u;
}

// The kernel that takes a call.  `aligned`: x and w start at 16-byte addresses.
constexpr uint32_t kLinGvChunk = 1024;  // k per chunk of k_linear_gemv
enum class LinRoute : uint32_t {
  kGemv,       // FAST, few tokens: k_linear_gemv
  kGemm,       // FAST prompts: k_linear_gemm
  kFast,       // FAST otherwise: k_linear_fast
  kGemvExact,  // one token: k_linear_gemv_exact
  kExactMfma,  // UE8M0 scales on both sides: k_linear_exact_mfma
  kTile,       // k_linear_tile + k_linear_sum
  kExact,      // any other: k_linear_exact
};
inline LinRoute lin_route(bool fast, uint32_t m, uint32_t n, uint32_t k, bool f32_scales, bool aligned) {
  constexpr uint64_t kMax32 = 0xFFFFFFFFull;  // row offsets, of the last tile's rows past n too
  const uint32_t G = (k + kLinGroup - 1u) / kLinGroup;
  // the GEMV where it measured faster than the MFMA tiles (graph replays,
  // us: wq_b m = 1 8.5 against 10.4, m = 2 10.9 against 10.7; wo_a m = 2 11.2
  // against 12.6, m = 3 14.7 against 13.1; wkv m = 4 4.9 against 7.9)
  const bool gemv = m == 1u || (m == 2u && n <= 8192u) || (m <= 4u && n <= 1024u);
  if (fast && gemv && k % kLinGvChunk == 0u && uint64_t(n) * k <= kMax32) return LinRoute::kGemv;
  if (fast && k % (4u * kLinGroup) == 0u) {
    // the prompt tiles from where they measured faster than k_linear_fast
    // (us: wq_b m = 8 11.7 against 12.0, m = 12 17.9 against 11.9; wo_b m = 12 24.3
    // against 13.8; wkv m = 64 14.6 against 17.8, m = 333 27.6 against 17.9)
    if (m > 8u && uint64_t(m) * n * k >= 300000000ull && (uint64_t(n) + 127u) * k <= kMax32) return LinRoute::kGemm;
    if (lin_fast_plan(m, n, G).cw) return LinRoute::kFast;
  }
  const bool vec = k % 16u == 0u && aligned;
  if (m == 1u && vec && uint64_t(n) * k <= kMax32 && (k == 1024u || k == 2048u || k == 4096u || k == 8192u))
    return LinRoute::kGemvExact;
  if (!vec || k % kLinGroup != 0u || (uint64_t(n) + 63u) * k > kMax32) return LinRoute::kExact;
  const bool tile = size_t(G) * n * sizeof(float) <= kLinPartBytes;  // one token's partials fit the workspace
  // the f32 MFMA: UE8M0 scales, whole groups.  Two to four tokens over a k
  // past 4,096 stay on the tiles (wo_b m = 4: 21.5 us against 24.1: 64-row
  // workgroups leave most CUs idle there)
  if (!f32_scales && (m > 4u || k <= 4096u) && !(tile && lin_exact_tiles(m, n, G))) return LinRoute::kExactMfma;
  return tile ? LinRoute::kTile : LinRoute::kExact;
}

}  // namespace s14

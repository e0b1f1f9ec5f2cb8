// How an attention launch runs (attention.hip): which kernel and form, over which work items. Host
// arithmetic only, without HIP, so that it can be walked on a machine without a GPU.
#pragma once

#include <algorithm>
#include <cstdint>

namespace ckv {

#ifndef CKV_ATTN_QG
#define CKV_ATTN_QG 2
#endif
constexpr int kAttnWaves = 4;
constexpr int kAttnQG = CKV_ATTN_QG;                // 16-query groups per wavefront
constexpr int kAttnBM = kAttnWaves * kAttnQG * 16;  // queries per workgroup
constexpr int kAttnBN = 64;                         // cache rows per tile
constexpr int kWaveChunk = 32;                      // cache rows per step of attn_wave_kernel's wavefronts

constexpr int kXcds = 8;  // MI355X: workgroups go round-robin to 8 XCDs, each with its own L2

// Which work item (query block qb, head h, cache split z) a workgroup takes. The hardware hands
// workgroup L of a 1-D grid to XCD L % 8, so items are assigned through L: the XCDs split evenly
// over the KV heads (8 / Hkv XCDs each), every item of one KV head lands on that head's XCDs (its
// K/V stay in their L2s and are read there by all `group` query heads together), consecutive items
// of an XCD cycle through the group's query heads on one query block and split, and query blocks
// go latest position first, alternating between the head's XCDs so their work stays balanced. The
// grid is padded to whole rounds of 8; a workgroup past a head's last item returns. With a KV-head
// count that does not divide 8, all heads are one group over all XCDs. The two divisions are
// multiplications by the host's reciprocals: hardware has no integer division, and four or five
// emulated ones were half a microsecond of every workgroup's start.
struct AttnMap {
  int nqb = 0, group = 0, xpk_log = 0, items = 0;  // items: of one KV head
  uint32_t inv_group = 0, inv_nqb = 0;
  uint32_t blocks = 0;  // the grid
};

// For x / d as a multiplication (div_by): ceil(2^32 / d) where that is exact for every x <= most
// (most d < 2^32), 0 elsewhere.
static uint32_t inverse_of(int64_t most, int64_t d) {
  return d > 1 && most * d < (1ll << 32) ? (uint32_t)(((1ll << 32) + d - 1) / d) : 0;
}

static AttnMap attn_map(int64_t nqb, int Hkv, int group, int64_t splits) {
  AttnMap m;
  if (kXcds % Hkv != 0) {
    group *= Hkv;
    Hkv = 1;
  }
  while ((Hkv << m.xpk_log) < kXcds) ++m.xpk_log;
  m.nqb = (int)nqb;
  m.group = group;
  m.items = (int)(group * nqb * splits);
  m.inv_group = inverse_of(m.items, group);
  m.inv_nqb = inverse_of(nqb * splits, nqb);
  m.blocks = (uint32_t)((((int64_t)m.items + (1 << m.xpk_log) - 1) >> m.xpk_log) * kXcds);
  return m;
}

// How a launch runs.
struct AttnPlan {
  bool wave = false;     // attn_wave_kernel, else attn_active_kernel (its splits are whole tiles)
  bool grouped = false;  // rows are the (token, query head) pairs of a KV head
  int qg = 0, waves = 0;
  int splits = 1, split_chunks = 0;
  AttnMap map;
};

// The (head_dim, QG, W, GROUPED) forms of attn_wave_kernel that attn_plan picks from.
#define CKV_WAVE_FORMS(X)                                                                  \
  X(128, 1, 4, true) X(128, 1, 8, true) X(128, 2, 8, true)                                  \
  X(128, 1, 4, false) X(128, 1, 8, false) X(128, 2, 4, false) X(128, 2, 8, false)           \
  X(64, 1, 4, true) X(64, 1, 8, true)                                                       \
  X(64, 1, 4, false) X(64, 1, 8, false) X(64, 2, 4, false) X(64, 2, 8, false)

// Where the 128-query workgroups are too few: below about one for each of the 256 CUs at head_dim
// 128 (us, 28 heads, this first: 768 causal rows, 168 workgroups, 19.7 against 20.6; 1000 of 8256
// rows, 224, 157 against 164; 1103 causal rows, 252, 27.8 against 27.1; 1500, 336, 41.1 against
// 36.5), below two at head_dim 64, where they also hold less work each (14 heads: 3000 causal rows,
// 336 workgroups, 37.6 against 46.5; 4000, 448, 58.9 against 61.8; 4500, 504, 72.4 against 69.8).
static bool wave_launch(int n, int Hq, int head_dim) {
  const int64_t blocks = (int64_t)((n + kAttnBM - 1) / kAttnBM) * Hq;
  return blocks < (head_dim == 128 ? 256 : 450);
}

constexpr int kWaveFill = 256;  // workgroups that a split launch aims at: one for each CU

// The most splits a launch takes: a workgroup has at most 32 (token, query head) rows, a split's
// four wavefronts a chunk each.
static int64_t most_splits(int n, int N, int Hq, int head_dim) {
  const int64_t chunks = (N + kWaveChunk - 1) / kWaveChunk;
  if (!wave_launch(n, Hq, head_dim) || chunks <= 16) return 1;
  return std::max<int64_t>(1, std::min<int64_t>(kWaveFill * 32 / ((int64_t)n * Hq), (chunks + 3) / 4));
}

// The plan without split 128-query workgroups.
static AttnPlan attn_base_plan(int n, int N, int Hq, int Hkv, int head_dim, int64_t workspace_bytes) {
  AttnPlan p;
  const int group = Hq / Hkv;
  if (!wave_launch(n, Hq, head_dim)) {
    p.map = attn_map((n + kAttnBM - 1) / kAttnBM, Hkv, group, 1);
    return p;
  }
  p.wave = true;
  p.grouped = group > 1 && (int64_t)n * group <= kAttnBM;
  const int rows = p.grouped ? n * group : n, heads = p.grouped ? Hkv : Hq;
  const int chunks = (N + kWaveChunk - 1) / kWaveChunk;
  const int b16 = (rows + 15) / 16 * heads, b32 = (rows + 31) / 32 * heads;
  // 16 rows a workgroup while those workgroups are all resident at once (two or four of four
  // wavefronts on a CU, by registers), else 32, which read each cache row half as often: 28 heads
  // of 128, 192 causal rows 5.9 against 7.2 us, 320 rows (560 workgroups) 9.8 against 9.0. A long
  // cache is read often enough to prefer 32 earlier at head_dim 128 (251 of 1103 rows 13.7 against
  // 14.1, 300 of 4000 34 against 43).
  const bool lng = chunks >= 24;
  if (rows <= 16) p.qg = 1;
  else if (lng) p.qg = head_dim == 64 && b16 <= 512 ? 1 : 2;
  else p.qg = b16 <= (head_dim == 64 ? 800 : 512) ? 1 : 2;
  // Grouped launches have forms of 16 rows, and at head_dim 128 of 32 rows by eight wavefronts. Up to
  // 64 KV heads the rules ask for no other; with more, the nearest of these.
  if (p.grouped && head_dim == 64) p.qg = 1;
  // 17 to 128 rows over 24 to 63 chunks at head_dim 128: a workgroup's own chain of them is the time
  // (5 queries of 28 heads over 1103 rows 13.9 us, over 1600 17.9), so 16 rows by four wavefronts,
  // split (8.8, 8.9); the three microseconds of the merge are not worth it at head_dim 64 (7.1 whole).
  const int64_t row_b = (int64_t)Hq * n * (head_dim + 4) * 4;
  const int64_t can = std::min<int64_t>(most_splits(n, N, Hq, head_dim), workspace_bytes / row_b);
  if (head_dim == 128 && rows > 16 && lng && chunks < 64) {
    const int64_t splits = std::min<int64_t>(std::min<int64_t>(can, kWaveFill / b16), chunks / 4);
    if (splits > 1) {
      p.qg = 1;
      p.waves = 4;
      p.split_chunks = (int)((chunks + splits - 1) / splits);
      p.splits = (chunks + p.split_chunks - 1) / p.split_chunks;
      p.map = attn_map(b16 / heads, Hkv, p.grouped ? 1 : group, p.splits);
      return p;
    }
  }
  const int blocks = p.qg == 1 ? b16 : b32;
  // Eight wavefronts halve a workgroup's chain where it is long, if the workgroups still fit (one
  // or two on a CU): 300 of 4000 rows 34 against 45 us with four, 768 causal rows 24.5 against 19.1.
  p.waves = (lng && (blocks <= 288 || (blocks <= 450 && chunks >= 128))) || (p.grouped && p.qg == 2) ? 8 : 4;
  // Splits cost the merge launch, about 3 us: taken for one token's rows from 17 chunks on (28
  // heads, 700 rows 7.1 against 8.5 us, 8288 rows 8.7 against 45), else where eight wavefronts
  // would have eight chunks each (150 of 1500 rows, 47 chunks, 8.5 us whole and 9.5 in two).
  int64_t splits = std::min<int64_t>(can, kWaveFill / std::max(blocks, 1));
  if (rows > 16 && chunks < 64) splits = 1;
  if (rows <= 16) p.waves = splits > 1 ? 4 : 8;
  splits = std::max<int64_t>(1, std::min<int64_t>(splits, (chunks + p.waves - 1) / p.waves));
  p.split_chunks = (int)((chunks + splits - 1) / splits);
  p.splits = (chunks + p.split_chunks - 1) / p.split_chunks;
  p.map = attn_map(blocks / heads, Hkv, p.grouped ? 1 : group, p.splits);
  return p;
}

// 128-query workgroups over splits of a long cache. Where a launch has few query blocks the small
// launches' form reads the cache once for every 16 or 32 rows, at half the large kernel's rate, and
// the large kernel unsplit is a chain of every tile on a part of the CUs. The splits that fill the
// card once: of q = n / 128 query blocks (a last block of few rows is little work) with positions
// spread over the cache, split z of s concerns those that reach it, about s (q + 1) / 2 + (q - 1) / 2 of
// a head's q s workgroups, and 512 (head_dim 64: 768) are resident at once.
static int64_t large_splits(int n, int N, int Hq, int head_dim) {
  const int64_t tiles = (N + kAttnBN - 1) / kAttnBN;
  if (tiles < 80) return 1;  // shorter caches: no form gained enough
  const double q = std::max(1.0, (double)n / kAttnBM), per_head = (head_dim == 128 ? 1024.0 : 1536.0) / Hq;
  const double s = (per_head - (q - 1)) / (q + 1) + 0.1;
  return s < 2.0 ? 1 : std::min<int64_t>({(int64_t)s, tiles / 4, 32});
}

// Estimates (us) of a base plan and of the large kernel in `splits`, fitted to 13,000 launches of
// seven head layouts (28 / 4, 32 / 8, 64 / 8, 32 / 32 and 8 / 2 heads of 128, 14 / 2, 32 / 8 and 16 / 16
// of 64; 3-3000 queries over 1103-32832 rows), within about 10 %: a workgroup's chain of chunks or
// tiles, or all chunks at the rate of the card, and the partial rows written and read.
static double base_plan_us(const AttnPlan& p, int n, int N, int Hq, int Hkv, int head_dim) {
  const bool d128 = head_dim == 128;
  if (!p.wave) return 4.0 + (d128 ? 1.35 : 0.95) * ((N + kAttnBN - 1) / kAttnBN);
  const int rows = p.grouped ? n * (Hq / Hkv) : n, heads = p.grouped ? Hkv : Hq;
  const double chunks = (N + kWaveChunk - 1) / kWaveChunk, blocks = (double)((rows + 16 * p.qg - 1) / (16 * p.qg)) * heads;
  const double chain = (int64_t)(chunks + p.splits * p.waves - 1) / (p.splits * p.waves);
  const double step = p.waves == 8 ? (d128 ? 1.9 : 1.05) : (d128 ? 1.4 : 0.9);
  const double work = p.qg == 1 ? (d128 ? 0.27 : 0.12) : (d128 ? 0.34 : 0.185);  // of a CU
  const double seen = p.grouped ? 1.0 : 0.5;  // half the cache, on average
  return 4.0 + std::max(chain * step, blocks * chunks * seen * work / 256) + (p.splits > 1 ? 4.0 : 0.0);
}
static double large_split_us(int n, int N, int Hq, int head_dim, int64_t splits) {
  const int64_t tiles = (N + kAttnBN - 1) / kAttnBN, chain = (tiles + splits - 1) / splits;
  const double partial_mb = (double)splits * n * Hq * (head_dim + 4) * 4e-6;
  return head_dim == 128 ? 10.0 + 2.1 * chain + 0.31 * partial_mb : 7.0 + 1.6 * chain + 0.45 * partial_mb;
}

// Bytes of partial rows at the most splits that a launch of this shape may take; 0: it never splits.
static int64_t attn_most_splits(int n, int N, int Hq, int head_dim) {
  return std::max(most_splits(n, N, Hq, head_dim), large_splits(n, N, Hq, head_dim));
}
static int64_t attn_workspace_bytes(int n, int N, int Hq, int head_dim) {
  const int64_t splits = attn_most_splits(n, N, Hq, head_dim);
  return splits > 1 ? splits * Hq * n * (head_dim + 4) * 4 : 0;
}

// The base plan, or the large kernel in splits where that is estimated to be clearly faster (the
// estimate of an unsplit small launch is the least certain): 28 heads of 128 (us, the base plan first),
// 130 of 8256 rows 63.7 and 45.0, 251 of 32832 232 and 135, 1153 of 8256 168 and 132; 14 heads of 64, 251
// of 32832 116 and 44.8, 1153 of 16400 127 and 76.7. Below 64 rows of a KV head the small launches' form
// stays ahead. Over 1651 shapes of the layouts above 0.90 of the base plan's time in the mean; 11 are
// more than 3 % slower than it, the worst 1.19 (64 / 8 heads of 128, 180 of 32832 rows, 235 and 279).
static AttnPlan attn_plan(int n, int N, int Hq, int Hkv, int head_dim, int64_t workspace_bytes) {
  AttnPlan p = attn_base_plan(n, N, Hq, Hkv, head_dim, workspace_bytes);
  const int group = Hq / Hkv;
  const int64_t splits = large_splits(n, N, Hq, head_dim);
  if (splits < 2 || (int64_t)n * group < 64 || workspace_bytes / ((int64_t)Hq * n * (head_dim + 4) * 4) < splits ||
      large_split_us(n, N, Hq, head_dim, splits) >
          (p.wave && p.splits == 1 ? 0.8 : 0.92) * base_plan_us(p, n, N, Hq, Hkv, head_dim))
    return p;
  const int tiles = (N + kAttnBN - 1) / kAttnBN;
  const int split_tiles = (int)((tiles + splits - 1) / splits);
  p = AttnPlan{};
  p.split_chunks = split_tiles * (kAttnBN / kWaveChunk);
  p.splits = (tiles + split_tiles - 1) / split_tiles;
  p.map = attn_map((n + kAttnBM - 1) / kAttnBM, Hkv, group, p.splits);
  return p;
}

}  // namespace ckv

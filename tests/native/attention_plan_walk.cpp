// Walks the attention launch plan (chunkkv_amd/csrc/attention_plan.hpp) over head counts, group sizes,
// query and cache lengths and workspace sizes, and checks every plan: its kernel form exists, its
// splits cover the cache, none empty, and fit the workspace, and its work items are each taken
// once. Prints the plans checked and the bad ones (the first ten in full).
#include "attention_plan.hpp"

#include <cstdio>
#include <vector>

using namespace ckv;

// div_by of attention.hip
static int divided(int x, int d, uint32_t inv) {
  return inv != 0 ? (int)(((uint64_t)(uint32_t)x * inv) >> 32) : d == 1 ? x : x / d;
}

static bool form_exists(const AttnPlan& p, int D) {
  if (!p.wave) return true;
#define CKV_IS(HD, QG, W, GR) if (D == HD && p.qg == QG && p.waves == W && p.grouped == GR) return true;
  CKV_WAVE_FORMS(CKV_IS)
#undef CKV_IS
  return false;
}

static bool items_once(const AttnPlan& p, int Hq, int Hkv) {
  const AttnMap& m = p.map;
  const int heads = p.grouped ? Hkv : Hq;
  std::vector<char> taken((size_t)heads * m.nqb * p.splits, 0);
  size_t n = 0;
  for (uint32_t L = 0; L < m.blocks; ++L) {  // attn_work_item of attention.hip
    const int xcd = L % kXcds, j = (int)((L / kXcds) << m.xpk_log) + (xcd & ((1 << m.xpk_log) - 1));
    if (j >= m.items) continue;
    const int rest = divided(j, m.group, m.inv_group), h = (xcd >> m.xpk_log) * m.group + (j - rest * m.group);
    const int z = divided(rest, m.nqb, m.inv_nqb), qb = m.nqb - 1 - (rest - z * m.nqb);
    if (h < 0 || h >= heads || z < 0 || z >= p.splits || qb < 0 || qb >= m.nqb) return false;
    char& t = taken[((size_t)z * m.nqb + qb) * heads + h];
    if (t) return false;
    t = 1, ++n;
  }
  return n == taken.size();
}

int main() {
  const int ns[] = {1, 2, 3, 5, 8, 9, 16, 17, 31, 32, 33, 40, 57, 63, 64, 65, 100, 127, 128, 129, 251, 320, 512, 777, 1103, 2000, 4097};
  const int Ns[] = {1, 31, 32, 33, 300, 512, 513, 767, 768, 1103, 2047, 2049, 4096, 8256, 32864, 131072};
  const int kvs[] = {1, 2, 3, 4, 5, 7, 8, 12, 16, 32, 40, 63, 64, 65, 66, 72, 73, 80, 96, 100, 127, 128, 129, 200, 255, 256};
  long checked = 0, bad = 0;
  for (int Hkv : kvs)
    for (int group = 1; group <= 16; ++group)
      for (int D : {64, 128})
        for (int n : ns)
          for (int N : Ns) {
            const int Hq = Hkv * group;
            const int64_t row_b = (int64_t)Hq * n * (D + 4) * 4, need = attn_workspace_bytes(n, N, Hq, D);
            for (int64_t ws : {need, (int64_t)0, need / 2, (int64_t)1 << 50}) {
              const AttnPlan p = attn_plan(n, N, Hq, Hkv, D, ws);
              const int64_t chunks = (N + kWaveChunk - 1) / kWaveChunk;
              bool ok = form_exists(p, D) && p.splits >= 1;
              if (p.splits > 1)
                ok = ok && p.splits * row_b <= ws && p.splits * row_b <= need && (int64_t)p.splits * p.split_chunks >= chunks &&
                     (int64_t)(p.splits - 1) * p.split_chunks < chunks;
              ok = ok && (p.wave || p.split_chunks % (kAttnBN / kWaveChunk) == 0);  // whole tiles
              ok = ok && (p.map.blocks > 3000 || items_once(p, Hq, Hkv));
              ++checked;
              if (!ok && bad++ < 10)
                std::printf("bad: Hq %d Hkv %d D %d n %d N %d workspace %lld: wave %d qg %d waves %d grouped %d splits %d x %d of %lld chunks\n",
                            Hq, Hkv, D, n, N, (long long)ws, p.wave, p.qg, p.waves, p.grouped, p.splits, p.split_chunks, (long long)chunks);
            }
          }
  // the large kernel in splits, at the shapes that the GPU test of it runs
  const int split[][5] = {{28, 4, 128, 5120, 130}, {7, 7, 128, 9001, 700}, {32, 8, 64, 9000, 251}, {12, 3, 64, 8300, 333}};
  for (const auto& t : split) {
    const AttnPlan p = attn_plan(t[4], t[3], t[0], t[1], t[2], (int64_t)1 << 50);
    if (p.wave || p.splits < 2) ++bad, std::printf("not split: %d queries over %d\n", t[4], t[3]);
  }
  std::printf("%ld %ld\n", checked, bad);
  return 0;
}

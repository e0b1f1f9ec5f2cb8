// The attention of a launch too small for 128-query workgroups to fill the chip: decode, short
// prompts, the few rows of a small blend (attention_plan.hpp says which). Included by attention.hip, whose layouts it shares.
//
// Bound: latency. A 128-query workgroup that walks the cache one 64-row tile at a time is a chain
// of dependent steps (load, barrier, product, softmax, product) as long as the cache, and a launch
// of 320 queries has only 84 of them on 256 CUs. Here a workgroup takes 16 QG query rows of one
// head and its W wavefronts share the cache: wavefront w owns the 32-row chunks w, w + W, ... with
// a softmax of its own, and the W partial results meet once, in LDS, at the end. Nothing in the
// loop waits for another wavefront (no barrier): the first chunk's rows are loaded before the
// positions arrive, the next chunk's as soon as its registers are free, and Q, K and V pass through
// a wavefront's own 32 rows of LDS, one after the other, from whole-row loads. (Loading K into the
// registers of its matrix operand directly saves the LDS trip but makes 16 neighbouring lanes read
// 16 rows, 16 bytes each, which the L1 serves at a quarter of the rate: 320 queries of 28 heads
// took 11.0 us that way, 9.0 us now.) GROUPED: as many (token, query head) rows of one KV head per
// workgroup, so that the group's heads share every row it loads (decode). Launches with few
// workgroups even so split the chunks over the grid; each split writes its unnormalised rows with
// their max and sum, and attn_combine_kernel merges them.
// Measured (graph replays, us, the 128-query kernel or its split and grouped forms before): 28
// heads of 128, 320 causal rows 11.4 -> 9.0, 251 rows over 1103 17.5 -> 13.7, one row over 8288
// 14 -> 8.7; 14 heads of 64, 320 causal rows 8.8 -> 5.2, 251 over 1103 16 -> 7.1.
#pragma once

namespace ckv {

// Between the stages in which a wavefront's lanes exchange rows through LDS (and before a stage's rows
// are overwritten): LDS runs one wavefront's operations in order, so this is no instruction, only an
// order of stores and loads that the compiler has to keep though no lane reads its own bytes.
__device__ __forceinline__ void wave_lds_stage() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");
}

template <int D, int QG, int W, bool GROUPED>
__global__ __launch_bounds__(W * 64) void attn_wave_kernel(
    int nqb, int map_group, int xpk_log, int items, uint32_t inv_group, uint32_t inv_nqb,
    const int64_t* __restrict__ pos, int n, int N, const char* __restrict__ kc, const char* __restrict__ vc,
    int64_t kv_hs_b, const char* __restrict__ q, int64_t q_hs_b, int64_t q_ts_b, int Hq, int group, uint32_t inv_gqa,
    float scale_log2, int split_chunks, char* __restrict__ out, float* __restrict__ ws, int32_t* __restrict__ err) {
  constexpr int DS = D / 32, DT = D / 16, CPR = D / 8, ROWB = D * 2;
  constexpr int ROWS = 16 * QG;               // query rows of the workgroup
  constexpr int LI = kWaveChunk * CPR / 64;   // 16-byte loads per lane and chunk, of K and of V
  constexpr int QI = ROWS * CPR / 64;         // of the workgroup's query rows
  constexpr int OP = D + 4;                   // pitch of a partial row in LDS (floats): distinct banks
  constexpr int V_B = W * kWaveChunk * ROWB, O_B = W * ROWS * OP * 4;
  __shared__ __attribute__((aligned(1024))) char lds[V_B > O_B ? V_B : O_B];  // Q, K, V rows in turn, then partial rows
  __shared__ float s_m[W][ROWS], s_l[W][ROWS];

  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64), lane = threadIdx.x % 64;
  const int g = lane / 16, lm = lane % 16;
  int qb, hq, z;
  if (!attn_work_item(nqb, map_group, xpk_log, items, inv_group, inv_nqb, qb, hq, z)) return;
  const int hk = GROUPED ? hq : div_by(hq, group, inv_gqa);
  if (GROUPED) hq *= group;  // the KV head's first query head
  const int n_rows = GROUPED ? n * group : n;
  int row_m[QG];  // token of this lane's rows (n: no query)
  int64_t p64[QG];
#pragma unroll
  for (int qg = 0; qg < QG; ++qg) {
    const int r = qb * ROWS + qg * 16 + lm;
    const int t = GROUPED ? div_by(r, group, inv_gqa) : r;
    row_m[qg] = r < n_rows ? t : n;
    p64[qg] = pos[min(row_m[qg], n - 1)];
  }

  // The chunk a wavefront starts with is known before the positions are: its rows load at once
  // (clamped to the cache's last row), after the queries.
  const char* kh = kc + (int64_t)hk * kv_hs_b;
  const char* vh = vc + (int64_t)hk * kv_hs_b;
  vec16 kr[LI], vr[LI], qr[QI];
  auto load = [&](vec16(&r)[LI], const char* rows, int c) {  // lane l of load i: piece i 64 + l of the chunk
    c = min(c, (N - 1) / kWaveChunk);
    const char* base = rows + (int64_t)c * (kWaveChunk * ROWB);
    const int last = N - 1 - c * kWaveChunk;
#pragma unroll
    for (int i = 0; i < LI; ++i) r[i] = ld16(base + min((i * 64 + lane) / CPR, last) * ROWB + (lane % CPR) * 16);
  };
#pragma unroll
  for (int i = 0; i < QI; ++i) {  // absent rows load the last token's query and store nothing
    const int r = min(qb * ROWS + (i * 64 + lane) / CPR, n_rows - 1);
    const int t = GROUPED ? div_by(r, group, inv_gqa) : r;
    qr[i] = ld16(q + (int64_t)(GROUPED ? hq + r - t * group : hq) * q_hs_b + (int64_t)t * q_ts_b + (lane % CPR) * 16);
  }
  const int begin = ws != nullptr ? z * split_chunks : 0;
  int c = begin + wave;
  load(kr, kh, c);
  load(vr, vh, c);
  // The operand of matrix step ds for row slot s: logical 16-byte piece 4 ds + g, kept at piece
  // (4 ds + g) ^ swz_k(s) of the slot.
  char* wl = lds + wave * kWaveChunk * ROWB;
  auto put = [&](int slot, const vec16& v) { *(vec16*)(wl + slot * ROWB + (((lane % CPR) ^ swz_k<CPR>(slot)) * 16)) = v; };
  auto operand = [&](int slot, int ds) {
    return *(const bf16x8*)(wl + slot * ROWB + (((4 * ds + g) ^ swz_k<CPR>(slot)) * 16));
  };
  bf16x8 qf[QG][DS];
#pragma unroll
  for (int i = 0; i < QI; ++i) put((i * 64 + lane) / CPR, qr[i]);
  wave_lds_stage();
#pragma unroll
  for (int qg = 0; qg < QG; ++qg)
#pragma unroll
    for (int ds = 0; ds < DS; ++ds) qf[qg][ds] = operand(qg * 16 + lm, ds);

  int my_pos[QG], wmax = -1, wmin = N;
#pragma unroll
  for (int qg = 0; qg < QG; ++qg) {
    int p = -1;
    if (row_m[qg] < n) {
      if (p64[qg] < 0 || p64[qg] >= N) flag_error(err, CKV_DEVICE_ERR_RANGE);
      p = p64[qg] < 0 ? 0 : p64[qg] >= N ? N - 1 : (int)p64[qg];
      wmin = min(wmin, p);
    }
    my_pos[qg] = p;
    wmax = max(wmax, p);
  }
  wmax = row16_reduce(wmax, [](int a, int b) { return max(a, b); });  // the lane groups hold the same rows
  wmin = row16_reduce(wmin, [](int a, int b) { return min(a, b); });
  wmax = __builtin_amdgcn_readfirstlane(wmax);
  wmin = __builtin_amdgcn_readfirstlane(wmin);
  int c_end = wmax < 0 ? 0 : wmax / kWaveChunk + 1;
  if (ws != nullptr) c_end = min(c_end, begin + split_chunks);

  f32x4 o[QG][DT], l_acc[QG];
  float m_run[QG];
  const bf16x8 ones = {(__bf16)1.f, (__bf16)1.f, (__bf16)1.f, (__bf16)1.f,
                       (__bf16)1.f, (__bf16)1.f, (__bf16)1.f, (__bf16)1.f};
#pragma unroll
  for (int qg = 0; qg < QG; ++qg) {
    m_run[qg] = -INFINITY;
    l_acc[qg] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) o[qg][dt] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  for (; c < c_end; c += W) {
    const int n0 = c * kWaveChunk;
    wave_lds_stage();
#pragma unroll
    for (int i = 0; i < LI; ++i) {  // K row r = 8 a + 4 t + b to slot 16 t + 4 a + b (kslot_row's inverse)
      const int r = (i * 64 + lane) / CPR;
      put(16 * ((r >> 2) & 1) + 4 * (r >> 3) + (r & 3), kr[i]);
    }
    if (c + W < c_end) load(kr, kh, c + W);  // lands while this chunk is worked on
    wave_lds_stage();
    f32x4 s[QG][2];
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int ds = 0; ds < DS; ++ds) {
        const bf16x8 a = operand(16 * t + lm, ds);
#pragma unroll
        for (int qg = 0; qg < QG; ++qg)
          s[qg][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, qf[qg][ds], ds == 0 ? f32x4{0.f, 0.f, 0.f, 0.f} : s[qg][t], 0, 0, 0);
      }
    // V over the K rows; rows past every query's position become zero (their weights are zero, and
    // a cache row not written yet may hold a NaN)
    const bool edge = n0 + kWaveChunk - 1 > wmax;
    wave_lds_stage();
#pragma unroll
    for (int i = 0; i < LI; ++i) {
      const int slot = (i * 64 + lane) / CPR;
      const vec16 v = edge && n0 + slot > wmax ? vec16{0, 0, 0, 0} : vr[i];
      *(vec16*)(wl + slot * ROWB + (((lane % CPR) ^ swz_v<CPR>(slot)) * 16)) = v;
    }
    if (c + W < c_end) load(vr, vh, c + W);
    wave_lds_stage();

    const bool need_mask = n0 + kWaveChunk - 1 > wmin;
    bf16x8 pb[QG];
#pragma unroll
    for (int qg = 0; qg < QG; ++qg) {
      float x[8];  // rows n0 + 8 g + j
#pragma unroll
      for (int j = 0; j < 8; ++j) x[j] = s[qg][j / 4][j % 4];
      if (need_mask) {
        const int lim = my_pos[qg] - n0 - 8 * g;
#pragma unroll
        for (int j = 0; j < 8; ++j)
          if (j > lim) x[j] = -INFINITY;
      }
      float bm = x[0];
#pragma unroll
      for (int j = 1; j < 8; ++j) bm = fmaxf(bm, x[j]);
      bm = group_max(bm) * scale_log2;
      const bool raise = bm > m_run[qg] + 8.f;
      if (__builtin_amdgcn_ballot_w64(raise)) {
        const float m_new = raise ? bm : m_run[qg];
        const float alpha = m_run[qg] == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m_run[qg] - m_new);
        l_acc[qg] *= alpha;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) o[qg][dt] *= alpha;
        m_run[qg] = m_new;
      }
      const float msub = m_run[qg] == -INFINITY ? 0.f : m_run[qg];
#pragma unroll
      for (int j = 0; j < 8; ++j)
        pb[qg][j] = (__bf16)__builtin_amdgcn_exp2f(__builtin_fmaf(x[j], scale_log2, -msub));
    }
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) {
      const bf16x8 a = v_operand<CPR>(wl, dt, g, lm);
#pragma unroll
      for (int qg = 0; qg < QG; ++qg) o[qg][dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, pb[qg], o[qg][dt], 0, 0, 0);
    }
#pragma unroll
    for (int qg = 0; qg < QG; ++qg) l_acc[qg] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ones, pb[qg], l_acc[qg], 0, 0, 0);
  }

  // Merge the wavefronts: each scales its rows to the common max and leaves them in LDS (over the
  // V chunks: every wavefront is past its last read of them), then all threads sum 8 columns each.
#pragma unroll
  for (int qg = 0; qg < QG; ++qg)
    if (g == 0) s_m[wave][qg * 16 + lm] = m_run[qg];
  __syncthreads();
  float* so = reinterpret_cast<float*>(lds);
#pragma unroll
  for (int qg = 0; qg < QG; ++qg) {
    const int r = qg * 16 + lm;
    float mx = s_m[0][r];
#pragma unroll
    for (int w = 1; w < W; ++w) mx = fmaxf(mx, s_m[w][r]);
    const float sc = m_run[qg] == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m_run[qg] - mx);
    if (g == 0) s_l[wave][r] = l_acc[qg][0] * sc;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) {
      const f32x4 v = o[qg][dt] * sc;
      *(f32x4*)(so + (wave * ROWS + r) * OP + dt * 16 + 4 * g) = v;
    }
  }
  __syncthreads();
  for (int it = threadIdx.x; it < ROWS * CPR; it += W * 64) {
    const int r = it / CPR, col = (it % CPR) * 8;
    const int rr = qb * ROWS + r;
    if (rr >= n_rows) break;  // later items are later rows
    f32x4 a = {0.f, 0.f, 0.f, 0.f}, b = a;
    float l = 0.f, mx = -INFINITY;
#pragma unroll
    for (int w = 0; w < W; ++w) {
      const float* pr = so + (w * ROWS + r) * OP + col;
      a += *(const f32x4*)pr;
      b += *(const f32x4*)(pr + 4);
      l += s_l[w][r];
      mx = fmaxf(mx, s_m[w][r]);
    }
    const int m = GROUPED ? div_by(rr, group, inv_gqa) : rr, h = GROUPED ? hq + rr - m * group : hq;
    if (ws != nullptr) {
      float* prow = ws + (((int64_t)z * Hq + h) * n + m) * (D + 4);  // 16-byte aligned rows
      *(f32x4*)(prow + col) = a;
      *(f32x4*)(prow + col + 4) = b;
      if (col == 0) {
        prow[D] = mx;
        prow[D + 1] = l;
      }
    } else {
      const float inv = 1.f / l;
      a *= inv;
      b *= inv;
      *(vec16*)(out + ((int64_t)m * Hq + h) * ROWB + col * 2) =
          vec16{f32x2_to_bf16x2_bits(a[0], a[1]), f32x2_to_bf16x2_bits(a[2], a[3]), f32x2_to_bf16x2_bits(b[0], b[1]),
                f32x2_to_bf16x2_bits(b[2], b[3])};
    }
  }
}

// Merge the splits of a split launch: for query m and head h, with (M_z, L_z, O_z) the partials
// of split z (max in the log2 domain, sum and unnormalised rows relative to M_z):
//   out = sum_z 2^(M_z - M) O_z / sum_z 2^(M_z - M) L_z,  M = max_z M_z  (splits with M_z = -inf
// saw no visible row and weigh 0). One workgroup per (query, head) with a wavefront for every four
// splits, up to kCombineMaxWaves: each loads its four partials together (one round trip up to 64
// splits; further groups of four follow) and merges them into a running (max, sum, row) with the
// online rescale; the wavefronts' results are merged through LDS. Lane d covers head-dim columns
// d, d + 64.
constexpr int kCombineMaxWaves = 16;
constexpr int kCombineParts = 4;  // partials in flight per wavefront

template <int D>
__global__ __launch_bounds__(kCombineMaxWaves * 64) void attn_combine_kernel(char* __restrict__ out,
                                                                             const float* __restrict__ ws, int n,
                                                                             int Hq, int splits) {
  constexpr int CW = D / 64;  // columns per lane
  constexpr int U = kCombineParts;
  const int waves = blockDim.x / 64;
  const int m = blockIdx.x, hq = blockIdx.y, lane = threadIdx.x % 64, wave = threadIdx.x / 64;
  const int64_t stride = (int64_t)Hq * n * (D + 4);
  const float* base = ws + ((int64_t)hq * n + m) * (D + 4);
  float M = -INFINITY, L = 0.f, acc[CW];
#pragma unroll
  for (int j = 0; j < CW; ++j) acc[j] = 0.f;
  for (int z0 = wave * U; z0 < splits; z0 += U * waves) {
    float mz[U], lz[U], oz[U][CW];
#pragma unroll
    for (int u = 0; u < U; ++u) {  // past the last split: the last one again, weighing nothing
      const float* pz = base + (int64_t)min(z0 + u, splits - 1) * stride;
      mz[u] = pz[D];
      lz[u] = pz[D + 1];
#pragma unroll
      for (int j = 0; j < CW; ++j) oz[u][j] = pz[lane + 64 * j];
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (z0 + u >= splits || mz[u] == -INFINITY) continue;  // uniform: the same partial for every lane
      const float mn = fmaxf(M, mz[u]);
      const float a = __builtin_amdgcn_exp2f(M - mn);  // 0 while M is still -inf
      const float b = __builtin_amdgcn_exp2f(mz[u] - mn);
      L = L * a + lz[u] * b;
#pragma unroll
      for (int j = 0; j < CW; ++j) acc[j] = acc[j] * a + oz[u][j] * b;
      M = mn;
    }
  }
  uint16_t* orow = reinterpret_cast<uint16_t*>(out + ((int64_t)m * Hq + hq) * (D * 2));
  if (waves > 1) {
    __shared__ float s_m[kCombineMaxWaves], s_l[kCombineMaxWaves], s_o[kCombineMaxWaves][D];
    if (lane == 0) {
      s_m[wave] = M;
      s_l[wave] = L;
    }
#pragma unroll
    for (int j = 0; j < CW; ++j) s_o[wave][lane + 64 * j] = acc[j];
    __syncthreads();
    if (wave != 0) return;
    // lane w % 16 weighs wavefront w; every read below is independent of the others
    const int w16 = lane % kCombineMaxWaves;
    const float mw = w16 < waves ? s_m[w16] : -INFINITY, lw = w16 < waves ? s_l[w16] : 0.f;
    float ov[kCombineMaxWaves][CW];
#pragma unroll
    for (int w = 0; w < kCombineMaxWaves; ++w)
#pragma unroll
      for (int j = 0; j < CW; ++j) ov[w][j] = s_o[min(w, waves - 1)][lane + 64 * j];
    const float mx = row16_reduce(mw, [](float a, float b) { return fmaxf(a, b); });
    const float sw = mw == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(mw - mx);
    L = row16_reduce(sw * lw, [](float a, float b) { return a + b; });
#pragma unroll
    for (int j = 0; j < CW; ++j) acc[j] = 0.f;
#pragma unroll
    for (int w = 0; w < kCombineMaxWaves; ++w) {
      const float s = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(sw), w));
#pragma unroll
      for (int j = 0; j < CW; ++j) acc[j] += s * ov[w][j];
    }
  }
  const float inv = 1.f / L;
#pragma unroll
  for (int j = 0; j < CW; ++j) orow[lane + 64 * j] = (uint16_t)f32_to_bf16_bits(acc[j] * inv);
}

}  // namespace ckv

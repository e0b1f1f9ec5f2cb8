// Attention of the active rows over the whole cache, with the causal mask given by positions:
// query row i (absolute position pos[i]) attends to cache rows j <= pos[i] of its KV head.
//
// Reference semantics (src/chunkkv/engine/torch_engine.py): the mask is materialised as a
// boolean (n_active x N) tensor, mask = active[:, None] >= arange(N)[None, :] (:157), and
// F.scaled_dot_product_attention(q, K, V, attn_mask=mask, enable_gqa=True) (:68-72) runs with
// the default scale 1/sqrt(head_dim); query head h reads KV head h / (Hq / Hkv). This kernel
// computes the same function from the positions alone: no mask tensor, no KV-head expansion.
//
// Design (gfx950, flash-attention forward): one workgroup = 4 wavefronts = 128 queries of one
// query head; it walks the cache in 64-row tiles up to the largest position among its queries
// (tiles past a wavefront's own queries are skipped by that wavefront). Both products run on
// the bf16 matrix cores (v_mfma_f32_16x16x32_bf16) in transposed form:
//   S^T = K Q^T   (A = K rows from LDS, B = the wavefront's Q rows held in registers)
//   O^T = V^T P^T (A = V^T rows from LDS, B = P straight from the S^T accumulators)
// so that every lane owns one query (lane % 16) for the whole computation: the online-softmax
// max/sum and the output rows live in that lane and only two xor-shuffles per tile combine the
// four lane groups. K/V tiles go from global memory straight into double-buffered LDS (no
// register staging, one barrier per tile), in swizzled rows that make the fragment reads
// conflict-free; V^T comes out of row-major V through transposing LDS reads. Scores and the output accumulate in
// fp32; P is rounded to bf16 for the second product (as fused SDPA kernels do). Launches with too
// few 128-query workgroups to fill the chip (decode, short prompts, small blends) run
// attention_wave.hpp's kernel instead, or, over a long cache, this one in splits of the cache whose
// partial rows attn_combine_kernel merges (attention_plan.hpp). Built with the MFMA VGPR form (no accumulator-register
// copies around the online-softmax rescale).
// Bound: issue and power together. The matrix cores run half of the cycles and the vector
// instructions most of the rest, so every vector instruction that is not softmax costs time: tile
// addresses are a kept offset on a uniform base (62 -> 8 instructions a tile), wavefront extremes
// are scalar (branches, not selects), the four lanes of a query agree on its max only where a lane
// asks to raise it. Measured (us, 28 heads of 128): 2976 rows over 8256, 216 -> 196 with the
// rows spread evenly (199 GFLOP: 1010 TFLOP/s) and 234 -> 216 as a blend keeps them, most in the chunks
// that moved (215 GFLOP: 996; 203-226 on other cards); 8256 causal rows 480 -> 449 (1089), 2000 51.2 ->
// 47.4; 14 heads of 64, 8256 causal rows 162 -> 144.
// A square bf16 product of 8192 reaches 1300-1400 on this card; inputs of zeros (no toggling) 10 %
// more than these. Not faster: tiles one ahead so that the matrix cores work beside the exponentials
// (209-214 / 478 before this form, with spills), V operands read ahead of their products (the same),
// eight wavefronts on one tile (233 / 476), 48 or 64 queries a wavefront (275 / 453, 322 / 649).
#include <algorithm>

#include "attention_plan.hpp"
#include "ckv_common.hpp"

namespace ckv {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

// Combine a lane's value with the lanes 16 and 32 away (the four lane groups of one query), with
// gfx950's row-swap permutes (VALU, no LDS round trip): each returns the lane's own value and
// its partner's, in an order that depends on the lane, so only order-free combinations are used.
__device__ __forceinline__ float group_max(float v) {
  auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
  auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1]));
}
// f over the 16 lanes of a row, in every lane (row rotations: VALU, no LDS round trip).
template <typename T, typename F>
__device__ __forceinline__ T row16_reduce(T v, F f) {
  static_assert(sizeof(T) == 4, "one VGPR");
  auto from = [](T x, auto ctrl) {
    return __builtin_bit_cast(T, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, x), decltype(ctrl)::value, 0xf, 0xf, false));
  };
  v = f(v, from(v, std::integral_constant<int, 0x128>{}));
  v = f(v, from(v, std::integral_constant<int, 0x124>{}));
  v = f(v, from(v, std::integral_constant<int, 0x122>{}));
  return f(v, from(v, std::integral_constant<int, 0x121>{}));
}

typedef short v4i16 __attribute__((ext_vector_type(4)));

// LDS tiles (K and V, 64 cache rows each) are unpadded rows of D x 2 bytes, CPR 16-byte chunks,
// filled by direct-to-LDS loads. Spreading over the banks comes from swizzles of the chunk index:
// chunk c of slot s holds logical chunk c ^ swz(s).
//  - K: swz_k(s) = s % CPR. The 16 lanes of one lane group read one logical chunk of 16
//    consecutive slots for an S^T operand (16-byte reads): 16 distinct physical chunks.
//  - V: swz_v(s) = 2 (s % 4) + 8 ((s / 8) % 2) (CPR = 16; 2 (s % 4) for CPR = 8). A transposing
//    read of a lane group covers 4 consecutive slots x 2 adjacent chunks x 2 halves; the swizzle
//    puts them, and the next lane group's 4 slots 8 rows on, on distinct 8-byte bank ranges.
//  - K slot s of a 32-row block holds cache row kslot_row(s): slot 16 t + 4 a + b <- row
//    8 a + 4 t + b, so the 16 slots one S^T operand reads give each lane 8 consecutive rows of
//    the output (the rows its P^T operand pairs with V). V slots hold rows in order.
// Without the swizzles the kernel takes 0.405 ms instead of 0.220 ms on the 2976-row case.
template <int CPR>
__device__ __forceinline__ int swz_k(int s) { return s % CPR; }
template <int CPR>
__device__ __forceinline__ int swz_v(int s) { return CPR >= 16 ? 2 * (s % 4) + 8 * ((s / 8) % 2) : 2 * (s % 4); }
__device__ __forceinline__ int kslot_row(int s) {
  const int k = s & 31;
  return (s & ~31) + 8 * ((k >> 2) & 3) + 4 * (k >> 4) + (k & 3);
}

// The A operand of O^T = V^T P^T for columns 16 dt .. + 16 of 32 V rows at vb (swizzled, row-major),
// through transposing 64-bit LDS loads: in each 16-lane group, lane m names row 4 h + m / 4 (of the
// group's 8 keys 8 g ..) at column 4 (m % 4) of the 16-column tile, and lane 4a + b receives column
// 4a + b of rows 4h + 0..3. So lane (g, lm) holds V[8 g + 4 h + e][16 dt + lm], e = 0..3: two loads
// (h = 0, 1) give the eight keys 8 g + e' the B operand (P^T) pairs with that lane. Element
// 16 dt + 4 (lm % 4) is logical chunk 2 dt + (lm % 4) / 2, byte 8 (lm % 2).
template <int CPR>
__device__ __forceinline__ bf16x8 v_operand(const char* vb, int dt, int g, int lm) {
  typedef __attribute__((address_space(3))) v4i16 lds_v4i16;
  auto rd = [&](int h) {
    const int row = 8 * g + 4 * h + lm / 4;
    return row * CPR * 16 + (((2 * dt + (lm % 4) / 2) ^ swz_v<CPR>(row)) * 16) + 8 * (lm % 2);
  };
  const v4i16 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4i16*)(vb + rd(0)));
  const v4i16 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4i16*)(vb + rd(1)));
  return __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
}

// x / d for d > 0, with inv = inverse_of(.., d).
__device__ __forceinline__ int div_by(int x, int d, uint32_t inv) {
  return inv != 0 ? (int)__umulhi((uint32_t)x, inv) : d == 1 ? x : x / d;
}
__device__ __forceinline__ bool attn_work_item(int nqb, int group, int xpk_log, int items, uint32_t inv_group,
                                               uint32_t inv_nqb, int& qb, int& h, int& z) {
  const int L = (int)blockIdx.x, xcd = L % kXcds;
  const int j = ((L / kXcds) << xpk_log) + (xcd & ((1 << xpk_log) - 1));
  const int rest = div_by(j, group, inv_group);
  h = (xcd >> xpk_log) * group + (j - rest * group);
  z = div_by(rest, nqb, inv_nqb);
  qb = nqb - 1 - (rest - z * nqb);
  return j < items;
}

// SPLIT: split z of the cache's tiles per workgroup, unnormalised rows with their max and sum to ws.
template <int D, bool SPLIT>
__global__ __launch_bounds__(kAttnWaves * 64) void attn_active_kernel(
    int nqb, int map_group, int xpk_log, int items, uint32_t inv_group, uint32_t inv_nqb,
    const int64_t* __restrict__ pos, int n, int N, const char* __restrict__ kc, const char* __restrict__ vc,
    int64_t kv_hs_b, const char* __restrict__ q, int64_t q_hs_b, int64_t q_ts_b, int Hq, int group, float scale_log2,
    char* __restrict__ out, int32_t* __restrict__ err, float* __restrict__ ws, int split_tiles) {
  constexpr int DS = D / 32;          // k-steps of S^T = K Q^T
  constexpr int DT = D / 16;          // 16-row tiles of O^T
  constexpr int CPR = D / 8;          // 16-byte chunks per cache row
  constexpr int ROWB = D * 2;        // bytes per cache row (and LDS slot)
  constexpr int NT = kAttnWaves * 64;
  static_assert(D % 32 == 0, "head_dim must be a multiple of 32");
  static_assert((kAttnBN * CPR) % NT == 0, "tile loads must tile the workgroup");
  static_assert((CPR & (CPR - 1)) == 0 && CPR >= 8, "swizzles need a power-of-two chunk count");

  // Two buffers per tensor: tile t + 1 loads into one while tile t is read from the other.
  __shared__ __attribute__((aligned(1024))) char k_lds0[kAttnBN * ROWB];
  __shared__ __attribute__((aligned(1024))) char k_lds1[kAttnBN * ROWB];
  __shared__ __attribute__((aligned(1024))) char v_lds0[kAttnBN * ROWB];
  __shared__ __attribute__((aligned(1024))) char v_lds1[kAttnBN * ROWB];
  __shared__ int blk_max_s[kAttnWaves];

  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64), lane = threadIdx.x % 64;
  const int g = lane / 16, lm = lane % 16;
  int qb, hq, z;
  if (!attn_work_item(nqb, map_group, xpk_log, items, inv_group, inv_nqb, qb, hq, z)) return;
  const int hk = hq / group;
  const int q0 = qb * kAttnBM + wave * kAttnQG * 16;
  // Positions of this lane's queries (-1 = no query); out-of-range positions are flagged and
  // clamped so that every read stays inside the cache.
  int my_pos[kAttnQG];
  int wmax = -1, wmin = N;
#pragma unroll
  for (int qg = 0; qg < kAttnQG; ++qg) {
    const int m = q0 + qg * 16 + lm;
    int p = -1;
    if (m < n) {
      const int64_t p64 = pos[m];
      if (p64 < 0 || p64 >= N) {
        flag_error(err, CKV_DEVICE_ERR_RANGE);
        p = p64 < 0 ? 0 : N - 1;
      } else {
        p = (int)p64;
      }
      wmin = min(wmin, p);
    }
    my_pos[qg] = p;
    wmax = max(wmax, p);
  }
  wmax = __builtin_amdgcn_readfirstlane(row16_reduce(wmax, [](int a, int b) { return max(a, b); }));
  wmin = __builtin_amdgcn_readfirstlane(row16_reduce(wmin, [](int a, int b) { return min(a, b); }));
  if (lane == 0) blk_max_s[wave] = wmax;
  __syncthreads();
  int bmax = blk_max_s[0];
#pragma unroll
  for (int w = 1; w < kAttnWaves; ++w) bmax = max(bmax, blk_max_s[w]);
  bmax = __builtin_amdgcn_readfirstlane(bmax);
  int n_tiles = bmax < 0 ? 0 : bmax / kAttnBN + 1;
  const int tile_begin = SPLIT ? z * split_tiles : 0;
  if (SPLIT) n_tiles = min(n_tiles, tile_begin + split_tiles);

  // Q fragments (B operand of S^T): query q0 + 16 qg + lm, head-dim 32 s + 8 g .. + 8.
  bf16x8 qf[kAttnQG][DS];
#pragma unroll
  for (int qg = 0; qg < kAttnQG; ++qg) {
    const int m = q0 + qg * 16 + lm;
#pragma unroll
    for (int s = 0; s < DS; ++s) {
      vec16 v = {0, 0, 0, 0};
      if (m < n) v = ld16(q + (int64_t)hq * q_hs_b + (int64_t)m * q_ts_b + (32 * s + 8 * g) * 2);
      qf[qg][s] = __builtin_bit_cast(bf16x8, v);
    }
  }

  f32x4 o[kAttnQG][DT];
  float m_run[kAttnQG], m_sub[kAttnQG];
  // The row sums come from one more MFMA per key block with an all-ones A operand: every row of its output is sum_k P^T[k][query], the sum of the bf16 weights that
  // multiply V (lane (g, lm) gets query lm's sum in each of its four values).
  f32x4 l_acc[kAttnQG];
  const bf16x8 ones = {(__bf16)1.f, (__bf16)1.f, (__bf16)1.f, (__bf16)1.f,
                       (__bf16)1.f, (__bf16)1.f, (__bf16)1.f, (__bf16)1.f};
#pragma unroll
  for (int qg = 0; qg < kAttnQG; ++qg) {
    m_run[qg] = -INFINITY;
    m_sub[qg] = 0.f;
    l_acc[qg] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) o[qg][dt] = f32x4{0.f, 0.f, 0.f, 0.f};
  }

  const char* kh = kc + (int64_t)hk * kv_hs_b;
  const char* vh = vc + (int64_t)hk * kv_hs_b;

  // Tile loads go straight from global memory to LDS (global_load_lds_dwordx4): load
  // instruction i of wavefront w fills the 1 KB block w * KI + i of a tile buffer, lane l its 16
  // bytes at l * 16, i.e. position P = (w KI + i) 64 + l = slot P / CPR, chunk P % CPR. No
  // registers stage the tile and no LDS store instructions run; rows past every query's position
  // load the last one's row instead: they are masked, but their zero weights meet the values, and a
  // cache row not written yet may hold a NaN (nor is there a row past the cache to read).
  constexpr int KI = (kAttnBN * CPR) / NT;  // load instructions per wavefront, tile and tensor
  static_assert(KI >= 1 && (kAttnBN * CPR) % NT == 0, "a tile must fill whole load instructions");
  // A lane's offsets in a tile are kept (K slots hold rows in kslot_row's order) and added to the
  // tile's uniform address: two 64-bit addresses built per load were a quarter of a tile's vector
  // instructions. Only a workgroup's last tile clamps its rows.
  int off_k[KI], off_v[KI];
#pragma unroll
  for (int i = 0; i < KI; ++i) {
    const int P = (wave * KI + i) * 64 + lane;
    const int slot = P / CPR, pc = P % CPR;
    off_k[i] = kslot_row(slot) * ROWB + (pc ^ swz_k<CPR>(slot)) * 16;
    off_v[i] = slot * ROWB + (pc ^ swz_v<CPR>(slot)) * 16;
  }
  typedef __attribute__((address_space(1))) void gvoid;
  typedef __attribute__((address_space(3))) void lvoid;
  auto issue = [&](int n0, char* kb, char* vb) {
    const char* kt = kh + (int64_t)n0 * ROWB;
    const char* vt = vh + (int64_t)n0 * ROWB;
    const int last = bmax - n0;  // >= 0: only tiles that some query sees are issued
    auto load = [&](const char* t, int off, char* to) {
      __builtin_amdgcn_global_load_lds((gvoid*)(t + (uint32_t)off), (lvoid*)to, 16, 0, 0);
    };
    if (last >= kAttnBN - 1) {  // uniform: a whole tile
#pragma unroll
      for (int i = 0; i < KI; ++i) {
        load(kt, off_k[i], kb + (wave * KI + i) * 1024);
        load(vt, off_v[i], vb + (wave * KI + i) * 1024);
      }
    } else {
      auto clamp = [&](int off) { return min(off / ROWB, last) * ROWB + off % ROWB; };
#pragma unroll
      for (int i = 0; i < KI; ++i) {
        load(kt, clamp(off_k[i]), kb + (wave * KI + i) * 1024);
        load(vt, clamp(off_v[i]), vb + (wave * KI + i) * 1024);
      }
    }
  };
  // S^T operand of (kb, t, ds) for lane (g, lm): slot 32 kb + 16 t + lm, logical chunk 4 ds + g.
  int k_rd[DS];
#pragma unroll
  for (int ds = 0; ds < DS; ++ds) k_rd[ds] = lm * ROWB + (((4 * ds + g) ^ swz_k<CPR>(lm)) * 16);
  if (tile_begin < n_tiles) issue(tile_begin * kAttnBN, k_lds0, v_lds0);

  // One tile; the loop below alternates the buffers (each call names its buffers directly, so
  // the compiler sees that the loads in flight never alias the buffer being read).
  auto body = [&](int tile, const char* k_lds, const char* v_lds, char* k_nxt, char* v_nxt) {
    const int n0 = tile * kAttnBN;
    __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): this wavefront's loads of the tile landed
    __syncthreads();  // every wavefront's loads landed and every wavefront is done with the other buffer
    if (tile + 1 < n_tiles) issue(n0 + kAttnBN, k_nxt, v_nxt);  // lands during the MFMAs below

    if (n0 > wmax) return;  // uniform per wavefront: no query of this wavefront reaches the tile
    const bool need_mask = n0 + kAttnBN - 1 > wmin;

    // S^T for the tile: lane (g, lm) gets query lm, rows n0 + 32 kb + 8 g + 4 t + e.
    constexpr int KB = kAttnBN / 32;
    f32x4 s[kAttnQG][KB][2];
#pragma unroll
    for (int kb = 0; kb < KB; ++kb)
#pragma unroll
      for (int ds = 0; ds < DS; ++ds) {  // the halves inside: dependent products four apart
#pragma unroll
        for (int t = 0; t < 2; ++t) {
          const bf16x8 a = *(const bf16x8*)(k_lds + (kb * 32 + 16 * t) * ROWB + k_rd[ds]);
#pragma unroll
          for (int qg = 0; qg < kAttnQG; ++qg)
            s[qg][kb][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, qf[qg][ds], ds == 0 ? f32x4{0.f, 0.f, 0.f, 0.f}
                                                                                       : s[qg][kb][t], 0, 0, 0);
        }
      }

    // Online softmax over the tile. The running max is only raised when a query's tile max
    // exceeds it by more than 2^8 (log2 domain): weights stay <= 256, the output rescale is
    // skipped for the whole wavefront otherwise, and the result is unchanged (the final division
    // uses the same max).
    bf16x8 pb[kAttnQG][KB];
#pragma unroll
    for (int qg = 0; qg < kAttnQG; ++qg) {
      // Raw scores of this lane (query lm, rows n0 + 32 kb + 8 g + 4 t + e); rows past the query's
      // position become -inf, on the tiles that reach past the lowest position only (uniform).
      float x[KB][8];
#pragma unroll
      for (int kb = 0; kb < KB; ++kb)
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
          for (int e = 0; e < 4; ++e) x[kb][4 * t + e] = s[qg][kb][t][e];
      if (need_mask) {
        const int lim = my_pos[qg] - n0 - 8 * g;  // row offset 32 kb + 4 t + e must stay <= lim
#pragma unroll
        for (int kb = 0; kb < KB; ++kb)
#pragma unroll
          for (int j = 0; j < 8; ++j)
            if (32 * kb + j > lim) x[kb][j] = -INFINITY;
      }
      float bm = -INFINITY;
#pragma unroll
      for (int kb = 0; kb < KB; ++kb)
#pragma unroll
        for (int j = 0; j < 8; ++j) bm = fmaxf(bm, x[kb][j]);
      // A lane asks for its own scores; the four lanes of a query agree on its max inside the branch.
      if (__builtin_amdgcn_ballot_w64(bm * scale_log2 > m_run[qg] + 8.f)) {  // uniform branch
        bm = group_max(bm) * scale_log2;           // the scale is > 0: max commutes
        const bool raise = bm > m_run[qg] + 8.f;  // also true on the first visible tile (m_run = -inf)
        const float m_new = raise ? bm : m_run[qg];
        const float alpha = m_run[qg] == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m_run[qg] - m_new);
        l_acc[qg] *= alpha;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) o[qg][dt] *= alpha;
        m_run[qg] = m_new;
        // with no visible row yet (absent queries) every score is -inf and subtracting 0 keeps p = 0
        m_sub[qg] = m_new == -INFINITY ? 0.f : m_new;
      }
      // p = 2^(score * scale - max) in one fma
#pragma unroll
      for (int kb = 0; kb < KB; ++kb)
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          pb[qg][kb][e] = (__bf16)__builtin_amdgcn_exp2f(__builtin_fmaf(x[kb][e], scale_log2, -m_sub[qg]));
        }
    }

    // O^T += V^T P^T: A = V^T rows dt*16 + lm, columns 32 kb + 8 g .. + 8.
#pragma unroll
    for (int kb = 0; kb < KB; ++kb)
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) {
        const bf16x8 a = v_operand<CPR>(v_lds + kb * 32 * ROWB, dt, g, lm);
#pragma unroll
        for (int qg = 0; qg < kAttnQG; ++qg)
          o[qg][dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, pb[qg][kb], o[qg][dt], 0, 0, 0);
        if (dt == DT - 1) {
#pragma unroll
          for (int qg = 0; qg < kAttnQG; ++qg)
            l_acc[qg] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ones, pb[qg][kb], l_acc[qg], 0, 0, 0);
        }
      }
  };
  for (int tile = tile_begin; tile < n_tiles; tile += 2) {
    body(tile, k_lds0, v_lds0, k_lds1, v_lds1);
    if (tile + 1 < n_tiles) body(tile + 1, k_lds1, v_lds1, k_lds0, v_lds0);
  }

  // Normalise and write: lane (g, lm) holds O[query][dt*16 + 4g + e], 4 bf16 = 8 bytes per tile.
#pragma unroll
  for (int qg = 0; qg < kAttnQG; ++qg) {
    const float l = l_acc[qg][0];
    const int m = q0 + qg * 16 + lm;
    if (m >= n) continue;
    if (SPLIT) {
      float* prow = ws + (((int64_t)z * Hq + hq) * n + m) * (D + 4);  // 16-byte aligned rows
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) *(f32x4*)(prow + dt * 16 + 4 * g) = o[qg][dt];
      if (g == 0) {
        prow[D] = m_run[qg];
        prow[D + 1] = l;
      }
      continue;
    }
    const float inv = 1.f / l;
    char* orow = out + ((int64_t)m * Hq + hq) * (D * 2);
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) {
      unsigned w[2];
#pragma unroll
      for (int h = 0; h < 2; ++h) w[h] = f32x2_to_bf16x2_bits(o[qg][dt][2 * h] * inv, o[qg][dt][2 * h + 1] * inv);
      *(uint2*)(orow + (dt * 16 + 4 * g) * 2) = uint2{w[0], w[1]};
    }
  }
}

}  // namespace ckv

#include "attention_wave.hpp"

extern "C" int64_t ckv_attention_workspace_bytes(int32_t n_queries, int32_t n_tokens, int32_t n_q_heads,
                                                 int32_t head_dim, int32_t* splits_out, int32_t* split_tiles_out) {
  using namespace ckv;
  const bool some = n_queries > 0 && n_tokens > 0 && n_q_heads > 0 && head_dim > 0;
  const int64_t splits = some ? attn_most_splits(n_queries, n_tokens, n_q_heads, head_dim) : 1;
  const int tiles = n_tokens > 0 ? (n_tokens + kAttnBN - 1) / kAttnBN : 0;
  if (splits_out != nullptr) *splits_out = (int32_t)splits;
  if (split_tiles_out != nullptr) *split_tiles_out = splits > 1 ? (int32_t)((tiles + splits - 1) / splits) : 0;
  return some ? attn_workspace_bytes(n_queries, n_tokens, n_q_heads, head_dim) : 0;
}

extern "C" int32_t ckv_attention_active(void* out, const void* q, int64_t q_head_stride, int64_t q_token_stride,
                                        const void* k_cache, const void* v_cache, int64_t kv_head_stride,
                                        const int64_t* positions, int32_t n_queries, int32_t n_tokens,
                                        int32_t n_q_heads, int32_t n_kv_heads, int32_t head_dim, int32_t dtype,
                                        double scale, void* workspace, int64_t workspace_bytes, int32_t* err,
                                        void* stream) {
  using namespace ckv;
  if (out == nullptr || q == nullptr || k_cache == nullptr || v_cache == nullptr || positions == nullptr)
    return CKV_ERR_INVALID_ARGUMENT;
  if (dtype != CKV_DTYPE_BF16 || (head_dim != 64 && head_dim != 128)) return CKV_ERR_INVALID_ARGUMENT;
  if (n_queries < 0 || n_tokens <= 0 || n_q_heads <= 0 || n_kv_heads <= 0 || n_q_heads % n_kv_heads != 0 ||
      !(scale > 0.0))
    return CKV_ERR_INVALID_ARGUMENT;
  if (q_token_stride % 8 || q_head_stride % 8 || kv_head_stride % 8) return CKV_ERR_INVALID_ARGUMENT;  // 16-byte rows
  if (((uintptr_t)out | (uintptr_t)q | (uintptr_t)k_cache | (uintptr_t)v_cache) % 16) return CKV_ERR_INVALID_ARGUMENT;
  if (q_token_stride < head_dim || kv_head_stride < (int64_t)n_tokens * head_dim) return CKV_ERR_OUT_OF_RANGE;
  if (n_queries == 0) return CKV_OK;
  if (n_q_heads > 65535) return CKV_ERR_TOO_LARGE;
  const float scale_log2 = (float)(scale * 1.4426950408889634);  // exp(x) = exp2(x log2 e)
  const int group = n_q_heads / n_kv_heads;
  hipStream_t st = (hipStream_t)stream;
  const AttnPlan plan = attn_plan(n_queries, n_tokens, n_q_heads, n_kv_heads, head_dim,
                                  workspace != nullptr && (uintptr_t)workspace % 16 == 0 ? workspace_bytes : 0);
  const AttnMap& map = plan.map;
  float* ws = plan.splits > 1 ? (float*)workspace : nullptr;
  if (plan.wave) {
    const uint32_t inv_gqa = inverse_of((int64_t)n_queries * group, group);
    auto launch = [&](auto kernel, int waves) {
      hipLaunchKernelGGL(kernel, dim3(map.blocks), dim3(waves * 64), 0, st, map.nqb, map.group, map.xpk_log, map.items,
                         map.inv_group, map.inv_nqb, positions, n_queries, n_tokens, (const char*)k_cache,
                         (const char*)v_cache, kv_head_stride * 2, (const char*)q, q_head_stride * 2, q_token_stride * 2,
                         n_q_heads, group, inv_gqa, scale_log2, plan.split_chunks, (char*)out, ws, err);
    };
#define CKV_WAVE(HD, QG, W, GR) \
  else if (head_dim == HD && plan.qg == QG && plan.waves == W && plan.grouped == GR) \
    launch(attn_wave_kernel<HD, QG, W, GR>, W);
    if (false) {
    }
    CKV_WAVE_FORMS(CKV_WAVE)
    else return CKV_ERR_INVALID_ARGUMENT;  // a plan outside the list
#undef CKV_WAVE
  } else {
    auto launch = [&](auto kernel) {
      hipLaunchKernelGGL(kernel, dim3(map.blocks), dim3(kAttnWaves * 64), 0, st, map.nqb, map.group, map.xpk_log, map.items,
                         map.inv_group, map.inv_nqb, positions, n_queries, n_tokens, (const char*)k_cache,
                         (const char*)v_cache, kv_head_stride * 2, (const char*)q, q_head_stride * 2, q_token_stride * 2,
                         n_q_heads, group, scale_log2, (char*)out, err, ws, plan.split_chunks / (kAttnBN / kWaveChunk));
    };
    if (head_dim == 128) ws != nullptr ? launch(attn_active_kernel<128, true>) : launch(attn_active_kernel<128, false>);
    else ws != nullptr ? launch(attn_active_kernel<64, true>) : launch(attn_active_kernel<64, false>);
  }
  CKV_RETURN_IF_LAUNCH_FAILED();
  if (ws != nullptr) {
    const dim3 grid((unsigned)n_queries, (unsigned)n_q_heads);
    const dim3 block(64 * (unsigned)std::min((plan.splits + kCombineParts - 1) / kCombineParts, kCombineMaxWaves));
    auto merge = [&](auto kernel) { hipLaunchKernelGGL(kernel, grid, block, 0, st, (char*)out, ws, n_queries, n_q_heads, plan.splits); };
    if (head_dim == 128) merge(attn_combine_kernel<128>);
    else merge(attn_combine_kernel<64>);
    CKV_RETURN_IF_LAUNCH_FAILED();
  }
  return CKV_OK;
}

// The model's projections at short requests: out = x W^T + bias in bf16 with fp32 accumulation, the
// function of torch.nn.functional.linear, which the engine keeps for everything larger.
//
// Reference semantics: the decoder's q/k/v/o and MLP projections (torch_engine.py:61-72), nn.Linear
// modules. Products accumulate in fp32, the bias is added in fp32, one rounding to bf16 at the end,
// as the libraries do.
//
// Bound: latency on both sides. At a 1.1k-token request of the 0.5B shape a projection of the kept
// rows is 0.5-4.4 GFLOP: the library's call takes about 20 us of host time (its heuristic runs on
// every call, this one 4) and its kernels 7-13 us, so the host is what the request waits for. Here
// a workgroup of four wavefronts takes a 64 x 64 tile, both operands run along K (x rows and W
// rows), so every load is whole 128-byte pieces of rows and every matrix operand a 16-byte LDS
// read. Rows are staged through registers four steps of 64 ahead into two LDS buffers (one barrier
// per step, which waits for no load); K is split over the grid where the tiles leave CUs idle, the
// fp32 partials summed in order by a second launch.
// Measured (us, graph replays, 251 rows, the library beside it): 1152 x 896 6.9 and 7.9, 896 x 896
// 6.6 and 7.1, 9728 x 896 13.9 and 12.8, 896 x 4864 11.4 and 11.9. 128 x 128 tiles won nowhere in
// the range that ckv_linear is for (9728 x 896 13.7).
#include <algorithm>

#include "ckv_common.hpp"

namespace ckv {

typedef __bf16 lin_bf16x8 __attribute__((ext_vector_type(8)));
typedef float lin_f32x4 __attribute__((ext_vector_type(4)));

constexpr int kLinThreads = 256;
constexpr int kLinTile = 64;  // rows of x and of W per workgroup
constexpr int kLinBK = 64;    // K per step: 128 bytes of a row, eight 16-byte pieces
constexpr int kLinAhead = 4;  // steps whose loads are in flight

// Piece c of row r of a staged tile sits at piece c ^ ((r / 2) % 8) of the row: the 16 rows one
// operand reads at one piece then cover all 64 banks.
__device__ __forceinline__ int lin_at(int r, int c) { return r * 128 + ((c ^ ((r >> 1) & 7)) << 4); }

// Barrier for LDS only: global loads in flight stay in flight.
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// Tile (tm, tn) of split z. The workgroups of one W tile (all row tiles of x) run on one XCD, one
// after the other: workgroup L of the grid goes to XCD L % 8, column tiles are dealt to the XCDs.
__global__ __launch_bounds__(kLinThreads) void linear_kernel(const char* __restrict__ x, int64_t x_rs_b,
                                                             const char* __restrict__ w, int M, int N, int K, int mt,
                                                             int nt, int steps, const char* __restrict__ bias,
                                                             char* __restrict__ out, float* __restrict__ part) {
  constexpr int BM = kLinTile, BN = kLinTile, kAhead = kLinAhead;
  constexpr int WM = BM / 2, WN = BN / 2;        // a wavefront's share of the tile
  constexpr int TM = WM / 16, TN = WN / 16;      // in 16 x 16 matrix tiles
  static_assert(kAhead % 2 == 0, "a step's LDS buffer is its parity in the group");
  constexpr int LA = BM * 8 / kLinThreads, LB = BN * 8 / kLinThreads;  // 16-byte pieces per thread and step
  __shared__ __attribute__((aligned(1024))) char lds[2][(BM + BN) * 128];
  const int L = (int)blockIdx.x, per = L >> 3;
  const int tn = (per / mt) * 8 + (L & 7), tm = per % mt, z = (int)blockIdx.y;
  if (tn >= nt) return;
  const int m0 = tm * BM, n0 = tn * BN;
  const int tid = threadIdx.x, wave = tid / 64, lane = tid % 64, g = lane / 16, lm = lane % 16;
  const int wm = (wave & 1) * WM, wn = (wave >> 1) * WN;
  const int k_begin = z * steps, k_end = min(K / kLinBK, k_begin + steps);

  // Thread t stages piece t % 8 of rows t / 8, t / 8 + 32, ...; rows past the end repeat the last.
  const char* pa[LA];
  const char* pb[LB];
  int at_a[LA], at_b[LB];
#pragma unroll
  for (int i = 0; i < LA; ++i) {
    const int r = tid / 8 + i * 32;
    pa[i] = x + (int64_t)min(m0 + r, M - 1) * x_rs_b + (tid % 8) * 16;
    at_a[i] = lin_at(r, tid % 8);
  }
#pragma unroll
  for (int i = 0; i < LB; ++i) {
    const int r = tid / 8 + i * 32;
    pb[i] = w + (int64_t)min(n0 + r, N - 1) * ((int64_t)K * 2) + (tid % 8) * 16;
    at_b[i] = BM * 128 + lin_at(r, tid % 8);
  }
  vec16 ra[kAhead][LA], rb[kAhead][LB];
  auto load = [&](int k, vec16(&a)[LA], vec16(&b)[LB]) {
    k = min(k, k_end - 1);  // past the end: the last step again, not used
#pragma unroll
    for (int i = 0; i < LB; ++i) b[i] = ld16(pb[i] + (int64_t)k * 128);
#pragma unroll
    for (int i = 0; i < LA; ++i) a[i] = ld16(pa[i] + (int64_t)k * 128);
  };
  auto stage = [&](char* to, const vec16(&a)[LA], const vec16(&b)[LB]) {
#pragma unroll
    for (int i = 0; i < LB; ++i) *(vec16*)(to + at_b[i]) = b[i];
#pragma unroll
    for (int i = 0; i < LA; ++i) *(vec16*)(to + at_a[i]) = a[i];
  };
  lin_f32x4 acc[TN][TM];  // lane (g, lm): columns 16 j + 4 g + e of row 16 i + lm
#pragma unroll
  for (int j = 0; j < TN; ++j)
#pragma unroll
    for (int i = 0; i < TM; ++i) acc[j][i] = lin_f32x4{0.f, 0.f, 0.f, 0.f};

#pragma unroll
  for (int s = 0; s < kAhead; ++s) {
    load(k_begin + s, ra[s], rb[s]);
    __builtin_amdgcn_sched_barrier(0);  // in this order, as the loop issues them: its waits count on it
  }
  // No branch leaves a group of kAhead steps (the compiler would wait for every load in flight
  // where the paths meet): the steps past the end are staged again and not used.
  for (int k = k_begin; k < k_end; k += kAhead) {
#pragma unroll
    for (int s = 0; s < kAhead; ++s) {
      char* buf = lds[s & 1];
      stage(buf, ra[s], rb[s]);
      lds_barrier();  // the step is in LDS; every wavefront is done with the other buffer's last step
      load(k + s + kAhead, ra[s], rb[s]);
      if (k + s < k_end) {  // uniform
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
          lin_bf16x8 fa[TM], fb[TN];
#pragma unroll
          for (int j = 0; j < TN; ++j) fb[j] = *(const lin_bf16x8*)(buf + BM * 128 + lin_at(wn + 16 * j + lm, 4 * ks + g));
#pragma unroll
          for (int i = 0; i < TM; ++i) fa[i] = *(const lin_bf16x8*)(buf + lin_at(wm + 16 * i + lm, 4 * ks + g));
#pragma unroll
          for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int i = 0; i < TM; ++i) acc[j][i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fb[j], fa[i], acc[j][i], 0, 0, 0);
        }
      }
    }
  }
#pragma unroll
  for (int j = 0; j < TN; ++j) {
    const int n = n0 + wn + 16 * j + 4 * g;
    if (n >= N) continue;  // N is a multiple of 8
    float b[4] = {0.f, 0.f, 0.f, 0.f};
    if (part == nullptr && bias != nullptr) {
      const uint2 v = *(const uint2*)(bias + (int64_t)n * 2);
      b[0] = bf16_bits_to_f32(v.x & 0xffffu);
      b[1] = bf16_bits_to_f32(v.x >> 16);
      b[2] = bf16_bits_to_f32(v.y & 0xffffu);
      b[3] = bf16_bits_to_f32(v.y >> 16);
    }
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      const int m = m0 + wm + 16 * i + lm;
      if (m >= M) continue;
      const lin_f32x4 v = acc[j][i];
      if (part != nullptr) {
        *(lin_f32x4*)(part + ((int64_t)z * M + m) * N + n) = v;
      } else {
        *(uint2*)(out + ((int64_t)m * N + n) * 2) =
            uint2{f32x2_to_bf16x2_bits(v[0] + b[0], v[1] + b[1]), f32x2_to_bf16x2_bits(v[2] + b[2], v[3] + b[3])};
      }
    }
  }
}

// out = the sum of `splits` partials in order, plus the bias: eight columns a thread.
template <int SPLITS>
__global__ __launch_bounds__(kLinThreads) void linear_sum_kernel(const float* __restrict__ part, int splits, int64_t mn,
                                                                 int N, const char* __restrict__ bias,
                                                                 char* __restrict__ out) {
  const int64_t e = ((int64_t)blockIdx.x * kLinThreads + threadIdx.x) * 8;
  if (e >= mn) return;
  lin_f32x4 a[SPLITS], b[SPLITS];
#pragma unroll
  for (int z = 0; z < SPLITS; ++z) {  // all in flight; past the last split the last one again
    const float* p = part + (int64_t)min(z, splits - 1) * mn + e;
    a[z] = *(const lin_f32x4*)p;
    b[z] = *(const lin_f32x4*)(p + 4);
  }
  float c[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  if (bias != nullptr) Elem<CKV_DTYPE_BF16>::unpack(ld16(bias + (e % N) * 2), c);
#pragma unroll
  for (int z = 1; z < SPLITS; ++z)
    if (z < splits) {
      a[0] += a[z];
      b[0] += b[z];
    }
  float o[8];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    o[i] = a[0][i] + c[i];
    o[4 + i] = b[0][i] + c[4 + i];
  }
  st16(out + e * 2, Elem<CKV_DTYPE_BF16>::pack(o));
}

// The splits of K and the steps of each. A split keeps eight steps (two groups in flight) and is
// worth its second launch only where the tiles fill less than three quarters of the CUs: 251 rows,
// 896 x 4864 (56 tiles) 11.4 us in four and 15.4 in two, 1152 x 896 (72 tiles, 14 steps) 6.9 whole
// and 7.7 in two.
struct LinPlan {
  int splits = 1, steps = 0;
};
constexpr int kLinMaxSplits = 8;

static LinPlan linear_plan(int64_t M, int64_t N, int64_t K, int64_t workspace_bytes) {
  LinPlan p;
  const int64_t total = K / kLinBK, tiles = ((M + kLinTile - 1) / kLinTile) * ((N + kLinTile - 1) / kLinTile);
  int64_t splits = tiles < 192 ? std::min<int64_t>(256 / tiles, total / 8) : 1;
  splits = std::max<int64_t>(1, std::min<int64_t>({splits, (int64_t)kLinMaxSplits, workspace_bytes / (M * N * 4)}));
  p.steps = (int)((total + splits - 1) / splits);
  p.splits = (int)((total + p.steps - 1) / p.steps);
  return p;
}

// Where calls issued one after the other gain from this: not for one row (decode replays a graph, so
// the host does not count, and the library's one-row kernels are faster: 1152 x 896 4.2 us against
// 6.2), and up to 5 GFLOP, about where the library's kernels take as long as its host call (1103 rows
// of 9728 x 896, 19 GFLOP: 24.6 us against 32). It is the host time that this bounds, 4 us a call
// against 20; the kernels alone (us, this first, graph replays over weights as a model reads them,
// without the committed GEMM table): 7B shapes, 2-32 rows, q|k|v 10.4-11.4 and 12.5-13.3, o 9.3-10.2 and
// 12.0, down 27-30.5 and 46-110, gate|up (to 16 rows) 54-56 and 54-55; 0.5B shapes, 2-24 rows, q|k|v
// and o 6.2-6.5 and 5.6, gate|up 7.0 and 8.7, down 7.2-7.9 and 12.8; 1103 rows of q|k|v and o 10.3 and
// 9.0, 251 of gate|up 17.8 and 15.1. By kernel time alone the lines would lie elsewhere (64 rows of
// 3584 x 18944, left to the library, take it 85.8 us and this 28.9).
constexpr int64_t kLinMaxWork = 2500000000;  // n_rows * n_out * n_in

}  // namespace ckv

extern "C" int64_t ckv_linear_workspace_bytes(int32_t n_rows, int32_t n_out, int32_t n_in) {
  using namespace ckv;
  if (n_rows < 2 || n_out <= 0 || n_in <= 0 || n_out % 8 || n_in % kLinBK) return -1;
  if ((int64_t)n_rows * n_out > kLinMaxWork / n_in) return -1;
  const LinPlan p = linear_plan(n_rows, n_out, n_in, INT64_MAX);
  return p.splits > 1 ? (int64_t)p.splits * n_rows * n_out * 4 : 0;
}

extern "C" int32_t ckv_linear(void* out, const void* x, int64_t x_row_stride, const void* weight, const void* bias,
                              int32_t n_rows, int32_t n_out, int32_t n_in, int32_t dtype, void* workspace,
                              int64_t workspace_bytes, void* stream) {
  using namespace ckv;
  if (n_rows < 0 || n_out <= 0 || n_in <= 0 || dtype != CKV_DTYPE_BF16 || n_in % kLinBK || n_out % 8 || x_row_stride % 8)
    return CKV_ERR_INVALID_ARGUMENT;
  if (x_row_stride < n_in) return CKV_ERR_OUT_OF_RANGE;
  if (n_rows == 0) return CKV_OK;
  if (out == nullptr || x == nullptr || weight == nullptr) return CKV_ERR_INVALID_ARGUMENT;
  if (((uintptr_t)out | (uintptr_t)x | (uintptr_t)weight | (uintptr_t)bias) % 16) return CKV_ERR_INVALID_ARGUMENT;
  const bool ws_ok = workspace != nullptr && (uintptr_t)workspace % 16 == 0;
  const LinPlan p = linear_plan(n_rows, n_out, n_in, ws_ok ? workspace_bytes : 0);
  hipStream_t st = (hipStream_t)stream;
  float* part = p.splits > 1 ? (float*)workspace : nullptr;
  const int64_t mt = ((int64_t)n_rows + kLinTile - 1) / kLinTile, nt = ((int64_t)n_out + kLinTile - 1) / kLinTile;
  const int64_t blocks = mt * ((nt + 7) / 8) * 8;
  if (blocks > 0xffffff) return CKV_ERR_TOO_LARGE;
  hipLaunchKernelGGL(linear_kernel, dim3((unsigned)blocks, (unsigned)p.splits), dim3(kLinThreads), 0, st, (const char*)x,
                     x_row_stride * 2, (const char*)weight, n_rows, n_out, n_in, (int)mt, (int)nt, p.steps,
                     (const char*)bias, (char*)out, part);
  CKV_RETURN_IF_LAUNCH_FAILED();
  if (part != nullptr) {
    const int64_t mn = (int64_t)n_rows * n_out;
    auto sum = [&](auto kernel) {
      hipLaunchKernelGGL(kernel, dim3((unsigned)((mn / 8 + kLinThreads - 1) / kLinThreads)), dim3(kLinThreads), 0, st,
                         part, p.splits, mn, n_out, (const char*)bias, (char*)out);
    };
    if (p.splits <= 2) sum(linear_sum_kernel<2>);
    else if (p.splits <= 4) sum(linear_sum_kernel<4>);
    else sum(linear_sum_kernel<kLinMaxSplits>);
    CKV_RETURN_IF_LAUNCH_FAILED();
  }
  return CKV_OK;
}

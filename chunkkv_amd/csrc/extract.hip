// Store-put extraction: copy token rows [start, start + len) of every layer's K and V out of the
// request's cache slabs into one new contiguous buffer per segment, for every reusable segment of
// the request in one launch.
//
// Reference semantics (src/chunkkv/engine/base.py:55-60): PrefillResult.chunk(start, end) builds
// a ChunkKV whose keys/values are `copy(k[:, :, start:end, :])` per layer, copy being
// `.contiguous()` for the torch engine (torch_engine.py:177); the runtime calls it once per
// reusable segment after every prefill (runtime.py:83-92), i.e. 2 x n_layers copy launches per
// segment. Here one launch moves all of them; the bytes are identical (a bit copy).
//
// Destination layout per segment s: [2][n_layers][H][len_s][D] (K layers, then V layers), so
// that layer l's keys (and values) are a contiguous (1, H, len_s, D) view.
//
// Design (gfx950): one workgroup = one (segment, 8-token tile, layer); 16-byte loads and
// stores; a thread walks (K/V, head, token, 16-byte column) items with the column fastest, so a
// wavefront reads and writes whole rows. Grid x = tile (fastest), y = segment, z = layer: the
// workgroups in flight together copy neighbouring tiles of one segment (159 -> 150 us for the
// 8k request's 24 segments x 28 layers against segment-fastest order with 16-token tiles).
#include "ckv_common.hpp"

namespace ckv {

constexpr int kExtractThreads = 256;
constexpr int kExtractTile = 8;

// Up to 64 segments by value (1 KB of kernel arguments): a table in device memory costs a pinned
// block and a copy in front of the launch, and each workgroup a dependent load of its span. The 8k
// request's whole call (24 segments x 320 tokens x 28 layers, calls back to back, both builds
// alternating, one line a card): 156.4-156.6 -> 149.2-149.4 us, 154.1 -> 146.3, 161.7 -> 155.8-156.7,
// 159.0 -> 154.8 (the last two within a few per cent of noise). 64 is a chosen size, not a measured
// edge: arguments hold about 250 segments (4 KB), and longer lists were not measured in this form.
constexpr int kExtractArgs = 64;
struct ExtractSpans {
  uint64_t dst[kExtractArgs];
  int32_t start[kExtractArgs], len[kExtractArgs];
};

__device__ __forceinline__ void extract_tile(const char* __restrict__ src_k, const char* __restrict__ src_v, int64_t ls_b,
                                             int64_t hs_b, int row_b, char* __restrict__ dst, int start, int len,
                                             int n_layers, int n_heads) {
  const int layer = blockIdx.z;
  const int t0 = blockIdx.x * kExtractTile;
  if (t0 >= len) return;  // uniform
  const int ntok = min(kExtractTile, len - t0);
  const int cpr = row_b / 16;
  const int items = 2 * n_heads * ntok * cpr;
  const int64_t head_b = (int64_t)len * row_b;  // one (head) block of the destination
  for (int i = threadIdx.x; i < items; i += kExtractThreads) {
    const int c = i % cpr;
    const int r = i / cpr;             // (kv, head, token) row
    const int tok = r % ntok;
    const int kh = r / ntok;           // kv * n_heads + head
    const int kv = kh / n_heads, h = kh % n_heads;
    const char* s = (kv ? src_v : src_k) + layer * ls_b + h * hs_b + (int64_t)(start + t0 + tok) * row_b + c * 16;
    char* d = dst + ((int64_t)(kv * n_layers + layer) * n_heads + h) * head_b + (int64_t)(t0 + tok) * row_b + c * 16;
    st16_stream(d, ld16_stream(s));
  }
}

__global__ __launch_bounds__(kExtractThreads) void extract_kernel(
    const char* __restrict__ src_k, const char* __restrict__ src_v, int64_t ls_b, int64_t hs_b, int row_b,
    const uint64_t* __restrict__ dst_tab, const int32_t* __restrict__ spans, int n_layers, int n_heads, int n_tokens,
    int32_t* __restrict__ err) {
  typedef __attribute__((address_space(1))) const int32_t gi32;
  const int seg = blockIdx.y;
  const int start = *(gi32*)(spans + 2 * seg), len = *(gi32*)(spans + 2 * seg + 1);
  if (start < 0 || len < 0 || (int64_t)start + len > n_tokens) {
    if (threadIdx.x == 0 && blockIdx.x == 0 && blockIdx.z == 0) flag_error(err, CKV_DEVICE_ERR_RANGE);
    return;
  }
  extract_tile(src_k, src_v, ls_b, hs_b, row_b, reinterpret_cast<char*>(dst_tab[seg]), start, len, n_layers, n_heads);
}

__global__ __launch_bounds__(kExtractThreads) void extract_args_kernel(
    const char* __restrict__ src_k, const char* __restrict__ src_v, int64_t ls_b, int64_t hs_b, int row_b, int n_layers,
    int n_heads, const ExtractSpans spans) {
  const int seg = blockIdx.y;
  extract_tile(src_k, src_v, ls_b, hs_b, row_b, reinterpret_cast<char*>(spans.dst[seg]), spans.start[seg],
               spans.len[seg], n_layers, n_heads);
}

// What both entry points check but for their tables.
static int32_t extract_check(const void* k_slab, const void* v_slab, int64_t layer_stride, int64_t head_stride,
                             int32_t n_spans, int32_t n_layers, int32_t n_heads, int32_t n_tokens, int32_t head_dim,
                             int32_t dtype, int64_t& eb) {
  if (k_slab == nullptr || v_slab == nullptr) return CKV_ERR_INVALID_ARGUMENT;
  if ((dtype != CKV_DTYPE_BF16 && dtype != CKV_DTYPE_F32) || head_dim <= 0 || n_spans < 0 || n_layers <= 0 ||
      n_heads <= 0 || n_tokens < 0)
    return CKV_ERR_INVALID_ARGUMENT;
  eb = dtype == CKV_DTYPE_BF16 ? 2 : 4;
  if (head_dim * eb % 16 || ((uintptr_t)k_slab | (uintptr_t)v_slab) % 16) return CKV_ERR_INVALID_ARGUMENT;
  if (head_stride < (int64_t)n_tokens * head_dim || layer_stride < head_stride * n_heads) return CKV_ERR_OUT_OF_RANGE;
  return CKV_OK;
}

}  // namespace ckv

extern "C" int32_t ckv_extract_chunks(const void* k_slab, const void* v_slab, int64_t layer_stride,
                                      int64_t head_stride, const uint64_t* dst_tab, const int32_t* spans,
                                      int32_t n_spans, int32_t max_len, int32_t n_layers, int32_t n_heads,
                                      int32_t n_tokens, int32_t head_dim, int32_t dtype, int32_t* err,
                                      void* stream) {
  using namespace ckv;
  if (dst_tab == nullptr || spans == nullptr || max_len < 0) return CKV_ERR_INVALID_ARGUMENT;
  int64_t eb = 0;
  const int32_t rc = extract_check(k_slab, v_slab, layer_stride, head_stride, n_spans, n_layers, n_heads, n_tokens,
                                   head_dim, dtype, eb);
  if (rc != CKV_OK) return rc;
  if (n_spans == 0 || max_len == 0) return CKV_OK;
  const int tiles = (max_len + kExtractTile - 1) / kExtractTile;
  if (n_spans > 65535 || n_layers > 65535) return CKV_ERR_TOO_LARGE;  // grid y and z
  hipLaunchKernelGGL(extract_kernel, dim3((unsigned)tiles, (unsigned)n_spans, (unsigned)n_layers),
                     dim3(kExtractThreads), 0, (hipStream_t)stream, (const char*)k_slab, (const char*)v_slab,
                     layer_stride * eb, head_stride * eb, (int)(head_dim * eb), dst_tab, spans, n_layers, n_heads, n_tokens, err);
  CKV_RETURN_IF_LAUNCH_FAILED();
  return CKV_OK;
}

extern "C" int32_t ckv_extract_chunks_host(const void* k_slab, const void* v_slab, int64_t layer_stride,
                                           int64_t head_stride, const uint64_t* dst, const int32_t* spans,
                                           int32_t n_spans, int32_t n_layers, int32_t n_heads, int32_t n_tokens,
                                           int32_t head_dim, int32_t dtype, void* stream) {
  using namespace ckv;
  if (dst == nullptr || spans == nullptr) return CKV_ERR_INVALID_ARGUMENT;
  int64_t eb = 0;
  const int32_t rc = extract_check(k_slab, v_slab, layer_stride, head_stride, n_spans, n_layers, n_heads, n_tokens,
                                   head_dim, dtype, eb);
  if (rc != CKV_OK) return rc;
  if (n_spans > kExtractArgs || n_layers > 65535) return CKV_ERR_TOO_LARGE;
  ExtractSpans args = {};
  int max_len = 0;
  for (int i = 0; i < n_spans; ++i) {
    const int start = spans[2 * i], len = spans[2 * i + 1];
    if (start < 0 || len < 0 || (int64_t)start + len > n_tokens) return CKV_ERR_OUT_OF_RANGE;
    if (len > 0 && (dst[i] == 0 || dst[i] % 16)) return CKV_ERR_INVALID_ARGUMENT;
    args.dst[i] = dst[i], args.start[i] = start, args.len[i] = len;
    max_len = len > max_len ? len : max_len;
  }
  if (max_len == 0) return CKV_OK;
  const int tiles = (max_len + kExtractTile - 1) / kExtractTile;
  hipLaunchKernelGGL(extract_args_kernel, dim3((unsigned)tiles, (unsigned)n_spans, (unsigned)n_layers),
                     dim3(kExtractThreads), 0, (hipStream_t)stream, (const char*)k_slab, (const char*)v_slab,
                     layer_stride * eb, head_stride * eb, (int)(head_dim * eb), n_layers, n_heads, args);
  CKV_RETURN_IF_LAUNCH_FAILED();
  return CKV_OK;
}

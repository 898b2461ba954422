// Fused q/k RMSNorm + NeoX RoPE + paged KV-cache write (gfx950).
//
// Replaces the Triton kernel of oxr_runtime/kernels.py:66-99 and its CPU
// restatement kernels.py:133-165.  One head (128 bf16 = 256 B) is owned by 16
// lanes, each holding 8 consecutive elements loaded with one 128-bit load, so
// a 64-lane wave works on 4 heads and every load and store is a full 128-bit
// access.  A workgroup takes up to 16 heads of one token, so its token's slot
// and position are scalars; waves of V heads only copy.
//
// What bounds it: HBM, once the instructions are few enough.  4000 tokens of
// 16/8 heads with k and v returned (83 MB): 15.1 us, 5.5 TB/s.  19.7 us with
// heads numbered over the whole batch (a 64-bit division per lane), V heads
// normed for nothing and the exchanges through LDS.
//
// The per-head arithmetic and its bit-exact rounding chain are in norm_rope.h.
#include <algorithm>

#include "norm_rope.h"

namespace oxr {
namespace {

constexpr int kHeadDim = kNormRopeDim;
constexpr int kLanesPerHead = 16;
constexpr int kMaxHeads = 16;  // heads per workgroup

template <bool kNeedKV>
__global__ __launch_bounds__(kMaxHeads* kLanesPerHead) void qk_norm_rope_store_kernel(
    const bf16_t* __restrict__ qkv, const bf16_t* __restrict__ q_weight, const bf16_t* __restrict__ k_weight,
    const bf16_t* __restrict__ cos_table, const bf16_t* __restrict__ sin_table, float eps,
    bf16_t* __restrict__ k_cache, bf16_t* __restrict__ v_cache, const int64_t* __restrict__ slots,
    int64_t num_slots, int num_heads, int num_kv_heads, int first_head, bf16_t* __restrict__ q_out,
    bf16_t* __restrict__ k_out, bf16_t* __restrict__ v_out, const int64_t* __restrict__ positions,
    int64_t table_rows) {
  const int heads_per_token = num_heads + 2 * num_kv_heads;
  const int64_t t = blockIdx.x;
  const int first = first_head + (int)(blockIdx.y * blockDim.x + threadIdx.x) / kLanesPerHead;
  const int s = threadIdx.x % kLanesPerHead;
  // Lanes past the token's last head keep running on that head so every lane
  // takes part in the exchanges below; they store nothing.
  const bool active = first < heads_per_token;
  const int head = min(first, heads_per_token - 1);

  const u32x4 raw = ld128(qkv + (t * heads_per_token + head) * kHeadDim + s * 8);
  const bool is_q = head < num_heads;
  const bool is_v = head >= num_heads + num_kv_heads;
  const int64_t slot = slots[t];
  const bool slot_ok = slot >= 0 && slot < num_slots;
  u32x4 value = raw;
  if (__builtin_amdgcn_ballot_w64(!is_v)) {  // wave-uniform
    // cos/sin row: the token's own row, or the table row of its position
    // (rope_cos[positions], language.py:204) when positions are given.
    int64_t trow = t;
    if (positions) {
      trow = positions[t];
      trow = trow < 0 ? 0 : (trow >= table_rows ? table_rows - 1 : trow);
    }
    const u32x4 normed = norm_rope_16(raw, is_q ? q_weight : k_weight, cos_table + trow * (kHeadDim / 2),
                                      sin_table + trow * (kHeadDim / 2), eps, s);
    if (!is_v) value = normed;
  }
  if (!active) return;

  if (is_q) {
    st128(q_out + (t * num_heads + head) * kHeadDim + s * 8, value);
  } else {
    const int kvh = head - num_heads - (is_v ? num_kv_heads : 0);
    if (slot_ok) st128((is_v ? v_cache : k_cache) + (slot * num_kv_heads + kvh) * kHeadDim + s * 8, value);
    if (kNeedKV) st128((is_v ? v_out : k_out) + (t * num_kv_heads + kvh) * kHeadDim + s * 8, value);
  }
}

}  // namespace
}  // namespace oxr

namespace oxr {
namespace {
int launch_qk(const oxr_bf16* qkv, const oxr_bf16* q_weight, const oxr_bf16* k_weight, const oxr_bf16* cos,
              const oxr_bf16* sin, float eps, oxr_bf16* k_cache, oxr_bf16* v_cache, const int64_t* slots,
              int64_t num_slots, int64_t n, int32_t num_heads, int32_t num_kv_heads, int32_t head_dim,
              oxr_bf16* q_out, oxr_bf16* k_out, oxr_bf16* v_out, const int64_t* positions, int64_t table_rows,
              oxr_stream_t stream) {
  OXR_RETURN_IF(n < 0 || num_heads <= 0 || num_kv_heads <= 0 || num_slots < 0, OXR_ERR_INVALID_ARG);
  OXR_RETURN_IF(head_dim != kHeadDim, OXR_ERR_UNSUPPORTED);
  OXR_RETURN_IF((k_out == nullptr) != (v_out == nullptr), OXR_ERR_INVALID_ARG);
  if (n == 0) return OXR_OK;
  OXR_RETURN_IF(!qkv || !q_weight || !k_weight || !cos || !sin || !k_cache || !v_cache || !slots || !q_out,
                OXR_ERR_INVALID_ARG);
  const int64_t heads = num_heads + 2 * (int64_t)num_kv_heads;
  const int64_t chunks = (heads + kMaxHeads - 1) / kMaxHeads;
  OXR_RETURN_IF(heads > INT32_MAX - kMaxHeads, OXR_ERR_UNSUPPORTED);
  const dim3 block(kWave * (unsigned)((std::min<int64_t>(heads, kMaxHeads) + 3) / 4));
  hipStream_t s = (hipStream_t)stream;
  const auto kernel = k_out ? qk_norm_rope_store_kernel<true> : qk_norm_rope_store_kernel<false>;
  constexpr int64_t kSlice = 1 << 23;  // tokens per launch: a launch holds less than 2^32 threads in x
  constexpr int64_t kChunks = 65535;   // and head chunks: its blocks in y
  for (int64_t t0 = 0; t0 < n; t0 += kSlice) {
    const int64_t table = positions ? 0 : t0 * (kHeadDim / 2), kv = t0 * num_kv_heads * kHeadDim;
    for (int64_t c0 = 0; c0 < chunks; c0 += kChunks) {
      const dim3 grid((unsigned)std::min(kSlice, n - t0), (unsigned)std::min(kChunks, chunks - c0));
      hipLaunchKernelGGL(kernel, grid, block, 0, s, qkv + t0 * heads * kHeadDim, q_weight, k_weight, cos + table,
                         sin + table, eps, k_cache, v_cache, slots + t0, num_slots, num_heads, num_kv_heads,
                         (int)(c0 * kMaxHeads), q_out + t0 * num_heads * kHeadDim, k_out ? k_out + kv : nullptr,
                         k_out ? v_out + kv : nullptr, positions ? positions + t0 : nullptr, table_rows);
    }
  }
  return OXR_LAUNCH_STATUS();
}
}  // namespace
}  // namespace oxr

extern "C" int oxr_qk_norm_rope_store(const oxr_bf16* qkv, const oxr_bf16* q_weight, const oxr_bf16* k_weight,
                                      const oxr_bf16* cos, const oxr_bf16* sin, float eps, oxr_bf16* k_cache,
                                      oxr_bf16* v_cache, const int64_t* slots, int64_t num_slots, int64_t n,
                                      int32_t num_heads, int32_t num_kv_heads, int32_t head_dim, oxr_bf16* q_out,
                                      oxr_bf16* k_out, oxr_bf16* v_out, oxr_stream_t stream) {
  return oxr::launch_qk(qkv, q_weight, k_weight, cos, sin, eps, k_cache, v_cache, slots, num_slots, n, num_heads,
                        num_kv_heads, head_dim, q_out, k_out, v_out, nullptr, 0, stream);
}

extern "C" int oxr_qk_norm_rope_store_at(const oxr_bf16* qkv, const oxr_bf16* q_weight, const oxr_bf16* k_weight,
                                         const oxr_bf16* cos_table, const oxr_bf16* sin_table, int64_t table_rows,
                                         const int64_t* positions, float eps, oxr_bf16* k_cache, oxr_bf16* v_cache,
                                         const int64_t* slots, int64_t num_slots, int64_t n, int32_t num_heads,
                                         int32_t num_kv_heads, int32_t head_dim, oxr_bf16* q_out, oxr_bf16* k_out,
                                         oxr_bf16* v_out, oxr_stream_t stream) {
  if (n > 0 && (!positions || table_rows <= 0)) return OXR_ERR_INVALID_ARG;
  return oxr::launch_qk(qkv, q_weight, k_weight, cos_table, sin_table, eps, k_cache, v_cache, slots, num_slots, n,
                        num_heads, num_kv_heads, head_dim, q_out, k_out, v_out, positions, table_rows, stream);
}

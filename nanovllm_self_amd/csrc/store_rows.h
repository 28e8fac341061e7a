// The KV-cache write of one launch's threads, shared by the write's own launch
// and the planning launch of a prefill call (which writes the step's tokens
// beside the plan).
#pragma once

#include "nvs_common.h"
#include "store_common.h"

namespace nvs {

// ---------------------------------------------------------------------------
// KV-cache write.  One thread owns 8 consecutive head_dim elements of one
// (token, kv_head) row of both K and V; lpr = head_dim / 8 lanes form a row.
// With IDENT the destination row is the token index itself (used by
// nvs_quantize_per_token), otherwise slot_mapping[token].
// ---------------------------------------------------------------------------
struct StoreArgs {
  const void* k;
  const void* v;
  int64_t k_ts, k_hs, v_ts, v_hs;
  const int32_t* slots;
  int64_t rows;         // num_tokens * H
  int64_t total_slots;  // num_blocks * block_size
  void* kc;
  void* vc;
  float* ks;
  float* vs;
  int H, D, lpr_log2;
};

template <int SRC, int DST, bool IDENT, bool HAS_V>
__device__ __forceinline__ void store_rows(const StoreArgs& a, int64_t gid) {
  const int lpr = 1 << a.lpr_log2;
  const int64_t row = gid >> a.lpr_log2;
  const int c = (int)(gid & (lpr - 1));
  const bool active = row < a.rows;
  const int64_t t = active ? row / a.H : 0;
  const int h = active ? (int)(row - t * a.H) : 0;
  int64_t slot = -1;
  if (active) slot = IDENT ? t : (int64_t)a.slots[t];
  const bool valid = active && slot >= 0 && slot < a.total_slots;

  constexpr int SRC_BYTES = (SRC == NVS_DTYPE_FP32) ? 4 : 2;
  float xk[8], xv[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) xk[i] = xv[i] = 0.0f;
  if (valid) {
    load8<SRC>((const char*)a.k + (t * a.k_ts + h * a.k_hs + c * 8) * SRC_BYTES, xk);
    if constexpr (HAS_V)
      load8<SRC>((const char*)a.v + (t * a.v_ts + h * a.v_hs + c * 8) * SRC_BYTES, xv);
  }
  const int64_t dst_row = slot * a.H + h;  // (block*bs + off) * H + h
  const int64_t dst_elem = dst_row * a.D + c * 8;

  if constexpr (DST == NVS_DTYPE_INT8 || DST == NVS_DTYPE_FP8_E4M3) {
    // All lanes of a row take part in the reduction, valid or not.
    constexpr float qmax = (DST == NVS_DTYPE_INT8) ? QuantInt8::kQmax : QuantFp8::kQmax;
    const float sk = quant_scale(row_absmax(xk, lpr), qmax);
    float sv = 0.0f;
    if constexpr (HAS_V) sv = quant_scale(row_absmax(xv, lpr), qmax);
    if (valid) {
      *reinterpret_cast<u32x2*>((uint8_t*)a.kc + dst_elem) = quant8<DST, SRC != NVS_DTYPE_FP32>(xk, sk);
      if (c == 0) a.ks[dst_row] = sk;
      if constexpr (HAS_V) {
        *reinterpret_cast<u32x2*>((uint8_t*)a.vc + dst_elem) = quant8<DST, SRC != NVS_DTYPE_FP32>(xv, sv);
        if (c == 0) a.vs[dst_row] = sv;
      }
    }
  } else {
    constexpr int DST_BYTES = (DST == NVS_DTYPE_FP32) ? 4 : 2;
    if (valid) {
      store8_float<DST>((char*)a.kc + dst_elem * DST_BYTES, xk);
      if constexpr (HAS_V) store8_float<DST>((char*)a.vc + dst_elem * DST_BYTES, xv);
    }
  }
}

// A write to make, validated: arguments and element types.
struct StoreJob {
  StoreArgs a;
  int src, dst;
};

// nvs_store_kvcache's checks and arguments (num_tokens > 0), and its launch.
int make_store_job(StoreJob& job, const void* k, const void* v, int src_dtype, int64_t k_tok_stride,
                   int64_t k_head_stride, int64_t v_tok_stride, int64_t v_head_stride, const int32_t* slot_mapping,
                   int64_t num_tokens, void* k_cache, void* v_cache, int cache_dtype, float* k_scale, float* v_scale,
                   int64_t num_blocks, int block_size, int num_kv_heads, int head_dim);
int launch_store_job(const StoreJob& job, hipStream_t stream);

}  // namespace nvs

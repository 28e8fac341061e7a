// The bf16 copy of a code cache's prefill keys and values that the MFMA
// tile-loop prefill kernel reads (layout and capacity: ShadowLayout in
// attention_common.h).
//
// Reference semantics: prefill_torch's dequantisation of a sequence's cached
// keys and values (nanovllm/layers/attention.py:268-273, 100-117):
// (code.float() * scale.float()).to(bf16), per token and kv head, with
// missing blocks read as zeros (the eager gather pads them with zeros).
//
// Work: tile s (64 consecutive keys of one prefill row, every kv head, K and
// V), or half of it when the copy has fewer tiles than work-groups, per
// work-group iteration; the plan kernel numbered the tiles row by row
// (ShadowLayout::base).  A work-group finds the row of its tile by a binary
// search over those numbers, writes the table entry (first half), and
// converts its token rows of K and of V: 16 lanes to a row (8 codes, one
// 8-byte load, a 16-byte store each), 16 rows per pass of 256 threads.
// Keys past the row's length are not written (the prefill kernel never
// reads them).
#include <algorithm>

#include "nvs_common.h"
#include "attention_common.h"

namespace nvs {

namespace {

constexpr int kShadowThreads = 256;

struct ShadowArgs {
  const uint8_t* kc;
  const uint8_t* vc;
  const float* ks;
  const float* vs;
  const int32_t* bt;
  int64_t bt_stride;
  int64_t NB;
  int bs;
  const int32_t* cu_k;
  int B, Hkv;
  const PlanHeader* hdr;
  ShadowLayout sh;
};

// Eight codes (bytes of w) times the row's scale, rounded to bf16 (one
// conversion per pair, round-to-nearest-even as torch's .to(bf16)).
template <int KV>
__device__ __forceinline__ u32x4 dequant8(u32x2 w, float sc) {
  u32x4 o;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    float f0, f1;
    if (i & 1)
      code_pair_to_f32<KV, true>(w[i >> 1], f0, f1);
    else
      code_pair_to_f32<KV, false>(w[i >> 1], f0, f1);
    o[i] = pack_bf16x2(f0 * sc, f1 * sc);
  }
  return o;
}

// The row of copy tile s: the largest b with base[b] <= s (base is
// non-decreasing with base[B] = total > s, so that row has tiles).  Sixty-four
// candidates a round, one a lane: a batch of up to 64 rows takes one load
// round trip.
__device__ __forceinline__ int row_of_tile(const int* base, int B, int s, int lane) {
  int lo = 0, hi = B;
  while (hi - lo > 1) {
    const int step = (hi - lo + 63) / 64, i = lo + lane * step;
    const int n = __popcll(__ballot(i < hi && base[min(i, hi - 1)] <= s));
    lo += (n - 1) * step;
    hi = min(lo + step, hi);
  }
  return __builtin_amdgcn_readfirstlane(lo);
}

// A work-group dequantises a piece of a tile: its 64 keys, or, while the grid
// holds them all, half, a quarter or an eighth of them.  Sixteen lanes take a
// token row (eight codes each; 16-byte loads would store every other 16 bytes,
// 10 % slower), two rows at a time a thread.  Bound by HBM in a long copy, by
// latency in a short one (the tile's row, block and scales are loads that
// wait for each other), which small pieces and few round trips shorten; more
// work-groups than the CUs hold keep the stream dense.  Tiles of 8 heads,
// fp8: 182 of them (71 MB) 23.5 -> 17.0 us, 504 39.2 -> 34.6, 717 51.7 ->
// 47.6; 833 of int8 66.2 -> 56.0 (before: whole or half tiles, 1024
// work-groups that loop, a row searched by halves).
constexpr int kShadowRows = kShadowThreads / 16;  // token rows of a pass
constexpr int kShadowPieces = 8;
constexpr int kShadowUnroll = 2;

template <int KV>
__global__ __launch_bounds__(kShadowThreads) void shadow_fill_kernel(ShadowArgs a) {
  if (a.hdr->shadow_on == 0) return;
  const int total = a.hdr->shadow_tiles;
  const int j = threadIdx.x & 15;
  const int rows = kShadowTile * a.Hkv;  // token rows of a tile (token-major, then kv head)
  int log_pieces = 0;
  while ((1 << log_pieces) < kShadowPieces && (int64_t)total << (log_pieces + 1) <= (int64_t)gridDim.x) ++log_pieces;
  const int span = kShadowTile >> log_pieces;  // keys of a piece
  for (int64_t u = blockIdx.x; u < (int64_t)total << log_pieces; u += gridDim.x) {
    const int s = (int)(u >> log_pieces), piece = (int)u & ((1 << log_pieces) - 1);
    const int b = row_of_tile(a.sh.base, a.B, s, threadIdx.x & 63);
    const int t = s - a.sh.base[b];  // < ST: the plan keeps a row's tiles within its table row
    if (threadIdx.x == 0 && piece == 0) a.sh.table[(int64_t)b * a.sh.ST + t] = s;
    const int K = a.cu_k[b + 1] - a.cu_k[b];
    // The tile's keys lie in one block (block_size is a multiple of 64).
    const int lb = (int)((uint32_t)(kShadowTile * t) / (uint32_t)a.bs);
    int blk = kShadowTile * (int64_t)t < K && lb < a.bt_stride ? a.bt[(int64_t)b * a.bt_stride + lb] : -1;
    if (blk >= a.NB) blk = -1;
    const int64_t row0 = blk >= 0 ? ((int64_t)blk * a.bs + (kShadowTile * t - lb * a.bs)) * a.Hkv : 0;
    const int keys = min(K - kShadowTile * t, kShadowTile);
    const int64_t out0 = (int64_t)s * rows;
    const int r_end = min(keys, span * (piece + 1)) * a.Hkv;
    for (int r0 = span * piece * a.Hkv + (int)(threadIdx.x >> 4); r0 < r_end; r0 += kShadowUnroll * kShadowRows) {
      u32x2 kw[kShadowUnroll], vw[kShadowUnroll];
      float ks[kShadowUnroll], vs[kShadowUnroll];
#pragma unroll
      for (int i = 0; i < kShadowUnroll; ++i) {
        const int r = min(r0 + i * kShadowRows, r_end - 1);
        const int64_t cr = row0 + (blk >= 0 ? r : 0);  // cache row (token, kv head)
        kw[i] = *reinterpret_cast<const u32x2*>(a.kc + cr * kHeadDim + 8 * j);
        vw[i] = *reinterpret_cast<const u32x2*>(a.vc + cr * kHeadDim + 8 * j);
        ks[i] = a.ks[cr];
        vs[i] = a.vs[cr];
      }
#pragma unroll
      for (int i = 0; i < kShadowUnroll; ++i) {
        const int r = r0 + i * kShadowRows;
        if (r >= r_end) break;
        u32x4 ko = dequant8<KV>(kw[i], ks[i]), vo = dequant8<KV>(vw[i], vs[i]);
        if (blk < 0) ko = vo = u32x4{0u, 0u, 0u, 0u};  // missing block: zeros
        *reinterpret_cast<u32x4*>(a.sh.k + (out0 + r) * kHeadDim + 8 * j) = ko;
        *reinterpret_cast<u32x4*>(a.sh.v + (out0 + r) * kHeadDim + 8 * j) = vo;
      }
    }
  }
}

}  // namespace

int launch_shadow_fill(const AttnParams& P, const Plan& plan, const ShadowLayout& sh, hipStream_t stream) {
  ShadowArgs a;
  a.kc = (const uint8_t*)P.kc;
  a.vc = (const uint8_t*)P.vc;
  a.ks = P.ks;
  a.vs = P.vs;
  a.bt = P.bt;
  a.bt_stride = P.bt_stride;
  a.NB = P.NB;
  a.bs = P.bs;
  a.cu_k = P.cu_k;
  a.B = P.B;
  a.Hkv = P.Hkv;
  a.hdr = plan.hdr;
  a.sh = sh;
  if (P.B <= 0 || sh.cap <= 0) return NVS_OK;
  // Up to four times the work-groups the CUs hold (8, 16, 32 and 64 a CU: 833
  // tiles 61.6, 56.3, 56.0 and 55.6 us), never more than the copy's pieces.
  const int wgs = (int)std::min<int64_t>(kShadowPieces * (int64_t)sh.cap, (int64_t)device_slots(32));
  dim3 grid((unsigned)std::max(1, wgs)), block(kShadowThreads);
  switch (P.cache_dtype) {
    case NVS_DTYPE_INT8:
      hipLaunchKernelGGL(shadow_fill_kernel<NVS_DTYPE_INT8>, grid, block, 0, stream, a);
      break;
    case NVS_DTYPE_FP8_E4M3:
      hipLaunchKernelGGL(shadow_fill_kernel<NVS_DTYPE_FP8_E4M3>, grid, block, 0, stream, a);
      break;
    default:
      set_error("paged_attention: no bf16 copy for cache dtype %d", P.cache_dtype);
      return NVS_ERR_UNSUPPORTED;
  }
  return check_launch("shadow_fill");
}

}  // namespace nvs

// Whole-block copies between a paged cache and a packed block snapshot: the
// KV handoff of prefill/decode disaggregation (pd_self/kv_connector.py).
//
//   export  kv_cache[:, :, src_block_ids]      (_export_kv_snapshot :94-110)
//   import  kv_cache[:, :, dst_block_ids[i]] = blocks[:, :, i]
//                                               (load_kv_item :282-311)
//
// The caches are [planes, num_blocks, block] arrays of bytes (planes = 2 x
// layers; a block is block_size x kv_heads x head_dim codes, or the
// block_size x kv_heads fp32 scales), so one kernel serves bf16, fp16, fp32,
// int8 and fp8 codes and the scales alike.  Copies must not overlap each
// other (distinct destination blocks, source and destination regions
// disjoint): the work-groups run in no particular order.
//
// Bound by HBM.  A work-group copies one 16-byte load and store a lane, both
// non-temporal: the dispatcher hands out the next chunk as soon as one ends, so
// the stream stays dense and in address order.  One wave a work-group for large
// blocks (72 planes x 16 blocks of 512 KiB, 604 MB each way: 184 us, 6.55 TB/s
// read and written; 195 with four waves), four for blocks of up to 256 KiB, of
// which one-wave chunks wait for the dispatcher (72 planes x 32 blocks of 8 KiB,
// what a code cache's scales are: 11.6 us, 9.4 with four waves, 9.8 before; of
// 128 KiB 106 and 104, 116 before).  Measured beside it at 512 KiB, gathering /
// scattering: 256 threads with four loads each, 8192 work-groups that loop,
// plain stores (before) 232 / 237 us; the same with non-temporal stores 211 /
// 223; two waves a chunk 193 / 192; one wave with the item split by divisions
// instead of the grid's dimensions 195 / 195, with two loads a lane 189 / 192.
#include <algorithm>

#include "nvs_common.h"

namespace nvs {
namespace {

constexpr int64_t kCopySmallBlock = 256 << 10;  // blocks of up to so many bytes are copied by four waves a chunk
// Largest grid dimensions; the kernel loops over what lies beyond.
constexpr int64_t kGridX = 1 << 24, kGridYZ = 65535;

struct CopyArgs {
  const char* src;
  char* dst;
  const int32_t* src_ids;  // NULL: copy i reads block i
  const int32_t* dst_ids;  // NULL: copy i writes block i
  int64_t src_nb, dst_nb;
  int64_t block_bytes;
  int64_t chunks;  // chunks per block
  int64_t copies;
  int64_t planes;
};

// Work-group (chunk, copy, plane).
template <int THREADS>
__global__ __launch_bounds__(THREADS) void copy_blocks_kernel(CopyArgs a) {
  for (int64_t plane = blockIdx.z; plane < a.planes; plane += gridDim.z) {
    for (int64_t i = blockIdx.y; i < a.copies; i += gridDim.y) {
      const int64_t s = a.src_ids ? a.src_ids[i] : i;
      const int64_t d = a.dst_ids ? a.dst_ids[i] : i;
      if (s < 0 || s >= a.src_nb || d < 0 || d >= a.dst_nb) continue;  // uniform per work-group
      const char* from = a.src + (plane * a.src_nb + s) * a.block_bytes;
      char* to = a.dst + (plane * a.dst_nb + d) * a.block_bytes;
      for (int64_t chunk = blockIdx.x; chunk < a.chunks; chunk += gridDim.x) {
        const int64_t off = (chunk * THREADS + threadIdx.x) * 16;
        if (off < a.block_bytes)
          __builtin_nontemporal_store(__builtin_nontemporal_load((const u32x4*)(from + off)), (u32x4*)(to + off));
      }
    }
  }
}

}  // namespace
}  // namespace nvs

using namespace nvs;

extern "C" int nvs_copy_blocks(const void* src, int64_t src_num_blocks, const int32_t* src_block_ids,
                               void* dst, int64_t dst_num_blocks, const int32_t* dst_block_ids,
                               int64_t num_planes, int64_t block_bytes, int64_t num_copies, void* stream) {
  clear_error();
  const char* who = "copy_blocks";
  NVS_REQUIRE(num_planes >= 0 && num_copies >= 0 && src_num_blocks >= 0 && dst_num_blocks >= 0,
              NVS_ERR_INVALID, "%s: negative size", who);
  NVS_REQUIRE(block_bytes > 0 && block_bytes % 16 == 0, NVS_ERR_INVALID,
              "%s: block_bytes %lld must be a positive multiple of 16", who, (long long)block_bytes);
  NVS_REQUIRE(src_block_ids || num_copies <= src_num_blocks, NVS_ERR_INVALID,
              "%s: %lld copies from a %lld-block source without ids", who, (long long)num_copies,
              (long long)src_num_blocks);
  NVS_REQUIRE(dst_block_ids || num_copies <= dst_num_blocks, NVS_ERR_INVALID,
              "%s: %lld copies into a %lld-block destination without ids", who, (long long)num_copies,
              (long long)dst_num_blocks);
  const int threads = block_bytes <= kCopySmallBlock ? 256 : 64;
  const int64_t chunks = (block_bytes + threads * 16 - 1) / (threads * 16);
  if (num_planes == 0 || num_copies == 0) return NVS_OK;
  NVS_REQUIRE(src && dst, NVS_ERR_INVALID, "%s: null pointer argument", who);
  NVS_REQUIRE(((uintptr_t)src % 16) == 0 && ((uintptr_t)dst % 16) == 0, NVS_ERR_INVALID,
              "%s: buffers must be 16-byte aligned", who);
  CopyArgs a;
  a.src = (const char*)src; a.dst = (char*)dst;
  a.src_ids = src_block_ids; a.dst_ids = dst_block_ids;
  a.src_nb = src_num_blocks; a.dst_nb = dst_num_blocks;
  a.block_bytes = block_bytes; a.chunks = chunks; a.copies = num_copies; a.planes = num_planes;
  const dim3 grid((unsigned)std::min(chunks, kGridX), (unsigned)std::min(num_copies, kGridYZ),
                  (unsigned)std::min(num_planes, kGridYZ));
  hipLaunchKernelGGL(threads == 256 ? copy_blocks_kernel<256> : copy_blocks_kernel<64>, grid, dim3(threads), 0,
                     (hipStream_t)stream, a);
  return check_launch(who);
}

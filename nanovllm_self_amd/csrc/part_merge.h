// The merge of prefill entries split along the keys: what the tile-loop
// kernel's units left in their slots of the workspace, joined by a
// log-sum-exp into output rows.
#pragma once

#include "nvs_common.h"
#include "attention_common.h"

namespace nvs {

struct PartMergeArgs {
  const PlanHeader* hdr;
  const SplitRow* rows;
  const char* slots;
  int units, hgroups, hpi, g;  // units of an entry; head groups, heads per item, group
  uint16_t* out;
  int64_t out_ts, out_hs;
  int f16;
  int wgs;  // work-groups of the launch that merge parts (0: none)
};

// Slot layout (a wave's part): the accumulators O^T[n][qb] of head_dim block
// n and q-block qb as 4 KiB each, register group k of the 64 lanes together:
// lane (qc, h) holds d = 32 n + 8 k + 4 h .. + 3 of row qc; then m and l.
//
// A work-group merges one wave's part of one unit (64 rows), its waves
// taking the (n, qb) blocks' halves, so that a few hundred units fill the
// chip.  It is bound by the slots' bytes, 132 KiB a part and unit, and their
// loads' latency, four parts in flight at a time: 152 slots 3.6 us, 504 slots
// 9.3 us (7 TB/s) beyond a launch that merges nothing (4.7 us).
__device__ __forceinline__ void merge_parts(const PartMergeArgs& a, int wg) {
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int n = w >> 2, qb = (w >> 1) & 1, kh = w & 1, qc = lane & 31, h = lane >> 5;
  const int items = a.hdr->n_split * a.units * 4;
  for (int item = wg; item < items; item += a.wgs) {
    const int kw = item & 3, u = (item >> 2) % a.units;
    const SplitRow row = a.rows[(item >> 2) / a.units];
    const char* base = a.slots + (int64_t)(row.slot + u) * kPartBytes + kw * kPartWaveBytes;
    const int64_t stride = (int64_t)a.units * kPartBytes;
    const int o_off = (2 * n + qb) * 4096 + 2 * kh * 1024 + lane * 16, m_off = 32768 + qb * 256 + lane * 4;
    float M = -INFINITY, L = 0.0f;
    f32x4 acc[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
    for (int c0 = 0; c0 < row.parts; c0 += 4) {
      float m[4], l[4];
      f32x4 o[4][2];
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const char* p = base + min(c0 + c, row.parts - 1) * stride;
        m[c] = *reinterpret_cast<const float*>(p + m_off);
        l[c] = *reinterpret_cast<const float*>(p + m_off + 512);
#pragma unroll
        for (int k = 0; k < 2; ++k) o[c][k] = *reinterpret_cast<const f32x4*>(p + o_off + 1024 * k);
      }
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        if (c0 + c >= row.parts) break;
        const float m_new = fmaxf(M, m[c]);
        const float al = M == -INFINITY ? 0.0f : fast_exp2(M - m_new);
        const float be = m[c] == -INFINITY ? 0.0f : fast_exp2(m[c] - m_new);
        M = m_new;
        L = L * al + l[c] * be;
#pragma unroll
        for (int k = 0; k < 2; ++k) acc[k] = acc[k] * al + o[c][k] * be;
      }
    }
    const int qbi = 2 * kw + qb, hkv = u / a.hgroups, hin = (u % a.hgroups) * a.hpi + qbi % a.hpi;
    const int pos = row.p0 + 32 * (qbi / a.hpi) + qc;
    if (hin < a.g && pos < row.L) {
      const float inv = L > 0.0f ? 1.0f / L : 0.0f;
      uint16_t* out = a.out + (int64_t)(row.q0 + pos) * a.out_ts + (int64_t)(hkv * a.g + hin) * a.out_hs + 32 * n +
                      16 * kh + 4 * h;
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        const f32x4 x = acc[k] * inv;
        u32x2 v;
        v[0] = a.f16 ? pack_f16x2(x[0], x[1]) : pack_bf16x2(x[0], x[1]);
        v[1] = a.f16 ? pack_f16x2(x[2], x[3]) : pack_bf16x2(x[2], x[3]);
        *reinterpret_cast<u32x2*>(out + 8 * k) = v;
      }
    }
  }
}

}  // namespace nvs

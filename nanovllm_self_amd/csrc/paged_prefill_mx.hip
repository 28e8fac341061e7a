// Varlen causal prefill attention for bf16 (or fp16) K/V on gfx950: one wave
// per SIMD, 64 query rows per wave, a hand-scheduled tile loop.
//
// Reference semantics: prefill_flashattn (nanovllm/layers/attention.py:303-375)
// and prefill_torch (:378-498): query row r of a sequence with L new and K
// visible keys attends keys j <= r + (K - L); GQA head map hq -> hq / g;
// softmax in fp32; output rounded to bf16 (fp16 for an fp16 cache, whose Q,
// K, V and P are fp16 and whose MFMA is the fp16 one, as the reference's
// flash path computes in the cache's dtype).  Paged mode reads K/V through
// block_tables (a missing block reads as zeros); local mode reads the step's
// own k/v rows (block_tables is None).
//
// Work item: (sequence, tile of P query positions, kv head, group of hpi
// query heads) on one 256-thread work-group (four waves, one per SIMD):
// hpi = min(8, the largest power of two <= g) heads share the item's K/V
// tiles and P = 256 / hpi positions fill 8 q-blocks of 32 rows; wave w owns
// q-blocks 2w and 2w + 1 (the same positions when hpi >= 2).
//
// All of a work-group's work is one inline-asm statement generated by
// gen_prefill_mx.py (prefill_mx_asm.inc).  Per 64-key tile and wave it runs
// 64 v_mfma_f32_32x32x16_bf16 (QK^T of the next tile, PV of the previous
// one), reads K/V operands from LDS into AGPR rings six operands ahead, and
// interleaves the online softmax of the current tile (running max with a
// row-sum check instead of a per-tile max, exponentials, bf16 packing, row
// sums) between the MFMAs, so the matrix pipe and the vector ALU run side
// by side in one wave.  Q^T (64 registers) and O^T (128) live in AGPRs; S
// and P are double buffered in VGPRs.  Tiles are copied HBM -> LDS by
// buffer loads that write LDS directly; rows past the keys and missing
// blocks fall outside the buffer resource and read as zero.  The pipeline
// runs on from one unit into the next: a unit's last iterations copy the
// next unit's first key tiles and run its first QK^T, and the next unit's
// first iteration runs the unit's last PV and stores its output (bf16 rows,
// staged through the wave's query stage and stored whole) beside its own
// work.
//
// LDS (per work-group): K tiles at 0 and 16 KiB, V tiles at 32, 48 and 64
// KiB (64 keys x 128 d bf16, 16-byte chunks XOR-swizzled per key; the V
// tiles rotate through the three, each filled an iteration before segment B
// reads it), then one 16 KiB query stage per wave (the next unit's 64 query
// rows, swizzled as the key tiles: 144 KiB in all), then the three claim
// slots.
#include <algorithm>
#include <cstdlib>
#include <string>

#include "nvs_common.h"
#include "attention_common.h"
#include "decode_wave.h"
#include "prefill_mx_asm.inc"

namespace nvs {

constexpr int kMxThreads = 256;
constexpr int kMxStageBytes = 16384;     // per wave: 64 query rows x 256 B
constexpr int kMxQStage = 81920;         // query stage: one kMxStageBytes per wave
constexpr int kMxLdsBytes = kMxQStage + 4 * kMxStageBytes;

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef int32_t i32x8 __attribute__((ext_vector_type(8)));
typedef int32_t i32x4 __attribute__((ext_vector_type(4)));
typedef int32_t i32x2 __attribute__((ext_vector_type(2)));

struct MxArgs {
  const uint16_t* q;
  int64_t q_ts, q_hs;
  const char* kc;  // paged caches
  const char* vc;
  const int32_t* bt;
  int bt_stride;
  int NB;
  int bs;
  const char* k;  // local k / v
  const char* v;
  int64_t k_ts, k_hs, v_ts, v_hs;
  int64_t Tk;  // rows of the local k / v
  const int32_t* cu_q;
  const int32_t* cu_k;
  int Hq, Hkv, g, hpi, hgroups;
  Plan plan;
  float scale_log2;
  uint16_t* out;
  int64_t out_ts, out_hs;
  const int* gate;  // run only where *gate == gate_run (null: always)
  int gate_run;
  // The call's decode rows, streamed first by the work-groups the plan
  // names (the kernel's DKV names their cache type).
  DecodeArgs dec;
  const int32_t* dec_bt;
  int dec_groups;  // decode groups the partial workspace has room for
  char* parts;     // slots of the units that cover a part of their keys (null: none)
};

// Tile ring depth of the decode waves in this kernel (one wave per SIMD,
// the prefill's occupancy): 3 (2 and 4 measured within 1 % of it on
// mixed_32b, bf16 and fp8).
#ifndef NVS_CODECODE_RING
#define NVS_CODECODE_RING 3
#endif
constexpr int kNoDecode = -1;

// Heads per item for a group of g query heads per kv head.
__host__ __device__ inline int mx_heads_per_item(int g) {
  int h = 1;
  while (2 * h <= g && 2 * h <= 8) h *= 2;
  return h;
}
int prefill_mx_positions(int g) { return 256 / mx_heads_per_item(g); }
int prefill_mx_units(int Hq, int Hkv) {
  const int g = Hq / Hkv, hpi = mx_heads_per_item(g);
  return Hkv * ((g + hpi - 1) / hpi);
}
int prefill_mx_wgs(int64_t units) {
  return (int)std::max<int64_t>(8, std::min<int64_t>((units + 7) & ~(int64_t)7, device_slots(1)) & ~(int64_t)7);
}

__device__ __forceinline__ int mx_swz(int key) { return ((key & 3) << 2) | ((key >> 2) & 3); }

__device__ __forceinline__ int mx_lane() {
  return __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
}

// Persistent, dynamically scheduled over the prefill list: unit u = (list
// entry, kv head, head group); units with u % 8 == x belong to XCD x and are
// claimed from its counter by the work-groups on it, except the first three
// rounds: the work-groups that start on the prefill at once take those by
// their number, back and forth (claimed one after the other, three to a
// work-group, 104 units of up to 10 tiles left most of the chip idle: 26.4
// us, now 22.0).  One asm statement (gen_prefill_mx.py) runs the rest: it
// claims each further unit three ahead, decodes units from their plan
// records, and streams their tiles through one pipeline that runs on from
// one unit into the next.  What it needs from here: lane constants (LDS
// operand addresses, fill, query-copy and output lane offsets), the call's
// constants in one VGPR (lane k holds constant k, read with v_readlane) and
// scalar inputs.
//
// With a decode cache type DKV, the first plan.hdr->dec_wgs work-groups (a
// multiple of 8, so as many on every XCD) first stream the call's decode
// rows, one decode wave per wave, and then join the prefill: the decode's
// HBM stream runs beside the prefill's MFMA work instead of before it.  The
// decode waves of XCD x form groups k = 8 j + x (Hkv waves of one XCD a
// group, as in the decode kernel), G groups in all; the merge of rows split
// across groups is a launch after this one.
template <bool PAGED, bool F16, int DKV>
__global__ __launch_bounds__(kMxThreads) __attribute__((amdgpu_waves_per_eu(1, 1))) void prefill_mx_kernel(
    MxArgs a, const PlanRecord* __restrict__ rec) {
  __shared__ __attribute__((aligned(1024))) char lds[kMxLdsBytes];
  __shared__ int s_claim[3];
  // Work-groups of this XCD that start on the prefill at once, and this
  // one's number among them (below 0: it streams decode rows first).
  int starters = gridDim.x >> 3, number = blockIdx.x >> 3;
  if constexpr (DKV != kNoDecode) {
    const int nd = __builtin_amdgcn_readfirstlane(a.plan.hdr->dec_wgs);
    starters -= nd >> 3;
    number -= nd >> 3;
    if ((int)blockIdx.x < nd) {
      const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
      const int lw = 4 * (int)(blockIdx.x >> 3) + wave;  // among the XCD's nd / 2 decode waves
      const int gx = (nd / 2) / a.Hkv;                     // whole groups an XCD holds
      const int G = min(8 * gx, a.dec_groups);
      const int h = lw % a.Hkv, k = 8 * (lw / a.Hkv) + (int)(blockIdx.x & 7);
      decode_wave<DKV, NVS_CODECODE_RING>(a.dec, a.dec_bt, a.dec.cu_q, a.dec.cu_k, h, k, G,
                                          4 * (int)blockIdx.x + wave, 4 * nd);
    }
  }
  if (a.gate && *a.gate != a.gate_run) return;  // the other prefill kernel serves this call
  const uint32_t lds_base = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)lds;
  const int per_entry = a.Hkv * a.hgroups;
  const int units = a.plan.hdr->n_prefill * per_entry;
  const int xcd = blockIdx.x & 7;
  int* counter = a.plan.hdr->prefill_next + xcd;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // Beside decode rows a long list is claimed throughout: the work-groups that
  // join late should not find the others' units dealt (2048 units beside 128
  // rows 1744 us, 1769 dealt; over 16 ragged batches of 1.0 .. 2.3 K units
  // claiming is 1.2 % slower, from 4.6 slower to 5.6 faster; over 16 of 150 ..
  // 1024 it is 6 % slower.  4416 units without decode rows 1125 claimed, 1120 ..
  // 1123 dealt).
  if (units > kSplitMaxUnits && starters < (int)(gridDim.x >> 3)) starters = 0, number = -1;
  if (number < 0) {  // or streamed decode rows: joins late
    if (threadIdx.x == 0)
      for (int i = 0; i < 3; ++i) s_claim[i] = 3 * starters + atomicAdd(counter, 1);
  } else if (threadIdx.x < 3) {
    const int i = threadIdx.x;
    s_claim[i] = i * starters + (i == 1 ? starters - 1 - number : number);
  }
  __syncthreads();
  const int u0 = __builtin_amdgcn_readfirstlane(8 * s_claim[0] + xcd);
  const int u1 = __builtin_amdgcn_readfirstlane(8 * s_claim[1] + xcd);
  const int u2 = __builtin_amdgcn_readfirstlane(8 * s_claim[2] + xcd);
  if (u0 >= units) return;  // the same for the whole work-group
  __syncthreads();          // the claim slots are read: the loop reuses them

  const int lane = mx_lane();
  const int qc = lane & 31, h = lane >> 5;
  const int krow = PAGED ? a.Hkv * 256 : (int)(a.k_ts * 2);  // = the value row stride
  const int qrts = (int)(a.q_ts * 2);
  const int orts = (int)(a.out_ts * 2);
  // K operands: key qc, d-step st (K buffer 0); V operands of V buffer 2
  // (the loop moves them to the first iteration's buffer, 0, and on).
  i32x8 kaddr, vaddr;
#pragma unroll
  for (int st = 0; st < 8; ++st) kaddr[st] = (int)lds_base + qc * 256 + (((2 * st + h) ^ mx_swz(qc)) << 4);
  {
    const int r = (lane >> 2) & 3, c = lane & 3, gp = (lane >> 4) & 1;
#pragma unroll
    for (int n = 0; n < 4; ++n)
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        const int ke = 4 * h + r + 8 * e;
        const int chunk = (4 * n + 2 * gp + (c >> 1)) ^ mx_swz(ke);
        vaddr[2 * n + e] = (int)lds_base + 32768 + 2 * 16384 + ke * 256 + chunk * 16 + 8 * (c & 1);
      }
  }
  // Fills: row 16 w + 4 i + lane / 16 of a tile, its 16-byte chunk lane % 16
  // into LDS slot chunk ^ swz(row).  Query copies: row 4 i + lane / 16 of a
  // q-block (+ 16 rows through the soffset), the same swizzle.
  i32x4 dmak, qlane;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int row = 16 * w + 4 * i + (lane >> 4);
    dmak[i] = row * krow + (((lane & 15) ^ mx_swz(row)) << 4);
    const int rq = 4 * i + (lane >> 4);
    qlane[i] = rq * qrts + (((lane & 15) ^ mx_swz(rq)) << 4);
  }
  // Output rows are staged through the query stage and stored four a store:
  // lane L stores chunk L % 16 of row 4 i + L / 16, read from its swizzled
  // slot (L % 16) ^ ((L / 16) << 2) ^ (i % 4) of the stage.
  const int ooff = (lane >> 4) * orts + 16 * (lane & 15);
  const int rl = (int)lds_base + kMxQStage + w * kMxStageBytes + (lane >> 4) * 256 +
                 (((lane & 15) ^ ((lane >> 4) << 2)) << 4);
  const int lanec = qc - 4 * h;

  // The call's constants (and the wave's q-block placement), lane k.
  int bank = 0;
  auto put = [&](int k, int v) { bank = lane == k ? v : bank; };
  auto put64 = [&](int k, const void* p) {
    put(k, (int)(uint32_t)(uint64_t)p);
    put(k + 1, (int)(uint32_t)((uint64_t)p >> 32));
  };
  put(0, a.hgroups - 1);
  put(1, a.hpi);
  put(2, a.g);
  put(3, a.Hq - 1);
#pragma unroll
  for (int qb = 0; qb < 2; ++qb) {
    const int qbi = 2 * w + qb;
    put(4 + qb, qbi % a.hpi);
    put(6 + qb, 32 * (qbi / a.hpi));
  }
  put64(8, PAGED ? (const void*)a.kc : (const void*)a.k);
  put64(10, PAGED ? (const void*)a.vc : (const void*)a.v);
  put(12, PAGED ? 0 : (int)(a.k_ts * 2));
  put(13, PAGED ? 256 : (int)(a.k_hs * 2));
  put(14, PAGED ? 256 : (int)(a.v_hs * 2));
  put64(15, a.q);
  put(17, qrts);
  put(18, (int)(a.q_hs * 2));
  put64(19, a.out);
  put(21, orts);
  put(22, (int)(a.out_hs * 2));
  put64(23, PAGED ? (const void*)a.bt : nullptr);
  put(25, PAGED ? 4 * a.bt_stride : 0);
  put64(26, a.parts + w * kPartWaveBytes);

  const int s_bs = PAGED ? a.bs : 64;
  const int s_nb = PAGED ? a.NB : 0;
  const int s_m0w = (int)lds_base + w * 4096;
  const int s_scale = __float_as_int(a.scale_log2);
  const uint64_t s_cnt = (uint64_t)counter;
  const int claim0 = xcd + 24 * starters;  // unit of the counter's value 0
  const int s_qst = (int)lds_base + kMxQStage + w * kMxStageBytes;
  const int s_qd = kMxQStage + w * kMxStageBytes;
  const uint32_t mpe = per_entry == 1 ? 0u : (uint32_t)((0x100000000ull + per_entry - 1) / per_entry);
  const int s_mpe = __builtin_amdgcn_readfirstlane((int)mpe);
  const int s_pe1 = __builtin_amdgcn_readfirstlane(per_entry == 1 ? -1 : 0);
  const uint64_t s_rec = (uint64_t)rec;
  const int s_q16 = 16 * qrts;
  const int s_slot = (int)(uint32_t)(uintptr_t)(__attribute__((address_space(3))) int*)s_claim;

#define NVS_MX_OPERANDS                                                                                   \
  : "+{v[200:207]}"(vaddr)                                                                                 \
  : "{v[192:199]}"(kaddr), "{v[208:211]}"(dmak), "{v[212:215]}"(qlane),                                  \
    "{v246}"(ooff), "{v247}"(lanec), "{v248}"(bank), "{v255}"(rl),                                        \
    "{s4}"(krow), "{s5}"(s_bs), "{s6}"(s_nb), "{s7}"(s_m0w), "{s8}"(s_scale), "{s9}"(w),                  \
    "{s[10:11]}"(s_cnt), "{s12}"(s_qst), "{s13}"(s_qd), "{s14}"(claim0), "{s15}"(units), "{s16}"(s_mpe),       \
    "{s17}"(per_entry), "{s[18:19]}"(s_rec), "{s20}"(s_q16), "{s21}"(s_slot), "{s22}"(u0), "{s23}"(u1),    \
    "{s37}"(s_pe1), "{s60}"(u2), "{s61}"(4 * orts)                                                        \
  : NVS_PREFILL_MX_CLOBBERS
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
  if constexpr (PAGED && !F16) {
    asm volatile(NVS_PREFILL_MX_ASM_PAGED NVS_MX_OPERANDS);
  } else if constexpr (!PAGED && !F16) {
    asm volatile(NVS_PREFILL_MX_ASM_LOCAL NVS_MX_OPERANDS);
  } else if constexpr (PAGED) {
    asm volatile(NVS_PREFILL_MX_ASM_PAGED_F16 NVS_MX_OPERANDS);
  } else {
    asm volatile(NVS_PREFILL_MX_ASM_LOCAL_F16 NVS_MX_OPERANDS);
  }
#pragma clang diagnostic pop
#undef NVS_MX_OPERANDS
}

// Whether the MFMA tile-loop kernel serves this call: bf16 or fp16 K/V (a
// bf16 / fp16 cache, or the local mode) and head_dim 128.  NVS_PREFILL_KERNEL=classic
// selects the classic kernel for every call.
bool prefill_mx_serves(const AttnParams& P) {
  static const bool off = [] {
    const char* e = std::getenv("NVS_PREFILL_KERNEL");
    return e && std::string(e) == "classic";
  }();
  if (off) return false;
  // Lane offsets of the fills and of the query copies are 32-bit: 64 key rows
  // and 32 query rows of their row strides must fit.
  if (64 * P.q_ts >= (1ll << 31)) return false;
  // Output rows are stored through a 32-bit buffer range of 32 rows.
  if (P.out_ts < kHeadDim || 64 * P.out_ts >= (1ll << 31)) return false;
  // Query and output head strides, in bytes, are 32-bit constants.
  if (P.q_hs * 2 >= (1ll << 31) || P.out_hs * 2 >= (1ll << 31)) return false;
  // Local mode: one lane offset serves the K and V fills (equal row strides);
  // row and head strides in bytes are 32-bit.
  if (P.bt == nullptr)
    return P.k_ts >= 0 && P.k_ts == P.v_ts && 128 * P.k_ts < (1ll << 31) && P.k_hs >= 0 && P.v_hs >= 0 &&
           2 * std::max(P.k_hs, P.v_hs) < (1ll << 31);
  if (P.cache_dtype != NVS_DTYPE_BF16 && P.cache_dtype != NVS_DTYPE_FP16) return false;
  // The loop's cache rows (block id x block_size + offset) and the bytes of
  // a block-table row are 32-bit.
  return P.NB * (int64_t)P.bs < (1ll << 31) && 4 * P.bt_stride < (1ll << 31);
}

int launch_prefill_mx(const AttnParams& P, const Plan& plan, hipStream_t stream, const CoDecode* co,
                      const SplitJob* split) {
  MxArgs a;
  a.q = (const uint16_t*)P.q; a.q_ts = P.q_ts; a.q_hs = P.q_hs;
  a.kc = (const char*)P.kc; a.vc = (const char*)P.vc;
  a.bt = P.bt; a.bt_stride = (int)P.bt_stride; a.NB = (int)P.NB; a.bs = P.bs;
  a.k = (const char*)P.k; a.v = (const char*)P.v;
  a.k_ts = P.k_ts; a.k_hs = P.k_hs; a.v_ts = P.v_ts; a.v_hs = P.v_hs; a.Tk = P.Tk;
  a.cu_q = P.cu_q; a.cu_k = P.cu_k;
  a.Hq = P.Hq; a.Hkv = P.Hkv; a.g = P.Hq / P.Hkv;
  a.hpi = mx_heads_per_item(a.g);
  a.hgroups = (a.g + a.hpi - 1) / a.hpi;
  a.plan = plan;
  a.scale_log2 = P.softmax_scale * 1.4426950408889634f;
  a.out = (uint16_t*)P.out; a.out_ts = P.out_ts; a.out_hs = P.out_hs;
  a.gate = P.gate; a.gate_run = P.gate_run;
  if (co) {
    a.dec = co->a;
    a.dec_bt = co->bt;
    a.dec_groups = co->groups;
  } else {
    a.dec = DecodeArgs{};
    a.dec_bt = nullptr;
    a.dec_groups = 0;
  }
  if (plan.ntq <= 0 || P.B <= 0) return NVS_OK;
  if (plan.pbm != 256 / a.hpi) {
    set_error("prefill: plan tile of %d positions does not match %d heads per item", plan.pbm, a.hpi);
    return NVS_ERR_INVALID;
  }
  // The plan sized the decode part, or the entries' parts, for as many.
  const int64_t wgs = co      ? co->wgs
                      : split ? split->wgs
                              : prefill_mx_wgs((int64_t)P.B * plan.ntq * prefill_mx_units(P.Hq, P.Hkv));
  a.parts = split ? split->at.slots : nullptr;
  const PlanRecord* rec = split ? split->at.rec : plan.rec;
  const bool f16 = P.cache_dtype == NVS_DTYPE_FP16;
  const dim3 grid((unsigned)wgs), block(kMxThreads);
  const int dkv = co ? co->kv : kNoDecode;
  if (P.bt == nullptr && !f16) {
    hipLaunchKernelGGL((prefill_mx_kernel<false, false, kNoDecode>), grid, block, 0, stream, a, rec);
  } else if (P.bt == nullptr) {
    hipLaunchKernelGGL((prefill_mx_kernel<false, true, kNoDecode>), grid, block, 0, stream, a, rec);
  } else if (f16) {
    if (dkv == NVS_DTYPE_FP16)
      hipLaunchKernelGGL((prefill_mx_kernel<true, true, NVS_DTYPE_FP16>), grid, block, 0, stream, a, rec);
    else
      hipLaunchKernelGGL((prefill_mx_kernel<true, true, kNoDecode>), grid, block, 0, stream, a, rec);
  } else {
    switch (dkv) {
      case NVS_DTYPE_BF16:
        hipLaunchKernelGGL((prefill_mx_kernel<true, false, NVS_DTYPE_BF16>), grid, block, 0, stream, a, rec);
        break;
      case NVS_DTYPE_FP8_E4M3:
        hipLaunchKernelGGL((prefill_mx_kernel<true, false, NVS_DTYPE_FP8_E4M3>), grid, block, 0, stream, a, rec);
        break;
      case NVS_DTYPE_INT8:
        hipLaunchKernelGGL((prefill_mx_kernel<true, false, NVS_DTYPE_INT8>), grid, block, 0, stream, a, rec);
        break;
      default:
        hipLaunchKernelGGL((prefill_mx_kernel<true, false, kNoDecode>), grid, block, 0, stream, a, rec);
    }
  }
  return check_launch("prefill_mx");
}

}  // namespace nvs

// The decode waves' arguments and the merge of their split rows, shared by
// the decode file (the merge's own launch: decode-only calls, and calls
// whose prefill launch streamed the decode rows) and the planning kernel
// (which runs the merge beside the plan in one launch when a paged call's
// decode launch comes before prefill rows).
#pragma once

#include "nvs_common.h"
#include "attention_common.h"

namespace nvs {

struct DecodeArgs {
  const uint16_t* q;
  int64_t q_ts, q_hs;
  const void* kc;
  const void* vc;
  const float* ks;
  const float* vs;
  int bt_stride;  // row stride == number of columns
  int NB;
  int Hq, Hkv, g, bs;
  float scale_log2;
  float* ws_o;   // [max_waves, 2 slots, g, 128]
  float* ws_ml;  // [max_waves, 2 slots, g, 2]
  int32_t* ws_rec;  // [4 + 4 waves]: (T, Kw), then per wave the split row it merges
  // New tokens (bf16) stored by the decode waves themselves: copied into a
  // bf16 cache, quantised per token and kv head into an fp8 / int8 one with
  // their scales into ks / vs (kn null: none).
  const uint16_t* kn;
  const uint16_t* vn;
  int64_t kn_ts, kn_hs, vn_ts, vn_hs;
  const int32_t* slots;
  int64_t total_slots;
  const int32_t* cu_q;
  const int32_t* cu_k;
  int B;
  int64_t T;  // query / output rows
  uint16_t* out;
  int64_t out_ts, out_hs;
  int f16;  // q and out are fp16 (an fp16 cache), else bf16
};

// First tile of decode group k of Kw over T tiles.
__device__ __forceinline__ int group_start(int T, int Kw, int k) { return (int)((int64_t)k * T / Kw); }

// The merge's state of head c0 + lane / 16 + 4 i (i < NH) of a row: running
// max, sum and the lane's eight output elements, 8 (lane % 16) .. + 7.  NH
// head passes at once, so a group of more than four heads waits for its
// partials' loads once rather than once per four heads.
template <int NH>
struct MergeState {
  float M[NH], L[NH];
  f32x4 o0[NH], o1[NH];
};

template <int NH>
__device__ __forceinline__ void merge_clear(MergeState<NH>& s) {
#pragma unroll
  for (int i = 0; i < NH; ++i) {
    s.M[i] = -INFINITY;
    s.L[i] = 0.0f;
    s.o0[i] = f32x4{0.f, 0.f, 0.f, 0.f};
    s.o1[i] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
}

// Adds the partial (m, l, o0, o1) to head pass i.
template <int NH>
__device__ __forceinline__ void merge_add(MergeState<NH>& s, int i, float m, float l, f32x4 o0, f32x4 o1) {
  const float m_new = fmaxf(s.M[i], m);
  const float al = s.M[i] == -INFINITY ? 0.0f : fast_exp2(s.M[i] - m_new);
  const float be = m == -INFINITY ? 0.0f : fast_exp2(m - m_new);
  s.M[i] = m_new;
  s.L[i] = s.L[i] * al + l * be;
  s.o0[i] = s.o0[i] * al + o0 * be;
  s.o1[i] = s.o1[i] * al + o1 * be;
}

// A row split across groups k .. k_last: output row, the slot of group k's
// partial (the others' is 0).
struct MergeRow {
  int k, h, k_last, slot_k, q_row;
};

// Partials whose loads are in flight together (a run).
constexpr int kMergeRun = 4;

// Adds the partials of groups first .. k_last in runs, the next run starting
// `stride` groups after the last one's start.
template <int NH>
__device__ __forceinline__ void merge_partials(const DecodeArgs& a, const MergeRow& r, int first, int stride, int c0,
                                               int lane, MergeState<NH>& s) {
  const int j = lane & 15;
  int cc[NH];
#pragma unroll
  for (int i = 0; i < NH; ++i) {
    const int c = c0 + (lane >> 4) + 4 * i;
    cc[i] = c < a.g ? c : 0;
  }
  for (int x0 = first; x0 <= r.k_last; x0 += stride) {
    f32x2 ml[kMergeRun][NH];
    f32x4 o0[kMergeRun][NH], o1[kMergeRun][NH];
#pragma unroll
    for (int u = 0; u < kMergeRun; ++u) {
      const int x = min(x0 + u, r.k_last);
#pragma unroll
      for (int i = 0; i < NH; ++i) {
        const int64_t base = (((int64_t)x * a.Hkv + r.h) * 2 + (x == r.k ? r.slot_k : 0)) * a.g + cc[i];
        ml[u][i] = *reinterpret_cast<const f32x2*>(a.ws_ml + base * 2);
        o0[u][i] = *reinterpret_cast<const f32x4*>(a.ws_o + base * kHeadDim + 8 * j);
        o1[u][i] = *reinterpret_cast<const f32x4*>(a.ws_o + base * kHeadDim + 8 * j + 4);
      }
    }
#pragma unroll
    for (int u = 0; u < kMergeRun; ++u) {
      if (x0 + u > r.k_last) break;
#pragma unroll
      for (int i = 0; i < NH; ++i) merge_add<NH>(s, i, ml[u][i][0], ml[u][i][1], o0[u][i], o1[u][i]);
    }
  }
}

// Normalises and writes the row's heads.
template <int NH>
__device__ __forceinline__ void merge_write(const DecodeArgs& a, const MergeRow& r, int c0, int lane,
                                            const MergeState<NH>& s) {
  const int j = lane & 15;
#pragma unroll
  for (int i = 0; i < NH; ++i) {
    const int c = c0 + (lane >> 4) + 4 * i;
    if (c >= a.g) continue;
    const float inv = s.L[i] > 0.0f ? 1.0f / s.L[i] : 0.0f;
    const f32x4 x0 = s.o0[i] * inv, x1 = s.o1[i] * inv;
    u32x4 v;
    if (a.f16) {
      v[0] = pack_f16x2(x0[0], x0[1]);
      v[1] = pack_f16x2(x0[2], x0[3]);
      v[2] = pack_f16x2(x1[0], x1[1]);
      v[3] = pack_f16x2(x1[2], x1[3]);
    } else {
      v[0] = pack_bf16x2(x0[0], x0[1]);
      v[1] = pack_bf16x2(x0[2], x0[3]);
      v[2] = pack_bf16x2(x1[0], x1[1]);
      v[3] = pack_bf16x2(x1[2], x1[3]);
    }
    *reinterpret_cast<u32x4*>(a.out + (int64_t)r.q_row * a.out_ts + (int64_t)(r.h * a.g + c) * a.out_hs + 8 * j) = v;
  }
}

template <int NH>
__device__ __forceinline__ void merge_heads(const DecodeArgs& a, const MergeRow& r, int c0, int lane) {
  MergeState<NH> s;
  merge_clear<NH>(s);
  merge_partials<NH>(a, r, r.k, kMergeRun, c0, lane, s);
  merge_write<NH>(a, r, c0, lane, s);
}

// A merge work-group is sixteen waves, one unit each.  A row of up to
// kMergeAlone partials is merged by its wave; longer ones may be merged by
// teams of waves, the work-group's waves shared evenly among up to kMergeTeams
// of them at a time.
constexpr int kMergeWaves = 16;
template <int NH>
constexpr int kMergeAlone = 16 / NH;

// The most of sixteen lanes' values (>= 0), the same in each row of sixteen.
__device__ __forceinline__ int most_of_16(int x) {
  x = max(x, __builtin_amdgcn_update_dpp(0, x, 0x128, 0xf, 0xf, false));  // row_ror 8, 4, 2, 1
  x = max(x, __builtin_amdgcn_update_dpp(0, x, 0x124, 0xf, 0xf, false));
  x = max(x, __builtin_amdgcn_update_dpp(0, x, 0x122, 0xf, 0xf, false));
  x = max(x, __builtin_amdgcn_update_dpp(0, x, 0x121, 0xf, 0xf, false));
  return __builtin_amdgcn_readfirstlane(x);
}
constexpr int kMergeTeams = 4;

struct MergeLds {
  MergeRow rows[kMergeWaves];  // k_last < 0: not a row for a team
  f32x2 ml[kMergeWaves][64];
  f32x4 o[kMergeWaves][2][64];
};

// Runs of partials that a row must have more of than a team's share of it for
// the team to pay.
template <int NH>
constexpr int kTeamRuns = 4 - NH;

// Whether a row of up to max_seqlen_k keys may have so many partials that a
// team merges it (more than 16, with two head passes 12): its tiles, over
// groups of kDecodeMinUnits or more, from the last tile of one on.
inline bool merge_teams(int max_seqlen_k, int group) {
  const int64_t tiles = ((int64_t)max_seqlen_k + kDecodeTile - 1) / kDecodeTile;
  return (tiles + kDecodeMinUnits - 2) / kDecodeMinUnits + 1 >
         kMergeRun * (1 + (group <= 4 ? kTeamRuns<1> : kTeamRuns<2>));
}

// Work-groups of a merge launch of `units` groups and kv heads.
inline int merge_wgs(int units, int Hkv) { return (units / Hkv + kMergeWaves - 1) / kMergeWaves * Hkv; }

// One head pass c0 .. c0 + 4 NH - 1 of the row r by `waves` waves (this wave
// the `part`-th of them, w among the work-group's): each takes every
// waves-th run of partials, and the first adds the others' states
// through LDS and writes.  Every wave of the work-group calls it (two
// barriers a head); r.k_last < 0 adds and writes nothing.
template <int NH>
__device__ __forceinline__ void merge_pass(const DecodeArgs& a, const MergeRow& r, int w, int part, int waves, int c0,
                                           int lane, MergeLds& lds) {
  MergeState<NH> s;
  merge_clear<NH>(s);
  if (r.k_last >= 0) merge_partials<NH>(a, r, r.k + kMergeRun * part, kMergeRun * waves, c0, lane, s);
#pragma unroll
  for (int i = 0; i < NH; ++i) {
    lds.ml[w][lane] = f32x2{s.M[i], s.L[i]};
    lds.o[w][0][lane] = s.o0[i];
    lds.o[w][1][lane] = s.o1[i];
    __syncthreads();
    if (part == 0 && r.k_last >= 0)
      for (int y = 1; y < waves; ++y) {
        const f32x2 ml = lds.ml[w + y][lane];
        merge_add<NH>(s, i, ml[0], ml[1], lds.o[w + y][0][lane], lds.o[w + y][1][lane]);
      }
    __syncthreads();
  }
  if (part == 0 && r.k_last >= 0) merge_write<NH>(a, r, c0, lane, s);
}

// The row merge unit `unit` = k Hkv + h owns: kv head h of the row recorded
// by decode wave k Hkv + h (the row that crosses the boundary after group k
// and starts inside group k's range); its partials sit in wave k Hkv + h
// (the recorded slot) and in waves x Hkv + h for groups x = k + 1 .. k_last
// (slot 0).  k_last = -1: none.
__device__ __forceinline__ MergeRow merge_row(const DecodeArgs& a, int unit, int units) {
  MergeRow r = {0, 0, -1, 0, 0};
  if (unit >= units) return r;
  r.k = unit / a.Hkv;
  r.h = unit - r.k * a.Hkv;
  // Header and record in one round trip.  Groups k >= Kw - 1 merge nothing (a
  // launch may hold more merge waves than the decode had groups; their
  // records are not this call's).
  const int T = a.ws_rec[0], Kw = a.ws_rec[1];
  const int32_t* rec = a.ws_rec + 4 + 4 * unit;
  const int rec_row = rec[0], rec_tiles = rec[1], rec_slot = rec[2], rec_on = rec[3];
  asm volatile("" ::"s"(T), "s"(Kw), "s"(rec_row), "s"(rec_tiles), "s"(rec_slot), "s"(rec_on));
  if (r.k >= Kw - 1 || rec_on == 0) return r;
  r.q_row = rec_row;
  r.slot_k = rec_slot;
  const int last = group_start(T, Kw, r.k + 1) - 1 + rec_tiles;  // the row's last tile
  r.k_last = (int)(((int64_t)(last + 1) * Kw - 1) / T);
  return r;
}

// Log-sum-exp merge of the rows split across groups, by work-group `wg`
// (every wave of the work-group calls it): kv head wg % Hkv of the sixteen
// groups from 16 (wg / Hkv), one a wave, so the kv heads of one row fall to
// different work-groups and a work-group reads neighbouring groups'
// partials.  Lane l
// serves head 4 p + l / 16 of the group (pass p) and head_dim elements
// 8 (l % 16) .. + 7; a pass over the partials keeps a running max, sum and
// output, for NH head passes together (two for groups of more than four).
// What bounds it is the chain of dependent loads, 0.7 .. 1.5 us a run of four
// partials (1.3 .. 1.8 us with two head passes).  With one wave a row
// throughout, a single conversation of 20 011 keys, whose row is split across
// all 156 groups, took 62.8 us here (now 8.8).  A team costs as much as a few
// runs (barriers, the states' way through LDS), and the work-group's shorter
// rows come before it: each work-group takes teams where its longest row is
// longer than all that (kTeamRuns), and rows of up to sixteen partials (eight
// with two head passes) stay with one wave in any case (33 rows of up to 14
// partials: 8.0 us alone, 9.5 with teams from nine on; 64 rows of about 5: 7.3,
// 12.5 with teams from five on).  With teams for every row past those, whole
// calls of rows of 17 partials beside ones of 16 were 10 .. 19 % slower than one
// wave a row (6 rows of 2000 keys, 32/8 heads 25.9 us, 23.0 alone), of 9 beside
// 8 with two head passes 20 .. 45 % (12 rows of 1000 keys, 32/2 heads 30.5, 21.4).
//
// A launch whose rows cannot have enough partials for a team (merge_teams) runs
// without TEAMS: no LDS, no barrier (eight rows of 128 .. 1024 keys, GPU time of
// the call 15.85 us with both, 15.50 without).
template <int NH, bool TEAMS>
__device__ __forceinline__ void merge_split_rows(const DecodeArgs& a, int units, int wg, MergeLds* lds) {
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int k = wg / a.Hkv * kMergeWaves + w;
  const MergeRow r = merge_row(a, k * a.Hkv + wg % a.Hkv, units);
  uint32_t rest = 0;  // the rows for teams, one bit a unit, the same for every wave
  if constexpr (TEAMS) {
    if (lane == 0) lds->rows[w] = r;
    __syncthreads();
    const MergeRow& y = lds->rows[lane & (kMergeWaves - 1)];
    const int partials = y.k_last >= 0 ? y.k_last - y.k + 1 : 0;
    rest = (uint32_t)__ballot(lane < kMergeWaves && partials > kMergeAlone<NH>);
    if (rest) {
      const int n = __popc(rest), waves = n == 1 ? kMergeWaves : n == 2 ? kMergeWaves / 2 : kMergeWaves / kMergeTeams;
      const int runs = (most_of_16(partials) + kMergeRun - 1) / kMergeRun;
      const int before = (most_of_16(partials > kMergeAlone<NH> ? 0 : partials) + kMergeRun - 1) / kMergeRun;
      const int rounds = (n + kMergeTeams - 1) / kMergeTeams;
      if (runs <= before + rounds * (kTeamRuns<NH> + (runs + waves - 1) / waves)) rest = 0;
    }
  }
  if (r.k_last >= 0 && !(rest >> w & 1))
    for (int c0 = 0; c0 < a.g; c0 += 4 * NH) merge_heads<NH>(a, r, c0, lane);
  if constexpr (!TEAMS) return;
  while (rest) {
    const int n = __popc(rest);
    const int waves = n == 1 ? kMergeWaves : n == 2 ? kMergeWaves / 2 : kMergeWaves / kMergeTeams;
    const int team = w / waves;
    MergeRow x = {0, 0, -1, 0, 0};
    for (int t = 0; t < kMergeWaves / waves && rest; ++t) {
      if (t == team) x = lds->rows[__ffs(rest) - 1];
      rest &= rest - 1;
    }
    x.k = __builtin_amdgcn_readfirstlane(x.k);
    x.h = __builtin_amdgcn_readfirstlane(x.h);
    x.k_last = __builtin_amdgcn_readfirstlane(x.k_last);
    x.slot_k = __builtin_amdgcn_readfirstlane(x.slot_k);
    x.q_row = __builtin_amdgcn_readfirstlane(x.q_row);
    for (int c0 = 0; c0 < a.g; c0 += 4 * NH) merge_pass<NH>(a, x, w, w % waves, waves, c0, lane, *lds);
  }
}

// A merge left to the plan launch: the decode launch's arguments and the
// number of merge waves ((groups - 1) x Hkv; 0: no row can be split).
struct MergeJob {
  DecodeArgs a;
  int units;
};

// Decode rows streamed by the MFMA prefill launch: their arguments and
// block tables, the cache type, the decode groups the partial workspace
// holds, and the work-groups the launch runs.
struct CoDecode {
  DecodeArgs a;
  const int32_t* bt;
  int kv;
  int groups;
  int wgs;
};

}  // namespace nvs

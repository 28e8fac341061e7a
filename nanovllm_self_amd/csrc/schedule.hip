// Planning kernel: the prefill work list from cu_seqlens, on the device and
// without a host round trip.
#include "nvs_common.h"
#include "attention_common.h"
#include "decode_merge.h"
#include "store_rows.h"
#include <type_traits>

namespace nvs {

struct PlanArgs {
  const int32_t* cu_q;
  const int32_t* cu_k;
  int B;
  int64_t T;
  int paged;
  const int32_t* bt;  // paged: block tables
  int64_t bt_stride;
  int64_t NB;
  int bs;
  Plan plan;
  int* shadow_base;  // code caches: per-row first tile of the bf16 copy (null: no copy)
  int shadow_cap;
  int shadow_st;     // tiles of a table row: a row's tiles past it are not copied
  int64_t Tk;        // rows of the local k / v (local mode)
  // Decode rows streamed by the prefill launch's first work-groups (co_wgs
  // > 0: the launch's work-group count; 0: the decode has a launch of its
  // own).  The plan picks how many from the decode bytes and the prefill
  // FLOPs at the per-CU rates below.
  int co_wgs;
  int32_t* dec_rec;  // the decode waves' header (T, Kw), zeroed here: with no decode work-group the
                     // merge after the prefill launch must find no groups, not a stale count
  int Hq, Hkv;
  float dec_tile_bytes;  // HBM bytes of one 32-key decode tile over all kv heads
  float dec_cu_bps;      // decode bytes per second one CU streams beside the prefill
  float dec_hbm_bps;     // decode bytes per second of the whole chip
  float pre_cu_flops;    // prefill FLOP per second of one CU
  float dec_finish;      // the decode should end by this fraction of the call
  // Entries split along the keys or put in order (split_slots: the slots there are).
  PlanRecord* rec;  // the list's records
  SplitRow* split_rows;
  int split_slots, split_wgs;
  int units;  // units of an entry
};

// Tiles of the bf16 copy for a prefill row with kl keys.
__device__ __forceinline__ int shadow_row_tiles(const PlanArgs& a, int np, int kl) {
  return np > 0 && kl > 0 ? min((kl + kShadowTile - 1) / kShadowTile, a.shadow_st) : 0;
}

// Block id of the tile of keys [64 t, 64 t + 64) of row b: -1 past the
// row's blocks or outside the pool.
__device__ __forceinline__ int tile_block(const PlanArgs& a, int b, int kl, int t) {
  const uint32_t lb = 64u * (uint32_t)t / (uint32_t)a.bs;
  if (64 * (int64_t)t >= kl || lb >= a.bt_stride) return -1;
  const int blk = a.bt[(int64_t)b * a.bt_stride + lb];
  return (blk >= 0 && blk < a.NB) ? blk : -1;
}

// x op the value of the lanes before it, step by step within the wave (data
// parallel primitives: a step takes a few cycles where a shuffle through LDS
// takes about a hundred).  Lanes a step does not reach take 0.
template <int CTRL, int ROWS, typename T>
__device__ __forceinline__ T lanes_before(T x) {
  return __builtin_bit_cast(T, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), CTRL, ROWS, 0xf, false));
}
template <typename T, typename F>
__device__ __forceinline__ T wave_scan(T x, F op) {
  x = op(x, lanes_before<0x111, 0xf>(x));  // row_shr 1, 2, 4, 8 within 16 lanes
  x = op(x, lanes_before<0x112, 0xf>(x));
  x = op(x, lanes_before<0x114, 0xf>(x));
  x = op(x, lanes_before<0x118, 0xf>(x));
  x = op(x, lanes_before<0x142, 0xa>(x));  // row_bcast 15: rows 1 and 3
  return op(x, lanes_before<0x143, 0xc>(x));  // row_bcast 31: rows 2 and 3
}
__device__ __forceinline__ int wave_scan_add(int x) { return wave_scan(x, [](int p, int q) { return p + q; }); }
__device__ __forceinline__ int wave_total(int x) { return __builtin_amdgcn_readlane(wave_scan_add(x), 63); }
__device__ __forceinline__ int wave_most(int x) {  // of values >= 0
  return __builtin_amdgcn_readlane(wave_scan(x, [](int p, int q) { return max(p, q); }), 63);
}
__device__ __forceinline__ float wave_most(float x) {  // of values >= 0
  return __builtin_bit_cast(float, wave_most(__builtin_bit_cast(int, x)));
}
__device__ __forceinline__ float wave_total(float x) {
  x = wave_scan(x, [](float p, float q) { return p + q; });
  return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, x), 63));
}

// Inclusive scan of one int per thread over the 1024-thread work-group: a
// scan inside each wave, then the 16 wave totals through LDS.  Also returns
// the work-group total.  Two barriers.
__device__ __forceinline__ int block_scan_1024(int v, int* lds, int& total) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  v = wave_scan_add(v);
  if (lane == 63) lds[w] = v;
  __syncthreads();
  int before = 0, all = 0;
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const int x = lds[i];
    before += i < w ? x : 0;
    all += x;
  }
  __syncthreads();
  total = all;
  return v + before;
}

// Row b's work: a decode row (q_len == 1 row of a paged call) or prefill
// query tiles (every other row); also its first query row and key count.
__device__ __forceinline__ void row_work(const PlanArgs& a, int b, bool& dec, int& np, int& q0, int& kl) {
  dec = false;
  np = 0;
  q0 = kl = 0;
  if (b >= a.B) return;
  q0 = a.cu_q[b];
  const int ql = a.cu_q[b + 1] - q0;
  kl = a.cu_k[b + 1] - a.cu_k[b];
  if (q0 < 0 || ql <= 0 || (int64_t)q0 + ql > a.T) return;  // malformed rows are skipped
  if (a.paged && ql == 1)
    dec = true;
  else
    np = min((ql + a.plan.pbm - 1) / a.plan.pbm, a.plan.ntq);
}

constexpr int kPlanThreads = 1024;
constexpr int kPlanWaves = kPlanThreads / 64;
static_assert(kPlanWaves == kMergeWaves, "a work-group of the plan launch holds the merge's waves");

// Sums of three floats per thread over the 1024-thread work-group (every
// thread gets them).  Two barriers.
__device__ __forceinline__ void block_sum3_1024(float (&v)[3], float (*lds)[3]) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
#pragma unroll
  for (int i = 0; i < 3; ++i) v[i] = wave_total(v[i]);
  if (lane == 0)
    for (int i = 0; i < 3; ++i) lds[w][i] = v[i];
  __syncthreads();
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    float all = 0.0f;
#pragma unroll
    for (int x = 0; x < kPlanWaves; ++x) all += lds[x][i];
    v[i] = all;
  }
  __syncthreads();
}

// Query-key pairs of a prefill row with L new and K visible keys under the
// causal mask (row r sees keys j <= r + K - L).
__device__ __forceinline__ float causal_pairs(int L, int K) {
  const float off = (float)(K - L);
  return K >= L ? (float)L * off + 0.5f * (float)L * (float)(L + 1) : 0.5f * (float)K * (float)(K + 1);
}

// Work-groups of the prefill launch that stream the decode rows before they
// join the prefill: the fewest whose decode, at dec_cu_bps a CU and at most
// dec_hbm_bps in all, ends by dec_finish of the call's estimated time (the
// prefill's CU time, its FLOPs at pre_cu_flops a CU, plus the decode's,
// shared by all work-groups); all of them when none does; none without
// decode rows.  Counts step in multiples of 8 (as many on every XCD) and of
// 2 Hkv (an XCD's decode waves form whole groups: at 24 work-groups and Hkv
// = 8 a third of them idled) when the launch holds such a step.
__device__ int pick_decode_wgs(const PlanArgs& a, float dec_rows, float dec_tiles, float pairs) {
  if (a.co_wgs <= 0 || dec_rows <= 0.0f) return 0;  // a keyless decode row still needs its zeros
  const int top = a.co_wgs & ~7;
  int step = 8;
  while (step % (2 * a.Hkv) != 0 && step <= top) step += 8;
  if (step > top) step = 8;
  const int lo = min(top, max(step, (2 * a.Hkv + 7) & ~7));
  const float bytes = dec_tiles * a.dec_tile_bytes;
  const float pre = pairs * 4.0f * (float)a.Hq * (float)kHeadDim / a.pre_cu_flops;  // CU seconds
  for (int nd = lo; nd <= top; nd += step) {
    const float td = bytes / fminf((float)nd * a.dec_cu_bps, a.dec_hbm_bps);
    const float t = (pre + (float)nd * td) / (float)a.co_wgs;
    if (td <= a.dec_finish * t) return nd;
  }
  return top;
}

// A row of the batch, as its entries need it.
struct RowFields {
  int b, q0, L, k0, K;
};

// The record of the entry of query tile qt (kv tiles t0 .. t1 of the row's
// visible ones), from its row.
__device__ __forceinline__ PlanRecord make_record(const PlanArgs& a, const RowFields& r, bool shadow, const int (&blk)[3],
                                                  int qt, int t0, int nt, int part) {
  PlanRecord rec;
  rec.part = part;
  rec.q0 = r.q0;
  rec.L = r.L;
  rec.k0 = r.k0;
  rec.K = r.K;
  rec.blk0 = blk[0];
  rec.blk1 = blk[1];
  rec.blk2 = blk[2];
  rec.off = r.K - r.L - 64 * t0;
  rec.b = r.b;
  if (a.paged) {
    const uint32_t tbs = shadow ? kShadowTile : a.bs;
    const uint32_t tst = shadow ? a.shadow_st : (uint32_t)a.bt_stride;
    rec.k0c = 0;
    rec.kf = r.K - 64 * t0;
    rec.bt_off = (int)(4 * (64 * (uint32_t)t0 / tbs));
    // None of a part that starts past the table row (more keys than it has
    // blocks for): they read as missing.
    rec.bt_bytes = max(0, (int)(4 * min(((uint32_t)max(r.K, 0) + tbs - 1) / tbs, tst)) - rec.bt_off);
  } else {
    const int64_t k0c = min(max((int64_t)r.k0, (int64_t)0), a.Tk);
    rec.k0c = (int)k0c + 64 * t0;
    rec.kf = (int)max((int64_t)0, min((int64_t)r.K, a.Tk - k0c)) - 64 * t0;
    rec.bt_off = rec.bt_bytes = 0;
  }
  rec.p0 = qt * a.plan.pbm;
  rec.ntiles = nt;
  return rec;
}

// Visible key tiles of query tile qt of a row, and those its first position
// sees a key of.
__device__ __forceinline__ int entry_tiles(const PlanArgs& a, int L, int K, int qt, int& first_sees) {
  const int p0 = qt * a.plan.pbm, off = K - L;
  const int kv_end = min(K, min(L, p0 + a.plan.pbm) + off);
  first_sees = p0 + off >= 0 ? (p0 + off) / 64 + 1 : 0;
  return (p0 < L && kv_end > 0) ? (kv_end + 63) / 64 : 0;
}

// ceil(x / y), 0 <= x < 2^20, y > 0: exact (the quotient's estimate is off
// by less than one).  The plan is a chain of dependent steps of one
// work-group: it avoids integer divisions, LDS reads that wait for each other
// and shuffles (six turns of 44 .. 294 tokens over cached ones, 18 entries:
// 13.8 us with the write, 11.1 without them; 552 entries: 8.0, 7.1).
__device__ __forceinline__ int ceil_div(int x, int y) {
  int q = (int)((float)x * __builtin_amdgcn_rcpf((float)y));
  q += q * y < x;
  q -= (q - 1) * y >= x;
  return q;
}

// An entry of nt key tiles in parts of at most about C: their tiles each
// (whole blocks of `step` tiles) and their number.  Every row sees a key of
// every part (first_sees: tiles the entry's first position sees a key of), so
// no row of a part stays without a running max.
__device__ __forceinline__ int part_tiles(int nt, int first_sees, int C, int step, int& parts) {
  const int most = max(1, ceil_div(nt, C));
  const int each = max(1, ceil_div(ceil_div(nt, most), step) * step);
  parts = max(1, min(ceil_div(nt, each), ceil_div(first_sees, each)));
  return each;
}

// Tiles a part may have at most, in rising order (8, 10, 12, 14, 16, 20, ..,
// 80, 96: four steps an octave); the last choice: no parts.  One a wave.
constexpr int kPartChoices = kPlanWaves;
__device__ __forceinline__ int part_choice(int i) {
  return i == kPartChoices - 1 ? 1 << 20 : (4 + (i & 3)) << (1 + (i >> 2));
}

// What the plan keeps of each row of a 1024-row step in LDS while the
// step's list entries are written, one entry per thread.
struct PlanRows {
  int end[kPlanThreads];  // inclusive prefix of the rows' entry counts
  int q0[kPlanThreads], L[kPlanThreads], k0[kPlanThreads], K[kPlanThreads];
  int blk[3][kPlanThreads];
};

// Entries weighed for a split: row, key tiles, tiles the first position sees
// (then the first slot, -1: none), tiles of a part and parts; what the
// buckets of part sizes hold, then their next place in the list; the list's
// places (entry << 10 | part).
constexpr int kPartBuckets = 64;
struct PlanEntries {
  int row[kSplitMaxEntries], nt[kSplitMaxEntries], sees[kSplitMaxEntries];
  int each[kSplitMaxEntries], parts[kSplitMaxEntries];
  int place[kSplitMaxEntries + kSplitSlots];
  float cost[kPartChoices];
  int tiles[kPlanWaves], deepest[kPlanWaves];  // of the waves' entries
  float load[kPlanWaves];
  int bucket[kPartBuckets];
  int longest, list, slots, rows;
};

// Estimated times of the call's prefill, in key tiles of a work-group that runs
// alone (1.06 us).  Two things bound it: the most tiles that one work-group
// gets, each unit with kPartSetup tiles' worth of set-up and output, and what
// the chip gets through, all the units' tiles at kPartBusy times an even
// share (256 work-groups at once take 1.6 us a tile; half as many, 1.1).
// Where the two are near each other each slows the other down (part_time).  A
// part's slot is written and read once (132 KiB each way): kPartMerge.
//
// Fitted to 312 batches (8/1, 16/8, 32/8 and 64/8 heads, 1 .. 32 rows of 4 ..
// 4000 tokens over 0 .. 16 K cached ones) with every choice of parts timed:
// the mean error is 4 %.  Before, a tile cost the same however many
// work-groups ran, and 123 of those batches were slower in their parts, or
// sorted, than row by row (32 turns of 200 tokens over 3 K, 32/8 heads: 441
// us, 362 row by row; 12 of 40 over 1.5 K: 64.7, 46.4).
constexpr float kPartSetup = 5.2f;
constexpr float kPartBusy = 1.54f;
constexpr float kPartMerge = 0.036f;
constexpr float kPartLaunch = 1.2f;
__device__ __forceinline__ float part_time(float most, float chip) {
  const float hi = fmaxf(most, chip), lo = fminf(most, chip);
  return hi + 0.26f * lo * lo * lo * __builtin_amdgcn_rcpf(hi * hi);
}

// The choices are weighed (2.5 us more of the plan) where parts or another
// order could bring a batch's time in row order down by more than kPartEarly
// and a fiftieth of it, and the best of them is taken where it is kPartWorth
// below the row order.
constexpr float kPartEarly = 8.0f;
constexpr float kPartWorth = 1.0f;

// The estimate for whole entries in row order, what no choice gets below, and
// (chip) the time of all tiles at the chip's rate; every thread calls it, after
// a barrier that follows the entries' writes.  The first three rounds of units
// are dealt by number (unit 8 k + x to work-group k of XCD x, back and forth);
// past them, the even share and half of the deepest entry of the last round.
__device__ __forceinline__ float row_order_cost(const PlanArgs& a, PlanEntries& ent, int entries, int wgs,
                                                float& least, float& chip) {
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int units = entries * a.units, most = wgs >> 3;  // at most 128 work-groups of an XCD
  const int j = lane & (kPlanWaves - 1);
  const int of_wave = ent.tiles[j];
  const int longest = wave_most(ent.deepest[j]);
  const float tiles = (float)wave_total(lane < kPlanWaves ? of_wave : 0) * a.units;
  const float each = __builtin_amdgcn_rcpf((float)wgs);
  const float share = (tiles + kPartSetup * units) * each;
  chip = kPartBusy * tiles * each;
  float load = (float)longest + kPartSetup;
  if (units > 8 * most) {
    float mine = 0.0f;
    if (tid < 8 * most) {
      const int x = tid & 7, k = tid >> 3;
#pragma unroll
      for (int i = 0; i < 3; ++i) {
        const int unit = 8 * (i * most + (i == 1 ? most - 1 - k : k)) + x;
        if (unit < units) mine += (float)ent.nt[ceil_div(unit + 1, a.units) - 1] + kPartSetup;
      }
    }
    // Past three rounds: entries from `last` on are the last round's.
    const int last = units > 24 * most ? entries - ceil_div(wgs, a.units) : entries;
    if (tid >= last && tid < entries) mine = fmaxf(mine, share + 0.5f * ((float)ent.nt[tid] + kPartSetup));
    mine = wave_most(mine);
    if (lane == 0) ent.load[w] = mine;
    __syncthreads();
    load = wave_most(ent.load[j]);
  }
  least = part_time(fmaxf(share, (float)min(longest, kSplitMinTiles) + kPartSetup), chip);
  return part_time(load, chip);
}

// The estimate for parts of at most C tiles, dealt longest first, by one wave
// over all entries; infinite where the parts need more slots than there are.
// Up to three rounds of units the deal is followed; past them, the even share
// and some of the longest.
constexpr float kPartUneven = 0.3f;
__device__ __forceinline__ float part_cost(const PlanArgs& a, const PlanEntries& ent, int* hist, int entries, int C,
                                           int step, int wgs, float chip, int lane) {
  int units = 0, slots = 0, longest = 0;
#pragma unroll 1
  for (int e = lane; e < entries; e += 64) {
    int parts;
    const int nt = ent.nt[e], each = part_tiles(nt, ent.sees[e], C, step, parts);
    units += parts;
    if (parts > 1) slots += parts;
    longest = max(longest, parts > 1 ? max(each, nt - (parts - 1) * each) : nt);
  }
  const int pieces = wave_total(units);
  units = pieces * a.units;
  slots = wave_total(slots) * a.units;
  longest = wave_most(longest);
  if (slots > a.split_slots) return INFINITY;
  const float merge = slots > 0 ? kPartLaunch + kPartMerge * slots : 0.0f;
  const int most = wgs >> 3;  // work-groups of an XCD
  if (units > 24 * most) {
    const float one = (float)longest + kPartSetup;
    const float share = chip * (1.0f / kPartBusy) + kPartSetup * units * __builtin_amdgcn_rcpf((float)wgs);
    return merge + part_time(fmaxf(one, share + kPartUneven * one), chip);
  }
  // Pieces by size, longest first: 64 buckets, then how many there are up to
  // each (the wave's own LDS: its operations complete in order).
  const float scale = 64.0f * __builtin_amdgcn_rcpf((float)(longest + 1));
  hist[lane] = 0;
  __builtin_amdgcn_wave_barrier();
#pragma unroll 1
  for (int e = lane; e < entries; e += 64) {
    int parts;
    const int nt = ent.nt[e], each = part_tiles(nt, ent.sees[e], C, step, parts);
    const int last = parts > 1 ? nt - (parts - 1) * each : nt;
    atomicAdd(&hist[min(63, (int)((float)(longest - last) * scale))], 1);
    if (parts > 1) atomicAdd(&hist[min(63, (int)((float)(longest - each) * scale))], parts - 1);
  }
  __builtin_amdgcn_wave_barrier();
  const int upto = wave_scan_add(hist[lane]);
  hist[lane] = upto;
  __builtin_amdgcn_wave_barrier();
  int piece[3], b[3] = {0, 0, 0};  // the first bucket that reaches past the piece
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    const int unit = 8 * (i * most + (i == 1 ? most - 1 - lane : lane));
    piece[i] = lane < most && unit < units ? ceil_div(unit + 1, a.units) - 1 : -1;
  }
#pragma unroll
  for (int s = 32; s >= 1; s >>= 1)
#pragma unroll
    for (int i = 0; i < 3; ++i)
      if (hist[b[i] + s - 1] <= piece[i]) b[i] += s;
  float load = 0.0f;
#pragma unroll
  for (int i = 0; i < 3; ++i)
    if (piece[i] >= 0) load += (float)longest - (float)b[i] * (1.0f / 64.0f) * (float)(longest + 1) + kPartSetup;
  return merge + part_time(wave_most(load), chip);
}

// The list of a batch of one step of rows (in `rows`, tot entries), longest
// units first, its entries split along the keys where that ends sooner.
// Returns the list's length, or -1, with nothing written, where the row order
// is as good: neighbouring units of a row share its keys in L2.  Every thread
// calls it.  A batch of more than kSplitMaxUnits units keeps the row order.
//
// Measured (the prefill kernel alone): six turns of 44 .. 294 tokens over
// 2 .. 16 K cached ones (32 / 8 heads, 144 units of 33 .. 249 tiles) unsplit
// 302 us, bound by the longest unit; in parts of up to 20, 28, 40, 56 and 92
// tiles 135, 151, 136, 150 and 139 us, and 14, 12, 9, 6 and 4 us of merge.
// Four prompts of 0.7 .. 1.2 K over up to 3.8 K cached (488 units of up to 75
// tiles, fp8): row by row 194 us, longest first 178, in parts of 64 171.
__device__ int plan_parts(const PlanArgs& a, const PlanRows& rows, PlanEntries& ent, bool shadow, int tot, int wgs) {
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int step = (a.paged && !shadow) ? a.bs / 64 : 1;
  int r = 0, qt = 0, nt = 0, sees = 0;
  if (tid < tot) {
    int hi = a.B - 1;
    while (r < hi) {
      const int mid = (r + hi) >> 1;
      if (rows.end[mid] > tid) hi = mid; else r = mid + 1;
    }
    qt = rows.end[r] - 1 - tid;
    nt = entry_tiles(a, rows.L[r], rows.K[r], qt, sees);
    ent.row[tid] = r;
    ent.nt[tid] = nt;
    ent.sees[tid] = sees;
  }
  const int wave_tiles = wave_total(nt), wave_deepest = wave_most(nt);
  if (lane == 0) {
    ent.tiles[w] = wave_tiles;
    ent.deepest[w] = wave_deepest;
  }
  if (tid < kPartBuckets) ent.bucket[tid] = 0;
  if (tid == kPartBuckets) ent.longest = ent.slots = ent.rows = 0;
  __syncthreads();
  float least, chip;
  const float row_order = row_order_cost(a, ent, tot, wgs, least, chip);
  if (0.98f * row_order <= least + kPartEarly) return -1;
  {
    const float c = part_cost(a, ent, ent.place + 64 * w, tot, part_choice(w), step, wgs, chip, lane);
    if (lane == 0) ent.cost[w] = c;
  }
  __syncthreads();
  // The least cost (the most parts' size of equal ones), by every wave.
  const float worth = 1.0f / (1.0f + (lane < kPartChoices ? ent.cost[lane] : INFINITY));
  const float top = wave_most(worth);
  const int best = 63 - __builtin_clzll(__ballot(lane < kPartChoices && worth == top));
  if (row_order <= ent.cost[best] + kPartWorth) return -1;
  int parts = 0, each = 0;
  if (tid < tot) {
    each = part_tiles(nt, sees, part_choice(best), step, parts);
    if (parts == 1) each = nt;
    ent.each[tid] = each;
    ent.parts[tid] = parts;
    atomicMax(&ent.longest, max(each, nt - (parts - 1) * each));
    int slot = -1;
    if (parts > 1) {
      slot = atomicAdd(&ent.slots, parts) * a.units;
      a.split_rows[atomicAdd(&ent.rows, 1)] = {slot, parts, rows.q0[r], rows.L[r], qt * a.plan.pbm};
    }
    ent.sees[tid] = slot;
  }
  __syncthreads();
  // Places by size, longest first, to a 64th of the longest (a 16th: 0.2 %
  // slower over the batches); an entry's last part by its own size, as the cost
  // has it.  Which of two parts of one bucket comes first, and the slots they
  // take, change with the run; their outputs do not.
  int bk = 0, bk_last = 0;
  const int last = nt - (parts - 1) * each;
  if (tid < tot) {
    const float scale = (float)kPartBuckets / (float)(ent.longest + 1);
    bk = min(kPartBuckets - 1, (int)((float)(ent.longest - each) * scale));
    bk_last = min(kPartBuckets - 1, (int)((float)(ent.longest - last) * scale));
    if (parts > 1) atomicAdd(&ent.bucket[bk], parts - 1);
    atomicAdd(&ent.bucket[bk_last], 1);
  }
  __syncthreads();
  if (tid < kPartBuckets) {
    const int n = ent.bucket[tid], end = wave_scan_add(n);
    ent.bucket[tid] = end - n;
    if (tid == kPartBuckets - 1) {
      ent.list = end;
      a.plan.hdr->n_split = ent.rows;
    }
  }
  __syncthreads();
  if (tid < tot) {
    const int at = parts > 1 ? atomicAdd(&ent.bucket[bk], parts - 1) : 0;
    const int at_last = atomicAdd(&ent.bucket[bk_last], 1);
#pragma unroll 1
    for (int c = 0; c < parts - 1; ++c) ent.place[at + c] = tid << 10 | c;
    ent.place[at_last] = tid << 10 | (parts - 1);
  }
  __syncthreads();
  const int list = ent.list;
#pragma unroll 1
  for (int i = tid; i < list; i += kPlanThreads) {
    const int e = ent.place[i] >> 10, c = ent.place[i] & 1023;
    const int b = ent.row[e];
    const RowFields row = {b, rows.q0[b], rows.L[b], rows.k0[b], rows.K[b]};
    const int n = ent.parts[e], tiles = ent.each[e], t0 = c * tiles;
    int blk[3];
    for (int t = 0; t < 3; ++t) {
      if (c == 0)
        blk[t] = rows.blk[t][b];
      else if (shadow)
        blk[t] = t0 + t < shadow_row_tiles(a, 1, row.K) ? a.shadow_base[b] + t0 + t : -1;
      else
        blk[t] = a.paged ? tile_block(a, b, row.K, t0 + t) : -1;
    }
    a.rec[i] = make_record(a, row, shadow, blk, rows.end[b] - 1 - e, t0, c == n - 1 ? ent.nt[e] - t0 : tiles,
                           n > 1 ? ent.sees[e] + c * a.units : -1);
  }
  return list;
}

template <bool PARTS>
struct PlanLds {
  struct NoEntries {};
  PlanRows rows;
  int scan[kPlanWaves];
  float sum[kPlanWaves][3];
  int decode;  // whether the batch has decode rows
  std::conditional_t<PARTS, PlanEntries, NoEntries> entries;
};

// The plan, by one work-group.
template <bool PARTS>
__device__ __forceinline__ void write_plan(const PlanArgs& a, PlanLds<PARTS>& lds) {
  int* scan_lds = lds.scan;
  float (*sum_lds)[3] = lds.sum;
  PlanRows& rows = lds.rows;
  const int tid = threadIdx.x;
  const Plan& pl = a.plan;
  if (tid < 8) pl.hdr->prefill_next[tid] = 0;
  if (tid == 0) lds.decode = 0;
  __syncthreads();
  if (!PARTS && tid == 0) pl.hdr->n_split = 0;
  // ---- code caches: the prefill rows' 64-key tiles of the bf16 copy, row
  // by row (an exclusive scan of ceil(k_len / 64)); the copy serves the call
  // if they fit.
  bool shadow = false;
  if (a.shadow_base) {
    int sbase = 0;
    for (int b0 = 0; b0 < a.B; b0 += kPlanThreads) {
      bool dec;
      int np, q0, kl, tot;
      row_work(a, b0 + tid, dec, np, q0, kl);
      const int nt = shadow_row_tiles(a, np, kl);
      const int incl = block_scan_1024(nt, scan_lds, tot);
      if (b0 + tid < a.B) a.shadow_base[b0 + tid] = sbase + incl - nt;
      sbase += tot;
    }
    shadow = sbase <= a.shadow_cap;
    if (tid == 0) {
      a.shadow_base[a.B] = sbase;
      pl.hdr->shadow_tiles = sbase;
      pl.hdr->shadow_on = shadow ? 1 : 0;
    }
  } else if (tid == 0) {
    pl.hdr->shadow_tiles = 0;
    pl.hdr->shadow_on = 0;
  }
  // ---- prefill tiles row by row (1024 rows per step: a scan of the rows'
  // tile counts), each row's tiles deepest first (most keys under the causal
  // mask).  Row-major order keeps the work-groups of an XCD on the same
  // sequence at the same time, so the K/V tiles they all read come from HBM
  // once and from L2 after that.  Each thread then writes entries e, e +
  // 1024, ... of the step, finding its row by a binary search of the prefix.
  int base = 0;
  // this thread's rows: decode rows and their tiles, prefill query-key pairs
  float dec_rows = 0.0f, dec_tiles = 0.0f, pairs = 0.0f;
  bool parted = false;
  int entries = 0;
  // The list entries of the rows in LDS (from row b0, tot entries), row by row.
  const auto write_rows = [&](int b0, int tot) {
#pragma unroll 1
    for (int e = tid; e < tot; e += kPlanThreads) {
      int lo = 0, hi = min(kPlanThreads, a.B - b0) - 1;  // the first row whose prefix passes e
      while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        if (rows.end[mid] > e) hi = mid; else lo = mid + 1;
      }
      const int r = lo, rb = b0 + r;
      const int qt = rows.end[r] - 1 - e;  // the row's first entry is its deepest tile
      const RowFields row = {rb, rows.q0[r], rows.L[r], rows.k0[r], rows.K[r]};
      const int blk[3] = {rows.blk[0][r], rows.blk[1][r], rows.blk[2][r]};
      int sees;
      pl.plist[base + e] = rb * pl.ntq + qt;
      a.rec[base + e] = make_record(a, row, shadow, blk, qt, 0, entry_tiles(a, row.L, row.K, qt, sees), -1);
    }
  };
  for (int b0 = 0; b0 < a.B; b0 += kPlanThreads) {
    bool dec;
    int np, q0, kl, tot;
    const int b = b0 + tid;
    row_work(a, b, dec, np, q0, kl);
    if (dec) {
      dec_rows += 1.0f;
      lds.decode = 1;
    }
    if (dec && kl > 0) dec_tiles += (float)((kl + kDecodeTile - 1) / kDecodeTile);
    if (np > 0) pairs += causal_pairs(a.cu_q[b + 1] - q0, kl);
    const int incl = block_scan_1024(np, scan_lds, tot);
    rows.end[tid] = incl;
    if (np > 0) {
      rows.q0[tid] = q0;
      rows.L[tid] = a.cu_q[b + 1] - q0;
      rows.k0[tid] = a.cu_k[b];
      rows.K[tid] = kl;
      if (shadow) {  // tiles of the copy (the thread wrote shadow_base[b] itself)
        const int sb = a.shadow_base[b], nt = shadow_row_tiles(a, np, kl);
        for (int t = 0; t < 3; ++t) rows.blk[t][tid] = t < nt ? sb + t : -1;
      } else {
        for (int t = 0; t < 3; ++t) rows.blk[t][tid] = a.paged ? tile_block(a, b, kl, t) : -1;
      }
    }
    __syncthreads();
    if constexpr (PARTS) {
      parted = a.B <= kPlanThreads && tot > 0 && tot <= kSplitMaxEntries && tot * a.units <= kSplitMaxUnits &&
               (!a.shadow_base || shadow);
      if (parted) {  // written below
        entries = tot;
        break;
      }
    }
    write_rows(b0, tot);
    __syncthreads();  // the next step's rows overwrite the LDS
    base += tot;
  }
  int dec_wgs = 0;
  if (a.co_wgs > 0 && tid < 2) a.dec_rec[tid] = 0;
  if (a.co_wgs > 0 && lds.decode) {  // the same for every thread
    float sums[3] = {dec_rows, dec_tiles, pairs};
    block_sum3_1024(sums, sum_lds);
    dec_wgs = pick_decode_wgs(a, sums[0], sums[1], sums[2]);
  }
  if constexpr (PARTS) {
    // The work-groups that stream decode rows join late.
    if (parted) {
      base = plan_parts(a, rows, lds.entries, shadow, entries, a.co_wgs > 0 ? max(8, a.co_wgs - dec_wgs) : a.split_wgs);
      parted = base >= 0;
      if (!parted) {
        base = 0;
        write_rows(0, entries);
        base = entries;
      }
    }
    if (!parted && tid == 0) pl.hdr->n_split = 0;
  }
  if (tid == 0) {
    pl.hdr->n_prefill = base;
    pl.hdr->dec_wgs = dec_wgs;
  }
}

// Work-group 0 writes the plan; the others (a paged call whose decode
// launch left its merge to this one) merge the decode rows split across
// groups, one merge wave per wave.
template <int NH>
__global__ __launch_bounds__(kPlanThreads) void plan_kernel(PlanArgs a, DecodeArgs m, int merge_units) {
  __shared__ union Lds {
    PlanLds<false> plan;
    MergeLds merge;
  } lds;
  if (blockIdx.x > 0)
    merge_split_rows<NH, true>(m, merge_units, (int)blockIdx.x - 1, &lds.merge);
  else
    write_plan<false>(a, lds.plan);
}

template <bool PARTS>
__global__ __launch_bounds__(kPlanThreads) void plan_only_kernel(PlanArgs a) {
  __shared__ PlanLds<PARTS> lds;
  write_plan<PARTS>(a, lds);
}

// The plan by work-group 0 and the write of the step's k / v by the others:
// neither reads what the other writes, and a small step's write (5 us) and
// plan (4 .. 13 us) are each mostly latency.  Chosen for writes of up to four
// work-groups a CU (the whole call, 32/8 heads, prompts of 250 tokens; a launch
// of its own and here: 250 tokens 19.0 and 16.8 us, 4000 (500 work-groups) 38.7
// and 35.0, 8000 (1000) 64.4 and 59.0; over fp8 4000 41.3 and 37.5, 8000 64.9
// and 63.1, 12 000 88.0 and 88.6).
template <bool PARTS, int SRC, int DST>
__global__ __launch_bounds__(kPlanThreads) void plan_store_kernel(PlanArgs a, StoreArgs st) {
  __shared__ PlanLds<PARTS> lds;
  if (blockIdx.x > 0)
    store_rows<SRC, DST, false, true>(st, (int64_t)(blockIdx.x - 1) * kPlanThreads + threadIdx.x);
  else
    write_plan<PARTS>(a, lds);
}

// The element types the plan launch writes.
static bool plan_stores(const StoreJob& job) {
  const int s = job.src, d = job.dst;
  return (s == NVS_DTYPE_FP16 && d == NVS_DTYPE_FP16) ||
         (s == NVS_DTYPE_BF16 && (d == NVS_DTYPE_BF16 || d == NVS_DTYPE_FP8_E4M3 || d == NVS_DTYPE_INT8));
}
static int64_t store_wgs(const StoreJob& job) {
  return ((job.a.rows << job.a.lpr_log2) + kPlanThreads - 1) / kPlanThreads;
}
bool plan_launch_stores(const StoreJob& job) { return plan_stores(job) && store_wgs(job) <= device_slots(4); }

template <bool PARTS>
static void launch_plan_store(const PlanArgs& a, const StoreJob& job, hipStream_t stream) {
  const dim3 grid((unsigned)(1 + store_wgs(job))), block(kPlanThreads);
  if (job.src == NVS_DTYPE_FP16)
    hipLaunchKernelGGL((plan_store_kernel<PARTS, NVS_DTYPE_FP16, NVS_DTYPE_FP16>), grid, block, 0, stream, a, job.a);
  else if (job.dst == NVS_DTYPE_BF16)
    hipLaunchKernelGGL((plan_store_kernel<PARTS, NVS_DTYPE_BF16, NVS_DTYPE_BF16>), grid, block, 0, stream, a, job.a);
  else if (job.dst == NVS_DTYPE_FP8_E4M3)
    hipLaunchKernelGGL((plan_store_kernel<PARTS, NVS_DTYPE_BF16, NVS_DTYPE_FP8_E4M3>), grid, block, 0, stream, a,
                       job.a);
  else
    hipLaunchKernelGGL((plan_store_kernel<PARTS, NVS_DTYPE_BF16, NVS_DTYPE_INT8>), grid, block, 0, stream, a, job.a);
}

static int g_cus[64] = {0};

int device_slots(int per_cu) {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) dev = 0;
  if (g_cus[dev] == 0) {
    int n = 0;
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0)
      n = 256;
    g_cus[dev] = n;
  }
  return g_cus[dev] * per_cu;
}

int launch_plan(const AttnParams& P, const Plan& plan, bool paged, hipStream_t stream, const ShadowLayout* shadow,
                const MergeJob* merge, const CoDecode* co, const SplitJob* split,
                const StoreJob* store) {
  PlanArgs a;
  a.cu_q = P.cu_q;
  a.cu_k = P.cu_k;
  a.B = P.B;
  a.T = P.T;
  a.paged = paged ? 1 : 0;
  a.bt = P.bt;
  a.bt_stride = P.bt_stride;
  a.NB = P.NB;
  a.bs = P.bs > 0 ? P.bs : 64;
  a.plan = plan;
  a.shadow_base = shadow ? shadow->base : nullptr;
  a.shadow_cap = shadow ? shadow->cap : 0;
  a.shadow_st = shadow ? shadow->ST : 0;
  a.Tk = P.Tk;
  a.rec = split ? split->at.rec : plan.rec;
  a.split_rows = split ? split->at.rows : nullptr;
  a.split_slots = split ? split->slots : 0;
  a.split_wgs = split ? split->wgs : 0;
  a.units = prefill_mx_units(P.Hq, P.Hkv);
  a.co_wgs = co ? co->wgs : 0;
  a.dec_rec = co ? co->a.ws_rec : nullptr;
  a.Hq = P.Hq;
  a.Hkv = P.Hkv;
  const float esz = (P.cache_dtype == NVS_DTYPE_BF16 || P.cache_dtype == NVS_DTYPE_FP16) ? 2.0f : 1.0f;
  a.dec_tile_bytes = (float)kDecodeTile * P.Hkv * (2.0f * kHeadDim * esz + (esz < 2.0f ? 8.0f : 0.0f));
  const CoDecodeRates r = co_decode_rates(P.cache_dtype);
  a.dec_cu_bps = r.cu_bps;
  a.dec_hbm_bps = r.hbm_bps;
  a.pre_cu_flops = r.pre_cu_flops;
  a.dec_finish = r.finish;
  DecodeArgs m = {};
  int units = 0;
  if (merge && merge->units > 0) {
    m = merge->a;
    units = merge->units;
  }
  const int grid = 1 + (units > 0 ? merge_wgs(units, m.Hkv) : 0);
  const bool parts = split != nullptr;
  const dim3 one(1), block(kPlanThreads);
  if (store)
    parts ? launch_plan_store<true>(a, *store, stream) : launch_plan_store<false>(a, *store, stream);
  else if (parts)
    hipLaunchKernelGGL(plan_only_kernel<true>, one, block, 0, stream, a);
  else if (units > 0)
    hipLaunchKernelGGL(m.g <= 4 ? plan_kernel<1> : plan_kernel<2>, dim3(grid), block, 0, stream, a, m, units);
  else
    hipLaunchKernelGGL(plan_only_kernel<false>, one, block, 0, stream, a);
  return check_launch("plan");
}

}  // namespace nvs

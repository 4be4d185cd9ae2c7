// The planner: from tokens-per-expert counts to the tables of one fused launch, by one workgroup in device memory.
#pragma once
#include <hip/hip_runtime.h>

#include <type_traits>

#include "../../../include/mxmoe_amd.h"
#include "mxmoe_launch.hpp"
#include "mxmoe_perm.hpp"
#include "mxmoe_plan.hpp"

namespace mxmoe {

// A block descriptor (not the QParams arrays of the launcher, whose padding bytes belong to the caller) may name an operand variant
// in q._pad[0]: 1 = the int4 codes of per-token activations as bf6 fragments (for the kernels whose w4a4 tiles run on the 6-bit float
// matrix path), 2 = per-token fp8 e4m3 codes instead of int8 ones (for the kernels whose w8a8 tiles run the fp8 instruction).
__host__ __device__ inline bool wants_bf6(const mxmoe_qparams& q) { return q._pad[0] == 1 && q.a_bits == 4 && q.w_bits == 4 && q.gsize == -1; }
__host__ __device__ inline bool wants_fp8(const mxmoe_qparams& q) { return q._pad[0] == 2 && q.a_bits == 8 && q.w_bits == 8 && q.gsize == -1; }

__host__ __device__ inline int act_tag_of(const mxmoe_qparams& q) {  // ref_bind.cu:461-473
  if (q.a_bits >= 16) return 0;
  if (wants_fp8(q)) return 5;
  if (q.a_bits == 8 && q.gsize == -1) return 1;
  if (wants_bf6(q)) return 4;
  if (q.a_bits == 4 && q.gsize == -1) return 2;
  if (q.a_bits == 4 && q.gsize == 128) return 3;
  return -1;
}

__host__ __device__ inline int fmt_of(const mxmoe_qparams& q) { return (int)classify(q); }

constexpr int kNumTags = 6;

// How a block's operands are laid out.
//   kPlain    activations as rows sorted by expert, the output as the GEMM's [rows, N] (the operators' layout);
//   kGateUp   the gate_up form of the tiles (TileArgs): activations are one store per tag that holds every token once, each problem
//             reads them through its part of `token_of_row` (the shared expert through `iota`), the output is [rows, N / 2];
//   kBehind   the block behind a gate_up form: as kPlain, but fp16 activations are read where that form left them (`act`).
struct LayerForm {
  enum Kind { kPlain = 0, kGateUp = 1, kBehind = 2 };
  int kind;
  const uint8_t* store[kNumTags];
  const uint8_t* scales[kNumTags];
  const int32_t* token_of_row;
  const int32_t* iota;
  const uint8_t* act;
};

struct PlanParams {
  const int64_t* recv;
  const mxmoe_block_desc* desc;
  const uint8_t* inp;
  const uint8_t* scale;
  uint8_t* out;
  uint8_t* plan;
  int E, Et, shared_rows;
  LayerForm form;
  PlanInfo info;
};

// The branch table a block is planned with.  Which experts get rows is not known here, so all of them count as blocks of the launch.
inline PlanInfo plan_info_of_block(const FusedKernel& k, const mxmoe_block_desc* h_desc, int et) {
  PlanInfo info = plan_of(k);
  long blocks = 0;
  bool w8a16 = false;
  for (int i = 0; i < et; ++i) {
    blocks += (h_desc[i].N + 255) / 256;
    w8a16 = w8a16 || fmt_of(h_desc[i].q) == (int)Fmt::W8A16;
  }
  info.few_blocks = info.narrow && blocks <= kPoleBlocks;
  if (!w8a16) info.has_slim = 0;  // (nothing to look for)
  for (int i = 1; i < et; ++i) info.unequal_k |= h_desc[i].K != h_desc[0].K;
  return info;
}

constexpr int kPlanThreads = 128;
constexpr int kMaxPlannedProblems = 4096;  // experts of a planned block (run as launches of kMaxProblems experts each)
static_assert(kMaxProblems <= kPlanThreads, "one thread per problem");
static_assert(kMaxBranches <= 64, "one lane per branch");

struct PlanPair {
  PlanParams p[2];
  int chunks;  // launches per block
  // Whether either block's tile shapes hang on its launch's totals (plan_block_body's TOTALS).
  bool totals() const { return p[0].info.may_pair || p[0].info.has_slim || p[1].info.may_pair || p[1].info.has_slim; }
  // Whether either block's experts differ in K (its LONG).
  bool longs() const { return p[0].info.unequal_k || p[1].info.unequal_k; }
  // f(TOTALS, LONG) with both as types.
  template <class F>
  void with_body(F&& f) const {
    if (totals()) longs() ? f(std::true_type{}, std::true_type{}) : f(std::true_type{}, std::false_type{});
    else longs() ? f(std::false_type{}, std::true_type{}) : f(std::false_type{}, std::false_type{});
  }
};

// One workgroup of two waves per launch, thread e = expert e0 + e of the launch's chunk of experts [e0, e0 + kMaxProblems) (the shared
// expert, if any, is expert E with `shared_rows` rows).  Everything the host launcher computes (launch_range), with the same
// functions and in the same order, so the two produce identical tables; prefix sums over experts are wave scans (a later chunk
// first sums what the experts before it occupy), and an entry finds its place from per-branch counts instead of a sequential walk.
// A chain of dependent steps that the whole forward waits for, so every step is kept short: what does not depend on the counts (the
// experts' descriptors, the kernel's branch table) is fetched first, by plan_block_prepare, while the counts are still being made;
// scans run on lane moves in the vector ALU; sums over the branches take one lane per branch.  Its code is
// cold in every launch and costs its fetching, so it is small: loops are rolled, and no division is left (a version with the branch walk
// unrolled into registers and 2.3 times the code was slower at 8192 tokens: 5.5 us for the walk alone).  Measured inside the workgroup from
// the counts to the end, Qwen1.5-MoE: 12.8 -> 7.3 us at 8192 tokens, 8.7 -> 5.2 us at 64.
struct PlanShared {
  static constexpr int kSums = 5;                    // rows, packed input, scales, output elements, fp16 input elements
  long tot[kSums][2];                                // per wave
  long base[kSums][2];                               // the same five, summed over the experts before this launch
  int cnt[kMaxBranches][2], til[kMaxBranches][2];    // per run-order rank and wave: entries, tiles
  int cnt_long[kMaxBranches][2], til_long[kMaxBranches][2];  // ... of which belong to long-K problems
  int kmin[2];
  unsigned load[2];                                  // launch_load_of, per wave
  unsigned tall[2];                                  // large tiles of the wave's problems with K = kmin (lower half), of the others (upper half)
  int long_tiles[2], long_tiles_kmin[2];             // large tiles of the wave's problems with K >= kLongK; of those with K = kmin
  // the kernel's branch table, from the kernel arguments: the planning functions walk it entry by entry, and each step of such a
  // walk through the argument segment costs a trip to the scalar cache
  PlanInfo info;
};

// Threads 0 .. kPlanThreads - 1 of the planning workgroup, before the counts are there: this thread's expert's descriptor (returned), the
// branch table and cleared counters in LDS.  A barrier must lie between this and plan_block_body.
__device__ __forceinline__ mxmoe_block_desc plan_block_prepare(const PlanParams& p, const int chunk, PlanShared& sh) {
  const int e = threadIdx.x, ge = chunk * kMaxProblems + e;
  mxmoe_block_desc d{};
  if (e < min(kMaxProblems, p.Et - chunk * kMaxProblems)) d = p.desc[ge];
  static_assert(sizeof(PlanInfo) % 4 == 0, "copied word by word");
  for (int i = e; i < (int)(sizeof(PlanInfo) / 4); i += kPlanThreads) reinterpret_cast<int*>(&sh.info)[i] = reinterpret_cast<const int*>(&p.info)[i];
  if (e < kMaxBranches) {
    sh.cnt[e][0] = sh.cnt[e][1] = sh.til[e][0] = sh.til[e][1] = 0;
    sh.cnt_long[e][0] = sh.cnt_long[e][1] = sh.til_long[e][0] = sh.til_long[e][1] = 0;  // (LONG)
  }
  return d;
}

// `recv`: the tokens-per-expert counts (device memory, or LDS when the planning workgroup counted them itself); `d`: what
// plan_block_prepare returned.  Every thread of the workgroup must call this (it holds workgroup barriers); threads with `active` false
// (those past kPlanThreads of a wider workgroup) only pass the barriers.
// TOTALS: with what a launch's totals decide, pairs of row segments and slim tiles.  In a body of its own, since a launch of few rows, which has neither, waits for the
// fetching of that code even where a test skips it: layer_head_kernel, us, skipped by a test / without it: 1 token of 64 experts 7.9 / 7.2, 32 tokens 7.8 / 7.5, 8 tokens of 60
// experts 8.9 / 8.4, 64 with a shared expert 9.7 / 8.7.
// LONG: some experts' K differ (PlanInfo::unequal_k): without, no problem is long against the launch's others, and what looks for those is left out the same way.
template <bool TOTALS, bool LONG, class Count>
__device__ __forceinline__ void plan_block_body(const PlanParams& p, const int chunk, const int chunks, const Count* recv, const mxmoe_block_desc& d, PlanShared& sh,
                                                const bool active) {
  const int e0 = chunk * kMaxProblems;                       // first expert of this launch
  const int ecnt = min(kMaxProblems, p.Et - e0);             // experts of this launch
  constexpr int kSums = PlanShared::kSums;
  const PlanInfo& info = sh.info;
  const int e = threadIdx.x, lane = e & 63, wave = e >> 6;
  const int ge = e0 + e;                             // this thread's expert
  const bool mine = active && e < ecnt;
  const PlanLayout lay(p.Et);
  FusedArgs* fa = reinterpret_cast<FusedArgs*>(p.plan + chunk * kFusedArgsStride);
  int64_t* table = reinterpret_cast<int64_t*>(p.plan + lay.table);
  const void** ptrs = reinterpret_cast<const void**>(p.plan + lay.ptrs);
  int64_t* misc = reinterpret_cast<int64_t*>(p.plan + lay.misc);
  mxmoe_dim3* sizes = reinterpret_cast<mxmoe_dim3*>(p.plan + lay.sizes);
  const int32_t** row_maps = reinterpret_cast<const int32_t**>(p.plan + lay.rows);
  const int kind = p.form.kind;

  // what one expert occupies: rows, packed activation elements, scales, output elements, fp16 input elements (in fp16 elements but the rows)
  auto footprint = [&](int x, const mxmoe_block_desc& dx, long (&f)[kSums]) {
    const long rows = x < p.E ? (long)recv[x] : (long)p.shared_rows;
    const int tag = act_tag_of(dx.q), K = (int)dx.K;
    const long qld = tag == 0 ? K : (tag == 1 || tag == 5 ? K / 2 : K / 4);  // fp16 elements per packed activation row (ref_bind.cu:491)
    const long sld = tag == 0 ? 0 : (tag == 3 ? K / 128 : 1);                // scales per row (ref_bind.cu:492)
    f[0] = rows;
    // packed activations: rows of qld elements, or (tag 4) whole blocks of 32 rows of K / 64 fragments
    f[1] = tag == 4 ? ((rows + 31) >> 5) * (long)(K >> 6) * (kBf6Frag / 2) : qld * rows;
    f[2] = sld * rows;
    f[3] = (long)(kind == LayerForm::kGateUp ? dx.N / 2 : dx.N) * rows;
    f[4] = (long)K * rows;
  };
  const int N = (int)d.N, K = (int)d.K, fmt = fmt_of(d.q), tag = act_tag_of(d.q);
  const bool scaled = tag != 0;
  long foot[kSums] = {0, 0, 0, 0, 0}, before_me[kSums] = {0, 0, 0, 0, 0}, rows = 0;
  PlanChoice choice;
  int have = 0;
  if (active) {
    // experts before this launch (none for the first: most blocks are one launch)
    if (e0 > 0) {
      long base[kSums] = {0, 0, 0, 0, 0};
      for (int x = e; x < e0; x += kPlanThreads) {
        long f[kSums];
        footprint(x, p.desc[x], f);
#pragma unroll
        for (int i = 0; i < kSums; ++i) base[i] += f[i];
      }
#pragma unroll
      for (int i = 0; i < kSums; ++i) {
        const long all = wave_last(wave_inclusive_scan(base[i]));
        if (lane == 0) sh.base[i][wave] = all;
      }
    } else if (lane < kSums) {
      sh.base[lane][wave] = 0;
    }
    if (mine) footprint(ge, d, foot);
    rows = foot[0];
    // exclusive sums over the experts of this launch before this one (those that the block's form has a use for)
    auto sum_before = [&](int i) {
      const long inc = wave_inclusive_scan(foot[i]);
      before_me[i] = inc - foot[i];
      const long all = wave_last(inc);
      if (lane == 0) sh.tot[i][wave] = all;
    };
    sum_before(0);
    sum_before(3);
    if (kind != LayerForm::kGateUp) {
      sum_before(1);
      sum_before(2);
    }
    if (kind == LayerForm::kBehind) sum_before(4);
    // smallest K of the launch's problems with rows: those above it run first inside their branch (see build_fused_tables)
    int km = K;
    if constexpr (LONG) {
      km = -wave_last(wave_inclusive_max(mine && rows > 0 ? -K : -0x7fffffff));
      if (lane == 0) sh.kmin[wave] = km;
    }
    // what this problem's tile shapes are, as far as the rest of the launch has no say in it, and the large tiles of the long problems
    // (launch_scope): whether one of K >= kLongK is above the launch's smallest is known behind the barrier
    have = mine ? plan_choose(info, fmt, (int)rows, N, choice) : 0;
    if (TOTALS && info.may_pair) {
      const unsigned load = (unsigned)wave_last((int)wave_inclusive_scan(have > 0 ? launch_load_of(choice, (int)rows, N, K) : 0u));  // (unsigned: the upper half takes all 16 bits)
      if (lane == 0) sh.load[wave] = load;
    }
    if (TOTALS && info.has_slim) {
      const unsigned tall = have > 0 ? (unsigned)choice.large_tiles : 0u;
      const unsigned all = (unsigned)wave_last((int)wave_inclusive_scan(K == km ? tall : tall << 16));
      if (lane == 0) sh.tall[wave] = all;
    }
    if constexpr (LONG) {
      const int large = have > 0 && K >= kLongK ? choice.large_tiles : 0;
      if (__ballot(large > 0) != 0) {
        const int all = wave_last(wave_inclusive_scan(large)), at_km = wave_last(wave_inclusive_scan(K == km ? large : 0));
        if (lane == 0) {
          sh.long_tiles[wave] = all;
          sh.long_tiles_kmin[wave] = at_km;
        }
      } else if (lane == 0) {
        sh.long_tiles[wave] = sh.long_tiles_kmin[wave] = 0;
      }
    }
  }
  __syncthreads();
  const int kmin = LONG ? min(sh.kmin[0], sh.kmin[1]) : K;
  const bool long_k = LONG && mine && K > kmin;
  const int long_tiles = !LONG ? 0 : sh.long_tiles[0] - (sh.kmin[0] == kmin ? sh.long_tiles_kmin[0] : 0) + sh.long_tiles[1] - (sh.kmin[1] == kmin ? sh.long_tiles_kmin[1] : 0);
  Segment sg[2];
  const int ns = have > 0 ? plan_split(info, fmt, (int)rows, N, choice, runs_long(K, kmin) ? min(long_tiles, kLongTiles) : info.few_blocks && integer_sums(fmt) ? choice.large_tiles : 0, sg) : 0;
  if (TOTALS && info.has_slim) {
    const unsigned t0 = sh.tall[0], t1 = sh.tall[1];
    const int at_kmin = (int)((!LONG || sh.kmin[0] == kmin ? t0 & 0xFFFF : 0) + (!LONG || sh.kmin[1] == kmin ? t1 & 0xFFFF : 0));
    const int all = (int)((t0 & 0xFFFF) + (t0 >> 16) + (t1 & 0xFFFF) + (t1 >> 16));
    take_slim_tiles(info, long_k ? all - at_kmin : at_kmin, (int)rows, N, K, sg, ns);
  }
  const PlanBranch& my_branch = info.b[info.order[min(lane, kMaxBranches - 1)]];  // lane r: the branch of rank r
  const int my_order = my_branch.index;
  unsigned pair = 0;  // the second segment goes beside the first: one item of two entries
  if (TOTALS && info.may_pair && ns == 2 && pairs_pay(fmt, (int)((sh.load[0] >> 16) + (sh.load[1] >> 16)), (int)((sh.load[0] & 0xFFFF) + (sh.load[1] & 0xFFFF)))) pair = pair_word(sg);
  int seg_rank[2] = {-1, -1}, seg_pos[2] = {0, 0}, seg_first[2] = {0, 0};
  // per branch in run order, this wave's entries and tiles
  for (int r = 0; active && r < info.nb; ++r) {
    const int b = __builtin_amdgcn_readlane(my_order, r);
    int mine_tiles = 0, which = -1;
#pragma unroll
    for (int j = 0; j < 2; ++j)
      if (j < ns && sg[j].branch == b && sg[j].tiles > 0 && !(j == 1 && pair)) {
        mine_tiles = sg[j].tiles + (pair ? sg[1].tiles : 0);
        which = j;
      }
    // entries of this branch in this wave, long-K problems first: position = matching lanes that run earlier, first tile = their tiles
    const uint64_t has = __ballot(which >= 0);
    if (has == 0) continue;  // (most branches of a kernel are not used by a given launch: their counters stay zero)
    const uint64_t has_long = LONG ? __ballot(which >= 0 && long_k) : 0, two = __ballot(which >= 0 && pair);
    const int inc_long = LONG ? wave_inclusive_scan(long_k ? mine_tiles : 0) : 0, inc_rest = wave_inclusive_scan(long_k ? 0 : mine_tiles);
    const int tt_long = LONG ? wave_last(inc_long) : 0, tt = tt_long + wave_last(inc_rest);
    const uint64_t before = (1ull << lane) - 1;
#pragma unroll
    for (int j = 0; j < 2; ++j)
      if (which == j) {
        seg_rank[j] = r;
        // position / first tile inside this wave's entries of its own class; the other wave's and the other class's are added below
        const uint64_t here = (long_k ? has_long : ~has_long) & before;
        seg_pos[j] = __popcll(has & here) + __popcll(two & here);
        seg_first[j] = long_k ? inc_long - mine_tiles : inc_rest - mine_tiles;
      }
    if (lane == 0) {
      sh.cnt[r][wave] = __popcll(has) + __popcll(two);
      sh.til[r][wave] = tt;
      if (LONG) {
        sh.cnt_long[r][wave] = __popcll(has_long) + __popcll(has_long & two);
        sh.til_long[r][wave] = tt_long;
      }
    }
  }
  if (pair) {
    seg_rank[1] = seg_rank[0];
    seg_pos[1] = seg_pos[0] + 1;
    seg_first[1] = seg_first[0] + sg[0].tiles;
  }
  __syncthreads();
  if (!active) return;
#pragma unroll
  for (int i = 0; i < kSums; ++i) before_me[i] += sh.base[i][0] + sh.base[i][1] + (wave == 1 ? sh.tot[i][0] : 0l);  // (a sum without a use stays garbage)
  const long first_row = before_me[0], inp_off = before_me[1], sc_off = before_me[2], out_off = before_me[3];
  if (mine) {
    table[ge] = tag;
    table[p.Et + ge] = first_row;
    if (kind != LayerForm::kGateUp) {
      table[2 * p.Et + ge] = inp_off;
      table[3 * p.Et + ge] = sc_off;
    }
    const void* a_ptr = p.inp + 2 * inp_off;
    const void* sa_ptr = scaled ? p.scale + 2 * sc_off : nullptr;
    if (kind == LayerForm::kGateUp) {
      a_ptr = p.form.store[tag];
      sa_ptr = scaled ? p.form.scales[tag] : nullptr;
      row_maps[ge] = ge < p.E ? p.form.token_of_row + first_row : p.form.iota;
    } else if (kind == LayerForm::kBehind && tag == 0) {
      a_ptr = p.form.act + 2 * before_me[4];
    }
    ptrs[ge] = a_ptr;
    ptrs[p.Et + ge] = d.B;
    ptrs[2 * p.Et + ge] = sa_ptr;
    ptrs[3 * p.Et + ge] = d.scale_b;
    ptrs[4 * p.Et + ge] = p.out + 2 * out_off;
    sizes[ge] = mxmoe_dim3{(uint32_t)rows, (uint32_t)N, (uint32_t)K};
    if (ge == p.E) misc[1] = (int64_t)(p.out + 2 * out_off);
  }
  // Branches in run order, one per lane (both waves hold the same): entries and tiles before each.
  const int b_til = lane < info.nb ? sh.til[lane][0] + sh.til[lane][1] : 0, b_cnt = lane < info.nb ? sh.cnt[lane][0] + sh.cnt[lane][1] : 0;
  const int t_long = LONG && lane < info.nb ? sh.til_long[lane][0] + sh.til_long[lane][1] : 0;
  const int til_inc = wave_inclusive_scan(b_til), cnt_inc = wave_inclusive_scan(b_cnt);
  const int total = wave_last(til_inc), ne = wave_last(cnt_inc);
  const int tile0 = til_inc - b_til, ent0 = cnt_inc - b_cnt;
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int r = max(seg_rank[j], 0);
    int pos = seg_pos[j] + __shfl(ent0, r), first = seg_first[j] + __shfl(tile0, r);
    if (seg_rank[j] >= 0) {
      // inside the branch: [long-K entries of wave 0][of wave 1][other entries of wave 0][of wave 1]
      if (long_k) {
        if (wave == 1) {
          pos += sh.cnt_long[r][0];
          first += sh.til_long[r][0];
        }
      } else {
        if (LONG) {
          pos += sh.cnt_long[r][0] + sh.cnt_long[r][1];
          first += sh.til_long[r][0] + sh.til_long[r][1];
        }
        if (wave == 1) {
          pos += sh.cnt[r][0] - (LONG ? sh.cnt_long[r][0] : 0);
          first += sh.til[r][0] - (LONG ? sh.til_long[r][0] : 0);
        }
      }
      fa->entry[pos] = FusedArgs::Entry{first, sg[j].row0, sg[j].rows, (int)((unsigned)(e | (sg[j].branch << 16)) | pair | (pair && j ? kPairSecond : 0u))};  // problem index relative to the launch's first
    }
  }
  if (wave == 0) {
    // Phases: every branch with tiles is one, or two (long_phase), in run order; those beyond the phase table share the last phase.
    const bool split = LONG && long_phase(my_branch, t_long, b_til - t_long);
    const uint64_t live = __ballot(b_til > 0), twice = LONG ? __ballot(split) : 0, lower = (1ull << lane) - 1;
    int ord = __popcll(live & lower), np = __popcll(live);
    int head_tiles = b_til, padded1 = 0;  // tiles of a branch's first phase; workgroups of its second
    if (LONG && twice) {                  // (a branch around code that most launches would fetch for nothing)
      ord += __popcll(twice & lower);
      np += __popcll(twice);
      if (split) {
        head_tiles = t_long;
        padded1 = ord + 1 < kMaxPhases - 1 ? (b_til - t_long + kNumXcd - 1) / kNumXcd * kNumXcd : 0;
      }
    }
    np = min(np, kMaxPhases);
    // workgroups of the phases that have a successor in the table
    const int padded0 = b_til > 0 && ord < kMaxPhases - 1 ? (head_tiles + kNumXcd - 1) / kNumXcd * kNumXcd : 0;
    const int wg0 = wave_inclusive_scan(padded0 + padded1) - padded0 - padded1;
    const int flat = wave_last(wave_inclusive_scan(b_til > 0 && ord < kMaxPhases && flat_phase(my_branch) ? 1 << ord : 0));
    auto begin = [&](int o, int first, int wg) {
      fa->phase_tile0[o] = first;
      fa->phase_wg0[o] = wg;
      if (o == np - 1) {  // the last phase: up to the last tile
        fa->phase_tile0[np] = total;
        fa->phase_wg0[np] = wg + (total - first + kNumXcd - 1) / kNumXcd * kNumXcd;
      }
    };
    if (b_til > 0 && ord < kMaxPhases) begin(ord, tile0, wg0);
    if (LONG && twice) {
      if (split && ord + 1 < kMaxPhases) begin(ord + 1, tile0 + t_long, wg0 + padded0);
    }
    if (lane == 0) {
      // rows routed: those of every launch without the shared expert's; the last launch knows them all
      if (chunk == chunks - 1) misc[0] = sh.base[0][0] + sh.base[0][1] + sh.tot[0][0] + sh.tot[0][1] - (p.Et > p.E ? p.shared_rows : 0);
      if (chunk == 0 && p.Et == p.E) misc[1] = 0;
      if (np == 0) fa->phase_tile0[0] = fa->phase_wg0[0] = fa->phase_tile0[1] = fa->phase_wg0[1] = 0;  // a plan without tiles still holds one (empty) phase range
      fa->num_phases = np;
      fa->phase_flat = flat;
      fa->num_entries = ne;
      fa->total_tiles = total;
      fa->problem_offset = e0;
      fa->As = reinterpret_cast<const uint8_t* const*>(ptrs);
      fa->Bs = reinterpret_cast<const uint8_t* const*>(ptrs + p.Et);
      fa->sa = reinterpret_cast<const _Float16* const*>(ptrs + 2 * p.Et);
      fa->sb = reinterpret_cast<const _Float16* const*>(ptrs + 3 * p.Et);
      fa->Cs = reinterpret_cast<_Float16* const*>(const_cast<void**>(ptrs + 4 * p.Et));
      fa->acc = nullptr;
      fa->sizes = sizes;
      fa->rows = row_maps;
    }
  }
}

// Kernel for the formats of `h_desc`, checked once on the host: every problem's format has a branch and its shape fits it (negative:
// none, see last_error()).
int resolve_kernel(int kernel_id, const mxmoe_block_desc* h_desc, int et);

}  // namespace mxmoe

// Device-side planning of the two fused launches of a layer forward.
//
// The reference's operators read the tokens-per-expert counts back to the host (`.cpu()`, mxmoe/kernels/src/ref_bind.cu:451) and
// build every table there: the per-expert {tag, first row, offsets} table of the quantisers (ref_bind.cu:475-505), the five pointer
// arrays and sizes of the launch (ref_bind.cu:362-404) and, in the generated launcher, the tile prefix sums
// (mxmoe/kernels/kernel_sketch.py:89-104).  Here one small kernel derives all of them from the counts where they are, in device
// memory, so that the host enqueues the whole forward without waiting for the routing: no synchronisation, nothing that depends
// on the counts in any launch argument, and therefore a sequence that a HIP graph can hold.
#include <hip/hip_runtime.h>

#include "../../include/mxmoe_amd.h"
#include "include/mxmoe_launch.hpp"
#include "include/mxmoe_plan.hpp"
#include "include/mxmoe_perm.hpp"
#include "include/mxmoe_plan_body.hpp"

namespace mxmoe {

template <bool TOTALS, bool LONG>
__global__ void __launch_bounds__(kPlanThreads) plan_block_kernel(const PlanPair pair) {
  // one workgroup per launch of each block of the layer (gate_up, down): all only read the counts
  __shared__ PlanShared sh;
  const PlanParams& p = pair.p[blockIdx.x / pair.chunks];
  const mxmoe_block_desc d = plan_block_prepare(p, blockIdx.x % pair.chunks, sh);
  __syncthreads();
  plan_block_body<TOTALS, LONG>(p, blockIdx.x % pair.chunks, pair.chunks, pair.p[0].recv, d, sh, true);
}

// Permutation and planning of a decode-sized batch (at most kPermChunk (token, slot) entries) in ONE launch: workgroup 0 builds the
// permutation, the others plan the layer's launches from counts they take from the routed ids themselves (a few hundred ids: cheaper
// than waiting for workgroup 0 in a second launch).  A forward of some tens of microseconds feels every launch it saves.
struct PermSmallArgs {
  const int32_t* ids;
  int total, E, topk, nbits;
  int64_t* recv;
  int32_t* dst;
  int64_t* perm;
  int64_t* slot;
  int32_t* row_of_slot;
};
template <bool TOTALS, bool LONG>
__global__ void __launch_bounds__(kPlanThreads) perm_plan_small_kernel(const PermSmallArgs a, const PlanPair pair) {
  extern __shared__ __align__(8) uint8_t pp_lds[];  // E int32 counters (workgroup 0) or E int64 counts (planning workgroups)
  if (blockIdx.x == 0) {
    perm_small_body(a.ids, a.total, a.E, a.topk, a.nbits, a.recv, a.dst, a.perm, a.slot, a.row_of_slot, reinterpret_cast<int32_t*>(pp_lds), threadIdx.x < 64);
    return;
  }
  __shared__ PlanShared sh;
  const int b = blockIdx.x - 1, chunk = b % pair.chunks;
  const mxmoe_block_desc d = plan_block_prepare(pair.p[b / pair.chunks], chunk, sh);
  int64_t* counts = reinterpret_cast<int64_t*>(pp_lds);
  unsigned long long* cnt = reinterpret_cast<unsigned long long*>(pp_lds);
  for (int e = threadIdx.x; e < a.E; e += kPlanThreads) counts[e] = 0;
  __syncthreads();
  for (int i = threadIdx.x; i < a.total; i += kPlanThreads) {
    const int e = a.ids[i];
    if (e >= 0 && e < a.E) atomicAdd(&cnt[e], 1ull);
  }
  __syncthreads();
  plan_block_body<TOTALS, LONG>(pair.p[b / pair.chunks], chunk, pair.chunks, counts, d, sh, true);
}

// The same for larger batches, after perm_hist_kernel has counted the experts per chunk of kPermChunk entries: the first `blocks`
// workgroups scatter their chunk (each summing the counts it needs: perm_scatter_body with raw counts), the others plan the
// layer's launches from the column sums of the same histogram.  Neither waits for the other, so the forward's serial head is two
// launches (count, scatter + plan) instead of four (count, scan, scatter, plan).
struct PermScatterArgs {
  const int32_t* ids;
  int total, E, topk, nbits, blocks;
  const int32_t* hist;
  int64_t* recv;
  int32_t* dst;
  int64_t* perm;
  int64_t* slot;
  int32_t* row_of_slot;
};
template <bool TOTALS, bool LONG>
__global__ void __launch_bounds__(kPlanThreads) perm_scatter_plan_kernel(const PermScatterArgs a, const PlanPair pair) {
  extern __shared__ __align__(8) uint8_t pp_lds[];  // E int32 ranks (scatter workgroups) or E int64 counts (planning workgroups)
  if ((int)blockIdx.x < a.blocks) {
    perm_scatter_body(a.ids, a.total, a.E, a.topk, a.nbits, a.hist, a.blocks, (int)blockIdx.x, true, a.recv, a.dst, a.perm, a.slot, a.row_of_slot,
                      reinterpret_cast<int32_t*>(pp_lds), threadIdx.x < 64);
    return;
  }
  __shared__ PlanShared sh;
  const int b = blockIdx.x - a.blocks, chunk = b % pair.chunks;
  const mxmoe_block_desc d = plan_block_prepare(pair.p[b / pair.chunks], chunk, sh);
  int64_t* counts = reinterpret_cast<int64_t*>(pp_lds);
  for (int e = threadIdx.x; e < a.E; e += kPlanThreads) {
    int v, before;
    perm_hist_row_sums(a.hist + (long)e * perm_hist_stride(a.blocks), a.blocks, 0, &v, &before);
    counts[e] = v;
  }
  __syncthreads();
  plan_block_body<TOTALS, LONG>(pair.p[b / pair.chunks], chunk, pair.chunks, counts, d, sh, true);
}

// Whether a kernel has a tile for the format and operand layout of every block.
static bool covers_blocks(const FusedKernel& k, const mxmoe_block_desc* h_desc, int et) {
  for (int i = 0; i < et; ++i) {
    Segment sg[2];
    const int f = fmt_of(h_desc[i].q);
    if (f == (int)Fmt::UNSUPPORTED || plan_segments(plan_of(k), f, 1, 256, sg) < 0) return false;
    // a kernel's w4a4 tiles take packed int4 rows or bf6 fragments, never both: the descriptor says which the block will get
    if (f == (int)Fmt::W4A4 && kernel_takes_bf6(k) != wants_bf6(h_desc[i].q)) return false;
    if (f == (int)Fmt::W8A8 && (kernel_variant(k, Fmt::W8A8) == kVariantFp8) != wants_fp8(h_desc[i].q)) return false;
    // 16-bit float blocks of a layer are fp16 (the activation step between the launches computes in fp16): no bfloat16 kernel here
    if (f == (int)Fmt::FP16 && kernel_variant(k, Fmt::FP16) != 0) return false;
  }
  return true;
}

// Kernel for the formats of `h_desc`, checked once on the host: every problem's format has a branch and its shape fits it.
int resolve_kernel(int kernel_id, const mxmoe_block_desc* h_desc, int et) {
  auto& reg = registry();
  auto covers = [&](const FusedKernel& k) { return covers_blocks(k, h_desc, et); };
  if (kernel_id < 0) {
    for (int i = 0; i < (int)reg.size() && kernel_id < 0; ++i)
      if (reg[i].policy == Policy::Fused && reg[i].max_rows_hint == 0 && covers(reg[i])) kernel_id = i;  // (row counts are not known here: no few-row kernel)
    if (kernel_id < 0) {
      last_error() = "quant type not supported";
      return -1;
    }
  }
  if (kernel_id >= (int)reg.size()) {
    last_error() = "kernel id out of range";
    return -2;
  }
  const FusedKernel& k = reg[kernel_id];
  if (!covers(k)) {
    last_error() = "quant type not supported";
    return -1;
  }
  for (int i = 0; i < et; ++i) {
    const mxmoe_dim3 sz{1, h_desc[i].N, h_desc[i].K};
    for (const BranchInfo& bi : k.branches)
      if ((int)bi.fmt == fmt_of(h_desc[i].q) && !shape_ok(bi, sz)) {
        char buf[200];
        snprintf(buf, sizeof buf, "problem %d: shape [N %u, K %u] not supported by tile %s (K %% %d, N %% 8)", i, sz.y, sz.z, fmt_name(bi.fmt, true), bi.k_multiple);
        last_error() = buf;
        return -3;
      }
    const int tag = act_tag_of(h_desc[i].q);
    if (tag < 0 || (tag == 3 && h_desc[i].K % 128)) {
      last_error() = tag < 0 ? "quant type not supported" : "group-128 activations need a row length that is a multiple of 128";
      return tag < 0 ? -1 : -3;
    }
  }
  return kernel_id;
}

}  // namespace mxmoe

using namespace mxmoe;

extern "C" {

size_t mxmoe_plan_bytes(int num_problems) { return PlanLayout(num_problems).total; }

size_t mxmoe_plan_offset(int which, int num_problems) {
  const PlanLayout lay(num_problems);
  switch (which) {
    case 0: return 0;
    case 1: return lay.table;
    case 2: return lay.ptrs;
    case 3: return lay.misc;
    case 4: return lay.sizes;
    default: return lay.total;
  }
}

int mxmoe_plan_select_kernel(int kernel_id, const mxmoe_block_desc* h_desc, int num_problems) {
  if (!h_desc || num_problems <= 0 || num_problems > kMaxPlannedProblems) {
    last_error() = "a planned block holds 1 to 4096 problems";
    return -3;
  }
  return resolve_kernel(kernel_id, h_desc, num_problems);
}

static int select_kernel_rows(const mxmoe_block_desc* h_desc, int num_experts, int num_tokens, int topk, int shared_rows, bool headless) {
  const int et = num_experts + (shared_rows > 0 ? 1 : 0);
  const int plain = mxmoe_plan_select_kernel(-1, h_desc, et);
  if (plain < 0) return plain;
  if (num_experts <= 0 || num_tokens <= 0 || topk <= 0 || shared_rows < 0) {
    last_error() = "experts, tokens and top-k must be positive";
    return -3;
  }
  // an even routing over the widest experts: every one of them gets a row before any gets two
  const long routed = (long)num_tokens * topk;
  const int live = (int)std::min<long>(num_experts, routed);
  std::vector<int> widest(num_experts);
  for (int i = 0; i < num_experts; ++i) widest[i] = i;
  std::stable_sort(widest.begin(), widest.end(), [&](int x, int y) { return h_desc[x].N > h_desc[y].N; });
  RowSummary s;
  for (int i = 0; i < num_experts; ++i) {
    const mxmoe_block_desc& d = h_desc[widest[i]];
    s.add((Fmt)fmt_of(d.q), i < live ? routed / live + (i < routed % live) : 0, d.N, d.K);
    s.add_format((Fmt)fmt_of(d.q));  // (any of them may get rows)
  }
  if (shared_rows > 0) s.add((Fmt)fmt_of(h_desc[num_experts].q), shared_rows, h_desc[num_experts].N, h_desc[num_experts].K);
  s.max_rows = std::max<long>(s.max_rows, num_tokens);  // one expert may get them all
  // an uneven routing has problems of several 16-row tiles well before the average reaches 16
  if (routed > 12l * num_experts) s.tall = s.live;
  s.headless = headless && num_tokens <= kDirectTokens && routed <= kDirectEntries;
  const int few = few_row_kernel(s, [&](const FusedKernel& k) { return covers_blocks(k, h_desc, et); });
  return few >= 0 && resolve_kernel(few, h_desc, et) == few ? few : plain;
}

int mxmoe_plan_select_kernel_rows(const mxmoe_block_desc* h_desc, int num_experts, int num_tokens, int topk, int shared_rows) {
  return select_kernel_rows(h_desc, num_experts, num_tokens, topk, shared_rows, false);
}

int mxmoe_layer_kernel(const mxmoe_block_desc* h_desc, int num_experts, int num_tokens, int topk, int shared_rows, int first) {
  // (fp8 blocks keep the limits of a layer with a head: 64 tokens, 768 blocks; beyond them both sides were not measured)
  const int et = num_experts + (shared_rows > 0 ? 1 : 0);
  bool fp8 = false;
  for (int i = 0; h_desc && i < et; ++i) fp8 = fp8 || wants_fp8(h_desc[i].q);
  const int kid = select_kernel_rows(h_desc, num_experts, num_tokens, topk, shared_rows, first && !fp8);
  const int lean = without_many_token_tiles(kid, [&](const FusedKernel& k) { return covers_blocks(k, h_desc, et); });
  return lean == kid || resolve_kernel(lean, h_desc, et) == lean ? lean : kid;
}

int mxmoe_plan_grid_bound(int kernel_id, const mxmoe_block_desc* h_desc, int num_experts, int routed_rows_max, int shared_rows) {
  const int et = num_experts + (shared_rows > 0 ? 1 : 0);
  const int kid = mxmoe_plan_select_kernel(kernel_id, h_desc, et);
  if (kid < 0) return kid;
  const PlanInfo pi = plan_info_of_block(registry()[kid], h_desc, et);
  // For every routed expert tiles(M) <= first + slope * (M - 1) for all M >= 1, with first = tiles(1) and slope the steepest rise
  // found by walking M over 64 rows of the format's largest tile (the planner's decisions repeat with that tile's period).  With at
  // most n = min(experts, rows) experts non-empty, the launch has at most (sum of the n largest `first`) + max slope * (rows - n) tiles.
  // A block that is long against the smallest K, or an integer one of few blocks of channels, may be planned as such in its launch (or not, when the block is run as several launches), beside
  // any number of others: the larger count holds, and with more of the others it takes shapes of less total cost and more each,
  // hence fewer tiles, so it is enough to look at the block with none.
  auto tiles_of = [&](int f, int m, int n, bool maybe_long) {
    int most = 0;
    PlanChoice c;
    if (plan_choose(pi, f, m, n, c) <= 0) return 0;
    for (int lk = 0; lk <= (maybe_long ? 1 : 0); ++lk) {
      Segment sg[2];
      const int ns = plan_split(pi, f, m, n, c, lk ? c.large_tiles : 0, sg);
      int t = 0;
      for (int j = 0; j < ns; ++j) t += sg[j].tiles;
      most = std::max(most, t);
    }
    return most;
  };
  uint32_t kmin = ~0u;
  for (int e = 0; e < et; ++e) kmin = std::min(kmin, (uint32_t)h_desc[e].K);
  // And tiles(M) <= extra + per_row * M, with per_row the columns per row of the shape that very long problems run on and extra the
  // largest excess over it: the smaller of the two sums holds.
  long shared_tiles = 0;
  double slope = 0, per_row = 0;
  long extras = 0;
  std::vector<int> firsts;
  struct Seen { int f, n, maybe_long, first, extra; double slope, per_row; };
  std::vector<Seen> seen;
  for (int e = 0; e < et; ++e) {
    const int f = fmt_of(h_desc[e].q), n = (int)h_desc[e].N;
    const bool maybe_long = runs_long((int)h_desc[e].K, (int)kmin) || (pi.few_blocks && integer_sums(f));
    if (e >= num_experts) {  // the shared expert's row count is known
      shared_tiles += tiles_of(f, shared_rows, n, maybe_long);
      continue;
    }
    const Seen* hit = nullptr;
    for (const Seen& sn : seen)
      if (sn.f == f && sn.n == n && sn.maybe_long == maybe_long) hit = &sn;
    if (!hit) {
      Segment sg[2];
      plan_segments(pi, f, 1 << 20, n, sg);
      const BranchInfo& bi = registry()[kid].branches[sg[0].branch];
      const int bm = bi.BM, cols = (n + bi.BN - 1) / bi.BN;
      Seen sn{f, n, maybe_long, tiles_of(f, 1, n, maybe_long), 0, 0.0, (double)cols / bm};
      // (a long block of one column may be short of kLongTiles tiles for that many row tiles)
      const int limit = std::min(std::max(routed_rows_max, 2), std::max(64, maybe_long ? kLongTiles + 1 : 0) * bm);
      for (int m = 1; m <= limit; ++m) {
        const int t = tiles_of(f, m, n, maybe_long);
        if (m > 1) sn.slope = std::max(sn.slope, (double)(t - sn.first) / (m - 1));
        sn.extra = std::max(sn.extra, t - (m / bm) * cols);
      }
      seen.push_back(sn);
      hit = &seen.back();
    }
    firsts.push_back(hit->first);
    slope = std::max(slope, hit->slope);
    per_row = std::max(per_row, hit->per_row);
    extras += hit->extra;
  }
  std::sort(firsts.begin(), firsts.end(), [](int x, int y) { return x > y; });
  const int nonempty = std::min((int)firsts.size(), routed_rows_max);
  long by_first = (long)(slope * (routed_rows_max - nonempty)) + 1;
  for (int i = 0; i < nonempty; ++i) by_first += firsts[i];
  const long by_rows = extras + (long)(per_row * routed_rows_max) + 1;
  long bound = shared_tiles + std::min(by_first, by_rows);
  if (pi.has_slim) bound += 2 * kSlimTiles;  // slim tiles: twice as many as the wide ones, which are at most that many then, of either length
  bound += (long)kNumXcd * (kMaxPhases + 1);  // every phase is padded to a multiple of the XCD count
  bound = (bound + kNumXcd - 1) / kNumXcd * kNumXcd;
  if (bound > (1l << 30)) {
    last_error() = "planned grid too large";
    return -3;
  }
  return (int)bound;
}

static int fill_plan_params(PlanParams& p, int kernel_id, const int64_t* d_recv, int num_experts, int shared_rows, const mxmoe_block_desc* d_desc,
                            const mxmoe_block_desc* h_desc, const void* inp_store, const void* scale_store, void* out_store, void* d_plan) {
  const int et = num_experts + (shared_rows > 0 ? 1 : 0);
  if (!d_recv || !d_desc || !h_desc || !inp_store || !out_store || !d_plan) {
    last_error() = "null pointer";
    return 5;
  }
  const int kid = mxmoe_plan_select_kernel(kernel_id, h_desc, et);
  if (kid < 0) return kid == -1 ? 1 : (kid == -2 ? 2 : 3);
  p.recv = d_recv;
  p.desc = d_desc;
  p.inp = reinterpret_cast<const uint8_t*>(inp_store);
  p.scale = reinterpret_cast<const uint8_t*>(scale_store);
  p.out = reinterpret_cast<uint8_t*>(out_store);
  p.plan = reinterpret_cast<uint8_t*>(d_plan);
  p.E = num_experts;
  p.Et = et;
  p.shared_rows = shared_rows;
  p.form = LayerForm{};
  p.info = plan_info_of_block(registry()[kid], h_desc, et);
  return 0;
}

static int launch_plan(PlanPair& pair, int blocks, void* stream) {
  pair.chunks = PlanLayout(pair.p[0].Et).chunks;
  pair.with_body([&](auto totals, auto longs) { hipLaunchKernelGGL((plan_block_kernel<decltype(totals)::value, decltype(longs)::value>), dim3(blocks * pair.chunks), dim3(kPlanThreads), 0, (hipStream_t)stream, pair); });
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) {
    last_error() = std::string("kernel launch failed: ") + hipGetErrorString(e);
    return 4;
  }
  return 0;
}

int mxmoe_plan_block(int kernel_id, const int64_t* d_recv, int num_experts, int shared_rows, const mxmoe_block_desc* d_desc, const mxmoe_block_desc* h_desc,
                     const void* inp_store, const void* scale_store, void* out_store, void* d_plan, void* stream) {
  PlanPair pair;
  const int rc = fill_plan_params(pair.p[0], kernel_id, d_recv, num_experts, shared_rows, d_desc, h_desc, inp_store, scale_store, out_store, d_plan);
  if (rc) return rc;
  pair.p[1] = pair.p[0];
  return launch_plan(pair, 1, stream);
}

int mxmoe_plan_layer(const mxmoe_plan_call* gate_up, const mxmoe_plan_call* down, const int64_t* d_recv, int num_experts, int shared_rows, void* stream) {
  if (!gate_up || !down) {
    last_error() = "null pointer";
    return 5;
  }
  PlanPair pair;
  const mxmoe_plan_call* c[2] = {gate_up, down};
  for (int i = 0; i < 2; ++i) {
    const int rc = fill_plan_params(pair.p[i], c[i]->kernel_id, d_recv, num_experts, shared_rows, c[i]->d_desc, c[i]->h_desc, c[i]->inp_store, c[i]->scale_store,
                                    c[i]->out_store, c[i]->d_plan);
    if (rc) return rc;
  }
  return launch_plan(pair, 2, stream);
}

int mxmoe_permute_plan_layer(const int32_t* topk_ids, int num_tokens, int topk, int num_experts, int32_t* dst_exp_sorted, int64_t* perm_indices, int64_t* src_slot,
                             int64_t* recv_tokens_per_exp, int32_t* row_of_slot, const mxmoe_plan_call* gate_up, const mxmoe_plan_call* down, int shared_rows, void* stream) {
  if (num_tokens <= 0 || topk <= 0 || num_experts <= 0 || num_experts > kMaxPlannedProblems || (long)num_tokens * topk > kPermChunk) {
    last_error() = "the one-launch permutation + planning takes at most 256 (token, slot) entries: use mxmoe_build_permutation_inv and mxmoe_plan_layer";
    return 3;
  }
  if (!topk_ids || !dst_exp_sorted || !perm_indices || !src_slot || !recv_tokens_per_exp || !gate_up || !down) {
    last_error() = "null pointer";
    return 5;
  }
  PlanPair pair;
  const mxmoe_plan_call* c[2] = {gate_up, down};
  for (int i = 0; i < 2; ++i) {
    const int rc = fill_plan_params(pair.p[i], c[i]->kernel_id, recv_tokens_per_exp, num_experts, shared_rows, c[i]->d_desc, c[i]->h_desc, c[i]->inp_store, c[i]->scale_store,
                                    c[i]->out_store, c[i]->d_plan);
    if (rc) return rc;
  }
  pair.chunks = PlanLayout(pair.p[0].Et).chunks;
  PermSmallArgs a;
  a.ids = topk_ids;
  a.total = num_tokens * topk;
  a.E = num_experts;
  a.topk = topk;
  a.nbits = 1;
  while ((1 << a.nbits) <= num_experts) ++a.nbits;  // ids 0..E (E = parked lanes)
  a.recv = recv_tokens_per_exp;
  a.dst = dst_exp_sorted;
  a.perm = perm_indices;
  a.slot = src_slot;
  a.row_of_slot = row_of_slot;
  pair.with_body([&](auto totals, auto longs) { hipLaunchKernelGGL((perm_plan_small_kernel<decltype(totals)::value, decltype(longs)::value>), dim3(1 + 2 * pair.chunks), dim3(kPlanThreads), (size_t)num_experts * 8, (hipStream_t)stream, a, pair); });
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) {
    last_error() = std::string("kernel launch failed: ") + hipGetErrorString(e);
    return 4;
  }
  return 0;
}

int mxmoe_permute_plan_layer_ws(const int32_t* topk_ids, int num_tokens, int topk, int num_experts, int32_t* dst_exp_sorted, int64_t* perm_indices, int64_t* src_slot,
                                int64_t* recv_tokens_per_exp, int32_t* row_of_slot, const mxmoe_plan_call* gate_up, const mxmoe_plan_call* down, int shared_rows,
                                void* workspace, void* stream) {
  if (num_tokens > 0 && topk > 0 && (long)num_tokens * topk <= kPermChunk)
    return mxmoe_permute_plan_layer(topk_ids, num_tokens, topk, num_experts, dst_exp_sorted, perm_indices, src_slot, recv_tokens_per_exp, row_of_slot, gate_up, down,
                                    shared_rows, stream);
  const long total = (long)num_tokens * topk;
  const long blocks = (total + kPermChunk - 1) / kPermChunk;
  if (num_tokens <= 0 || topk <= 0 || num_experts <= 0 || num_experts > kMaxPlannedProblems || blocks * num_experts > kPermFusedScanMax) {
    last_error() = "the two-launch permutation + planning takes batches whose (chunks of 256 entries) x experts is at most 16384: use mxmoe_build_permutation_inv and mxmoe_plan_layer";
    return 3;
  }
  if (!topk_ids || !dst_exp_sorted || !perm_indices || !src_slot || !recv_tokens_per_exp || !gate_up || !down || !workspace) {
    last_error() = "null pointer";
    return 5;
  }
  if (reinterpret_cast<uintptr_t>(workspace) & 15) {
    last_error() = "the workspace of the two-launch permutation + planning must be 16-byte aligned";
    return 3;
  }
  PlanPair pair;
  const mxmoe_plan_call* c[2] = {gate_up, down};
  for (int i = 0; i < 2; ++i) {
    const int rc = fill_plan_params(pair.p[i], c[i]->kernel_id, recv_tokens_per_exp, num_experts, shared_rows, c[i]->d_desc, c[i]->h_desc, c[i]->inp_store, c[i]->scale_store,
                                    c[i]->out_store, c[i]->d_plan);
    if (rc) return rc;
  }
  pair.chunks = PlanLayout(pair.p[0].Et).chunks;
  PermScatterArgs a;
  a.ids = topk_ids;
  a.total = (int)total;
  a.E = num_experts;
  a.topk = topk;
  a.nbits = 1;
  while ((1 << a.nbits) <= num_experts) ++a.nbits;  // ids 0..E (E = parked lanes)
  a.blocks = (int)blocks;
  a.hist = reinterpret_cast<const int32_t*>(workspace);
  a.recv = recv_tokens_per_exp;
  a.dst = dst_exp_sorted;
  a.perm = perm_indices;
  a.slot = src_slot;
  a.row_of_slot = row_of_slot;
  launch_perm_hist(topk_ids, a.total, num_experts, reinterpret_cast<int32_t*>(workspace), true, (hipStream_t)stream);
  pair.with_body([&](auto totals, auto longs) { hipLaunchKernelGGL((perm_scatter_plan_kernel<decltype(totals)::value, decltype(longs)::value>), dim3(a.blocks + 2 * pair.chunks), dim3(kPlanThreads), (size_t)num_experts * 8, (hipStream_t)stream, a, pair); });
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) {
    last_error() = std::string("kernel launch failed: ") + hipGetErrorString(e);
    return 4;
  }
  return 0;
}

int mxmoe_group_gemm_planned(int kernel_id, const void* d_plan, int num_problems, int grid, void* stream) {
  auto& reg = registry();
  if (kernel_id < 0 || kernel_id >= (int)reg.size()) {
    last_error() = "kernel id out of range";
    return 2;
  }
  if (!d_plan || grid <= 0 || num_problems <= 0 || num_problems > kMaxPlannedProblems) {
    last_error() = "null plan, empty grid or bad problem count";
    return 5;
  }
  const FusedKernel& k = reg[kernel_id];
  // one launch per chunk of kMaxProblems experts, each reading its own tables (workgroups past a launch's tiles leave at once)
  const int chunks = PlanLayout(num_problems).chunks;
  for (int c = 0; c < chunks; ++c) {
    const hipError_t e = k.launch_planned(reinterpret_cast<const FusedArgs*>(reinterpret_cast<const uint8_t*>(d_plan) + c * kFusedArgsStride), grid, k.lds_bytes, (hipStream_t)stream);
    if (e != hipSuccess) {
      last_error() = std::string("kernel launch failed: ") + hipGetErrorString(e);
      return 4;
    }
  }
  return 0;
}

}  // extern "C"

// The planned layer forward in its short form: three to five launches from (hidden, expert ids, weights) to the layer's output.
//
//   head      permutation by expert, the tables of both GroupGEMMs, and every token quantised once per activation format: three
//             jobs that need nothing of each other, in one launch;
//   gate_up   the fused GroupGEMM in its gate_up form (TileArgs): rows gathered by token, output silu(gate) * up;
//   rows      rotation + quantisation of those rows for the second block (left out when every second block reads fp16 rows);
//   down      the fused GroupGEMM of the second block;
//   combine   un-permute, top-k weighted sum, shared expert.
//
// Few tokens on the kernels for few rows need no head (layer_first_kernel); what is left of it in front of gate_up is the tokens' quantisation, where first blocks take quantised ones.
//
// Against the form that writes an activation row per destination (top-k of them per token, after the permutation is known) and stores
// gate and up: the head is one launch instead of two or three in sequence, activations take 1 / top-k of the space, and 8 bytes per
// intermediate value are neither written nor read.  The same kernels' arithmetic, bit for bit.  Measured, that form -> this one, us a
// pass: DeepSeek-V2-Lite w4a16 / w3a16 47.7 -> 35.2 (1 token), 98.7 -> 84.9 (32), 163 -> 139 (201); Qwen1.5-MoE w4a4 456 -> 402 (8192,
// of which the head 47 -> 24, the activation step 107 -> 72); Mixtral w4a4 / w8a8 / w4a16 3368 -> 3249 (8192).
#include <algorithm>
#include <climits>
#include <hip/hip_runtime.h>

#include <memory>
#include <string>
#include <vector>

#include "../../include/mxmoe_amd.h"
#include "include/mxmoe_launch.hpp"
#include "include/mxmoe_perm.hpp"
#include "include/mxmoe_plan.hpp"
#include "include/mxmoe_plan_body.hpp"
#include "include/mxmoe_rows.hpp"

namespace mxmoe {

// Threads of the head's workgroups: kHeadSmall up to kHeadSmallMax entries (tokens x top-k), kHeadLarge beyond.  A small batch's head is a
// chain of latencies, and its tokens are better off on many CUs; workgroups that count a larger batch's ids are bound by their own
// instructions (32768 ids: 7.7 us with 256 threads, 3.3 with 1024), but tokens in workgroups of 1024 threads fill the chip worse
// (head of 8192 tokens: 24.3 / 25.3 / 28.9 us with 256 / 512 / 1024 threads, of 2049 tokens with top-6: 17.4 / 16.3 / 19.4).
constexpr int kHeadSmall = 256, kHeadLarge = 512;
constexpr int kHeadSmallMax = 4096;
// Experts of the short form: its permutation workgroups keep up to 26 counters per expert in LDS (52 KiB at this many).
constexpr int kHeadMaxExperts = 512;
// Entries (tokens x top-k) up to which every workgroup that needs counts takes them from the ids themselves, all of them: 128 KiB of ids
// out of L2 and as many LDS counter updates take some 6 us, which the token workgroups of the same launch hide; beyond, the cost
// per workgroup would grow with the batch, and a counting launch (perm_hist_kernel) goes first.  Its counts are summed by every workgroup
// that needs them, so that form in turn ends at kPermFusedScanMax counts (mxmoe_layer_supported): with 64 experts or more, here.
constexpr int kHeadCountMax = 65536;

struct HeadArgs {
  const int32_t* ids;
  int total, E, topk, nbits;
  int perm_wgs;          // workgroups of one entry per thread
  int chunks;            // chunks of kPermChunk entries
  const int32_t* hist;   // per-chunk counts, expert-major (perm_hist_stride), or null: count the ids
  int64_t* recv;         // [E] tokens per expert
  int32_t* dst_exp;      // [total] expert of each sorted row
  int32_t* token_of_row; // [total]
  int32_t* row_of_slot;  // [total] sorted row of each (token, slot), -1 when its expert id is out of range
  // tokens
  const _Float16* hidden;  // [T][n]
  int T;
  unsigned tags;           // bit per tag: formats every token is written in
  int rotate;              // 0 never, 1 quantised formats, 2 also fp16
  float scale;             // 1 / sqrt(n)
  uint8_t* store[kNumTags];
  _Float16* scales[kNumTags];
};

// Counts of every expert over all ids (all) and over those before entry `base` (before; not counted when null), by a whole workgroup.
// `copies`: LDS for kCountCopies (all) or twice as many counters per expert: lane l adds to copy l % kCountCopies, since lanes that hit one
// counter take turns (60 experts: four or five of 64 lanes on average, twenty under a skewed routing).
constexpr int kCountCopies = 8;
template <int TH>
__device__ __forceinline__ void count_ids(const int32_t* __restrict__ ids, int total, int E, int base, int32_t* before, int32_t* all, int32_t* copies) {
  const int sets = before ? 2 : 1;
  // the first ids are on their way while the counters are cleared (a barrier waits for every load in front of it, so this one round trip
  // also covers whatever the caller has just requested)
  constexpr int kFirst = TH == kHeadSmall ? 8 : 4;
  int first[kFirst];
#pragma unroll
  for (int k = 0; k < kFirst; ++k) first[k] = (int)threadIdx.x + k * TH < total ? gload<int>(ids + threadIdx.x + k * TH) : -1;
  for (int i = threadIdx.x; i < sets * kCountCopies * E; i += TH) copies[i] = 0;
  __syncthreads();
  int32_t* const mine = copies + (threadIdx.x % kCountCopies) * E;
  // (an entry counts in one set only: those before `base` are added to both results at the end)
  auto add = [&](int idx, int e) {
    if (e >= 0 && e < E) atomicAdd(mine + (before && idx < base ? kCountCopies * E : 0) + e, 1);
  };
#pragma unroll 1
  for (int k = 0; k < kFirst && k * TH < total; ++k) {  // (rolled: cold code costs its fetch)
    add(threadIdx.x + k * TH, first[0]);
#pragma unroll
    for (int j = 0; j + 1 < kFirst; ++j) first[j] = first[j + 1];
  }
  int done = kFirst * TH;
  if constexpr (TH == kHeadLarge) {  // 16 bytes per lane and load, eight loads in flight: two round trips for 32768 ids
    const int n4 = (reinterpret_cast<uintptr_t>(ids) & 15) == 0 ? total >> 2 : 0;
    constexpr int kAhead = 8;
    for (int i0 = done / 4 + (int)threadIdx.x; i0 < n4; i0 += kAhead * TH) {
      v4i v[kAhead];
#pragma unroll
      for (int k = 0; k < kAhead; ++k) v[k] = gload<v4i>(reinterpret_cast<const v4i*>(ids) + min(i0 + k * TH, n4 - 1));
#pragma unroll
      for (int k = 0; k < kAhead; ++k) {
        const int i = i0 + k * TH;
        if (i < n4) {
#pragma unroll
          for (int j = 0; j < 4; ++j) add(4 * i + j, v[k][j]);
        }
      }
    }
    done = max(n4 << 2, done);
  }
  for (int i = done + (int)threadIdx.x; i < total; i += TH) add(i, ids[i]);
  __syncthreads();
  for (int e = threadIdx.x; e < E; e += TH) {
    int n = 0, nb = 0;
#pragma unroll
    for (int c = 0; c < kCountCopies; ++c) {
      n += copies[c * E + e];
      if (before) nb += copies[(kCountCopies + c) * E + e];
    }
    all[e] = n + nb;
    if (before) before[e] = nb;
  }
  __syncthreads();
}

// TH consecutive entries of the stable permutation by expert: each wave places 64.
template <int TH>
__device__ __forceinline__ void head_scatter(const HeadArgs& a, int block, int32_t* lds) {
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  constexpr int kWavesHere = TH / 64;
  int32_t *all = lds, *run = lds + a.E, *in_wave = lds + 2 * a.E;  // [E] totals, [E] first row of this workgroup's entries, [waves][E] entries per wave
  const int idx = block * TH + threadIdx.x;
  const bool ok = idx < a.total;
  int e = ok ? a.ids[idx] : -1;
  if (e < 0 || e >= a.E) e = a.E;  // parked on a dummy id, never written
  for (int i = threadIdx.x; i < kWavesHere * a.E; i += TH) in_wave[i] = 0;
  if (a.hist) {
    for (int x = threadIdx.x; x < a.E; x += TH) {
      int v, before;
      perm_hist_row_sums(a.hist + (long)x * perm_hist_stride(a.chunks), a.chunks, block * (TH / kPermChunk), &v, &before);
      all[x] = v;
      run[x] = before;
    }
    __syncthreads();
  } else {
    count_ids<TH>(a.ids, a.total, a.E, block * TH, run, all, lds + (2 + kWavesHere) * a.E);
  }
  const uint64_t same = match_same(e, a.nbits);
  const int before = __popcll(same & ((1ull << lane) - 1));
  if (e < a.E && before == 0) in_wave[wave * a.E + e] = __popcll(same);
  if (wave == 0) {  // first row of every expert = exclusive scan of the totals
    int carry = 0;
    for (int x0 = 0; x0 < a.E; x0 += 64) {
      const int x = x0 + lane;
      const int v = x < a.E ? all[x] : 0;
      const int inc = wave_inclusive_scan(v);
      if (x < a.E) {
        run[x] += carry + inc - v;
        if (block == 0) a.recv[x] = v;
      }
      carry += wave_last(inc);
    }
  }
  __syncthreads();
  if (e < a.E) {
    int pos = run[e] + before;
    for (int w = 0; w < wave; ++w) pos += in_wave[w * a.E + e];
    a.dst_exp[pos] = e;
    a.token_of_row[pos] = idx / a.topk;
    a.row_of_slot[idx] = pos;
  } else if (ok) {
    a.row_of_slot[idx] = -1;
  }
}

// One token by one wave: its row of n = 512 * NI values in every format of the layer's first block, at row t of the format's store.
template <int NI>
__device__ __forceinline__ void head_token(const HeadArgs& a, int t, int lane) {
  constexpr int n = 512 * NI;
  asm volatile("" : "+v"(lane));  // (else every address below becomes a register pair of its own that the loop over tokens carries along)
  const _Float16* srow = a.hidden + (long)t * n;
  v8h h[NI];
#pragma unroll
  for (int i = 0; i < NI; ++i) h[i] = *reinterpret_cast<const v8h*>(srow + lane * 8 + 512 * i);
  if (a.rotate != 0) {
    wave_rotate<NI>(h, lane, a.scale);
  } else {
#pragma unroll
    for (int i = 0; i < NI; ++i) h[i] = quiet(h[i]);
  }
  if (a.tags & 1u) {  // fp16: only when every row is rotated (else the GEMM reads the tokens where they are)
    _Float16* out = reinterpret_cast<_Float16*>(a.store[0]) + (long)t * n;
#pragma unroll
    for (int i = 0; i < NI; ++i) *reinterpret_cast<v8h*>(out + lane * 8 + 512 * i) = h[i];
  }
  // fp16 division: fp32 quotient of two fp16 values, rounded to fp16; a zero row gets 1 (quantize.cuh:258)
  auto scale_of = [](float amax, float upper) {
    const float scale = round_h(amax / upper);
    return scale == 0.0f ? 1.0f : scale;
  };
  if (a.tags & 8u) {  // tag 3: int4, one scale per 128 values = the 16 chunks held by an aligned group of 16 lanes
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      const int c = lane + 64 * i;
      HalfMax gmax;
      gmax.add(h[i]);
      const float scale = scale_of(row16_max_abs(gmax.get()), 7.0f);
      if ((c & 15) == 0) a.scales[3][(long)t * (n >> 7) + (c >> 4)] = (_Float16)scale;
      *reinterpret_cast<unsigned*>(a.store[3] + (long)t * (n / 2) + lane * 4 + 256 * i) = HalfDiv(scale).int4(h[i]);
    }
  }
  if ((a.tags & 0x26u) == 0) return;
  HalfMax half_max;
#pragma unroll
  for (int i = 0; i < NI; ++i) half_max.add(h[i]);
  const float amax = wave_max_abs(half_max.get());
  if (a.tags & 2u) {  // tag 1: int8 per token
    const float scale = scale_of(amax, 127.0f);
    const HalfDiv half(scale);
    if (lane == 0) a.scales[1][t] = (_Float16)scale;
#pragma unroll
    for (int i = 0; i < NI; ++i) *reinterpret_cast<uint2*>(a.store[1] + (long)t * n + lane * 8 + 512 * i) = half.int8(h[i]);
  }
  if (a.tags & 0x20u) {  // tag 5: fp8 e4m3 per token
    const float scale = scale_of(amax, 448.0f);
    const ScaleDiv div(scale);
    if (lane == 0) a.scales[5][t] = (_Float16)scale;
#pragma unroll
    for (int i = 0; i < NI; ++i) *reinterpret_cast<uint2*>(a.store[5] + (long)t * n + lane * 8 + 512 * i) = fp8_chunk_codes(h[i], div);
  }
  if (a.tags & 4u) {  // tag 2: int4 per token
    const float scale = scale_of(amax, 7.0f);
    const HalfDiv half(scale);
    if (lane == 0) a.scales[2][t] = (_Float16)scale;
#pragma unroll
    for (int i = 0; i < NI; ++i) *reinterpret_cast<unsigned*>(a.store[2] + (long)t * (n / 2) + lane * 4 + 256 * i) = half.int4(h[i]);
  }
}

// The tables of launch `wg` of both blocks' launches, from the ids (or from counts per chunk of them).
template <int TH, bool TOTALS, bool LONG>
__device__ __forceinline__ void head_plan(const HeadArgs& a, const PlanPair& pair, int wg, PlanShared& sh, int32_t* lds) {
  const PlanParams& p = pair.p[wg / pair.chunks];
  const int chunk = wg % pair.chunks;
  mxmoe_block_desc d{};
  const bool plans = __builtin_amdgcn_readfirstlane(threadIdx.x) < kPlanThreads;
  if (plans) d = plan_block_prepare(p, chunk, sh);
  if (a.hist) {
    for (int e = threadIdx.x; e < a.E; e += TH) {
      int v, before;
      perm_hist_row_sums(a.hist + (long)e * perm_hist_stride(a.chunks), a.chunks, 0, &v, &before);
      lds[e] = v;
    }
    __syncthreads();
  } else {
    count_ids<TH>(a.ids, a.total, a.E, 0, nullptr, lds, lds + a.E);
  }
  plan_block_body<TOTALS, LONG>(p, chunk, pair.chunks, lds, d, sh, plans);
}

// Workgroups: planning first (the longest chain of dependent steps), then the permutation's entries, then tokens, one per wave.
template <int NI, int TH, bool TOTALS, bool LONG>
__global__ void __launch_bounds__(TH) layer_head_kernel(const HeadArgs a, const PlanPair pair) {
  extern __shared__ __align__(16) int32_t head_lds[];
  const int plan_wgs = 2 * pair.chunks;
  int wg = blockIdx.x;
  if (wg < plan_wgs) {
    __builtin_amdgcn_s_setprio(3);  // one chain of dependent steps against the token waves' full issue slots on the same SIMDs
    __shared__ PlanShared sh;
    head_plan<TH, TOTALS, LONG>(a, pair, wg, sh, head_lds);
    return;
  }
  wg -= plan_wgs;
  if (wg < a.perm_wgs) {
    __builtin_amdgcn_s_setprio(2);
    head_scatter<TH>(a, wg, head_lds);
    return;
  }
  wg -= a.perm_wgs;
  const int token_wgs = (int)gridDim.x - plan_wgs - a.perm_wgs;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  for (int t = wg * (TH / 64) + wave; t < a.T; t += token_wgs * (TH / 64)) head_token<NI>(a, t, lane);
}

// Few tokens: a workgroup of gate_up finds its problem from the ids itself, so that the launch waits for no head.  The permutation and the tables of both blocks, which the launches behind
// need, are made beside it by the first workgroups.  What is left in front is the quantisation of the tokens (layer_tokens_kernel), where first blocks take quantised ones.
// Grid: (column tiles of a routed expert) x (1 for those, shared_slots rows of the shared expert's tiles, one row per expert that may have tokens).  A workgroup counts the ids in LDS, takes
// the slot-th expert with rows, lists its rows, and runs their row tiles one after the other (an expert of more than one is rare but under a skewed routing, and its
// weights come from L2 then).  DEAL (fp16 weights and more than 32 tokens): where at most half of the grid's rows have an expert, since most tokens take the same ones as the padding of a captured batch does, the others
// come to the experts in turn and take row tiles of those of more than two.  64 tokens on the same four of 60 fp16 experts, us a layer: one tile after the other 71.6, dealt 62.8 (behind a head, on the tiles of 64 rows, 62.1).
// Elsewhere one after the other is the better of both or what was gained does not pay the look (0.4 us of a layer): weight-only 32 tokens 28.3 / 28.7, 128 tokens 64.4 / 53.6 (79.3 behind a head), integer tiles of 32 rows 36.8 / 37.3.
// What a launch of few tokens consists of is latency: a layer's, with the head in front -> without, us: 64 experts top-6 and a shared one, w4a16 / w3a16, 29 -> 22 (1 token), 54 -> 46 (8),
// 77 -> 71 (32), w8a16 / w2a16 31 -> 23 (1), 65 -> 54 (8), 96 -> 85 (32); 60 experts top-4, w4a16 24 -> 18 (1), 55 -> 49 (16), 72 -> 68 (64), skewed 68 -> 64 (64), fp16 35 -> 27 (1),
// 108 -> 99 (8), 217 -> 212 (64); 8 experts of N = 28 672 / 4096, w4a16 64 -> 58 (1), 134 -> 126 (16).  One or two ids per thread: up to 512 of them, and no more tokens than the kernels for few rows take.
// 257 .. 512 of them, 64 experts top-6 and a shared one, us a layer, head -> none: w4a16 / w3a16 79 -> 74 (44 tokens), 77 -> 70 (52, skewed), w8a16 / w2a16 101 -> 87, 96 -> 84, fp16 249 -> 243 (44), 262 -> 252 (64),
// skewed 258 -> 249, w4a4 82 -> 78, 83 -> 80, 82 -> 76, w4a4 / w8a8 104 -> 98, 107 -> 101, 104 -> 97, beside fp8 106 -> 99, 108 -> 102, 104 -> 98, four formats 120 -> 112, 124 -> 117, 122 -> 113.
static_assert(kDirectEntries == 2 * kHeadSmall, "one or two ids per thread");
struct DirectArgs {
  const mxmoe_block_desc* desc;
  const uint8_t* hidden;
  _Float16* act;
  int hidden_size, inter, inter_shared;
  int cols, shared_rows, shared_slots;  // column tiles of a routed expert; rows of the grid that hold a row tile's column tiles of the shared expert, and all of its row tiles'
  int shared_step;                      // rows of such a tile
  unsigned topk_inverse;  // ceil(2^16 / top-k): (i * topk_inverse) >> 16 = i / top-k for i < kDirectEntries and top-k <= 64
  int entries;            // ids in LDS: one or two per thread
  int tile_lds;           // bytes of LDS that the tiles use
};
constexpr size_t direct_lds(int entries, int E) { return (size_t)entries * 4 + (size_t)kWaves * entries + (size_t)E * 4; }

// A tile type of the launch: whether it is that of a format, and the tag of its activations.  (fp8 or int8 codes: a kernel holds the tile of one of them.)
template <class T>
struct DirectTile;
template <int WBITS, int WAVES>
struct DirectTile<SkinnyWoTile<WBITS, 64, 1, WAVES>> {
  static constexpr int kTag = 0;
  __device__ static bool takes(int a_bits, int w_bits, int) { return a_bits >= 16 && w_bits == WBITS; }
  template <class RowOf>
  __device__ static __forceinline__ void run(const TileArgs& t, uint8_t* smem, RowOf&& row_of) {
    SkinnyWoTile<WBITS, 64, 1, WAVES>::template run_rows<true>(t, smem, row_of);
  }
};
template <Op OP>
struct DirectTile<WxAxNarrowTile<OP>> {
  static constexpr int kTag = OP == Op::I4 ? 2 : OP == Op::I8 ? 1 : 5;
  __device__ static bool takes(int a_bits, int, int gsize) { return a_bits == (OP == Op::I4 ? 4 : 8) && gsize == -1; }
  template <class RowOf>
  __device__ static __forceinline__ void run(const TileArgs& t, uint8_t* smem, RowOf&& row_of) {
    WxAxNarrowTile<OP>::template run_rows<true, false>(t, smem, row_of);
  }
};
template <>
struct DirectTile<WxAxGNarrowTile> {
  static constexpr int kTag = 3;
  __device__ static bool takes(int a_bits, int, int gsize) { return a_bits == 4 && gsize == 128; }
  template <class RowOf>
  __device__ static __forceinline__ void run(const TileArgs& t, uint8_t* smem, RowOf&& row_of) {
    WxAxGNarrowTile::run_rows<true>(t, smem, row_of);
  }
};

template <bool DEAL, class... Tiles>
__global__ void __launch_bounds__(kThreads, 3) layer_first_kernel(const HeadArgs a, const PlanPair pair, const DirectArgs x) {
  static_assert(kThreads == kHeadSmall && ((Tiles::BN == 64) && ...), "one or two ids per thread; 32 outputs a tile");
  static_assert(!DEAL || ((Tiles::BM == 16) && ...), "row tiles of one height are dealt out");
  extern __shared__ __align__(16) uint8_t first_lds[];
  const int col0 = blockIdx.x, E = a.E;
  int slot = (int)blockIdx.y - 1;
  if (slot < 0) {
    if (col0 < 2 * pair.chunks) {
      __builtin_amdgcn_s_setprio(3);
      constexpr size_t kPlanBytes = (sizeof(PlanShared) + 15) & ~(size_t)15;
      // (one planner body for every layer: nothing waits for it as long as gate_up runs)
      head_plan<kHeadSmall, true, true>(a, pair, col0, *reinterpret_cast<PlanShared*>(first_lds), reinterpret_cast<int32_t*>(first_lds + kPlanBytes));
    } else if (col0 < 2 * pair.chunks + a.perm_wgs) {
      __builtin_amdgcn_s_setprio(2);
      head_scatter<kHeadSmall>(a, col0 - 2 * pair.chunks, reinterpret_cast<int32_t*>(first_lds));
    }
    return;
  }
  const bool shared = slot < x.shared_slots;
  int col = col0, shared_m0 = 0;
  if (shared) {
    int row = slot;
    for (; row >= x.shared_rows; row -= x.shared_rows) shared_m0 += x.shared_step;
    col += row * x.cols;
  }
  if (col0 >= x.cols || col * 32 >= (shared ? x.inter_shared : x.inter)) return;
  slot -= x.shared_slots;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  int32_t* const all_ids = reinterpret_cast<int32_t*>(first_lds + x.tile_lds);
  uint8_t* const rows = reinterpret_cast<uint8_t*>(all_ids + x.entries) + wave * x.entries;  // this wave's copy of the problem's tokens
  int32_t* const count = all_ids + x.entries + kWaves * x.entries / 4;
  const bool two = x.entries > kThreads;
  const int id = (int)threadIdx.x < a.total ? gload<int>(a.ids + threadIdx.x) : -1;
  const int id2 = two && (int)threadIdx.x + kThreads < a.total ? gload<int>(a.ids + threadIdx.x + kThreads) : -1;
  for (int i = threadIdx.x; i < E; i += kThreads) count[i] = 0;
  __syncthreads();
  all_ids[threadIdx.x] = id;
  if (id >= 0 && id < E) atomicAdd(count + id, 1);
  if (two) {
    all_ids[threadIdx.x + kThreads] = id2;
    if (id2 >= 0 && id2 < E) atomicAdd(count + id2, 1);
  }
  __syncthreads();
  int e = shared ? E : -1, before = 0;  // the problem's expert; rows of the experts before it
  auto find = [&](int k) {              // the k-th expert with rows; returns k less those with rows where there are no more than k
    for (int x0 = 0; x0 < E; x0 += 64) {
      const int c = x0 + lane < E ? count[x0 + lane] : 0;
      const uint64_t hit = __ballot(c > 0);
      const int hits = __popcll(hit);
      uint64_t take = ~0ull;  // experts of these 64 in front of the problem's
      if (!shared && k < hits) {
        const uint64_t it = __ballot(c > 0 && __popcll(hit & ((1ull << lane) - 1)) == k);
        e = x0 + __builtin_ctzll(it);
        take = it - 1;
      }
      before += wave_last(wave_inclusive_scan((take >> lane & 1) ? c : 0));
      if (!shared && e >= 0) break;
      k -= hits;
    }
    return k;
  };
  const int past = find(slot);
  const int slots = (int)gridDim.y - 1 - x.shared_slots;
  int tile0 = 0;
  if (e < 0) {  // (every wave of the workgroup has come to the same)
    if constexpr (!DEAL) return;
    const int live = slot - past;
    if (live == 0 || 2 * live > slots) return;
    tile0 = slot / live;
    slot -= tile0 * live;
    before = 0;
    find(slot);
  }
  int M = 0;
  if (shared) {
    M = min(a.T, shared_m0 + x.shared_step);
  } else {
    for (int i0 = 0; i0 < a.total; i0 += 64) {
      const bool mine = all_ids[i0 + lane] == e;
      const uint64_t which = __ballot(mine);
      if (mine) rows[M + __popcll(which & ((1ull << lane) - 1))] = (uint8_t)((i0 + lane) * x.topk_inverse >> 16);
      M += __popcll(which);
    }
    __builtin_amdgcn_wave_barrier();
    if (DEAL && tile0 > 0 && (M <= 32 || tile0 * 16 >= M)) return;
  }
  TileArgs t;
  const mxmoe_block_desc* d = x.desc + e;
  t.B = reinterpret_cast<const uint8_t*>(cload(&d->B));
  t.sb = reinterpret_cast<const _Float16*>(cload(&d->scale_b));
  t.C = x.act + (long)before * x.inter;
  t.acc_dump = nullptr;
  t.M = M;
  t.N = 2 * (shared ? x.inter_shared : x.inter);
  t.K = x.hidden_size;
  t.tile_m = 0;
  t.tile_n = col;
  t.rows = nullptr;
  const int a_bits = cload(&d->q.a_bits), w_bits = cload(&d->q.w_bits), gsize = cload(&d->q.gsize);
  auto token_of = [&](int m) { return shared ? m : (int)rows[m]; };
  auto run = [&](auto type) {
    using T = typename decltype(type)::type;
    using D = DirectTile<T>;
    if (!D::takes(a_bits, w_bits, gsize)) return;
    t.A = D::kTag == 0 ? x.hidden : a.store[D::kTag];
    t.sa = D::kTag == 0 ? nullptr : a.scales[D::kTag];
    const int m_first = shared_m0 + tile0 * T::BM;
    int m_step = T::BM;
    if (DEAL && !shared && M > 32) {
      int live = 0;
      for (int x0 = 0; x0 < E; x0 += 64) live += __popcll(__ballot(x0 + lane < E && count[x0 + lane] > 0));
      if (2 * live <= slots) m_step *= (slots - slot + live - 1) / live;  // (as many rows of the grid come to this expert)
    }
#pragma unroll 1
    for (int m0 = m_first; m0 < M; m0 += m_step) {
      if (m0 > m_first) __syncthreads();  // the reduction behind the previous tile has been read
      t.row0 = m0;
      D::run(t, first_lds, token_of);
    }
  };
  (run(TileType<Tiles>{}), ...);
}

// The tokens of the launch behind it, one per wave (the token part of layer_head_kernel).
template <int NI>
__global__ void __launch_bounds__(kHeadSmall) layer_tokens_kernel(const HeadArgs a) {
  const int t = blockIdx.x * (kHeadSmall / 64) + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (t < a.T) head_token<NI>(a, t, threadIdx.x & 63);
}

// A launch for first blocks of few tokens, and its tiles.
using LaunchFirstFn = void (*)(const HeadArgs&, const PlanPair&, const DirectArgs&, dim3, size_t, hipStream_t);
struct FirstLaunch {
  LaunchFirstFn fn, deals;  // deals: with row tiles dealt to spare rows of the grid, or null
  std::vector<BranchInfo> tiles;
};
template <bool DEAL, class... Tiles>
void launch_first(const HeadArgs& a, const PlanPair& pair, const DirectArgs& x, dim3 grid, size_t lds, hipStream_t s) {
  hipLaunchKernelGGL((layer_first_kernel<DEAL, Tiles...>), grid, dim3(kThreads), lds, s, a, pair, x);
}
template <class... Tiles>
FirstLaunch first_of() {
  LaunchFirstFn deals = nullptr;
  if constexpr (((Tiles::kABits == 16) && ...) && ((Tiles::kWBits == 16) || ...)) deals = &launch_first<true, Tiles...>;
  return {&launch_first<false, Tiles...>, deals, {BranchOf<Tiles>::get()...}};
}
template <int WBITS>
using FewTokenTile = SkinnyWoTile<WBITS, 64, 1, 3>;

// Whether a launch's tile computes what kernel k does for a block of format f, to the bit, whatever its rows: k has that tile, and where its tables could name another one of the format, the sums are the
// same in any (integers; group-scaled w4a4, whose additions are in the order of the groups).
static bool same_sums(const FusedKernel& k, Fmt f, const BranchInfo& tile) {
  bool has = false;
  for (const BranchInfo& b : k.branches) {
    if (b.fmt != f) continue;
    const bool same = b.BM == tile.BM && b.BN == tile.BN && b.variant == tile.variant;
    if (!same && (b.variant || tile.variant || !(integer_sums((int)f) || f == Fmt::W4A4G128))) return false;
    has = has || same;
  }
  return has;
}

// The launch for a layer whose first block runs on kernel k: the one of fewest formats that takes each block as k would, or null (a kernel for many rows; one whose tables may take a larger tile with other
// sums than the 64-channel one's).  With fp16 weights and more tokens than two row tiles hold, the one that deals row tiles out.
static LaunchFirstFn first_launch_of(const FusedKernel& k, const mxmoe_block_desc* h_desc, int et, int num_tokens) {
  using I4 = WxAxNarrowTile<Op::I4>;
  using I8 = WxAxNarrowTile<Op::I8>;
  using F8 = WxAxNarrowTile<Op::F8>;
  static const FirstLaunch launches[] = {
      first_of<FewTokenTile<4>, FewTokenTile<3>, FewTokenTile<2>>(),
      first_of<I4, I8>(),
      first_of<I4, F8>(),
      first_of<FewTokenTile<4>, FewTokenTile<3>, FewTokenTile<2>, FewTokenTile<8>, FewTokenTile<16>>(),
      first_of<I4, I8, WxAxGNarrowTile, FewTokenTile<4>, FewTokenTile<3>, FewTokenTile<2>, FewTokenTile<8>>(),
      first_of<I4, F8, WxAxGNarrowTile, FewTokenTile<4>, FewTokenTile<3>, FewTokenTile<2>, FewTokenTile<8>>(),
  };
  auto takes = [&](const FirstLaunch& l, Fmt f) { return std::any_of(l.tiles.begin(), l.tiles.end(), [&](const BranchInfo& t) { return t.fmt == f && same_sums(k, f, t); }); };
  for (const FirstLaunch& l : launches) {
    bool all = true, fp16 = false;
    for (int i = 0; i < et && all; ++i) {
      const Fmt f = (Fmt)fmt_of(h_desc[i].q);
      all = takes(l, f);
      fp16 = fp16 || f == Fmt::FP16;
    }
    if (all) return fp16 && l.deals && num_tokens > 32 ? l.deals : l.fn;
  }
  return nullptr;
}

// gate_up without a head in front of it, as far as it follows from the layer, the batch and kernel `kg` of the first block: its launch, or null where the layer has a head.  The one place of this
// rule: the choice of the kernel asks for it (mxmoe_layer_starts_with_gate_up) and so does the handle.
struct FirstForm {
  LaunchFirstFn fn;
  DirectArgs x;
  dim3 grid;
  size_t lds;
};
constexpr size_t kFirstLdsMax = 40 * 1024;  // (counters of many experts would take the room of a workgroup)
static FirstForm first_form(const mxmoe_layer_desc* d, const FusedKernel& kg) {
  const int et = d->num_experts + (d->has_shared ? 1 : 0), total = d->num_tokens * d->topk;
  FirstForm f{};
  if (d->num_tokens > kDirectTokens || total > kDirectEntries || d->topk > 64) return f;
  for (int i = 0; i < et; ++i) {
    const mxmoe_block_desc& b = d->h_gate_up[i];
    const int n = i < d->num_experts ? d->inter : d->inter_shared;
    if ((int)b.N != 2 * n || (int)b.K != d->hidden || n % 32) return f;
    if (d->rotate == 2 && act_tag_of(b.q) == 0) return f;  // (rotated fp16 tokens are made by a head)
  }
  DirectArgs& x = f.x;
  x.desc = d->d_gate_up;
  x.act = reinterpret_cast<_Float16*>(d->act);
  x.hidden_size = d->hidden;
  x.inter = d->inter;
  x.inter_shared = d->has_shared ? d->inter_shared : 0;
  x.cols = d->inter / 32;
  x.shared_rows = (x.inter_shared / 32 + x.cols - 1) / x.cols;
  x.shared_step = d->has_shared && d->h_gate_up[d->num_experts].q.a_bits < 16 && d->h_gate_up[d->num_experts].q.gsize != 128 ? 32 : 16;  // (BM of the format's tile)
  x.shared_slots = x.shared_rows * ((d->num_tokens + x.shared_step - 1) / x.shared_step);
  x.topk_inverse = (65536 + d->topk - 1) / d->topk;
  x.entries = total <= kThreads ? kThreads : kDirectEntries;
  x.tile_lds = kg.lds_bytes;
  const int front = 2 * PlanLayout(et).chunks + (total + kHeadSmall - 1) / kHeadSmall;  // workgroups that plan, and that write the permutation
  f.grid = dim3(std::max(x.cols, front), 1 + x.shared_slots + std::min(total, d->num_experts));
  f.lds = std::max(kg.lds_bytes + direct_lds(x.entries, d->num_experts), sizeof(PlanShared) + 16 + (size_t)(2 + kHeadSmall / 64 + 2 * kCountCopies) * d->num_experts * sizeof(int32_t));
  if (f.lds <= kFirstLdsMax) f.fn = first_launch_of(kg, d->h_gate_up, et, d->num_tokens);
  return f;
}

// What a layer keeps for one (tokens, top-k): its description and both launches' planning parameters.
struct LayerForward {
  mxmoe_layer_desc d;
  HeadArgs head;
  PlanPair pair;
  int et, threads, token_wgs;
  bool fp16_first;   // a first block reads the tokens as they are (its tiles load them straight into LDS)
  bool rows_step;    // a second block takes quantised (or rotated) rows
  RowsBehind rows;
  FirstForm first;
};

static int check_launch() {
  const hipError_t e = hipGetLastError();
  if (e == hipSuccess) return 0;
  last_error() = std::string("kernel launch failed: ") + hipGetErrorString(e);
  return 4;
}

}  // namespace mxmoe

using namespace mxmoe;

extern "C" {

int mxmoe_layer_supported(const mxmoe_layer_desc* d) {
  if (!d || !d->h_gate_up || !d->h_down) return 0;
  const int k = d->hidden, e = d->num_experts, et = e + (d->has_shared ? 1 : 0);
  if (d->num_tokens <= 0 || d->topk <= 0 || e <= 0 || e > kHeadMaxExperts || (long)d->num_tokens * d->topk > (1l << 24)) return 0;
  if (k < 512 || k > 4096 || (k & (k - 1)) || d->inter <= 0) return 0;
  const long total = (long)d->num_tokens * d->topk, blocks = (total + kPermChunk - 1) / kPermChunk;
  if (total > kHeadCountMax && blocks * e > kPermFusedScanMax) return 0;
  if ((long)d->num_tokens * k * 2 >= (long)kGatherBytes) return 0;  // offsets into a token store
  const int kg = resolve_kernel(d->kernel_gate_up, d->h_gate_up, et), kd = resolve_kernel(d->kernel_down, d->h_down, et);
  if (kg < 0 || kd < 0 || !registry()[kg].launch_gate_up) return 0;
  for (int i = 0; i < et; ++i) {
    const mxmoe_block_desc& g = d->h_gate_up[i];
    if (g.N % 64 || (long)g.N * g.K * 2 >= (long)kGatherBytes) return 0;  // gate and up each whole 32-channel blocks; offsets into fp16 weights
    if (act_tag_of(g.q) < 0 || act_tag_of(g.q) == 4 || act_tag_of(d->h_down[i].q) < 0 || act_tag_of(d->h_down[i].q) == 4) return 0;
  }
  return 1;
}

int mxmoe_layer_create(const mxmoe_layer_desc* d, void** handle) {
  if (!d || !handle) {
    last_error() = "null pointer";
    return 5;
  }
  if (!mxmoe_layer_supported(d)) {
    last_error() = "layer shape not supported by the short form of the forward";
    return 3;
  }
  const int et = d->num_experts + (d->has_shared ? 1 : 0);
  if (!d->d_gate_up || !d->d_down || !d->act || !d->down_inp || !d->down_scales || !d->down_out || !d->plan_gate_up || !d->plan_down || !d->dst_exp || !d->token_of_row ||
      !d->row_of_slot || !d->iota || !d->recv || !d->workspace || (reinterpret_cast<uintptr_t>(d->workspace) & 15)) {
    last_error() = "null pointer, or a workspace that is not 16-byte aligned";
    return 5;
  }
  std::unique_ptr<LayerForward> f(new LayerForward());
  f->d = *d;
  f->et = et;
  const int shared_rows = d->has_shared ? d->num_tokens : 0;
  unsigned tags = 0, tags_behind = 0;
  for (int i = 0; i < et; ++i) {
    tags |= 1u << act_tag_of(d->h_gate_up[i].q);
    tags_behind |= 1u << act_tag_of(d->h_down[i].q);
  }
  f->fp16_first = (tags & 1u) && d->rotate != 2;
  if (f->fp16_first) tags &= ~1u;
  for (int i = 0; i < kNumTags; ++i)
    if ((tags >> i & 1) && (!d->token_store[i] || (i > 0 && !d->token_scales[i]))) {
      last_error() = "missing token store of a format the layer uses";
      return 5;
    }
  f->rows_step = d->rotate == 2 || (tags_behind & ~1u);

  HeadArgs& h = f->head;
  h = HeadArgs{};
  h.total = d->num_tokens * d->topk;
  h.E = d->num_experts;
  h.topk = d->topk;
  h.nbits = 1;
  while ((1 << h.nbits) <= d->num_experts) ++h.nbits;  // ids 0..E (E = parked lanes)
  f->threads = h.total <= kHeadSmallMax ? kHeadSmall : kHeadLarge;
  h.perm_wgs = (h.total + f->threads - 1) / f->threads;
  h.chunks = (h.total + kPermChunk - 1) / kPermChunk;
  h.hist = h.total > kHeadCountMax ? reinterpret_cast<const int32_t*>(d->workspace) : nullptr;
  h.recv = d->recv;
  h.dst_exp = d->dst_exp;
  h.token_of_row = d->token_of_row;
  h.row_of_slot = d->row_of_slot;
  h.T = d->num_tokens;
  h.tags = tags;
  h.rotate = d->rotate;
  h.scale = 1.0f / sqrtf((float)d->hidden);
  for (int i = 0; i < kNumTags; ++i) {
    h.store[i] = reinterpret_cast<uint8_t*>(d->token_store[i]);
    h.scales[i] = reinterpret_cast<_Float16*>(d->token_scales[i]);
  }
  int dev = 0, cus = 256;
  (void)hipGetDevice(&dev);
  (void)hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
  const int per_wg = f->threads / 64;
  f->token_wgs = tags ? std::min((d->num_tokens + per_wg - 1) / per_wg, cus * 32 / per_wg) : 0;

  auto fill = [&](PlanParams& p, int kernel_id, const mxmoe_block_desc* desc, const mxmoe_block_desc* h_desc, void* out, void* plan) {
    p = PlanParams{};
    const int kid = resolve_kernel(kernel_id, h_desc, et);
    p.recv = d->recv;
    p.desc = desc;
    p.out = reinterpret_cast<uint8_t*>(out);
    p.plan = reinterpret_cast<uint8_t*>(plan);
    p.E = d->num_experts;
    p.Et = et;
    p.shared_rows = shared_rows;
    p.info = plan_info_of_block(registry()[kid], h_desc, et);
    // a problem has two row segments only with more rows than its format's lowest shape: for a handful of tokens the planner need not look for pairs
    int low = INT_MAX;
    for (const BranchInfo& b : registry()[kid].branches)
      if (!is_weight_only(b.fmt)) low = std::min(low, b.BM);
    if ((long)d->num_tokens * d->topk <= low) p.info.may_pair = 0;
    if ((long)d->num_tokens * d->topk <= 32) p.info.has_slim = 0;  // (nor for 128-row tiles)
    return kid;
  };
  f->d.kernel_gate_up = fill(f->pair.p[0], d->kernel_gate_up, d->d_gate_up, d->h_gate_up, d->act, d->plan_gate_up);
  f->d.kernel_down = fill(f->pair.p[1], d->kernel_down, d->d_down, d->h_down, d->down_out, d->plan_down);
  f->pair.chunks = PlanLayout(et).chunks;
  LayerForm& g = f->pair.p[0].form;
  g.kind = LayerForm::kGateUp;
  for (int i = 0; i < kNumTags; ++i) {
    g.store[i] = reinterpret_cast<const uint8_t*>(d->token_store[i]);
    g.scales[i] = reinterpret_cast<const uint8_t*>(d->token_scales[i]);
  }
  g.token_of_row = d->token_of_row;
  g.iota = d->iota;
  PlanParams& pd = f->pair.p[1];
  pd.inp = reinterpret_cast<const uint8_t*>(d->down_inp);
  pd.scale = reinterpret_cast<const uint8_t*>(d->down_scales);
  pd.form.kind = d->rotate == 2 ? LayerForm::kPlain : LayerForm::kBehind;
  pd.form.act = reinterpret_cast<const uint8_t*>(d->act);

  f->first = first_form(d, registry()[f->d.kernel_gate_up]);

  RowsBehind& r = f->rows;
  r = RowsBehind{};
  r.rows = d->act;
  r.plan_gate_up = reinterpret_cast<const uint8_t*>(d->plan_gate_up);
  r.plan_down = reinterpret_cast<const uint8_t*>(d->plan_down);
  r.inp_store = reinterpret_cast<uint8_t*>(d->down_inp);
  r.scale_store = reinterpret_cast<_Float16*>(d->down_scales);
  r.dst_exp = d->dst_exp;
  r.n = d->inter;
  r.n_shared = d->inter_shared;
  r.rows_capacity = h.total;
  r.num_tokens = d->num_tokens;
  r.num_experts = d->num_experts;
  r.has_shared = d->has_shared != 0;
  r.variants = (tags_behind & 0x30u) != 0;
  r.rotate = d->rotate;
  r.had_k = d->had_k;
  r.had_f = d->had_f;
  r.had_signs = d->had_signs;
  *handle = f.release();
  return 0;
}

int mxmoe_layer_starts_with_gate_up(const mxmoe_layer_desc* d) {
  if (!mxmoe_layer_supported(d)) return 0;
  return first_form(d, registry()[resolve_kernel(d->kernel_gate_up, d->h_gate_up, d->num_experts + (d->has_shared ? 1 : 0))]).fn != nullptr;
}

int mxmoe_layer_has_head(const void* handle) { return handle && !reinterpret_cast<const LayerForward*>(handle)->first.fn; }

void mxmoe_layer_destroy(void* handle) { delete reinterpret_cast<LayerForward*>(handle); }

int mxmoe_layer_run(const void* handle, const void* hidden, const int32_t* topk_ids, const float* topk_weights, void* out, void* stream) {
  if (!handle || !hidden || !topk_ids || !topk_weights || !out) {
    last_error() = "null pointer";
    return 5;
  }
  const LayerForward& f = *reinterpret_cast<const LayerForward*>(handle);
  const mxmoe_layer_desc& d = f.d;
  if (f.fp16_first && (reinterpret_cast<uintptr_t>(hidden) & 15)) {
    last_error() = "hidden must be 16-byte aligned: first blocks of 16-bit activations read the tokens where they are, in 16-byte pieces";
    return 3;
  }
  hipStream_t s = (hipStream_t)stream;
  HeadArgs h = f.head;
  PlanPair pair = f.pair;
  h.ids = topk_ids;
  h.hidden = reinterpret_cast<const _Float16*>(hidden);
  if (f.fp16_first) pair.p[0].form.store[0] = reinterpret_cast<const uint8_t*>(hidden);
  const FusedKernel &kg = registry()[d.kernel_gate_up], &kd = registry()[d.kernel_down];
  auto gemm = [&](LaunchPlannedFn fn, const FusedKernel& k, const void* plan, int launch_grid) {
    for (int c = 0; c < pair.chunks; ++c) {
      const hipError_t e = fn(reinterpret_cast<const FusedArgs*>(reinterpret_cast<const uint8_t*>(plan) + c * kFusedArgsStride), launch_grid, k.lds_bytes, s);
      if (e != hipSuccess) {
        last_error() = std::string("kernel launch failed: ") + hipGetErrorString(e);
        return 4;
      }
    }
    return 0;
  };
  // by the row length: f(number of 512-value pieces)
  auto by_length = [&](auto&& f) {
    switch (d.hidden / 512) {
      case 1: f(std::integral_constant<int, 1>{}); break;
      case 2: f(std::integral_constant<int, 2>{}); break;
      case 4: f(std::integral_constant<int, 4>{}); break;
      default: f(std::integral_constant<int, 8>{}); break;
    }
  };
  if (f.first.fn) {
    DirectArgs x = f.first.x;
    x.hidden = reinterpret_cast<const uint8_t*>(hidden);
    if (h.tags) by_length([&](auto ni) { hipLaunchKernelGGL((layer_tokens_kernel<decltype(ni)::value>), dim3((h.T + 3) / 4), dim3(kHeadSmall), 0, s, h); });
    if (const int rc = check_launch()) return rc;
    f.first.fn(h, pair, x, f.first.grid, f.first.lds, s);
    if (const int rc = check_launch()) return rc;
  } else {
    if (h.hist) launch_perm_hist(topk_ids, h.total, h.E, const_cast<int32_t*>(h.hist), true, s);
    const dim3 grid(2 * pair.chunks + h.perm_wgs + f.token_wgs), block(f.threads);
    const size_t lds = (size_t)(2 + f.threads / 64 + 2 * kCountCopies) * h.E * sizeof(int32_t);
    by_length([&](auto ni) {
      constexpr int NI = decltype(ni)::value;
      pair.with_body([&](auto totals, auto longs) {
        constexpr bool kTotals = decltype(totals)::value, kLong = decltype(longs)::value;
        if (f.threads == kHeadSmall) hipLaunchKernelGGL((layer_head_kernel<NI, kHeadSmall, kTotals, kLong>), grid, block, lds, s, h, pair);
        else hipLaunchKernelGGL((layer_head_kernel<NI, kHeadLarge, kTotals, kLong>), grid, block, lds, s, h, pair);
      });
    });
    if (const int rc = check_launch()) return rc;
    if (const int rc = gemm(kg.launch_gate_up, kg, d.plan_gate_up, d.grid_gate_up)) return rc;
  }
  if (f.rows_step)
    if (const int rc = quant_rows_behind(f.rows, s)) return rc;
  if (const int rc = gemm(kd.launch_planned, kd, d.plan_down, d.grid_down)) return rc;
  return mxmoe_combine_planned(d.down_out, d.plan_down, f.et, topk_weights, d.row_of_slot, d.num_tokens, d.topk, d.hidden, out, stream);
}

}  // extern "C"

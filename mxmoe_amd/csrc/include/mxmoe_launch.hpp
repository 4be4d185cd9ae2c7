// Fused one-launch GroupGEMM: tile scheduler, per-problem branch dispatch, host launcher and kernel registry.
//
// Mirrors the reference's generated `groupgemm_hz_fused_<i>` pair (kernel + host launcher,
// mxmoe/kernels/compose_kernel.py:150-295, mxmoe/kernels/kernel_sketch.py:82-145) with these differences:
//  * one workgroup per tile instead of a persistent grid: the hardware dispatcher hands out tiles as
//    workgroups retire, which balances the mixed tile costs of a mixed-precision launch;
//  * the tile prefix sum and the per-problem branch index travel in the kernel-argument segment, so a launch
//    performs no allocation, no host-to-device copy and no synchronisation (the reference does
//    cudaMalloc + cudaMemcpy + cudaFree per call, kernel_sketch.py:102-104,142-143);
//  * workgroup ids are remapped so that each of the 8 XCDs (one L2 each; workgroups are dealt round-robin)
//    receives one contiguous run of the tile list, i.e. whole experts, and re-reads of an expert's weights
//    and activations by neighbouring tiles stay inside one L2;
//  * a qcfg may own several tile shapes; the host picks one per problem from its row count.
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdio>
#include <cstring>
#include <string>
#include <vector>

#include "mxmoe_tiles.hpp"
#include "mxmoe_grp_tiles.hpp"
#include "mxmoe_few_tiles.hpp"
#include "mxmoe_bf6_tiles.hpp"
#include "mxmoe_wo_tiles.hpp"

namespace mxmoe {

constexpr int kMaxProblems = 120;  // per launch (the tables ride in the 4 KB kernel argument block); longer problem lists are split into several launches
constexpr int kMaxEntries = 2 * kMaxProblems;  // a problem is run as at most two row segments, each with its own tile shape
constexpr int kNumXcd = 8;
constexpr int kMaxPhases = 8;

struct FusedArgs {
  const uint8_t* const* As;
  const uint8_t* const* Bs;
  const _Float16* const* sa;
  const _Float16* const* sb;
  _Float16* const* Cs;
  int32_t* const* acc;  // optional accumulator dumps (null, or per-problem pointers which may themselves be null)
  const mxmoe_dim3* sizes;
  int problem_offset;   // first problem of this launch inside the arrays above
  int num_entries;
  int total_tiles;
  // Phases: the entries are sorted so that the most expensive tile shapes come first (workgroups are dispatched in index order,
  // so the cheap tiles fill the tail of the launch).  Phase p covers tiles [phase_tile0[p], phase_tile0[p+1]) and workgroups
  // [phase_wg0[p], phase_wg0[p+1]); inside a phase, workgroup v maps to tile (v % 8) * chunk + v / 8 so that each XCD (one L2)
  // works on a contiguous run of tiles.
  int num_phases;
  int phase_tile0[kMaxPhases + 1];
  int phase_wg0[kMaxPhases + 1];
  // Bit p set: phase p maps workgroup v to tile v.  For the skinny weight-only tiles, which share no operand with their neighbours
  // (every tile streams its own weights once): dealing them round-robin to the XCDs balances the memory traffic tile by tile,
  // where contiguous runs would leave the XCD that holds a few long problems behind.
  int phase_flat;
  // One entry per row segment of a problem, 16 bytes so that a workgroup fetches its entry with one scalar load: first tile of the
  // entry (exclusive prefix sum of tiles), first row of the segment inside its problem, rows of the segment, and
  // problem (relative to problem_offset) | tile type << 16 | the fields of a pair (pair_word).
  struct Entry {
    int first, row0, rows, problem_branch;
  };
  Entry entry[kMaxEntries];
  const int32_t* const* rows;  // gate_up form (see TileArgs): per problem, the activation row behind each of its rows
};
static_assert(sizeof(FusedArgs) <= 4096, "kernel arguments are limited to 4 KB");

// Activation bytes that a group of row tiles may hold (see locate_tile): half of an XCD's 4 MB L2.
#ifndef MXMOE_GROUP_BYTES
#define MXMOE_GROUP_BYTES (2 << 20)
#endif

// A pair: the two row segments of one problem as neighbouring entries whose tiles are dealt out column by column, so that the tiles of both
// shapes that read a block of weight rows run at the same time and the block is fetched once.  (As phases of their own, the launch went through
// all of its weights a second time for the remainder tiles; with more weights than the caches hold, that was the launch's time.)
// Both shapes' column tiles are equally wide.  Fields of problem_branch, on both entries: bits 21 .. 28 the second segment's row tiles (0: no pair), bit 29 set on
// the second entry.
constexpr unsigned kPairSecond = 1u << 29;
__host__ __device__ inline int entry_problem(int pb) { return pb & 0xFFFF; }
__host__ __device__ inline int entry_branch(int pb) { return (int)((unsigned)pb >> 16 & 31u); }
__host__ __device__ inline int pair_width(int pb) { return (int)((unsigned)pb >> 21 & 255u); }

// Where a tile of an entry (of a pair: of both entries) lies.
struct TileAt {
  int m, n;
  bool second;  // in the pair's second segment
};
// Local index -> (row tile, column tile) as tile_scheduler.cuh:40-49, but row tile fastest: neighbouring workgroups then share
// one block of weight rows and sweep the problem's activations.  The 64 workgroups that an XCD runs at a time only share
// what its 4 MB L2 still holds, and they drift apart along K, so a problem whose activations exceed the L2 ends up
// streaming them once per column tile.  Such a problem is walked in groups of row tiles holding at most 2 MB of
// activations, each group against all column tiles: the group's activations stay resident whatever the drift, and a block
// of weights is fetched once per group by row tiles that start together.  The plain order is kept where the estimate of
// its traffic (activations once per 64 / grid_m column tiles, weights once) is below half of the grouped order's (weights
// once per group, activations once): very long rows, of which only one or two row tiles fit.
// BM, BN, bits: of the entry's tile shape (of a pair: of its first segment, which the last group shares with the second).
__host__ __device__ __forceinline__ TileAt locate_tile(int local, int rows, int N, int K, int BM, int BN, int a_bits, int w_bits, int problem_branch) {
  const int grid_m = (rows + BM - 1) / BM;
  const int beside = pair_width(problem_branch);
  if (grid_m == 1 && beside == 0) return TileAt{0, local, false};
  const int raw_bytes = BM * (K / 8) * a_bits, tile_bytes = raw_bytes > 1 ? raw_bytes : 1;
  int g = 0, r = local, rows_g = grid_m;  // group, index inside it, its row tiles
  bool last = true;
  if ((long)grid_m * tile_bytes > MXMOE_GROUP_BYTES && tile_bytes <= MXMOE_GROUP_BYTES) {  // (a single row tile beyond the budget cannot stay resident either)
    const int rg = MXMOE_GROUP_BYTES / tile_bytes, groups = (grid_m + rg - 1) / rg;
    const int grid_n = (N + BN - 1) / BN;
    const float a_bytes = (float)grid_m * (float)tile_bytes;
    const float b_bytes = (float)N * (float)(K / 8) * (float)w_bits;
    const float cols = (float)grid_n * (float)grid_m * (1.0f / 64.0f);
    if ((float)groups * b_bytes + a_bytes < 2.0f * ((cols > 1.0f ? cols : 1.0f) * a_bytes + b_bytes)) {
      g = local / (rg * grid_n);
      g = g < groups ? g : groups - 1;
      r = local - g * (rg * grid_n);
      last = g == groups - 1;
      rows_g = last ? grid_m - g * rg : rg;
      g *= rg;
    }
  }
  const int width = rows_g + (last ? beside : 0);
  const int col = r / width, at = r - col * width;
  if (beside == 0 || at < rows_g) return TileAt{g + at, col, false};
  return TileAt{at - rows_g, col, true};
}

// Whether a kernel of these tiles may be given pairs (PlanInfo::may_pair): some of them are of a format that has them (weight-only tiles have 16-bit activations and
// less than 16 bits a weight, group-scaled ones are bound by their arithmetic), and it is not one of those for few rows.  Those run lists of at most 64 rows, which
// have nothing to pair, in a few microseconds, of which the looking for pairs was a part.
template <class T>
constexpr bool kPairs = T::kABits == T::kWBits;
template <int BM>
constexpr bool kPairs<WxAxGTile<BM>> = false;
template <>
inline constexpr bool kPairs<WxAxGNarrowTile> = false;
template <class T>
constexpr bool kNarrow = false;
template <Op OP>
constexpr bool kNarrow<WxAxNarrowTile<OP>> = true;
template <class... Tiles>
constexpr bool kMayPair = (kPairs<Tiles> || ...) && !(kNarrow<Tiles> || ...);

// f(TileType<T>{}) with T the tile of branch `branch`: the compile-time dispatch over a kernel's tiles.
template <class T>
struct TileType {
  using type = T;
};
template <int I, class F>
__device__ __forceinline__ void with_branch(std::integral_constant<int, I>, int, F&&) {}
template <class T, class... Rest, int I, class F>
__device__ __forceinline__ void with_branch(std::integral_constant<int, I>, int branch, F&& f) {
  if (branch == I) f(TileType<T>{});
  else with_branch<Rest...>(std::integral_constant<int, I + 1>{}, branch, f);
}

// Waves per SIMD the register allocator should aim for: 2 (two co-resident workgroups per CU, 256 registers per lane) unless a
// tile keeps more than 128 accumulator registers per lane, which needs the full 512-register budget of a lone wave.
// A kernel made only of tiles that ask for more waves (the few-token weight-only tiles: latency-bound streams that gain from every
// further workgroup in flight) is compiled for the smallest number any of its tiles asks for.
template <class... Tiles>
constexpr int kWavesPerSimd = ((Tiles::kAccRegs > 128) || ...) ? 1 : std::min({Tiles::kWavesWanted...});

// Tables are read through the constant address space: what a workgroup reads from them is the same for all lanes and is not
// written while the kernel runs (a planned launch's tables were written by the planning kernel before it), so every read is a
// scalar load, whether the table came in the kernel arguments or lies in device memory.
#define MXMOE_CONST __attribute__((address_space(4)))
template <class T>
__device__ __forceinline__ T cload(const T* p) {
  return *(const MXMOE_CONST T*)(p);
}
__host__ __device__ __forceinline__ int uni(int v) {
#if defined(__HIP_DEVICE_COMPILE__)
  return __builtin_amdgcn_readfirstlane(v);
#else
  return v;
#endif
}

// Tile that workgroup `wg` of a launch runs, or -1 when it has none (tile_scheduler.cuh:25-37 maps a persistent block's linear
// index the same way; here the index is the workgroup id).  Compiled for the host as well: the scheduler tests replay a whole grid
// through this very function.
template <class ArgsPtr>
__host__ __device__ __forceinline__ int tile_of_workgroup(ArgsPtr args, int wg) {
  const int num_phases = uni(args->num_phases);
  // A planned launch is sized for the worst routing: workgroups past the last phase have no tile (without this test they would
  // be folded back into the last phase by the XCD remap below and run one of its tiles a second time), and a launch whose plan
  // holds no tile at all has nothing else in its tables that may be read.
  if (num_phases <= 0 || wg >= uni(args->phase_wg0[num_phases])) return -1;
  int ph = 0;
  while (ph + 1 < num_phases && wg >= uni(args->phase_wg0[ph + 1])) ++ph;
  const int v = wg - uni(args->phase_wg0[ph]);
  const int tile0 = uni(args->phase_tile0[ph]);
  const int ntiles = uni(args->phase_tile0[ph + 1]) - tile0;
  const int chunk = (ntiles + kNumXcd - 1) / kNumXcd;
  const int pt = (uni(args->phase_flat) >> ph & 1) ? v : (v % kNumXcd) * chunk + v / kNumXcd;
  return pt < ntiles ? tile0 + pt : -1;
}

template <bool GU, class ArgsPtr, class... Tiles>
__device__ __forceinline__ void fused_body(ArgsPtr args, uint8_t* smem) {
  const int tile = tile_of_workgroup(args, (int)blockIdx.x);
  if (tile < 0) return;
  // tile_scheduler.cuh:25-37 — the entry that holds the tile: last entry whose first tile is <= tile (binary search here; all
  // indices are wave-uniform, so these are scalar loads)
  int lo = 0, hi = uni(args->num_entries) - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (uni(args->entry[mid].first) <= tile) lo = mid; else hi = mid - 1;
  }
  int en_first = uni(args->entry[lo].first), en_row0 = uni(args->entry[lo].row0), en_rows = uni(args->entry[lo].rows), en_pb = uni(args->entry[lo].problem_branch);
  if (kMayPair<Tiles...> && ((unsigned)en_pb & kPairSecond)) {  // found by its index among the second segment's: a pair's tiles are counted from the first segment on
    --lo;
    en_first = uni(args->entry[lo].first);
    en_row0 = uni(args->entry[lo].row0);
    en_rows = uni(args->entry[lo].rows);
    en_pb = uni(args->entry[lo].problem_branch);
  }
  const int gp = uni(args->problem_offset) + entry_problem(en_pb);
  const mxmoe_dim3* sizes = args->sizes;
  const uint8_t* const* As = args->As;
  const uint8_t* const* Bs = args->Bs;
  const _Float16* const* sa = args->sa;
  const _Float16* const* sb = args->sb;
  _Float16* const* Cs = args->Cs;
  int32_t* const* acc = args->acc;
  TileArgs t;
  t.A = cload(As + gp);
  t.B = cload(Bs + gp);
  t.sa = sa ? cload(sa + gp) : nullptr;
  t.sb = sb ? cload(sb + gp) : nullptr;
  t.C = cload(Cs + gp);
  t.acc_dump = acc ? cload(acc + gp) : nullptr;
  t.N = uni((int)cload(&sizes[gp].y));
  t.K = uni((int)cload(&sizes[gp].z));
  t.rows = nullptr;
  if constexpr (GU) t.rows = cload(args->rows + gp);
  int branch = entry_branch(en_pb), local = tile - en_first;
  if (kMayPair<Tiles...> && pair_width(en_pb) != 0) {  // which of the two shapes it is comes out of the place; from here on a tile like any other
    TileAt at{0, 0, false};
    int bm = 0;
    with_branch<Tiles...>(std::integral_constant<int, 0>{}, branch, [&](auto tile_type) {
      using T = typename decltype(tile_type)::type;
      at = locate_tile(local, en_rows, t.N, t.K, T::BM, T::BN, T::kABits, T::kWBits, en_pb);
      bm = T::BM;
    });
    if (uni(at.second)) {
      en_row0 = uni(args->entry[lo + 1].row0);
      en_rows = uni(args->entry[lo + 1].rows);
      branch = entry_branch(uni(args->entry[lo + 1].problem_branch));
      local = uni(at.n * pair_width(en_pb) + at.m);
    } else {  // (the first segment is whole tiles) as the one row tile of its own segment
      en_row0 += uni(at.m * bm);
      en_rows = uni(bm);
      local = uni(at.n);
    }
  }
  t.row0 = en_row0;
  t.M = t.row0 + en_rows;  // rows past the segment are treated like rows past the problem
  with_branch<Tiles...>(std::integral_constant<int, 0>{}, branch, [&](auto tile_type) {
    using T = typename decltype(tile_type)::type;
    const TileAt at = locate_tile(local, en_rows, t.N, t.K, T::BM, T::BN, T::kABits, T::kWBits, 0);
    t.tile_m = at.m;
    t.tile_n = at.n;
    T::template run<GU>(t, smem);
  });
}

template <class... Tiles>
__global__ void __launch_bounds__(kThreads, kWavesPerSimd<Tiles...>) fused_group_gemm_kernel(const FusedArgs args) {
  extern __shared__ __align__(16) uint8_t smem[];
  fused_body<false, const FusedArgs*, Tiles...>(&args, smem);
}

// The same kernel with its tables in device memory, where a planning kernel wrote them from the tokens-per-expert counts: the
// host then needs no copy of the counts, so a layer forward neither synchronises nor depends on its routing when it is enqueued
// (or captured into a graph).  The grid is sized for the worst case; workgroups past the planned tiles leave at once.
// GU: the tiles' gate_up form (TileArgs::rows).
template <bool GU, class... Tiles>
__global__ void __launch_bounds__(kThreads, kWavesPerSimd<Tiles...>) fused_group_gemm_planned_kernel(const FusedArgs* __restrict__ args) {
  extern __shared__ __align__(16) uint8_t smem[];
  fused_body<GU, const MXMOE_CONST FusedArgs*, Tiles...>((const MXMOE_CONST FusedArgs*)args, smem);
}

// ------------------------------------------------------------------ host side ------------------------------------------------------------------

enum class Fmt { FP16, W8A8, W4A4, W4A16, W3A16, W2A16, W4A4G128, W8A16, UNSUPPORTED };

// Format of a problem from its QParams.  Weight-only formats come with one (scale, zero) pair per channel and 128-wide K group or
// per channel (group size -1): the tiles are the same, the packer repeats a per-channel pair for every group.
__host__ __device__ inline Fmt classify(const mxmoe_qparams& q) {
  if (q.a_bits >= 16 && q.w_bits >= 16) return Fmt::FP16;
  if (q.a_bits == 8 && q.w_bits == 8 && q.gsize == -1 && q.sym) return Fmt::W8A8;
  if (q.a_bits == 4 && q.w_bits == 4 && q.gsize == -1 && q.sym) return Fmt::W4A4;
  if (q.a_bits == 4 && q.w_bits == 4 && q.gsize == 128 && q.sym) return Fmt::W4A4G128;
  if (q.a_bits >= 16 && (q.gsize == 128 || q.gsize == -1)) {
    if (q.w_bits == 8) return Fmt::W8A16;
    if (q.w_bits == 4) return Fmt::W4A16;
    if (q.w_bits == 3) return Fmt::W3A16;
    if (q.w_bits == 2) return Fmt::W2A16;
  }
  return Fmt::UNSUPPORTED;
}
__host__ __device__ inline bool is_weight_only(Fmt f) { return f == Fmt::W8A16 || f == Fmt::W4A16 || f == Fmt::W3A16 || f == Fmt::W2A16; }

inline const char* fmt_name(Fmt f, bool sym) {
  switch (f) {
    case Fmt::FP16: return "fp16";
    case Fmt::W8A8: return "w8a8_g-1_sym";
    case Fmt::W4A4: return "w4a4_g-1_sym";
    case Fmt::W8A16: return sym ? "w8a16_g128_sym" : "w8a16_g128_asym";
    case Fmt::W4A16: return sym ? "w4a16_g128_sym" : "w4a16_g128_asym";
    case Fmt::W3A16: return sym ? "w3a16_g128_sym" : "w3a16_g128_asym";
    case Fmt::W2A16: return sym ? "w2a16_g128_sym" : "w2a16_g128_asym";
    case Fmt::W4A4G128: return "w4a4_g128_sym";
    default: return "unsupported";
  }
}

struct BranchInfo {
  Fmt fmt;
  int a_bits, w_bits;  // of an element of either operand as the tile reads it (kABits, kWBits: what the order of a problem's tiles goes by)
  int BM, BN, BK, WGM, WGN;
  int lds_bytes;
  int k_multiple;  // K must be a multiple of this
  int max_m;       // largest M this branch accepts (skinny weight-only tiles), or 0 = any
  int k_min = 0;   // smallest K this branch accepts, or 0 = one k_multiple
  // What QParams cannot say about the operands a branch takes: 0 as the format's table in the header says; 1 both operands of w4a4 as
  // bf6 fragments (the tiles on the 6-bit float matrix path); 2 both operands of w8a8 as fp8 e4m3 codes with fp32 accumulation
  // (w8a8_g-1_sym_E4M3, mxmoe/kernels/tile_config.py:45: QParams (8, 8, -1, sym) there as well).  A kernel with such a branch is
  // never chosen automatically: the caller names it, because only the caller knows what its operands hold.
  int variant = 0;
  int n_multiple = 8;  // N must be a multiple of this
};
constexpr int kVariantBf6 = 1, kVariantFp8 = 2, kVariantBf16 = 3;

template <class T>
struct BranchOf;
template <Op OP, int BM, int BN, int WGM, int WGN>
struct BranchOf<MfmaTile<OP, BM, BN, WGM, WGN>> {
  static BranchInfo get() {
    using T = MfmaTile<OP, BM, BN, WGM, WGN>;
    const Fmt f = OP == Op::I8 ? Fmt::W8A8 : (OP == Op::I4 ? Fmt::W4A4 : Fmt::FP16);
    // bfloat16 problems carry the QParams of fp16 ones (16 / 16 bits): which of the two a kernel computes is the kernel's variant
    return BranchInfo{f, T::kABits, T::kWBits, BM, BN, T::BK, WGM, WGN, T::kLdsBytes, T::BK, 0, 0, OP == Op::BF16 ? kVariantBf16 : 0};
  }
};
template <int BM>
struct BranchOf<WxAxGTile<BM>> {
  static BranchInfo get() {
    using T = WxAxGTile<BM>;
    return BranchInfo{Fmt::W4A4G128, T::kABits, T::kWBits, BM, T::BN, T::BK, 1, 4, T::kLdsBytes, T::BK, 0};
  }
};
template <>
struct BranchOf<WxAxGNarrowTile> {
  static BranchInfo get() {
    using T = WxAxGNarrowTile;
    return BranchInfo{Fmt::W4A4G128, T::kABits, T::kWBits, T::BM, T::BN, T::BK, 1, 1, T::kLdsBytes, T::BK, 0};
  }
};
template <Op OP, int BM, int BN>
struct BranchOf<WxAxTile<OP, BM, BN>> {
  static BranchInfo get() {
    using T = WxAxTile<OP, BM, BN>;
    return BranchInfo{OP == Op::I4 ? Fmt::W4A4 : Fmt::W8A8, T::kABits, T::kWBits, BM, BN, T::BK, 1, 4, T::kLdsBytes, T::BK, 0, 0, OP == Op::F8 ? kVariantFp8 : 0};
  }
};
template <Op OP>
struct BranchOf<WxAxNarrowTile<OP>> {
  static BranchInfo get() {
    using T = WxAxNarrowTile<OP>;
    return BranchInfo{OP == Op::I4 ? Fmt::W4A4 : Fmt::W8A8, T::kABits, T::kWBits, T::BM, T::BN, T::BK, 1, 1, T::kLdsBytes, T::BK, 0, 0, OP == Op::F8 ? kVariantFp8 : 0};
  }
};
template <int BM>
struct BranchOf<Bf6Tile<BM>> {
  // same format as the int4 tiles on the int8 instruction; what differs is the layout both operands are handed over in (6-bit
  // fragments), so the two kinds never share a kernel: the kernel a caller picks says which layout its operands have
  static BranchInfo get() {
    using T = Bf6Tile<BM>;
    return BranchInfo{Fmt::W4A4, T::kABits, T::kWBits, BM, T::BN, T::BK, 1, 4, T::kLdsBytes, 128, 0, 256, kVariantBf6};
  }
};
template <int WBITS, int BN, int MB, int WAVES>
struct BranchOf<SkinnyWoTile<WBITS, BN, MB, WAVES>> {
  static BranchInfo get() {
    using T = SkinnyWoTile<WBITS, BN, MB, WAVES>;
    return BranchInfo{WBITS == 16 ? Fmt::FP16 : WBITS == 8 ? Fmt::W8A16 : WBITS == 4 ? Fmt::W4A16 : WBITS == 3 ? Fmt::W3A16 : Fmt::W2A16, T::kABits, T::kWBits, T::BM, BN, 128, 1, 4, T::kLdsBytes, 128, 0, 0, 0, 16};
  }
};

using LaunchFn = hipError_t (*)(const FusedArgs&, int grid, int lds, hipStream_t);
using LaunchPlannedFn = hipError_t (*)(const FusedArgs* d_args, int grid, int lds, hipStream_t);

// How a registered kernel walks a problem list (the reference generates one host launcher per policy, kernel_sketch.py:82-145
// fused, :148-274 sequential, :277-406 multi-stream):
//   Fused       one launch over all problems;
//   Sequential  one launch per run of consecutive problems of equal format, all on the caller's stream;
//   MultiStream the same launches dealt round-robin to side streams that fork from and join the caller's stream.
enum class Policy { Fused = 0, Sequential = 1, MultiStream = 2 };

struct FusedKernel {
  std::string name;  // "[qcfg: (BM,BN,BK) (WGM,WGN,1) 2], ...<fn name>" — same shape as registry.cuh:42-70
  std::vector<BranchInfo> branches;
  int lds_bytes;
  LaunchFn launch;
  Policy policy;
  mxmoe_func_t func;  // the kernel as a function of the reference's FuncType (registry.cuh:28-39)
  LaunchPlannedFn launch_planned;  // the same kernel reading its tables from device memory (device-side planning)
  LaunchPlannedFn launch_gate_up;  // ... with its tiles in their gate_up form; null for kernels that are not a layer's
  int plan_index;                  // index into plan_infos()
  // Largest row count per problem this kernel is meant for, 0 = any.  A kernel with a limit is preferred by the automatic choice when
  // every problem of the list stays within it (the few-token kernels: same results, more workgroups per CU).
  int max_rows_hint;
};

inline std::vector<FusedKernel>& registry() {
  static std::vector<FusedKernel> r;
  return r;
}

inline std::string& last_error() {
  static thread_local std::string e;
  return e;
}

template <int WBITS, int BM, int BN>
struct BranchOf<WoMfmaTile<WBITS, BM, BN>> {
  static BranchInfo get() {
    using T = WoMfmaTile<WBITS, BM, BN>;
    return BranchInfo{WBITS == 8 ? Fmt::W8A16 : WBITS == 4 ? Fmt::W4A16 : WBITS == 3 ? Fmt::W3A16 : Fmt::W2A16, T::kABits, T::kWBits, BM, BN, 128, T::WM, 4 / T::WM, T::kLdsBytes, 128, 0, 0, 0, 16};
  }
};

// Run time of one tile of a branch relative to the 128 x 256 tile of the same format (same K), from the kernel-profile table
// measured on MI355X (ms per 256 tiles at K = 2048).  Small tiles pay a fixed prologue / epilogue and use the matrix pipe less
// well; the weight-only entries compare the skinny streaming tile with the 128 x 128 dequantise-to-fp16 tile (the 128 x 256
// one, four waves side by side with twice the tokens each, does twice the work in 1.5 times the time).
// The 32-token few-token tile costs the same for every bit width (it waits for memory, not for bytes), and two of them must not
// look cheaper than one 128 x 256 tile, which runs half its loop for a problem of 33 .. 64 rows.  (Its 4-, 3- and 2-bit entries are from before it walked K as
// one stream, which took a fifth off its time: what 33 .. 128 rows run on has not been weighed again since.)
inline double tile_cost(const BranchInfo& b) {
  struct Row { Fmt f; int bm, bn; double c; };
  static const Row table[] = {
      // (inside a fused kernel the small integer tiles run at the occupancy of the largest one, which costs them part of the
      // advantage they show as single-tile kernels in the profile table)
      {Fmt::W4A4, 128, 256, 1.00}, {Fmt::W4A4, 64, 256, 0.58}, {Fmt::W4A4, 32, 256, 0.48}, {Fmt::W4A4, 32, 64, 0.13},
      {Fmt::W8A8, 128, 256, 1.00}, {Fmt::W8A8, 64, 256, 0.74}, {Fmt::W8A8, 32, 256, 0.56}, {Fmt::W8A8, 32, 64, 0.155},
      {Fmt::FP16, 128, 256, 1.00}, {Fmt::FP16, 64, 256, 0.69}, {Fmt::FP16, 32, 256, 0.53}, {Fmt::FP16, 16, 64, 0.30}, {Fmt::FP16, 128, 128, 0.57}, {Fmt::FP16, 256, 128, 1.09},
      {Fmt::W4A16, 16, 128, 0.37}, {Fmt::W4A16, 16, 64, 0.20}, {Fmt::W4A16, 32, 128, 0.50}, {Fmt::W4A16, 128, 128, 1.00}, {Fmt::W4A16, 128, 256, 1.50},
      {Fmt::W3A16, 16, 128, 0.31}, {Fmt::W3A16, 16, 64, 0.20}, {Fmt::W3A16, 32, 128, 0.50}, {Fmt::W3A16, 128, 128, 1.00}, {Fmt::W3A16, 128, 256, 1.50},
      {Fmt::W2A16, 16, 128, 0.25}, {Fmt::W2A16, 16, 64, 0.20}, {Fmt::W2A16, 32, 128, 0.50}, {Fmt::W2A16, 128, 128, 1.00}, {Fmt::W2A16, 128, 256, 1.50},
      {Fmt::W8A16, 16, 128, 0.60}, {Fmt::W8A16, 16, 64, 0.35}, {Fmt::W8A16, 32, 128, 0.66}, {Fmt::W8A16, 128, 128, 1.00}, {Fmt::W8A16, 128, 256, 1.50},
      {Fmt::W4A4G128, 64, 256, 1.00}, {Fmt::W4A4G128, 32, 256, 0.60}, {Fmt::W4A4G128, 16, 64, 0.16},
  };
  for (const Row& r : table)
    if (r.f == b.fmt && r.bm == b.BM && r.bn == b.BN) return r.c;
  return (0.22 + 0.78 * b.BM / 128.0) * b.BN / 256.0;  // shapes without a measurement
}

// Rough run time of one tile across formats, used only to order the tile list (expensive shapes first): the matrix pipe runs
// fp16 at half the int8 rate, and int4 operands are widened to int8.
inline double branch_cost(const BranchInfo& b) {
  const double per_k = b.fmt == Fmt::FP16 ? 2.0 : is_weight_only(b.fmt) ? 1.2 : (b.fmt == Fmt::W8A8 ? 1.25 : 1.0);
  return tile_cost(b) * per_k;
}

// What the planners (the host launcher and the device-side planning kernel) need to know of a kernel's branches, as plain data.
constexpr int kMaxBranches = 32;
struct PlanBranch {
  int index;             // position among the kernel's branches
  int fmt, BM, BN;
  int bm_log2, bn_log2;  // tile dimensions are powers of two (register_fused): the planners shift instead of dividing
  double cost;           // tile_cost
  double cost_per_row;   // tile_cost / BM
};
// A phase of such tiles keeps the plain workgroup order (no XCD remap): the few-token weight-only tiles stream their own weights
// and share nothing but a few rows of activations with their neighbours.
__host__ __device__ inline bool flat_phase(const PlanBranch& b) { return b.BM <= 16 || (is_weight_only((Fmt)b.fmt) && b.BM < 128); }
// Whether the tiles of a shape's problems above the launch's smallest K (a shared expert's second block, two or four times as long as the routed experts') are a phase of their own,
// so that every XCD gets an eighth of them as well as of the others.  In one phase the XCDs get equal numbers of tiles, and the first of them all the long ones, which the launch then
// waited for while half of the chip was idle (a second block of 64 experts and a shared one of twice their width, 2049 tokens: CUs busy 0.52 of the time, 173 us).  Layers, us, one phase / two: 64 experts
// top-6 and a shared one, 2049 tokens, w4a16 385 / 332, w4a4 and w8a8 267 / 259; 60 experts top-4 and one four times as wide, w4a4 and w8a8 64 tokens 112 / 103, 2049 tokens 283 / 259, w4a16 / w3a16
// 442 / 339, 8192 tokens 1375 / 1051.  No lower limit: both layers in five mixes, even and skewed, 129 .. 400 tokens, two phases take 0.96 .. 1.01 of one's time (the planner with the code for it 0.2 to 0.5 us more, shared tiles of few rows
// are mostly flat phases), 512 tokens 0.94 .. 1.02, 777 0.89 .. 1.01.
__host__ __device__ inline bool long_phase(const PlanBranch& b, int long_tiles, int other_tiles) { return long_tiles > 0 && other_tiles > 0 && !flat_phase(b); }
// Tiles of size 2^lg that cover `x`.
__host__ __device__ inline int tiles_over(int x, int lg) { return (x + (1 << lg) - 1) >> lg; }
constexpr int kNumFmts = (int)Fmt::UNSUPPORTED;
struct PlanInfo {
  int nb;                       // branches
  // Narrow integer tiles among them; and, where a launch is planned with them, whether it has few blocks of channels (kPoleBlocks).
  int narrow, few_blocks;
  int may_pair;  // a format that has pairs (pairs_pay) comes in several shapes, and it is no kernel for few rows
  // A 128 x 256 tile that has a 128 x 128 one for launches of few tiles (kSlimTiles): branches, and whether there is such a pair of shapes.  The slim one stands behind
  // the formats' branches in b: problems are planned without it.
  int wide, slim, has_slim;
  int unequal_k;  // (the device planner's) the experts of the block differ in K
  uint8_t order[kMaxBranches];  // positions in b, most expensive tile first (branch_cost); ties keep the registration order
  uint8_t fmt_start[kNumFmts + 4];
  // by format, in registration order inside a format: those of format f are b[fmt_start[f]] .. b[fmt_start[f + 1] - 1], and the planners
  // look at no other branch
  PlanBranch b[kMaxBranches];
};
static_assert(sizeof(PlanInfo) % 8 == 0, "copied word by word");

struct Segment {
  int row0, rows, branch, tiles;
  int bm_log2, bn_log2;  // of two segments: their tiles
};

// Blocks of 256 channels, over all problems of a launch, up to which a 64-row integer tile sets the launch's time when it runs beside narrow ones: they stream
// their weights at the rate of the machine and are done in less than half of its time, during which it shares its CU with them.  There, problems of 33 .. 64 rows
// (and up to 128) take narrow tiles too (same sums: integers).  Eight problems of 45 .. 2 rows, K = 2048 / 14 336, us, 64-row tiles / narrow ones / a kernel of wide tiles
// alone: 128 blocks w4a4 16.6 / 13.5 / 13.4, 82 / 63 / 60, w8a8 26.5 / 21.8 / 19.9, 146 / 118 / 107; 64 blocks w4a4 13.9 / 10.0 / 13.0, 60 / 40 / 56.  Beyond, the
// narrow tiles lose what they gain: 256 blocks 22.1 / 19.9 / 17.8; 512 blocks (64 problems) 31.8 / 32.2 / 32.0, half of them of 40 rows 33.6 / 39.0 / 31.8.
constexpr int kPoleBlocks = 128;
__host__ __device__ inline bool integer_sums(int f) { return f == (int)Fmt::W4A4 || f == (int)Fmt::W8A8; }

// Tiles of a launch's long-K problems, all of them together, from which on it is as busy with them as with the rest (a quarter of the 512
// workgroups that run at a time).
constexpr int kLongTiles = 128;
// Whether a problem of a launch whose smallest K is `kmin` counts as long: above that, and a tile of it takes long at all (a 128 x 256
// weight-only tile 2.4 us per 128 of K: 40 us, a whole launch of few-row experts).
constexpr int kLongK = 2048;
__host__ __device__ inline bool runs_long(int K, int kmin) { return K > kmin && K >= kLongK; }

// The fields of a pair of segments (FusedArgs::Entry); 0 where their column tiles differ.
__host__ __device__ inline unsigned pair_word(const Segment (&s)[2]) {
  if (s[0].bn_log2 != s[1].bn_log2) return 0;
  const unsigned width = (unsigned)tiles_over(s[1].rows, s[1].bm_log2);
  return width <= 255 ? width << 21 : 0;
}
// Whether the two row segments of a problem are dealt out as a pair.  What a pair saves is the second trip of its weights from memory;
// what it costs is that cheap tiles no longer come last, where they fill the end of the launch.  `launch_tiles` counts the launch's tiles in the shapes that are cheapest
// per row, `launch_cols` what there is to fetch: blocks of 256 channels, each K / 4096 times (a megabyte with 8 bits).  512 tiles run at a time.  With
// fewer, large ones that come first get a CU each; around that number the second trip is worth it only of weights that the 256 MB last-level cache does not keep beside
// the rest; with many, always.  From 2219 lists (N = 2048 .. 28 672, K = 1408 .. 14 336, 1 .. 64 problems, even and uneven rows), time of pairs over that of phases, 8-bit and 16-bit
// operands, by tiles and weights:
//                    under 60 MB    60 .. 130    130 .. 250    250 .. 500    500 .. 1000    more    at worst
//   150 .. 300       1.01           1.02         1.03          1.02          1.01           0.99    1.42
//   301 .. 448       1.00           1.00         0.98          0.99          0.92           0.88    1.36
//   449 .. 512       0.99           1.01         0.96          0.91          0.88           0.88    1.11
//   513 .. 700       1.01           1.04         0.98          0.93          0.89           0.99    1.19
//   701 .. 1100      1.00           0.98         0.92          0.84          0.86           0.89    1.12
//   beyond           -              0.97         0.94          0.87          0.82           0.84    1.13
// us, phases / pairs: 16 problems of 180 rows, N = 4096, K = 14 336 (512 tiles) w8a8 311 / 253, fp16 721 / 544, fp8 309 / 230; one of 546 rows, N = 28 672, K = 4096 (560 tiles,
// 117 MB) w8a8 74 / 89; 64 of 192 rows, N = 2816, K = 2048 w8a8 155 / 114, fp16 310 / 232; 8 of 300 rows, N = 4096, K = 14 336 (384 tiles) w8a8 184 / 247.
// int4 operands take half the time to fetch and as long to multiply: 1.06 .. 1.14 up to 700 tiles and 250 MB, 1.01 .. 1.06 up to 1100, beyond that 0.98 from 250 MB on, 1.02 .. 1.05 below.
// Weight-only tiles are bound by their arithmetic: 135 rows 134 / 149, 267 rows 209 / 273.
constexpr int kPairTiles = 448, kPairTilesMany = 700, kPairTilesInt4 = 1000, kPairCols = 192, kPairColsInt4 = 768;
__host__ __device__ inline bool pairs_pay(int f, int launch_tiles, int launch_cols) {
  if (f == (int)Fmt::W4A4) return launch_tiles > kPairTilesInt4 && launch_cols > kPairColsInt4;
  if (f != (int)Fmt::W8A8 && f != (int)Fmt::FP16) return false;
  return launch_tiles > kPairTilesMany || (launch_tiles > kPairTiles && launch_cols > (f == (int)Fmt::FP16 ? kPairCols / 2 : kPairCols));
}

// Large tiles of a launch's problems of one length (the smallest K; any longer one) up to which the 128 x 128 tile of 8-bit weights runs in the place of the 128 x 256
// one: twice as many find a CU each, and one takes 0.8 of the time; with more, what counts is the work, of which the wide tile does twice as much in 1.5 times the
// time.  us, slim / wide, weights from memory, by wide tiles: N = 2048, K = 1408 96 rows 18.3 / 24.8 (8), 25.4 / 28.7 (128), 36.2 / 32.7 (256); N = 4096, K = 4096 96 rows
// 44.7 / 59.4 (16), 58.3 / 65.3 (128), 89.4 / 81.0 (256), 192 rows 57.3 / 63.7 (128), 384 rows 78.8 / 68.1 (192); K = 14 336 96 rows 185 / 206 (64), 214 / 225 (128), 292 / 272 (256);
// N = 2816, K = 2048 384 rows 29.8 / 34.8 (66), 37.4 / 36.2 (132).  A wide tile of up to 64 rows runs half its loop: there the slim one is ahead only in launches of
// few tiles of few steps in K (tiles times K up to kSlimWorkHalf): 33 rows, K = 1408 18.3 / 19.5 (8), 19.9 / 19.6 (32); K = 2048 24.7 / 25.6 (11), 25.2 / 26.1 (44), 30.3 / 29.6 (88);
// K = 4096 44.0 / 45.4 (16), 51.4 / 48.4 (32), 54.1 / 52.2 (64); K = 14 336 181 / 171 (16).  Few tiles of one length beside many of another: the longer ones start
// first and end last, the shorter ones fill the end, so that what counts is again the time of one (wide everywhere -> counted apart, N = 2048: 60 problems of 130 rows, K = 1408, and
// one of 2000, K = 5632 228 -> 146; 30 of 200 rows, K = 2048, and 8 of K = 4096 158 -> 118; 30 of K = 4096 and 8 of K = 2048 166 -> 148).
constexpr int kSlimTiles = 128, kSlimWorkHalf = 48 * 2048;
// The choice of tile shapes for an M x N problem, as far as it does not depend on the rest of the launch.
struct PlanPick {
  int branch = -1, bm = 0, tiles = 0, bm_log2 = 0, bn_log2 = 0;
  double cost = 0;
  __host__ __device__ void offer(const PlanBranch& b, int t, double c, double eps) {
    if (branch < 0 || c < cost - eps || (c < cost + eps && b.BM > bm)) {
      branch = b.index;
      bm = b.BM;
      bm_log2 = b.bm_log2;
      bn_log2 = b.bn_log2;
      tiles = t;
      cost = c;
    }
  }
};
struct PlanChoice {
  PlanPick unit, whole;  // cheapest per row of the problem; cheapest for all of it (cost of a block run with one shape = row tiles * column tiles * tile_cost)
  int full = 0;          // rows that fill whole tiles of `unit`
  double full_cost = 0;
  // Tiles in the largest shape, what a problem adds to its launch's large tiles and one of long K to its `long_tiles` (clamped where more makes no difference), or 0
  // when it takes a shorter shape anyway or there is no other.
  int large_tiles = 0;
};

constexpr int kLargeTilesTop = (kSlimTiles > kLongTiles ? kSlimTiles : kLongTiles) + 1;

// What a problem adds to its launch's `launch_tiles` (upper half) and `launch_cols` (lower half).  Clamped where more makes no difference: the sums over a wave's
// problems stay within 16 bits each.
static_assert(64 * (kPairTilesInt4 + 1) < 1 << 16 && 64 * (kPairColsInt4 + 1) < 1 << 16, "two sums in a word");
__host__ __device__ inline unsigned launch_load_of(const PlanChoice& c, int M, int N, int K) {
  const unsigned tm = tiles_over(M, c.unit.bm_log2), tn = tiles_over(N, c.unit.bn_log2), blocks = tiles_over(N, 8);
  const unsigned tiles = tm > kPairTilesInt4 || tn > kPairTilesInt4 || tm * tn > kPairTilesInt4 ? kPairTilesInt4 + 1 : tm * tn;
  const unsigned cols = blocks > kPairColsInt4 || K > (kPairColsInt4 << 12) || blocks * (unsigned)K > (kPairColsInt4 << 12) ? kPairColsInt4 + 1 : blocks * (unsigned)K >> 12;
  return tiles << 16 | cols;
}

// Returns 1, or 0 for M == 0, or -1 when the kernel has no tile for `f`.  Rolled loops here and below on purpose: the device planner runs
// this once per launch, when none of its code is in the instruction cache, and what it costs there is the fetching of its instructions.
__host__ __device__ inline int plan_choose(const PlanInfo& k, int f, int M, int N, PlanChoice& c) {
  if (f < 0 || f >= kNumFmts) return -1;
  const int lo = k.fmt_start[f], hi = k.fmt_start[f + 1];
  if (lo == hi) return -1;
  if (M <= 0) return 0;
#pragma unroll 1
  for (int i = lo; i < hi; ++i) {
    const PlanBranch& b = k.b[i];
    const int tm = tiles_over(M, b.bm_log2), tn = tiles_over(N, b.bn_log2), rows = M >> b.bm_log2 << b.bm_log2;
    c.whole.offer(b, tm * tn, (double)tm * tn * b.cost, 1e-9);
    const int had = c.unit.branch;
    c.unit.offer(b, (M >> b.bm_log2) * tn, b.cost_per_row * tn, 1e-12);
    if (c.unit.branch != had) {
      c.full = rows;
      c.full_cost = (double)(M >> b.bm_log2) * tn * b.cost;
    }
  }
  if (hi - lo > 1 && (c.full > 0 || c.whole.branch == c.unit.branch)) c.large_tiles = c.whole.tiles < kLargeTilesTop ? c.whole.tiles : kLargeTilesTop;
  return 1;
}

// Split the M rows of an M x N problem (M > 0, `c` from plan_choose) into at most two segments: whole tiles of the shape that is cheapest
// per output element, then the remainder with the shape that covers it most cheaply.  Returns the number of segments.
//
// `long_tiles`: 0, or for a problem of long K (runs_long: a shared expert behind several intermediates' width, say) the sum of large_tiles
// over all such problems of its launch.  Their tiles run that many times longer than the others', and a launch is not over before they
// are: as long as there are too few of them to share the chip with the rest, what counts is the time of one.  Where the choice by
// total cost takes the largest shape, such a problem takes the one of the smallest max(tile_cost, t / kLongTiles) instead, t being the
// cost of its own tiles and two thirds of what the launch's other long problems add to them (taken in proportion to their large tiles).  It is
// the launch's sum that is asked, since short tiles are 2 to 2.5 times the work.  c problems of K = 4096, N = 2048 beside one of K = 2048, us, large
// shape / shapes by each problem alone / this rule: w4a16 64 rows 52 / 37 / 33 (c = 6), 55 / 58 / 44 (15), 107 / 202 / 107 (60); 200 rows 69 / 48 / 48
// (4), 73 / 102 / 74 (12); 600 rows 557 / 998 / 557 (60); w4a4 128 rows 31 / 28 / 23 (8), 70 / 95 / 70 (60); fp16 128 rows 57 / 75 / 52 (8), 246 / 441 / 246 (60).
// Weight-only formats take the 32-token tile up to some 600 rows that way.  The 16-, 8- and 4-bit operand formats do it up to one large row
// tile only: their shorter tiles need half as long, not a third, for a quarter of the rows (201 .. 800 rows measured slower).  Down launch with 60 experts and a shared expert of four times their width, us,
// large shape -> this rule: w4a16 / w3a16 103 -> 36 (100 tokens), 103 -> 40 (201), 106 -> 58 (400); w4a4 45 -> 31, w4a4 / w8a8 49 -> 40, fp16
// 151 -> 128 (100); 64 experts and twice the width: w4a16 / w3a16 61 -> 37 (128), 60 -> 41 (201), 80 -> 67 (600), w8a16 / w2a16 60 -> 44 (128).
__host__ __device__ inline int plan_split(const PlanInfo& k, int f, int M, int N, const PlanChoice& c, int long_tiles, Segment out[2]) {
  const int lo = k.fmt_start[f], hi = k.fmt_start[f + 1];
  if (long_tiles > 0 && long_tiles < kLongTiles && c.large_tiles > 0 && (M <= 128 || is_weight_only((Fmt)f))) {
    PlanPick quick;  // soonest done on a part of the chip (both terms times 3 * kLongTiles * own tiles)
    const double own = (double)(3 * kLongTiles) * c.whole.tiles, shared = c.whole.tiles + 2.0 * long_tiles;
#pragma unroll 1
    for (int i = lo; i < hi; ++i) {
      const PlanBranch& b = k.b[i];
      const int tiles = tiles_over(M, b.bm_log2) * tiles_over(N, b.bn_log2);
      const double one = own * b.cost, all = (double)tiles * b.cost * shared;
      quick.offer(b, tiles, all > one ? all : one, 1e-9);
    }
    if (quick.branch != c.unit.branch) {
      out[0] = Segment{0, M, quick.branch, quick.tiles, 0, 0};
      return 1;
    }
  }
  const int rem = M - c.full;
  out[0] = Segment{0, M, c.whole.branch, c.whole.tiles, 0, 0};
  if (rem == 0 || c.full == 0) return 1;
  PlanPick rest;
  int all_unit = 0;  // tiles of the whole problem in the shape that is cheapest per row
#pragma unroll 1
  for (int i = lo; i < hi; ++i) {
    const PlanBranch& b = k.b[i];
    const int tm = tiles_over(rem, b.bm_log2), tn = tiles_over(N, b.bn_log2);
    rest.offer(b, tm * tn, (double)tm * tn * b.cost, 1e-9);
    if (b.index == c.unit.branch) all_unit = tiles_over(M, b.bm_log2) * tn;
  }
  if (rest.branch == c.unit.branch) {
    out[0] = Segment{0, M, c.unit.branch, all_unit, 0, 0};
    return 1;
  }
  if (c.whole.cost <= c.full_cost + rest.cost + 1e-9) return 1;
  out[0] = Segment{0, c.full, c.unit.branch, c.unit.tiles, c.unit.bm_log2, c.unit.bn_log2};
  out[1] = Segment{c.full, rem, rest.branch, rest.tiles, rest.bm_log2, rest.bn_log2};
  return 2;
}

// The segments of an M x N x K problem in a launch with `launch_tiles` large tiles for problems of its length: where those are few, wide ones become slim ones (kSlimTiles).
__host__ __device__ inline void take_slim_tiles(const PlanInfo& k, int launch_tiles, int M, int N, int K, Segment sg[2], int ns) {
  if (!k.has_slim || launch_tiles > kSlimTiles || (M <= 64 && (long)launch_tiles * K > kSlimWorkHalf)) return;
#pragma unroll
  for (int j = 0; j < 2; ++j)  // (unrolled: indexed by a loop, the segments would not stay in the planner's registers)
    if (j < ns && sg[j].branch == k.wide) {
      sg[j].branch = k.slim;
      sg[j].tiles = tiles_over(sg[j].rows, 7) * tiles_over(N, 7);
    }
}

// Both steps for a problem by itself: the number of segments (0 for M == 0), or -1 when the kernel has no tile for `f`.
inline int plan_segments(const PlanInfo& k, int f, int M, int N, Segment out[2]) {
  PlanChoice c;
  const int rc = plan_choose(k, f, M, N, c);
  return rc <= 0 ? rc : plan_split(k, f, M, N, c, 0, out);
}

inline PlanInfo make_plan_info(const std::vector<BranchInfo>& branches) {
  PlanInfo k;
  std::memset(&k, 0, sizeof k);
  k.nb = std::min((int)branches.size(), kMaxBranches);
  for (int i = 0; i < k.nb; ++i) k.narrow |= integer_sums((int)branches[i].fmt) && branches[i].BN == 64;
  for (int i = 0; i < k.nb && !k.narrow; ++i)  // (kMayPair)
    for (int j = 0; j < i; ++j) k.may_pair |= branches[i].fmt == branches[j].fmt && !is_weight_only(branches[i].fmt) && branches[i].fmt != Fmt::W4A4G128;
  auto log2_of = [](int v) {
    int lg = 0;
    while ((1 << lg) < v) ++lg;
    return lg;
  };
  for (int i = 0; i < k.nb; ++i)
    for (int j = 0; j < k.nb; ++j)
      if (branches[i].fmt == Fmt::W8A16 && branches[j].fmt == Fmt::W8A16 && branches[i].BM == 128 && branches[j].BM == 128 && branches[i].BN == 256 && branches[j].BN == 128) {
        k.wide = i;
        k.slim = j;
        k.has_slim = 1;
      }
  int at = 0;
  auto add = [&](int i) {
    const double cost = tile_cost(branches[i]);
    k.b[at++] = PlanBranch{i, (int)branches[i].fmt, branches[i].BM, branches[i].BN, log2_of(branches[i].BM), log2_of(branches[i].BN), cost, cost / branches[i].BM};
  };
  for (int f = 0; f < kNumFmts; ++f) {
    k.fmt_start[f] = (uint8_t)at;
    for (int i = 0; i < k.nb; ++i)
      if ((int)branches[i].fmt == f && !(k.has_slim && i == k.slim)) add(i);
  }
  k.fmt_start[kNumFmts] = (uint8_t)at;
  if (k.has_slim) add(k.slim);
  std::vector<int> order(k.nb);
  for (int i = 0; i < k.nb; ++i) order[i] = i;
  std::stable_sort(order.begin(), order.end(), [&](int x, int y) { return branch_cost(branches[x]) > branch_cost(branches[y]); });
  for (int r = 0; r < k.nb; ++r)
    for (int i = 0; i < k.nb; ++i)
      if (k.b[i].index == order[r]) k.order[r] = (uint8_t)i;
  return k;
}

inline std::vector<PlanInfo>& plan_infos() {
  static std::vector<PlanInfo> v;
  return v;
}
inline const PlanInfo& plan_of(const FusedKernel& k) { return plan_infos()[k.plan_index]; }

template <class... Tiles>
hipError_t launch_fused(const FusedArgs& a, int grid, int lds, hipStream_t s) {
  // more than 64 KB of dynamic LDS must be opted into, once per device (kept out of library load time: no HIP call before first use)
  static bool lds_opted_in[64] = {};
  if (lds > 64 * 1024) {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return hipGetLastError();
    if (dev >= 0 && dev < 64 && !lds_opted_in[dev]) {
      const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&fused_group_gemm_kernel<Tiles...>), hipFuncAttributeMaxDynamicSharedMemorySize, lds);
      if (e != hipSuccess) return e;
      lds_opted_in[dev] = true;
    }
  }
  hipLaunchKernelGGL((fused_group_gemm_kernel<Tiles...>), dim3(grid), dim3(kThreads), lds, s, a);
  return hipGetLastError();
}

template <bool GU, class... Tiles>
hipError_t launch_fused_planned(const FusedArgs* d_args, int grid, int lds, hipStream_t s) {
  static bool lds_opted_in[64] = {};
  if (lds > 64 * 1024) {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return hipGetLastError();
    if (dev >= 0 && dev < 64 && !lds_opted_in[dev]) {
      const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&fused_group_gemm_planned_kernel<GU, Tiles...>), hipFuncAttributeMaxDynamicSharedMemorySize, lds);
      if (e != hipSuccess) return e;
      lds_opted_in[dev] = true;
    }
  }
  hipLaunchKernelGGL((fused_group_gemm_planned_kernel<GU, Tiles...>), dim3(grid), dim3(kThreads), lds, s, d_args);
  return hipGetLastError();
}

inline int group_gemm(int kernel_id, const void* const* As, const void* const* Bs, const void* const* sa, const void* const* sb, void* const* Cs,
                      int32_t* const* acc, const mxmoe_dim3* d_sizes, const mxmoe_dim3* h_sizes, const mxmoe_qparams* h_q, int count, hipStream_t stream);

// Stream the FuncType functions launch on (that type has no stream argument; the reference launches on stream 0,
// kernel_sketch.py:123), and the status of the calling thread's last FuncType call (that type returns void).
inline hipStream_t& func_stream() {
  static thread_local hipStream_t s = nullptr;
  return s;
}
inline int& func_status() {
  static thread_local int rc = 0;
  return rc;
}

inline int checked_group_gemm(int kernel_id, const void* const* As, const void* const* Bs, const void* const* sa, const void* const* sb, void* const* Cs,
                              void* const* Ds, int32_t* const* acc, const mxmoe_dim3* d_sizes, const mxmoe_dim3* h_sizes, const mxmoe_qparams* h_q, int count,
                              hipStream_t stream) {
  if (count < 0 || (count > 0 && (!As || !Bs || !Cs || !d_sizes || !h_sizes || !h_q))) {
    last_error() = "null argument";
    return 5;
  }
  // Ds is accepted and never read, as in the reference's kernels (hz_fused.cuh:89,110 store through ptr_Cs only; its own caller
  // passes a second array with the same entries, test.cu:446-459): results go to Cs.
  (void)Ds;
  return group_gemm(kernel_id, As, Bs, sa, sb, Cs, acc, d_sizes, h_sizes, h_q, count, stream);
}

// One C function of the reference's FuncType per registered kernel: the template instance is the function, its static member the
// registry index it launches.  A failure is reported like the reference's launcher reports CUDA errors (message on stderr,
// helper.h:186-193) but the process is left alive; mxmoe_last_status() returns the code.
template <int POLICY, class... Tiles>
struct FuncThunk {
  static inline int kernel_id = -1;
  static void call(mxmoe_half** As, mxmoe_half** Bs, mxmoe_half** sa, mxmoe_half** sb, mxmoe_half** Cs, mxmoe_half** Ds, int64_t*, int64_t*, int64_t*, int64_t*,
                   mxmoe_dim3* d_sizes, mxmoe_dim3* h_sizes, mxmoe_qparams*, mxmoe_qparams* h_q, int problem_count) {
    const int rc = checked_group_gemm(kernel_id, (const void* const*)As, (const void* const*)Bs, (const void* const*)sa, (const void* const*)sb, (void* const*)Cs,
                                      (void* const*)Ds, nullptr, d_sizes, h_sizes, h_q, problem_count, func_stream());
    func_status() = rc;
    if (rc != 0) fprintf(stderr, "mxmoe: %s\n", last_error().c_str());
  }
};

template <class... Tiles>
int register_fused(const char* fn_name, Policy policy = Policy::Fused, int max_rows_hint = 0, LaunchPlannedFn launch_gate_up = nullptr) {
  static_assert(sizeof...(Tiles) <= kMaxBranches, "the planners' branch table holds kMaxBranches tile shapes per kernel");
  static_assert((((Tiles::BM & (Tiles::BM - 1)) == 0 && (Tiles::BN & (Tiles::BN - 1)) == 0) && ...), "the planners shift: tile dimensions are powers of two");
  FusedKernel k;
  k.policy = policy;
  k.max_rows_hint = max_rows_hint;
  k.branches = {BranchOf<Tiles>::get()...};
  k.lds_bytes = 0;
  std::string n;
  for (const auto& b : k.branches) {
    char buf[160];
    snprintf(buf, sizeof buf, "[%s%s: (%d,%d,%d) (%d,%d,1) 2], ", b.variant == kVariantBf16 ? "bf16" : fmt_name(b.fmt, b.fmt == Fmt::W8A8 || b.fmt == Fmt::W4A4),
             b.variant == kVariantFp8 ? "_E4M3" : "", b.BM, b.BN,
             b.BK, b.WGM, b.WGN);
    n += buf;
    k.lds_bytes = std::max(k.lds_bytes, b.lds_bytes);
  }
  k.name = n + fn_name;
  k.launch = &launch_fused<Tiles...>;
  k.launch_planned = &launch_fused_planned<false, Tiles...>;
  k.launch_gate_up = launch_gate_up;
  k.plan_index = (int)plan_infos().size();
  plan_infos().push_back(make_plan_info(k.branches));
  const int id = (int)registry().size();
  switch (policy) {
    case Policy::Fused: FuncThunk<0, Tiles...>::kernel_id = id; k.func = &FuncThunk<0, Tiles...>::call; break;
    case Policy::Sequential: FuncThunk<1, Tiles...>::kernel_id = id; k.func = &FuncThunk<1, Tiles...>::call; break;
    default: FuncThunk<2, Tiles...>::kernel_id = id; k.func = &FuncThunk<2, Tiles...>::call; break;
  }
  registry().push_back(k);
  return id;
}

// A kernel that a layer's first block may run on: its tiles in both forms.
template <class... Tiles>
int register_layer_kernel(const char* fn_name, Policy policy, int max_rows_hint = 0) {
  return register_fused<Tiles...>(fn_name, policy, max_rows_hint, &launch_fused_planned<true, Tiles...>);
}

// Operand variant (BranchInfo::variant) of the kernel's tiles for format `f`, 0 when it has none or the plain ones.
inline int kernel_variant(const FusedKernel& k, Fmt f) {
  for (const BranchInfo& b : k.branches)
    if (b.fmt == f && b.variant) return b.variant;
  return 0;
}
inline bool kernel_takes_bf6(const FusedKernel& k) { return kernel_variant(k, Fmt::W4A4) == kVariantBf6; }
inline bool kernel_has_variants(const FusedKernel& k) {
  for (const BranchInfo& b : k.branches)
    if (b.variant) return true;
  return false;
}

// A kernel can run a problem list when it has a branch for every format in it.  The automatic choice (kernel_id = -1) never
// falls on a kernel with operand variants (bf6 fragments, fp8 codes): QParams do not say what the operands hold, so those kernels
// are asked for by id.
inline bool kernel_covers(const FusedKernel& k, const mxmoe_qparams* q, int count) {
  for (int i = 0; i < count; ++i) {
    const Fmt f = classify(q[i]);
    Segment sg[2];
    if (f == Fmt::UNSUPPORTED || plan_segments(plan_of(k), (int)f, 1, 256, sg) < 0) return false;
  }
  return true;
}

// The problems of a launch that have rows, as far as the choice of a kernel for few rows looks at them.  The launcher fills it from its list; the planned
// forward, which does not know its routing on the host, with what an even routing would give (mxmoe_plan_select_kernel_rows).
struct RowSummary {
  int live = 0, tall = 0;         // problems; those of more than 16 rows
  long rows = 0, max_rows = 0;
  long blocks = 0;                // of 256 channels
  uint32_t max_k = 0;
  bool headless = false;          // a planned layer of few tokens: no head in front of gate_up on these kernels (layer_first_kernel)
  bool w4a4 = false, w8a8 = false, other = false, any_fp16 = false;  // formats among them
  bool fp16 = true;                                // no other format than this one
  void add_format(Fmt f) {
    (f == Fmt::W4A4 ? w4a4 : f == Fmt::W8A8 ? w8a8 : other) = true;
    fp16 = fp16 && f == Fmt::FP16;
    any_fp16 = any_fp16 || f == Fmt::FP16;
  }
  void add(Fmt f, long m, uint32_t N, uint32_t K) {
    if (m == 0) return;
    add_format(f);
    ++live;
    tall += m > 16;
    rows += m;
    max_rows = std::max(max_rows, m);
    blocks += (N + 255) / 256;
    max_k = std::max(max_k, K);
  }
};
inline RowSummary row_summary(const mxmoe_dim3* h_sizes, const mxmoe_qparams* h_q, int count) {
  RowSummary s;
  for (int i = 0; i < count; ++i) s.add(classify(h_q[i]), h_sizes[i].x, h_sizes[i].y, h_sizes[i].z);
  return s;
}

// Lists of few rows with w4a4 or w8a8 problems go to the kernels that hold the narrow integer tile (WxAxNarrowTile, for problems of up to 32 rows; more take
// 64-row tiles): no problem above 64 rows, at most 768 blocks of 256 channels over all problems, and few rows per problem on average.  A narrow tile reads the rows
// of its problem as often as there are 64-channel columns, so it loses with rows what it gains where the wide tiles leave the chip idle: by blocks, in rounds of 256 or 512
// workgroups.  One launch over weights from memory, time against the wide kernel's (w4a4 / w8a8 / half and half, then a third weight-only):
//   64 .. 128 blocks:              2 .. 24 rows 0.43 .. 0.96;  one problem of 48 rows 0.58 .. 0.97
//   132 .. 256 blocks:             8 rows 0.83 .. 1.05, 12 0.84 .. 1.08, 24 0.89 .. 1.20;  one problem of 36 rows 1.04 .. 1.45 (its 64-row tile is what the launch waits for)
//   K = 1408, 320 blocks:          8 rows 0.95 / 0.86 / 0.93, 12 0.95 / 0.90 / 0.95, 24 1.04 / 1.01 / 1.06;  with weight-only 192 and 256 blocks, 16 rows 0.90 and 0.95
//   K = 1408, 480 and 512 blocks:  4 rows 1.03, 1.06 / 0.97, 0.97 / 1.01, 1.01, 8 1.05, 1.09 / 1.03, 1.05 / 1.05, 1.06, 24 1.20 .. 1.26;  with weight-only 1.07 .. 1.11 at 1 .. 24
//   K = 2048, 660 blocks:          8 rows 0.97 / 0.96 / 0.93, 12 1.00 / 1.00 / 0.96, 16 1.03 / 1.03 / 0.98, 24 1.11 / 1.11 / 1.02;  with weight-only, 16 rows 0.98, 24 1.10
//   K = 4096, 448 blocks:          8 rows 0.97 / 0.94 / 0.99, 12 1.01 / 0.94 / 0.98, 16 1.05 / 0.96 / 1.00, 24 1.11 / 1.02 / 1.06;  with weight-only, 16 rows 0.99, 24 1.06
// Whole layers, planned, us, wide -> as chosen here: 60 experts top-4, w4a4 / w8a8 half and half 45 -> 35 (1 token), 65 -> 58 (8), 99 -> 89 (32), 106 -> 97 (64); with a shared
// expert of four times the width 58 -> 42 (1), 80 -> 70 (8), 122 -> 120 (64), under a skewed routing 93 -> 98 (32), 113 -> 114 (64); 64 experts top-6 and a shared one 50 -> 41 (1), 81 -> 74 (8),
// 117 -> 110 (32), 121 -> 117 (64), skewed 112 -> 119 (64: the planned forward does not know its routing); 8 experts of N = 28 672 / 4096, K = 4096 / 14 336, whose second
// block alone is within the limit of blocks, 126 -> 94 (1), 230 -> 199 (8), 240 -> 209 (64).  More than 768 blocks: lists of 770 .. 902 at 8 rows 0.91 .. 1.01, but the gate_up form of those 8
// experts' first block (896) 1.00 .. 1.05 in w4a4 layers of 1 .. 32 tokens, 1.12 skewed.
// A 128-row tile beside them would take the third workgroup of a CU (244 registers, 161 without): 60 experts 77 -> 83 (32).
// (Launches of fewer than 8 blocks would run at 0.35 .. 0.6 of the wide kernel's time as well; the planning rules for long problems are stated, and tested, on lists of two or three
// small problems in the wide shapes.)
// The kernels for fp8 beside w4a4 (groupgemm_hz_fused_wxax_e4m3_few) by the same rules, us a layer: 60 experts top-4 40 -> 30 (1 token), 64 -> 55 (8), 94 -> 84 (32), 100 -> 92 (64); with a
// shared expert, skewed, 53 -> 38 (1), 79 -> 67 (16), 105 -> 97 (64); 8 experts 103 -> 67 (1), 216 -> 184 (8), 232 -> 200 (64).  That with group-scaled w4a4 and weight-only problems
// (groupgemm_hz_fused_all_e4m3_few: tiles of 64 channels alone, 155 registers; with the many-token tiles beside them, 255 registers, 8 experts, 64 tokens, took 343 us, not 265), four formats: 60 experts
// 54 -> 32 (1), 78 -> 62 (8), 100 -> 101 (32); with a shared expert 75 -> 42 (1), 110 -> 92 (16), 140 -> 124 (64); 8 experts 228 -> 84 (1), 307 -> 213 (8), 326 -> 265 (64).
// Where such a layer starts with gate_up on these kernels (layer_first_kernel, 4 us less in front of it), up to 1024 blocks and 12 rows: 8 experts, first block of 896 blocks, us a layer, w4a4 119 -> 115 (4
// tokens), 148 -> 144 (32), w4a4 / w8a8 skewed 146 -> 137 (4), 173 -> 167 (16), 201 -> 199 (48), 211 -> 219 (64), with w4a16 208 -> 202 (16), 212 -> 210 (48), 216 -> 222 (64);
// 90 experts of N = 2816 top-6 (990 blocks) w4a4 96 -> 91 (44), 98 -> 95 (64), skewed 85 -> 76, 90 -> 83, w4a4 / w8a8 125 -> 117, 126 -> 119, skewed 105 -> 94, 114 -> 107.
// Where a layer starts with gate_up, up to 128 tokens: kDirectTokens.
constexpr int kFewRowsMax = 64, kFewBlocks = 768, kFewBlocksHeadless = 1024, kFewBlocksMin = 8;
// Tokens and (token, slot) pairs up to which a planned layer has no head in front of gate_up on the kernels for few rows (layer_first_kernel: one or two pairs per thread of a
// workgroup).  Above 64 tokens, us a layer, wide kernels behind a head -> without, evenly routed / skewed: 60 experts top-4 w4a4 80 -> 73 / 72 -> 64 (66 tokens), 80 -> 75 / 82 -> 73 (128), w4a4 / w8a8
// 99 -> 88 / 89 -> 79, 102 -> 93 / 101 -> 91, w4a4 / w8a8 / w4a16 102 -> 90 / 92 -> 81, 105 -> 95 / 103 -> 95, w4a16 / w3a16 75 -> 65 / 84 -> 65, 78 -> 70 / 97 -> 81, w8a16 / w2a16 96 -> 82 / 98 -> 79, 99 -> 88 /
// 105 -> 97, with a shared expert 97 -> 89, 114 -> 107, 129 -> 121, 95 -> 78, 112 -> 97 (66); 64 experts top-6 and a shared one 93 -> 88, 117 -> 111, 122 -> 115, 96 -> 81, 114 -> 98 (84); 32 experts top-4 w4a4 57 -> 52 / 66 -> 57 (96), w4a4 / w8a8 69 -> 65 / 76 -> 67 (127),
// w4a16 / w3a16 52 -> 45 / 80 -> 58 (72); 24 experts top-2, K = 4096, w4a4 74 -> 65 / 68 -> 64 (100).  fp16 (weights read
// once per 16 rows from L2 outweigh the head) 223 -> 210 / 186 -> 189 (66), 223 -> 214 / 224 -> 231 (128), with a shared expert 278 -> 298: up to 64.
// Errors of weight-only problems against float64 in the 2-norm, many-token tiles (whose weights are rounded to fp16) / 64-channel tiles, K = 2048: w8 2.88e-4 / 2.06e-4, w4 2.89e-4 / 2.06e-4, w3 2.82e-4 /
// 2.13e-4, w2 2.22e-4 / 2.09e-4 (the output's own rounding is 2.0e-4 of each).
constexpr int kDirectTokens = 128, kDirectEntries = 512;
// The largest problem that those kernels take in a launch.
inline long few_rows_max(const RowSummary& s) { return s.headless && !s.any_fp16 ? kDirectTokens : kFewRowsMax; }
inline bool holds_narrow(const FusedKernel& k) { return plan_of(k).narrow; }
// Rows per problem, on average, up to which those kernels are chosen.
inline int few_rows_limit(const RowSummary& s) {
  if (s.blocks <= kPoleBlocks) return 24;
  if (s.blocks > kFewBlocks) return 12;
  if (s.max_k < 2048 && s.blocks > 384) return s.other ? 2 : 5;
  if (s.other || (s.w4a4 && s.w8a8 && s.max_k >= 2048)) return 16;
  return s.max_k < 2048 ? 8 : 12;
}
inline bool few_rows(const RowSummary& s) {
  if (!(s.w4a4 || s.w8a8) || s.max_rows > few_rows_max(s) || s.blocks < kFewBlocksMin || s.blocks > (s.headless ? kFewBlocksHeadless : kFewBlocks)) return false;
  if (s.blocks > kPoleBlocks && s.blocks <= 256 && s.max_rows > 32) return false;
  return s.rows <= few_rows_limit(s) * s.live;
}
// A list of weight-only problems of few rows takes a kernel made of 16-row few-token tiles (FusedKernel::max_rows_hint), unless more than a quarter of its
// problems need several of them: then the kernels that also hold the 32-row few-token tile do better, whatever the largest count.
// Of those kernels, the one of 64-channel tiles against that of 128: twice the workgroups, 125 registers (four workgroups per CU) against 164.
// Up to 6 rows per problem on average; the activations, read once per tile, weigh more with more.  A whole layer, us, 128 -> 64 channels: 64 experts top-6 and
// a shared one, w4a16 / w3a16, 30.2 -> 28.2 (1 token), 42.7 -> 39.2 (4), 64 -> 61 (16), 75 -> 73 (64); 60 experts top-4 and a shared one 33.6 -> 29.0 (1),
// 58 -> 51 (16); 8 experts of N = 28 672 / 4096 61.6 -> 52.1 (1), 144 -> 140 (16), but 144 -> 150 (32: 8 rows each).  (Launches of fewer than 8 blocks
// would take 0.73 .. 0.81 of the time as well: 7 blocks of K = 2048, 1 row, 7.6 -> 5.9.)
// The same for lists with fp16 or 8-bit weight-only problems (a kernel of its own, 142 registers: three workgroups per CU), against the kernels of wider tiles, us a layer: 60 experts top-4
// fp16 67 -> 35 (1 token), 86 -> 73 (4), 131 -> 108 (8), 166 -> 158 (16), 207 -> 196 (32), 216 -> 217 (64), with a shared expert 143 -> 68 (1), 208 -> 141 (16), 288 -> 232 (64); 8 experts of N = 28 672 /
// 4096 fp16 327 -> 173 (1), 583 -> 447 (16), 622 -> 521 (32: 8 rows each), 639 -> 614 (48), 642 -> 705 (64): weights of 16 bits outweigh the activations for longer, up to 12 rows.  w8a16 / w2a16 half and
// half, 64 experts top-6 and a shared one 37 -> 31 (1), 71 -> 65 (8), 103 -> 96 (32), 8 experts 100 -> 80 (1), 204 -> 200 (8), 213 -> 215 (32).
// Where a layer starts with gate_up on these kernels (no head in front of it), up to 10 rows, or 8 where K is above 2048 and the head less of the layer's time, us a layer: 64 experts top-6 and a shared one, 58 tokens w4a16 / w3a16 80 -> 74, skewed 80 -> 71, w8a16 / w2a16
// 108 -> 92, 106 -> 89, 64 tokens 81 -> 75, 108 -> 93; 60 experts top-8, 64 tokens 76 -> 70, 100 -> 88; 8 experts of N = 28 672 / 4096 w4a16 161 -> 154 (28), 172 -> 166 (32), 175 -> 172 (40), 180 -> 180 (48),
// w8a16 / w2a16 219 -> 210 (28), 222 -> 219 (32), 226 -> 230 (40), 234 -> 243 (48).
constexpr int kFewTokenRows = 6, kFewTokenRowsHeadless = 10, kFewTokenRowsHeadlessLong = 8, kFewTokenRowsFp16 = 12;
inline int few_token_rows(const RowSummary& s) {
  if (s.fp16) return kFewTokenRowsFp16;
  if (!s.headless) return kFewTokenRows;
  return s.max_k > 2048 ? kFewTokenRowsHeadlessLong : kFewTokenRowsHeadless;
}
inline bool only_narrow_few_token(const FusedKernel& k) {
  for (const BranchInfo& b : k.branches)
    if (b.a_bits != 16 || b.BN != 64) return false;
  return true;
}

// The kernel made for the few rows of a launch, or -1 where there is none or the plain kernels do better.  `covers(k)`: whether kernel k has a tile for every
// problem's format (and operand layout).  The one place of this choice: the launcher and the planned forward both come here.
template <class Covers>
int few_row_kernel(const RowSummary& s, Covers&& covers) {
  auto& reg = registry();
  auto first = [&](auto&& wanted) {
    for (int i = 0; i < (int)reg.size(); ++i)
      if (reg[i].policy == Policy::Fused && wanted(reg[i]) && covers(reg[i])) return i;
    return -1;
  };
  if (few_rows(s)) {
    const int kid = first(holds_narrow);
    if (kid >= 0) return kid;
  }
  if (4 * s.tall > s.live) return -1;
  if (s.max_rows <= few_rows_max(s) && s.rows <= few_token_rows(s) * s.live && s.blocks >= kFewBlocksMin) {
    const int kid = first(only_narrow_few_token);
    if (kid >= 0) return kid;
  }
  return first([&](const FusedKernel& k) { return k.max_rows_hint > 0 && s.max_rows <= k.max_rows_hint; });
}

// K a multiple of the tile's K step, N a multiple of 8 (16 for the weight-only layouts and the few-token tiles)
inline bool shape_ok(const BranchInfo& bi, const mxmoe_dim3& sz) {
  return sz.z != 0 && sz.z % bi.k_multiple == 0 && (int)sz.z >= bi.k_min && sz.y % bi.n_multiple == 0;
}

// Whether kernel k's tiles take the shapes of a list's problems (an fp16 problem may have one that the few-token tiles do not take).
inline bool fits_shapes(const FusedKernel& k, const mxmoe_dim3* h_sizes, const mxmoe_qparams* h_q, int count) {
  for (int i = 0; i < count; ++i)
    for (const BranchInfo& b : k.branches)
      if (h_sizes[i].x != 0 && b.fmt == classify(h_q[i]) && !shape_ok(b, h_sizes[i])) return false;
  return true;
}

// Of the kernels with narrow tiles, the one for a layer: without many-token tiles where there is one.  A launch of more formats than w4a4 and w8a8 by itself is chosen with them (lists of up to 64 rows
// a problem); in a layer of few tokens a problem of more than a row tile is rare, and they cost every tile of the launch its third workgroup per CU.  w4a4 / w8a8 / w4a16, us a layer, with /
// without them: 64 experts top-6 and a shared one 38.7 / 37.8 (1 token), 93 / 90 (16), 108 / 106 (32); 60 experts top-4 and a shared one 89 / 83 (16), 109 / 102 (32), 121 / 113 (64).
template <class Covers>
int without_many_token_tiles(int kid, Covers&& covers) {
  auto many = [](const FusedKernel& k) {
    for (const BranchInfo& b : k.branches)
      if (b.BM == 128) return true;
    return false;
  };
  auto& reg = registry();
  if (kid < 0 || !holds_narrow(reg[kid]) || !many(reg[kid])) return kid;
  for (int i = 0; i < (int)reg.size(); ++i)
    if (reg[i].policy == Policy::Fused && holds_narrow(reg[i]) && !many(reg[i]) && covers(reg[i])) return i;
  return kid;
}

// The kernel for a layer's list of few rows whose operands are those of kernel `kernel_id` (its operand variants, which QParams do not name; plain ones where it is negative), or kernel_id.
inline int few_row_sibling(int kernel_id, const mxmoe_dim3* h_sizes, const mxmoe_qparams* h_q, int count) {
  auto covers = [&](const FusedKernel& k) {
    for (int i = 0; i < count; ++i) {
      const Fmt f = classify(h_q[i]);
      if (kernel_variant(k, f) != (kernel_id < 0 ? 0 : kernel_variant(registry()[kernel_id], f))) return false;
    }
    return (kernel_id >= 0 || !kernel_has_variants(k)) && kernel_covers(k, h_q, count) && fits_shapes(k, h_sizes, h_q, count);
  };
  const int kid = without_many_token_tiles(few_row_kernel(row_summary(h_sizes, h_q, count), covers), covers);
  return kid >= 0 ? kid : kernel_id;
}

// The kernel the launcher picks when the caller names none: one made for few rows, or the first fused kernel without operand variants that has a tile for every
// format.
inline int auto_kernel(const mxmoe_dim3* h_sizes, const mxmoe_qparams* h_q, int count) {
  auto covers = [&](const FusedKernel& k) { return !kernel_has_variants(k) && kernel_covers(k, h_q, count); };
  const int few = few_row_kernel(row_summary(h_sizes, h_q, count), [&](const FusedKernel& k) { return covers(k) && fits_shapes(k, h_sizes, h_q, count); });
  if (few >= 0) return few;
  auto& reg = registry();
  for (int i = 0; i < (int)reg.size(); ++i)
    if (reg[i].policy == Policy::Fused && reg[i].max_rows_hint == 0 && covers(reg[i])) return i;
  return -1;
}

// What the planning of one launch's problems has in common: its smallest K, its tiles (where it may have pairs), its large tiles and those of its long problems, whether it has
// few blocks; and what was chosen for each problem on the way, so that the tables do not choose again.  Problems without rows
// have no part in it: a list plans the same with and without them (the device planner sees every expert, the operators leave out empty ones).
struct LaunchScope {
  int kmin = 0x7fffffff, long_tiles = 0, launch_tiles = 0, launch_cols = 0;
  int tall_tiles[2] = {0, 0};  // of the problems of the smallest K, of the others
  bool few_blocks = false;
  int8_t have[kMaxProblems];          // plan_choose's answer for each problem (-1 too where its format is not supported)
  union {
    PlanChoice choice[kMaxProblems];  // where that is 1
  };
  LaunchScope() {}  // (leaves the arrays alone)
  // A problem of `M` rows, N and K of `sz`, whose shapes are `c`: plan_split in this launch.
  int split(const PlanInfo& pi, int f, int M, const mxmoe_dim3& sz, const PlanChoice& c, Segment out[2]) const {
    const int ns = plan_split(pi, f, M, (int)sz.y, c, runs_long((int)sz.z, kmin) ? long_tiles : few_blocks && integer_sums(f) ? c.large_tiles : 0, out);
    take_slim_tiles(pi, tall_tiles[(int)sz.z > kmin], M, (int)sz.y, (int)sz.z, out, ns);
    return ns;
  }
  // The number of segments of problem i (0 without rows), or -1 when the kernel has no tile for it.
  int segments(const PlanInfo& pi, int i, const mxmoe_dim3& sz, int f, Segment out[2]) const {
    return have[i] <= 0 ? have[i] : split(pi, f, (int)sz.x, sz, choice[i], out);
  }
};
inline void launch_scope(const PlanInfo& pi, const mxmoe_dim3* h_sizes, const mxmoe_qparams* h_q, int n, LaunchScope& s) {
  s.kmin = 0x7fffffff;
  s.long_tiles = s.launch_tiles = s.launch_cols = s.tall_tiles[0] = s.tall_tiles[1] = 0;
  long blocks = 0;
  for (int i = 0; i < n; ++i)
    if (h_sizes[i].x != 0) {
      s.kmin = std::min(s.kmin, (int)h_sizes[i].z);
      blocks += (h_sizes[i].y + 255) / 256;
    }
  s.few_blocks = pi.narrow && blocks <= kPoleBlocks;
  for (int i = 0; i < n; ++i) {
    const Fmt f = classify(h_q[i]);
    PlanChoice& c = s.choice[i];
    c = PlanChoice{};
    s.have[i] = f == Fmt::UNSUPPORTED ? -1 : (int8_t)plan_choose(pi, (int)f, (int)h_sizes[i].x, (int)h_sizes[i].y, c);
    if (s.have[i] <= 0) continue;
    if (pi.may_pair) {
      const unsigned load = launch_load_of(c, (int)h_sizes[i].x, (int)h_sizes[i].y, (int)h_sizes[i].z);
      s.launch_tiles += (int)(load >> 16);
      s.launch_cols += (int)(load & 0xFFFF);
    }
    s.tall_tiles[(int)h_sizes[i].z > s.kmin] += c.large_tiles;
    if (runs_long((int)h_sizes[i].z, s.kmin)) s.long_tiles = std::min(s.long_tiles + c.large_tiles, kLongTiles);
  }
}

// Tile tables of one launch over problems [base, base + n) (n <= kMaxProblems): entries, phases, totals of `a`; *grid receives the
// workgroups to launch.  Host-only arithmetic.
inline int build_fused_tables(const FusedKernel& k, const mxmoe_dim3* h_sizes, const mxmoe_qparams* h_q, int base, int n, FusedArgs& a, int* grid) {
  a.problem_offset = base;
  a.phase_flat = 0;
  const PlanInfo& pi = plan_of(k);
  struct Entry {
    int row0, rows, problem, branch, tiles;
    unsigned pair;
    int phase_branch;  // whose phase it runs in: its own, or that of the pair's first segment
  };
  Entry entries[kMaxEntries];
  int nent = 0;
  LaunchScope scope;
  launch_scope(pi, h_sizes + base, h_q + base, n, scope);
  for (int i = 0; i < n; ++i) {
    const mxmoe_dim3& sz = h_sizes[base + i];
    const Fmt f = classify(h_q[base + i]);
    Segment sg[2];
    const int ns = scope.segments(pi, i, sz, (int)f, sg);
    if (ns < 0) {
      last_error() = "quant type not supported";
      return 1;
    }
    for (int j = 0; j < ns; ++j) {
      const BranchInfo& bi = k.branches[sg[j].branch];
      if (!shape_ok(bi, sz)) {
        char buf[200];
        snprintf(buf, sizeof buf, "problem %d: shape [%u,%u,%u] not supported by tile %s (K %% %d, N %% 8)", base + i, sz.x, sz.y, sz.z, fmt_name(bi.fmt, true), bi.k_multiple);
        last_error() = buf;
        return 3;
      }
      const unsigned pair = ns == 2 && pi.may_pair && pairs_pay((int)f, scope.launch_tiles, scope.launch_cols) ? pair_word(sg) : 0;
      entries[nent++] = Entry{sg[j].row0, sg[j].rows, i, sg[j].branch, sg[j].tiles, pair | (pair && j ? kPairSecond : 0u), sg[pair ? 0 : j].branch};
    }
  }
  // Most expensive tile shape first.  Inside a shape, the problems whose K is above the launch's smallest K go first (their tiles
  // run longest: a shared expert with a wider intermediate, say; workgroups are dispatched in index order, and the longest
  // jobs first is what keeps the tail of the launch short), then the others, as a phase of their own (long_phase); problems keep their order otherwise (neighbouring tiles
  // share operands).
  int total = 0, ne = 0, wg = 0, np = 0;
  for (int oi = 0; oi < pi.nb; ++oi) {
    const PlanBranch& pb = pi.b[pi.order[oi]];
    const int b = pb.index;
    const int tile0 = total;
    int rest0 = total;  // first tile of the problems of the smallest K
    for (int pass = 0; pass < 2; ++pass) {
      if (pass == 1) rest0 = total;
      for (int ei = 0; ei < nent; ++ei) {
        const Entry& en = entries[ei];
        if (en.phase_branch != b || en.tiles == 0 || ((int)h_sizes[base + en.problem].z > scope.kmin) != (pass == 0)) continue;
        a.entry[ne] = FusedArgs::Entry{total, en.row0, en.rows, (int)((unsigned)(en.problem | (en.branch << 16)) | en.pair)};
        total += en.tiles;
        ++ne;
      }
    }
    if (total == tile0) continue;
    const bool split = long_phase(pb, rest0 - tile0, total - rest0);
    for (int part = 0; part < (split ? 2 : 1); ++part) {
      const int first = part ? rest0 : tile0, last = split && part == 0 ? rest0 : total;
      // phases beyond the table share its last one (their relative order is kept)
      if (np < kMaxPhases) {
        a.phase_tile0[np] = first;
        a.phase_wg0[np] = wg;
        if (flat_phase(pb)) a.phase_flat |= 1 << np;
        ++np;
      }
      const int p0 = a.phase_tile0[np - 1];
      wg = a.phase_wg0[np - 1] + (last - p0 + kNumXcd - 1) / kNumXcd * kNumXcd;
    }
  }
  a.num_entries = ne;
  a.total_tiles = total;
  a.num_phases = np;
  a.phase_tile0[np] = total;
  a.phase_wg0[np] = wg;
  *grid = wg;
  return 0;
}

// One launch over problems [base, base + n) of the caller's arrays with kernel `k` (n <= kMaxProblems).
inline int launch_range(const FusedKernel& k, const void* const* As, const void* const* Bs, const void* const* sa, const void* const* sb, void* const* Cs,
                        int32_t* const* acc, const mxmoe_dim3* d_sizes, const mxmoe_dim3* h_sizes, const mxmoe_qparams* h_q, int base, int n, hipStream_t stream) {
  FusedArgs a;
  std::memset(&a, 0, sizeof a);
  a.As = reinterpret_cast<const uint8_t* const*>(As);
  a.Bs = reinterpret_cast<const uint8_t* const*>(Bs);
  a.sa = reinterpret_cast<const _Float16* const*>(sa);
  a.sb = reinterpret_cast<const _Float16* const*>(sb);
  a.Cs = reinterpret_cast<_Float16* const*>(Cs);
  a.acc = acc;
  a.sizes = d_sizes;
  int grid = 0;
  if (const int rc = build_fused_tables(k, h_sizes, h_q, base, n, a, &grid)) return rc;
  if (a.total_tiles == 0) return 0;
  const hipError_t e = k.launch(a, grid, k.lds_bytes, stream);
  if (e != hipSuccess) {
    last_error() = std::string("kernel launch failed: ") + hipGetErrorString(e);
    return 4;
  }
  return 0;
}

// Problems of the launch that starts at `base`: up to kMaxProblems, under the other policies than Fused of one format (kernel_sketch.py:192-246
// compares the QParams of neighbours the same way).
inline int launch_length(const FusedKernel& k, const mxmoe_qparams* h_q, int base, int count) {
  const mxmoe_qparams& a = h_q[base];
  int n = 1;
  while (base + n < count && n < kMaxProblems) {
    const mxmoe_qparams& b = h_q[base + n];
    if (k.policy != Policy::Fused && !(a.a_bits == b.a_bits && a.w_bits == b.w_bits && a.gsize == b.gsize && a.sym == b.sym)) break;
    ++n;
  }
  return n;
}

// Side streams of the multi-stream policy, created on first use per device (default priority, non-blocking) and kept for the
// life of the process, with the events that fork them from and join them to the caller's stream.
constexpr int kSideStreams = 4;
struct SideStreams {
  hipStream_t stream[kSideStreams];
  hipEvent_t fork, join[kSideStreams];
  bool ready;
};
inline SideStreams* side_streams() {
  static SideStreams pool[64] = {};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return nullptr;
  SideStreams& p = pool[dev];
  if (!p.ready) {
    if (hipEventCreateWithFlags(&p.fork, hipEventDisableTiming) != hipSuccess) return nullptr;
    for (int i = 0; i < kSideStreams; ++i)
      if (hipStreamCreateWithFlags(&p.stream[i], hipStreamNonBlocking) != hipSuccess || hipEventCreateWithFlags(&p.join[i], hipEventDisableTiming) != hipSuccess) return nullptr;
    p.ready = true;
  }
  return &p;
}

// Host launcher.  Array arguments as in the reference FuncType (registry.cuh:28-39): every pointer array and
// d_sizes / d_q live in device memory, h_sizes / h_q are their host mirrors.  ld* and d_q are accepted and unused.
inline int group_gemm(int kernel_id, const void* const* As, const void* const* Bs, const void* const* sa, const void* const* sb, void* const* Cs,
                      int32_t* const* acc, const mxmoe_dim3* d_sizes, const mxmoe_dim3* h_sizes, const mxmoe_qparams* h_q, int count, hipStream_t stream) {
  if (count <= 0) return 0;
  auto& reg = registry();
  if (kernel_id < 0) {
    kernel_id = auto_kernel(h_sizes, h_q, count);
    if (kernel_id < 0) {
      last_error() = "quant type not supported";  // same message as the reference launcher (compose_kernel.py:433)
      return 1;
    }
  }
  if (kernel_id >= (int)reg.size()) {
    last_error() = "kernel id out of range";
    return 2;
  }
  const FusedKernel& k = reg[kernel_id];
  for (int i = 0; i < count; ++i) {  // the tiles read the scales unconditionally: refuse a launch whose scale arrays are missing
    const Fmt f = classify(h_q[i]);
    const bool wa = f == Fmt::W8A8 || f == Fmt::W4A4 || f == Fmt::W4A4G128;
    const bool wo = is_weight_only(f);
    if (h_sizes[i].x != 0 && ((wa && (!sa || !sb)) || (wo && !sb))) {
      last_error() = "scale arrays are required for quantised formats";
      return 5;
    }
  }
  auto run = [&](int base, int n, hipStream_t s) { return launch_range(k, As, Bs, sa, sb, Cs, acc, d_sizes, h_sizes, h_q, base, n, s); };
  if (k.policy == Policy::Fused) {
    for (int base = 0; base < count; base += kMaxProblems)
      if (const int rc = run(base, std::min(kMaxProblems, count - base), stream)) return rc;
    return 0;
  }
  SideStreams* side = nullptr;
  if (k.policy == Policy::MultiStream) {
    side = side_streams();
    if (!side || hipEventRecord(side->fork, stream) != hipSuccess) {
      last_error() = "could not set up the side streams of the multi-stream policy";
      return 4;
    }
  }
  int nrun = 0, rc = 0;
  unsigned used = 0;
  for (int base = 0; base < count && rc == 0;) {
    const int n = launch_length(k, h_q, base, count);
    hipStream_t s = stream;
    if (side) {
      const int si = nrun % kSideStreams;
      s = side->stream[si];
      if (!(used >> si & 1) && hipStreamWaitEvent(s, side->fork, 0) != hipSuccess) rc = 4;
      used |= 1u << si;
    }
    if (rc == 0) rc = run(base, n, s);
    base += n;
    ++nrun;
  }
  if (side) {  // join whatever was forked, also after a failure, so that the caller's stream stays ordered after the side work
    for (int si = 0; si < kSideStreams; ++si)
      if (used >> si & 1)
        if (hipEventRecord(side->join[si], side->stream[si]) != hipSuccess || hipStreamWaitEvent(stream, side->join[si], 0) != hipSuccess) rc = rc ? rc : 4;
    if (rc == 4 && last_error().empty()) last_error() = "stream fork / join failed";
  }
  return rc;
}

}  // namespace mxmoe

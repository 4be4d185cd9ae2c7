// The planned layer forward in its short form: four or five launches from (hidden, expert ids, weights) to the layer's output.
//
//   head      permutation by expert, the tables of both GroupGEMMs, and every token quantised once per activation format: three
//             jobs that need nothing of each other, in one launch;
//   gate_up   the fused GroupGEMM in its gate_up form (TileArgs): rows gathered by token, output silu(gate) * up;
//   rows      rotation + quantisation of those rows for the second block (left out when every second block reads fp16 rows);
//   down      the fused GroupGEMM of the second block;
//   combine   un-permute, top-k weighted sum, shared expert.
//
// Against the form that writes an activation row per destination (top-k of them per token, after the permutation is known) and stores
// gate and up: the head is one launch instead of two or three in sequence, activations take 1 / top-k of the space, and 8 bytes per
// intermediate value are neither written nor read.  The same kernels' arithmetic, bit for bit.  Measured, that form -> this one, us a
// pass: DeepSeek-V2-Lite w4a16 / w3a16 47.7 -> 35.2 (1 token), 98.7 -> 84.9 (32), 163 -> 139 (201); Qwen1.5-MoE w4a4 456 -> 402 (8192,
// of which the head 47 -> 24, the activation step 107 -> 72); Mixtral w4a4 / w8a8 / w4a16 3368 -> 3249 (8192).
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

constexpr int kHeadThreads = 256;
// Experts of the short form: its permutation workgroups keep six counters per expert in LDS (24 KiB at this many).
constexpr int kHeadMaxExperts = 1024;
// Entries (tokens x top-k) up to which every workgroup that needs counts takes them from the ids themselves, all of them: 128 KiB of ids
// out of L2 and as many LDS counter updates take some 6 us, which the token workgroups of the same launch hide; beyond, the cost
// per workgroup would grow with the batch, and a counting launch (perm_hist_kernel) goes first.
constexpr int kHeadCountMax = 65536;

struct HeadArgs {
  const int32_t* ids;
  int total, E, topk, nbits;
  int perm_wgs;          // workgroups of kPermChunk entries each
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
__device__ __forceinline__ void count_ids(const int32_t* __restrict__ ids, int total, int E, int base, int32_t* before, int32_t* all) {
  for (int e = threadIdx.x; e < E; e += kHeadThreads) {
    all[e] = 0;
    if (before) before[e] = 0;
  }
  __syncthreads();
  auto add = [&](int idx, int e) {
    if (e >= 0 && e < E) {
      atomicAdd(&all[e], 1);
      if (before && idx < base) atomicAdd(&before[e], 1);
    }
  };
  if ((reinterpret_cast<uintptr_t>(ids) & 15) == 0) {  // 16 bytes per lane and load, eight loads in flight: a handful of round trips for a full batch
    const int n4 = total >> 2;
    constexpr int kAhead = 8;
    for (int i0 = threadIdx.x; i0 < n4; i0 += kAhead * kHeadThreads) {
      v4i v[kAhead];
#pragma unroll
      for (int k = 0; k < kAhead; ++k) v[k] = reinterpret_cast<const v4i*>(ids)[min(i0 + k * kHeadThreads, n4 - 1)];
#pragma unroll
      for (int k = 0; k < kAhead; ++k) {
        const int i = i0 + k * kHeadThreads;
        if (i < n4) {
#pragma unroll
          for (int j = 0; j < 4; ++j) add(4 * i + j, v[k][j]);
        }
      }
    }
    for (int i = (n4 << 2) + threadIdx.x; i < total; i += kHeadThreads) add(i, ids[i]);
  } else {
    for (int i = threadIdx.x; i < total; i += kHeadThreads) add(i, ids[i]);
  }
  __syncthreads();
}

// One chunk of the stable permutation by expert: each wave places 64 consecutive entries.
__device__ __forceinline__ void head_scatter(const HeadArgs& a, int block, int32_t* lds) {
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  int32_t *all = lds, *run = lds + a.E, *in_wave = lds + 2 * a.E;  // [E] totals, [E] first row of this chunk's entries, [4][E] entries per wave
  const int idx = block * kPermChunk + wave * 64 + lane;
  const bool ok = idx < a.total;
  int e = ok ? a.ids[idx] : -1;
  if (e < 0 || e >= a.E) e = a.E;  // parked on a dummy id, never written
  for (int i = threadIdx.x; i < 4 * a.E; i += kHeadThreads) in_wave[i] = 0;
  if (a.hist) {
    for (int x = threadIdx.x; x < a.E; x += kHeadThreads) {
      int v, before;
      perm_hist_row_sums(a.hist + (long)x * perm_hist_stride(a.perm_wgs), a.perm_wgs, block, &v, &before);
      all[x] = v;
      run[x] = before;
    }
    __syncthreads();
  } else {
    count_ids(a.ids, a.total, a.E, block * kPermChunk, run, all);
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
  const _Float16* srow = a.hidden + (long)t * n;
  float v[NI][8];
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    const v8h g = *reinterpret_cast<const v8h*>(srow + (lane + 64 * i) * 8);
#pragma unroll
    for (int j = 0; j < 8; ++j) v[i][j] = (float)g[j];
  }
  if (a.rotate != 0) wave_rotate<NI>(v, lane, a.scale);
  if (a.tags & 1u) {  // fp16: only when every row is rotated (else the GEMM reads the tokens where they are)
    _Float16* out = reinterpret_cast<_Float16*>(a.store[0]) + (long)t * n;
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      v8h o;
#pragma unroll
      for (int j = 0; j < 8; ++j) o[j] = (_Float16)v[i][j];
      *reinterpret_cast<v8h*>(out + (lane + 64 * i) * 8) = o;
    }
  }
  auto codes4 = [&](const float (&x)[8], float scale) {
    const ScaleDiv div(scale);
    unsigned w = 0;
#pragma unroll
    for (int j = 0; j < 8; ++j) w = push_code<4>(w, code_word(fminf(fmaxf(round_h(div(x[j])), -7.0f), 7.0f)));
    return w;
  };
  // fp16 division: fp32 quotient of two fp16 values, rounded to fp16; a zero row gets 1 (quantize.cuh:258)
  auto scale_of = [](float amax, float upper) {
    const float scale = round_h(amax / upper);
    return scale == 0.0f ? 1.0f : scale;
  };
  if (a.tags & 8u) {  // tag 3: int4, one scale per 128 values = the 16 chunks held by an aligned group of 16 lanes
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      const int c = lane + 64 * i;
      float gmax = 0.0f;
#pragma unroll
      for (int j = 0; j < 8; ++j) gmax = fmaxf(gmax, fabsf(v[i][j]));
      const float scale = scale_of(row16_max(gmax), 7.0f);
      if ((c & 15) == 0) a.scales[3][(long)t * (n >> 7) + (c >> 4)] = (_Float16)scale;
      *reinterpret_cast<unsigned*>(a.store[3] + (long)t * (n / 2) + c * 4) = codes4(v[i], scale);
    }
  }
  if ((a.tags & 0x26u) == 0) return;
  float amax = 0.0f;
#pragma unroll
  for (int i = 0; i < NI; ++i)
#pragma unroll
    for (int j = 0; j < 8; ++j) amax = fmaxf(amax, fabsf(v[i][j]));
  amax = wave_max(amax);
  if (a.tags & 2u) {  // tag 1: int8 per token
    const float scale = scale_of(amax, 127.0f);
    const ScaleDiv div(scale);
    if (lane == 0) a.scales[1][t] = (_Float16)scale;
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      uint2 w{0, 0};
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        w.x = push_code<8>(w.x, code_word(fminf(fmaxf(round_h(div(v[i][j])), -127.0f), 127.0f)));
        w.y = push_code<8>(w.y, code_word(fminf(fmaxf(round_h(div(v[i][j + 4])), -127.0f), 127.0f)));
      }
      *reinterpret_cast<uint2*>(a.store[1] + (long)t * n + (lane + 64 * i) * 8) = w;
    }
  }
  if (a.tags & 0x20u) {  // tag 5: fp8 e4m3 per token
    const float scale = scale_of(amax, 448.0f);
    const ScaleDiv div(scale);
    if (lane == 0) a.scales[5][t] = (_Float16)scale;
#pragma unroll
    for (int i = 0; i < NI; ++i) *reinterpret_cast<uint2*>(a.store[5] + (long)t * n + (lane + 64 * i) * 8) = fp8_chunk_codes(v[i], div);
  }
  if (a.tags & 4u) {  // tag 2: int4 per token
    const float scale = scale_of(amax, 7.0f);
    if (lane == 0) a.scales[2][t] = (_Float16)scale;
#pragma unroll
    for (int i = 0; i < NI; ++i) *reinterpret_cast<unsigned*>(a.store[2] + (long)t * (n / 2) + (lane + 64 * i) * 4) = codes4(v[i], scale);
  }
}

// Workgroups: planning first (the longest chain of dependent steps), then the permutation's chunks, then tokens, four per workgroup.
template <int NI>
__global__ void __launch_bounds__(kHeadThreads) layer_head_kernel(const HeadArgs a, const PlanPair pair) {
  extern __shared__ __align__(16) int32_t head_lds[];
  const int plan_wgs = 2 * pair.chunks;
  int wg = blockIdx.x;
  if (wg < plan_wgs) {
    if (a.hist) {
      for (int e = threadIdx.x; e < a.E; e += kHeadThreads) {
        int v, before;
        perm_hist_row_sums(a.hist + (long)e * perm_hist_stride(a.perm_wgs), a.perm_wgs, 0, &v, &before);
        head_lds[e] = v;
      }
      __syncthreads();
    } else {
      count_ids(a.ids, a.total, a.E, 0, nullptr, head_lds);
    }
    if (threadIdx.x < kPlanThreads) plan_block_body(pair.p[wg / pair.chunks], wg % pair.chunks, pair.chunks, head_lds);
    return;
  }
  wg -= plan_wgs;
  if (wg < a.perm_wgs) {
    head_scatter(a, wg, head_lds);
    return;
  }
  wg -= a.perm_wgs;
  const int token_wgs = (int)gridDim.x - plan_wgs - a.perm_wgs;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  for (int t = wg * 4 + wave; t < a.T; t += token_wgs * 4) head_token<NI>(a, t, lane);
}

// What a layer keeps for one (tokens, top-k): its description and both launches' planning parameters.
struct LayerForward {
  mxmoe_layer_desc d;
  HeadArgs head;
  PlanPair pair;
  int et, token_wgs;
  bool fp16_first;   // a first block reads the tokens as they are
  bool rows_step;    // a second block takes quantised (or rotated) rows
  RowsBehind rows;
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
  h.perm_wgs = (h.total + kPermChunk - 1) / kPermChunk;
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
  f->token_wgs = tags ? std::min((d->num_tokens + 3) / 4, cus * 8) : 0;

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
    p.info = plan_of(registry()[kid]);
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

void mxmoe_layer_destroy(void* handle) { delete reinterpret_cast<LayerForward*>(handle); }

int mxmoe_layer_run(const void* handle, const void* hidden, const int32_t* topk_ids, const float* topk_weights, void* out, void* stream) {
  if (!handle || !hidden || !topk_ids || !topk_weights || !out) {
    last_error() = "null pointer";
    return 5;
  }
  const LayerForward& f = *reinterpret_cast<const LayerForward*>(handle);
  const mxmoe_layer_desc& d = f.d;
  hipStream_t s = (hipStream_t)stream;
  HeadArgs h = f.head;
  PlanPair pair = f.pair;
  h.ids = topk_ids;
  h.hidden = reinterpret_cast<const _Float16*>(hidden);
  if (f.fp16_first) pair.p[0].form.store[0] = reinterpret_cast<const uint8_t*>(hidden);
  if (h.hist) launch_perm_hist(topk_ids, h.total, h.E, const_cast<int32_t*>(h.hist), true, s);
  const dim3 grid(2 * pair.chunks + h.perm_wgs + f.token_wgs), block(kHeadThreads);
  const size_t lds = (size_t)6 * h.E * sizeof(int32_t);
  switch (d.hidden / 512) {
    case 1: hipLaunchKernelGGL((layer_head_kernel<1>), grid, block, lds, s, h, pair); break;
    case 2: hipLaunchKernelGGL((layer_head_kernel<2>), grid, block, lds, s, h, pair); break;
    case 4: hipLaunchKernelGGL((layer_head_kernel<4>), grid, block, lds, s, h, pair); break;
    default: hipLaunchKernelGGL((layer_head_kernel<8>), grid, block, lds, s, h, pair); break;
  }
  if (const int rc = check_launch()) return rc;
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
  const FusedKernel &kg = registry()[d.kernel_gate_up], &kd = registry()[d.kernel_down];
  if (const int rc = gemm(kg.launch_gate_up, kg, d.plan_gate_up, d.grid_gate_up)) return rc;
  if (f.rows_step)
    if (const int rc = quant_rows_behind(f.rows, s)) return rc;
  if (const int rc = gemm(kd.launch_planned, kd, d.plan_down, d.grid_down)) return rc;
  return mxmoe_combine_planned(d.down_out, d.plan_down, f.et, topk_weights, d.row_of_slot, d.num_tokens, d.topk, d.hidden, out, stream);
}

}  // extern "C"

// Row arithmetic shared by the activation quantisers: rounding, the division by a row's scale, codes, lane exchanges and the Sylvester
// rotation of a row held by one wave.  Every step is a fixed sequence of correctly rounded operations (FMA contraction is off), so
// codes and scales are reproducible bit for bit on a CPU.
#pragma once
#include <hip/hip_runtime.h>

#include "mxmoe_tiles.hpp"

namespace mxmoe {

// Load of a value that no kernel of this launch writes (routing arrays, expert table), through the constant address space: with a
// wave-uniform address it is a scalar load into scalar registers, off the vector register budget.
template <class T>
__device__ __forceinline__ T const_load(const T* p) {
  return *(const __attribute__((address_space(4))) T*)(p);
}

__device__ __forceinline__ float round_h(float v) { return (float)(_Float16)v; }

// Integer code of a value already clamped to the code range, as the low bits of a word: the addition of 1.5 * 2^23 rounds to an
// integer by itself (to nearest, ties to even: rintf) and leaves its two's complement in the low mantissa bits.  push_code<BITS>
// shifts a word of codes right by BITS and puts the new code on top: after 32 / BITS pushes the first code sits in the lowest bits.
__device__ __forceinline__ unsigned code_word(float clamped) { return __float_as_uint(clamped + 12582912.0f); }
template <int BITS>
__device__ __forceinline__ unsigned push_code(unsigned w, unsigned code) {
  return __builtin_amdgcn_alignbit(code, w, BITS);
}

// v / s in fp32 for fp16-valued v and s, given r = 1.0f / s: the rounded product v * r corrected once with its exact remainder.
// With r the correctly rounded reciprocal this is the correctly rounded quotient, i.e. bit for bit what the division instruction
// sequence returns, for every pair of fp16 values (checked with exact integer arithmetic over all 2^20 mantissa pairs in
// tests/test_oracle_quant.py); a row's elements share one scale, so the division proper is done once per row.
// An infinite scale (a row that already holds an infinity) keeps the plain result: finite / inf = 0.
struct ScaleDiv {
  float r, s;
  __device__ __forceinline__ explicit ScaleDiv(float scale) : r(1.0f / scale), s(__builtin_isinf(scale) ? 0.0f : scale) {}
  __device__ __forceinline__ float operator()(float v) const {
    const float q0 = v * r;
    const float e = __builtin_fmaf(-s, q0, v);
    return __builtin_fmaf(e, r, q0);
  }
};

// Value of lane (l ^ M), M = 1 .. 8: data-parallel-primitive moves inside a row of 16 lanes, in the vector ALU (quad permutations;
// l ^ 4 = mirror of 8 lanes, then of 4; l ^ 8 = a rotation of the row by 8).
template <int M>
__device__ __forceinline__ float lane_xor(float v) {
  int x = __float_as_int(v);
  if constexpr (M == 1) {
    x = __builtin_amdgcn_update_dpp(0, x, 0xB1, 0xF, 0xF, true);   // quad_perm [1,0,3,2]
  } else if constexpr (M == 2) {
    x = __builtin_amdgcn_update_dpp(0, x, 0x4E, 0xF, 0xF, true);   // quad_perm [2,3,0,1]
  } else if constexpr (M == 4) {
    x = __builtin_amdgcn_update_dpp(0, x, 0x141, 0xF, 0xF, true);  // row_half_mirror: l ^ 7
    x = __builtin_amdgcn_update_dpp(0, x, 0x1B, 0xF, 0xF, true);   // quad_perm [3,2,1,0]: l ^ 3
  } else {
    static_assert(M == 8, "larger distances: lane_butterfly");
    x = __builtin_amdgcn_update_dpp(0, x, 0x128, 0xF, 0xF, true);  // row_ror:8: lane (l + 8) mod 16 = l ^ 8
  }
  return __int_as_float(x);
}

// One butterfly stage across lanes of two values at once: lane pairs (l, l ^ M) end up with (own + other) in the lower lane of the pair
// and (other - own) in the upper one, each rounded once.
// M <= 8: an exchange and one fused multiply-add with own's sign (the product with +-1 is exact) per value.
// M = 16, 32: the half-wave swap instructions of gfx950 turn the lane distance into a register distance: after the swap one register
// holds the lower partners of both values and the other the upper ones, a sum and a difference do the stage, and a second swap puts
// the results back: two instructions per value in the vector ALU, where a lane exchange of that distance through the LDS crossbar
// (ds_bpermute) shares one LDS pipe among the four SIMDs of a CU.
template <int M>
__device__ __forceinline__ void lane_butterfly(float& a, float& b, int lane) {
  if constexpr (M <= 8) {
    const float sgn = (lane & M) ? -1.0f : 1.0f;
    a = __builtin_fmaf(sgn, a, lane_xor<M>(a));
    b = __builtin_fmaf(sgn, b, lane_xor<M>(b));
  } else {
    static_assert(M == 16 || M == 32, "a wave has 64 lanes");
    auto swap = [](float x, float y) {
      if constexpr (M == 16) return __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(y), false, false);
      else return __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(y), false, false);
    };
    const auto t = swap(a, b);
    const float lo = __uint_as_float(t[0]), hi = __uint_as_float(t[1]);
    const float sum = lo + hi, dif = lo - hi;
    const auto r = swap(sum, dif);
    a = __uint_as_float(r[0]);
    b = __uint_as_float(r[1]);
  }
}

// Largest value over the wave of values that are not negative (or NaN-free in general), in every lane; vector ALU only.
__device__ __forceinline__ float wave_max(float v) {
  v = fmaxf(v, lane_xor<1>(v));
  v = fmaxf(v, lane_xor<2>(v));
  v = fmaxf(v, lane_xor<4>(v));
  v = fmaxf(v, lane_xor<8>(v));
  const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
  const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1]));
}
// Largest value over each aligned group of 16 lanes.
__device__ __forceinline__ float row16_max(float v) {
  v = fmaxf(v, lane_xor<8>(v));
  v = fmaxf(v, lane_xor<4>(v));
  v = fmaxf(v, lane_xor<2>(v));
  return fmaxf(v, lane_xor<1>(v));
}

// ---- tag 5: per-token fp8 (OCP e4m3) codes for the kernels whose w8a8 tiles run the fp8 matrix instruction.  scale = max|x| / 448
// (the largest e4m3 number) in fp16 like the integer scales; code = e4m3(clamp(fp16(x / scale), +-448)), round to nearest even; rows
// are stored like int8 rows, one byte per value.
template <class Div>
__device__ __forceinline__ uint2 fp8_chunk_codes(const float (&v)[8], const Div& div) {
  float r[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) r[j] = fminf(fmaxf(round_h(div(v[j])), -448.0f), 448.0f);
  int lo = 0, hi = 0;
  lo = __builtin_amdgcn_cvt_pk_fp8_f32(r[0], r[1], lo, false);
  lo = __builtin_amdgcn_cvt_pk_fp8_f32(r[2], r[3], lo, true);
  hi = __builtin_amdgcn_cvt_pk_fp8_f32(r[4], r[5], hi, false);
  hi = __builtin_amdgcn_cvt_pk_fp8_f32(r[6], r[7], hi, true);
  return make_uint2((unsigned)lo, (unsigned)hi);
}

// H_n x * scale for a row of n = 512 * NI values held by one wave (lane l: the NI chunks l + 64 i of 8 values), every level rounded
// to fp32 in ascending order of stride and the scaled result rounded to fp16: strides 1, 2, 4 inside a chunk, 8 .. 256 across
// lanes, 512 and up across the chunks of a lane.
template <int NI>
__device__ __forceinline__ void wave_rotate(float (&v)[NI][8], int lane, float scale) {
#pragma unroll
  for (int i = 0; i < NI; ++i)
#pragma unroll
    for (int h = 1; h < 8; h <<= 1)
#pragma unroll
      for (int j = 0; j < 8; ++j)
        if (!(j & h)) {
          const float p = v[i][j], q = v[i][j + h];
          v[i][j] = p + q;
          v[i][j + h] = p - q;
        }
  auto lane_stage = [&](auto mc) {
#pragma unroll
    for (int i = 0; i < NI; ++i)
#pragma unroll
      for (int j = 0; j < 8; j += 2) lane_butterfly<decltype(mc)::value>(v[i][j], v[i][j + 1], lane);
  };
  lane_stage(std::integral_constant<int, 1>{});
  lane_stage(std::integral_constant<int, 2>{});
  lane_stage(std::integral_constant<int, 4>{});
  lane_stage(std::integral_constant<int, 8>{});
  lane_stage(std::integral_constant<int, 16>{});
  lane_stage(std::integral_constant<int, 32>{});
#pragma unroll
  for (int hi = 1; hi < NI; hi <<= 1)
#pragma unroll
    for (int i = 0; i < NI; ++i)
      if (!(i & hi)) {
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          const float p = v[i][j], q = v[i + hi][j];
          v[i][j] = p + q;
          v[i + hi][j] = p - q;
        }
      }
#pragma unroll
  for (int i = 0; i < NI; ++i)
#pragma unroll
    for (int j = 0; j < 8; ++j) v[i][j] = round_h(keep_f32(v[i][j] * scale));
}

// The activation step behind a gate_up form (act_kernels.hip): rows that are already silu(gate) * up -> rotation, quantisation,
// packing into the store of the second block, for the rows of experts whose second block is not fp16 (or all rows when every row is
// rotated).  Everything that depends on the routing is read from the two plan buffers.
struct RowsBehind {
  const void* rows;  // [rows_capacity][n] fp16, rows sorted by expert; the shared expert's [num_tokens][n_shared] where the gate_up plan put them
  const uint8_t *plan_gate_up, *plan_down;
  uint8_t* inp_store;
  _Float16* scale_store;
  const int32_t* dst_exp;  // expert of each routed row
  int n, n_shared, rows_capacity, num_tokens, num_experts;
  bool has_shared, variants;
  int rotate, had_k, had_f;
  const float* had_signs;
};
int quant_rows_behind(const RowsBehind& b, hipStream_t stream);

}  // namespace mxmoe

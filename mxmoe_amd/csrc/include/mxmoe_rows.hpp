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

// A finished row is held as what it is, fp16 values, eight to a chunk: half the registers of fp32 copies, and two values to an instruction in its maximum and its
// codes.  (The quantisers are bound by their vector instructions: a code of int8 takes 3.75 and of int4 4.25, in fp32 it took 7.75 and 8; a value of the maximum half a one instead of
// one and a half.)

// Largest magnitude: two values of a chunk per instruction, NaN ignored as fmaxf ignores it.
struct HalfMax {
  unsigned m = 0;  // an fp16 value in the low half
  __device__ __forceinline__ void add(const v8h& h) {
    const v4i w = __builtin_bit_cast(v4i, h);
#pragma unroll
    for (int d = 0; d < 4; ++d) asm("v_max3_f16 %0, |%1|, |%1|, %2 op_sel:[0,1,0,0]" : "=v"(m) : "v"(w[d]), "v"(m));
  }
  __device__ __forceinline__ float get() const { return (float)__builtin_bit_cast(_Float16, (unsigned short)m); }
};
// The same of a row held in fp32.
struct FloatMax {
  float m = 0.0f;
  __device__ __forceinline__ void add(const float (&v)[8]) {
#pragma unroll
    for (int j = 0; j < 8; ++j) m = fmaxf(m, fabsf(v[j]));
  }
  __device__ __forceinline__ float get() const { return m; }
};
template <class Chunk>
using AbsMax = std::conditional_t<std::is_same_v<Chunk, v8h>, HalfMax, FloatMax>;
// A chunk as packed halves: of a row that is held so, or of one held in fp32 (values that are fp16 numbers).
__device__ __forceinline__ const v8h& as_half(const v8h& h) { return h; }
__device__ __forceinline__ v8h as_half(const float (&v)[8]) {
  v8h h;
#pragma unroll
  for (int j = 0; j < 8; ++j) h[j] = (_Float16)v[j];
  return h;
}
// A row that goes on as it was read: signalling NaNs become quiet ones, as a trip through fp32 makes them.
__device__ __forceinline__ v8h quiet(const v8h& h) { return __builtin_elementwise_canonicalize(h); }

// Integer codes of a row whose scale is known: clamp(fp16(v / scale), +-UPPER) rounded to the nearest integer, ties to even.  Two values at a time in fp16: value and
// scale times the power of two that brings the scale into 1 .. 2 (a scale below the normal numbers: into 2^-9 .. 1), the product with the reciprocal corrected
// once with its remainder, and 1536 added, where fp16 numbers are integers, so that the code's two's complement is left in the low mantissa bits.  The same
// code as from the fp32 quotient for every value and scale that a row can have (test_codes_from_packed_halves_are_those_of_the_fp32_quotient goes through all
// of them).  An infinite scale (a row that holds an infinity) keeps the plain product: finite / inf = 0.
struct HalfDiv {
  v2h up, s, r;  // both halves alike
  __device__ __forceinline__ explicit HalfDiv(float scale) {
    const int e = (__float_as_int(scale) >> 23) - 127;  // scale > 0
    const float f = __int_as_float((127 + min(max(-e, -15), 15)) << 23);
    const _Float16 hu = (_Float16)f, hs = (_Float16)(__builtin_isinf(scale) ? 0.0f : scale * f), hr = (_Float16)__builtin_amdgcn_rcpf(scale * f);
    up = v2h{hu, hu};
    s = v2h{hs, hs};
    r = v2h{hr, hr};
  }
  template <int UPPER>
  __device__ __forceinline__ unsigned codes(v2h v) const {
    const v2h x = v * up;
    const v2h q0 = x * r;
    v2h q = __builtin_elementwise_fma(__builtin_elementwise_fma(-q0, s, x), r, q0);
    const _Float16 top = UPPER, magic = 1536;
    q = __builtin_elementwise_min(__builtin_elementwise_max(q, v2h{-top, -top}), v2h{top, top});
    return __builtin_bit_cast(unsigned, q + v2h{magic, magic});
  }
  template <int UPPER>
  __device__ __forceinline__ void codes8(const v8h& h, unsigned (&w)[4]) const {
#pragma unroll
    for (int d = 0; d < 4; ++d) w[d] = codes<UPPER>(v2h{h[2 * d], h[2 * d + 1]});
  }
  // eight int8 codes, the first in the lowest byte
  __device__ __forceinline__ uint2 int8(const v8h& h) const {
    unsigned w[4];
    codes8<127>(h, w);
    return make_uint2(__builtin_amdgcn_perm(w[1], w[0], 0x06040200), __builtin_amdgcn_perm(w[3], w[2], 0x06040200));
  }
  // eight int4 codes, the first in the lowest bits
  __device__ __forceinline__ unsigned int4(const v8h& h) const {
    unsigned w[4];
    codes8<7>(h, w);
    const unsigned a = __builtin_amdgcn_perm(w[1], w[0], 0x06020400), b = __builtin_amdgcn_perm(w[3], w[2], 0x06020400);  // codes 0 2 1 3, 4 6 5 7
    const unsigned even = __builtin_amdgcn_perm(b, a, 0x05040100), odd = __builtin_amdgcn_perm(b, a, 0x07060302);
    return (even & 0x0F0F0F0Fu) | (odd << 4 & 0xF0F0F0F0u);
  }
};

// H_8 of a chunk of fp16 values, in fp32: strides 1, 2, 4.  The first stage takes the halves as they are (mixed-precision fused multiply-adds by one and minus one:
// sums and differences rounded once, without conversions in front).
__device__ __forceinline__ void chunk_h8(const v8h& h, float (&v)[8]) {
  float one = 1.0f;
  asm("" : "+s"(one));  // (a multiplication by a visible 1 would be folded away, and with it the mixed-precision form)
#pragma unroll
  for (int j = 0; j < 8; j += 2) {
    v[j] = __builtin_fmaf((float)h[j + 1], one, (float)h[j]);
    v[j + 1] = __builtin_fmaf((float)h[j + 1], -one, (float)h[j]);
  }
#pragma unroll
  for (int st = 2; st < 8; st <<= 1)
#pragma unroll
    for (int j = 0; j < 8; ++j)
      if (!(j & st)) {
        const float p = v[j], q = v[j + st];
        v[j] = p + q;
        v[j + st] = p - q;
      }
}

// fp16(v * scale), the product rounded to fp32 first; `mx` follows the largest magnitude (of the products: their maximum, rounded, is that of the rounded ones)
__device__ __forceinline__ v8h scale_chunk(const float (&v)[8], float scale, float& mx) {
  v8h h;
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const float p = keep_f32(v[j] * scale);
    h[j] = (_Float16)p;
    mx = fmaxf(mx, fabsf(p));
  }
  return h;
}

// The chunk on the exact grid of the dense stage: rint(h * to_grid) / 16, a number of at most 2^13 in steps of 1/16.  One fused operation rounds to the grid
// (beside 1.5 * 2^19 an fp32 number has steps of 1/16), one takes the offset off and converts; both are exact otherwise.
__device__ __forceinline__ v8h snap_chunk(const v8h& h, float to_grid) {
  const float to16 = to_grid * 0.0625f;
  float one = 1.0f, off = 786432.0f;
  asm("" : "+s"(one), "+s"(off));
  v8h q;
#pragma unroll
  for (int j = 0; j < 8; ++j) q[j] = (_Float16)__builtin_fmaf(__builtin_fmaf((float)h[j], to16, off), one, -off);
  return q;
}

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

// The stage across lanes l ^ M for the eight values of a chunk.
// M = 4: the partner is four lanes up for the even quads of a row of 16 lanes and four lanes down for the odd ones, so an addition with its exchange built in writes
// the even quads and a subtraction the odd ones (bank masks): two instructions a value, where an exchange of that distance takes two by itself.  (Two wait
// states are due between a vector write and a lane exchange that reads it: the compiler does not see into the block.)
template <int M>
__device__ __forceinline__ void lane_stage(float (&v)[8], int lane) {
  if constexpr (M == 4) {
    float o[8];
#define MXMOE_XOR4(n, src) "\n\tv_add_f32_dpp %" #n ", %" #src ", %" #src " row_shl:4 row_mask:0xf bank_mask:0x5\n\tv_sub_f32_dpp %" #n ", %" #src ", %" #src " row_shr:4 row_mask:0xf bank_mask:0xa"
    asm("s_nop 1" MXMOE_XOR4(0, 8) MXMOE_XOR4(1, 9) MXMOE_XOR4(2, 10) MXMOE_XOR4(3, 11) MXMOE_XOR4(4, 12) MXMOE_XOR4(5, 13) MXMOE_XOR4(6, 14) MXMOE_XOR4(7, 15) "\n\ts_nop 1"
        : "=&v"(o[0]), "=&v"(o[1]), "=&v"(o[2]), "=&v"(o[3]), "=&v"(o[4]), "=&v"(o[5]), "=&v"(o[6]), "=&v"(o[7])
        : "v"(v[0]), "v"(v[1]), "v"(v[2]), "v"(v[3]), "v"(v[4]), "v"(v[5]), "v"(v[6]), "v"(v[7]));
#undef MXMOE_XOR4
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = o[j];
  } else {
#pragma unroll
    for (int j = 0; j < 8; j += 2) lane_butterfly<M>(v[j], v[j + 1], lane);
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
// The same of magnitudes (no NaN, no sign), whose bit patterns order like the values: one instruction a step, as the lane exchange is part of an integer
// maximum and nothing has to be made canonical.
__device__ __forceinline__ unsigned max_xor8421(unsigned x) {
  auto dpp = [](unsigned v, auto ctrl) { return (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, decltype(ctrl)::value, 0xF, 0xF, true); };
  x = max(x, dpp(x, std::integral_constant<int, 0xB1>{}));         // quad_perm [1,0,3,2]
  x = max(x, dpp(x, std::integral_constant<int, 0x4E>{}));         // quad_perm [2,3,0,1]: a quad is alike
  x = max(x, dpp(x, std::integral_constant<int, 0x141>{}));        // row_half_mirror: the other quad of 8 lanes
  return max(x, dpp(x, std::integral_constant<int, 0x128>{}));     // row_ror:8
}
__device__ __forceinline__ float wave_max_abs(float v) {
  unsigned x = max_xor8421(__float_as_uint(v));
  const auto a = __builtin_amdgcn_permlane16_swap(x, x, false, false);
  x = max(a[0], a[1]);
  const auto b = __builtin_amdgcn_permlane32_swap(x, x, false, false);
  return __uint_as_float(max(b[0], b[1]));
}
// ... over each aligned group of 16 lanes.
__device__ __forceinline__ float row16_max_abs(float v) { return __uint_as_float(max_xor8421(__float_as_uint(v))); }

// ---- tag 5: per-token fp8 (OCP e4m3) codes for the kernels whose w8a8 tiles run the fp8 matrix instruction.  scale = max|x| / 448
// (the largest e4m3 number) in fp16 like the integer scales; code = e4m3(clamp(fp16(x / scale), +-448)), round to nearest even; rows
// are stored like int8 rows, one byte per value.
template <class Chunk>
__device__ __forceinline__ uint2 fp8_chunk_codes(const Chunk& h, const ScaleDiv& div) {
  float r[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) r[j] = fminf(fmaxf(round_h(div((float)h[j])), -448.0f), 448.0f);
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
__device__ __forceinline__ void wave_rotate(v8h (&h)[NI], int lane, float scale) {
  float v[NI][8];
#pragma unroll
  for (int i = 0; i < NI; ++i) {  // (chunk by chunk: stage by stage over all of them takes more registers)
    chunk_h8(h[i], v[i]);
    lane_stage<1>(v[i], lane);
    lane_stage<2>(v[i], lane);
    lane_stage<4>(v[i], lane);
    lane_stage<8>(v[i], lane);
    lane_stage<16>(v[i], lane);
    lane_stage<32>(v[i], lane);
  }
  // Chunk by chunk, stage by stage: the compiler otherwise follows single results through all the stages and keeps the operands of the others (rows of 4096 values: 162
  // registers instead of 121 in the layer's first kernel, 182 instead of 142 in row_quant_wave_kernel, of which 16 384 rows take 64.6 us instead of 58.4).
  auto formed = [](float (&x)[8]) {
    asm volatile("" : "+v"(x[0]), "+v"(x[1]), "+v"(x[2]), "+v"(x[3]), "+v"(x[4]), "+v"(x[5]), "+v"(x[6]), "+v"(x[7]));
  };
#pragma unroll
  for (int i = 0; i < NI; ++i) formed(v[i]);
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
        formed(v[i]);
        formed(v[i + hi]);
      }
#pragma unroll
  for (int i = 0; i < NI; ++i)
#pragma unroll
    for (int j = 0; j < 8; ++j) h[i][j] = (_Float16)keep_f32(v[i][j] * scale);
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

// WxAxNarrowTile: w4a4 / w8a8 (int8 or fp8) tile for launches with fewer workgroups than the chip has room for (decode batches on a few experts).
//
// 32 tokens x 64 channels per workgroup, K dealt to the four waves in contiguous quarters, against 32 x 256 with all of K per wave (WxAxTile): four times the
// workgroups and a quarter of the steps in each, for problems whose weight stream is all there is.  The 128 workgroups that the wide tile makes of eight
// experts of N = 4096, K = 14336 leave half of the CUs idle: w4a4 and w8a8 half and half 90 us whatever the number of tokens, 62 here (w8a8 alone 97 -> 82, w4a4
// 56 -> 44); by blocks, rows and formats, and for whole layers: few_rows in mxmoe_launch.hpp.  The partial sums are integers: the same result in any order.  (fp8: fp32 sums, added in the waves' order;
// their errors in the 2-norm, 1.2e-5 .. 1.5e-5, are those of the wide tile's single chain, to three digits.)
//
// A wave streams the fragments of its channels (64 bytes of K of 32 channels are 2 KB, WxAxTile's layout) and of all 32 token rows straight into registers, kAhead
// K slices ahead, without LDS or barriers; every load is an untracked one (gload16_untracked) awaited with the exact number of younger loads.  Rows past M
// re-read the last one: a token is a column of the product, and such columns are not stored.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "mxmoe_tiles.hpp"

namespace mxmoe {

template <Op OP>
struct WxAxNarrowTile {
  static_assert(OP == Op::I4 || OP == Op::I8 || OP == Op::F8, "integer sums, which may be added in any order, or fp8, whose partial sums are added in the waves' order");
  static constexpr int BM = 32, BN = 64, FN = 2;
  static constexpr int BK = kRowBytes * 8 / OpTraits<OP>::kBitsPerElem;
  static constexpr int kLdsBytes = kWaves * FN * 4 * 64 * 16;  // partial sums
  static constexpr int kAccRegs = FN * 16;
  static constexpr int kWavesWanted = 2;
  static constexpr int kABits = OpTraits<OP>::kBitsPerElem, kWBits = kABits;
  // K slices in flight per wave: with 6 and 8 the registers (203, 251) leave two workgroups per CU. Planned layers of w4a4 and w8a8
  // experts, us at 3 / 4 / 6 / 8: 60 experts top-4, 32 tokens 76.7 / 77.5 / 84.4 / 87.1; with the shared expert 104.9 / 99.7 / 110.4 / 110.5
  static constexpr int kAhead = 4;
  static constexpr int kLoads = 2 * FN + 2;  // loads per slice: weight fragments, then token fragments

  // 16 bytes per lane from a uniform address and a lane offset below 4 GiB
  __device__ static __forceinline__ v4i load16(const uint8_t* base, unsigned voff) {
    v4i v;
    asm volatile("global_load_dwordx4 %0, %1, %2" : "=v"(v) : "v"(voff), "s"(base) : "memory");
    return v;
  }

  template <bool GU>
  __device__ static __forceinline__ void run(const TileArgs& t, uint8_t* __restrict__ smem) {
    run_rows<GU, GU>(t, smem, [&](int m) {
      if constexpr (GU) return gload4_untracked(t.rows + m);
      else return m;
    });
  }
  // `row_of(m)`: the row of A (and of sa) behind row m of the problem; IN_FLIGHT: it comes from an untracked load.
  template <bool GU, bool IN_FLIGHT, class RowOf>
  __device__ static __forceinline__ void run_rows(const TileArgs& t, uint8_t* __restrict__ smem, RowOf&& row_of) {
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int M = t.M, N = GU ? t.N / 2 : t.N;  // N: output channels
    const unsigned row_bytes = (unsigned)((long)t.K * kABits / 8);
    const int KT = (int)(row_bytes / kRowBytes);
    constexpr int BNO = GU ? BN / 2 : BN;       // output channels of the tile (gate_up form: block 0 = gate, block 1 = up channels)
    const int m0 = t.row0 + t.tile_m * BM, n0 = t.tile_n * BNO;
    const int lrow = lane & 31, nq = (lane >> 5) * 4;
    const int KW = (KT + kWaves - 1) / kWaves;
    const int k0 = min(KT, wave * KW), k1 = min(KT, k0 + KW);

    // what the epilogue needs of this wave's outputs: rows q = wave of every four-channel run (see below)
    const int m = min(m0 + lrow, M - 1);
    int src = row_of(m);
    const _Float16* sb_ptr[FN];
    typedef int v2i __attribute__((ext_vector_type(2)));
    v2i sb_bits[FN];
#pragma unroll
    for (int j = 0; j < FN; ++j) {
      sb_ptr[j] = t.sb + (GU ? j * N + min(n0 + wave * 8 + nq, N - 4) : min(n0 + j * 32 + wave * 8 + nq, N - 4));
      asm volatile("global_load_dwordx2 %0, %1, off" : "=v"(sb_bits[j]) : "v"(sb_ptr[j]) : "memory");
    }

    const int nblk = (N + 31) / 32;
    const uint8_t* bbase[FN];  // blocks past N re-read the last one; their results are never stored
#pragma unroll
    for (int j = 0; j < FN; ++j) bbase[j] = t.B + (long)(GU ? min(n0 / 32, nblk - 1) + j * nblk : min(n0 / 32 + j, nblk - 1)) * KT * 2048;
    v4i w[kAhead][FN][2], x[kAhead][2];
    const uint8_t* const xbase = GU ? t.A : t.A + (long)m0 * row_bytes;
    unsigned xoff = 0;
    auto load_w = [&](auto dc, int kt) {
#pragma unroll
      for (int j = 0; j < FN; ++j)
#pragma unroll
        for (int s = 0; s < 2; ++s) w[decltype(dc)::value][j][s] = load16(bbase[j] + (long)kt * 2048 + s * 1024, lane * 16);
    };
    auto load_x = [&](auto dc, int kt) {
#pragma unroll
      for (int s = 0; s < 2; ++s) x[decltype(dc)::value][s] = load16(xbase + (long)kt * kRowBytes + s * 32, xoff);
    };
    int sa_bits = 0;
    const int klast = max(k1 - 1, 0);
    // (a wave without slices loads the last slice of K and multiplies nothing)
    static_for<kAhead>([&](auto dc) {
      constexpr int d = decltype(dc)::value;
      load_w(dc, min(k0 + d, klast));
      if constexpr (d == 0) {
        if constexpr (IN_FLIGHT) vm_wait_for<FN + 2 * FN>(src);  // (younger: the channel scales and the fragments above)
        xoff = (unsigned)(GU ? src : src - m0) * row_bytes + (lane >> 5) * 16;  // (a gate_up form's store is below 2 GiB)
        sa_bits = gload2_untracked(t.sa + src);
      }
      load_x(dc, min(k0 + d, klast));
    });

    typename OpTraits<OP>::Acc acc[FN];
#pragma unroll
    for (int j = 0; j < FN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[j][r] = 0;
    auto landed = [&](auto dc, auto nc) {
      constexpr int d = decltype(dc)::value, n = decltype(nc)::value;
#pragma unroll
      for (int j = 0; j < FN; ++j)
#pragma unroll
        for (int s = 0; s < 2; ++s) vm_wait_for<n>(w[d][j][s]);
#pragma unroll
      for (int s = 0; s < 2; ++s) vm_wait_for<n>(x[d][s]);
    };
    auto multiply = [&](auto dc) {
      constexpr int d = decltype(dc)::value;
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        if constexpr (OP == Op::I4) {  // int4 pairs widened to bytes holding 16 v (WxAxTile::widen)
          const v4i xl = (x[d][s] << 4) & (int)0xF0F0F0F0, xh = x[d][s] & (int)0xF0F0F0F0;
#pragma unroll
          for (int j = 0; j < FN; ++j) {
            const v4i wl = (w[d][j][s] << 4) & (int)0xF0F0F0F0, wh = w[d][j][s] & (int)0xF0F0F0F0;
            acc[j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(wl, xl, acc[j], 0, 0, 0);
            acc[j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(wh, xh, acc[j], 0, 0, 0);
          }
        } else if constexpr (OP == Op::I8) {
#pragma unroll
          for (int j = 0; j < FN; ++j) acc[j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(w[d][j][s], x[d][s], acc[j], 0, 0, 0);
        }
      }
      if constexpr (OP == Op::F8) {
#pragma unroll
        for (int j = 0; j < FN; ++j) WxAxTile<OP, 32, 256>::mma_slice(acc[j], w[d][j][0], w[d][j][1], x[d][0], x[d][1]);
      }
      __builtin_amdgcn_sched_barrier(0);
    };
    int kt = k0;
#pragma unroll 1
    for (; kt + kAhead < k1; kt += kAhead)
      static_for<kAhead>([&](auto dc) {
        landed(dc, std::integral_constant<int, (kAhead - 1) * kLoads>{});
        multiply(dc);
        const int kn = min(kt + kAhead + decltype(dc)::value, klast);
        load_w(dc, kn);
        load_x(dc, kn);
        __builtin_amdgcn_sched_barrier(0);
      });
    static_for<kAhead>([&](auto dc) {  // the last slices of the range
      constexpr int d = decltype(dc)::value;
      landed(dc, std::integral_constant<int, (kAhead - 1 - d) * kLoads>{});
      if (kt + d < k1) multiply(dc);
    });
    vm_wait_for<0>(sa_bits);
#pragma unroll
    for (int j = 0; j < FN; ++j) vm_wait_for<0>(sb_bits[j]);

    // the four waves' sums meet in LDS; wave q adds and stores channels 8 q + nq .. + 3 of every 32-channel block
    typedef decltype(acc[0][0] + acc[0][0]) Sum;
    typedef Sum v4s __attribute__((ext_vector_type(4)));
    v4s* red = reinterpret_cast<v4s*>(smem);
#pragma unroll
    for (int j = 0; j < FN; ++j)
#pragma unroll
      for (int q = 0; q < 4; ++q) red[((wave * FN + j) * 4 + q) * 64 + lane] = v4s{acc[j][4 * q], acc[j][4 * q + 1], acc[j][4 * q + 2], acc[j][4 * q + 3]};
    __syncthreads();
    const _Float16 sa_h = __builtin_bit_cast(_Float16, (unsigned short)sa_bits);
    const float s_a = (float)sa_h * (OP == Op::I4 ? 0.00390625f : 1.0f);  // (the int4 accumulator holds 256 * sum)
    v4h o[FN];
    const bool live = m0 + lrow < M;
#pragma unroll
    for (int j = 0; j < FN; ++j) {
      v4s sum = red[(j * 4 + wave) * 64 + lane];
#pragma unroll
      for (int v = 1; v < kWaves; ++v) sum += red[((v * FN + j) * 4 + wave) * 64 + lane];
      const v4h s_b = __builtin_bit_cast(v4h, sb_bits[j]);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float sc = s_a * (float)s_b[e];
        o[j][e] = (_Float16)keep_f32((float)sum[e] * sc);
      }
      if (!GU && t.acc_dump) {  // parity tests only
        const int n = n0 + j * 32 + wave * 8 + nq;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const Sum v = sum[e];
          const int a = __builtin_bit_cast(int, v);
          if (live && n < N) gstore<int>(t.acc_dump + (long)(m0 + lrow) * N + n + e, OP == Op::I4 ? a >> 8 : a);
        }
      }
    }
    if constexpr (GU) {
      v4h y;
#pragma unroll
      for (int e = 0; e < 4; ++e) y[e] = silu_mul_half(o[0][e], o[1][e]);
      const int n = n0 + wave * 8 + nq;
      if (live && n < N) gstore<v4h>(t.C + (long)(m0 + lrow) * N + n, y);
    } else {
#pragma unroll
      for (int j = 0; j < FN; ++j) {
        const int n = n0 + j * 32 + wave * 8 + nq;
        if (live && n < N) gstore<v4h>(t.C + (long)(m0 + lrow) * N + n, o[j]);
      }
    }
  }
};

}  // namespace mxmoe

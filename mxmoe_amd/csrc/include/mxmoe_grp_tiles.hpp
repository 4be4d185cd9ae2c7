// WxAxGTile: w4a4 with group-128 symmetric scales on both operands (w4a4_g128_sym).
//
// Every K slice of the int4 tiles is 128 values = one quantisation group, so the integer accumulators of a slice are complete
// per-group sums: after each slice they are converted, multiplied by the product of the token's and the channel's scale of that
// group and added to fp32 accumulators, groups in ascending order (the reference rescales each group's integer fragment into an
// fp32 fragment the same way, mxmoe/kernels/src/include/cta_gemm.cuh:613-772).
//
// Operands: activations int4 rows [M, K/2] with scales [M, K/128]; weights in MFMA fragment order as for w4a4 (mxmoe_tiles.hpp,
// WxAxTile) with scales stored group-major [K/128, N], so that the scales of a tile's channels for one group are contiguous.
// BM x 256 outputs per workgroup, 4 waves x 64 channels.  Activations go global -> registers -> LDS (3-stage ring, one barrier
// per slice), weights global -> registers one slice ahead, a group's scales global -> registers as soon as the last group's are used; every load is an
// ordinary load whose waits the compiler places.  Indices past the ends (rows past M, channel blocks past N, slices past K) are clamped
// to the last valid one: such results are computed and never stored.
//
// Bound: the vector ALU.  A 32 x 32 block of a slice is four matrix instructions (128 cycles of the matrix pipe) and, written out, 80 vector ones to rescale
// it (320 cycles), besides the widening of its operands.  The products of the scales, 32 of those 80, therefore come out of the matrix pipe too, which
// has the time: the outer product of 32 channel scales and 32 token scales is one more matrix instruction, exact (22 bits of product, everything else
// it adds is zero) and in the layout of the sums.  Every block is then 16 conversions, multiplications and additions, and the operands of the blocks to come
// are widened between the matrix instructions.  64 problems of N = 2816, K = 2048, weights from memory, us: 30 rows 65 -> 54, 192 rows 175 -> 151,
// 546 rows 431 -> 363.  (The order alone, blocks rescaled beside the next block's matrix instructions, changed nothing: the other wave of the SIMD fills the gaps.)
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "mxmoe_tiles.hpp"

namespace mxmoe {

template <int BM_>
struct WxAxGTile {
  static constexpr int BM = BM_, BN = 256, BK = 128;
  static constexpr int FM = BM / 32, FN = 2;
  static_assert(BM == 32 || BM == 64, "two sets of accumulators (int32 per group, fp32 running sum) must fit 256 registers");
  static constexpr int kStageBytes = BM * kRowBytes, kStages = 3;
  static constexpr int kLdsBytes = kStages * kStageBytes;
  static constexpr int kAccRegs = 2 * FM * FN * 16;
  static constexpr int kWavesWanted = 2;  // waves per SIMD a kernel of such tiles is compiled for
  static constexpr int kABits = 4, kWBits = 4;  // bits per activation / weight element
  static constexpr int kPieces = BM / 16;                       // 1 KB pieces (16 rows) of one activation slice
  static constexpr int kQ = (kPieces + kWaves - 1) / kWaves;    // pieces a wave copies per slice

  template <bool GU>
  __device__ static __forceinline__ void run(const TileArgs& t, uint8_t* __restrict__ smem) {
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int M = t.M, N = GU ? t.N / 2 : t.N;  // N: output channels (gate_up form: block 0 of a wave = gate, block 1 = up channels)
    const int G = t.K / 128;  // K slices = quantisation groups
    const long row_bytes = t.K / 2;
    const int m0 = t.row0 + t.tile_m * BM, n0 = t.tile_n * (GU ? BN / 2 : BN);
    const int lrow = lane & 31, nq = (lane >> 5) * 4;

    // ---- activations: global -> registers -> LDS ----
    auto row_of = [&](int m) {  // the stored row behind row m (clamped to the last valid one)
      if constexpr (GU) return gload<int>(t.rows + min(m, M - 1));
      else return min(m, M - 1);
    };
    const uint8_t* a_src[kQ];
    int a_lds[kQ];
    bool a_mine[kQ];
#pragma unroll
    for (int q = 0; q < kQ; ++q) {
      const int piece = wave + kWaves * q;
      a_mine[q] = piece < kPieces;
      const int row = (a_mine[q] ? piece : 0) * 16 + (lane >> 2);
      a_src[q] = t.A + (long)row_of(m0 + row) * row_bytes + (lane & 3) * 16;
      a_lds[q] = row * kRowBytes + (((lane & 3) ^ lds_swizzle(row)) << 4);
    }
    auto a_gload = [&](int kt, v4i (&r)[kQ]) {
#pragma unroll
      for (int q = 0; q < kQ; ++q) r[q] = gload<v4i>(a_src[q] + (long)min(kt, G - 1) * kRowBytes);
    };
    auto a_swrite = [&](int stage, const v4i (&r)[kQ]) {
#pragma unroll
      for (int q = 0; q < kQ; ++q)
        if (a_mine[q]) *reinterpret_cast<v4i*>(smem + stage * kStageBytes + a_lds[q]) = r[q];
    };
    const int fa = lrow * kRowBytes;
    const int sw = lds_swizzle(lrow);
    // ---- weights: fragment (block j, k-step s) of slice kt at ((nb * G + kt) * 2 + s) * 1 KB ----
    const int nblk = (N + 31) / 32;
    const uint8_t* bptr[FN];
#pragma unroll
    for (int j = 0; j < FN; ++j)
      bptr[j] = t.B + (long)(GU ? min(n0 / 32 + wave, nblk - 1) + j * nblk : min(n0 / 32 + wave * FN + j, nblk - 1)) * G * 2048 + lane * 16;
    auto b_gload = [&](int j, int s, int kt) { return gload<v4i>(bptr[j] + ((long)min(kt, G - 1) * 2 + s) * 1024); };

    // ---- scales of one group.  Their products come out of the matrix pipe in the layout of the sums: channel scales as a 32 x 16 operand with all but its
    // first column zero, token scales likewise, so a lane loads one of each per block (lanes 32 .. 63 hold columns 8 .. 15 and mask what they load)
    const _Float16* sa_ptr[FM];
#pragma unroll
    for (int i = 0; i < FM; ++i) sa_ptr[i] = t.sa + (long)row_of(m0 + i * 32 + lrow) * G;
    int sb_at[FN];
#pragma unroll
    for (int j = 0; j < FN; ++j) sb_at[j] = GU ? j * N + min(n0 + wave * 32 + lrow, N - 1) : min(n0 + wave * 64 + j * 32 + lrow, N - 1);
    const int first_column = lane < 32 ? 0xFFFF : 0;
    int sa_next[FM], sb_next[FN];  // of the next group, as bits
    auto s_load = [&](int kt) {
      const int g = min(kt, G - 1);
#pragma unroll
      for (int i = 0; i < FM; ++i) sa_next[i] = gload<unsigned short>(sa_ptr[i] + g);
#pragma unroll
      for (int j = 0; j < FN; ++j) sb_next[j] = gload<unsigned short>(t.sb + (long)g * t.N + sb_at[j]);
    };

    v16f facc[FM][FN];    // 256 times the outputs: the integer sums are of 16 * code products (int4 widened in place), a power of two either way
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int j = 0; j < FN; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r) facc[i][j][r] = 0.0f;

    v4i stg[kQ];          // activation slice kt+2 on its way to LDS
    v4i wb[FN][2];        // packed weight fragments, each loaded for the next slice when it has been widened for this one
    v4i pa[2];            // packed activation fragments of one block
    v4i aop[FM][2][2];    // operands of a slice: [block][k-step][low / high nibbles]
    v4i bop[FN][2][2];
    v4i sa_op[FM], sb_op[FN];
#pragma unroll
    for (int i = 0; i < FM; ++i) sa_op[i] = v4i{};
#pragma unroll
    for (int j = 0; j < FN; ++j) sb_op[j] = v4i{};

    // nibble n of a byte -> int8 holding 16 * signed(n): quarter x of a block's fragments
    auto widen = [](const v4i (&p)[2], v4i (&o)[2][2], int x) {
      if (x & 1) o[x >> 1][1] = p[x >> 1] & (int)0xF0F0F0F0;
      else o[x >> 1][0] = (p[x >> 1] << 4) & (int)0xF0F0F0F0;
    };
    auto a_sread = [&](int stage, int i) {
#pragma unroll
      for (int s = 0; s < 2; ++s)
        pa[s] = *reinterpret_cast<const v4i*>(smem + stage * kStageBytes + fa + i * 32 * kRowBytes + ((((lane >> 5) + 2 * s) ^ sw) << 4));
    };
    auto b_load = [&](int j, int kt) {
#pragma unroll
      for (int s = 0; s < 2; ++s) wb[j][s] = b_gload(j, s, kt);
    };

    a_gload(0, stg);
#pragma unroll
    for (int j = 0; j < FN; ++j) b_load(j, 0);
    s_load(0);
    a_swrite(0, stg);
    a_gload(1, stg);
    __syncthreads();
    a_sread(0, 0);
#pragma unroll
    for (int x = 0; x < 4; ++x) {
      widen(pa, aop[0], x);
      widen(wb[0], bop[0], x);
    }
    b_load(0, 1);

    constexpr int kBlocks = FM * FN;  // block b of a slice: token block b / FN, channel block b % FN
    int stage = 0;
#pragma unroll 1
    for (int kt = 0; kt < G; ++kt) {
      const int nstage = stage == kStages - 1 ? 0 : stage + 1;
#pragma unroll
      for (int i = 0; i < FM; ++i) sa_op[i][0] = sa_next[i] & first_column;
#pragma unroll
      for (int j = 0; j < FN; ++j) sb_op[j][0] = sb_next[j] & first_column;
      s_load(kt + 1);
      a_swrite(nstage, stg);  // slice kt+1, fetched during the previous slice
      a_gload(kt + 2, stg);
      static_for<kBlocks>([&](auto bc) {
        constexpr int b = decltype(bc)::value, i = b / FN, j = b % FN;
        if constexpr (b == 0 && FM == 2) a_sread(stage, 1);
        if constexpr (b == kBlocks - 2) {
          __syncthreads();  // slice kt+1 is in LDS for everybody (and everybody is done with the stage that slice kt+2 will overwrite)
          a_sread(nstage, 0);
        }
        const v16f sc = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(v8h, sb_op[j]), __builtin_bit_cast(v8h, sa_op[i]), v16f{}, 0, 0, 0);
        v16i c;
        // four matrix instructions, and the operands whose registers are free widened beside them
        static_for<4>([&](auto xc) {
          constexpr int x = decltype(xc)::value;
          if constexpr (x == 0) c = __builtin_amdgcn_mfma_i32_32x32x32_i8(bop[j][0][0], aop[i][0][0], v16i{}, 0, 0, 0);
          else c = __builtin_amdgcn_mfma_i32_32x32x32_i8(bop[j][x >> 1][x & 1], aop[i][x >> 1][x & 1], c, 0, 0, 0);
          if constexpr (b == 0) widen(wb[1], bop[1], x);
          if constexpr (FM == 2 && b == 1) widen(pa, aop[1], x);
          if constexpr (FM == 2 && b == 2) widen(pa, aop[0], x);
          __builtin_amdgcn_sched_barrier(0);
        });
        if constexpr (b == 0) b_load(1, kt + 1);
        if constexpr (b == kBlocks - 1) {
#pragma unroll
          for (int x = 0; x < 4; ++x) {
            if constexpr (FM == 1) widen(pa, aop[0], x);
            widen(wb[0], bop[0], x);
          }
          b_load(0, kt + 2);
        }
#pragma unroll
        for (int r = 0; r < 16; ++r) facc[i][j][r] = facc[i][j][r] + (float)c[r] * sc[r];
        __builtin_amdgcn_sched_barrier(0);
      });
      stage = nstage;
    }
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int j = 0; j < FN; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r) facc[i][j][r] *= 0.00390625f;  // exact

    // ---- epilogue: lane holds token lane & 31 and channels 8*(r/4) + 4*(lane >> 5) + (r & 3) of each 32 x 32 block ----
#pragma unroll
    for (int i = 0; i < FM; ++i) {
      const int m = m0 + i * 32 + lrow;
#pragma unroll
      for (int j = 0; j < (GU ? 1 : FN); ++j)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int n = n0 + wave * (GU ? 32 : 64) + j * 32 + q * 8 + nq;
          if (m < M && n < N) {
            v4h o;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              if constexpr (GU) o[e] = silu_mul_half((_Float16)facc[i][0][q * 4 + e], (_Float16)facc[i][1][q * 4 + e]);
              else o[e] = (_Float16)facc[i][j][q * 4 + e];
            }
            gstore(t.C + (long)m * N + n, o);
            if (!GU && t.acc_dump) {  // parity tests only: the fp32 sums as bit patterns
#pragma unroll
              for (int e = 0; e < 4; ++e) {
                const float f = facc[i][j][q * 4 + e];  // a copy: a bit cast applied to a vector element reads element 0
                gstore(t.acc_dump + (long)m * N + n + e, __float_as_int(f));
              }
            }
          }
        }
    }
  }
};

// The same problems with few rows: 16 tokens x 64 channels per workgroup, the groups dealt to the four waves one by one.  A round is four groups: a wave's integer sums of
// its group, times their scales, go to LDS, and behind the barrier wave q adds the four groups' products to its quarter of the outputs in group order, which is all that has to happen in
// order: the same additions as above, bit for bit.  Operands and scales stream straight into registers, kAhead rounds ahead; rows past M re-read the last one.
// Bound: the weights' bytes; with few problems the latency of a round, of which there are a quarter as many as groups, in four times the workgroups.  Layers of four formats, a third of the
// problems in this one, on narrow tiles but for these / with these too, us: eight experts of N = 28 672 / 4096, K = 4096 / 14 336 193 / 88 (1 token), 283 / 222 (8); 60 experts top-4 and a shared
// one 56 / 43, 81 / 75.
struct WxAxGNarrowTile {
  static constexpr int BM = 16, BN = 64, BK = 128, NB = BN / 16;
  static constexpr int kRoundBytes = kWaves * NB * 64 * 16;
  static constexpr int kLdsBytes = 2 * kRoundBytes;  // a round's products are read while the next one's are written
  static constexpr int kAccRegs = NB * 4 + 4;
  static constexpr int kWavesWanted = 2;
  static constexpr int kABits = 4, kWBits = 4;
  static constexpr int kAhead = 3;

  template <bool GU>
  __device__ static __forceinline__ void run(const TileArgs& t, uint8_t* __restrict__ smem) {
    run_rows<GU>(t, smem, [&](int m) {
      if constexpr (GU) return gload<int>(t.rows + m);
      else return m;
    });
  }
  // `row_of(m)`: the row of A (and of sa) behind row m of the problem.
  template <bool GU, class RowOf>
  __device__ static __forceinline__ void run_rows(const TileArgs& t, uint8_t* __restrict__ smem, RowOf&& row_of) {
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lm = lane & 15, lg = lane >> 4;
    const int M = t.M, N = GU ? t.N / 2 : t.N;  // N: output channels
    const int G = t.K / 128, rounds = (G + kWaves - 1) / kWaves;
    const int m0 = t.row0 + t.tile_m * BM, n0 = t.tile_n * (GU ? BN / 2 : BN);
    const int src = row_of(min(m0 + lm, M - 1));
    const uint8_t* const xp = t.A + (long)src * (t.K / 2) + lg * 16;
    const _Float16* const sa = t.sa + (long)src * G;
    // 16 channels of the tile: half of a 32-channel block of fragments, of which lane (lm, lg) takes the 16-byte piece lg of channel lm's 64 bytes of a slice
    const int nblk = (N + 31) / 32;
    const uint8_t* wp[NB];
    int ch[NB];  // first of the four channels whose products this lane gets
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      const int blk = GU ? min(n0 / 32, nblk - 1) + b / 2 * nblk : min(n0 / 32 + b / 2, nblk - 1);
      wp[b] = t.B + (long)blk * G * 2048 + (lg >> 1) * 1024 + ((lg & 1) * 32 + b % 2 * 16 + lm) * 16;
      ch[b] = GU ? b / 2 * N + min(n0 + b % 2 * 16 + lg * 4, N - 4) : min(n0 + b * 16 + lg * 4, N - 4);
    }
    v4i w[kAhead][NB], x[kAhead];
    v4h s_b[kAhead][NB];
    _Float16 s_a[kAhead];
    auto load = [&](auto dc, int round) {
      constexpr int d = decltype(dc)::value;
      const int g = min(round * kWaves + wave, G - 1);
#pragma unroll
      for (int b = 0; b < NB; ++b) w[d][b] = gload<v4i>(wp[b] + (long)g * 2048);
      x[d] = gload<v4i>(xp + (long)g * kRowBytes);
#pragma unroll
      for (int b = 0; b < NB; ++b) s_b[d][b] = gload<v4h>(t.sb + (long)g * t.N + ch[b]);
      s_a[d] = gload<_Float16>(sa + g);
    };
    static_for<kAhead>([&](auto dc) { load(dc, decltype(dc)::value); });
    __builtin_amdgcn_sched_barrier(0);

    v4f sum = {0.f, 0.f, 0.f, 0.f};  // 256 times this lane's outputs: channels 4 lg .. + 3 of 16-channel block `wave`, token lm
    auto multiply = [&](auto dc, int round) {
      constexpr int d = decltype(dc)::value;
      v4f* const out = reinterpret_cast<v4f*>(smem + (round & 1) * kRoundBytes);
      const v4i xl = (x[d] << 4) & (int)0xF0F0F0F0, xh = x[d] & (int)0xF0F0F0F0;  // int4 pairs widened to bytes holding 16 v
      const float a = (float)s_a[d];
#pragma unroll
      for (int b = 0; b < NB; ++b) {
        const v4i wl = (w[d][b] << 4) & (int)0xF0F0F0F0, wh = w[d][b] & (int)0xF0F0F0F0;
        v4i c = __builtin_amdgcn_mfma_i32_16x16x64_i8(wl, xl, v4i{}, 0, 0, 0);
        c = __builtin_amdgcn_mfma_i32_16x16x64_i8(wh, xh, c, 0, 0, 0);
        v4f p;
#pragma unroll
        for (int e = 0; e < 4; ++e) p[e] = (float)c[e] * (a * (float)s_b[d][b][e]);
        out[(wave * NB + b) * 64 + lane] = p;
      }
      __builtin_amdgcn_sched_barrier(0);
    };
    auto add = [&](int round) {
      const v4f* const in = reinterpret_cast<const v4f*>(smem + (round & 1) * kRoundBytes);
      v4f p[kWaves];
#pragma unroll
      for (int v = 0; v < kWaves; ++v) p[v] = in[(v * NB + wave) * 64 + lane];
#pragma unroll
      for (int v = 0; v < kWaves; ++v)
        if (round * kWaves + v < G) {
#pragma unroll
          for (int e = 0; e < 4; ++e) sum[e] = sum[e] + p[v][e];
        }
    };
#pragma unroll 1
    for (int r0 = 0; r0 < rounds; r0 += kAhead)
      static_for<kAhead>([&](auto dc) {
        const int round = r0 + decltype(dc)::value;
        if (round >= rounds) return;  // (uniform)
        multiply(dc, round);
        load(dc, round + kAhead);
        __builtin_amdgcn_sched_barrier(0);
        __syncthreads();  // (behind it nobody reads the products of the round before the last any more: the next round overwrites those)
        add(round);
      });
    v4h o;
#pragma unroll
    for (int e = 0; e < 4; ++e) o[e] = (_Float16)(sum[e] * 0.00390625f);  // exact
    const int m = m0 + lm;
    if constexpr (GU) {  // waves 0 and 1 hold gate channels, 2 and 3 the up channels of the same outputs
      v4h* const up = reinterpret_cast<v4h*>(smem);
      __syncthreads();
      if (wave >= 2) up[(wave - 2) * 64 + lane] = o;
      __syncthreads();
      if (wave < 2) {
        const v4h u = up[wave * 64 + lane];
#pragma unroll
        for (int e = 0; e < 4; ++e) o[e] = silu_mul_half(o[e], u[e]);
        const int n = n0 + wave * 16 + lg * 4;
        if (m < M && n < N) gstore<v4h>(t.C + (long)m * N + n, o);
      }
    } else {
      const int n = n0 + wave * 16 + lg * 4;
      if (m < M && n < N) {
        gstore<v4h>(t.C + (long)m * N + n, o);
        if (t.acc_dump) {  // parity tests only: the fp32 sums as bit patterns
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const float f = sum[e] * 0.00390625f;
            gstore<int>(t.acc_dump + (long)m * N + n + e, __float_as_int(f));
          }
        }
      }
    }
  }
};

}  // namespace mxmoe

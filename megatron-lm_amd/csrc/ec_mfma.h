// ec_mfma.h — GF(2^8) matrix-vector products on the matrix cores, for the
// codes past the unrolled VALU kernels (k > 16 or m > 4), shared by the flat
// (ec_flat.hip) and batched (ec_update.hip) kernels.
//
// Multiplication by a coefficient is linear over GF(2): output bit r of c * x
// is the parity of (row r of an 8 x 8 bit matrix of c) AND x.  An m x k code
// is an 8m x 8k bit matrix, and the parity bytes of one column of k bytes are
// the matrix's product with the column's 8k bits, each sum taken mod 2.  The
// products are 0 or 1 and the sums at most 8k <= 256, so the scaled fp4 MFMA
// (v_mfma_scale_f32_32x32x64_f8f6f4) computes them exactly.
//
//   Operands.  B is the data: a dword holding one byte of four shards at one
//   column becomes the 32 fp4 values of a lane with five VALU ops, because a
//   nibble of 1, 2 or 4 is the fp4 number 0.5, 1 or 2: three masks keep the
//   bits where they are, the top bit of each nibble is shifted down.  A holds
//   the reciprocal wherever the bit matrix has a one, so every product is 1.
//   Results.  The accumulators start at 2^23, so a sum's bits are the low
//   mantissa bits.  A's scale of row r is 2^r (its MX block scale, free) and
//   B's is 2^8 for odd byte columns, whose products go to the same
//   accumulator as the even ones: accumulator r then holds the parity bit of
//   two adjacent bytes at mantissa bits r and 8 + r, and seven bit selects
//   merge the eight accumulators of an output byte into two finished bytes
//   (3.75 VALU ops per output byte, against 8.75 with one byte each).  The
//   lower sum must stay below 2^8: PAIR = false keeps every column in its own
//   accumulator for the one matrix where it may not (a row of 256 ones, see
//   mfma_pair_ok).
//
// VALU ops per column of k bytes in and m out: 1.75 k + 3.75 m, against
// 1.125 k m + 1.25 k for the permute tables (RS(24,8): 72 against 246).
#pragma once

#include "ec_device.h"

namespace ec {
namespace {

typedef int v8i32 __attribute__((ext_vector_type(8)));
typedef float v16f32 __attribute__((ext_vector_type(16)));

constexpr int kFmtFp4 = 4;         // operand format selector of f8f6f4: e2m1
constexpr int kScaleOne = 127;     // E8M0 block scale 2^0

constexpr uint8_t cx_gf_mul(uint32_t a, uint32_t b) {
  uint32_t r = 0;
  for (int i = 0; i < 8; ++i) {
    if ((b >> i) & 1u) r ^= a << i;
  }
  for (int i = 14; i >= 8; --i)
    if ((r >> i) & 1u) r ^= 0x11Du << (i - 8);
  return (uint8_t)r;
}

// Row `bit` of the bit matrix of c: bit b is set when c * 2^b has bit `bit`.
constexpr uint8_t cx_bit_row(uint32_t c, int bit) {
  uint32_t w = 0;
  for (int b = 0; b < 8; ++b) w |= ((uint32_t)(cx_gf_mul(c, 1u << b) >> bit) & 1u) << b;
  return (uint8_t)w;
}

// cx_bit_row(., bit) is linear in c, so the permute tables of a multiply
// resolve it for four coefficients at once.
struct BitRowTabs {
  PermTab t[8];
};

constexpr BitRowTabs make_bit_row_tabs() {
  BitRowTabs r{};
  for (int bit = 0; bit < 8; ++bit) {
    uint32_t w[5] = {0, 0, 0, 0, 0};
    for (uint32_t a = 0; a < 8; ++a) {
      w[a >> 2] |= (uint32_t)cx_bit_row(a, bit) << (8 * (a & 3));
      w[2 + (a >> 2)] |= (uint32_t)cx_bit_row(a << 3, bit) << (8 * (a & 3));
    }
    for (uint32_t a = 0; a < 4; ++a) w[4] |= (uint32_t)cx_bit_row(a << 6, bit) << (8 * a);
    r.t[bit] = PermTab{w[0], w[1], w[2], w[3], w[4]};
  }
  return r;
}

__device__ const BitRowTabs g_bit_rows = make_bit_row_tabs();

// The kernels are instantiated for KH = ceil(k / 4) and MH = ceil(m / 2).  Lane
// half h of a wave holds shards 8 kt + 2 i + h (i < 4; i < 2 in the last group
// when KH is odd) and outputs 4 mt + 2 s + h (s < 2; s < 1 in the last tile
// when MH is odd), so what a code leaves unused of its last group or tile is
// left out of the loops as far as possible.
constexpr int mfma_groups(int kh) { return (kh + 1) / 2; }
constexpr int mfma_tiles(int mh) { return (mh + 1) / 2; }
constexpr int mfma_words(int kh, int kt) { return 2 * kt + 1 < kh ? 4 : 2; }   // i < this
constexpr int mfma_outs(int mh, int mt) { return 2 * mt + 1 < mh ? 2 : 1; }     // s < this

// The coefficients as the kernels take them: m rows padded to 32 bytes, zeros
// past k and m, each group of eight in the order of the lane halves (h, i).
struct MfmaCoeff {
  uint8_t c[EC_MAX_M][EC_MAX_K];
};

inline MfmaCoeff mfma_coeff(const uint8_t* coeff, int k, int m) {
  MfmaCoeff r{};
  for (int i = 0; i < m; ++i)
    for (int j = 0; j < k; ++j)
      r.c[i][(j & ~7) + 4 * (j & 1) + ((j & 7) >> 1)] = coeff[i * k + j];
  return r;
}

// Whether every sum of the code stays below 2^8, as PAIR needs: always for
// k < 32; for k = 32 unless some bit row is all ones, which takes 32 equal
// coefficients.
inline bool mfma_pair_ok(const uint8_t* coeff, int k, int m) {
  if (k * 8 < 256) return true;
  for (int i = 0; i < m; ++i) {
    bool equal = true, full = false;
    for (int j = 1; j < k; ++j) equal &= coeff[i * k + j] == coeff[i * k];
    for (int bit = 0; bit < 8; ++bit) full |= cx_bit_row(coeff[i * k], bit) == 0xff;
    if (equal && full) return false;
  }
  return true;
}

__device__ __forceinline__ v8i32 fp4_operand(uint32_t q0, uint32_t q1, uint32_t q2, uint32_t q3) {
  return v8i32{(int)q0, (int)q1, (int)q2, (int)q3, 0, 0, 0, 0};
}

// The code's bit matrix in the A layout (lane l: row l % 32 of each tile, K
// values 32 (l / 32) .. + 31).  Row order: the 16 accumulators of lane half h
// are the 8 bits of outputs h and 2 + h of the tile.  Up to kCodeRegs dwords
// stay in registers; larger codes are read from LDS at each use (RS(32,16):
// 16 KiB, half of the LDS rate at the full MFMA rate).
constexpr int kCodeRegs = 32;

template <int KH, int MH>
struct MfmaCode {
  static constexpr int KT = mfma_groups(KH), MT = mfma_tiles(MH);
  static constexpr bool kInLds = KT * MT * 4 > kCodeRegs;
  struct Lds {
    uint4 a[kInLds ? KT * MT : 1][64];
  };
  uint4 a[kInLds ? 1 : KT][kInLds ? 1 : MT];
  const uint4* lds;
  int row_scale;

  __device__ __forceinline__ v8i32 operand(int kt, int mt) const {
    const uint4 v = kInLds ? lds[(kt * MT + mt) * 64] : a[kInLds ? 0 : kt][kInLds ? 0 : mt];
    return fp4_operand(v.x, v.y, v.z, v.w);
  }

  // B lanes of a workgroup; with kInLds the caller has a barrier after it.
  template <int B>
  __device__ __forceinline__ void load(const MfmaCoeff& coeff, Lds& shared) {
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    const uint32_t row = lane & 31u, half = lane >> 5;
    const uint32_t r = (row & 3u) + 4u * (row >> 3);
    const uint32_t out = 2u * (r >> 3) + ((row >> 2) & 1u);
    const PermTab t = g_bit_rows.t[r & 7u];
    row_scale = kScaleOne + (int)(r & 7u);
    lds = &shared.a[0][lane];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int kt = 0; kt < KT; ++kt) {
        if (kInLds && (kt * MT + mt) % (B / 64) != (int)wave) continue;
        const uint32_t c = *reinterpret_cast<const uint32_t*>(
            &coeff.c[mt * kMfmaOutputs + out][kt * kMfmaShards + half * 4]);
        const uint32_t w = mac1(0u, t, fields(c));
        const uint4 v = make_uint4((w & 0x11111111u) << 2, w & 0x22222222u,
                                   (w & 0x44444444u) >> 2, (w >> 1) & 0x44444444u);
        if constexpr (kInLds) shared.a[kt * MT + mt][lane] = v;
        else a[kt][mt] = v;
      }
  }
};

__device__ __forceinline__ v8i32 fp4_bits(uint32_t w) {
  return fp4_operand(w & 0x11111111u, w & 0x22222222u, w & 0x44444444u, (w >> 3) & 0x11111111u);
}

// Eight accumulators (bits 0..7 of one output) into the low 16 bits: byte 0
// the parity bits of the even column, byte 1 those of the odd one.
__device__ __forceinline__ uint32_t merge_bits(const v16f32& acc, int first) {
  uint32_t r = __float_as_uint(acc[first]);
#pragma unroll
  for (int b = 1; b < 8; ++b)   // bits keep of the accumulator, the others of r
    r = __builtin_amdgcn_bitop3_b32(__float_as_uint(acc[first + b]), r, 0x101u << b, 0xe4);
  return r;
}

// Keeps what is computed from a after what was computed before the fence.
__device__ __forceinline__ void step_fence(uint32_t& a) { asm volatile("" : "+v"(a)); }

// t[kt][d][c]: byte column 4 d + c of the lane's shards of group kt, one byte
// per shard, from x[kt][i], 16 bytes of shard 8 kt + 2 i + h (h: the lane's
// half).
// With FENCE all of them are taken here, so that x's registers are free for
// other loads; without, the compiler takes each when it is used.
template <int KH, bool FENCE>
__device__ __forceinline__ void mfma_columns(uint32_t (&t)[mfma_groups(KH)][4][4],
                                             const uint4 (&x)[mfma_groups(KH)][4]) {
#pragma unroll
  for (int kt = 0; kt < mfma_groups(KH); ++kt)
#pragma unroll
    for (int d = 0; d < 4; ++d) {
      uint32_t(&o)[4] = t[kt][d];
      const uint32_t w0 = word(x[kt][0], d), w1 = word(x[kt][1], d);
      if (mfma_words(KH, kt) == 2) {
        o[0] = perm(w1, w0, 0x0c0c0400u);
        o[1] = perm(w1, w0, 0x0c0c0501u);
        o[2] = perm(w1, w0, 0x0c0c0602u);
        o[3] = perm(w1, w0, 0x0c0c0703u);
      } else {
        const uint32_t w2 = word(x[kt][2], d), w3 = word(x[kt][3], d);
        const uint32_t a01 = perm(w1, w0, 0x05010400u), a23 = perm(w3, w2, 0x05010400u);
        const uint32_t b01 = perm(w1, w0, 0x07030602u), b23 = perm(w3, w2, 0x07030602u);
        o[0] = perm(a23, a01, 0x05040100u);
        o[1] = perm(a23, a01, 0x07060302u);
        o[2] = perm(b23, b01, 0x05040100u);
        o[3] = perm(b23, b01, 0x07060302u);
      }
#pragma unroll
      for (int c = 0; c < 4; ++c)
        if (FENCE) step_fence(o[c]);
    }
}

// out[mt][s] = 16 bytes of output 4 mt + 2 s + h for the columns t of the
// lane's shards (mfma_columns).  Lanes l and l + 32 hold the same 16 byte
// columns of different shards.
// Two columns at a time: 16 MT accumulators, so that two or more waves fit a
// SIMD and one's bit selects run beside another's MFMAs.  step_fence orders
// the steps: without it the compiler starts them all at once (512 registers,
// or spills).
template <int KH, int MH, bool PAIR>
__device__ __forceinline__ void mfma_matvec16(uint4 (&out)[mfma_tiles(MH)][2],
                                              uint32_t (&t)[mfma_groups(KH)][4][4],
                                              const MfmaCode<KH, MH>& code) {
  constexpr int KT = mfma_groups(KH), MT = mfma_tiles(MH);
  constexpr int kAccs = PAIR ? 1 : 2;   // accumulator sets for two columns
  v16f32 base;
#pragma unroll
  for (int r = 0; r < 16; ++r) base[r] = 8388608.0f;
#pragma unroll
  for (int d = 0; d < 4; ++d) {
    uint32_t half[2][MT][2];   // two finished bytes of each output
#pragma unroll
    for (int q = 0; q < 2; ++q) {
#pragma unroll
      for (int kt = 0; kt < KT; ++kt) {
        step_fence(t[kt][d][2 * q]);
        step_fence(t[kt][d][2 * q + 1]);
      }
      v16f32 acc[MT][kAccs];
#pragma unroll
      for (int kt = 0; kt < KT; ++kt)
#pragma unroll
        for (int c = 0; c < 2; ++c) {
          const v8i32 b = fp4_bits(t[kt][d][2 * q + c]);
          const int w = PAIR ? 0 : c;
          const bool first = kt == 0 && (!PAIR || c == 0);
#pragma unroll
          for (int mt = 0; mt < MT; ++mt)
            acc[mt][w] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(
                code.operand(kt, mt), b, first ? base : acc[mt][w], kFmtFp4, kFmtFp4, 0,
                code.row_scale, 0, PAIR && c ? kScaleOne + 8 : kScaleOne);
        }
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int s = 0; s < mfma_outs(MH, mt); ++s) {
          const uint32_t lo = merge_bits(acc[mt][0], 8 * s);
          half[q][mt][s] =
              PAIR ? lo : perm(merge_bits(acc[mt][kAccs - 1], 8 * s), lo, 0x0c0c0400u);
          step_fence(half[q][mt][s]);
        }
    }
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int s = 0; s < mfma_outs(MH, mt); ++s) {
        const uint32_t v = perm(half[1][mt][s], half[0][mt][s], 0x05040100u);
        if (d == 0) out[mt][s].x = v;
        else if (d == 1) out[mt][s].y = v;
        else if (d == 2) out[mt][s].z = v;
        else out[mt][s].w = v;
      }
  }
}

}  // namespace
}  // namespace ec

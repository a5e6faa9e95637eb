// ec_update.hip — ec_parity_update (update_kernel of ec_update.h for
// k <= 16, m <= 4) and the batched kernels for wide codes
// (batched_core_kernel on the matrix cores; batched_wide_kernel and
// update_wide_kernel on permute tables, k at run time; up to
// EC_MAX_K x EC_MAX_M).  ec_batched.hip and ec_batched_copy.hip reach the first
// two through batched_wide(), ec_parity_update the third.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <array>
#include <utility>

#include "ec_device.h"
#include "ec_mfma.h"
#include "ec_update.h"

namespace ec {
namespace {

// --------------------------------------- batched kernels for wide codes --
// The batched encode/decode and the parity update for codes past the
// instantiated fast path (k > 16 or m > 4): k at run time, M a template
// parameter, one 16-byte chunk per lane (4 KiB tiles).  A workgroup stages
// its stripe's descriptors and the m x k tables in LDS; fast tiles issue the
// unit loads in groups of kWideGroup; tiles with unit ends or misaligned
// addresses take the units one at a time, with one unaligned load each at a
// clamped address (load_clip).  On views of one flat buffer that is as fast as
// the aligned tiles (300 tensors in 64 KiB units, us, aligned / views: RS(10,6)
// 398 / 388, RS(17,1) 241 / 223): enough waves run to hide the single load.

struct BatchWideArgs {
  const uint64_t* dptr;  // [n_stripes][k] (update: new units, 0 = unchanged)
  const uint32_t* dlen;  // [n_stripes][k]
  const uint64_t* optr;  // update: [n_stripes][k] old units; otherwise unused
  const uint64_t* pptr;  // [n_stripes][m]
  const uint32_t* olen;  // [n_stripes][m] valid output bytes, or null = whole units
  uint8_t coeff[EC_MAX_M * EC_MAX_K];  // row-major m x k
  uint32_t unit_bytes;
  uint32_t tiles_per_unit;
  uint32_t tiles_per_block;
  uint32_t blocks_per_unit;
  FastDiv by_blocks;  // division by blocks_per_unit
  int k;
};

template <int M>
struct WideStripe {
  PermTab tab[M * EC_MAX_K];
  const uint8_t* d[EC_MAX_K];
  const uint8_t* o[EC_MAX_K];
  uint32_t len[EC_MAX_K];
  uint8_t* p[M];
  uint32_t plen[M];
};

// Tables and stripe s's descriptors into LDS.  Returns, after a barrier,
// whether any unit or output address is not 16-byte aligned (uniform).
// Lanes 0..k-1 read the data descriptors, lanes 32..32+M-1 the parity ones
// (k <= 32, M <= 16): B >= 64.
template <int M, int B>
__device__ __forceinline__ bool stage_wide(WideStripe<M>& w, const BatchWideArgs& a, uint32_t s,
                                           bool update) {
  static_assert(B >= 64, "stage_wide needs lanes 0..47");
  const int k = a.k;
  const uint32_t t = threadIdx.x;
  for (uint32_t i = t; i < (uint32_t)(M * k); i += B) w.tab[i] = dev_perm_tab(a.coeff[i]);
  if (t < (uint32_t)k) {
    // Dense arrays: the length (and in an update the old unit's address) is
    // read together with the address, not after it.
    const uint8_t* d = reinterpret_cast<const uint8_t*>(a.dptr[(uint64_t)s * k + t]);
    const uint32_t dl = a.dlen[(uint64_t)s * k + t];
    const uint8_t* o0 = update ? reinterpret_cast<const uint8_t*>(a.optr[(uint64_t)s * k + t])
                               : nullptr;
    const uint32_t l = d ? dl : 0u;
    const uint8_t* o = d ? o0 : nullptr;
    w.d[t] = d;
    w.o[t] = o;
    w.len[t] = l < a.unit_bytes ? l : a.unit_bytes;
  } else if (t >= 32 && t < 32 + M) {
    const uint32_t i = t - 32;
    uint8_t* p = reinterpret_cast<uint8_t*>(a.pptr[(uint64_t)s * M + i]);
    const uint32_t l = p ? (a.olen ? a.olen[(uint64_t)s * M + i] : a.unit_bytes) : 0u;
    w.p[i] = p;
    w.plen[i] = l < a.unit_bytes ? l : a.unit_bytes;
  }
  __syncthreads();
  uintptr_t bits = 0;
  for (int j = 0; j < k; ++j)
    bits |= reinterpret_cast<uintptr_t>(w.d[j]) | reinterpret_cast<uintptr_t>(w.o[j]);
#pragma unroll
  for (int i = 0; i < M; ++i) bits |= reinterpret_cast<uintptr_t>(w.p[i]);
  return (bits & 15u) != 0;
}

template <int M>
__device__ __forceinline__ void wide_mac(uint32_t (&acc)[M][4], const uint4& x,
                                         const PermTab* col, int k) {
  Fields f[4];
#pragma unroll
  for (int dd = 0; dd < 4; ++dd) f[dd] = fields(word(x, dd));
#pragma unroll
  for (int i = 0; i < M; ++i) {
    asm volatile("" ::: "memory");
    const PermTab t = col[i * k];
#pragma unroll
    for (int dd = 0; dd < 4; ++dd) acc[i][dd] = mac1(acc[i][dd], t, f[dd]);
  }
}

template <int M, int B>
__global__ void __launch_bounds__(B) batched_wide_kernel(const BatchWideArgs a) {
  constexpr uint32_t kWideTile = B * 16u;
  __shared__ WideStripe<M> w;
  const uint32_t s = fast_div(blockIdx.x, a.by_blocks);
  const uint32_t t0 = (blockIdx.x - s * a.blocks_per_unit) * a.tiles_per_block;
  const uint32_t t1 = min(t0 + a.tiles_per_block, a.tiles_per_unit);
  const bool misaligned = stage_wide<M, B>(w, a, s, false);
  const int k = a.k;
  for (uint32_t t = t0; t < t1; ++t) {
    const uint32_t lo = t * kWideTile, hi = lo + kWideTile;
    uint32_t off = lo + threadIdx.x * 16u;
    bool edge = misaligned;
    for (int j = 0; j < k; ++j) edge |= w.len[j] > lo && w.len[j] < hi;
#pragma unroll
    for (int i = 0; i < M; ++i) edge |= w.plen[i] < hi;
    uint32_t acc[M][4] = {};
    if (!edge) {
      for (int j0 = 0; j0 < k; j0 += kWideGroup) {
        uint4 x[kWideGroup];
#pragma unroll
        for (int g = 0; g < kWideGroup; ++g) {
          const int j = j0 + g;
          x[g] = j < k && w.len[j] >= hi ? load_stream(w.d[j] + off) : make_uint4(0, 0, 0, 0);
        }
#pragma unroll
        for (int g = 0; g < kWideGroup; ++g) {
          if (j0 + g >= k) break;
          wide_mac<M>(acc, x[g], &w.tab[j0 + g], k);
        }
      }
#pragma unroll
      for (int i = 0; i < M; ++i)
        store_stream(w.p[i] + off, make_uint4(acc[i][0], acc[i][1], acc[i][2], acc[i][3]));
    } else {
      // Within the other path's registers: with this one's values computed ahead
      // of the branch and all its addresses read together RS(10,6) took 93, five
      // waves per SIMD instead of six (64 KiB units, 400 us against 386).
      asm volatile("" : "+v"(off));
      if (off >= a.unit_bytes) continue;
#pragma unroll 1
      for (int j = 0; j < k; ++j) {
        if (off >= w.len[j]) continue;
        wide_mac<M>(acc, load_clip(w.d[j], off, w.len[j]), &w.tab[j], k);
      }
#pragma unroll
      for (int i = 0; i < M; ++i) {
        asm volatile("" ::: "memory");   // each address right before its use
        store_clip(w.p[i], off, w.plen[i],
                   make_uint4(acc[i][0], acc[i][1], acc[i][2], acc[i][3]));
      }
    }
  }
}

// parity[s][i] ^= C[i][j] * (new[s][j] ^ old[s][j]) for the changed units.
template <int M, int B>
__global__ void __launch_bounds__(B) update_wide_kernel(const BatchWideArgs a) {
  constexpr uint32_t kWideTile = B * 16u;
  __shared__ WideStripe<M> w;
  const uint32_t s = fast_div(blockIdx.x, a.by_blocks);
  const uint32_t t0 = (blockIdx.x - s * a.blocks_per_unit) * a.tiles_per_block;
  const uint32_t t1 = min(t0 + a.tiles_per_block, a.tiles_per_unit);
  stage_wide<M, B>(w, a, s, true);
  const int k = a.k;
  uint32_t longest = 0;   // past the longest changed unit the delta is zero
  for (int j = 0; j < k; ++j) longest = w.len[j] > longest ? w.len[j] : longest;
  for (uint32_t t = t0; t < t1; ++t) {
    const uint32_t off = t * kWideTile + threadIdx.x * 16u;
    if (off >= longest) continue;
    // The products go on top of the parity itself, loaded first: with registers
    // of their own for both m = 16 took 200, two waves per SIMD instead of five
    // (RS(32,16) 1 % update in 1 MiB units 147 us against 132).
    uint32_t acc[M][4];
#pragma unroll
    for (int i = 0; i < M; ++i) {
      const uint4 v = load_any(w.p[i] + off);
#pragma unroll
      for (int dd = 0; dd < 4; ++dd) acc[i][dd] = word(v, dd);
    }
#pragma unroll 1
    for (int j = 0; j < k; ++j) {
      if (w.d[j] == nullptr || off >= w.len[j]) continue;  // unchanged unit, or past its end
      const uint4 vn = load_clip(w.d[j], off, w.len[j]);
      const uint4 vo = load_clip(w.o[j], off, w.len[j]);
      wide_mac<M>(acc, make_uint4(vn.x ^ vo.x, vn.y ^ vo.y, vn.z ^ vo.z, vn.w ^ vo.w),
                  &w.tab[j], k);
    }
    asm volatile("" ::: "memory");   // the addresses are read again
#pragma unroll
    for (int i = 0; i < M; ++i)
      store_any(w.p[i] + off, make_uint4(acc[i][0], acc[i][1], acc[i][2], acc[i][3]));
  }
}

// The encode and decode of wide codes on the matrix cores (ec_mfma.h): a wave
// codes 512 bytes of every unit of a stripe per step, lane l and lane l + 32
// the same columns of the even and the odd units.  A workgroup stages its
// stripe's descriptors in LDS once for the steps it walks.  Units and outputs
// at any address and of any length take the same path: a unit is read at
// clamped addresses and the chunk that holds its end shifted into place.
struct BatchCoreArgs {
  const uint64_t* dptr;  // [n_stripes][k]
  const uint32_t* dlen;  // [n_stripes][k]
  const uint64_t* pptr;  // [n_stripes][m]
  const uint32_t* olen;  // [n_stripes][m] valid output bytes, or null = whole units
  MfmaCoeff coeff;
  uint32_t unit_bytes;
  uint32_t steps_per_unit;   // ceil(unit_bytes / 512)
  uint32_t steps_per_block;  // consecutive steps one workgroup walks
  uint32_t blocks_per_unit;
  FastDiv by_blocks;         // division by blocks_per_unit
  int k, m;
};

constexpr uint32_t kCoreStep = 512;   // bytes of each unit per wave and step

template <int KH, int MH>
struct CoreLds {
  const uint8_t* d[EC_MAX_K];
  uint32_t len[EC_MAX_K];
  uint8_t* p[EC_MAX_M];
  uint32_t plen[EC_MAX_M];
  typename MfmaCode<KH, MH>::Lds code;
};

template <int KH, int MH, bool PAIR>
__global__ void __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(2)))
batched_core_kernel(const BatchCoreArgs a) {
  constexpr int KT = mfma_groups(KH), MT = mfma_tiles(MH);
  constexpr uint32_t kWaves = kBlock / 64;
  __shared__ CoreLds<KH, MH> w;
  const uint32_t s = fast_div(blockIdx.x, a.by_blocks);
  const uint32_t s0 = (blockIdx.x - s * a.blocks_per_unit) * a.steps_per_block;
  const uint32_t s1 = min(s0 + a.steps_per_block, a.steps_per_unit);
  const uint32_t t = threadIdx.x;
  if (t < EC_MAX_K) {
    const bool in = (int)t < a.k;
    const uint64_t d = in ? a.dptr[(uint64_t)s * a.k + t] : 0u;
    const uint32_t l = in ? a.dlen[(uint64_t)s * a.k + t] : 0u;
    w.d[t] = reinterpret_cast<const uint8_t*>(d);
    w.len[t] = d ? (l < a.unit_bytes ? l : a.unit_bytes) : 0u;
  } else if (t >= 64 && t < 64 + EC_MAX_M) {
    const uint32_t i = t - 64;
    const bool in = (int)i < a.m;
    const uint64_t q = in ? a.pptr[(uint64_t)s * a.m + i] : 0u;
    const uint32_t l = !in ? 0u : a.olen ? a.olen[(uint64_t)s * a.m + i] : a.unit_bytes;
    w.p[i] = reinterpret_cast<uint8_t*>(q);
    w.plen[i] = q ? (l < a.unit_bytes ? l : a.unit_bytes) : 0u;
  }
  MfmaCode<KH, MH> code;
  code.template load<kBlock>(a.coeff, w.code);
  __syncthreads();
  const uint32_t lane = t & 63u, half = lane >> 5;
  for (uint32_t step = s0 + __builtin_amdgcn_readfirstlane(t >> 6); step < s1; step += kWaves) {
    const uint32_t lo = step * kCoreStep, off = lo + (lane & 31u) * 16u;
    uint4 x[KT][4];
#pragma unroll
    for (int kt = 0; kt < KT; ++kt)
#pragma unroll
      for (int i = 0; i < mfma_words(KH, kt); ++i) {
        const uint32_t j = 8 * kt + 2 * i + half;
        const uint32_t l = w.len[j];
        x[kt][i] = load_any(l > lo ? clip_address(w.d[j], off, l) : g_zeros);
      }
#pragma unroll
    for (int kt = 0; kt < KT; ++kt)
#pragma unroll
      for (int i = 0; i < mfma_words(KH, kt); ++i) {
        const uint32_t j = 8 * kt + 2 * i + half;
        const uint32_t l = w.len[j];
        if (l > lo && l < lo + kCoreStep)
          x[kt][i] = l >= 16u ? clip_chunk(x[kt][i], off, l)
                     : off < l ? load_short(w.d[j], l) : x[kt][i];
      }
    uint32_t c[KT][4][4];
    mfma_columns<KH, false>(c, x);
    uint4 out[MT][2];
    mfma_matvec16<KH, MH, PAIR>(out, c, code);
    asm volatile("" ::: "memory");   // the descriptors stay in LDS
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int q = 0; q < mfma_outs(MH, mt); ++q) {
        const uint32_t o = 4 * mt + 2 * q + half;
        store_clip(w.p[o], off, w.plen[o], out[mt][q]);
      }
  }
}

template <int KH, int MH>
int launch_core(const uint8_t* coeff, int k, int m, const uint64_t* dptr, const uint32_t* dlen,
                const uint64_t* pptr, const uint32_t* olen, uint32_t n_stripes,
                uint32_t unit_bytes, hipStream_t st) {
  BatchCoreArgs a;
  a.dptr = dptr;
  a.dlen = dlen;
  a.pptr = pptr;
  a.olen = olen;
  a.coeff = mfma_coeff(coeff, k, m);
  a.k = k;
  a.m = m;
  a.unit_bytes = unit_bytes;
  a.steps_per_unit = (unit_bytes + kCoreStep - 1) / kCoreStep;
  // Spans of span_bytes per workgroup, shorter where fewer than 2048
  // workgroups would be left, a step per wave at least.
  const uint64_t total = (uint64_t)n_stripes * a.steps_per_unit;
  uint64_t spb = span_bytes(unit_bytes) / kCoreStep;
  if (total / spb < 2048) spb = total / 2048;
  if (spb < kBlock / 64) spb = kBlock / 64;
  if (spb > a.steps_per_unit) spb = a.steps_per_unit;
  a.steps_per_block = (uint32_t)spb;
  a.blocks_per_unit = (a.steps_per_unit + a.steps_per_block - 1) / a.steps_per_block;
  a.by_blocks = make_fastdiv(a.blocks_per_unit);
  if ((uint64_t)n_stripes * a.blocks_per_unit > 0x7fffffffull) return EC_ERANGE;
  bool pair = true;
  if constexpr (KH == EC_MAX_K / 4) pair = mfma_pair_ok(coeff, k, m);
  // As many launches as the grid's limit asks for (units of a few bytes: one
  // launch holds 2^24 stripes).
  const uint32_t most = (uint32_t)(max_grid(kBlock) / a.blocks_per_unit);
  for (uint32_t left = n_stripes; left != 0;) {
    const uint32_t n = left < most ? left : most;
    const dim3 grid(n * a.blocks_per_unit), block(kBlock);
    if (pair)
      hipLaunchKernelGGL((batched_core_kernel<KH, MH, true>), grid, block, 0, st, a);
    else if constexpr (KH == EC_MAX_K / 4)
      hipLaunchKernelGGL((batched_core_kernel<KH, MH, false>), grid, block, 0, st, a);
    left -= n;
    a.dptr += (uint64_t)n * k;
    a.dlen += (uint64_t)n * k;
    a.pptr += (uint64_t)n * m;
    if (a.olen) a.olen += (uint64_t)n * m;
  }
  return hip_status();
}

using CoreFn = int (*)(const uint8_t*, int, int, const uint64_t*, const uint32_t*,
                       const uint64_t*, const uint32_t*, uint32_t, uint32_t, hipStream_t);
template <int KH, int MH>
constexpr CoreFn core_entry() {
  if constexpr (core_reached(KH, MH)) return &launch_core<KH, MH>;
  else return nullptr;
}
template <int KH, int... Ms>
constexpr auto core_row(std::integer_sequence<int, Ms...>) {
  return std::array<CoreFn, sizeof...(Ms)>{core_entry<KH, Ms + 1>()...};
}
template <int... Ks>
constexpr auto core_table(std::integer_sequence<int, Ks...>) {
  return std::array<std::array<CoreFn, EC_MAX_M / 2>, sizeof...(Ks)>{
      core_row<Ks + 1>(std::make_integer_sequence<int, EC_MAX_M / 2>{})...};
}
const auto kCoreTable = core_table(std::make_integer_sequence<int, EC_MAX_K / 4>{});

// The update's launch shape (update_kernel in ec_update.h): lanes per
// workgroup, 16-byte chunks per lane, and log2 of the interleaved slices of
// the grid (0: launch order).  Measured on MI355X for config 5's 1 % update
// (RS(12,4), 3,152 changed 64 KiB units in 2,993 stripes, 1.98 GB of
// traffic), microseconds per launch by lanes x chunks and slices 1 / 8:
//   256 x 1  322.8 / 311.3     256 x 2  331.6 / 322.0     256 x 4  328.4 / 324.5
//   128 x 1  331.5 / 309.7     128 x 2  331.0 / 319.6
//    64 x 1  311.3 / 308.6      64 x 2  365.4 / 320.2      64 x 4  334.1 / 324.5
// and 64 x 1 over 4 / 16 / 32 slices 307.2 / 314.0 / 315.8: one wavefront on
// a 1 KiB tile in 4 slices, 0.806 of the HBM roofline against 0.767 for the
// former 256 x 1 in launch order.  More chunks per lane (more loads in
// flight per lane, fewer workgroups) lost everywhere.
constexpr int kUpdateBlock = 64;
constexpr int kUpdateChunks = 1;
constexpr uint32_t kUpdateSliceShift = 2;

template <int K, int M>
int update_fast(const uint8_t* coeff, const uint64_t* nptr, const uint64_t* optr,
                const uint32_t* len, const uint64_t* pptr, uint32_t n_stripes,
                uint32_t unit_bytes, hipStream_t st) {
  return launch_update<K, M, kUpdateBlock, kUpdateChunks>(coeff, nptr, optr, len, pptr, n_stripes,
                                                          unit_bytes, kUpdateSliceShift, st);
}

// Wide codes through the batched kernels: encode / decode (update = false,
// optr unused) or the parity update, with B-lane workgroups on B * 16-byte
// tiles: the encode walks spans of `span` bytes (0: span_bytes()) keeping at
// least 2048 workgroups, the update one tile per workgroup.
// span: bytes of each unit that a workgroup walks (0: span_bytes).
template <int M, int B, bool UPDATE>
int launch_batched_wide_b(const uint8_t* coeff, int k, const uint64_t* dptr, const uint32_t* dlen,
                          const uint64_t* optr, const uint64_t* pptr, const uint32_t* olen,
                          uint32_t n_stripes, uint32_t unit_bytes, hipStream_t st,
                          uint32_t span) {
  BatchWideArgs a;
  a.dptr = dptr;
  a.dlen = dlen;
  a.optr = optr;
  a.pptr = pptr;
  a.olen = olen;
  for (int t = 0; t < M * k; ++t) a.coeff[t] = coeff[t];
  a.k = k;
  a.unit_bytes = unit_bytes;
  a.tiles_per_unit = (unit_bytes / 16u + B - 1) / B;
  const uint64_t total_tiles = (uint64_t)n_stripes * a.tiles_per_unit;
  uint64_t tpb = 1;
  if (!UPDATE) {
    tpb = (span ? span : span_bytes(unit_bytes)) / (B * 16u);
    if (tpb < 1) tpb = 1;
    if (total_tiles / tpb < 2048) tpb = total_tiles / 2048;
  } else {
    tpb = (total_tiles + 0x3fffffffull) >> 30;
  }
  if (tpb < 1) tpb = 1;
  if (tpb > a.tiles_per_unit) tpb = a.tiles_per_unit;
  a.tiles_per_block = (uint32_t)tpb;
  a.blocks_per_unit = (a.tiles_per_unit + a.tiles_per_block - 1) / a.tiles_per_block;
  a.by_blocks = make_fastdiv(a.blocks_per_unit);
  const uint64_t blocks = (uint64_t)n_stripes * a.blocks_per_unit;
  if (blocks > 0x7fffffffull) return EC_ERANGE;
  if constexpr (UPDATE)
    hipLaunchKernelGGL((update_wide_kernel<M, B>), dim3((unsigned)blocks), dim3(B), 0, st, a);
  else
    hipLaunchKernelGGL((batched_wide_kernel<M, B>), dim3((unsigned)blocks), dim3(B), 0, st, a);
  return hip_status();
}

// Encode and decode with m <= 4 run one-wavefront workgroups on one 1 KiB
// tile each, like the fixed-size batched kernel; wider outputs and the update
// keep 256-lane workgroups.  Both keep launch order for every unit size:
// the fixed-size kernel's 8 slices for large units (SpanGrid) gained nothing
// here and cost up to 11 %.  Measured on MI355X when all wide codes ran on these
// tables (HBM traffic, GB/s, 8 GiB buffers; of these codes only decodes of one
// to three positions still do): one wavefront against 256 lanes with m = 4,
// RS(20,4) over 4 MiB units, encode 5041 -> 5314, decode 4886 -> 5136; with
// m >= 6 the per-workgroup table build (m * k tables) made one-wavefront
// workgroups 5 % slower (RS(16,6) over 64 KiB units 4995 -> 4747).
template <int M>
int launch_batched_wide(const uint8_t* coeff, int k, const uint64_t* dptr, const uint32_t* dlen,
                        const uint64_t* pptr, const uint32_t* olen, uint32_t n_stripes,
                        uint32_t unit_bytes, hipStream_t st) {
  constexpr int B = M <= 4 ? 64 : kBlock;
  return launch_batched_wide_b<M, B, false>(coeff, k, dptr, dlen, nullptr, pptr, olen, n_stripes,
                                            unit_bytes, st, M <= 4 ? B * 16 : 0);
}

template <int M>
int launch_update_wide(const uint8_t* coeff, int k, const uint64_t* nptr, const uint64_t* optr,
                       const uint32_t* len, const uint64_t* pptr, uint32_t n_stripes,
                       uint32_t unit_bytes, hipStream_t st) {
  return launch_batched_wide_b<M, kBlock, true>(coeff, k, nptr, len, optr, pptr, nullptr,
                                                n_stripes, unit_bytes, st, 0);
}

using UpdFn = int (*)(const uint8_t*, const uint64_t*, const uint64_t*, const uint32_t*,
                      const uint64_t*, uint32_t, uint32_t, hipStream_t);

template <int K, int... Ms>
constexpr auto upd_row(std::integer_sequence<int, Ms...>) {
  return std::array<UpdFn, sizeof...(Ms)>{&update_fast<K, Ms + 1>...};
}
template <int... Ks>
constexpr auto upd_table(std::integer_sequence<int, Ks...>) {
  return std::array<std::array<UpdFn, kFastMaxM>, sizeof...(Ks)>{
      upd_row<Ks + 1>(std::make_integer_sequence<int, kFastMaxM>{})...};
}
const auto kUpdTable = upd_table(std::make_integer_sequence<int, kFastMaxK>{});
using BatchWideFn = int (*)(const uint8_t*, int, const uint64_t*, const uint32_t*,
                            const uint64_t*, const uint32_t*, uint32_t, uint32_t, hipStream_t);
template <int M>
constexpr BatchWideFn batch_wide_entry() {
  if constexpr (batch_table_reached(M)) return &launch_batched_wide<M>;
  else return nullptr;
}
using UpdWideFn = int (*)(const uint8_t*, int, const uint64_t*, const uint64_t*, const uint32_t*,
                          const uint64_t*, uint32_t, uint32_t, hipStream_t);
template <int... Ms>
constexpr auto batch_wide_table(std::integer_sequence<int, Ms...>) {
  return std::array<BatchWideFn, sizeof...(Ms)>{batch_wide_entry<Ms + 1>()...};
}
template <int... Ms>
constexpr auto upd_wide_table(std::integer_sequence<int, Ms...>) {
  return std::array<UpdWideFn, sizeof...(Ms)>{&launch_update_wide<Ms + 1>...};
}
const auto kBatchWideTable = batch_wide_table(std::make_integer_sequence<int, EC_MAX_M>{});
const auto kUpdWideTable = upd_wide_table(std::make_integer_sequence<int, EC_MAX_M>{});

}  // namespace

int batched_wide(int k, int m, const uint8_t* coeff, const uint64_t* dptr, const uint32_t* dlen,
                 const uint64_t* pptr, const uint32_t* olen, uint32_t n_stripes,
                 uint32_t unit_bytes, hipStream_t st) {
  if (m < 1 || m > EC_MAX_M || k < 1 || k > EC_MAX_K || fast_shape(k, m)) return EC_ERANGE;
  if (batch_tables(k, m, (uint64_t)n_stripes * unit_bytes))
    return kBatchWideTable[m - 1](coeff, k, dptr, dlen, pptr, olen, n_stripes, unit_bytes, st);
  return kCoreTable[(k - 1) / 4][(m - 1) / 2](coeff, k, m, dptr, dlen, pptr, olen, n_stripes,
                                              unit_bytes, st);
}

}  // namespace ec

extern "C" {

int ec_parity_update(const uint8_t* coeff, int k, int m, const uint64_t* d_new_ptrs,
                     const uint64_t* d_old_ptrs, const uint32_t* d_len,
                     const uint64_t* d_parity_ptrs, uint32_t n_stripes, uint32_t unit_bytes,
                     ec_stream_t stream) {
  int s = ec::check_batch(coeff, k, m, d_new_ptrs, d_old_ptrs, d_parity_ptrs, unit_bytes);
  if (s != EC_OK) return s;
  if (!d_len) return EC_EINVAL;
  if (n_stripes == 0) return EC_OK;
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  if (!ec::fast_shape(k, m))
    return ec::kUpdWideTable[m - 1](coeff, k, d_new_ptrs, d_old_ptrs, d_len, d_parity_ptrs,
                                    n_stripes, unit_bytes, st);
  return ec::kUpdTable[k - 1][m - 1](coeff, d_new_ptrs, d_old_ptrs, d_len, d_parity_ptrs,
                                     n_stripes, unit_bytes, st);
}

}  // extern "C"

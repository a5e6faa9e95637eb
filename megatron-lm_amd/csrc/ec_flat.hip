// ec_flat.hip — the flat-shard kernels and entry points of the C ABI:
// ec_xor_encode, ec_rs_encode, ec_rs_decode (k equal-size shards in, m out),
// and ec_stream_create / ec_stream_destroy.  Helpers, the GF multiply and
// the streaming accesses are in ec_device.h.
#include <hip/hip_ext.h>
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <array>
#include <utility>
#include <vector>

#include "ec_device.h"
#include "ec_mfma.h"

namespace ec {
namespace {

// ------------------------------------------------ fast matrix-vector kernel --
// parity_i = XOR_j C[i][j] * data_j over n16 16-byte chunks; all pointers
// 16-byte aligned.  Encode and decode both run this kernel (decode with the
// host-inverted rows over the survivors).

template <int K, int M>
struct RsArgs {
  const uint8_t* data[K];
  uint8_t* out[M];
  PermTab tab[M][K];
  uint64_t n16;
};

// Lanes per workgroup of the flat kernels: one wavefront for the small codes
// (tables in registers, k * m <= 20), two for the wider ones, with
// workgroups in launch order: workgroup b streams 1 or 2 KiB of every shard
// at column b * BLOCK, and the round-robin dispatch over the 8 XCDs deals
// consecutive 1-2 KiB columns to different XCDs.  Measured on MI355X over
// 256 MiB shards (HBM traffic, GB/s; the former 256-lane workgroups that
// streamed each shard at two places half a shard apart first): RS(6,3) 5887 -> 6404 (one wave),
// 6309 (two waves); RS(8,2) 5900 -> 6319 / 6381; RS(4,1) 5942 -> 6347 /
// 6377; RS(12,4) 5687 -> 6087 / 6253; RS(16,4) over 128 MiB 6116 -> 6291 /
// 6335.  RS(6,3) with one wave over 64 MiB to 1 GiB shards: 6393-6547
// (5657-6097 before).  Smaller workgroups also made the rate less dependent
// on the box: the 256-lane kernel ran RS(6,3) at 393 to 424 us per launch on
// three boxes, the 64/128-lane ones at 376 to 386.  The two-window order lost
// with them (RS(6,3) one wave: 6202 vs 6404 at 256 MiB), and so did
// interleaved slices, workgroup b taking column (b mod 2^s) * ceil(n / 2^s) +
// b / 2^s (RS(6,3) over 6 x 256 MiB, us per launch, one box: launch order
// 373, 8 slices, one per XCD, 378-381, 32 slices 406, 256 slices 447).
template <int K, int M>
constexpr int flat_block() {
  return K * M <= 20 ? 64 : 128;
}

// Three forms of the same kernel, chosen per code by flat_form:
//  - kFormLanes: a per-lane grid-stride loop over 16-byte chunks, global nt
//    loads and stores (each lane computes its own 64-bit addresses);
//  - kFormPass: workgroup b codes the B chunks at chunk b * B of every shard
//    in one pass, global nt loads and stores on a wave-uniform base (kernel
//    argument plus b * B * 16, a scalar) plus the lane's 16-byte offset;
//  - kFormPassSc1: the same with nt+sc1 buffer stores on that base
//    (store_wave).
// The pass forms cover shards up to 16 GiB in one grid (grid_of); PASSES
// adds a wave-uniform grid-stride loop for larger ones (the loop costs
// 0.5-1 % where it is not needed: RS(6,3) over 6 x 256 MiB 372.9 us
// loop-free against 376.3 with the loop).
enum FlatForm : int { kFormLanes = 0, kFormPass = 1, kFormPassSc1 = 2 };

// Every shape with k <= 16, m <= 4 was timed in all three forms over 128 MiB
// shards on two boxes (HIP events, 3 interleaved rounds each).  A pass form
// is used where it beat kFormLanes by at least 0.5 % on the mean of both
// boxes (time relative to kFormLanes):
//   kFormPassSc1: RS(1,1) 0.981, RS(1,2) 0.972, RS(1,3) 0.988, RS(4,3) 0.991,
//                 RS(4,4) 0.984, RS(5,3) 0.993, RS(6,3) 0.992
//   kFormPass:    RS(1,4) 0.982, RS(4,1) 0.988, RS(7,2) 0.982, RS(12,1) 0.993,
//                 RS(13,1) 0.989, RS(16,1) 0.960
// kFormLanes was ahead for most codes with k >= 7 (by up to 3-4 %: RS(10,3)
// 1.022 / 1.041 for the pass forms, RS(9,2) 1.025 / 1.029), and the rest lie
// within 0.5 %.  The headline shape, RS(6,3) over 6 x 256 MiB, on one box:
// 375.9 us in the former library (kFormLanes) against 371.2 in this one
// (kFormPassSc1).
template <int K, int M>
constexpr int flat_form() {
  constexpr int kSc1[][2] = {{1, 1}, {1, 2}, {1, 3}, {4, 3}, {4, 4}, {5, 3}, {6, 3}};
  constexpr int kPass[][2] = {{1, 4}, {4, 1}, {7, 2}, {12, 1}, {13, 1}, {16, 1}};
  for (const auto& p : kSc1)
    if (p[0] == K && p[1] == M) return kFormPassSc1;
  for (const auto& p : kPass)
    if (p[0] == K && p[1] == M) return kFormPass;
  return kFormLanes;
}

template <int K, int M, int FORM, bool PASSES>
__global__ void __launch_bounds__((flat_block<K, M>())) rs_kernel(const RsArgs<K, M> a) {
  constexpr int B = flat_block<K, M>();
  __shared__ PermTab tab[M][K];
  {
    // M * K <= 64 tables: one per lane of the first B lanes, looped for
    // B = 64 < M * K
    for (int q = threadIdx.x; q < M * K; q += B) tab[q / K][q % K] = a.tab[q / K][q % K];
    __syncthreads();
  }
  if constexpr (FORM == kFormLanes) {
    const uint64_t stride = (uint64_t)gridDim.x * B;
    for (uint64_t idx = (uint64_t)blockIdx.x * B + threadIdx.x; idx < a.n16; idx += stride) {
      uint4 x[K];
#pragma unroll
      for (int j = 0; j < K; ++j) x[j] = load_stream(a.data[j] + idx * 16);
      uint32_t acc[M][4] = {};
      gf_matvec16<K, M>(acc, x, tab);
#pragma unroll
      for (int i = 0; i < M; ++i)
        store_stream(a.out[i] + idx * 16, make_uint4(acc[i][0], acc[i][1], acc[i][2], acc[i][3]));
    }
  } else {
    const uint64_t stride = PASSES ? (uint64_t)gridDim.x * B : 0;
    for (uint64_t base = (uint64_t)blockIdx.x * B; base < a.n16; base += stride) {
      if (base + threadIdx.x < a.n16) {
        const uint32_t lane = threadIdx.x * 16u;
        uint4 x[K];
#pragma unroll
        for (int j = 0; j < K; ++j) x[j] = load_stream(a.data[j] + base * 16 + lane);
        uint32_t acc[M][4] = {};
        gf_matvec16<K, M>(acc, x, tab);
#pragma unroll
        for (int i = 0; i < M; ++i) {
          const uint4 v = make_uint4(acc[i][0], acc[i][1], acc[i][2], acc[i][3]);
          if constexpr (FORM == kFormPassSc1)
            store_wave<kPolicyNt | kPolicySc1>(a.out[i] + base * 16, lane, v);
          else
            store_stream(a.out[i] + base * 16 + lane, v);
        }
      }
      if (!PASSES) break;
    }
  }
}

// ------------------------------------------------------------- XOR kernel --

template <int K>
struct XorArgs {
  const uint8_t* data[K];
  uint8_t* out;
  uint64_t n16;
};

__device__ __forceinline__ uint4 xor3v(const uint4& a, const uint4& b, const uint4& c) {
  return make_uint4(xor3(a.x, b.x, c.x), xor3(a.y, b.y, c.y), xor3(a.z, b.z, c.z),
                    xor3(a.w, b.w, c.w));
}

// XOR parity: one-wavefront workgroups in launch order, one chunk per lane,
// nt buffer loads on the workgroup's wave-uniform base (as the pass forms of
// rs_kernel address it).  Measured on MI355X for XOR(4) (HBM traffic, GB/s):
// over 64 MiB shards 6482 vs 6357 for the former 512-lane workgroups with two
// chunks per lane (6399 with 128 lanes, 6288 with 256); over 256 MiB 6621 vs
// 6555.  The parity store of k > 1 is an sc1 buffer store.  XOR(4) over
// 4 x 64 MiB, same box: global nt loads with a plain global store 52.7 us,
// with an sc1 buffer store 50.9, nt buffer loads with the sc1 buffer store
// 48.9; on another box nt+sc1 stores took 54.8 us against 50.5 for sc1 ones
// (a plain store had beaten a streaming one: 6470 against 6360 GB/s).  The
// copy (k = 1) keeps the streaming global store, whose measured alternatives
// were within 1 %.
constexpr int kXorBlock = 64;

template <int K, bool PASSES>
__global__ void __launch_bounds__(kXorBlock) xor_kernel(const XorArgs<K> a) {
  const uint64_t stride = PASSES ? (uint64_t)gridDim.x * kXorBlock : 0;
  for (uint64_t base = (uint64_t)blockIdx.x * kXorBlock; base < a.n16; base += stride) {
    if (base + threadIdx.x < a.n16) {
      const uint32_t lane = threadIdx.x * 16u;
      uint4 x[K];
#pragma unroll
      for (int j = 0; j < K; ++j) x[j] = load_wave(a.data[j] + base * 16, lane);
      uint4 acc = x[0];
      int j = 1;
#pragma unroll
      for (; j + 1 < K; j += 2) acc = xor3v(acc, x[j], x[j + 1]);
      if (j < K)
        acc = make_uint4(acc.x ^ x[j].x, acc.y ^ x[j].y, acc.z ^ x[j].z, acc.w ^ x[j].w);
      if (K == 1)
        store_stream(a.out + base * 16 + lane, acc);
      else
        store_wave<kPolicySc1>(a.out + base * 16, lane, acc);
    }
    if (!PASSES) break;
  }
}

// ------------------------------------------------------------- any shards --
// Shards of any byte size (16 and more) at any alignment, in one launch: a
// frame of 16-byte chunks that starts `head` bytes into the shards (so that
// the outputs, or most of them, are aligned there) goes through the vector
// code with unaligned accesses.  The up to 15 bytes before and after it are
// the first and the last bytes of one more 16-byte chunk each, at the shards'
// start and at their end: it is loaded and coded whole, and only its own
// bytes are stored, one by one (the others belong to the frame).  Whole chunks
// at aligned addresses keep rs_kernel and xor_kernel.
struct Frame {
  uint64_t nbytes;  // of a shard
  uint64_t n16;     // chunks
  uint32_t head;    // bytes before them
  uint32_t tail;    // bytes after them
};

// A step of the launch: 0 and 1 the head and the tail where there are any,
// then the frame's.  Everything here is uniform over the workgroup (or wave).
struct Step {
  uint64_t at;         // byte offset of the step's first chunk
  uint64_t chunks;     // chunks from there to the frame's end (an edge: 1)
  uint32_t from, to;   // bytes of the chunk to store: 0, 16 except at an edge
};

__device__ __forceinline__ uint32_t edge_steps(const Frame& f) {
  return (f.head != 0) + (f.tail != 0);
}

__device__ __forceinline__ Step step_of(const Frame& f, uint64_t step, uint32_t chunks_per_step) {
  const uint32_t edges = edge_steps(f);
  if (step >= edges) {
    const uint64_t first = (step - edges) * chunks_per_step;
    return {f.head + first * 16, f.n16 - first, 0u, 16u};
  }
  if (f.head != 0 && step == 0) return {0, 1, 0u, f.head};
  return {f.nbytes - 16, 1, 16u - f.tail, 16u};
}

__device__ __forceinline__ bool whole(const Step& s) { return s.to - s.from == 16u; }

__device__ __forceinline__ void store_edge(uint8_t* p, const Step& s, const uint4& v) {
  store_bytes(p, s.from, s.to, v);
}

template <int M>
__device__ __forceinline__ void store_outputs(uint8_t* const (&out)[M], uint64_t off, const Step& s,
                                              const uint32_t (&acc)[M][4]) {
  if (whole(s)) {
#pragma unroll
    for (int i = 0; i < M; ++i)
      store_any(out[i] + off, make_uint4(acc[i][0], acc[i][1], acc[i][2], acc[i][3]));
  } else {
#pragma unroll
    for (int i = 0; i < M; ++i)
      store_edge(out[i] + off, s, make_uint4(acc[i][0], acc[i][1], acc[i][2], acc[i][3]));
  }
}

template <int K, int M>
struct AnyArgs {
  const uint8_t* data[K];
  uint8_t* out[M];
  PermTab tab[M][K];
  Frame f;
};

template <int K, int M, bool PASSES>
__global__ void __launch_bounds__((flat_block<K, M>())) any_kernel(const AnyArgs<K, M> a) {
  constexpr int B = flat_block<K, M>();
  __shared__ PermTab tab[M][K];
  for (int q = threadIdx.x; q < M * K; q += B) tab[q / K][q % K] = a.tab[q / K][q % K];
  __syncthreads();
  const uint64_t steps = PASSES ? edge_steps(a.f) + (a.f.n16 + B - 1) / B : 0;
  for (uint64_t step = blockIdx.x;;) {
    const Step s = step_of(a.f, step, B);
    if (threadIdx.x < s.chunks) {
      const uint32_t lane = threadIdx.x * 16u;
      uint4 x[K];
#pragma unroll
      for (int j = 0; j < K; ++j) x[j] = load_any(a.data[j] + s.at + lane);
      uint32_t acc[M][4] = {};
      gf_matvec16<K, M>(acc, x, tab);
      pin_products(acc);
      store_outputs(a.out, s.at + lane, s, acc);
    }
    step += gridDim.x;
    if (!PASSES || step >= steps) break;
  }
}

template <int K>
struct AnyXorArgs {
  const uint8_t* data[K];
  uint8_t* out;
  Frame f;
};

template <int K>
__global__ void __launch_bounds__(kXorBlock) any_xor_kernel(const AnyXorArgs<K> a) {
  const uint64_t steps = edge_steps(a.f) + (a.f.n16 + kXorBlock - 1) / kXorBlock;
  for (uint64_t step = blockIdx.x; step < steps; step += gridDim.x) {
    const Step s = step_of(a.f, step, kXorBlock);
    if (threadIdx.x >= s.chunks) continue;
    const uint32_t lane = threadIdx.x * 16u;
    uint4 x[K];
#pragma unroll
    for (int j = 0; j < K; ++j) x[j] = load_any(a.data[j] + s.at + lane);
    uint4 acc = x[0];
    int j = 1;
#pragma unroll
    for (; j + 1 < K; j += 2) acc = xor3v(acc, x[j], x[j + 1]);
    if (j < K) acc = make_uint4(acc.x ^ x[j].x, acc.y ^ x[j].y, acc.z ^ x[j].z, acc.w ^ x[j].w);
    if (whole(s))
      store_any(a.out + s.at + lane, acc);
    else
      store_edge(a.out + s.at + lane, s, acc);
  }
}

// Shards of less than 16 bytes, any k and m: a lane per byte and output, all
// in one workgroup.  Every output is coded before any is stored, since an
// output may lie over an input.
struct TinyArgs {
  const uint8_t* data[EC_MAX_K];
  uint8_t* out[EC_MAX_M];
  uint8_t coeff[EC_MAX_M * EC_MAX_K];
  uint32_t n;
  int k, m;
};

constexpr int kTinyBlock = 16 * EC_MAX_M;

__global__ void __launch_bounds__(kTinyBlock) tiny_kernel(const TinyArgs a) {
  const uint32_t b = threadIdx.x & 15u;
  const int i = threadIdx.x >> 4;
  const bool mine = b < a.n && i < a.m;
  uint8_t acc = 0;
  if (mine)
    for (int j = 0; j < a.k; ++j) acc ^= dev_gf_mul(a.coeff[i * a.k + j], gptr(a.data[j])[b]);
  __syncthreads();
  if (mine) gptr(a.out[i])[b] = acc;
}

// ------------------------------------------------------------ table kernel --
// Codes past the unrolled kernels for which the permute tables cost less than
// the matrix cores (flat_route in routes.h), any size and alignment: see
// kWideGroup in ec_device.h.
struct TableArgs {
  const uint8_t* data[EC_MAX_K];
  uint8_t* out[EC_MAX_M];
  uint8_t coeff[EC_MAX_M * EC_MAX_K];  // row-major m x k
  Frame f;
  int k;
};

// 128-lane workgroups in launch order.  Measured on MI355X (HBM traffic,
// TB/s, 64 MiB shards): RS(17,1) 6.1, RS(20,2) 5.8, RS(6,12) 5.5, RS(10,12)
// 4.6; 256-lane workgroups that streamed each shard at two places half a shard
// apart were 1-6 % slower.  Shards of 64 MiB + 5 B at the rate of whole chunks
// (us, on the matrix cores before / here): RS(17,1) 216 / 196, RS(6,9) 203 / 178,
// RS(10,10) 326 / 277, RS(4,16) 283 / 241, XOR of 32 381 / 362.
constexpr int kTableBlock = 128;

template <int M>
__global__ void __launch_bounds__(kTableBlock) table_kernel(const TableArgs a) {
  __shared__ PermTab tab[M * EC_MAX_K];
  const int k = a.k;
  for (int t = threadIdx.x; t < M * k; t += kTableBlock) tab[t] = dev_perm_tab(a.coeff[t]);
  __syncthreads();
  const uint64_t steps = edge_steps(a.f) + (a.f.n16 + kTableBlock - 1) / kTableBlock;
  for (uint64_t step = blockIdx.x; step < steps; step += gridDim.x) {
    const Step s = step_of(a.f, step, kTableBlock);
    if (threadIdx.x >= s.chunks) continue;
    uint32_t lane = threadIdx.x * 16u;
    asm volatile("" : "+v"(lane));   // no address is kept over the steps
    uint32_t acc[M][4] = {};
    for (int j0 = 0; j0 < k; j0 += kWideGroup) {
      uint4 x[kWideGroup];
#pragma unroll
      for (int g = 0; g < kWideGroup; ++g)
        x[g] = j0 + g < k ? load_any(a.data[j0 + g] + s.at + lane) : make_uint4(0, 0, 0, 0);
#pragma unroll
      for (int g = 0; g < kWideGroup; g += kWidePair<M>()) {
        if (j0 + g >= k) break;
        if constexpr (kWidePair<M>() == 2) {
          // Two coefficients per step (three XOR3 instead of two XOR3 and
          // two XOR).  x[g + 1] is zero past k and a zero byte's products
          // are zero, so the pair form is exact for an odd k as well.
          Fields fa[4], fb[4];
#pragma unroll
          for (int dd = 0; dd < 4; ++dd) {
            fa[dd] = fields(word(x[g], dd));
            fb[dd] = fields(word(x[g + 1], dd));
          }
          const int jb = j0 + g + 1 < k ? j0 + g + 1 : j0 + g;
#pragma unroll
          for (int i = 0; i < M; ++i) {
            // Read each table right before its uses (see gf_matvec16).
            asm volatile("" ::: "memory");
            const PermTab ta = tab[i * k + j0 + g], tb = tab[i * k + jb];
#pragma unroll
            for (int dd = 0; dd < 4; ++dd) acc[i][dd] = mac2(acc[i][dd], ta, fa[dd], tb, fb[dd]);
          }
        } else {
          Fields f[4];
#pragma unroll
          for (int dd = 0; dd < 4; ++dd) f[dd] = fields(word(x[g], dd));
#pragma unroll
          for (int i = 0; i < M; ++i) {
            asm volatile("" ::: "memory");
            const PermTab t = tab[i * k + j0 + g];
#pragma unroll
            for (int dd = 0; dd < 4; ++dd) acc[i][dd] = mac1(acc[i][dd], t, f[dd]);
          }
        }
      }
    }
    pin_products(acc);
    if (whole(s)) {
#pragma unroll
      for (int i = 0; i < M; ++i)
        store_any(a.out[i] + s.at + lane, make_uint4(acc[i][0], acc[i][1], acc[i][2], acc[i][3]));
    } else {
#pragma unroll
      for (int i = 0; i < M; ++i)
        store_edge(a.out[i] + s.at, s, make_uint4(acc[i][0], acc[i][1], acc[i][2], acc[i][3]));
    }
  }
}

// ------------------------------------------------------------ wide kernels --
// Codes past the unrolled kernels, any alignment and size, on the matrix cores
// (ec_mfma.h).  A wave codes 32 chunks (512 bytes of each shard) per step:
// lane l and lane l + 32 load the same columns of the even and the odd shards,
// and store those of the even and the odd outputs.
//   m > 4 (wide_kernel): the MFMAs and bit selects take about as long as the
// memory traffic, so waves stay and load their next step while they code one.
// Measured on MI355X (HBM traffic, TB/s; the former run-time-k kernel on
// permute tables first): RS(24,8) over 32 MiB shards 4.08 -> 5.38 (one step
// per wave without the loads ahead 5.19), RS(32,16) 2.69 -> 3.93 (3.10),
// RS(20,12) 3.57 -> 4.27 (3.80), RS(16,8) over 64 MiB 4.47 -> 5.61 (5.16).
// With the MFMAs taken out the same kernel moves 5.7-6.0.  By counters the
// matrix cores work 42 % of the time and the vector ALUs 40 % (RS(24,8));
// RS(32,16) 66 and 40.
//   m <= 4 (wide_narrow_kernel): memory-bound, one step per wave and none
// ahead: RS(20,4) over 64 MiB 5.70 -> 6.12 (with loads ahead 5.6), RS(24,4)
// 5.62 -> 5.90.
struct WideArgs {
  const uint8_t* data[EC_MAX_K];   // data[k] = data[k - 1] when k is odd
  uint8_t* out[EC_MAX_M];
  MfmaCoeff coeff;
  Frame f;
  int k, m;
};

// even or odd by the lane's half.  Both are read into scalar registers first:
// the compiler would otherwise select the address to read them from, one
// dependent vector load each.
template <typename T>
__device__ __forceinline__ T* of_half(uint32_t half, T* even, T* odd) {
  asm volatile("" : "+s"(even), "+s"(odd));
  return half ? odd : even;
}

constexpr int kWideBlock = 256;
constexpr int kWideChunks = 32;   // chunks of a wave's step

template <int KH, int MH>
struct WideLds {
  const uint8_t* data[EC_MAX_K];
  uint8_t* out[EC_MAX_M];
  typename MfmaCode<KH, MH>::Lds code;
};

// The loads of a step: x[kt][i] of shard 8 kt + 2 i + h, 16 bytes at off.
template <int KH>
__device__ __forceinline__ void wide_loads(uint4 (&x)[mfma_groups(KH)][4],
                                           const uint8_t* const* data, int k, uint32_t half,
                                           uint64_t off) {
#pragma unroll
  for (int kt = 0; kt < mfma_groups(KH); ++kt)
#pragma unroll
    for (int i = 0; i < mfma_words(KH, kt); ++i) {
      const int even = 8 * kt + 2 * i;
      if (even < 4 * KH - 3 || even < k)   // uniform: the first always, k > 4 (KH - 1)
        x[kt][i] = load_any(data[even + half] + off);
      else
        x[kt][i] = make_uint4(0u, 0u, 0u, 0u);
    }
}

template <int KH, int MH, bool PAIR>
__global__ void __launch_bounds__(kWideBlock) __attribute__((amdgpu_waves_per_eu(2)))
wide_kernel(const WideArgs a) {
  constexpr int KT = mfma_groups(KH), MT = mfma_tiles(MH);
  __shared__ WideLds<KH, MH> lds;
  if (threadIdx.x < EC_MAX_K) lds.data[threadIdx.x] = a.data[threadIdx.x];
  else if (threadIdx.x < EC_MAX_K + EC_MAX_M)
    lds.out[threadIdx.x - EC_MAX_K] = a.out[threadIdx.x - EC_MAX_K];
  MfmaCode<KH, MH> code;
  code.template load<kWideBlock>(a.coeff, lds.code);
  __syncthreads();
  const uint32_t lane = threadIdx.x & 63u, col = lane & 31u, half = lane >> 5;
  const uint64_t steps = edge_steps(a.f) + (a.f.n16 + kWideChunks - 1) / kWideChunks;
  const uint64_t stride = (uint64_t)gridDim.x * (kWideBlock / 64);
  uint64_t step = (uint64_t)blockIdx.x * (kWideBlock / 64) +
                  __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (step >= steps) return;
  Step s = step_of(a.f, step, kWideChunks);
  uint64_t off = s.at + (col < s.chunks ? col * 16u : 0u);   // past the end: the first chunk
  uint4 x[KT][4];
  wide_loads<KH>(x, lds.data, a.k, half, off);
  for (;;) {
    uint32_t t[KT][4][4];
    mfma_columns<KH, true>(t, x);
    // The next step's loads are in flight while this one is coded.
    const Step now = s;
    const uint64_t at = off;
    const bool mine = col < now.chunks;
    step += stride;
    const bool more = step < steps;   // uniform
    asm volatile("" ::: "memory");    // the addresses stay in LDS
    if (more) {
      s = step_of(a.f, step, kWideChunks);
      off = s.at + (col < s.chunks ? col * 16u : 0u);
      wide_loads<KH>(x, lds.data, a.k, half, off);
    }
    uint4 out[MT][2];
    mfma_matvec16<KH, MH, PAIR>(out, t, code);
    asm volatile("" ::: "memory");
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int q = 0; q < mfma_outs(MH, mt); ++q) {
        const uint32_t o = 4 * mt + 2 * q + half;
        if (!mine || (int)o >= a.m) continue;
        if (whole(now))
          store_any(lds.out[o] + at, out[mt][q]);
        else
          store_edge(lds.out[o] + at, now, out[mt][q]);
      }
    if (!more) break;
  }
}

template <int KH, int MH, bool PAIR>
__global__ void __launch_bounds__(kWideBlock)
__attribute__((amdgpu_waves_per_eu(2))) wide_narrow_kernel(const WideArgs a) {
  constexpr int KT = mfma_groups(KH);
  static_assert(mfma_tiles(MH) == 1 && !MfmaCode<KH, MH>::kInLds, "m <= 4");
  const uint32_t lane = threadIdx.x & 63u, col = lane & 31u, half = lane >> 5;
  const uint64_t steps = edge_steps(a.f) + (a.f.n16 + kWideChunks - 1) / kWideChunks;
  const uint64_t stride = (uint64_t)gridDim.x * (kWideBlock / 64);
  uint64_t step = (uint64_t)blockIdx.x * (kWideBlock / 64) +
                  __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (step >= steps) return;
  const uint8_t* data[KT][4];
  uint8_t* outp[2];
#pragma unroll
  for (int kt = 0; kt < KT; ++kt)
#pragma unroll
    for (int i = 0; i < mfma_words(KH, kt); ++i)
      data[kt][i] = of_half(half, a.data[8 * kt + 2 * i], a.data[8 * kt + 2 * i + 1]);
#pragma unroll
  for (int q = 0; q < mfma_outs(MH, 0); ++q) outp[q] = of_half(half, a.out[2 * q], a.out[2 * q + 1]);
  __shared__ typename MfmaCode<KH, MH>::Lds unused;
  MfmaCode<KH, MH> code;
  code.template load<kWideBlock>(a.coeff, unused);
  for (; step < steps; step += stride) {
    const Step s = step_of(a.f, step, kWideChunks);
    const bool mine = col < s.chunks;
    const uint64_t off = s.at + (mine ? col * 16u : 0u);   // past the end: the first chunk
    uint4 x[KT][4];
#pragma unroll
    for (int kt = 0; kt < KT; ++kt)
#pragma unroll
      for (int i = 0; i < mfma_words(KH, kt); ++i) {
        const int even = 8 * kt + 2 * i;
        if (even < 4 * KH - 3 || even < a.k)   // uniform, as in wide_loads
          x[kt][i] = load_any(data[kt][i] + off);
        else
          x[kt][i] = make_uint4(0u, 0u, 0u, 0u);
      }
    uint32_t t[KT][4][4];
    mfma_columns<KH, false>(t, x);
    uint4 out[1][2];
    mfma_matvec16<KH, MH, PAIR>(out, t, code);
#pragma unroll
    for (int q = 0; q < mfma_outs(MH, 0); ++q) {
      if (!mine || (int)(2 * q + half) >= a.m) continue;
      if (whole(s))
        store_any(outp[q] + off, out[0][q]);
      else
        store_edge(outp[q] + off, s, out[0][q]);
    }
  }
}

// ---------------------------------------------------------- host launch --

template <int K, int M>
int launch_rs(const uint8_t* coeff, const uint8_t* const* d, uint8_t* const* o, uint64_t n16,
              hipStream_t st) {
  RsArgs<K, M> a;
  for (int j = 0; j < K; ++j) a.data[j] = d[j];
  for (int i = 0; i < M; ++i) a.out[i] = o[i];
  for (int i = 0; i < M; ++i)
    for (int j = 0; j < K; ++j) a.tab[i][j] = perm_tab(coeff[i * K + j]);
  a.n16 = n16;
  constexpr int B = flat_block<K, M>();
  constexpr int F = flat_form<K, M>();
  const unsigned grid = grid_of(n16, B);
  if constexpr (F == kFormLanes) {
    hipLaunchKernelGGL((rs_kernel<K, M, F, false>), dim3(grid), dim3(B), 0, st, a);
  } else {
    if ((uint64_t)grid * B >= n16)
      hipLaunchKernelGGL((rs_kernel<K, M, F, false>), dim3(grid), dim3(B), 0, st, a);
    else
      hipLaunchKernelGGL((rs_kernel<K, M, F, true>), dim3(grid), dim3(B), 0, st, a);
  }
  return hip_status();
}

using WideFn = int (*)(const uint8_t*, int, int, const uint8_t* const*, uint8_t* const*,
                       const Frame&, hipStream_t);
WideFn wide_fn(int k, int m);

inline uint64_t frame_steps(const Frame& f, uint64_t chunks_per_step) {
  return (f.head != 0) + (f.tail != 0) + (f.n16 + chunks_per_step - 1) / chunks_per_step;
}

template <int K, int M>
int launch_any(const uint8_t* coeff, const uint8_t* const* d, uint8_t* const* o, const Frame& f,
               hipStream_t st) {
  AnyArgs<K, M> a;
  for (int j = 0; j < K; ++j) a.data[j] = d[j];
  for (int i = 0; i < M; ++i) a.out[i] = o[i];
  for (int i = 0; i < M; ++i)
    for (int j = 0; j < K; ++j) a.tab[i][j] = perm_tab(coeff[i * K + j]);
  a.f = f;
  constexpr int B = flat_block<K, M>();
  const uint64_t steps = frame_steps(f, B);
  const unsigned grid = (unsigned)(steps < max_grid(B) ? steps : max_grid(B));
  if (grid == steps)
    hipLaunchKernelGGL((any_kernel<K, M, false>), dim3(grid), dim3(B), 0, st, a);
  else if constexpr (M <= kFastMaxM)
    hipLaunchKernelGGL((any_kernel<K, M, true>), dim3(grid), dim3(B), 0, st, a);
  else   // more steps than one grid
    return wide_fn(K, M)(coeff, K, M, d, o, f, st);
  return hip_status();
}

template <int K>
int launch_any_xor(const uint8_t* const* d, uint8_t* o, const Frame& f, hipStream_t st) {
  AnyXorArgs<K> a;
  for (int j = 0; j < K; ++j) a.data[j] = d[j];
  a.out = o;
  a.f = f;
  const uint64_t steps = frame_steps(f, kXorBlock);
  const uint64_t grid = steps < max_grid(kXorBlock) ? steps : max_grid(kXorBlock);
  hipLaunchKernelGGL((any_xor_kernel<K>), dim3((unsigned)grid), dim3(kXorBlock), 0, st, a);
  return hip_status();
}

// Workgroups of a wide_kernel launch.  About one for each that the chip holds
// for the deep codes (2 waves per SIMD), several where more waves fit: capped
// at 1024 / 4096, RS(24,8) over 32 MiB 199.7 / 209.3 us, RS(32,16) 410 / 420,
// RS(20,12) 251 / 261, but RS(16,8) over 64 MiB 294.7 / 287.2, RS(16,6) 267 / 263.
constexpr uint64_t kWideGridDeep = 1024, kWideGrid = 4096;

template <int KH, int MH>
int launch_wide(const uint8_t* coeff, int k, int m, const uint8_t* const* d, uint8_t* const* o,
                const Frame& f, hipStream_t st) {
  WideArgs a;
  // With k odd the upper lanes read the last shard as well (their
  // coefficients for it are zero).
  for (int j = 0; j < EC_MAX_K; ++j) a.data[j] = j < k ? d[j] : j == k ? d[k - 1] : nullptr;
  for (int i = 0; i < EC_MAX_M; ++i) a.out[i] = i < m ? o[i] : nullptr;
  a.coeff = mfma_coeff(coeff, k, m);
  a.f = f;
  a.k = k;
  a.m = m;
  constexpr uint64_t kWaves = kWideBlock / 64;
  const uint64_t blocks = (frame_steps(f, kWideChunks) + kWaves - 1) / kWaves;
  const uint64_t cap = MH <= 2 ? max_grid(kWideBlock) : mfma_groups(KH) >= 3 ? kWideGridDeep : kWideGrid;
  const dim3 grid((unsigned)(blocks < cap ? blocks : cap)), block(kWideBlock);
  bool pair = true;
  if constexpr (KH == EC_MAX_K / 4) pair = mfma_pair_ok(coeff, k, m);
  if constexpr (MH <= 2) {
    if (pair)
      hipLaunchKernelGGL((wide_narrow_kernel<KH, MH, true>), grid, block, 0, st, a);
    else if constexpr (KH == EC_MAX_K / 4)
      hipLaunchKernelGGL((wide_narrow_kernel<KH, MH, false>), grid, block, 0, st, a);
  } else {
    if (pair)
      hipLaunchKernelGGL((wide_kernel<KH, MH, true>), grid, block, 0, st, a);
    else if constexpr (KH == EC_MAX_K / 4)
      hipLaunchKernelGGL((wide_kernel<KH, MH, false>), grid, block, 0, st, a);
  }
  return hip_status();
}

template <int M>
int launch_table(const uint8_t* coeff, int k, const uint8_t* const* d, uint8_t* const* o,
                 const Frame& f, hipStream_t st) {
  TableArgs a;
  for (int j = 0; j < k; ++j) a.data[j] = d[j];
  for (int i = 0; i < M; ++i) a.out[i] = o[i];
  for (int t = 0; t < M * k; ++t) a.coeff[t] = coeff[t];
  a.f = f;
  a.k = k;
  const uint64_t steps = frame_steps(f, kTableBlock);
  const uint64_t grid = steps < max_grid(kTableBlock) ? steps : max_grid(kTableBlock);
  hipLaunchKernelGGL((table_kernel<M>), dim3((unsigned)grid), dim3(kTableBlock), 0, st, a);
  return hip_status();
}

template <int K>
int launch_xor(const uint8_t* const* d, uint8_t* o, uint64_t n16, hipStream_t st) {
  XorArgs<K> a;
  for (int j = 0; j < K; ++j) a.data[j] = d[j];
  a.out = o;
  a.n16 = n16;
  const unsigned grid = grid_of(n16, kXorBlock);
  if ((uint64_t)grid * kXorBlock >= n16)
    hipLaunchKernelGGL((xor_kernel<K, false>), dim3(grid), dim3(kXorBlock), 0, st, a);
  else
    hipLaunchKernelGGL((xor_kernel<K, true>), dim3(grid), dim3(kXorBlock), 0, st, a);
  return hip_status();
}

using RsFn = int (*)(const uint8_t*, const uint8_t* const*, uint8_t* const*, uint64_t,
                     hipStream_t);
using XorFn = int (*)(const uint8_t* const*, uint8_t*, uint64_t, hipStream_t);
using AnyFn = int (*)(const uint8_t*, const uint8_t* const*, uint8_t* const*, const Frame&,
                      hipStream_t);
using AnyXorFn = int (*)(const uint8_t* const*, uint8_t*, const Frame&, hipStream_t);

template <int K, int... Ms>
constexpr auto rs_row(std::integer_sequence<int, Ms...>) {
  return std::array<RsFn, sizeof...(Ms)>{&launch_rs<K, Ms + 1>...};
}
template <int... Ks>
constexpr auto rs_table(std::integer_sequence<int, Ks...>) {
  return std::array<std::array<RsFn, kFastMaxM>, sizeof...(Ks)>{
      rs_row<Ks + 1>(std::make_integer_sequence<int, kFastMaxM>{})...};
}
template <int... Ks>
constexpr auto xor_table(std::integer_sequence<int, Ks...>) {
  return std::array<XorFn, sizeof...(Ks)>{&launch_xor<Ks + 1>...};
}
template <int K, int M>
constexpr AnyFn any_entry() {
  if constexpr (any_reached(K, M)) return &launch_any<K, M>;
  else return nullptr;
}
template <int K, int... Ms>
constexpr auto any_row(std::integer_sequence<int, Ms...>) {
  return std::array<AnyFn, sizeof...(Ms)>{any_entry<K, Ms + 1>()...};
}
template <int... Ks>
constexpr auto any_table(std::integer_sequence<int, Ks...>) {
  return std::array<std::array<AnyFn, kAnyMaxM>, sizeof...(Ks)>{any_row<Ks + 1>(std::make_integer_sequence<int, kAnyMaxM>{})...};
}
template <int... Ks>
constexpr auto any_xor_table(std::integer_sequence<int, Ks...>) {
  return std::array<AnyXorFn, sizeof...(Ks)>{&launch_any_xor<Ks + 1>...};
}
using TableFn = int (*)(const uint8_t*, int, const uint8_t* const*, uint8_t* const*, const Frame&,
                        hipStream_t);
template <int M>
constexpr TableFn table_entry() {
  if constexpr (table_reached(M)) return &launch_table<M>;
  else return nullptr;
}
template <int... Ms>
constexpr auto table_table(std::integer_sequence<int, Ms...>) {
  return std::array<TableFn, sizeof...(Ms)>{table_entry<Ms + 1>()...};
}
template <int KH, int MH>
constexpr WideFn wide_entry() {
  if constexpr (core_reached(KH, MH)) return &launch_wide<KH, MH>;
  else return nullptr;
}
template <int KH, int... Ms>
constexpr auto wide_row(std::integer_sequence<int, Ms...>) {
  return std::array<WideFn, sizeof...(Ms)>{wide_entry<KH, Ms + 1>()...};
}
constexpr int kWideKH = EC_MAX_K / 4, kWideMH = EC_MAX_M / 2;
template <int... Ks>
constexpr auto wide_table(std::integer_sequence<int, Ks...>) {
  return std::array<std::array<WideFn, kWideMH>, sizeof...(Ks)>{
      wide_row<Ks + 1>(std::make_integer_sequence<int, kWideMH>{})...};
}

const auto kRsTable = rs_table(std::make_integer_sequence<int, kFastMaxK>{});
const auto kXorTable = xor_table(std::make_integer_sequence<int, kFastMaxK>{});
const auto kAnyTable = any_table(std::make_integer_sequence<int, kFastMaxK>{});
const auto kAnyXorTable = any_xor_table(std::make_integer_sequence<int, kFastMaxK>{});
const auto kTableTable = table_table(std::make_integer_sequence<int, EC_MAX_M>{});
const auto kWideTable = wide_table(std::make_integer_sequence<int, kWideKH>{});

WideFn wide_fn(int k, int m) {
  return kWideTable[(k - 1) / 4][(m - 1) / 2];
}

// The address modulo 16 that most of n addresses share.
inline uint32_t usual_skew(uint8_t* const* a, int n) {
  int count[16] = {};
  for (int i = 0; i < n; ++i) ++count[reinterpret_cast<uintptr_t>(a[i]) & 15u];
  uint32_t best = 0;
  for (uint32_t s = 1; s < 16; ++s)
    if (count[s] > count[best]) best = s;
  return best;
}

inline bool all_aligned(const uint8_t* const* a, int n) {
  uintptr_t bits = 0;
  for (int i = 0; i < n; ++i) bits |= reinterpret_cast<uintptr_t>(a[i]);
  return (bits & 15u) == 0;
}

// The frame of nbytes-long shards with outputs o: its chunks start where most
// outputs are 16-byte aligned.
inline Frame frame_of(uint8_t* const* o, int m, uint64_t nbytes) {
  Frame f;
  f.nbytes = nbytes;
  const uint32_t skew = usual_skew(o, m);
  f.head = skew ? 16u - skew : 0u;
  if (f.head > nbytes) f.head = (uint32_t)nbytes;
  f.n16 = (nbytes - f.head) / 16;
  f.tail = (uint32_t)(nbytes - f.head - f.n16 * 16);
  return f;
}

int launch_tiny(const uint8_t* coeff, int k, int m, const uint8_t* const* d, uint8_t* const* o,
                uint64_t n, hipStream_t st) {
  TinyArgs a;
  for (int j = 0; j < k; ++j) a.data[j] = d[j];
  for (int i = 0; i < m; ++i) a.out[i] = o[i];
  for (int t = 0; t < m * k; ++t) a.coeff[t] = coeff[t];
  a.n = (uint32_t)n;
  a.k = k;
  a.m = m;
  hipLaunchKernelGGL(tiny_kernel, dim3(1), dim3(kTinyBlock), 0, st, a);
  return hip_status();
}

int matvec(const uint8_t* coeff, int k, int m, const uint8_t* const* d, uint8_t* const* o,
           uint64_t nbytes, hipStream_t st) {
  if (!coeff || !d || !o) return EC_EINVAL;
  if (k < 1 || m < 1) return EC_EINVAL;
  if (k > EC_MAX_K || m > EC_MAX_M) return EC_ERANGE;
  if (nbytes == 0) return EC_OK;  // empty shards may have null addresses
  for (int j = 0; j < k; ++j)
    if (!d[j]) return EC_EINVAL;
  for (int i = 0; i < m; ++i)
    if (!o[i]) return EC_EINVAL;
  const bool aligned = nbytes % 16 == 0 && all_aligned(d, k) && all_aligned(o, m);
  switch (flat_route(k, m, nbytes, aligned)) {
    case FlatRoute::kTiny:
      return launch_tiny(coeff, k, m, d, o, nbytes, st);
    case FlatRoute::kAligned:
      return kRsTable[k - 1][m - 1](coeff, d, o, nbytes / 16, st);
    case FlatRoute::kAny:
      return kAnyTable[k - 1][m - 1](coeff, d, o, frame_of(o, m, nbytes), st);
    case FlatRoute::kTable:
      return kTableTable[m - 1](coeff, k, d, o, frame_of(o, m, nbytes), st);
    case FlatRoute::kWide:
      break;
  }
  return wide_fn(k, m)(coeff, k, m, d, o, frame_of(o, m, nbytes), st);
}

}  // namespace
}  // namespace ec

extern "C" {

int ec_xor_encode(const uint8_t* const* d_data, int k, uint8_t* d_parity, uint64_t nbytes,
                  ec_stream_t stream) {
  if (!d_data || k < 1) return EC_EINVAL;
  if (k > EC_MAX_K) return EC_ERANGE;
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  if (nbytes == 0) return EC_OK;  // empty shards may have null addresses
  if (!d_parity) return EC_EINVAL;
  for (int j = 0; j < k; ++j)
    if (!d_data[j]) return EC_EINVAL;
  uint8_t* const out[1] = {d_parity};
  if (k > ec::kFastMaxK || nbytes < 16) {
    uint8_t ones[EC_MAX_K];
    for (int j = 0; j < k; ++j) ones[j] = 1;  // 1*x = x
    return ec::matvec(ones, k, 1, d_data, out, nbytes, st);
  }
  if (nbytes % 16 == 0 && ec::all_aligned(d_data, k) && ec::all_aligned(out, 1))
    return ec::kXorTable[k - 1](d_data, d_parity, nbytes / 16, st);
  return ec::kAnyXorTable[k - 1](d_data, d_parity, ec::frame_of(out, 1, nbytes), st);
}

int ec_rs_encode(const uint8_t* coeff, int k, int m, const uint8_t* const* d_data,
                 uint8_t* const* d_parity, uint64_t nbytes, ec_stream_t stream) {
  return ec::matvec(coeff, k, m, d_data, d_parity, nbytes, reinterpret_cast<hipStream_t>(stream));
}

int ec_rs_decode(const uint8_t* rows, int k, int e, const uint8_t* const* d_survivors,
                 uint8_t* const* d_out, uint64_t nbytes, ec_stream_t stream) {
  return ec::matvec(rows, k, e, d_survivors, d_out, nbytes, reinterpret_cast<hipStream_t>(stream));
}

int ec_stream_create(int device, int n_cus, ec_stream_t* out) {
  if (!out) return EC_EINVAL;
  *out = nullptr;
  int count = 0;
  if (hipGetDeviceCount(&count) != hipSuccess) return EC_EHIP;
  if (device < 0 || device >= count) return EC_EINVAL;
  int cus = 0;
  if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device) != hipSuccess ||
      cus <= 0)
    return EC_EHIP;
  const int n = (n_cus <= 0 || n_cus > cus) ? cus : n_cus;
  std::vector<uint32_t> mask((cus + 31) / 32, 0u);
  for (int c = 0; c < n; ++c) mask[c / 32] |= 1u << (c % 32);
  int prev = 0;
  if (hipGetDevice(&prev) != hipSuccess) return EC_EHIP;
  if (prev != device && hipSetDevice(device) != hipSuccess) return EC_EHIP;
  hipStream_t st = nullptr;
  const hipError_t e =
      hipExtStreamCreateWithCUMask(&st, static_cast<uint32_t>(mask.size()), mask.data());
  if (prev != device) (void)hipSetDevice(prev);
  if (e != hipSuccess) {
    (void)hipGetLastError();
    return EC_EHIP;
  }
  *out = st;
  return EC_OK;
}

int ec_stream_destroy(ec_stream_t stream) {
  if (!stream) return EC_EINVAL;
  return hipStreamDestroy(reinterpret_cast<hipStream_t>(stream)) == hipSuccess ? EC_OK : EC_EHIP;
}

}  // extern "C"

// routes.h — which kernel a flat call takes, by the code's shape and the
// shards' size and alignment.  No device code: the dispatch tables are filled
// by the same functions, and a host test checks the rule over every shape.
#pragma once

#include <stdint.h>

#include "ec_mi355.h"

namespace ec {

constexpr int kFastMaxK = 16;   // shapes of the fully unrolled kernels
constexpr int kFastMaxM = 4;
constexpr bool fast_shape(int k, int m) { return k <= kFastMaxK && m <= kFastMaxM; }

constexpr int kMfmaShards = 8;     // shards per 64-deep K step of the matrix cores
constexpr int kMfmaOutputs = 4;    // parity shards per 32-row tile

// What a code costs on the permute tables and on the matrix cores: SIMD cycles
// per 512 byte columns, 4 per VALU op (1.125 k m + 1.25 k ops per column
// against the transposes, expansions and bit selects of ec_mfma.h) and 32 per
// MFMA; the two kinds measured about additive.
constexpr int table_cost(int k, int m) { return 36 * k * m + 40 * k; }
constexpr int core_cost(int k, int m) {
  const int kt = (k + kMfmaShards - 1) / kMfmaShards, mt = (m + kMfmaOutputs - 1) / kMfmaOutputs;
  return 512 * kt * mt + 448 * kt + 240 * ((m + 1) / 2);
}

// Whether the permute tables take fewer cycles than the matrix cores for a
// code past the unrolled kernels.
constexpr bool table_pays(int k, int m) { return table_cost(k, m) <= core_cost(k, m); }

// Codes past the unrolled kernels that any_kernel is instantiated for: they
// are the ones it is fastest at.  Over 64 MiB + 5 B shards on MI355X (us,
// any_kernel / table_kernel / matrix cores): RS(5,5) 112 / 114 / 135, RS(8,5)
// 142 / 148 / 154, RS(12,5) 189 / 204 / 231, RS(10,6) 183 / 198 / 224, RS(8,6)
// 155 / 165 / 167, RS(12,7) 235 / 257 / 254, RS(6,8) 161 / 166 / 174, RS(11,8)
// 247 / 277 / 255.
constexpr int kAnyMaxM = 8, kAnyDeepMaxK = 12;
constexpr bool any_shape(int k, int m) {
  return fast_shape(k, m) || (k <= kAnyDeepMaxK && m <= kAnyMaxM);
}

// Up to this shard size too few waves run to be bound by either's arithmetic
// and the matrix cores' shorter chains win for every code but the cheapest
// (2 MiB shards, us, tables / matrix cores: RS(20,2) 11.9 / 10.7, RS(6,12) 11.3
// / 10.5, RS(16,5) 14.1 / 12.2).
constexpr uint64_t kTableMinBytes = 2u << 20;

// table_kernel, with k at run time, waits longer for its LDS tables than the
// cost says, the more so the fewer waves run.  Its time over that of the matrix
// cores on MI355X, by the ratio r of the two costs, over shards of 3 MiB / 4 MiB
// / 64 MiB of odd sizes:
//   r <= 0.7         RS(17,1) 0.85 0.78 0.91, RS(24,1) 0.87 0.83 0.96, RS(6,9)
//     0.92 0.82 0.87, RS(17,2) 0.98 0.85 0.96, RS(4,16) 1.01 0.92 0.83
//   0.7 < r <= 0.9   RS(13,5) 1.18 0.97 0.92, RS(17,3) 1.11 0.94 0.96, RS(20,2)
//     0.99 0.84 1.03, RS(20,5) 1.17 0.98 0.94, RS(10,12) 1.01 0.94 0.92
//   r > 0.9          RS(13,6) 1.28 1.05 1.00, RS(16,5) 1.24 1.00 1.02, RS(13,7)
//     1.25 1.10 1.05, RS(7,12) 1.17 0.98 1.09
constexpr bool table_kernel_pays(int k, int m, uint64_t nbytes) {
  const int table = table_cost(k, m), core = core_cost(k, m);
  return 10 * table <= 7 * core || (10 * table <= 9 * core && nbytes > 2 * kTableMinBytes);
}

enum class FlatRoute {
  kTiny,      // tiny_kernel: less than one chunk
  kAligned,   // rs_kernel, xor_kernel: whole chunks at aligned addresses
  kAny,       // any_kernel, any_xor_kernel: unrolled tables
  kTable,     // table_kernel: permute tables, k at run time
  kWide,      // wide_kernel, wide_narrow_kernel: the matrix cores
};

// aligned: every shard at a 16-byte-aligned address and of whole chunks.  It
// chooses between two kernels of the unrolled shapes only; past them any size
// and alignment takes the kernel that its code runs fastest on.
constexpr FlatRoute flat_route(int k, int m, uint64_t nbytes, bool aligned) {
  if (nbytes < 16) return FlatRoute::kTiny;
  if (fast_shape(k, m)) return aligned ? FlatRoute::kAligned : FlatRoute::kAny;
  if (nbytes <= kTableMinBytes) return FlatRoute::kWide;
  if (any_shape(k, m)) return table_pays(k, m) ? FlatRoute::kAny : FlatRoute::kWide;
  return table_kernel_pays(k, m, nbytes) ? FlatRoute::kTable : FlatRoute::kWide;
}

// Whether the batched encode or decode of a code past the unrolled kernels runs
// on permute tables: where they clearly cost less and enough stripes run to be
// bound by it (us, tables / matrix cores, 100 tensors in 64 KiB units: RS(10,6)
// 293 / 316, RS(20,2) 176 / 192; RS(6,8) 406 / 394, RS(20,4) 216 / 208, RS(24,8)
// 341 / 243, RS(32,16) 588 / 390; RS(10,6) over 5 MB of 16 KiB stripes 25.0 /
// 21.2).  position_bytes: the bytes of each position, all stripes together.
constexpr bool batch_tables_pay(int k, int m) {
  return !fast_shape(k, m) && 4 * table_cost(k, m) <= 3 * core_cost(k, m);
}
constexpr uint64_t kBatchTableBytes = 16u << 20;
constexpr bool batch_tables(int k, int m, uint64_t position_bytes) {
  return batch_tables_pay(k, m) && position_bytes > kBatchTableBytes;
}

// Which kernels some call reaches: the only ones that are instantiated.  Those
// of the matrix cores are shared by the codes with the same kh = ceil(k / 4) and
// mh = ceil(m / 2).
constexpr bool any_reached(int k, int m) {
  return fast_shape(k, m) || (any_shape(k, m) && table_pays(k, m));
}
constexpr bool table_reached(int m) {
  for (int k = 1; k <= EC_MAX_K; ++k)
    if (flat_route(k, m, UINT64_MAX, true) == FlatRoute::kTable) return true;
  return false;
}
constexpr bool core_reached(int kh, int mh) { return !fast_shape(4 * kh, 2 * mh); }
constexpr bool batch_table_reached(int m) {
  for (int k = 1; k <= EC_MAX_K; ++k)
    if (batch_tables_pay(k, m)) return true;
  return false;
}

// Workgroups of one launch at most; more work loops in the kernel.  HIP refuses
// a grid of 2^32 lanes and more.
constexpr uint64_t max_grid(uint64_t lanes) {
  constexpr uint64_t kMax = 1u << 24;
  return kMax * lanes < (1ull << 32) ? kMax : 0xffffffffull / lanes;
}

}  // namespace ec

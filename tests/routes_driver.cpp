// Checks ec::flat_route (megatron-lm_amd/csrc/routes.h) over every shape: the
// kernel of a code past the unrolled ones does not depend on whether its
// shards are whole chunks at aligned addresses, and every route has a kernel
// for the shapes that take it.  Built with g++.
#include <cstdint>
#include <cstdio>

#include "routes.h"

using ec::FlatRoute;

int main() {
  int bad = 0;
  const uint64_t two = ec::kTableMinBytes;
  const uint64_t sizes[] = {1, 15, 16, 4096, two, two + 1, 2 * two, 2 * two + 1, (64u << 20) + 5};
  for (int k = 1; k <= EC_MAX_K; ++k)
    for (int m = 1; m <= EC_MAX_M; ++m)
      for (uint64_t n : sizes) {
        const FlatRoute odd = ec::flat_route(k, m, n, false), even = ec::flat_route(k, m, n, true);
        bool ok = false;
        if (n < 16) ok = odd == FlatRoute::kTiny && even == odd;
        else if (ec::fast_shape(k, m)) ok = odd == FlatRoute::kAny && even == FlatRoute::kAligned;
        else if (even != odd) ok = false;
        else if (odd == FlatRoute::kAny) ok = n > two && ec::any_shape(k, m) && ec::table_pays(k, m);
        else if (odd == FlatRoute::kTable) ok = n > two && !ec::any_shape(k, m) && ec::table_pays(k, m);
        else ok = odd == FlatRoute::kWide;
        // single losses of wide codes and XOR of many shards: tables at any size past the small ones
        if (m == 1 && k > ec::kFastMaxK && n > two) ok = ok && odd == FlatRoute::kTable;
        // a kernel for every route (past any_kernel's one grid its codes go to the matrix cores)
        if (odd == FlatRoute::kAny) ok = ok && ec::any_reached(k, m);
        if (odd == FlatRoute::kTable) ok = ok && ec::table_reached(m);
        if (odd == FlatRoute::kWide || (odd == FlatRoute::kAny && m > ec::kFastMaxM))
          ok = ok && ec::core_reached((k - 1) / 4 + 1, (m - 1) / 2 + 1);
        if (ec::batch_tables(k, m, n)) ok = ok && n > ec::kBatchTableBytes && ec::batch_table_reached(m);
        else if (!ec::fast_shape(k, m)) ok = ok && ec::core_reached((k - 1) / 4 + 1, (m - 1) / 2 + 1);
        if (!ok) {
          std::printf("RS(%d,%d) over %llu bytes: route %d, aligned %d\n", k, m,
                      (unsigned long long)n, (int)odd, (int)even);
          ++bad;
        }
      }
  for (uint64_t lanes = 64; lanes <= 1024; lanes += 64)   // HIP's limit, and one pass over 16 GiB
    if (ec::max_grid(lanes) * lanes >= 1ull << 32 || ec::max_grid(lanes) * lanes < 1u << 30) {
      std::printf("max_grid(%llu) = %llu\n", (unsigned long long)lanes,
                  (unsigned long long)ec::max_grid(lanes));
      ++bad;
    }
  if (bad) return 1;
  std::printf("routes driver ok\n");
  return 0;
}

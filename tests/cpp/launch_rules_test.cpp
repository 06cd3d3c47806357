// Unit test of the host's launch sizes (final184_amd/csrc/launch_rules.hpp).
#include <cstdio>
#include <cstdlib>

#include "../../final184_amd/csrc/launch_rules.hpp"

#define CHECK(c)                                               \
  do {                                                         \
    if (!(c)) {                                                \
      std::printf("CHECK failed line %d: %s\n", __LINE__, #c); \
      std::exit(1);                                            \
    }                                                          \
  } while (0)

using namespace vgi;

int main() {
  const uint32_t precs[] = {VGI_PREC_FP32, VGI_PREC_FP16, VGI_PREC_BF16, VGI_PREC_FP16X2};
  // every trace that a wavefront a block could launch launches: below 2^32 work-items
  for (uint64_t exp = 20; exp < 32; exp++)
    for (int64_t off = -1; off <= 1; off++) {
      const uint64_t blocks = ((1ull << exp) + off * 4) / 64 + (off > 0);
      if (blocks * 64 >= (1ull << 32)) continue;
      for (uint32_t prec : precs)
        for (int sorted = 0; sorted < 2; sorted++)
          for (uint32_t diffuse : {0u, 1u, 9u, 11u, 32u})
            for (uint32_t spec = 0; spec < 2; spec++) {
              const uint32_t w = trace_wavefronts(blocks, diffuse + spec, diffuse, sorted != 0, prec);
              CHECK(w >= 1 && w <= 4);
              CHECK(blocks * 64 * w < (1ull << 32));
              // and no fewer than the rule for smaller launches gives, where they fit
              const uint32_t w0 = trace_wavefronts(1u << 20, diffuse + spec, diffuse, sorted != 0, prec);
              if (blocks >= (1u << 20)) CHECK(w == w0 || blocks * 64 * (w + 1) >= (1ull << 32));
            }
    }
  CHECK(trace_wavefronts((1u << 24) - 1, 10, 9, true, VGI_PREC_FP16) == 4);
  CHECK(trace_wavefronts(1u << 24, 10, 9, true, VGI_PREC_FP16) == 3);
  CHECK(trace_wavefronts((1u << 26) - 1, 10, 9, true, VGI_PREC_FP16) == 1);
  CHECK(trace_wavefronts(0, 10, 9, false, VGI_PREC_FP32) >= 1);
  // the overflow path, which runs on the same workgroups, has at least one a CU
  for (uint64_t seen : {0ull, 1ull, 8ull, 100ull, 171ull, 172ull, 5000ull, 1ull << 30})
    for (uint64_t cap : {1ull, 65ull, 1100ull, 1ull << 31}) {
      const uint32_t g = voxelize_workgroups(seen, cap, 256);
      CHECK(g >= 256);
      CHECK(g <= 256 || g <= cap);
      if (seen && seen <= cap) CHECK(g >= seen);
    }
  CHECK(voxelize_workgroups(0, 1ull << 20, 256) == 2048 && voxelize_workgroups(800, 1ull << 20, 256) == 964);
  std::printf("LAUNCH RULES OK\n");
  return 0;
}

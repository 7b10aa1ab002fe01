// Host-only check of the builds' plan (ps_plan): what it accepts has room for
// uniform keys -- in the groups, in the bytes that count 32 neighbouring
// quotients -- so a build is handed over for its keys, not for its size.
// Built with hipcc for the host alone by tests/test_build_plan.py; prints
// "build plans ok" when nothing failed.
#include <cmath>
#include <cstdio>

#include "../../gpuquotientfilters_amd/csrc/gqf_dbuild.hpp"

using namespace gqf;

static int fails = 0;
static void fail(const char* what, uint64_t n, uint32_t q) {
  if (++fails <= 10) std::printf("FAIL %s n=%llu q=%u\n", what, (unsigned long long)n, q);
}

int main() {
  for (uint32_t sparse : {PS_SPARSE_SQF, PS_SPARSE_RSQF})
    for (uint32_t q = 18; q <= 28; ++q)
      for (uint32_t r = 4; r <= 9; ++r)
        for (double load = 0.01; load < 40; load *= 1.02) {
          const uint64_t n = (uint64_t)(load * (double)(1ull << q));
          PsPlan p;
          if (!ps_plan(n, q, r, sparse, &p)) {
            // ordinary loads of the sizes that the form is for stay accepted
            if (q >= 22 && q <= 26 && r <= 8 && load >= 0.25 && load <= 0.95 && n > 256 * 7600) fail("refused", n, q);
            continue;
          }
          const double mean = (double)n / p.ngroups, block = 32.0 * (double)n / (double)(1ull << q);
          if (mean + 3 * std::sqrt(mean) > p.cap) fail("no room in a group", n, q);
          if (block + 3 * std::sqrt(block) > 255) fail("too many keys in 32 quotients", n, q);
          if (p.cap > PS_TILE || p.cap % 64 || p.tile > PS_TILE || (uint64_t)p.ngroups << p.qb != 1ull << q)
            fail("geometry", n, q);
        }
  if (!fails) std::printf("build plans ok\n");
  return fails ? 1 : 0;
}

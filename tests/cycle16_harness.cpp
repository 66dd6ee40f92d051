// The digit form of composed cycle maps (eithot_amd/csrc/plan.cpp:
// cycle_digits) and the kernel's arithmetic on it (cycle.hip), evaluated on
// the host for the CPU tests; compiled by the test with hipcc, never part of
// the product.
#include "../eithot_amd/csrc/maps.hpp"
#include "../eithot_amd/csrc/plan.cpp"

using namespace eithot;

// Over every step-th of the N positions: the digit permutations of `n` maps
// (bc, R, C, m each) against the maps.  Returns how many there are (0: none),
// or -1 - p at the first position p that differs.
extern "C" int64_t c16_digits(int n, const int64_t* maps, int64_t N, int64_t step) {
  CycleTable t;
  for (int k = 0; k < n; ++k) t.maps.push_back({maps[4 * k], maps[4 * k + 1], maps[4 * k + 2], maps[4 * k + 3]});
  cycle_digits(t, N);
  if (t.digits.size() > t.maps.size()) return -1;
  for (int64_t p = 0; p < N && !t.digits.empty(); p += step) {
    uint64_t q = (uint64_t)p;
    for (size_t k = t.maps.size(); k-- > 0;) {
      const CycleMap& M = t.maps[k];
      const uint64_t b = q / M.bc, r = q - b * M.bc, c = r / M.m, x = r - c * M.m;
      const uint64_t j = c / M.R, i = c - j * M.R;
      q = b * M.bc + (i * M.C + j) * M.m + x;
    }
    uint32_t s = (uint32_t)p;
    for (const CycleDigits& d : t.digits) {
      uint64_t prod = 1;
      const uint32_t in = s;
      s = 0;
      for (int k = 0; k < d.n; ++k) {
        const uint32_t w = d.stride[k] - (k ? d.radix[k - 1] * d.stride[k - 1] : 0);
        FD31 f;
        if (k) f.init((uint32_t)prod);
        s += (k ? f.div(in) : in) * w;
        prod *= d.radix[k];
      }
      if ((int64_t)prod != N) return -1 - p;
    }
    if (s != q) return -1 - p;
  }
  return (int64_t)t.digits.size();
}

// The first x < 2^31 of those given, near multiples of d and random, whose
// division by d in two instructions is wrong; -1: none.
extern "C" int64_t c16_div(uint32_t d, int n, const uint32_t* x) {
  FD31 f;
  f.init(d);
  for (int k = 0; k < n; ++k) {
    const uint32_t m = x[k] / d * d;
    for (uint32_t v : {x[k], m, m ? m - 1 : 0, 0x7fffffffu})
      if (f.div(v) != v / d) return v;
  }
  return -1;
}

// The first cell size in [16, n) whose groups are not whole items: more than
// 64 lanes of 16 bytes, or a last group under 16 bytes; -1: none.
extern "C" int64_t c16_groups(uint32_t n) {
  for (uint32_t U = 16; U < n; ++U) {
    const uint32_t G = cycle_cell_group(U);
    if (G < 16 || G > 1024 || G > U || (U % G && U % G < 16)) return U;
  }
  return -1;
}

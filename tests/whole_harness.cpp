// Host emulation of the whole-permutation passes (eithot_amd/csrc/whole.hip)
// for the CPU tests: the planner's geometry and the kernels' index
// arithmetic, with every access checked against its buffer.  Compiled by the
// test with hipcc, never part of the product.
#include <cstdint>
#include <cstring>
#include <vector>

#include "../eithot_amd/csrc/whole_plan.cpp"

using namespace eithot;

namespace {

struct Emu {
  const WholeGeom& g;
  uint8_t* data;
  uint64_t end;
  bool bad = false;

  // the tile's input runs, 16-byte chunks as the kernel moves them
  std::vector<uint8_t> load(uint32_t tau, uint64_t region) {
    std::vector<uint8_t> lds(g.lds_tile, 0xEE);
    const WholeTile x = whole_tile(g, tau);
    const uint32_t run = whole_len_in(g, x) * g.w;
    for (uint32_t t = 0; t < g.nin * g.fcin.d; ++t) {
      const uint32_t rho = g.fcin.div(t), c = (t - rho * g.fcin.d) * 16;
      uint32_t rel;
      if (!whole_in_run(g, x, rho, &rel) || c >= run) continue;
      const uint64_t off = region + x.in + rel;
      const uint32_t at = whole_row(g, rho) + c;
      if (off + run > end || at + 16 > lds.size() || (at % (g.w > 4 ? g.w : 4))) {
        bad = true;
        return lds;
      }
      for (uint32_t b = 0; b < 16; ++b)
        lds[at + b] = off + c + b < end ? data[off + c + b] : 0;
    }
    return lds;
  }
  void store(uint32_t tau, uint64_t region, const std::vector<uint8_t>& lds) {
    const WholeTile x = whole_tile(g, tau);
    const uint32_t len = whole_len_out(g, x), V = 16 / g.w;
    for (uint32_t t = 0; t < g.nout * g.fcout.d; ++t) {
      const uint32_t rho = g.fcout.div(t);
      uint32_t p = (t - rho * g.fcout.d) * V, l, n = V;
      uint32_t rel;
      if (!whole_out_run(g, x, rho, &rel, &l) || p >= len) continue;
      const uint64_t off = region + x.out + rel;
      if (len < V) n = len, p = 0;
      else if (p + V > len) p = len - V;
      for (uint32_t e = 0; e < n; ++e) {
        const uint32_t s = l + (g.jout > 1 ? whole_elem(g, p + e) : whole_elem1(g, p + e));
        const uint64_t o = off + (uint64_t)(p + e) * g.w;
        if (s % g.w || s + g.w > lds.size() || o + g.w > end) {
          bad = true;
          return;
        }
        std::memcpy(data + o, lds.data() + s, g.w);
      }
    }
  }
};

}  // namespace

// Runs the pass plan_whole chooses over `data`; returns its mode, 0 when there is none, -1 on an access out of
// bounds.  *tiles and *lds: its tiles per region and LDS bytes.
extern "C" int wh_run(const int64_t* dims, const int* perm1, int rank, int64_t elem, int cus,
                      int passes, int weak, uint8_t* data, int64_t* tiles, int64_t* lds) {
  const WholePass p = plan_whole(dims, perm1, rank, (size_t)elem, cus, 160 * 1024, passes, weak != 0);
  if (p.mode == WHOLE_NONE) return 0;
  const WholeGeom& g = p.g;
  *tiles = g.tiles;
  *lds = p.lds;
  if (p.lds < whole_lds_bytes(g) || p.lds > 160 * 1024) return -1;
  Emu e{g, data, g.B * g.region};
  std::vector<int> named(g.tiles, 0);  // every tile is some workgroup's, once
  for (uint32_t i = 0; i < g.tiles; ++i) {
    const uint32_t t = whole_nth(g, i);
    if (t >= g.tiles || named[t]++) return -1;
  }
  for (uint64_t b = 0; b < g.B && !e.bad; ++b) {
    const uint64_t region = b * g.region;
    if (p.mode == WHOLE_RESIDENT) {
      std::vector<std::vector<uint8_t>> held;
      for (uint32_t t = 0; t < g.tiles && !e.bad; ++t) held.push_back(e.load(t, region));
      for (uint32_t t = g.tiles; t-- > 0 && !e.bad;) e.store(t, region, held[t]);
      continue;
    }
    if ((int64_t)g.nin * g.fcin.d > (int64_t)p.threads * kWholeHold) return -1;
    for (uint32_t first = 0; first < g.tiles && !e.bad; ++first) {
      bool leads = true;
      for (uint32_t q = whole_tile(g, first).next; q != first; q = whole_tile(g, q).next)
        leads = leads && q > first;
      if (!leads) continue;
      uint32_t x = first;
      std::vector<uint8_t> held = e.load(x, region);
      for (uint32_t y = whole_tile(g, x).next; y != first && !e.bad; y = whole_tile(g, y).next) {
        std::vector<uint8_t> next = e.load(y, region);
        e.store(x, region, held);
        held.swap(next);
        x = y;
      }
      if (!e.bad) e.store(x, region, held);
    }
  }
  return e.bad ? -1 : p.mode;
}

// Whole-permutation passes: a tensor transposed by ONE kernel that reads and
// writes every byte once, instead of the plan's sequence of passes.
//
// The tensor is cut into tiles: a tile holds t[k] consecutive indices of
// every dim k, so that it is made of runs contiguous in the input layout and
// also of runs contiguous in the output layout.  A workgroup loads a tile
// along its input runs into LDS and stores it along its output runs.  Two
// forms differ in when a store may overwrite what other tiles still read:
//
//  * orbit (WHOLE_ORBIT): the dims' lengths and tile lengths read the same in
//    input and output order (d[perm[k]] == d[k]: a square matrix, a reversed
//    (a, b, b, a), ...).  Output tiles then lie exactly where input tiles
//    lie, so the tiles form cycles, each moved by one workgroup.
//  * resident (WHOLE_RESIDENT): the tensor is a batch of regions, each small
//    enough that all its tiles are held in the LDS of the chip at once.  The
//    region's workgroups load their tiles, meet at a counter in device
//    memory, and store.
//
// This header holds the geometry and the index arithmetic, shared by the
// kernels, the planner and the CPU tests.
#pragma once

#include <cstdint>
#include <vector>

#include "maps.hpp"

namespace eithot {

constexpr int kWholeDims = 8;
constexpr int kWholeHold = 8;  // 16-byte loads one thread holds (orbit)
constexpr uint32_t kWholeRegions = 16384;  // regions of one resident pass, at most

enum WholeMode : int { WHOLE_NONE = 0, WHOLE_ORBIT = 1, WHOLE_RESIDENT = 2 };

struct WholeGeom {
  uint32_t r = 0;                // dims, input order, fastest first
  uint32_t w = 0;                // element bytes (a power of two, at most 16)
  uint32_t jin = 0, jout = 0;    // dims in an input run / an output run
  uint32_t len_in = 0, len_out = 0;  // elements of a run of a full tile
  uint32_t nin = 0, nout = 0;    // runs of a full tile
  uint32_t rs = 0;               // LDS bytes from one input run to the next
  uint32_t vl = 31, g2 = 0;      // g2 further bytes after every 2^vl input runs
  uint32_t lds_tile = 0;         // LDS bytes of the tile's elements
  uint32_t tiles = 0;            // tiles per region
  uint32_t dst_stride[kWholeDims] = {0};  // orbit: tile index step of block coordinate k, moved
  uint32_t d[kWholeDims], t[kWholeDims];   // extent; tile extent
  uint32_t ls[kWholeDims];                 // LDS bytes per index
  uint64_t gin[kWholeDims], gout[kWholeDims];  // bytes per index, input / output layout
  uint32_t odim[kWholeDims];               // output order: input dim of output dim k
  uint32_t ot[kWholeDims], ols[kWholeDims];  // t and ls in output order
  uint64_t ogout[kWholeDims];              // gout in output order
  FD32 fnb[kWholeDims];                    // tiles along dim k
  FD32 ft[kWholeDims], oft[kWholeDims];    // tile extents, input and output order
  FD32 fcin, fcout;                        // 16-byte chunks per run
  FD32 ftiles;
  uint32_t per = 1, wgs = 0;     // resident: tiles one workgroup holds (1 or 2), workgroups per region
  FD32 fwgs;
  // Order in which workgroups take a matrix's tiles: along dim 0 within
  // groups of sg tiles (the last group: slast), then along dim 1, then the
  // next group.  sg = 0: index order.
  uint32_t sg = 0, sna = 1, slast = 1;  // sna: tiles along dim 0
  FD32 fsgroup, fsg, fslast;
  uint64_t region = 0, B = 1;              // bytes per region, regions
};

struct WholePass {
  int mode = WHOLE_NONE;
  int threads = 256;
  int64_t lds = 0;  // LDS bytes per workgroup
  WholeGeom g;
};

// LDS layout of a workgroup: control words, the input runs' byte offsets from
// the tile's first element, the output runs' (offset, LDS offset) pairs, the
// LDS offsets of one output run's elements (runs over several dims only), the
// tile.  Offsets are 32-bit: the planner takes no tile that spans 4 GB.
constexpr uint32_t kWholeCtl = 16;
EH_HD uint32_t whole_in_bytes(const WholeGeom& g) { return (g.nin * 4 + 15) / 16 * 16; }
EH_HD uint32_t whole_out_bytes(const WholeGeom& g) { return (g.nout * 8 + 15) / 16 * 16; }
EH_HD uint32_t whole_otab_bytes(const WholeGeom& g) {
  return g.jout > 1 ? (g.len_out * 4 + 15) / 16 * 16 : 0;
}
EH_HD uint32_t whole_lds_bytes(const WholeGeom& g) {
  return kWholeCtl + whole_in_bytes(g) + whole_out_bytes(g) + whole_otab_bytes(g) + g.lds_tile;
}

// Tile index of the i-th tile in the order that workgroups take them.
EH_HD uint32_t whole_nth(const WholeGeom& g, uint32_t i) {
  if (!g.sg) return i;
  const uint32_t grp = g.fsgroup.div(i), in = i - grp * g.fsgroup.d;
  const bool last = (grp + 1) * g.sg > g.sna;
  const uint32_t y = last ? g.fslast.div(in) : g.fsg.div(in);
  return grp * g.sg + (in - y * (last ? g.slast : g.sg)) + y * g.sna;
}

// One tile: the extents it has (short at the far edges) and the byte offsets
// of its first element within the region, input and output layout.  The
// functions take the most dims they handle as ND: kernels instantiated for
// few dims keep the others' constants out of their scalar registers.
struct WholeTile {
  uint32_t ext[kWholeDims];
  uint64_t in, out;
  uint32_t next;  // orbit: the tile whose place the transposed tile takes
};
template <int ND = kWholeDims>
EH_HD WholeTile whole_tile(const WholeGeom& g, uint32_t tau) {
  WholeTile x;
  x.in = x.out = 0;
  x.next = 0;
#pragma unroll
  for (int k = 0; k < ND; ++k) {
    x.ext[k] = 1;
    if (k < (int)g.r) {
      const uint32_t q = g.fnb[k].div(tau);
      const uint32_t c = tau - q * g.fnb[k].d;
      tau = q;
      const uint32_t o = c * g.t[k];
      const uint32_t left = g.d[k] - o;
      x.ext[k] = left < g.t[k] ? left : g.t[k];
      x.in += (uint64_t)o * g.gin[k];
      x.out += (uint64_t)o * g.gout[k];
      x.next += c * g.dst_stride[k];
    }
  }
  return x;
}

// Elements of this tile's input (output) runs.
template <int ND = kWholeDims>
EH_HD uint32_t whole_len_in(const WholeGeom& g, const WholeTile& x) {
  uint32_t n = 1;
#pragma unroll
  for (int k = 0; k < ND; ++k)
    if (k < (int)g.jin) n *= x.ext[k];
  return n;
}
template <int ND = kWholeDims>
EH_HD uint32_t whole_len_out(const WholeGeom& g, const WholeTile& x) {
  uint32_t n = 1;
#pragma unroll
  for (int k = 0; k < ND; ++k) {
    bool in = false;
#pragma unroll
    for (int j = 0; j < ND; ++j) in = in || (j < (int)g.jout && g.odim[j] == (uint32_t)k);
    if (in) n *= x.ext[k];
  }
  return n;
}

// Byte offset of input run rho from the tile's first element; false when the
// tile is short of it.  Runs number the indices of dims jin.. (radix t).
template <int ND = kWholeDims>
EH_HD bool whole_in_run(const WholeGeom& g, const WholeTile& x, uint32_t rho, uint32_t* off) {
  uint32_t a = 0;
  bool ok = true;
#pragma unroll
  for (int k = 0; k < ND; ++k)
    if (k >= (int)g.jin && k < (int)g.r) {
      const uint32_t q = g.ft[k].div(rho);
      const uint32_t i = rho - q * g.t[k];
      rho = q;
      ok = ok && i < x.ext[k];
      a += i * (uint32_t)g.gin[k];
    }
  *off = a;
  return ok;
}
// LDS offset of input run rho.
EH_HD uint32_t whole_row(const WholeGeom& g, uint32_t rho) { return rho * g.rs + (rho >> g.vl) * g.g2; }

// Byte offset of output run rho in the output layout and the LDS offset of
// its first element.
template <int ND = kWholeDims>
EH_HD bool whole_out_run(const WholeGeom& g, const WholeTile& x, uint32_t rho, uint32_t* off,
                         uint32_t* lds) {
  uint32_t a = 0;
  uint32_t l = 0;
  bool ok = true;
#pragma unroll
  for (int k = 0; k < ND; ++k)
    if (k >= (int)g.jout && k < (int)g.r) {
      const uint32_t q = g.oft[k].div(rho);
      const uint32_t i = rho - q * g.ot[k];
      rho = q;
      uint32_t e = 1;
#pragma unroll
      for (int j = 0; j < ND; ++j) e = g.odim[k] == (uint32_t)j ? x.ext[j] : e;
      ok = ok && i < e;
      a += i * (uint32_t)g.ogout[k];
      l += i * g.ols[k];
    }
  *off = a;
  *lds = l;
  return ok;
}
// LDS offset of element p of an output run from the run's first element:
// runs over one dim, and over several (mixed radix over the run's dims, of
// which all but the last are whole).
EH_HD uint32_t whole_elem1(const WholeGeom& g, uint32_t p) { return p * g.ols[0] + (p >> g.vl) * g.g2; }
template <int ND = kWholeDims>
EH_HD uint32_t whole_elem(const WholeGeom& g, uint32_t p) {
  uint32_t l = 0;
#pragma unroll
  for (int k = 0; k < ND; ++k)
    if (k < (int)g.jout) {
      const uint32_t q = g.oft[k].div(p);
      l += (p - q * g.ot[k]) * g.ols[k];
      p = q;
    }
  return l;
}

// Where resident passes meet: per region kWholeSubs counters, a root counter
// (zero between passes) and a word that the region's last workgroup steps.
constexpr uint32_t kWholeSubs = 16;
struct WholeCtl {
  uint32_t* failed = nullptr;  // set by a workgroup that gave up waiting
  uint32_t *open = nullptr, *root = nullptr, *sub = nullptr;
  uint32_t slots = 0;                // regions the words serve
  uint64_t patience = 0;             // ticks of the 100 MHz clock
  uint32_t* host_failed = nullptr;   // pinned host word, set along with *failed
};
constexpr uint64_t whole_ctl_words(uint32_t slots) { return 32 + (uint64_t)slots * (2 + kWholeSubs); }
inline void whole_ctl_at(WholeCtl& c, uint32_t* words, uint32_t slots) {
  c.failed = words;
  c.open = words + 32;
  c.root = c.open + slots;
  c.sub = c.root + slots;
  c.slots = slots;
}

// Plans the whole-permutation pass of a tensor (perm1 1-based) for a chip of
// `cus` CUs with lds_max bytes of LDS each; mode WHOLE_NONE when neither
// form fits.  `passes` is the pass count of the tensor's ordinary plan, and
// `weak` whether its only pass, when there is one, is worth replacing.
WholePass plan_whole(const int64_t* dims, const int* perm1, int rank, size_t elem, int cus,
                     int64_t lds_max, int passes, bool weak);

// The resident pass of a tensor among many in one launch: 32 KiB tiles,
// workgroups of kWholeBatchThreads.
constexpr int kWholeBatchThreads = 512;
WholePass plan_whole_batched(const int64_t* dims, const int* perm1, int rank, size_t elem, int cus,
                             int64_t lds_max);

}  // namespace eithot

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
//    memory, and store.  Where they do not meet (the chip is shared), none
//    stores and the last one moves the region alone.
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
  uint32_t od[kWholeDims], ogin[kWholeDims];  // resident: extents and gin in output order
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

// Byte offset in a region's input layout of element o of its output layout
// (r dims; WholeGeom's od and ogin).
EH_HD uint32_t whole_source(uint32_t r, const uint32_t* od, const uint32_t* ogin, uint32_t o) {
  uint32_t a = 0;
#pragma unroll
  for (int k = 0; k < kWholeDims; ++k)
    if (k < (int)r) {
      const uint32_t q = o / od[k];
      a += (o - q * od[k]) * ogin[k];
      o = q;
    }
  return a;
}

// ---------------------------------------------------------------------------
// Meeting of a region's workgroups.
//
// The workgroups that load a region must all be on the chip before one of
// them may store.  Nothing guarantees that: other processes' workgroups, or a
// stream that sees part of the chip, can keep the missing ones out for as
// long as the present ones wait.  So a wait is bounded, and ends in ONE
// decision for the region, taken by a compare-and-swap on its word: either
// the last workgroup to arrive opens the region and all of them store, or one
// that has waited long enough calls the pass off and none of them does.  All
// workgroups still arrive once (those that start later too), and the last
// one to arrive at a region called off finds it as it was, with everybody
// else gone or leaving, and moves it alone through host memory.
//
// Per region: kWholeSubs counters and a root counter (zero between passes)
// and the word, 4 * passes + flags.  For all regions of a device: the time
// of the last pass called off, for a while after which workgroups wait less
// (what kept one region's workgroups apart keeps the next one's), and a lock
// on the host memory.
// ---------------------------------------------------------------------------
constexpr uint32_t kWholeSubs = 16;
constexpr uint32_t kCalledOff = 1;   // this pass of the region
constexpr uint32_t kWasCalledOff = 2;  // the one before
struct WholeCtl {
  uint32_t *open = nullptr, *root = nullptr, *sub = nullptr;
  uint32_t slots = 0;            // regions these words serve
  uint32_t* recent = nullptr;    // time of the last pass called off, 2^20 ticks
  uint32_t* lock = nullptr;      // 1: a workgroup uses `room`
  char* room = nullptr;          // pinned host memory, as large as the largest region
  uint64_t patience = 0;         // ticks of the 100 MHz clock
};
constexpr uint64_t whole_ctl_words(uint32_t slots) { return (uint64_t)slots * (2 + kWholeSubs); }
inline void whole_ctl_at(WholeCtl& c, uint32_t* words, uint32_t slots) {
  c.open = words;
  c.root = c.open + slots;
  c.sub = c.root + slots;
  c.slots = slots;
}

enum WholeMeet : uint32_t { MEET_STORE = 0, MEET_LEAVE = 1, MEET_ALONE = 2 };

// W gives the words: add, get, set, cas (true when it swapped), now (ticks),
// pause.  The counters are spread (each on a line of its own: one address
// takes about 30 ns per addition).
template <class W>
EH_HD bool whole_arrive(const WholeCtl& c, uint32_t slot, uint32_t t, uint32_t n) {
  const uint32_t subs = n <= kWholeSubs ? 1 : kWholeSubs;
  const uint32_t j = t % subs, members = (n - j + subs - 1) / subs;
  uint32_t* sub = c.sub + (uint64_t)j * c.slots + slot;
  if (W::add(sub, 1) != members - 1) return false;
  W::set(sub, 0);
  if (subs == 1) return true;
  if (W::add(c.root + slot, 1) != subs - 1) return false;
  W::set(c.root + slot, 0);
  return true;
}

// What workgroup t of the region's n does, having loaded its part; `word` is
// the region's word as it was before it arrived.
template <class W>
EH_HD WholeMeet whole_meet(const WholeCtl& c, uint32_t slot, uint32_t t, uint32_t n, uint32_t word) {
  uint32_t* open = c.open + slot;
  if (whole_arrive<W>(c, slot, t, n))
    return !(word & kCalledOff) && W::cas(open, word, (word | 3) + 1) ? MEET_STORE : MEET_ALONE;
  if (word & kCalledOff) return MEET_LEAVE;
  const uint64_t t0 = W::now();
  // a second after a pass was called off: 1 ms at most
  const bool soon = (uint32_t)(t0 >> 20) - W::get(c.recent) < 96;
  const uint64_t patience = soon && c.patience > 100000 ? 100000 : c.patience;
  for (;;) {
    const uint32_t now = W::get(open);
    if ((now | 3) != (word | 3)) return now & kWasCalledOff ? MEET_LEAVE : MEET_STORE;
    if (now & kCalledOff) return MEET_LEAVE;
    if (W::now() - t0 > patience) {
      if (W::cas(open, word, word | kCalledOff)) {
        W::set(c.recent, (uint32_t)(W::now() >> 20));
        return MEET_LEAVE;
      }
    } else {
      W::pause();
    }
  }
}

// Ends a pass that MEET_ALONE's workgroup has done.
template <class W>
EH_HD void whole_done_alone(uint32_t* open, uint32_t word) {
  W::set(open, ((word | 3) + 1) | kWasCalledOff);
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

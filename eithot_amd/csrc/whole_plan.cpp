// Geometry of the whole-permutation passes (whole.hpp): which tensors one
// pass can move, and the tiles it moves them in.  Host code only.
#include "whole.hpp"

#include <algorithm>

namespace eithot {
namespace {

// A tensor's permutation with unit dims dropped, dims adjacent in both
// orders merged, a leading dim that stays in front folded into the element
// (cut into words of w bytes again) and a trailing dim that stays last taken
// as the batch.
struct Canon {
  std::vector<int64_t> d;
  std::vector<int> p;  // output dim k is input dim p[k]
  int64_t B = 1;
  uint32_t w = 1;
};

bool canonical(const int64_t* dims, const int* perm1, int rank, size_t elem, Canon& c) {
  std::vector<int> id(rank, -1), order;
  std::vector<int64_t> d;
  for (int i = 0; i < rank; ++i)
    if (dims[i] > 1) {
      id[i] = (int)d.size();
      d.push_back(dims[i]);
    }
  for (int k = 0; k < rank; ++k)
    if (id[perm1[k] - 1] >= 0) order.push_back(id[perm1[k] - 1]);
  std::vector<int> head(d.size(), 1), run(d.size());
  for (size_t k = 0; k + 1 < order.size(); ++k)
    if (order[k + 1] == order[k] + 1) head[order[k + 1]] = 0;
  for (size_t a = 0; a < d.size(); ++a) {
    if (head[a]) c.d.push_back(1);
    run[a] = (int)c.d.size() - 1;
    c.d.back() *= d[a];
  }
  for (int a : order)
    if (head[a]) c.p.push_back(run[a]);
  int64_t unit = (int64_t)elem;
  if (!c.p.empty() && c.p[0] == 0) {
    unit *= c.d[0];
    c.d.erase(c.d.begin());
    c.p.erase(c.p.begin());
    for (int& v : c.p) --v;
  }
  if (!c.p.empty() && c.p.back() == (int)c.d.size() - 1) {
    c.B = c.d.back();
    c.d.pop_back();
    c.p.pop_back();
  }
  if (c.d.size() < 2) return false;
  while (c.w < 16 && unit % (c.w * 2) == 0) c.w *= 2;
  if (unit > (int64_t)c.w) {
    c.d.insert(c.d.begin(), unit / c.w);
    for (int& v : c.p) ++v;
    c.p.insert(c.p.begin(), 0);
  }
  if (c.d.size() > (size_t)kWholeDims) return false;
  for (int64_t v : c.d)
    if (v >= (1ll << 31)) return false;
  return true;
}

uint32_t chunks(uint64_t elems, uint32_t w) { return (uint32_t)((elems * w + 15) / 16); }

// Every field of g but tiles of unequal places (dst_stride); false when the
// numbers leave their types.
bool build(const Canon& c, const std::vector<int64_t>& t, WholeGeom& g) {
  g = WholeGeom();
  const uint32_t r = (uint32_t)c.d.size();
  g.r = r;
  g.w = c.w;
  g.B = (uint64_t)c.B;
  uint64_t s = c.w;
  uint64_t ntile = 1;
  for (uint32_t k = 0; k < (uint32_t)kWholeDims; ++k) {
    g.d[k] = k < r ? (uint32_t)c.d[k] : 1;
    g.t[k] = k < r ? (uint32_t)t[k] : 1;
    g.gin[k] = k < r ? s : 0;
    s *= g.d[k];
    g.ft[k].init(g.t[k]);
    const uint64_t nb = (g.d[k] + g.t[k] - 1) / g.t[k];
    g.fnb[k].init(nb);
    ntile *= nb;
    if (ntile >= (1ull << 31)) return false;
  }
  g.region = s;
  g.tiles = (uint32_t)ntile;
  g.ftiles.init(ntile);
  uint64_t so = c.w;
  for (uint32_t k = 0; k < (uint32_t)kWholeDims; ++k) {
    g.gout[k] = 0;
    g.odim[k] = k;
  }
  for (uint32_t k = 0; k < r; ++k) {
    g.odim[k] = (uint32_t)c.p[k];
    g.gout[c.p[k]] = so;
    so *= g.d[c.p[k]];
  }
  // runs: leading dims that the tile holds whole, and the next one's part
  g.jin = g.jout = 1;
  // (an input run of whole 16-byte chunks ends there: the next one follows it
  // in memory all the same, and LDS rows are padded between runs)
  uint64_t in_bytes = (uint64_t)g.t[0] * g.w;
  while (g.jin < r && g.t[g.jin - 1] == g.d[g.jin - 1] && g.t[g.jin] > 1 &&
         !(in_bytes % 16 == 0 && in_bytes >= 64))
    in_bytes *= g.t[g.jin++];
  while (g.jout < r && g.t[g.odim[g.jout - 1]] == g.d[g.odim[g.jout - 1]] && g.t[g.odim[g.jout]] > 1)
    ++g.jout;
  uint64_t li = 1, lo = 1, ni = 1, no = 1;
  for (uint32_t k = 0; k < r; ++k) (k < g.jin ? li : ni) *= g.t[k];
  for (uint32_t k = 0; k < r; ++k) (k < g.jout ? lo : no) *= g.t[g.odim[k]];
  if (li * ni * g.w > 160 * 1024) return false;
  g.len_in = (uint32_t)li;
  g.len_out = (uint32_t)lo;
  g.nin = (uint32_t)ni;
  g.nout = (uint32_t)no;
  g.fcin.init(chunks(li, g.w));
  g.fcout.init(chunks(lo, g.w));
  // LDS rows: an odd number of banks apart (whole 16-byte chunks fit, so a
  // run's last chunk may be stored whole), so that the elements of an output
  // run, one row each, lie in different banks.  Elements under 4 bytes are
  // gathered V to a 16-byte store: further bytes after every V rows keep the
  // stores' first elements apart too, when an output run is one dim that
  // starts the rows and is cut at multiples of V.
  const uint32_t gr = g.w > 4 ? g.w : 4, V = 16 / g.w;
  uint32_t rows = (chunks(li, g.w) * 16 + gr - 1) / gr;
  g.rs = (rows | 1) * gr;
  const uint32_t q0 = g.odim[0];
  if (g.w < 4 && g.jout == 1 && q0 == g.jin && g.t[q0] % V == 0) {
    g.vl = g.w == 1 ? 4 : 3;
    g.g2 = gr;
  }
  uint64_t nat = g.w, mul = 1;
  for (uint32_t k = 0; k < (uint32_t)kWholeDims; ++k) {
    if (k >= r) {
      g.ls[k] = 0;
    } else if (k < g.jin) {
      g.ls[k] = (uint32_t)nat;
      nat *= g.t[k];
    } else {
      // rows of dims after the first lie whole groups of V rows apart, so
      // the group padding adds up along with them
      g.ls[k] = (uint32_t)(mul * g.rs + (k > g.jin ? (mul >> g.vl) * g.g2 : 0));
      mul *= g.t[k];
    }
  }
  const uint64_t lt = ni * g.rs + (ni >> g.vl) * g.g2 + 16;
  g.lds_tile = (uint32_t)((lt + 15) / 16 * 16);
  for (uint32_t k = 0; k < (uint32_t)kWholeDims; ++k) {
    const uint32_t a = g.odim[k];
    g.ot[k] = g.t[a];
    g.oft[k].init(g.t[a]);
    g.ols[k] = g.ls[a];
    g.ogout[k] = g.gout[a];
    g.od[k] = g.d[a];
    g.ogin[k] = (uint32_t)g.gin[a];
  }
  // offsets within a tile stay below 4 GB (a 16-byte access past them too)
  unsigned __int128 sin = 64, sout = 64;
  for (uint32_t k = 0; k < r; ++k) {
    sin += (unsigned __int128)g.t[k] * g.gin[k];
    sout += (unsigned __int128)g.t[k] * g.gout[k];
  }
  return lt < 200 * 1024 && sin < (1ull << 32) && sout < (1ull << 32);
}

// Tile extents within `cap` bytes of LDS: the shorter of the input and the
// output run is doubled (its first dim that is not whole) while it fits; an
// extent then shrinks to what its tile count needs, in whole 16-byte chunks
// for the runs' last dims.  Dims of one class keep one extent.  `tight` also
// grows by half where doubling does not fit: fuller tiles, fewer whole lines.
bool choose(const Canon& c, const std::vector<int>& cls, int64_t cap, int64_t max_chunks,
            WholeGeom& g, bool tight = false) {
  const int r = (int)c.d.size();
  std::vector<int64_t> t(r, 1);
  if (!build(c, t, g)) return false;
  auto set = [&](std::vector<int64_t>& v, int k, int64_t x) {
    for (int j = 0; j < r; ++j)
      if (cls[j] == cls[k]) v[j] = x;
  };
  auto run_bytes = [&](bool out) {
    int64_t n = c.w;
    for (int k = 0; k < r; ++k) {
      const int a = out ? c.p[k] : k;
      n *= t[a];
      if (t[a] < c.d[a]) break;
    }
    return n;
  };
  auto grow = [&](bool out) {
    for (int k = 0; k < r; ++k) {
      const int a = out ? c.p[k] : k;
      if (t[a] == c.d[a]) continue;
      for (int64_t f = 8; f > 4; f -= 2) {  // twice, then half as much again
        std::vector<int64_t> v = t;
        set(v, a, std::min<int64_t>(c.d[a], (f * t[a] + 3) / 4));
        WholeGeom h;
        if (v[a] > t[a] && build(c, v, h) && (int64_t)whole_lds_bytes(h) <= cap &&
            (int64_t)h.nin * h.fcin.d <= max_chunks) {
          t = v;
          return true;
        }
        if (!tight) break;
      }
      return false;
    }
    return false;
  };
  for (;;) {
    const bool first = run_bytes(true) < run_bytes(false);
    if (!grow(first) && !grow(!first)) break;
  }
  const int64_t V = 16 / c.w;
  for (int k = 0; k < r; ++k) {
    if (t[k] == c.d[k]) continue;
    const int64_t nb = (c.d[k] + t[k] - 1) / t[k];
    int64_t x = (c.d[k] + nb - 1) / nb;
    // whole 128-byte lines where that leaves the last tile nearly full
    // (7248^2 of 4 bytes: 64 wide 78 us, 48 wide 85 us), else whole chunks
    const int64_t line = std::max<int64_t>(128 / c.w, 1);
    const int64_t xl = (x + line - 1) / line * line;
    if (x > line && xl <= t[k] && nb * xl - c.d[k] <= c.d[k] / 16) x = xl;
    else if (x > V) x = std::min<int64_t>((x + V - 1) / V * V, t[k]);
    set(t, k, x);
  }
  return build(c, t, g) && (int64_t)whole_lds_bytes(g) <= cap &&
         (int64_t)g.nin * g.fcin.d <= max_chunks;
}

// The order of tiles (see WholeGeom::sg), for matrices: groups of 8 columns
// of tiles moved squares 5 to 18 % faster than rows of tiles (7248^2 of 4
// bytes 79.9 -> 75.3 us, 10001^2 of 1 byte 70 -> 57 us; groups of 4 and 16
// lie between).  With further dims in between, index order is the faster one
// ((96, 75, 75, 96) reversed: 122 us, 156 us in groups).
void order_tiles(WholeGeom& g) {
  const uint32_t na = g.fnb[0].d, nb = g.fnb[1].d;
  if (g.r != 2 || na < 2 || nb < 2) return;
  constexpr uint32_t G = 8;
  g.sg = G;
  g.sna = na;
  g.slast = na % G ? na % G : G;
  g.fsgroup.init((uint64_t)G * nb);
  g.fsg.init(G);
  g.fslast.init(g.slast);
}

void per_workgroup(WholeGeom& g, uint32_t per) {
  g.per = per;
  g.wgs = (g.tiles + per - 1) / per;
  g.fwgs.init(g.wgs);
}

int64_t short_run(const WholeGeom& g) { return (int64_t)std::min(g.len_in, g.len_out) * g.w; }

}  // namespace

WholePass plan_whole_batched(const int64_t* dims, const int* perm1, int rank, size_t elem, int cus,
                             int64_t lds_max) {
  WholePass none, w;
  Canon c;
  if (!canonical(dims, perm1, rank, elem, c) || c.B > (int64_t)kWholeRegions) return none;
  std::vector<int> cls(c.d.size());
  for (size_t k = 0; k < cls.size(); ++k) cls[k] = (int)k;
  // of every workgroup of the launch: three of 512 threads to a CU.  512
  // tensors of 1.5 GB took 1115 us, with two larger ones to a CU 1157, with
  // three of 384 or 256 threads 1210 and 1396, with four 1190 (38 KiB, 256
  // threads; 1303 of 512); 40 tensors 148 us, 192, 153 and 200, and 200
  constexpr int64_t kLds = 52 * 1024;
  if (kLds > lds_max || !choose(c, cls, kLds, kWholeBatchThreads * kWholeHold, w.g, true)) return none;
  // large regions: two tiles per workgroup, so that fewer of them wait for
  // the rest of their region to start
  per_workgroup(w.g, w.g.tiles > 16 ? 2 : 1);
  const int64_t slots = (int64_t)cus * std::min<int64_t>(lds_max / kLds, 2048 / kWholeBatchThreads);
  if ((int64_t)w.g.wgs > slots / 2 || short_run(w.g) < 32) return none;
  w.threads = kWholeBatchThreads;
  w.lds = (whole_lds_bytes(w.g) + 127) / 128 * 128;
  w.mode = WHOLE_RESIDENT;
  order_tiles(w.g);
  return w;
}

WholePass plan_whole(const int64_t* dims, const int* perm1, int rank, size_t elem, int cus,
                     int64_t lds_max, int passes, bool weak) {
  WholePass none, w;
  Canon c;
  if (!canonical(dims, perm1, rank, elem, c)) return none;
  const int r = (int)c.d.size();
  if (passes < 2 && !weak) return none;

  struct Step {
    int64_t lds;  // KiB
    int threads;
    uint32_t per;
  };
  constexpr Step kSteps[] = {{6, 256, 1},  {10, 256, 1},  {19, 256, 1},  {38, 256, 1},
                             {78, 512, 2}, {156, 1024, 2}};
  // resident: tiles as small as keeps the workgroups of a small tensor below
  // three per CU (77 KB: 17 -> 9.5 us, 4.4 MB: 33 -> 13 us, 1 MB of bytes:
  // 59 -> 10 us against the ordinary passes; meeting costs 2 to 5 us), and
  // 64 KiB tiles, two workgroups per CU and a second tile of each in
  // registers, for larger ones and batches (210 MB in regions of 3.6 MB:
  // 158 -> 100 us; one tile each 114, 32 KiB tiles 99, but 38 instead of 43 us
  // for 52 MB of bytes and 121 instead of 117 for 236 MB; 128 KiB 130).  A
  // region takes at most half of the workgroups the chip holds: the others'
  // room is for what else runs, so that its workgroups meet soon.
  if (c.B <= (int64_t)kWholeRegions) {
    std::vector<int> cls(r);
    for (int k = 0; k < r; ++k) cls[k] = k;
    for (const Step& st : kSteps) {
      if (st.lds * 1024 > lds_max) break;
      if (!choose(c, cls, st.lds * 1024, st.threads * kWholeHold, w.g)) continue;
      const int64_t lds = (whole_lds_bytes(w.g) + 127) / 128 * 128;
      const int64_t slots = (int64_t)cus * std::min<int64_t>(lds_max / lds, 2048 / st.threads);
      per_workgroup(w.g, st.per);
      if ((int64_t)w.g.wgs > slots / 2) continue;
      if (st.lds <= 38 && c.B * (int64_t)w.g.tiles > 3 * cus) continue;
      const bool big = (uint64_t)c.B * w.g.region > (64ull << 20);
      if (short_run(w.g) < (big ? 128 : 32)) continue;
      w.threads = st.threads;
      w.lds = lds;
      w.mode = WHOLE_RESIDENT;
      order_tiles(w.g);
      break;
    }
  }

  // orbit: every dim of a cycle of the permutation has one length
  bool alike = passes >= 2;
  for (int k = 0; k < r; ++k) alike = alike && c.d[c.p[k]] == c.d[k];
  if (alike) {
    std::vector<int> cls(r, -1);
    for (int k = 0; k < r; ++k)
      for (int j = k; cls[j] < 0; j = c.p[j]) cls[j] = k;
    WholePass o;
    if (choose(c, cls, 38 * 1024, 512 * kWholeHold, o.g)) {
      std::vector<int> inv(r);
      for (int k = 0; k < r; ++k) inv[c.p[k]] = k;
      uint32_t nbs[kWholeDims], s = 1;
      for (int k = 0; k < r; ++k) {
        nbs[k] = s;
        s *= o.g.fnb[k].d;
      }
      for (int k = 0; k < r; ++k) o.g.dst_stride[k] = nbs[inv[k]];
      const int64_t slots = (int64_t)o.g.nin * o.g.fcin.d;  // 16-byte loads of a tile
      o.threads = (int)std::min<int64_t>(512, std::max<int64_t>(64, ((slots + 7) / 8 + 63) / 64 * 64));
      o.lds = (whole_lds_bytes(o.g) + 127) / 128 * 128;
      o.mode = WHOLE_ORBIT;
      order_tiles(o.g);
      // runs that end with a short whole dim lie far apart in one of the
      // layouts: 128 to 256 bytes of them cost more than two ordinary passes
      // ((32, 15, 15, 15, 15, 32) reversed: 159 us, 216 here); 384 bytes, or
      // parts of a longer dim, cost less ((96, 75, 75, 96): 153 -> 102 us,
      // 384 x 384 matrices: 135 -> 73 us)
      const int64_t run = short_run(o.g);
      const bool whole_dim = o.g.t[0] == o.g.d[0] || o.g.ot[0] == o.g.d[o.g.odim[0]];
      const bool several = o.g.jin > 1 || o.g.jout > 1;
      if (slots <= (int64_t)o.threads * kWholeHold && (uint64_t)o.g.tiles * o.g.B < (1ull << 31) &&
          run >= (several ? 512 : whole_dim ? 256 : 128))
        return o;
    }
  }
  return w.mode == WHOLE_NONE ? none : w;
}

}  // namespace eithot

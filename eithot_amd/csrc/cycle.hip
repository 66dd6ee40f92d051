// Cycle following of cells of at least 16 bytes on gfx950.
//
// A pass moves whole cells of U bytes along the cycles of a permutation of
// cell positions, cut into segments (plan.hpp: CycleTable).  It is bound by
// memory where cells are whole lines, by partly used lines elsewhere, and by
// the arithmetic of source positions where several maps are composed.  An
// item is one segment of one matrix and one group of at most 1 KiB of every
// cell; it owns
// ceil(group / 16) consecutive lanes of a wave, any count, as many items to a
// wave as fit.  Lane l moves bytes 16 l .. 16 l + 15 of the group, the last
// lane the group's last 16 bytes, whatever the cell's size and address: the
// hardware splits an unaligned access at line boundaries, which costs less
// than realigning in registers did (cells of 4-byte words 2.1-3.2 TB/s).
// Where the last lane overlaps the one before it, both load the same old
// bytes in one instruction and store the same bytes in one instruction.
//
// A wave walks its segments p -> src(p), writing cell(p) <- old cell(src(p)),
// with D loads in flight: each store to a position waits for the load of the
// cell that follows it, and loads return in order, so the position's own old
// cell has been read before it is overwritten.  The last write of a segment
// takes the cell saved in a boundary slot before the pass (cut cycles), or
// the one the item read from its first position (whole cycles).
#include <hip/hip_runtime.h>

#include <algorithm>

#include "kernels.hpp"
#include "maps.hpp"

namespace eithot {
namespace {

typedef uint32_t C16 __attribute__((ext_vector_type(4)));
typedef uint32_t C16u __attribute__((ext_vector_type(4), aligned(1)));  // at any address

// One digit permutation of positions: it takes p to p * w[0] plus the sum
// over k >= 1 of (p / P_k) * w[k], mod 2^32, with P_k the product of the
// first k radices: p's digits d_k are p / P_k - r_k * (p / P_(k+1)), so
// w[k] = stride_k - r_(k-1) * stride_(k-1).
struct CycStage {
  uint32_t n, w[kMaxCycleDigits];
  FD31 fp[kMaxCycleDigits];  // fp[k]: division by P_k, k >= 1
};
struct Cyc16Args {
  char* data;  // first cell of matrix 0
  uint64_t RCU;
  uint32_t U, G, groups, lanes, per_wave, nseg, nslots;
  const CycleSeg* segs;
  const uint32_t* slots;
  char* boundary;
  uint64_t B, items;
  FD32 flanes;
  FD64 fgroups, fnseg;
  uint32_t nstages;
  CycStage st[kMaxCycleMaps];
};

// Source of cell position p: at most S digit permutations of at most K
// digits, K - 1 independent divisions of two instructions and as many
// multiply-adds each (the maps they are made of take three chained divisions
// of six instructions each).
template <int S, int K>
__device__ __forceinline__ uint32_t cyc16_src(const Cyc16Args& a, uint32_t p) {
#pragma unroll
  for (int j = 0; j < S; ++j) {
    if (j > 0 && j >= (int)a.nstages) continue;
    const CycStage& g = a.st[j];
    uint32_t s = p * g.w[0];
#pragma unroll
    for (int k = 1; k < K; ++k)
      if (k < (int)g.n) s += g.fp[k].div(p) * g.w[k];
    p = s;
  }
  return p;
}

// NT bit 0: non-temporal loads, bit 1: stores
template <int NT>
__device__ __forceinline__ C16 get16(const char* p) {
  if constexpr (NT & 1) return __builtin_nontemporal_load(reinterpret_cast<const C16u*>(p));
  return *reinterpret_cast<const C16u*>(p);
}
template <int NT>
__device__ __forceinline__ void set16(char* p, const C16& v) {
  if constexpr (NT & 2) __builtin_nontemporal_store((C16u)v, reinterpret_cast<C16u*>(p));
  else *reinterpret_cast<C16u*>(p) = v;
}

template <int D, int NT, int S, int K>
__global__ __launch_bounds__(256) void k_cycle16(Cyc16Args a) {
  const uint64_t gtid = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const uint32_t lw = threadIdx.x & 63;
  const uint32_t sub = a.flanes.div(lw), lane = lw - sub * a.lanes;
  const uint64_t item = (gtid >> 6) * a.per_wave + sub;
  if (sub >= a.per_wave || item >= a.items) return;
  const uint64_t rest = a.fgroups.div(item);
  const uint32_t g = (uint32_t)(item - rest * a.groups);
  const uint64_t b = a.fnseg.div(rest);
  const uint64_t s = rest - b * a.nseg;
  const uint32_t r0 = g * a.G, n = a.U - r0 < a.G ? a.U - r0 : a.G;
  if (lane * 16 >= n) return;  // the cell's last group may be shorter
  const uint32_t off = r0 + (lane * 16 + 16 <= n ? lane * 16 : n - 16);
  char* m = a.data + b * a.RCU + off;
  const CycleSeg sg = a.segs[s];
  uint32_t p = sg.start;
  auto cell = [&](uint32_t q) { return m + (uint64_t)q * a.U; };
  const C16 last = sg.src_slot < 0
                       ? get16<0>(cell(p))
                       : get16<0>(a.boundary + (b * a.nslots + (uint64_t)sg.src_slot) * a.U + off);
  for (uint32_t t = 0; t < sg.len; t += D) {
    C16 v[D];
    uint32_t q[D], pp = p;
#pragma unroll
    for (int k = 0; k < D; ++k) q[k] = pp = cyc16_src<S, K>(a, pp);
#pragma unroll
    for (int k = 0; k < D; ++k)
      if (t + k < sg.len) v[k] = t + k + 1 == sg.len ? last : get16<NT>(cell(q[k]));
    uint32_t dst = p;
#pragma unroll
    for (int k = 0; k < D; ++k)
      if (t + k < sg.len) {
        set16<NT>(cell(dst), v[k]);
        dst = q[k];
      }
    p = q[D - 1];
  }
}

// The cells at the first positions of cut segments, to their boundary slots:
// lanes of 16 bytes, a cell's last ones as above (copied twice).
__global__ __launch_bounds__(256) void k_cycle16_save(Cyc16Args a, uint32_t cpc, FD64 fcpc,
                                                      FD64 fnslots) {
  const uint64_t total = a.B * a.nslots * cpc;
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  for (uint64_t t = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; t < total; t += stride) {
    const uint64_t cell = fcpc.div(t);  // b * nslots + slot
    const uint32_t c = (uint32_t)(t - cell * cpc) * 16;
    const uint32_t off = c + 16 <= a.U ? c : a.U - 16;
    const uint64_t b = fnslots.div(cell), s = cell - b * a.nslots;
    set16<0>(a.boundary + cell * a.U + off, get16<0>(a.data + b * a.RCU + (uint64_t)a.slots[s] * a.U + off));
  }
}

template <int D, int NT>
void launch_form(const Cyc16Args& a, uint32_t blocks, hipStream_t st) {
  uint32_t n = 0;
  for (uint32_t k = 0; k < a.nstages; ++k) n = std::max(n, a.st[k].n);
  if (a.nstages == 1 && n <= 4)
    hipLaunchKernelGGL((k_cycle16<D, NT, 1, 4>), dim3(blocks), dim3(256), 0, st, a);
  else if (a.nstages == 1)
    hipLaunchKernelGGL((k_cycle16<D, NT, 1, kMaxCycleDigits>), dim3(blocks), dim3(256), 0, st, a);
  else if (a.nstages <= 2 && n <= 5)
    hipLaunchKernelGGL((k_cycle16<D, NT, 2, 5>), dim3(blocks), dim3(256), 0, st, a);
  else
    hipLaunchKernelGGL((k_cycle16<D, NT, kMaxCycleMaps, kMaxCycleDigits>), dim3(blocks), dim3(256), 0,
                       st, a);
}
template <int D>
void launch_nt(const Cyc16Args& a, int nt, uint32_t blocks, hipStream_t st) {
  if (nt == 3) launch_form<D, 3>(a, blocks, st);
  else if (nt == 2) launch_form<D, 2>(a, blocks, st);
  else launch_form<D, 0>(a, blocks, st);
}

}  // namespace

bool cycle16_takes(const Op& op, const LaunchCfg& cfg) {
  return cfg.cycle_variant == 0 && op.cyc && op.U >= 16 && op.U < (1ll << 31) &&
         !op.cyc->digits.empty() && op.cyc->digits.size() <= (size_t)kMaxCycleMaps;
}

hipError_t launch_cycle16(const Op& op, char* data, char* scratch, int64_t scratch_bytes,
                          const LaunchCfg& cfg, hipStream_t stream, const void* table) {
  const CycleTable& t = *op.cyc;
  if (t.segs.empty()) return hipSuccess;  // fixed points only
  const uint64_t need = (uint64_t)op.B * t.slots.size() * (uint64_t)op.U;
  if (need && (!scratch || (uint64_t)scratch_bytes < need)) return hipErrorInvalidValue;
  Cyc16Args a{};
  a.data = data + op.base;
  a.RCU = (uint64_t)op.R * op.C * op.U;
  a.U = (uint32_t)op.U;
  a.G = cycle_cell_group(a.U);
  a.groups = (a.U + a.G - 1) / a.G;
  a.lanes = (a.G + 15) / 16;
  a.per_wave = 64 / a.lanes;
  a.nseg = (uint32_t)t.segs.size();
  a.nslots = (uint32_t)t.slots.size();
  a.segs = reinterpret_cast<const CycleSeg*>(table);
  a.slots = reinterpret_cast<const uint32_t*>((const char*)table + t.segs.size() * sizeof(CycleSeg));
  a.boundary = scratch;
  a.B = (uint64_t)op.B;
  a.items = a.B * a.nseg * a.groups;
  a.flanes.init(a.lanes);
  a.fgroups.init(a.groups);
  a.fnseg.init(a.nseg);
  a.nstages = (uint32_t)t.digits.size();
  for (size_t j = 0; j < t.digits.size(); ++j) {
    const CycleDigits& d = t.digits[j];
    CycStage& g = a.st[j];
    g.n = (uint32_t)d.n;
    uint64_t prod = 1;
    for (int k = 0; k < d.n; ++k) {
      g.w[k] = d.stride[k] - (k ? d.radix[k - 1] * d.stride[k - 1] : 0);
      if (k) g.fp[k].init((uint32_t)prod);
      prod *= d.radix[k];
    }
  }
  const uint64_t waves = (a.items + a.per_wave - 1) / a.per_wave;
  const uint64_t blocks = (waves + 3) / 4;
  if (blocks >= (1ull << 31)) return hipErrorInvalidValue;
  if (a.nslots) {
    const uint32_t cpc = (a.U + 15) / 16;
    FD64 fcpc(cpc), fns(a.nslots);
    const uint64_t total = a.B * a.nslots * cpc;
    hipLaunchKernelGGL(k_cycle16_save, dim3((uint32_t)std::min<uint64_t>((total + 255) / 256, 256ull * 64)),
                       dim3(256), 0, stream, a, cpc, fcpc, fns);
  }
  // cells of at least 512 bytes in whole aligned 16-byte words: non-temporal
  // loads and stores, measured 1.7 % faster on 512-byte cells and 2-7 % on
  // larger ones; smaller cells lose up to 70 % with them (neighbouring cells
  // share cache lines that the hints evict).  Smaller ones in passes of at
  // least 512 MiB: non-temporal stores only, 2-6 % faster on 128-464-byte
  // cells of 0.8-4 GB passes; a 231 MB pass, which the 256 MB last-level
  // cache could hold, was 30 % slower with them.
  int nt = 0;
  if (op.U % 16 == 0 && (uintptr_t)a.data % 16 == 0)
    nt = op.U >= 512 ? 3 : a.B * a.RCU >= (512ull << 20) ? 2 : 0;
  // Steps of 8 positions, or of 2 or 4 where segments average no more: a step
  // computes the sources of all its positions (over cycles of mostly 6, mean
  // 8, a third more than it moves).
  if (t.mean && t.mean <= 2) launch_nt<2>(a, nt, (uint32_t)blocks, stream);
  else if (t.mean && t.mean <= 4) launch_nt<4>(a, nt, (uint32_t)blocks, stream);
  else launch_nt<8>(a, nt, (uint32_t)blocks, stream);
  return hipGetLastError();
}

}  // namespace eithot

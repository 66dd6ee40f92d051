// gfx950 kernels of the whole-permutation passes (whole.hpp).
#include <hip/hip_runtime.h>

#include <algorithm>

#include "kernels.hpp"
#include "whole.hpp"

namespace eithot {
namespace {

typedef uint32_t V16 __attribute__((ext_vector_type(4)));
// global accesses of 16 bytes at any address (runs start where the tensor's
// lengths put them); the hardware splits them at line boundaries
typedef uint32_t V16u __attribute__((ext_vector_type(4), aligned(1)));

template <int WL>
struct ElemOf;
template <>
struct ElemOf<0> {
  using T = uint8_t;
};
template <>
struct ElemOf<1> {
  using T = uint16_t;
};
template <>
struct ElemOf<2> {
  using T = uint32_t;
};
template <>
struct ElemOf<3> {
  using T = uint64_t;
};
template <>
struct ElemOf<4> {
  using T = V16;
};
// an element at any global address
template <int WL>
struct Loose {
  typename ElemOf<WL>::T v;
} __attribute__((packed));

template <int WL>
union Chunk {
  typename ElemOf<WL>::T e[16 >> WL];
  V16 v;
};

// 16 bytes to LDS at a multiple of max(4, element) bytes
template <int WL>
__device__ __forceinline__ void put_chunk(unsigned char* p, const V16& v) {
  if constexpr (WL == 4) {
    *reinterpret_cast<V16*>(p) = v;
  } else if constexpr (WL == 3) {
    reinterpret_cast<uint64_t*>(p)[0] = (uint64_t)v[0] | ((uint64_t)v[1] << 32);
    reinterpret_cast<uint64_t*>(p)[1] = (uint64_t)v[2] | ((uint64_t)v[3] << 32);
  } else {
    uint32_t* q = reinterpret_cast<uint32_t*>(p);
    q[0] = v[0];
    q[1] = v[1];
    q[2] = v[2];
    q[3] = v[3];
  }
}

// LDS areas of a workgroup (whole.hpp)
struct Areas {
  uint32_t* in;    // input runs: offsets from the tile's first element
  uint2* out;      // output runs: the same, and their LDS offsets
  uint32_t* otab;  // LDS offsets of an output run's elements
  unsigned char* tile;
};
__device__ __forceinline__ Areas areas(const WholeGeom& g, unsigned char* lds) {
  Areas a;
  a.in = reinterpret_cast<uint32_t*>(lds + kWholeCtl);
  a.out = reinterpret_cast<uint2*>(lds + kWholeCtl + whole_in_bytes(g));
  a.otab = reinterpret_cast<uint32_t*>(lds + kWholeCtl + whole_in_bytes(g) + whole_out_bytes(g));
  a.tile = reinterpret_cast<unsigned char*>(a.otab) + whole_otab_bytes(g);
  return a;
}

constexpr uint32_t kNoRun = ~0u;

template <int ND>
__device__ __forceinline__ void list_in(const WholeGeom& g, const WholeTile& x, const Areas& a) {
  for (uint32_t e = threadIdx.x; e < g.nin; e += blockDim.x) {
    uint32_t off;
    const bool ok = whole_in_run<ND>(g, x, e, &off);
    a.in[e] = ok ? off : kNoRun;
  }
}
template <int ND>
__device__ __forceinline__ void list_out(const WholeGeom& g, const WholeTile& x, const Areas& a) {
  for (uint32_t e = threadIdx.x; e < g.nout; e += blockDim.x) {
    uint32_t off, l;
    const bool ok = whole_out_run<ND>(g, x, e, &off, &l);
    a.out[e] = make_uint2(ok ? off : kNoRun, l);
  }
}
template <bool MULTI, int ND>
__device__ __forceinline__ void list_elems(const WholeGeom& g, const Areas& a) {
  if (MULTI)
    for (uint32_t e = threadIdx.x; e < g.len_out; e += blockDim.x) a.otab[e] = whole_elem<ND>(g, e);
}

// A thread's walk over the 16-byte chunks t = threadIdx.x + i * blockDim.x of
// a tile's runs, `per` to a run: the run and the chunk within it step by
// constants, so only the first takes a division.
struct Walk {
  uint32_t rho, c, drho, dc, per;
  __device__ __forceinline__ Walk(const FD32& f) {
    per = f.d;
    rho = f.div(threadIdx.x);
    c = threadIdx.x - rho * per;
    drho = f.div(blockDim.x);
    dc = blockDim.x - drho * per;
  }
  __device__ __forceinline__ void step() {
    c += dc;
    rho += drho;
    const bool wrap = c >= per;
    c -= wrap ? per : 0;
    rho += wrap ? 1 : 0;
  }
};

// Issues the loads of up to 8 chunks of the tile's input runs (src: the
// tile's first element, room: the tensor's bytes from there on); at[u] is
// chunk u's place in LDS, kNoRun for none.  Bytes read past a run's end are
// never used; a chunk that would leave the tensor (whose size is at least 16
// bytes) reads its last 16 bytes and shifts them down.
__device__ __forceinline__ void get_chunks(const WholeGeom& g, const char* src, uint64_t room,
                                           uint32_t run_bytes, const Areas& a, Walk& k, V16 (&v)[8],
                                           uint32_t (&at)[8]) {
  const uint32_t lim = room < kNoRun ? (uint32_t)room : kNoRun;
#pragma unroll
  for (int u = 0; u < 8; ++u) {
    at[u] = kNoRun;
    if (k.rho < g.nin) {
      const uint32_t run = a.in[k.rho], c = k.c * 16;
      if (run != kNoRun && c < run_bytes) {
        at[u] = whole_row(g, k.rho) + c;
        const uint32_t off = run + c;
        if (off + 16 <= lim) {
          v[u] = *reinterpret_cast<const V16u*>(src + off);
        } else {
          const V16 e = *reinterpret_cast<const V16u*>(src + (int64_t)room - 16);
          const uint32_t s = (uint32_t)((uint64_t)off + 16 - room) * 8;
          const uint64_t lo = (uint64_t)e[0] | ((uint64_t)e[1] << 32);
          const uint64_t hi = (uint64_t)e[2] | ((uint64_t)e[3] << 32);
          const uint64_t l = s < 64 ? (lo >> s) | (hi << 1 << (63 - s)) : hi >> (s - 64);
          const uint64_t h = s < 64 ? hi >> s : 0;
          v[u] = V16{(uint32_t)l, (uint32_t)(l >> 32), (uint32_t)h, (uint32_t)(h >> 32)};
        }
      }
    }
    k.step();
  }
}
template <int WL>
__device__ __forceinline__ void put_chunks(const Areas& a, const V16 (&v)[8], const uint32_t (&at)[8]) {
#pragma unroll
  for (int u = 0; u < 8; ++u)
    if (at[u] != kNoRun) put_chunk<WL>(a.tile + at[u], v[u]);
}

// Stores the tile along its output runs (dst: its first element's place): 16
// bytes per thread gathered from LDS element by element; a run's last store
// is moved back to end with the run (its first elements are stored twice,
// with the same values).
template <int WL, bool MULTI, int ND>
__device__ __forceinline__ void tile_store(const WholeGeom& g, const WholeTile& x, char* dst,
                                           const Areas& a) {
  using E = typename ElemOf<WL>::T;
  constexpr uint32_t V = 16u >> WL;
  const uint32_t len = whole_len_out<ND>(g, x);
  Walk k(g.fcout);
  for (; k.rho < g.nout; k.step()) {
    const uint2 run = a.out[k.rho];
    uint32_t p = k.c * V;
    if (run.x == kNoRun || p >= len) continue;
    const unsigned char* l = a.tile + run.y;
    // runs over one dim: V elements from a multiple of V (or any place
    // without the group padding) lie a constant step apart
    const bool tail = p + V > len;
    if (len >= V && !(tail && !MULTI && g.g2)) {
      if (tail) p = len - V;
      Chunk<WL> q;
      if constexpr (MULTI) {
#pragma unroll
        for (uint32_t e = 0; e < V; ++e) q.e[e] = *reinterpret_cast<const E*>(l + a.otab[p + e]);
      } else {
        const unsigned char* s = l + whole_elem1(g, p);
#pragma unroll
        for (uint32_t e = 0; e < V; ++e) q.e[e] = *reinterpret_cast<const E*>(s + e * g.ols[0]);
      }
      *reinterpret_cast<V16u*>(dst + (run.x + (p << WL))) = q.v;
    } else {
      for (; p < len; ++p)
        reinterpret_cast<Loose<WL>*>(dst + (run.x + (p << WL)))->v =
            *reinterpret_cast<const E*>(l + (MULTI ? a.otab[p] : whole_elem1(g, p)));
    }
  }
}

// ---------------------------------------------------------------------------
// resident form
// ---------------------------------------------------------------------------
struct Words {
  static __device__ __forceinline__ uint32_t add(uint32_t* p, uint32_t v) {
    return __hip_atomic_fetch_add(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  static __device__ __forceinline__ uint32_t get(uint32_t* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  static __device__ __forceinline__ void set(uint32_t* p, uint32_t v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  static __device__ __forceinline__ bool cas(uint32_t* p, uint32_t from, uint32_t to) {
    return __hip_atomic_compare_exchange_strong(p, &from, to, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                                __HIP_MEMORY_SCOPE_AGENT);
  }
  static __device__ __forceinline__ uint64_t now() { return __builtin_amdgcn_s_memrealtime(); }
  static __device__ __forceinline__ void pause() { __builtin_amdgcn_s_sleep(1); }
};

// Constant memory read late: the compiler may not load through the result
// ahead of this point.
template <typename T>
using Const = const T __attribute__((address_space(4)));
template <typename T>
__device__ __forceinline__ Const<T>* late(Const<T>* p) {
  asm volatile("" : "+s"(p));
  return p;
}

// The region at `base` moved by one workgroup, in output order into host
// memory and back: what the last workgroup does where the others have left.
// Regions of other launches may want the host memory too; whoever holds its
// lock runs and lets go of it.  g and c are read late: loaded with the rest
// at the kernel's start, they and what is made of them cost every workgroup
// registers (64 MiB of pairs: 33.6 us, 32.1 so).
template <int WL>
__device__ __forceinline__ void move_alone(Const<WholeGeom>* g, Const<WholeCtl>* c, char* base) {
  using E = typename ElemOf<WL>::T;
  uint32_t* lock = c->lock;
  char* room = c->room;
  uint32_t od[kWholeDims], ogin[kWholeDims];
#pragma unroll
  for (int k = 0; k < kWholeDims; ++k) {
    od[k] = g->od[k];
    ogin[k] = g->ogin[k];
  }
  if (threadIdx.x == 0)
    while (!Words::cas(lock, 0, 1)) Words::pause();
  __syncthreads();
  __threadfence_system();
  const uint32_t bytes = (uint32_t)g->region, n = bytes >> WL, n16 = bytes / 16;
  for (uint32_t o = threadIdx.x; o < n; o += blockDim.x)
    reinterpret_cast<E*>(room)[o] =
        reinterpret_cast<const Loose<WL>*>(base + whole_source(g->r, od, ogin, o))->v;
  __threadfence_system();  // written through, and no stale copy is read
  __syncthreads();
  __threadfence_system();
  for (uint32_t o = threadIdx.x; o < n16; o += blockDim.x)
    reinterpret_cast<V16u*>(base)[o] = reinterpret_cast<const V16*>(room)[o];
  for (uint32_t o = n16 * 16 + threadIdx.x; o < bytes; o += blockDim.x) base[o] = room[o];
  __threadfence_system();
  __syncthreads();
  if (threadIdx.x == 0) Words::set(lock, 0);
}

// Tiles t * per .. of region b, meeting its region's other workgroups at
// `slot`.  The first is held in LDS, a second one in registers until the
// first is stored.  No data passes between workgroups: the counters only
// order a region's loads, which are complete once in LDS or waited for,
// before its stores, so they need no cache flush.  True when the workgroup is
// to move the region alone, and then to set the region's word to the second
// word of LDS.
template <int WL, bool MULTI, int ND, bool PAIR>
__device__ __forceinline__ bool resident_body(const WholeGeom& g, char* data, uint32_t b, uint32_t t,
                                              uint32_t slot, const WholeCtl& c,
                                              unsigned char* lds) {
  uint32_t* ctl = reinterpret_cast<uint32_t*>(lds);
  uint32_t word = 0;
  if (threadIdx.x == 0) word = Words::get(c.open + slot);
  const WholeTile x = whole_tile<ND>(g, whole_nth(g, PAIR ? t * g.per : t));
  const uint64_t region = (uint64_t)b * g.region, room = g.B * g.region - region;
  char* base = data + region;
  const Areas a = areas(g, lds);
  list_in<ND>(g, x, a);
  list_out<ND>(g, x, a);
  list_elems<MULTI, ND>(g, a);
  __syncthreads();
  const uint32_t run_bytes = whole_len_in<ND>(g, x) << WL;
  for (Walk k(g.fcin); k.rho < g.nin;) {
    V16 v[8];
    uint32_t at[8];
    get_chunks(g, base + x.in, room - x.in, run_bytes, a, k, v, at);
    put_chunks<WL>(a, v, at);
  }
  const bool second = PAIR && g.per == 2 && 2 * t + 1 < g.tiles;
  WholeTile y = x;
  V16 hv[8];
  uint32_t hat[8];
  if (second) {
    y = whole_tile<ND>(g, whole_nth(g, 2 * t + 1));
    __syncthreads();  // the list of x's input runs has been read
    list_in<ND>(g, y, a);
    __syncthreads();
    Walk k(g.fcin);
    get_chunks(g, base + y.in, room - y.in, whole_len_in<ND>(g, y) << WL, a, k, hv, hat);
    __builtin_amdgcn_s_waitcnt(0);
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    ctl[0] = whole_meet<Words>(c, slot, t, g.wgs, word);
    ctl[1] = word;
  }
  __syncthreads();
  if (ctl[0] != MEET_STORE) return ctl[0] == MEET_ALONE;
  tile_store<WL, MULTI, ND>(g, x, base + x.out, a);
  if (second) {
    __syncthreads();  // x has been read out of LDS, and its lists
    put_chunks<WL>(a, hv, hat);
    list_out<ND>(g, y, a);
    __syncthreads();
    tile_store<WL, MULTI, ND>(g, y, base + y.out, a);
  }
  return false;
}

struct WholeItem {
  uint32_t op, b, t, slot;
};
struct WholeOp {
  WholeGeom g;
  char* data;
  int variant;  // log2(word) * 4 + (runs over several dims) * 2 + (at most 4 dims)
};
// The rest of a workgroup that resident_body has told to move region b alone.
template <int WL>
__device__ __forceinline__ void finish_alone(Const<WholeGeom>* g, Const<WholeCtl>* c, char* data,
                                             uint32_t b, uint32_t slot, const unsigned char* lds) {
  move_alone<WL>(g, c, data + (uint64_t)b * g->region);
  if (threadIdx.x == 0)
    whole_done_alone<Words>(c->open + slot, reinterpret_cast<const uint32_t*>(lds)[1]);
}
struct ResidentArgs {  // of k_resident, as it gets them
  WholeGeom g;
  char* data;
  WholeCtl c;
};
struct BatchArgs {  // of k_resident_batch
  const WholeOp* ops;
  const WholeItem* items;
  WholeCtl c;
};

// One tile, or two, per workgroup.  The workgroups of a region have
// consecutive block indices, and workgroups start in that order on each XCD,
// so those of the earliest unfinished region all run as soon as that many are
// resident, which the planner keeps to half of the chip's room.  Launches of
// resident passes of one process follow each other (the runtime chains them),
// so no two share that room, nor the words.  Where the room is short all the
// same (other processes), regions are called off and moved alone.
template <int WL, bool MULTI, int ND, bool PAIR>
__global__ __launch_bounds__(1024) void k_resident(WholeGeom g, char* data, WholeCtl c) {
  extern __shared__ __align__(16) unsigned char lds[];
  const uint32_t b = g.fwgs.div(blockIdx.x);
  if (resident_body<WL, MULTI, ND, PAIR>(g, data, b, blockIdx.x - b * g.wgs, b, c, lds)) {
    Const<ResidentArgs>* a = late((Const<ResidentArgs>*)__builtin_amdgcn_kernarg_segment_ptr());
    finish_alone<WL>(&a->g, &a->c, a->data, b, b, lds);
  }
}

// The same over the regions of many tensors: workgroup i takes item i.
__global__ __launch_bounds__(kWholeBatchThreads) void k_resident_batch(const WholeOp* __restrict__ ops,
                                                        const WholeItem* __restrict__ items,
                                                        WholeCtl c) {
  extern __shared__ __align__(16) unsigned char lds[];
  const WholeItem i = items[blockIdx.x];
  const WholeOp& o = ops[i.op];
  const WholeGeom& g = o.g;
  bool alone = false;
#define EH_WHOLE(WL, MULTI, ND)                                                       \
  case (WL)*4 + (MULTI)*2 + (ND == 4):                                                \
    alone = resident_body<WL, MULTI, ND, true>(g, o.data, i.b, i.t, i.slot, c, lds);  \
    break;
#define EH_WHOLE_W(WL)                                                                \
  EH_WHOLE(WL, false, 4) EH_WHOLE(WL, true, 4) EH_WHOLE(WL, false, 8) EH_WHOLE(WL, true, 8)
  switch (o.variant) {
    EH_WHOLE_W(0)
    EH_WHOLE_W(1)
    EH_WHOLE_W(2)
    EH_WHOLE_W(3)
    EH_WHOLE_W(4)
  }
  if (!alone) return;
  Const<BatchArgs>* ka = late((Const<BatchArgs>*)__builtin_amdgcn_kernarg_segment_ptr());
  Const<WholeOp>* op = (Const<WholeOp>*)(ka->ops + i.op);
  switch (op->variant >> 2) {
    case 0: finish_alone<0>(&op->g, &ka->c, op->data, i.b, i.slot, lds); break;
    case 1: finish_alone<1>(&op->g, &ka->c, op->data, i.b, i.slot, lds); break;
    case 2: finish_alone<2>(&op->g, &ka->c, op->data, i.b, i.slot, lds); break;
    case 3: finish_alone<3>(&op->g, &ka->c, op->data, i.b, i.slot, lds); break;
    case 4: finish_alone<4>(&op->g, &ka->c, op->data, i.b, i.slot, lds); break;
  }
#undef EH_WHOLE_W
#undef EH_WHOLE
}

// the words of a device's resident passes over single tensors, after those
// of all its resident passes (each on a line of its own)
__device__ uint32_t g_ctl[64 + whole_ctl_words(kWholeRegions)];

// ---------------------------------------------------------------------------
// orbit form
// ---------------------------------------------------------------------------
// One cycle of tiles per workgroup: its tile with the lowest index leads,
// the workgroups of the others leave.  The tile whose place the transposed
// one takes is loaded into registers ahead of it and goes to LDS after it.
template <int WL, bool MULTI, int ND>
__global__ __launch_bounds__(512) void k_orbit(WholeGeom g, char* data) {
  extern __shared__ __align__(16) unsigned char lds[];
  const uint32_t b = g.ftiles.div(blockIdx.x);
  const uint32_t first = whole_nth(g, blockIdx.x - b * g.tiles);
  WholeTile x = whole_tile<ND>(g, first);
  for (uint32_t q = x.next; q != first; q = whole_tile<ND>(g, q).next)
    if (q < first) return;
  char* base = data + (uint64_t)b * g.region;
  const uint64_t room = (g.B - b) * g.region;
  const Areas a = areas(g, lds);
  list_in<ND>(g, x, a);
  list_elems<MULTI, ND>(g, a);
  __syncthreads();
  V16 v[8];
  uint32_t at[8];
  Walk k(g.fcin);
  get_chunks(g, base + x.in, room - x.in, whole_len_in<ND>(g, x) << WL, a, k, v, at);
  for (;;) {
    const bool more = x.next != first;
    WholeTile y = x;
    V16 nv[8];
    uint32_t nat[8];
    if (more) {
      y = whole_tile<ND>(g, x.next);
      __syncthreads();  // the list of x's input runs has been read
      list_in<ND>(g, y, a);
      __syncthreads();
      Walk ky(g.fcin);
      get_chunks(g, base + y.in, room - y.in, whole_len_in<ND>(g, y) << WL, a, ky, nv, nat);
    }
    list_out<ND>(g, x, a);
    put_chunks<WL>(a, v, at);
    __builtin_amdgcn_s_waitcnt(0);  // y is read before x is stored over it
    __syncthreads();
    tile_store<WL, MULTI, ND>(g, x, base + x.out, a);
    if (!more) break;
    __syncthreads();
    x = y;
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      v[u] = nv[u];
      at[u] = nat[u];
    }
  }
}

template <int WL, bool MULTI, int ND>
hipError_t launch_i(const WholePass& p, char* data, const WholeCtl& c, hipStream_t st) {
  const dim3 block(p.threads);
  const uint32_t per_region = p.mode == WHOLE_ORBIT ? p.g.tiles : p.g.wgs;
  const dim3 grid((uint32_t)(per_region * p.g.B));
  if (p.mode == WHOLE_ORBIT)
    hipLaunchKernelGGL((k_orbit<WL, MULTI, ND>), grid, block, (size_t)p.lds, st, p.g, data);
  else if (p.g.per == 2)
    hipLaunchKernelGGL((k_resident<WL, MULTI, ND, true>), grid, block, (size_t)p.lds, st, p.g, data, c);
  else
    hipLaunchKernelGGL((k_resident<WL, MULTI, ND, false>), grid, block, (size_t)p.lds, st, p.g, data, c);
  return hipGetLastError();
}
template <int WL>
hipError_t launch_w(const WholePass& p, char* data, const WholeCtl& c, hipStream_t st) {
  const bool multi = p.g.jout > 1;
  if (p.g.r <= 4)
    return multi ? launch_i<WL, true, 4>(p, data, c, st) : launch_i<WL, false, 4>(p, data, c, st);
  return multi ? launch_i<WL, true, kWholeDims>(p, data, c, st)
               : launch_i<WL, false, kWholeDims>(p, data, c, st);
}
template <int WL>
void configure_w(int64_t bytes, hipError_t& e) {
  for (const void* fn :
       {(const void*)k_resident<WL, false, 4, false>, (const void*)k_resident<WL, true, 4, false>,
        (const void*)k_resident<WL, false, kWholeDims, false>,
        (const void*)k_resident<WL, true, kWholeDims, false>,
        (const void*)k_resident<WL, false, 4, true>, (const void*)k_resident<WL, true, 4, true>,
        (const void*)k_resident<WL, false, kWholeDims, true>,
        (const void*)k_resident<WL, true, kWholeDims, true>}) {
    const hipError_t r = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
    if (r != hipSuccess) e = r;
  }
}

}  // namespace

hipError_t launch_whole(const WholePass& p, char* data, const WholeCtl& ctl, hipStream_t st) {
  switch (p.g.w) {
    case 16: return launch_w<4>(p, data, ctl, st);
    case 8: return launch_w<3>(p, data, ctl, st);
    case 4: return launch_w<2>(p, data, ctl, st);
    case 2: return launch_w<1>(p, data, ctl, st);
    default: return launch_w<0>(p, data, ctl, st);
  }
}

hipError_t whole_ctl_device(WholeCtl& c) {
  void* p = nullptr;
  const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(g_ctl));
  if (e != hipSuccess) return e;
  c.recent = (uint32_t*)p;
  c.lock = (uint32_t*)p + 32;
  whole_ctl_at(c, (uint32_t*)p + 64, kWholeRegions);
  return e;
}

hipError_t configure_whole(int64_t bytes) {
  hipError_t e = hipSuccess;
  configure_w<0>(bytes, e);
  configure_w<1>(bytes, e);
  configure_w<2>(bytes, e);
  configure_w<3>(bytes, e);
  configure_w<4>(bytes, e);
  return e;
}

// ---------------------------------------------------------------------------
// many tensors in one launch
// ---------------------------------------------------------------------------
struct WholeBatch {
  char* mem = nullptr;  // ops, items and counters
  WholeOp* ops = nullptr;
  WholeItem* items = nullptr;
  WholeCtl ctl;
  uint32_t grid = 0;
  int64_t lds = 0;
};

hipError_t whole_batch_build(const std::vector<std::pair<const WholePass*, char*>>& passes,
                             const WholeCtl& ctl, WholeBatch** out) {
  *out = nullptr;
  std::vector<WholeOp> ops;
  std::vector<WholeItem> items;
  uint64_t slots = 0;
  int64_t lds = 0;
  for (const auto& p : passes) {
    const WholeGeom& g = p.first->g;
    const uint32_t op = (uint32_t)ops.size();
    int wl = 0;
    while ((1u << wl) < g.w) ++wl;
    ops.push_back({g, p.second, wl * 4 + (g.jout > 1 ? 2 : 0) + (g.r <= 4 ? 1 : 0)});
    lds = std::max(lds, p.first->lds);
    for (uint32_t b = 0; b < g.B; ++b, ++slots)
      for (uint32_t t = 0; t < g.wgs; ++t) items.push_back({op, b, t, (uint32_t)slots});
  }
  if (items.empty()) return hipSuccess;
  if (items.size() >= (1ull << 31)) return hipErrorInvalidValue;
  auto up = [](size_t n) { return (n + 255) / 256 * 256; };
  const size_t ob = up(ops.size() * sizeof(WholeOp)), ib = up(items.size() * sizeof(WholeItem));
  const size_t cb = whole_ctl_words((uint32_t)slots) * sizeof(uint32_t);
  auto* w = new WholeBatch;
  hipError_t e = hipMalloc((void**)&w->mem, ob + ib + cb);
  if (e == hipSuccess)
    e = hipMemcpy(w->mem, ops.data(), ops.size() * sizeof(WholeOp), hipMemcpyHostToDevice);
  if (e == hipSuccess)
    e = hipMemcpy(w->mem + ob, items.data(), items.size() * sizeof(WholeItem), hipMemcpyHostToDevice);
  if (e == hipSuccess) e = hipMemset(w->mem + ob + ib, 0, cb);
  if (e == hipSuccess) e = hipStreamSynchronize(nullptr);
  if (e != hipSuccess) {
    whole_batch_free(w);
    return e;
  }
  w->ops = (WholeOp*)w->mem;
  w->items = (WholeItem*)(w->mem + ob);
  w->ctl = ctl;
  whole_ctl_at(w->ctl, (uint32_t*)(w->mem + ob + ib), (uint32_t)slots);
  w->grid = (uint32_t)items.size();
  w->lds = lds;
  *out = w;
  return hipSuccess;
}

hipError_t whole_batch_enqueue(const WholeBatch* w, hipStream_t st) {
  if (!w) return hipSuccess;
  hipLaunchKernelGGL(k_resident_batch, dim3(w->grid), dim3(kWholeBatchThreads), (size_t)w->lds, st,
                     w->ops, w->items, w->ctl);
  return hipGetLastError();
}

void whole_batch_free(WholeBatch* w) {
  if (!w) return;
  if (w->mem) (void)hipFree(w->mem);
  delete w;
}

}  // namespace eithot

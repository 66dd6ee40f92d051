// Host runs of the resident passes' meeting (eithot_amd/csrc/whole.hpp) for
// the CPU tests: threads stand for workgroups, a limited number of which runs
// at a time, over real regions.  Compiled by the test with hipcc, never part
// of the product.
#include <atomic>
#include <chrono>
#include <condition_variable>
#include <mutex>
#include <thread>

#include "whole_harness.cpp"

namespace {

struct HostWords {
  static uint32_t add(uint32_t* p, uint32_t v) { return __atomic_fetch_add(p, v, __ATOMIC_SEQ_CST); }
  static uint32_t get(uint32_t* p) { return __atomic_load_n(p, __ATOMIC_SEQ_CST); }
  static void set(uint32_t* p, uint32_t v) { __atomic_store_n(p, v, __ATOMIC_SEQ_CST); }
  static bool cas(uint32_t* p, uint32_t from, uint32_t to) {
    return __atomic_compare_exchange_n(p, &from, to, false, __ATOMIC_SEQ_CST, __ATOMIC_SEQ_CST);
  }
  static uint64_t now() {  // 100 MHz
    return (uint64_t)std::chrono::steady_clock::now().time_since_epoch().count() / 10;
  }
  static void pause() { std::this_thread::yield(); }
};

// the chip: workgroups start in order while there is room, and leave it at
// their end; two launches (two processes) share it
struct Chip {
  std::mutex mu;
  std::condition_variable cv;
  int room;
  void enter() {
    std::unique_lock<std::mutex> lk(mu);
    cv.wait(lk, [&] { return room > 0; });
    --room;
  }
  void leave() {
    std::lock_guard<std::mutex> lk(mu);
    ++room;
    cv.notify_all();
  }
};

struct Launch {
  const WholePass& p;
  Emu e;
  WholeCtl c;
  std::vector<uint32_t> words;
  std::vector<uint8_t> room;
  uint32_t recent = 0, lock = 0;
  std::atomic<int> alone{0};
  std::atomic<bool> bad{false};

  Launch(const WholePass& w, uint8_t* data, uint64_t patience)
      : p(w), e{w.g, data, w.g.B * w.g.region}, words(whole_ctl_words((uint32_t)w.g.B), 0),
        room(w.g.region) {
    whole_ctl_at(c, words.data(), (uint32_t)w.g.B);
    c.recent = &recent;
    c.lock = &lock;
    c.room = (char*)room.data();
    c.patience = patience;
  }
  void workgroup(uint32_t block) {
    const WholeGeom& g = p.g;
    const uint32_t b = g.fwgs.div(block), t = block - b * g.wgs;
    const uint64_t region = b * g.region;
    const uint32_t word = HostWords::get(c.open + b);
    Emu mine = e;
    std::vector<std::vector<uint8_t>> held;
    for (uint32_t i = t * g.per; i < g.tiles && i < (t + 1) * g.per; ++i)
      held.push_back(mine.load(whole_nth(g, i), region));
    const WholeMeet how = whole_meet<HostWords>(c, b, t, g.wgs, word);
    if (how == MEET_STORE)
      for (uint32_t i = 0; i < held.size(); ++i) mine.store(whole_nth(g, t * g.per + i), region, held[i]);
    if (how == MEET_ALONE) {
      while (!HostWords::cas(c.lock, 0, 1)) HostWords::pause();
      for (uint32_t o = 0; o < g.region / g.w; ++o)
        std::memcpy(c.room + (uint64_t)o * g.w, e.data + region + whole_source(g.r, g.od, g.ogin, o), g.w);
      std::memcpy(e.data + region, c.room, g.region);
      HostWords::set(c.lock, 0);
      whole_done_alone<HostWords>(c.open + b, word);
      ++alone;
    }
    if (mine.bad) bad = true;
  }
  void run(Chip& chip) {
    std::vector<std::thread> th;
    const uint32_t n = (uint32_t)(p.g.B * p.g.wgs);
    for (uint32_t i = 0; i < n; ++i) {
      chip.enter();
      th.emplace_back([this, i, &chip] {
        workgroup(i);
        chip.leave();
      });
    }
    for (auto& t : th) t.join();
  }
};

}  // namespace

// Two launches of the resident pass of one shape, over data[0] and data[1],
// `rounds` times each on a chip with room for `room` workgroups.  batched:
// the pass of a tensor among many.  Returns the regions that were moved
// alone, -1 when the shape has no such pass, -2 on an access out of bounds,
// -3 when words are left changed.  *wgs: workgroups of a region.
extern "C" int wm_run(const int64_t* dims, const int* perm1, int rank, int64_t elem, int cus,
                      int batched, int room, int64_t patience, int rounds, uint8_t* data0,
                      uint8_t* data1, int64_t* wgs) {
  const WholePass p = batched ? plan_whole_batched(dims, perm1, rank, (size_t)elem, cus, 160 * 1024)
                              : plan_whole(dims, perm1, rank, (size_t)elem, cus, 160 * 1024, 3, true);
  if (p.mode != WHOLE_RESIDENT) return -1;
  *wgs = p.g.wgs;
  Chip chip;
  chip.room = room;
  Launch a(p, data0, (uint64_t)patience), b(p, data1, (uint64_t)patience);
  for (int k = 0; k < rounds; ++k) {
    std::thread other([&] { b.run(chip); });
    a.run(chip);
    other.join();
  }
  for (Launch* l : {&a, &b}) {
    if (l->bad) return -2;
    for (size_t i = (size_t)p.g.B; i < l->words.size(); ++i)
      if (l->words[i]) return -3;
    for (uint64_t r = 0; r < p.g.B; ++r)
      if (l->words[r] / 4 != (uint32_t)rounds || (l->words[r] & kCalledOff)) return -3;
    if (l->lock) return -3;
  }
  return a.alone + b.alone;
}

// The tiles of a resident pass as its workgroups hold them, moved once:
// whole_harness.cpp's wh_run for the pairs of tiles of a workgroup and for
// the passes of batches.  Returns its workgroups per region, 0 when there is
// no such pass, -1 on an access out of bounds or a tile that a workgroup
// cannot hold.
extern "C" int wm_once(const int64_t* dims, const int* perm1, int rank, int64_t elem, int cus,
                       int batched, int64_t lds_max, uint8_t* data, int64_t* per) {
  const WholePass p = batched ? plan_whole_batched(dims, perm1, rank, (size_t)elem, cus, lds_max)
                              : plan_whole(dims, perm1, rank, (size_t)elem, cus, lds_max, 3, true);
  if (p.mode != WHOLE_RESIDENT) return 0;
  const WholeGeom& g = p.g;
  *per = g.per;
  if (p.lds < whole_lds_bytes(g) || p.lds > lds_max) return -1;
  if (g.per < 1 || g.per > 2 || g.wgs != (g.tiles + g.per - 1) / g.per) return -1;
  // a second tile waits in 8 registers of 16 bytes per thread
  if (g.per == 2 && (int64_t)g.nin * g.fcin.d > (int64_t)p.threads * kWholeHold) return -1;
  if (batched && p.threads != kWholeBatchThreads) return -1;
  Emu e{g, data, g.B * g.region};
  std::vector<int> named(g.tiles, 0);
  for (uint64_t b = 0; b < g.B && !e.bad; ++b) {
    std::vector<std::pair<uint32_t, std::vector<uint8_t>>> held;
    for (uint32_t t = 0; t < g.wgs && !e.bad; ++t)
      for (uint32_t j = 0; j < g.per && g.per * t + j < g.tiles; ++j) {
        const uint32_t tau = whole_nth(g, g.per * t + j);
        if (tau >= g.tiles || (b == 0 && named[tau]++)) return -1;
        held.emplace_back(tau, e.load(tau, b * g.region));
      }
    if (held.size() != g.tiles) return -1;
    while (!held.empty() && !e.bad) {
      e.store(held.back().first, b * g.region, held.back().second);
      held.pop_back();
    }
  }
  return e.bad ? -1 : (int)g.wgs;
}

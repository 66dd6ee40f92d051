// Host checks of the planner's cached pass tables (eithot_amd/csrc/plan.cpp)
// for the CPU tests.  Compiled by the test with hipcc, never part of the
// product.
#include <chrono>

#include "../eithot_amd/csrc/plan.cpp"

using namespace eithot;

// Plans a shape twice and looks at the cycle tables that the first plan
// holds, which a running call may be reading: 0 when the second planning has
// left them alone, else 1 + the index of the pass.  *tables: how many there were.
extern "C" int pt_replan(const int64_t* dims, const int* perm1, int rank, int64_t elem, int64_t other,
                         int* tables) {
  DeviceProfile prof;
  Plan a, b;
  *tables = 0;
  if (make_plan(dims, perm1, rank, (size_t)elem, 1, 0.05, prof, 0, a)) return -1;
  struct Seen {
    const CycleSeg* segs;
    const CycleDigits* digits;
    size_t nsegs, ndigits;
    uint32_t mean, first;
  };
  auto look = [](const CycleTable& t) {
    return Seen{t.segs.data(), t.digits.data(), t.segs.size(), t.digits.size(), t.mean,
                t.segs.empty() ? 0 : t.segs[0].start};
  };
  std::vector<Seen> before;
  for (const Op& o : a.ops) before.push_back(o.cyc ? look(*o.cyc) : Seen{});
  // the same cells, of another size, and the same shape again
  if (make_plan(dims, perm1, rank, (size_t)(elem * other), 1, 0.05, prof, 0, b)) return -1;
  if (make_plan(dims, perm1, rank, (size_t)elem, 1, 0.05, prof, 0, b)) return -1;
  for (size_t i = 0; i < a.ops.size(); ++i) {
    if (!a.ops[i].cyc) continue;
    ++*tables;
    const Seen x = before[i], y = look(*a.ops[i].cyc);
    if (x.segs != y.segs || x.digits != y.digits || x.nsegs != y.nsegs || x.ndigits != y.ndigits ||
        x.mean != y.mean || x.first != y.first || (x.nsegs && !x.ndigits))
      return 1 + (int)i;
  }
  return 0;
}

// Shortest of `reps` planning times (ms), with or without cycle passes of small cells.
extern "C" double pt_plan_ms(const int64_t* dims, const int* perm1, int rank, int64_t elem, int small,
                             int reps) {
  DeviceProfile prof;
  prof.cycle_small = small;
  double best = 1e300;
  for (int k = 0; k < reps; ++k) {
    Plan p;
    const auto t0 = std::chrono::steady_clock::now();
    if (make_plan(dims, perm1, rank, (size_t)elem, 1, 0.05, prof, 0, p)) return -1;
    best = std::min(best, std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count());
  }
  return best;
}

// Internal runtime state shared by the C-ABI translation units.
#pragma once

#include <hip/hip_runtime.h>

#include <atomic>
#include <memory>
#include <mutex>
#include <string>
#include <vector>

#include "kernels.hpp"
#include "plan.hpp"
#include "plan_cache.hpp"
#include "whole.hpp"

namespace eithot {

using PlanPtr = std::shared_ptr<const Plan>;

// Per-device state.  Two locks:
//   mu         the plan cache;
//   enqueue_mu held from the first use of the arena or of pass tables to the
//              event recorded after a call's last pass: arena growth or
//              shrinking, table eviction and every launch that uses them are
//              mutually exclusive, so no thread launches into memory another
//              thread frees.  Lock order: enqueue_mu, then mu.
struct GraphMem;

struct Device {
  int id = 0;
  DeviceProfile prof;
  LaunchCfg cfg;
  std::mutex mu;
  LruCache<Plan> plans{kPlanCacheEntries, kPlanCacheHostBytes};
  std::mutex enqueue_mu;
  char* arena = nullptr;             // scratch for staged passes and cycle boundaries
  int64_t arena_bytes = 0;
  hipEvent_t arena_ready = nullptr;  // recorded after the last pass that used the arena
  // Resident whole-permutation passes share the chip with no other of their
  // kind (whole.hip): each waits, on the device, for the one before.  All
  // under enqueue_mu.
  hipEvent_t whole_ready = nullptr;
  bool whole_elsewhere = false;      // the last one ran on a stream other than the null stream
  int null_sees_all = 0;             // the null stream has every CU: 1, not: -1
  WholeCtl whole_ctl;
  // bytes at whole_ctl.room: a power of two, 1 to 64 MiB.  A smaller room
  // before it stays, for the passes in flight and the batches that name it.
  uint64_t whole_room = 0;
  // device bytes of the pass tables uploaded for plans of this cache (and
  // not yet freed; an evicted plan a request still holds counts until freed)
  std::atomic<int64_t> cached_tables{0};

  // plans cached per device, and the host bytes of their pass tables
  static constexpr size_t kPlanCacheEntries = 8192;
  static constexpr uint64_t kPlanCacheHostBytes = 16ull << 30;

  // The cached plan for these arguments, planned on first sight (outside
  // the cache lock).  The caller's reference keeps the plan alive even if
  // the cache evicts it.  small false: without cycle passes of small cells,
  // for callers that cannot give their tables and boundary cells a place.
  PlanPtr plan_for(const int64_t* dims, const int* perm1, int rank, size_t elem, int n_sub,
                   double alpha, int* rc, bool small = true);
  // hardware profile / launch configuration with the tuning knobs applied
  DeviceProfile profile() const;
  LaunchCfg launch_cfg() const;
  // With enqueue_mu held: keeps the device bytes the library holds (arena
  // plus the resident tables of cached plans) within `budget` by freeing the
  // tables of other cached plans, least recently used first, and shrinking
  // an arena larger than `keep` needs.
  void trim_locked(int64_t budget, const Plan* keep);
  // With enqueue_mu held: arena of at least `bytes`, ordered after its last
  // user on `stream`.
  int reserve_arena_locked(int64_t bytes, hipStream_t stream);
  int release_arena_after_locked(hipStream_t stream);
  // Memory that graphs have let go of (GraphMem, chained), freed by the next
  // call.  Not under enqueue_mu: graphs end on any thread.
  std::atomic<GraphMem*> retired{nullptr};
  void free_retired();

  // With enqueue_mu held: whether a call of `plan` on `stream` runs its
  // whole-permutation pass, which run_plan then launches.  Resident passes
  // are left out of stream captures (a replay could not be chained) and of
  // streams that see part of the chip.
  bool takes_whole_locked(const Plan& plan, hipStream_t stream);
  // Resident passes over regions of up to `region` bytes on `stream` go
  // between these two (false: the device or the stream can run none now);
  // batches, which launch later, make sure of their room.
  bool whole_room_locked(uint64_t region);
  bool whole_begin_locked(uint64_t region, hipStream_t stream);
  void whole_end_locked(hipStream_t stream);
  // Device bytes the library holds for plain transposes on this device.
  int64_t held_bytes();
};

// Cache key of a plan: the arguments and the tuning epoch.
std::string plan_key(const int64_t* dims, const int* perm1, int rank, size_t elem, int n_sub,
                     double alpha);
Device* device_ctx(int* err);
int fail(int code, const char* fmt, ...);
void set_peak(size_t bytes);
void set_whole(int mode);
int validate(const void* dev, const int64_t* dims, const int* perm, int order, size_t elem);
// Enqueues the plan's passes on `stream`.  min_groups_cap > 0 lowers the
// launch configuration's workgroup floor per pass to at most that (callers
// whose passes share the GPU with other work).  tables: the passes' tables as
// copy_tables lays them out, instead of the plan's own copies.  whole: what
// takes_whole_locked has said.
int run_plan(Device* d, const Plan& plan, char* data, char* scratch, int64_t scratch_bytes,
             hipStream_t stream, std::vector<float>* times, bool whole, int64_t min_groups_cap = 0,
             const char* tables = nullptr);

}  // namespace eithot

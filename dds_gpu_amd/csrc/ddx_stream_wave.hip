// The streaming solver with one wave64 per search (ddx_wave.hpp): what ddx_stream.hip's kernel does
// with lanes or 16-lane teams, each deal's leads on waves of their own.
//
// A deal's latency is its slowest lead's, and a lead's speed is its search's: a search on a wave
// runs at 1.15M nodes/s alone, as in a batch, where a 16-lane team ran at 115k under full load and
// one lane at 20-150k. 1,500 eight-card deals through a ring of 256 slots: 1,011 ms with one lane per
// search, 52 ms with waves; 40,000 of them in a ring that holds all 932 and 283 ms, although 196,608
// lanes then stand against 4,096 waves. (80 VGPRs: 87 scalar registers are spilled to vector lanes, 12
// vector registers to scratch.)
//
// The ring is ddx_stream.hip's. Reading the host's counters costs a PCIe round trip, so only the
// first kPollers waves do it, whether idle or between the nodes of a search, and publish what they
// see in device memory; idle waves watch that. A job is reserved (atomic add) before it exists: an
// idle wave holds the next job number and waits until the deal is produced, so deals are taken in
// order and at once. Slot contents are read with system-scope relaxed loads, which bypass the
// caches: no acquire is needed to see them, and an acquire at system scope would invalidate the TT
// lines of every search on the chip.
#include <hip/hip_runtime.h>

#include "ddx_stream.h"

#if !DDX_TT_SIG && !DDX_SHARED_TT
#include "ddx_wave.hpp"

using namespace ddx;

namespace {

constexpr int kPollers = 8;

template <class V>
__device__ __forceinline__ V load_sys(const V* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}
template <class V>
__device__ __forceinline__ V load_dev(const V* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

}  // namespace

__global__ __launch_bounds__(1024) __attribute__((amdgpu_waves_per_eu(6, 6))) void stream_kernel_wave(StreamArgs a) {
  const long long search = (long long)blockIdx.x * (blockDim.x >> 6) + uni((int)(threadIdx.x >> 6));
  if (search >= a.lanes.searches) return;  // in the last block (no wave waits for another)
  WaveSearch W;
  W.init(a.lanes, search);
  const int jpd = a.jobs_per_deal;
  u32 jobs_done = 0, rounds = 0;
  // Shows the waves what the host has queued. End flags first: the host sets eof only after its
  // last produced. (By all lanes alike, as everything here: a branch on the lane would make the
  // compiler linearise the search, ddx_wave.hpp; a deal took 1.6 times as long.)
  auto look = [&]() {
    const unsigned long long e = (uni(load_sys(&a.ctl->eof)) ? 1u : 0u) | (uni(load_sys(&a.ctl->stop)) ? 2u : 0u);
    if (e) __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "");  // eof before the last produced
    const unsigned long long p = uni((u64)load_sys(&a.ctl->produced));
    if (p != uni((u64)load_dev(a.seen))) __hip_atomic_fetch_max(a.seen, p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (e & ~uni((u64)load_dev(a.seen + 1))) {
      // produced is complete before the flags say so
      __hip_atomic_fetch_or(a.seen + 1, e, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_AGENT);
    }
  };
  // Called at every trick start of a search: whether it must end.
  auto poll = [&]() -> bool {
    if ((++rounds & 255) != 0) return false;
    W.flush();
    if (search < kPollers) look();
    // (From the host itself: the polling waves may have ended at eof, and stop can come later.)
    return (rounds & 2047) == 0 && uni(load_sys(&a.ctl->stop)) != 0;
  };
  for (;;) {
    const long long job = (long long)one_lane_add(&a.counters[0], 1);
    const long long p = job / jpd;
    // Until the job's deal is produced, or no more will be.
    bool mine = false;
    for (;;) {
      if (search < kPollers) look();
      const u32 end = uni((u32)load_dev(a.seen + 1));
      if (end) __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");  // a set eof: the count is final
      mine = (long long)uni((u64)load_dev(a.seen)) > p && !(end & 2);
      if (mine || end) break;
      __builtin_amdgcn_s_sleep(64);
    }
    if (!mine) break;
    const long long slot = (long long)uni(load_sys(a.work + p % a.work_ring));
    const u64* h = a.hands + 4 * slot;
    W.new_deal(uni(load_sys(h)), uni(load_sys(h + 1)), uni(load_sys(h + 2)), uni(load_sys(h + 3)));
    const bool done = W.solve_job(
        jpd, (int)(job % jpd), a.seed_mode, poll,
        [&](int i) {  // bytes of 20-byte records: read as aligned words
          const long long at = 20 * slot + i;
          return (int)(uni(load_sys((const u32*)a.seeds + at / 4)) >> (8 * (at & 3)) & 0xFF);
        },
        [&](int i, int tricks) {
          a.out[20 * slot + i] = (uint8_t)tricks;
        });
    if (!done) break;
    jobs_done++;
    W.flush();
    // Count the job; its deal's last one publishes the slot.
    __threadfence_system();
    if (one_lane_add(&a.deal_done[slot], 1u) == (u32)jpd - 1) {
      __hip_atomic_store(&a.deal_done[slot], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      __threadfence_system();
      const u64 pos = one_lane_add(&a.counters[1], 1);
      one_lane_publish(&a.comp[pos % a.ring], (u32)slot + 1);
    }
  }
  if (search < kPollers) look();  // a stop that ended this wave's search reaches the idle waves
  W.flush();
  const u64 mine = W.totals();
  for (int i = 0; i < 3; i++) one_lane_add(&a.counters[2 + i], lane_get(mine, i));  // nodes, probes, hits
  one_lane_add(&a.counters[5], jobs_done);
  a.lanes.gen[search] = W.gen;
}

namespace ddx {

int stream_wave_grid(int device, long long asked, StreamGrid* g) {
  int cus = 0;
  HIPCHECK(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device));
  *g = stream_grid(asked, cus);
  return DDX_OK;
}

int launch_stream_wave(const StreamArgs& a, const StreamGrid& g, hipStream_t s) {
  hipLaunchKernelGGL(stream_kernel_wave, dim3((unsigned)g.blocks), dim3(64 * g.waves), 0, s, a);
  HIPCHECK(hipGetLastError());
  return DDX_OK;
}

}  // namespace ddx

#else
namespace ddx {

int stream_wave_grid(int, long long, StreamGrid* g) {
  *g = {0, 0, 0};
  return DDX_OK;
}
int launch_stream_wave(const StreamArgs&, const StreamGrid&, hipStream_t) { return DDX_E_ARG; }

}  // namespace ddx
#endif

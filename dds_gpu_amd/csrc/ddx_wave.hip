// One wave64 per search: the batch kernel for everything but saturated batches of very many
// searches (ddx_gpu.hip says which calls come here).
//
// What bounds a search with one lane of its own is that the 64 lanes of a wave run 64 unrelated
// searches: 18% of the lanes are active in an average instruction, a search alone in its wave
// advances at 150k nodes/s and one among 63 others at 20-30k. A batch then lasts as long as its
// heaviest job does at that rate, while most of the chip is idle. Here a wave runs one search, its
// state is uniform and lives in scalar registers, and the lanes serve the parts of a node that are
// parallel (ddx_wave.hpp). Measured: one search alone 1.15M nodes/s (nine-card endings); with
// every wave slot filled 2.9e9 nodes/s on eight-card endings, 3.3e9 on full deals -- above the
// lane kernel's 1.9e9 with 65,536 lanes, below its 3.8e9 with 196,608 lanes held to three waves
// per SIMD while its job queue lasts. 256 seven-card endings on 1,280 searches: 157 ms with lanes,
// 8.4 ms here; 500 nine-card endings 1,602 -> 96 ms; 65,536 eight-card endings on 196,608
// searches 829 -> 385 ms. (Times of random batches, both ways on the same deals; their heaviest jobs
// make batches of other deals differ by a quarter.)
//
// With every slot filled the kernel is bound by the scalar unit (one instruction per four cycles
// and SIMD: 181 scalar, 114 vector instructions and 22 jumps per node, the scalar ones 85% of the
// time). Alone, a node's 330 instructions take four cycles each and it waits half as long again:
// for jumps (38 cycles when taken), the TT and the way between the vector and the scalar unit. Six
// waves per SIMD (80 VGPRs; 83 scalar registers spilled to vector lanes, 5 vector registers to
// scratch): 5 and 6 measure 390 and 380 ms on 65,536 eight-card endings (and one search alone the same within 1%); 4 were 6% slower
// than 6, and 8 spill many more vector registers and cost one search 7%.
#include <hip/hip_runtime.h>

#include "ddx_wave.h"

#if !DDX_TT_SIG && !DDX_SHARED_TT
#include "ddx_wave.hpp"

using namespace ddx;

__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(6, 6))) void solve_kernel_wave(WaveArgs a) {
  const long long search = blockIdx.x, S = gridDim.x;
  WaveSearch W;
  W.init(a.lanes, search);
  u64 reported = 0;
  u32 jobs_done = 0, rounds = 0;
  // Called at every trick start: progress for the host and the stop flag, now and then.
  auto poll = [&]() -> bool {
    if ((++rounds & 255) == 0) {
      W.flush();
      a.wave_prog[2 * search] = jobs_done;  // (by all lanes: no branch, ddx_wave.hpp)
      a.wave_prog[2 * search + 1] = reported;
      if ((rounds & 1023) == 0 && uni((int)*a.stop)) return true;
    }
    return false;
  };
  const int jpd = a.jobs_per_deal;
  for (long long job = search; job < a.jobs;) {
    const long long deal = job / jpd;
    const u64* h = a.hands + 4 * deal;
    W.new_deal(uni(h[0]), uni(h[1]), uni(h[2]), uni(h[3]));
    const bool done = W.solve_job(
        jpd, (int)(job % jpd), a.seed_mode, poll,
        [&](int i) { return a.seeds ? (int)uni((u32)a.seeds[20 * deal + i]) : 7; },
        [&](int i, int tricks) {
          a.out[20 * deal + i] = (uint8_t)tricks;
        });
    if (!done) break;
    jobs_done++;
    W.flush();
    reported = lane_get(W.totals(), 0);
    job = S + (long long)one_lane_add(a.counters, 1);
  }
  W.flush();
  const u64 mine = W.totals();
  for (int i = 0; i < 5; i++) one_lane_add(a.counters + (i < 3 ? 1 + i : 3 + i), lane_get(mine, i));
  one_lane_add(a.counters + 4, jobs_done);
  a.wave_prog[2 * search] = jobs_done;
  a.wave_prog[2 * search + 1] = reported;
  a.lanes.gen[search] = W.gen;
}

namespace ddx {

int wave_capacity(int device, int* waves) {
  int per_cu = 0, cus = 0;
  HIPCHECK(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, solve_kernel_wave, 64, 0));
  HIPCHECK(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device));
  *waves = per_cu * cus;
  return DDX_OK;
}

int launch_wave_solve(const WaveArgs& a, long long searches, hipStream_t s) {
  hipLaunchKernelGGL(solve_kernel_wave, dim3((unsigned)searches), dim3(64), 0, s, a);
  HIPCHECK(hipGetLastError());
  return DDX_OK;
}

}  // namespace ddx

#else
namespace ddx {

int wave_capacity(int, int* waves) {
  *waves = 0;
  return DDX_OK;
}
int launch_wave_solve(const WaveArgs&, long long, hipStream_t) { return DDX_E_ARG; }

}  // namespace ddx
#endif

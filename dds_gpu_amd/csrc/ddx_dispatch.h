// Which configurations a batch handle accepts, which kernel runs a batch, and the grid of a stream:
// host logic only, without HIP, so that it can be checked on the CPU over every configuration.
#pragma once
#include "ddx.h"

namespace ddx {

constexpr int kTeamLanes = 16;  // lanes per search of a team

inline bool gpu_config_ok(const ddx_gpu_config& c, int min_log2, int max_log2) {
  if (c.tt_log2 < min_log2 || c.tt_log2 > max_log2 || (c.jobs_per_deal != 5 && c.jobs_per_deal != 20) ||
      c.seed_mode < 0 || c.seed_mode > 3)
    return false;
  if (c.block < 64 || c.block > 256 || c.block % 64 || c.lanes < 64 || c.lanes % 64 || c.lanes % c.block) return false;
  if ((c.team != 1 && c.team != kTeamLanes) || c.schedule < 0 || c.schedule > 3) return false;
  if (c.schedule == DDX_SCHED_THREAD && c.profile) return false;
  const bool split_schedule = c.schedule == DDX_SCHED_SPLIT && !c.profile;
  if (c.waves_per_simd != 0 && (c.waves_per_simd < 3 || c.waves_per_simd > 4 || !split_schedule)) return false;
  if (c.lds_lines != 0 && (c.lds_lines != 3 || c.team != 1 || !split_schedule || c.waves_per_simd == 4)) return false;
  if (c.split_min_nodes < 0) return false;
  return c.split_min_nodes == 0 || (c.team == 1 && split_schedule && !c.lds_lines && c.waves_per_simd != 4);
}

enum class BatchKernel {
  kNone,      // nothing to solve
  kWave,      // one wave per search (ddx_wave.hip)
  kSplit,     // the lane kernels (ddx_gpu.hip): splitting of the tail,
  kLds,       // the LDS cache of tag lines,
  kHeld,      // held to waves_per_simd waves,
  kSchedule,  // or by schedule, profile and, with a profile, team
};
struct Dispatch {
  BatchKernel kernel;
  long long searches;  // the kernel uses this many of the handle's TTs, stacks and generations
  int waves_per_simd;  // lane kernels: 0, 3 or 4 (beside a stream never the compiler's own 230 to 260 VGPRs
                       // where there is a kernel held to 168)
};

// Batches run with one wave per search (ddx_wave.hip), but for three kinds, which stay on lanes.
//
// The measuring options (stage profile, LDS line cache, splitting) exist in the lane kernels only.
//
// saturated: more than 65,536 lanes with more than two jobs each. Two jobs a lane are where lanes
// begin to win for full deals under a time limit, the work that such lane counts are tuned for: on
// 196,608 lanes for 80 s, 100,000 deals (2.5 jobs a lane, TT_LOG2 12) give 53,854 whole tables with
// lanes and 38,409 with waves, 78,000 deals (2.0, TT_LOG2 11) 42,134 and 33,562, 20,000 deals (0.5,
// 40 s) 10,048 and 17,769. Lanes start every job early and leave the heavy ones for last. Batches that
// run to their end are the other way round up to many jobs a lane: eight-card endings 807 ms with
// lanes and 380 with waves at 1.7 jobs a lane, 827 and 487 at 2.2, 1,150 and 895 at 4.1, 1,800 and 1,746
// at 8.1; six-card endings 180 and 178 at 4.1, 311 and 354 at 8.1. (65,536 lanes or fewer, two waves per
// SIMD at most, enter 1.9e9 nodes/s and waves 2.9e9 to 3.3e9.)
//
// corner: at most 1,024 lanes with more than eight jobs each. No figure speaks for lanes here: 3,000
// ten-card deals on 1,024 lanes take 16.4 s, and 0.80 s with waves; 1,700 eight-card ones 1.33 s
// and 44 ms. (Beside it another batch of 351 ms takes 355-378 ms all that time, or 405 ms once.) Such a
// handle's long batches run as they always have, on the 16 waves that its lanes fill, because the test
// of stop requests (tests/test_gpu.py) takes it that the former batch still runs after 1.5 s. With team 16
// and 16 times the lanes, the same number of searches runs on waves.
//
// Beside an open stream both of these rules are off: most lane kernels need more registers than the
// stream leaves (kRoomVgprs below), and would wait until it is closed.
//
// wave_cap: waves of the wave kernel that the device holds at once; 0 in builds without it. beside:
// a stream is open on the device.
inline Dispatch dispatch(const ddx_gpu_config& c, int wave_cap, long long jobs, bool beside) {
  if (jobs <= 0) return {BatchKernel::kNone, 0, 0};
  const bool measuring = c.profile || c.lds_lines || c.split_min_nodes > 0;
  const bool saturated = c.team == 1 && c.lanes > 65536 && jobs > 2 * c.lanes;
  const bool corner = c.team == 1 && c.lanes <= 1024 && jobs > 8 * c.lanes;
  if (wave_cap > 0 && !measuring && (beside || (!saturated && !corner))) {
    long long s = c.lanes / c.team;
    if (s > wave_cap) s = wave_cap;
    return {BatchKernel::kWave, s < jobs ? s : jobs, 0};
  }
  const int w = beside && !c.waves_per_simd ? 3 : c.waves_per_simd;
  if (c.split_min_nodes > 0) return {BatchKernel::kSplit, c.lanes, w};
  if (c.lds_lines) return {BatchKernel::kLds, c.lanes, w};
  if (c.waves_per_simd) return {BatchKernel::kHeld, c.lanes, w};
  // Teams have a lane kernel only for the stage profile.
  return {BatchKernel::kSchedule, c.profile ? c.lanes / c.team : c.lanes, 0};
}

// The wave-per-search stream kernel stays on the device until the stream is closed, and the net's
// kernels, whose seeds the stream may wait for, have to start meanwhile. A SIMD has 512 VGPRs and a
// wave of the stream takes 80. So a stream has at most 16 waves per CU, and they come in one block
// per CU, two of which no CU can hold: every SIMD has four waves of it and 192 VGPRs left, in which
// the net's small kernels (ddx_mlp.hip) find room on every CU. (The node rate of 4 and 6 waves per
// SIMD differs by 10%.) Fewer searches make smaller blocks, so that they still spread over the CUs.
constexpr int kStreamWavesPerCu = 16, kStreamVgprs = 80, kSimdVgprs = 512;
constexpr int kRoomVgprs = kSimdVgprs - kStreamWavesPerCu / 4 * kStreamVgprs;  // per SIMD, beside a stream

struct StreamGrid {
  long long searches;
  int blocks, waves;  // waves per block; the last block may hold fewer searches
};
inline StreamGrid stream_grid(long long asked, int cus) {
  const long long most = (long long)kStreamWavesPerCu * cus, n = asked < most ? asked : most;
  const int waves = (int)((n + cus - 1) / cus);
  return {n, (int)((n + waves - 1) / waves), waves};
}

}  // namespace ddx

// The streaming kernels' shared arguments, and the wave-per-search stream kernel's launch
// (ddx_stream_wave.hip).
#pragma once
#include "ddx_dispatch.h"
#include "ddx_lanes.hpp"

namespace ddx {

struct StreamCtl {
  long long produced;
  int eof;
  int stop;
  long long pad[6];
};

struct StreamArgs {
  LaneView lanes;
  const u64* hands;
  const uint8_t* seeds;
  uint8_t* out;
  const u32* work;
  u32* comp;
  StreamCtl* ctl;
  unsigned long long* counters;  // [0] next job, [1] comp_head, [2] nodes, [3] probes, [4] hits, [5] jobs
  u32* deal_done;                // per slot
  long long ring, work_ring;
  int jobs_per_deal, seed_mode;
  unsigned long long* seen;      // device: the host's counters as the polling waves last saw them:
                                 // [0] produced, [1] end flags (1 = eof, 2 = stop)
};

// The wave-per-search stream kernel's grid for this many searches; no searches in the builds that
// have no such kernel (signature entries, shared TT).
int stream_wave_grid(int device, long long asked, StreamGrid* g);
int launch_stream_wave(const StreamArgs& a, const StreamGrid& g, hipStream_t s);

}  // namespace ddx

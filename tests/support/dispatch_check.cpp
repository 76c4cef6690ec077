// Every configuration that a batch handle accepts, against the storage it allocates (lanes / team
// TTs, stacks and generations): no batch size may reach a kernel that indexes past them, an empty
// batch reaches none. And the stream's grid: its searches, in at most a block per CU. Prints the
// configurations tried, the batches, and the faults.
#include <stdio.h>

#include <initializer_list>

#include "ddx_dispatch.h"

using namespace ddx;

int main() {
  long configs = 0, batches = 0, bad = 0;
  const long long lanes[] = {64, 128, 256, 1024, 1280, 4096, 65536, 65792, 131072, 196608};
  for (long long L : lanes)
    for (int block = 64; block <= 256; block += 64)
      for (int team : {1, 2, 16})
        for (int schedule = -1; schedule <= 4; schedule++)
          for (int profile : {0, 1})
            for (int waves = 0; waves <= 5; waves++)
              for (int lds : {0, 3})
                for (int split : {0, 64})
                  for (int jpd : {5, 20}) {
                    ddx_gpu_config c{0, L, 10, jpd, schedule, 0, block, profile, team, 0, waves, lds, split};
                    if (!gpu_config_ok(c, 9, 20)) continue;
                    configs++;
                    for (int mode = 0; mode < 4; mode++) {
                      const int cap = mode & 1 ? 6144 : 0;
                      const bool beside = mode & 2;
                      if (cap == 0 && team != 1) continue;  // the builds without wave kernels have no teams
                      for (long long n : {0ll, 1ll, 12ll, 13ll, 409ll, 410ll, 2000ll, 13107ll, 26215ll, 100000ll}) {
                        const Dispatch d = dispatch(c, cap, n * jpd, beside);
                        batches++;
                        const bool none = d.kernel == BatchKernel::kNone, wave = d.kernel == BatchKernel::kWave;
                        if (d.searches > L / team || none != (n == 0) || none != (d.searches == 0)) bad++;
                        if (wave && (d.searches > cap || d.searches > n * jpd || profile || lds || split)) bad++;
                        if (!wave && !none && d.searches != (profile ? L / team : L)) bad++;  // the lane kernels' grids
                        // Beside a stream: waves, or a lane kernel held to 168 or 128 VGPRs, but for the profile.
                        if (beside && cap && !none && !wave && !profile && d.waves_per_simd < 3) bad++;
                        if (!beside && !none && !wave && d.waves_per_simd != waves) bad++;
                      }
                    }
                  }
  for (int cus = 1; cus <= 320; cus++)
    for (long long n : {1ll, 4ll, 64ll, 255ll, 256ll, 257ll, 2048ll, 4096ll, 65536ll, 196608ll}) {
      const StreamGrid g = stream_grid(n, cus);
      const bool covers = (long long)g.blocks * g.waves >= g.searches && (long long)(g.blocks - 1) * g.waves < g.searches;
      const bool most = g.searches == n || g.searches == 16ll * cus;
      if (!covers || !most || g.searches < 1 || g.searches > n || g.blocks > cus || g.waves < 1 || g.waves > 16) bad++;
    }
  // A full block leaves kRoomVgprs on every SIMD, and no room for a second one.
  if (kRoomVgprs != 512 - 4 * kStreamVgprs || 8 * kStreamVgprs <= 512) bad++;
  printf("%ld %ld %ld\n", configs, batches, bad);
  return bad != 0;
}

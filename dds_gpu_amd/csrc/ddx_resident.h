// How many streams are open on each device. A stream's kernel stays there until it is closed, and
// kernels that need most of a CU (the net's large ones, ddx_mlp.hip) would wait for that.
//
// Such a kernel is launched under the lock and only while the device has no stream. ddx_stream_open
// counts its stream first and then synchronizes the device (lanes_alloc), so that every large kernel
// launched before has ended when the stream's starts. One count serves all builds of the library in
// a process: ddx_host.cpp.
#pragma once
#include <mutex>

namespace ddx {

struct Resident {
  std::mutex mu;
  int& streams(int device) { return n[device >= 0 && device < kDevices ? device : kDevices]; }

 private:
  static constexpr int kDevices = 64;
  int n[kDevices + 1] = {};  // the last: every device beyond
};
Resident& resident();

inline void count_stream(int device, int by) {
  std::lock_guard<std::mutex> lock(resident().mu);
  resident().streams(device) += by;
}

}  // namespace ddx

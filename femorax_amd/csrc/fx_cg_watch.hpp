// The host's side of a CG solve that runs on the device: it queues iterations ahead of the progress
// the device writes to pinned memory, and ends once the device has stopped. Host code only, over
// any Device, so that it runs against a scripted one as well:
//   int it(), bool done()       the progress and the stop, as the device has written them
//   int launch(int i)           queue iterations from i on (one, or a captured group of them)
//   int idle(bool&)             whether everything queued has run
//   int stalled()               the error of a device that has run its work without reporting it
#pragma once

#include <cstdint>
#include <thread>

namespace fx {

// A wait on memory that the device writes. Each look pauses the core and every 64th offers it to
// another thread (a serving process has a waiting thread per solver); true where it is time to ask
// whether the device still runs at all. A 48^3 block solved to 1e-8 takes 20.3 ms, 22.8 where the
// host looks without a pause.
struct DeviceWait {
  uint32_t looks = 0;
  bool pause() {
    ++looks;
    if (looks % 64) __builtin_ia32_pause();
    else std::this_thread::yield();
    return looks % 4096 == 0;
  }
};

// Iterations queued beyond the last one the device has reported: enough to hide the host's launch
// times, and the only iterations that run as no-ops after the stop (three or four launches each;
// polling by copies in groups of up to 64 iterations ran 30 of them on average).
constexpr int kQueueAhead = 8;

enum class CgNext { kQueue, kWait, kStop, kStalled };

// `launched` of at most max_it iterations are queued, in groups of `group`.
inline CgNext cg_next(int launched, int max_it, int group, int it, bool done) {
  if (done) return CgNext::kStop;
  return launched < max_it && launched - it < kQueueAhead + group - 1 ? CgNext::kQueue : CgNext::kWait;
}

// The same once the stream has been found idle, from progress read after that: the host was held up
// for as long as the queue took, and goes on. Where the product of iteration i + 1 reports iteration
// i (box_forms_direction), the last of an idle queue is not reported yet; more than one unreported,
// or none left to queue, is a device that ran its work without a result.
inline CgNext cg_next_idle(int launched, int max_it, int it, bool done) {
  if (done) return CgNext::kStop;
  return launched < max_it && launched - it <= 1 ? CgNext::kQueue : CgNext::kStalled;
}

template <typename Device>
int cg_watch(Device& dev, int max_it, int group) {
  DeviceWait wait;
  for (int launched = 0;;) {
    const int it = dev.it();
    CgNext next = cg_next(launched, max_it, group, it, dev.done());
    if (next == CgNext::kWait) {
      if (!wait.pause()) continue;
      bool idle = false;
      if (int rc = dev.idle(idle)) return rc;
      if (!idle) continue;
      next = cg_next_idle(launched, max_it, dev.it(), dev.done());
    }
    if (next == CgNext::kStop) return 0;
    if (next == CgNext::kStalled) return dev.stalled();
    if (next == CgNext::kQueue) {
      if (int rc = dev.launch(launched)) return rc;
      launched += group;
      wait = DeviceWait{};
    }
  }
}

}  // namespace fx

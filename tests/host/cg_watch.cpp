// cg_watch over a scripted device: solves that stop after `stop` iterations (or at max_it), reported
// at once or by the iteration that follows, one at a time or in captured groups, on a host that is
// kept up to date or held up until everything queued has run. Prints the first solve that fails.
#include <algorithm>
#include <cstdio>
#include <random>

#include "../../femorax_amd/csrc/fx_cg_watch.hpp"

namespace {

constexpr int kStalledCode = 77;

struct Device {
  int max_it, stop, group;
  bool next_reports;  // iteration i is reported by the product of iteration i + 1 (the tiles form the direction)
  int held_up;        // in 64ths: how often the host is held up between its look and the stream's query
  int broken_at;      // iterations from here on run without a report
  std::mt19937 rng;
  int queued = 0, ran = 0, reported = 0;
  bool stopped = false;

  void run(int n) {
    for (; n > 0 && ran < queued && !stopped; --n) {
      ++ran;
      if (ran > broken_at) continue;
      // the last of a captured group, and the last of all, decide by themselves
      const bool decides = !next_reports || (group > 1 && ran % group == 0) || ran == max_it;
      if (next_reports && ran > 1) report(ran - 1);
      if (decides && !stopped) report(ran);
    }
    if (stopped) ran = queued;  // no-ops
  }
  void report(int i) {
    if (stopped) return;
    reported = i;
    if (i >= stop || i >= max_it) stopped = true;
  }
  int it() {
    run(rng() % 2048 == 0);  // the device goes on between the looks
    return reported;
  }
  bool done() const { return stopped; }
  int launch(int i) {
    if (i != queued) return 1;
    queued += group;
    return 0;
  }
  int idle(bool& is) {
    if (static_cast<int>(rng() % 64) < held_up) run(queued);
    is = ran >= queued;
    return 0;
  }
  int stalled() { return kStalledCode; }
};

int solve(int max_it, int stop, int group, bool next_reports, int held_up, int broken_at, unsigned seed) {
  Device d{max_it, stop, group, next_reports, held_up, broken_at, std::mt19937(seed)};
  if (stop <= 0 || max_it <= 0) d.stopped = true;  // decided before the first iteration
  const int rc = fx::cg_watch(d, max_it, group);
  if (rc == 0 && (!d.stopped || d.reported != std::max(0, std::min(stop, max_it)))) return 2;
  return rc;
}

}  // namespace

int main() {
  constexpr int kNever = 1 << 30;
  for (int group : {1, 8})
    for (bool next_reports : {false, true})
      for (int held_up : {0, 1, 64})
        for (int max_it : {0, 1, 7, 8, 9, 64, 200})
          for (int stop : {0, 1, 6, 17, kNever})
            for (unsigned seed = 0; seed < 3; ++seed)
              if (int rc = solve(max_it, stop, group, next_reports, held_up, kNever, seed)) {
                std::printf("code %d: group %d, reported by the next %d, held up %d, at most %d iterations, stop after %d\n",
                            rc, group, next_reports, held_up, max_it, stop);
                return 1;
              }
  // a device that stops reporting is an error, not an endless wait
  for (int group : {1, 8})
    for (int broken_at : {0, 3, 20})
      if (solve(200, kNever, group, false, 64, broken_at, 1) != kStalledCode) {
        std::printf("group %d: no error from a device that reports nothing past iteration %d\n", group, broken_at);
        return 1;
      }
  std::puts("ok");
  return 0;
}

// Steps that the engine runs in a schedule of its own choice (StepLaunch in
// storm_amd/csrc/launch_policy.h) on made-up transport rates: the schedule
// watch learns nothing from them.  Prints one "ok" line per check; exits 1 on
// the first failure.
#include <cstdio>
#include <cstdlib>
#include <stdexcept>

#include "launch_policy.h"

using storm::gpu::LaunchPolicy;
using storm::gpu::StepLaunch;

namespace {

constexpr int32_t kPass = STORM_GPU_SCHEDULE_PASS, kRefill = STORM_GPU_SCHEDULE_REFILL;

void check(bool c, const char *what) {
  if (!c) {
    std::printf("FAIL %s\n", what);
    std::exit(1);
  }
}

// rates that jump by up to 40% from step to step
double noisy(int step) { return 1.0 + 0.4 * ((step * 2654435761u >> 16) % 101u) / 100.0; }

// one step: the schedule it ran in
int32_t run(LaunchPolicy &p, int32_t set, double rate) {
  StepLaunch l(p, set);
  const int32_t ran = p.schedule;
  l.restore();
  l.done(rate, 1.0);
  return ran;
}

bool same_watch(const LaunchPolicy &a, const LaunchPolicy &b) {
  return a.schedule == b.schedule && a.watch_state == b.watch_state && a.watch_n == b.watch_n &&
         a.watch_every == b.watch_every && a.watch_prev == b.watch_prev;
}

}  // namespace

int main() {
  // 500 steps, each held to passes: no probe, no switch, no count
  {
    LaunchPolicy p;
    p.schedule = kRefill;
    const LaunchPolicy before = p;
    for (int k = 0; k < 500; ++k) {
      check(run(p, kPass, noisy(k)) == kPass, "held: runs the schedule set");
      check(same_watch(p, before), "held: the watch stays as it was");
    }
    std::printf("held steps ok\n");
  }
  // own and held steps in turn: the policy is what the own steps alone make it,
  // but for the probes, each of which the held step after it drops
  {
    LaunchPolicy p;
    p.schedule = kRefill;
    int probes = 0;
    for (int k = 0; k < 400; ++k) {
      if (run(p, -1, noisy(2 * k)) == kPass) ++probes;
      run(p, kPass, 100.0 * noisy(2 * k + 1));
      check(p.schedule == kRefill && p.watch_state == 0, "in turn: no switch on the held steps' rates");
    }
    check(probes > 0, "in turn: the own steps still probe");
    std::printf("alternating steps ok\n");
  }
  // a probe that did not end (its step threw) before a held step
  {
    LaunchPolicy p;
    p.schedule = kRefill;
    for (int k = 0; k < 16; ++k) run(p, -1, 1.0);
    try {
      StepLaunch l(p, -1);
      check(p.schedule == kPass && p.watch_state == 1, "thrown: the 17th step probes");
      throw std::runtime_error("a step that fails");
    } catch (const std::runtime_error &) {
    }
    run(p, kPass, 5.0);
    check(p.schedule == kRefill && p.watch_state == 0 && p.watch_n == 0, "thrown: the probe is dropped");
    std::printf("dropped probe ok\n");
  }
  // a held step that throws leaves the engine's own schedule
  {
    LaunchPolicy p;
    p.schedule = kRefill;
    try {
      StepLaunch l(p, kPass);
      check(p.schedule == kPass, "held, thrown: runs the schedule set");
      throw std::runtime_error("a step that fails");
    } catch (const std::runtime_error &) {
    }
    check(p.schedule == kRefill, "held, thrown: the own schedule is back");
    std::printf("held step that throws ok\n");
  }
  return 0;
}

// pcg_wait.hh — the host's side of a PCG run's progress in pinned memory: what a look at it says, and the wait for more.
#pragma once
#include <cstdint>
#include <thread>

#include "ik_internal.hh"

namespace ik {

// Whether run `run` has started, as the device's last store to the mirror says; then `state` is iterations << 2 | done
// and `flagged` whether the element kernels ahead of the run found an invalid element. The device stores the flags
// behind a fence before the run's first state, so they are there with any state of the run. (A copy of the flag enqueued
// ahead of the run is not: only a synchronisation of its stream makes its target readable.)
inline bool pcgLook(const PcgMirror& m, uint32_t run, unsigned& state, bool& flagged) {
  const unsigned long long s = __atomic_load_n(&m.state, __ATOMIC_ACQUIRE);
  if ((uint32_t)(s >> 32) != run) return false;
  state   = (unsigned)s;
  flagged = m.err[0] != ~0ull || m.err[1] != ~0ull;
  return true;
}

// Looks until look() says true, with check() now and then for what would make it wait without end. After a short while
// each look leaves the core to any other thread that is ready (where there is none it comes back in a fraction of a
// microsecond): otherwise solves by more threads than cores wait for each other by the scheduler's time slices, 4 ms each
// time (400 hand-overs between two waiting threads on one core: 1.6 s against a millisecond).
template <class Look, class Check>
void pcgSpin(Look look, Check check) {
  for (unsigned spin = 1; !look(); ++spin) {
    if (spin % 4096 == 0) check();
    if (spin < 64)
      __builtin_ia32_pause();
    else
      std::this_thread::yield();
  }
}

}  // namespace ik

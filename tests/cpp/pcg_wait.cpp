// pcg_wait.cpp — the host's side of a PCG run's progress (ikarus_amd/csrc/pcg_wait.hh) on the CPU: a plain struct stands
// for the pinned mirror, threads for the device and for other solves.
#include <cstdio>
#include <cstring>

#include "../../ikarus_amd/csrc/pcg_wait.hh"

namespace {

int bad = 0;
void expect(bool ok, const char* what) {
  if (ok) return;
  std::printf("FAILED: %s\n", what);
  ++bad;
}

constexpr unsigned long long kNone = ~0ull;
unsigned long long stateOf(uint32_t run, unsigned iters, unsigned done) {
  return (unsigned long long)run << 32 | iters << 2 | done;
}

// an invalid element is known with the run's first state, from what the device stored with it alone
void flags() {
  ik::PcgMirror m{};
  unsigned state = 77;
  bool flagged   = true;
  m.err[0] = m.err[1] = kNone;
  m.state             = stateOf(4, 12, 1);
  expect(!ik::pcgLook(m, 5, state, flagged) && state == 77, "another run's state is not this run's");
  m.state = stateOf(5, 0, 0);
  expect(ik::pcgLook(m, 5, state, flagged) && state == 0 && !flagged, "first state, no invalid element");
  m.state = stateOf(5, 8, 0);
  expect(ik::pcgLook(m, 5, state, flagged) && state == 32 && !flagged, "progress");
  for (int k = 0; k < 2; ++k)  // det C of an element, a singular D of one
    for (unsigned done : {0u, 1u, 2u}) {
      m.err[0] = m.err[1] = kNone;
      m.err[k]            = 0;  // element 0
      m.state             = stateOf(6 + k, 0, done);
      expect(ik::pcgLook(m, 6 + k, state, flagged) && flagged && (state & 3) == done, "an invalid element");
    }
}

}  // namespace

int main(int argc, char** argv) {
  if (argc > 1 && !std::strcmp(argv[1], "flags")) flags();
  std::printf(bad ? "FAILED\n" : "OK\n");
  return bad ? 1 : 0;
}

// pcg_record.hh — what the recording thread of a PCG convergence test writes: the run's scalars and, in pinned host
// memory, its progress.
#pragma once
#include "ik_internal.hh"

namespace ik {

// not after every iteration: a store to host memory takes the kernel a microsecond or two more
__device__ inline void pcgPublish(const PcgScalars* sc, double rr, int iters, int done) {
  if (!done && iters % kPcgPublish) return;
  PcgMirror* m = sc->mirror;
  if (done) {
    m->rr = rr;
    m->bb = sc->bb;
    __threadfence_system();
  }
  __hip_atomic_store(&m->state, (unsigned long long)sc->run << 32 | (unsigned)iters << 2 | (unsigned)done,
                     __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}
__device__ inline void pcgRecord(PcgScalars* sc, double rr, double rz, double beta, bool converged, int maxIter) {
  int iters = sc->iters, done = 1;
  sc->rr    = rr;
  if (!converged) {
    sc->beta   = beta;
    sc->rz_new = rz;
    sc->iters  = ++iters;
    done       = iters >= maxIter ? 2 : 0;
  }
  if (done) sc->done = done;
  pcgPublish(sc, rr, iters, done);
}

}  // namespace ik

// sparse.hip — sliced-ELL 3x3-block SpMV, reductions and the preconditioned CG solvers.
//
// FP64 Jacobi-PCG follows Eigen's ConjugateGradient with DiagonalPreconditioner, the reference's
// si_ConjugateGradient (ikarus/solver/linearsolver/linearsolver.cpp:23-24): x0 = 0,
// stop when ||r||^2 < tol^2 ||b||^2, iteration count as Eigen reports it.
// The mixed form runs the same recurrence in FP32 on an FP32 tangent with a 3x3 block-Jacobi
// preconditioner, wrapped in FP64 iterative refinement (r = b - K x accumulated in FP64).
//
// All PCG scalars live on the device; each kernel reads a `done` flag so the host can enqueue
// iterations ahead of the test: the iterate after convergence is exactly the one Eigen's loop returns.
#include "ik_internal.hh"
#include "pcg_record.hh"
#include "pcg_wait.hh"
#include "wave_reduce.hh"

namespace ik {
namespace {

// Block rows per wavefront of the SpMV lane layouts: FP64 values 3 lanes per row (21 rows, lane 63 idles),
// FP32 values one lane per row (64 rows). G wavefronts share the rows of one, taking every G-th block each, so that a
// small matrix still puts enough loads in flight: a lane's blocks are a chain of round trips to the caches.
template <typename TV>
constexpr int spmvRowsPerWave() {
  return sizeof(TV) == 4 ? 64 : 21;
}
constexpr int SPMV_BS = 256;
template <typename TV, int G>
constexpr int spmvRowsPerBlock() {
  return SPMV_BS / 64 / G * spmvRowsPerWave<TV>();
}

// block-wide sum; result valid in thread 0
template <int BS>
__device__ inline double blockSum(double v) {
  __shared__ double red[BS / 64];
  v = waveSum(v);
  const int w = threadIdx.x >> 6, l = threadIdx.x & 63;
  if (l == 0) red[w] = v;
  __syncthreads();
  double s = 0.0;
  if (threadIdx.x == 0)
#pragma unroll
    for (int i = 0; i < BS / 64; ++i) s += red[i];
  __syncthreads();
  return s;
}

// y = K x over the sliced-ELL block storage (slice of kSellRows = 64 block rows, block j of row r of slice s
// at slot sellStart[s] + 64 j + r, 9 values per slot); optional fused partial dot d = sum_i x_i y_i per
// block. Two lane layouts:
//  FP64 values: lane (r, k), row r = lane / 3 (21 rows per wavefront), output component k: for a fixed j the
//   wavefront's 21 rows read 21 adjacent 72-byte blocks (1,512 contiguous bytes), each lane its block row.
//  FP32 values: one lane per block row, the 3 outputs of the row per lane, a wavefront = one slice: for a
//   fixed j the 64 lanes read 64 adjacent 36-byte blocks (2304 contiguous bytes). Each lane runs to the
//   slice's longest row; padding slots hold zeros with the row's own column.
// 64^3 pattern, alone: FP32 48.6 us against 62.3 us for 3 lanes per row over CSR (21 rows per wavefront);
// FP64 108.4 us against 119.3 us for the former layout with one lane per block entry (7 rows per wavefront).
// Both issue the loads of 3 blocks before summing their products (FP64: 2, 4, 5, 6 and 9 gave 111.3, 111.9, 114.8,
// 116.5 and 121.1 us; FP32 53.2 us against 56.3, 60.9 and 68.4 us for 2, 4 and 6).
constexpr int SPMV_UNROLL = 3;
static_assert(kSellRows == 64, "one slice per wavefront");

// a[k] = sum of (K x)[3 row + k], k = 0..2, over the slots j = g, g + G, ... of the slice of row `row` (a lane per row)
template <int G, typename TA, typename TV, typename TX>
__device__ inline void rowSell3(const int32_t* __restrict__ sellStart, const int32_t* __restrict__ scol,
                                const TV* __restrict__ val, const TX* __restrict__ x, int64_t row, int g, TA a[3]) {
  const int64_t s = row >> 6;
  const int r     = (int)(row & 63);
  const int32_t s0 = sellStart[s];
  const int w      = (sellStart[s + 1] - s0) >> 6;
  const TV* v0     = val + ((int64_t)s0 + r) * 9;
  const int32_t* C = scol + s0 + r;
  TA a0 = TA(0), a1 = TA(0), a2 = TA(0);
#pragma unroll SPMV_UNROLL
  for (int j = g; j < w; j += G) {
    const int64_t c = (int64_t)C[j * kSellRows] * 3;
    const TA x0 = (TA)x[c], x1 = (TA)x[c + 1], x2 = (TA)x[c + 2];
    const TV* v = v0 + (int64_t)j * (kSellRows * 9);
    a0 += (TA)v[0] * x0 + (TA)v[1] * x1 + (TA)v[2] * x2;
    a1 += (TA)v[3] * x0 + (TA)v[4] * x1 + (TA)v[5] * x2;
    a2 += (TA)v[6] * x0 + (TA)v[7] * x1 + (TA)v[8] * x2;
  }
  a[0] = a0;
  a[1] = a1;
  a[2] = a2;
}

// (K x)[3 row + k] over the blocks j = g, g + G, ... of row `row` (FP64 lane layout). The lane keeps one sum per
// column l, a_l = sum_j K_j[k][l] x_j[l] in block order, and returns a_0 + (a_1 + a_2).
template <int G, typename TA, typename TV, typename TX>
__device__ inline TA rowSell1(const int32_t* __restrict__ rowptr, const int32_t* __restrict__ sellStart,
                              const int32_t* __restrict__ scol, const TV* __restrict__ val,
                              const TX* __restrict__ x, int64_t row, int k, int g) {
  const int64_t base = (int64_t)sellStart[row >> 6] + (row & 63);
  const TV* v0       = val + base * 9 + 3 * k;
  const int32_t* C   = scol + base;
  const int n        = rowptr[row + 1] - rowptr[row];
  TA a0 = TA(0), a1 = TA(0), a2 = TA(0);
  int j = g;
  for (; j + (SPMV_UNROLL - 1) * G < n; j += SPMV_UNROLL * G) {
    int32_t c[SPMV_UNROLL];
    TV v[SPMV_UNROLL][3];
#pragma unroll
    for (int u = 0; u < SPMV_UNROLL; ++u) {
      c[u] = C[(j + u * G) * kSellRows];
#pragma unroll
      for (int l = 0; l < 3; ++l) v[u][l] = v0[(int64_t)(j + u * G) * (kSellRows * 9) + l];
    }
#pragma unroll
    for (int u = 0; u < SPMV_UNROLL; ++u) {
      const int64_t xc = (int64_t)c[u] * 3;
      a0 += (TA)v[u][0] * (TA)x[xc];
      a1 += (TA)v[u][1] * (TA)x[xc + 1];
      a2 += (TA)v[u][2] * (TA)x[xc + 2];
    }
  }
  for (; j < n; j += G) {
    const TV* vj     = v0 + (int64_t)j * (kSellRows * 9);
    const int64_t xc = (int64_t)C[j * kSellRows] * 3;
    a0 += (TA)vj[0] * (TA)x[xc];
    a1 += (TA)vj[1] * (TA)x[xc + 1];
    a2 += (TA)vj[2] * (TA)x[xc + 2];
  }
  return a0 + (a1 + a2);
}

// The rows of row block rb: out(i, x_i, y_i) is called once for each entry i = 3 row + k of y = K x, accumulated in TA.
// With G > 1 the partial sums of the G wavefronts that share rows meet in LDS, summed in wavefront order.
template <int G, typename TA, typename TV, typename TX, typename F>
__device__ inline void spmvRows(const int32_t* __restrict__ rowptr, const int32_t* __restrict__ sellStart,
                                const int32_t* __restrict__ scol, const TV* __restrict__ val,
                                const TX* __restrict__ x, int64_t nrows, unsigned rb, F out) {
  constexpr int NO = sizeof(TV) == 4 ? 3 : 1;  // outputs per lane
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, g = wave % G;
  const int rl      = sizeof(TV) == 4 ? lane : lane / 3;
  const int k       = sizeof(TV) == 4 ? 0 : lane - 3 * rl;
  const int64_t row = (int64_t)rb * spmvRowsPerBlock<TV, G>() + wave / G * spmvRowsPerWave<TV>() + rl;
  const bool in     = rl < spmvRowsPerWave<TV>() && row < nrows;
  TA a[NO];
  if (in) {
    if constexpr (NO == 3)
      rowSell3<G, TA>(sellStart, scol, val, x, row, g, a);
    else
      a[0] = rowSell1<G, TA>(rowptr, sellStart, scol, val, x, row, k, g);
  }
  if constexpr (G > 1) {
    __shared__ TA part[SPMV_BS / 64][NO][64];
    if (in)
#pragma unroll
      for (int o = 0; o < NO; ++o) part[wave][o][lane] = a[o];
    __syncthreads();
    if (in && g == 0)
#pragma unroll
      for (int w = 1; w < G; ++w)
#pragma unroll
        for (int o = 0; o < NO; ++o) a[o] += part[wave + w][o][lane];
  }
  if (in && g == 0)
#pragma unroll
    for (int o = 0; o < NO; ++o) out(row * 3 + k + o, a[o]);
}

// rev: workgroup i takes row block gridDim.x - 1 - i (the partial stays at the row block's index, so the fold
// order and y are the same either way). The PCG loops alternate the direction from one iteration to the next:
// the matrix (FP32 259 MB, FP64 518 MB, plus 29 MB of column indices) is larger than the 256 MB last-level
// cache, and a pass in one direction evicts what the next pass in the same direction reads first, while a pass
// in the other direction starts on the part just read (64^3: FP64 134.4 -> 119.0 us, FP32 57.0 -> 53.3 us).
template <typename TV, typename TX, bool DOT, int G>
__global__ __launch_bounds__(SPMV_BS) void spmvKernel(const int32_t* __restrict__ rowptr,
                                                               const int32_t* __restrict__ sellStart,
                                                               const int32_t* __restrict__ scol,
                                                               const TV* __restrict__ val, const TX* __restrict__ x,
                                                               TX* __restrict__ y, int64_t nrows,
                                                               double* __restrict__ partial,
                                                               const PcgScalars* __restrict__ sc, int rev) {
  if (sc && sc->done) return;
  const unsigned rb = rev ? gridDim.x - 1u - blockIdx.x : blockIdx.x;
  double d = 0.0;
  spmvRows<G, TX>(rowptr, sellStart, scol, val, x, nrows, rb, [&](int64_t i, TX yi) {
    y[i] = yi;
    if (DOT) d += (double)x[i] * (double)yi;
  });
  if (DOT) {
    const double s = blockSum<SPMV_BS>(d);
    if (threadIdx.x == 0) partial[rb] = s;
  }
}

// Convergence test and beta of a PCG iteration from the update kernel's partials (r.r, r.z). Every calling block folds
// them in the same fixed order, so all blocks agree bitwise; the one with `record` writes the scalars. test() returns
// false when the iteration has converged. beta = r.z / (r.z of the previous iterate), which only the update kernel
// writes. fetch() issues the loads, so that they are in flight with the caller's.
template <int BS>
struct PcgTest {
  const double* __restrict__ partial;
  int nb;
  PcgScalars* __restrict__ sc;
  double rr, rz, threshold, rzPrev;
  __device__ void fetch(const double* __restrict__ part, int n, PcgScalars* __restrict__ scalars) {
    partial   = part;
    nb        = n;
    sc        = scalars;
    const bool in = (int)threadIdx.x < nb;
    rr        = in ? partial[threadIdx.x] : 0.0;
    rz        = in ? partial[nb + threadIdx.x] : 0.0;
    threshold = sc->threshold;
    rzPrev    = sc->rz;
  }
  __device__ void wait() {
    arrived(rr);
    arrived(rz);
  }
  __device__ bool test(int maxIter, bool record, double& beta) {
    __shared__ double bc[2];
    for (int i = threadIdx.x + BS; i < nb; i += BS) {
      rr += partial[i];
      rz += partial[nb + i];
    }
    rr = blockSum<BS>(rr);
    rz = blockSum<BS>(rz);
    if (threadIdx.x == 0) {
      bc[0] = rr;
      bc[1] = rz;
    }
    __syncthreads();
    rr              = bc[0];
    rz              = bc[1];
    const bool conv = rr < threshold;
    beta            = rz / rzPrev;
    if (record && threadIdx.x == 0) pcgRecord(sc, rr, rz, beta, conv, maxIter);
    return !conv;
  }
};

// The first half of a PCG iteration in one launch, for small systems whose kernels are bound by launch and latency:
// with `test` the convergence test and beta of the previous iteration (else beta as recorded), then q = K p with
// p = z + beta p_old formed at every read (the neighbours' too: twice the gathered bytes, which stay in the caches
// at these sizes), p stored beside p_old's buffer, and p.q partials. Lanes as spmvRows (G wavefronts share the rows);
// the loads of a lane's first DEPTH blocks, of z and p_old included, are in flight while the block folds the partials.
template <typename TV, int G>
__global__ __launch_bounds__(SPMV_BS) void pcgDirectionSpmv(
    const int32_t* __restrict__ rowptr, const int32_t* __restrict__ sellStart, const int32_t* __restrict__ scol,
    const TV* __restrict__ val, const TV* __restrict__ z, const TV* __restrict__ pOld, TV* __restrict__ p,
    TV* __restrict__ q, int64_t nrows, const double* __restrict__ partial, int nb, double* __restrict__ pq,
    PcgScalars* __restrict__ sc, int maxIter, int test) {
  int done = sc->done;
  PcgTest<SPMV_BS> t;
  if (test) t.fetch(partial, nb, sc);
  double bt        = sc->beta;
  constexpr int NO = sizeof(TV) == 4 ? 3 : 1;  // outputs per lane
  constexpr int DEPTH = 4;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, g = wave % G;
  const int rl      = sizeof(TV) == 4 ? lane : lane / 3;
  const int k       = sizeof(TV) == 4 ? 0 : lane - 3 * rl;
  const int64_t row = (int64_t)blockIdx.x * spmvRowsPerBlock<TV, G>() + wave / G * spmvRowsPerWave<TV>() + rl;
  const bool in     = rl < spmvRowsPerWave<TV>() && row < nrows;
  const int64_t base = in ? (int64_t)sellStart[row >> 6] + (row & 63) : 0;
  const int w        = in ? rowptr[row + 1] - rowptr[row] : 0;
  const int32_t* C   = scol + base;
  const TV* v0       = val + base * 9 + 3 * k;
  TV v[DEPTH][3 * NO], zc[DEPTH][3], pc[DEPTH][3], zr[NO], pr[NO];
  auto load = [&](int j, TV (&vj)[3 * NO], TV (&zj)[3], TV (&pj)[3]) {
    const int64_t c = (int64_t)C[j * kSellRows] * 3;
#pragma unroll
    for (int l = 0; l < 3 * NO; ++l) vj[l] = v0[(int64_t)j * (kSellRows * 9) + l];
#pragma unroll
    for (int l = 0; l < 3; ++l) {
      zj[l] = z[c + l];
      pj[l] = pOld[c + l];
    }
  };
#pragma unroll
  for (int u = 0; u < DEPTH; ++u)
    if (g + u * G < w) load(g + u * G, v[u], zc[u], pc[u]);
  if (in)
#pragma unroll
    for (int o = 0; o < NO; ++o) {
      zr[o] = z[row * 3 + k + o];
      pr[o] = pOld[row * 3 + k + o];
    }
#pragma unroll
  for (int u = 0; u < DEPTH; ++u) {
    arrived(v[u]);
    arrived(zc[u]);
    arrived(pc[u]);
  }
  arrived(zr);
  arrived(pr);
  if (test) t.wait();
  if (done) return;
  if (test && !t.test(maxIter, blockIdx.x == 0, bt)) return;
  const TV beta = (TV)bt;
  TV a[NO][3];  // one sum per output and column
#pragma unroll
  for (int o = 0; o < NO; ++o) a[o][0] = a[o][1] = a[o][2] = TV(0);
  auto add = [&](const TV (&vj)[3 * NO], const TV (&zj)[3], const TV (&pj)[3]) {
#pragma unroll
    for (int l = 0; l < 3; ++l) {
      const TV x = zj[l] + beta * pj[l];
#pragma unroll
      for (int o = 0; o < NO; ++o) a[o][l] += vj[3 * o + l] * x;
    }
  };
#pragma unroll
  for (int u = 0; u < DEPTH; ++u)
    if (g + u * G < w) add(v[u], zc[u], pc[u]);
  for (int j = g + DEPTH * G; j < w; j += G) {
    load(j, v[0], zc[0], pc[0]);
    add(v[0], zc[0], pc[0]);
  }
  TV y[NO];
#pragma unroll
  for (int o = 0; o < NO; ++o) y[o] = a[o][0] + (a[o][1] + a[o][2]);
  if constexpr (G > 1) {
    __shared__ TV part[SPMV_BS / 64][NO][64];
#pragma unroll
    for (int o = 0; o < NO; ++o) part[wave][o][lane] = y[o];
    __syncthreads();
    if (g == 0)
#pragma unroll
      for (int wv = 1; wv < G; ++wv)
#pragma unroll
        for (int o = 0; o < NO; ++o) y[o] += part[wave + wv][o][lane];
  }
  double d = 0.0;
  if (in && g == 0)
#pragma unroll
    for (int o = 0; o < NO; ++o) {
      const int64_t i = row * 3 + k + o;
      const TV pi     = zr[o] + beta * pr[o];
      p[i]            = pi;
      q[i]            = y[o];
      d += (double)pi * (double)y[o];
    }
  const double s = blockSum<SPMV_BS>(d);
  if (threadIdx.x == 0) pq[blockIdx.x] = s;
}

// the convergence test of the last iteration of a chunk of them, before the host looks at the flag
__global__ __launch_bounds__(256) void pcgTestKernel(const double* __restrict__ partial, int nb,
                                                     PcgScalars* __restrict__ sc, int maxIter) {
  if (sc->done) return;
  PcgTest<256> t;
  t.fetch(partial, nb, sc);
  double beta;
  (void)t.test(maxIter, true, beta);
}

// r = b - K x with FP64 accumulation (K may be FP32); used by iterative refinement. Same lane layouts.
template <typename TV, int G>
__global__ __launch_bounds__(SPMV_BS) void residualKernel(const int32_t* __restrict__ rowptr,
                                                                   const int32_t* __restrict__ sellStart,
                                                                   const int32_t* __restrict__ scol,
                                                                   const TV* __restrict__ val,
                                                                   const double* __restrict__ x,
                                                                   const double* __restrict__ b,
                                                                   double* __restrict__ r, int64_t nrows,
                                                                   double* __restrict__ partial) {
  double d = 0.0;
  spmvRows<G, double>(rowptr, sellStart, scol, val, x, nrows, blockIdx.x, [&](int64_t i, double kx) {
    const double ri = b[i] - kx;
    r[i]            = ri;
    d += ri * ri;
  });
  const double s = blockSum<SPMV_BS>(d);
  if (threadIdx.x == 0) partial[blockIdx.x] = s;
}

// partial dot products (grid-stride, fixed grid) — deterministic given the launch shape
__global__ __launch_bounds__(256) void dotKernel(const double* __restrict__ a, const double* __restrict__ b,
                                                 int64_t n, double* __restrict__ partial) {
  double s = 0.0;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) s += a[i] * b[i];
  s = blockSum<256>(s);
  if (threadIdx.x == 0) partial[blockIdx.x] = s;
}

__global__ __launch_bounds__(1024) void foldKernel(const double* __restrict__ partial, int n,
                                                   double* __restrict__ out) {
  double s = 0.0;
  for (int i = threadIdx.x; i < n; i += 1024) s += partial[i];
  s = blockSum<1024>(s);
  if (threadIdx.x == 0) *out = s;
}

__global__ void axpyKernel(double a, const double* __restrict__ x, double* __restrict__ y, int64_t n) {
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) y[i] += a * x[i];
}

// ---------------- PCG (Jacobi, FP64) ----------------
__global__ void jacobiDiagKernel(const int32_t* __restrict__ diag, const double* __restrict__ K, int64_t nrows,
                                 double* __restrict__ dinv) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= nrows * 3) return;
  const int64_t node = i / 3;
  const int k        = (int)(i - node * 3);
  const double d     = K[(int64_t)diag[node] * 9 + k * 4];
  dinv[i]            = d != 0.0 ? 1.0 / d : 1.0;
}

// r = b, x = 0, p = Dinv r (with z: z = Dinv r and p = 0); partials of rr and rz
__global__ __launch_bounds__(256) void pcgInitKernel(const double* __restrict__ b, const double* __restrict__ dinv,
                                                     double* __restrict__ x, double* __restrict__ r,
                                                     double* __restrict__ p, double* __restrict__ zOut, int64_t n,
                                                     double* __restrict__ partial /* 2*grid */) {
  double rr = 0.0, rz = 0.0;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) {
    const double bi = b[i];
    x[i]            = 0.0;
    r[i]            = bi;
    const double z  = dinv[i] * bi;
    p[i]            = zOut ? 0.0 : z;
    if (zOut) zOut[i] = z;
    rr += bi * bi;
    rz += bi * z;
  }
  rr = blockSum<256>(rr);
  rz = blockSum<256>(rz);
  if (threadIdx.x == 0) {
    partial[blockIdx.x]             = rr;
    partial[gridDim.x + blockIdx.x] = rz;
  }
}

__global__ __launch_bounds__(1024) void pcgInitFold(const double* __restrict__ partial, int nb, double tol2,
                                                    PcgScalars* __restrict__ sc, PcgMirror* mirror, uint32_t run,
                                                    const unsigned long long* __restrict__ err) {
  double rr = 0.0, rz = 0.0;
  for (int i = threadIdx.x; i < nb; i += 1024) {
    rr += partial[i];
    rz += partial[nb + i];
  }
  rr = blockSum<1024>(rr);
  rz = blockSum<1024>(rz);
  if (threadIdx.x == 0) {
    sc->bb        = rr;
    sc->rr        = rr;
    sc->rz        = rz;
    sc->rz_new    = rz;
    const double thr = tol2 * rr;
    sc->threshold = thr > 2.2250738585072014e-308 ? thr : 2.2250738585072014e-308;
    sc->iters     = 0;
    sc->halt      = 0;
    sc->done      = (rr == 0.0 || rr < sc->threshold) ? 1 : 0;
    sc->alpha = sc->beta = 0.0;
    sc->mirror           = mirror;
    sc->run              = run;
    mirror->err[0]       = err[0];
    mirror->err[1]       = err[1];
    __threadfence_system();
    pcgPublish(sc, rr, 0, sc->done);
  }
}

// First stage of the p.q fold: block b sums its slice of the SpMV's per-block partials, in order, into
// pq2[b] (kPqBlocks values). A single block summing one partial per SpMV block took 17 us per iteration at
// 1 M elements (38,631 partials); the update kernel folds the kPqBlocks values itself. Launches of at most
// kPqDirect SpMV blocks skip this stage: every update block then folds the SpMV's partials directly.
constexpr int kPqBlocks = 64;
constexpr int kPqDirect = 2048;
__global__ __launch_bounds__(256) void pcgPqFold(const double* __restrict__ partial, int nb,
                                                 double* __restrict__ pq2, const PcgScalars* __restrict__ sc) {
  if (sc->done) return;
  const int chunk = (nb + kPqBlocks - 1) / kPqBlocks;
  const int lo = blockIdx.x * chunk, hi = lo + chunk < nb ? lo + chunk : nb;
  double s = 0.0;
  for (int i = lo + threadIdx.x; i < hi; i += 256) s += partial[i];
  s = blockSum<256>(s);
  if (threadIdx.x == 0) pq2[blockIdx.x] = s;
}

// alpha = r.z / p.q (every block folds the npq values pq[] -- pcgPqFold's kPqBlocks sums or the SpMV's
// partials -- in the same order, so all blocks agree bitwise; block 0 records the scalars), then
// x += alpha p, r -= alpha q with partials of r.r and r.z (z = M^-1 r, stored when zOut is given)
template <typename T, bool BLOCK>
__global__ __launch_bounds__(256) void pcgUpdateKernel(T* __restrict__ x, T* __restrict__ r,
                                                       const T* __restrict__ p, const T* __restrict__ q,
                                                       const T* __restrict__ pre, T* __restrict__ zOut,
                                                       int64_t n, PcgScalars* __restrict__ sc,
                                                       const double* __restrict__ pq, int npq,
                                                       double* __restrict__ partial /* 2*grid */) {
  const int done = sc->done;
  // N entries per unit: one, or a node's three with the 3x3 block of the preconditioner
  constexpr int N = BLOCK ? 3 : 1;
  struct Unit {
    T x[N], r[N], p[N], q[N], m[N * N];
  };
  auto load = [&](int64_t u, Unit& v) {
#pragma unroll
    for (int k = 0; k < N; ++k) {
      v.x[k] = x[u * N + k];
      v.r[k] = r[u * N + k];
      v.p[k] = p[u * N + k];
      v.q[k] = q[u * N + k];
    }
#pragma unroll
    for (int k = 0; k < N * N; ++k) v.m[k] = pre[u * N * N + k];
  };
  const int64_t nu = n / N;
  int64_t u        = (int64_t)blockIdx.x * 256 + threadIdx.x;
  Unit v;
  if (u < nu) load(u, v);
  const double rzNew = sc->rz_new;  // r.z of the current iterate (set by the previous p update)
  double pqSum       = (int)threadIdx.x < npq ? pq[threadIdx.x] : 0.0;
  arrived(v.x);
  arrived(v.r);
  arrived(v.p);
  arrived(v.q);
  arrived(v.m);
  arrived(pqSum);
  if (done) return;
  __shared__ double alphaS;
  {
    for (int i = threadIdx.x + 256; i < npq; i += 256) pqSum += pq[i];
    pqSum = blockSum<256>(pqSum);
    if (threadIdx.x == 0) {
      alphaS = rzNew / pqSum;
      if (blockIdx.x == 0) {
        sc->rz    = rzNew;
        sc->pq    = pqSum;
        sc->alpha = alphaS;
      }
    }
    __syncthreads();
  }
  const T alpha = (T)alphaS;
  double rr = 0.0, rz = 0.0;
  while (u < nu) {
    T z[N];
#pragma unroll
    for (int k = 0; k < N; ++k) {
      x[u * N + k] = v.x[k] + alpha * v.p[k];
      v.r[k] -= alpha * v.q[k];
      r[u * N + k] = v.r[k];
      rr += (double)v.r[k] * (double)v.r[k];
    }
#pragma unroll
    for (int k = 0; k < N; ++k) {
      if constexpr (BLOCK)
        z[k] = v.m[3 * k] * v.r[0] + v.m[3 * k + 1] * v.r[1] + v.m[3 * k + 2] * v.r[2];
      else
        z[k] = v.m[0] * v.r[0];
      if (zOut) zOut[u * N + k] = z[k];
      rz += (double)v.r[k] * (double)z[k];
    }
    u += (int64_t)gridDim.x * 256;
    if (u < nu) load(u, v);
  }
  rr = blockSum<256>(rr);
  rz = blockSum<256>(rz);
  if (threadIdx.x == 0) {
    partial[blockIdx.x]             = rr;
    partial[gridDim.x + blockIdx.x] = rz;
  }
}

// Convergence test, beta and p = M^-1 r + beta p in one launch
template <typename T, bool BLOCK>
__global__ __launch_bounds__(256) void pcgBetaPKernel(T* __restrict__ p, const T* __restrict__ r,
                                                      const T* __restrict__ pre, int64_t n,
                                                      const double* __restrict__ partial, int nb,
                                                      PcgScalars* __restrict__ sc, int maxIter) {
  const int done = sc->done;
  PcgTest<256> t;
  t.fetch(partial, nb, sc);
  constexpr int N = BLOCK ? 3 : 1;
  struct Unit {
    T r[N], p[N], m[N * N];
  };
  auto load = [&](int64_t u, Unit& v) {
#pragma unroll
    for (int k = 0; k < N; ++k) {
      v.r[k] = r[u * N + k];
      v.p[k] = p[u * N + k];
    }
#pragma unroll
    for (int k = 0; k < N * N; ++k) v.m[k] = pre[u * N * N + k];
  };
  const int64_t nu = n / N;
  int64_t u        = (int64_t)blockIdx.x * 256 + threadIdx.x;
  Unit v;
  if (u < nu) load(u, v);
  arrived(v.r);
  arrived(v.p);
  arrived(v.m);
  t.wait();
  if (done) return;
  double bt;
  if (!t.test(maxIter, blockIdx.x == 0, bt)) return;
  const T beta = (T)bt;
  while (u < nu) {
#pragma unroll
    for (int k = 0; k < N; ++k) {
      if constexpr (BLOCK)
        p[u * N + k] = v.m[3 * k] * v.r[0] + v.m[3 * k + 1] * v.r[1] + v.m[3 * k + 2] * v.r[2] + beta * v.p[k];
      else
        p[u * N + k] = v.m[0] * v.r[0] + beta * v.p[0];
    }
    u += (int64_t)gridDim.x * 256;
    if (u < nu) load(u, v);
  }
}

// ---------------- FP32 block-Jacobi helpers ----------------
__global__ void blockInvKernel(const int32_t* __restrict__ diag, const float* __restrict__ K, int64_t nrows,
                               float* __restrict__ binv) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= nrows) return;
  const float* A = K + (int64_t)diag[i] * 9;
  // invert in double for robustness, store FP32
  const double a00 = A[0], a01 = A[1], a02 = A[2], a10 = A[3], a11 = A[4], a12 = A[5], a20 = A[6], a21 = A[7],
               a22 = A[8];
  const double det = a00 * (a11 * a22 - a12 * a21) - a01 * (a10 * a22 - a12 * a20) + a02 * (a10 * a21 - a11 * a20);
  float* B = binv + i * 9;
  if (det == 0.0) {
    for (int k = 0; k < 9; ++k) B[k] = (k % 4 == 0) ? 1.0f : 0.0f;
    return;
  }
  const double id = 1.0 / det;
  B[0] = (float)((a11 * a22 - a12 * a21) * id);
  B[1] = (float)((a02 * a21 - a01 * a22) * id);
  B[2] = (float)((a01 * a12 - a02 * a11) * id);
  B[3] = (float)((a12 * a20 - a10 * a22) * id);
  B[4] = (float)((a00 * a22 - a02 * a20) * id);
  B[5] = (float)((a02 * a10 - a00 * a12) * id);
  B[6] = (float)((a10 * a21 - a11 * a20) * id);
  B[7] = (float)((a01 * a20 - a00 * a21) * id);
  B[8] = (float)((a00 * a11 - a01 * a10) * id);
}

// FP32 PCG init from an FP64 right-hand side scaled by 1/s (s = ||r||, keeps FP32 in range)
__global__ __launch_bounds__(256) void pcgInitF32(const double* __restrict__ b, double invScale,
                                                  const float* __restrict__ binv, float* __restrict__ x,
                                                  float* __restrict__ r, float* __restrict__ p,
                                                  float* __restrict__ zOut, int64_t nn,
                                                  double* __restrict__ partial) {
  double rr = 0.0, rz = 0.0;
  for (int64_t nd = (int64_t)blockIdx.x * 256 + threadIdx.x; nd < nn; nd += (int64_t)gridDim.x * 256) {
    float rl[3];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      rl[k]         = (float)(b[nd * 3 + k] * invScale);
      r[nd * 3 + k] = rl[k];
      x[nd * 3 + k] = 0.0f;
      rr += (double)rl[k] * (double)rl[k];
    }
    const float* B = binv + nd * 9;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      const float z = B[k * 3] * rl[0] + B[k * 3 + 1] * rl[1] + B[k * 3 + 2] * rl[2];
      p[nd * 3 + k] = zOut ? 0.0f : z;
      if (zOut) zOut[nd * 3 + k] = z;
      rz += (double)rl[k] * (double)z;
    }
  }
  rr = blockSum<256>(rr);
  rz = blockSum<256>(rz);
  if (threadIdx.x == 0) {
    partial[blockIdx.x]             = rr;
    partial[gridDim.x + blockIdx.x] = rz;
  }
}

// two-level form: r = b / s, x = 0 and r.r partials (z and p follow from the coarse correction); clears the done
// flag, which the coarse kernels read before the init fold sets it
__global__ __launch_bounds__(256) void pcgInitR32(const double* __restrict__ b, double invScale,
                                                  float* __restrict__ x, float* __restrict__ r, int64_t n,
                                                  double* __restrict__ partial, PcgScalars* __restrict__ sc) {
  if (blockIdx.x == 0 && threadIdx.x == 0) sc->done = 0;
  double rr = 0.0;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) {
    const float ri = (float)(b[i] * invScale);
    r[i]           = ri;
    x[i]           = 0.0f;
    rr += (double)ri * (double)ri;
  }
  rr = blockSum<256>(rr);
  if (threadIdx.x == 0) partial[blockIdx.x] = rr;
}

// x64 += scale * x32
__global__ void accumulateF32(double* __restrict__ x, const float* __restrict__ d, double scale, int64_t n) {
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256)
    x[i] += scale * (double)d[i];
}

inline int vecGrid(int64_t n) {
  int64_t g = (n + 255) / 256;
  if (g > kReduceBlocks) g = kReduceBlocks;
  return (int)(g < 1 ? 1 : g);
}

}  // namespace

static double* pq2(ik_handle* h) { return h->partial.p + h->partial.n - 8 - kPqBlocks; }
// the PCG SpMV's per-block p.q partials, apart from the vector kernels' partials at the start (the update
// kernel reads the former while its blocks write the latter)
static double* pqPartials(ik_handle* h) { return h->partial.p + 2 * kReduceBlocks; }

// Wavefronts that share a row group of the SpMV (G), and whether the PCG forms its direction inside the SpMV. us per
// PCG iteration, hex8 grids of 20^3 / 27^3 / 34^3 / 42^3 / 52^3 elements (9,261 to 148,877 nodes):
//  FP64 Jacobi        G = 1: 16.5 / 18.6 / 24.5 / 37.6 / 65.0   G = 4: 12.8 / 18.3 / 27.8 / 40.2 / 69.0
//                     G = 4, direction in the SpMV: 12.8 / 19.4 / 28.9 / 47.8 / 94.2 (8^3: 10.6 against 13.0 for G = 1)
//  FP32 block Jacobi  G = 1: 17.9 / 19.3 / 19.7 / 23.9 / 37.4   G = 4: 15.8 / 17.1 / 19.1 / 24.3 / 37.5
//                     G = 4, direction in the SpMV: 10.9 / 13.5 / 16.6 / 23.5 / 38.7
// Shuffled element order at 42^3: FP64 43.0 (G = 1) and 49.1; FP32 34.8 (G = 1), 29.2 and 36.5 with the direction.
// Small systems lack wavefronts and are bound by the chain of loads of one row and by launches (a host that launches
// slowly: 198 ms against 154 for ten plane load steps at 2,210 nodes with the same split), so the split and the launch
// saved count; large ones are bound by bytes and prefer long runs of one wavefront.
constexpr int64_t kSplitRows64 = 15000, kSplitRows32 = 120000;
constexpr int64_t kDirectionRows64 = kSplitRows64, kDirectionRows32 = 50000;
constexpr int kSplit = 4;
template <typename TV>
static bool directionInSpmv(int64_t nn) {
  return nn <= (sizeof(TV) == 4 ? kDirectionRows32 : kDirectionRows64);
}
// calls f(std::integral_constant<int, G>) for the split of TV's layout on nn rows
template <typename TV, typename F>
static void withSplit(int64_t nn, F f) {
  if (nn <= (sizeof(TV) == 4 ? kSplitRows32 : kSplitRows64))
    f(std::integral_constant<int, kSplit>{});
  else
    f(std::integral_constant<int, 1>{});
}
template <typename TV>
static unsigned spmvGrid(int64_t nn) {
  unsigned g = 0;
  withSplit<TV>(nn, [&](auto G) {
    constexpr int R = spmvRowsPerBlock<TV, decltype(G)::value>();
    g               = (unsigned)((nn + R - 1) / R);
  });
  return g;
}

// partial[] holds one launch's per-block partials at its start, the PCG SpMV's partials from 2 kReduceBlocks
// on, the p.q first-stage sums (kPqBlocks) in a region of their own before the last 8 entries, and fold
// results in its last entry
static void ensureWork(ik_handle* h) {
  const int64_t spmvBlocks = std::max(spmvGrid<double>(h->nn), spmvGrid<float>(h->nn));
  h->partial.ensure((size_t)(2 * kReduceBlocks + spmvBlocks) + kPqBlocks + 8);
  h->sc.ensure(1);
  if (!h->pcg) {
    IK_HIP(hipHostMalloc((void**)&h->pcg, sizeof(PcgMirror), hipHostMallocCoherent));
    h->pcg->state = 0;
  }
  if (!h->hred) IK_HIP(hipHostMalloc((void**)&h->hred, sizeof(double) * 4, hipHostMallocDefault));
}

// y = K x (partial: with x.y partials per block, and skipped once sc->done)
template <typename TV, typename TX>
static void launchSpmv(ik_handle* h, const TV* K, const TX* x, TX* y, double* partial, const PcgScalars* sc, int rev) {
  ScopedKernelTimer t(h, KSPMV);
  const unsigned grid = spmvGrid<TV>(h->nn);
  withSplit<TV>(h->nn, [&](auto G) {
    constexpr int g = decltype(G)::value;
    if (partial)
      hipLaunchKernelGGL((spmvKernel<TV, TX, true, g>), dim3(grid), dim3(SPMV_BS), 0, h->stream, h->rowptr.p,
                         h->sellStart.p, h->scol.p, K, x, y, h->nn, partial, sc, rev);
    else
      hipLaunchKernelGGL((spmvKernel<TV, TX, false, g>), dim3(grid), dim3(SPMV_BS), 0, h->stream, h->rowptr.p,
                         h->sellStart.p, h->scol.p, K, x, y, h->nn, nullptr, nullptr, 0);
  });
}

void spmv64(ik_handle* h, const double* x, double* y) {
  ensureWork(h);
  launchSpmv<double, double>(h, h->K64.p, x, y, nullptr, nullptr, 0);
}

double dot(ik_handle* h, const double* a, const double* b, int64_t n) {
  ensureWork(h);
  const int g = vecGrid(n);
  hipLaunchKernelGGL(dotKernel, dim3(g), dim3(256), 0, h->stream, a, b, n, h->partial.p);
  return foldPartials(h, g);
}

double* partialsFor(ik_handle* h, int nb) {
  ensureWork(h);
  require(nb >= 1 && nb <= kReduceBlocks, IK_EINVAL, "internal error: too many reduction partials");
  return h->partial.p;
}

double foldPartials(ik_handle* h, int nb) {
  hipLaunchKernelGGL(foldKernel, dim3(1), dim3(1024), 0, h->stream, h->partial.p, nb, h->partial.p + h->partial.n - 1);
  IK_HIP(hipMemcpyAsync(h->hred, h->partial.p + h->partial.n - 1, sizeof(double), hipMemcpyDeviceToHost, h->stream));
  IK_HIP(hipStreamSynchronize(h->stream));
  finishErrCheck(h);
  return h->hred[0];
}

void axpy(ik_handle* h, double a, const double* x, double* y, int64_t n) {
  hipLaunchKernelGGL(axpyKernel, dim3(vecGrid(n)), dim3(256), 0, h->stream, a, x, y, n);
}

// Iterations are enqueued at most kPcgAhead beyond the count that the device last wrote into the handle's pinned
// mirror: enough that it never waits for the host (the four left when a count arrives take it 40 us or more), and few
// launches after convergence (they return at once, one and a half to two us each). Against 32, then 64 iterations
// between reads of the flag with the stream drained: two-level solve at 64^3 13.45 -> 12.44 ms, FP32 block Jacobi at
// 20^3 8.4 -> 7.2 ms, ten load steps of the 64 x 16 plane 147-154 -> 132-138 ms. 4 / 8 / 12 / 16 / 24 iterations
// between the counts, four more ahead: the two-level solve 12.6 / 12.44 / 12.41 / 12.44 / 12.67 ms, the others within
// their noise.
constexpr int kPcgAhead = 12;
static_assert(kPcgAhead > kPcgPublish + 1, "the device publishes within what may be enqueued");

// State of the current PCG run (iterations << 2 | done); `before` until the run has started. An assembly whose error
// flag is still to be read (errPending) is settled by the flag the run reports: if it is raised, here.
static unsigned pcgState(ik_handle* h, unsigned before) {
  unsigned state = before;
  bool flagged   = false;
  if (!pcgLook(*h->pcg, h->pcgRun, state, flagged)) return before;
  if (flagged) finishErrCheck(h, true);
  h->errPending = false;
  return state;
}

// waits for a state after `before`
static unsigned pcgWait(ik_handle* h, unsigned before) {
  bool idle      = false;
  unsigned state = before;
  pcgSpin(
      [&] {
        state = pcgState(h, before);
        if (state == before && idle) throw Error{IK_EHIP, "internal error: the PCG run ended without a result"};
        return state != before;
      },
      [&] {  // a launch or device that failed: an error here, not a wait without end
        const hipError_t query = hipStreamQuery(h->stream);
        idle                   = query == hipSuccess;
        if (query == hipErrorNotReady)
          (void)hipGetLastError();
        else
          IK_HIP(query);
      });
  return state;
}

// The iterations of one PCG solve, after its init kernels: enqueued until the done flag or maxIter. p holds
// the first direction, or zero with z = M^-1 r when z is given (the direction is then formed inside the SpMV,
// alternating between p and p2). coarse: the two-level form's vector kernels instead of update and direction.
template <typename T>
static void pcgLoop(ik_handle* h, const T* K, T* x, T* r, T* p, T* p2, T* z, T* q, const T* pre, int64_t n,
                    int grid, int maxIter, bool coarse) {
  const unsigned sgrid = spmvGrid<T>(h->nn);
  unsigned state = 0;
  for (int enq = 0;; ++enq) {
    if (z && enq == maxIter)  // the last iteration's test, which no direction follows
      hipLaunchKernelGGL(pcgTestKernel, dim3(1), dim3(256), 0, h->stream, h->partial.p, grid, h->sc.p, maxIter);
    state = pcgState(h, state);
    while (!(state & 3) && (enq == maxIter || enq - (int)(state >> 2) >= kPcgAhead)) state = pcgWait(h, state);
    if (state & 3) break;
    if (z) {
      if (enq > 0) std::swap(p, p2);
      ScopedKernelTimer t(h, KSPMV);
      hipLaunchKernelGGL((pcgDirectionSpmv<T, kSplit>), dim3(sgrid), dim3(SPMV_BS), 0, h->stream, h->rowptr.p,
                         h->sellStart.p, h->scol.p, K, z, p, p2, q, h->nn, h->partial.p, grid, pqPartials(h),
                         h->sc.p, maxIter, enq > 0 ? 1 : 0);
    } else {
      launchSpmv<T, T>(h, K, p, q, pqPartials(h), h->sc.p, enq & 1);
    }
    const double* pqSrc = pqPartials(h);
    int npq             = (int)sgrid;
    if (sgrid > (unsigned)kPqDirect) {
      hipLaunchKernelGGL(pcgPqFold, dim3(kPqBlocks), dim3(256), 0, h->stream, pqPartials(h), (int)sgrid, pq2(h),
                         h->sc.p);
      pqSrc = pq2(h);
      npq   = kPqBlocks;
    }
    if constexpr (std::is_same<T, float>::value)
      if (coarse) {
        coarseIteration(h, pqSrc, npq, x, r, p, q, pre, grid, h->partial.p, maxIter);
        continue;
      }
    constexpr bool B = std::is_same<T, float>::value;  // FP64: diagonal preconditioner, FP32: 3x3 blocks
    hipLaunchKernelGGL((pcgUpdateKernel<T, B>), dim3(grid), dim3(256), 0, h->stream, x, r, z ? p2 : p, q, pre, z, n,
                       h->sc.p, pqSrc, npq, h->partial.p);
    if (!z)
      hipLaunchKernelGGL((pcgBetaPKernel<T, B>), dim3(grid), dim3(256), 0, h->stream, p, r, pre, n, h->partial.p,
                         grid, h->sc.p, maxIter);
  }
}

void pcgJacobi64(ik_handle* h, const double* b, double* x, double rtol, int maxIter, int* iters, double* relres) {
  ensureWork(h);
  const int64_t n  = h->ndof;
  const bool fused = directionInSpmv<double>(h->nn);
  h->pr.ensure(n);
  h->pp.ensure(n);
  h->pq.ensure(n);
  h->pdiag.ensure(n);
  if (fused) {
    h->pz.ensure(n);
    h->pb.ensure(n);
  }
  double* z   = fused ? h->pz.p : nullptr;
  const int g = vecGrid(n);
  hipLaunchKernelGGL(jacobiDiagKernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, h->stream, h->diagBlk.p,
                     h->K64.p, h->nn, h->pdiag.p);
  hipLaunchKernelGGL(pcgInitKernel, dim3(g), dim3(256), 0, h->stream, b, h->pdiag.p, x, h->pr.p, h->pp.p, z, n,
                     h->partial.p);
  hipLaunchKernelGGL(pcgInitFold, dim3(1), dim3(1024), 0, h->stream, h->partial.p, g, rtol * rtol, h->sc.p,
                     h->pcg, ++h->pcgRun, h->errFlag.p);
  if (maxIter <= 0) maxIter = (int)(2 * n);
  pcgLoop<double>(h, h->K64.p, x, h->pr.p, h->pp.p, h->pb.p, z, h->pq.p, h->pdiag.p, n, g, maxIter, false);
  *iters  = (int)((unsigned)h->pcg->state >> 2);
  *relres = h->pcg->bb > 0 ? std::sqrt(h->pcg->rr / h->pcg->bb) : 0.0;
}

void pcgMixed(ik_handle* h, const double* b, double* x, const ik_solver_opts* o, ik_solver_info* info,
              double bnormKnown) {
  ensureWork(h);
  const bool twoLevel = o->kind == IK_PCG_TWOLEVEL_FP32_IR;
  const bool fused    = !twoLevel && directionInSpmv<float>(h->nn);
  const int64_t n = h->ndof;
  h->fr.ensure(n);
  h->fp.ensure(n);
  h->fq.ensure(n);
  h->fx.ensure(n);
  h->fdiag.ensure((size_t)h->nn * 9);
  h->pr.ensure(n);
  if (fused) {
    h->fz.ensure(n);
    h->fp2.ensure(n);
  }
  float* z    = fused ? h->fz.p : nullptr;
  const int g = vecGrid(n);
  // vector kernels over nodes: 512 blocks (the p update folds 2 partials per block in every block; 512 vs
  // 1024 blocks measured 2.28 vs 2.31 s on the 64^3 mixed Newton path)
  const int gn = std::min(vecGrid(h->nn), 512);
  const unsigned sgrid = spmvGrid<float>(h->nn);
  hipLaunchKernelGGL(blockInvKernel, dim3((unsigned)((h->nn + 255) / 256)), dim3(256), 0, h->stream, h->diagBlk.p,
                     h->K32.p, h->nn, h->fdiag.p);
  if (twoLevel) coarsePrepare(h);
  // x = 0, r = b
  launchZero(x, n, h->stream);
  IK_HIP(hipMemcpyAsync(h->pr.p, b, n * sizeof(double), hipMemcpyDeviceToDevice, h->stream));
  const double bnorm = bnormKnown >= 0.0 ? bnormKnown : std::sqrt(dot(h, b, b, n));
  info->iterations  = 0;
  info->refinements = 0;
  info->converged   = 0;
  if (bnorm == 0.0) {
    info->rel_residual = 0.0;
    info->converged    = 1;
    return;
  }
  const int maxIter = o->max_iter > 0 ? o->max_iter : (int)(2 * n);
  double rnorm      = bnorm;
  const int maxRef  = o->max_refine > 0 ? o->max_refine : 10;
  for (int sweep = 0; sweep < maxRef; ++sweep) {
    // inner FP32 PCG on K32 d = r / ||r||, to half the reduction the outer tolerance still needs (an inexact
    // Newton step asks for little), but never below inner_rtol
    const double innerTol = std::max(o->inner_rtol, 0.5 * o->rtol * bnorm / rnorm);
    if (twoLevel) {
      hipLaunchKernelGGL(pcgInitR32, dim3(gn), dim3(256), 0, h->stream, h->pr.p, 1.0 / rnorm, h->fx.p, h->fr.p, n,
                         h->partial.p, h->sc.p);
      coarseApply(h, h->fr.p, h->fp.p, nullptr, h->fdiag.p, gn, h->partial.p);  // p = z
    } else {
      hipLaunchKernelGGL(pcgInitF32, dim3(gn), dim3(256), 0, h->stream, h->pr.p, 1.0 / rnorm, h->fdiag.p, h->fx.p,
                         h->fr.p, h->fp.p, z, h->nn, h->partial.p);
    }
    hipLaunchKernelGGL(pcgInitFold, dim3(1), dim3(1024), 0, h->stream, h->partial.p, gn, innerTol * innerTol,
                       h->sc.p, h->pcg, ++h->pcgRun, h->errFlag.p);
    pcgLoop<float>(h, h->K32.p, h->fx.p, h->fr.p, h->fp.p, h->fp2.p, z, h->fq.p, h->fdiag.p, n, gn, maxIter, twoLevel);
    info->iterations += (int)((unsigned)h->pcg->state >> 2) + 1;
    info->refinements += 1;
    // x += ||r|| d ; r = b - K x in FP64
    hipLaunchKernelGGL(accumulateF32, dim3(g), dim3(256), 0, h->stream, x, h->fx.p, rnorm, n);
    withSplit<float>(h->nn, [&](auto G) {
      constexpr int gs = decltype(G)::value;
      hipLaunchKernelGGL((residualKernel<float, gs>), dim3(sgrid), dim3(SPMV_BS), 0, h->stream, h->rowptr.p,
                         h->sellStart.p, h->scol.p, h->K32.p, x, b, h->pr.p, h->nn, h->partial.p);
    });
    rnorm              = std::sqrt(foldPartials(h, (int)sgrid));
    info->rel_residual = rnorm / bnorm;
    if (info->rel_residual <= o->rtol) {
      info->converged = 1;
      break;
    }
  }
  if (twoLevel) coarseRecord(h, info->iterations, info->rel_residual);
}

}  // namespace ik

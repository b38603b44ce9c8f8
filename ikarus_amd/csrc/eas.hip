// eas.hip — EAS (enhanced Green-Lagrange strain, 21 modes) hex8 element: residual, condensed tangent and
// the internal-variable update.
//
// Restates EnhancedAssumedStrains (ikarus/finiteelements/mechanics/enhancedassumedstrains.hh:225-434)
// with the E21 ansatz (strainenhancements/easvariants/linearandglstrains.hh:22-39,280-328),
// T0 = T(xi_0) * detJ(xi_0) (easvariants/helperfunctions.hh:19-25; T from ikarus/utils/tensorutils.hh:440-465)
// and the GreenLagrangeStrain enhancement (easfunctions/greenlagrangestrain.hh:41-141):
//   E_enh = E(u) + M alpha,  M(xi) = T0^{-1} Mtilde(xi) / detJ(xi)
//   K_uu = sum (B^T C B + kg) dV,  R_u = sum B^T S dV,  D = sum M^T C M dV,  L = sum M^T C B dV,
//   Rt = sum M^T S dV,  K = K_uu - L^T D^{-1} L (upper, mirrored),  R = R_u - L^T D^{-1} Rt,
//   alpha <- alpha - D^{-1}(Rt + L du_e) on CORRECTION_UPDATED, with D, L, Rt of the state the tangent
//   was assembled at (the reference recomputes them at that same state).
//
// One contraction gives everything but the geometric stiffness: with the 6 x 48 matrix N = [M | B | 0] per Gauss point
// (21 mode columns, 24 displacement columns) and CN = [C dV M | C dV B | S dV | 0], sum over the points of N^T CN holds
// D, L, Rt, the material part of K_uu and R_u as one symmetric 48 x 48 array of 16 x 16 matrix-core tiles; block
// elimination of the 21 mode rows in those tiles leaves K and R. Outputs go to the same element-by-element staging as
// the plain element (36 upper blocks + 24 residual entries), plus the cache of the alpha update.
#include "ik_internal.hh"
#include "wave_reduce.hh"

namespace ik {
namespace {

constexpr int NE = 21;  // enhanced modes
typedef double v2d __attribute__((ext_vector_type(2)));
typedef double v4d __attribute__((ext_vector_type(4)));

// The alpha-update cache of an element: the rows What = Db^-1 Lb^-1 [.| L | Rt] of the block elimination
// D = Lb Db Lb^T (panels p of mode rows 4 p .. 4 p + 3, the last of row 20 alone), as the chunks in which the
// element kernel holds them (row k of a panel, column c of [D | L | Rt]): columns 16..31 of panel p at
// 64 p + 16 k + (c - 16), columns 32..45 at 320 + 56 p + 14 k + (c - 32), columns 4 (p + 1)..15 of panels 0-2 behind
// 600, columns 21..45 of row 20 at 696. The stride is a multiple of 64 bytes.
constexpr int kEasCache = 728;
__host__ __device__ constexpr int cacheLow(int p) { return p == 0 ? 600 : (p == 1 ? 648 : 680); }

__host__ __device__ constexpr int vI(int v) { return v < 3 ? v : (v == 3 ? 1 : 0); }
__host__ __device__ constexpr int vJ(int v) { return v < 3 ? v : (v == 5 ? 1 : 2); }
__host__ __device__ constexpr int sym6(int p, int q) {
  return p <= q ? p * 6 - (p * (p - 1)) / 2 + (q - p) : q * 6 - (q * (q - 1)) / 2 + (p - q);
}
__host__ __device__ constexpr int upperBlock(int a, int b) { return 8 * a - (a * (a - 1)) / 2 + (b - a); }

// E21 ansatz in reference coordinates (linearandglstrains.hh:300-322): column c has one nonzero, in Voigt row
// kRowOf(c), of value f_c(x, y, z) with x = 2 xi - 1 etc., a product of the coordinates in the mask (bit 0: x, 1: y,
// 2: z).
__host__ __device__ constexpr int kRowOf(int c) {
  return c < 3 ? c : (c < 9 ? 3 + (c - 3) / 2 : (c < 15 ? 3 + (c - 9) / 2 : (c - 15) / 2));
}
__host__ __device__ constexpr int monomialOf(int c) {
  constexpr int m[NE] = {1, 2, 4, 2, 4, 1, 4, 1, 2, 3, 5, 3, 6, 5, 6, 3, 5, 3, 6, 5, 6};
  return m[c];
}
// both as 3-bit fields, for a lane's own column
constexpr unsigned long long packModes(bool rows) {
  unsigned long long v = 0;
  for (int c = 0; c < NE; ++c) v |= (unsigned long long)(rows ? kRowOf(c) : monomialOf(c)) << (3 * c);
  return v;
}

__device__ inline double det3(const double A[3][3]) {
  return A[0][0] * (A[1][1] * A[2][2] - A[1][2] * A[2][1]) - A[0][1] * (A[1][0] * A[2][2] - A[1][2] * A[2][0]) +
         A[0][2] * (A[1][0] * A[2][1] - A[1][1] * A[2][0]);
}

// value of lane `lane` (uniform) of a 64-bit register, as two 32-bit lane reads into scalar registers
__device__ inline double readLane(double x, int lane) {
  const unsigned long long b = __builtin_bit_cast(unsigned long long, x);
  const unsigned lo          = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)b, lane);
  const unsigned hi          = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)(b >> 32), lane);
  return __builtin_bit_cast(double, ((unsigned long long)hi << 32) | lo);
}

// min(a, |b|); the compiler's fmin first quiets both operands, an instruction each
__device__ inline double minAbs(double a, double b) {
  double m;
  asm("v_min_f64 %0, %1, |%2|" : "=v"(m) : "v"(a), "v"(b));
  return m;
}
__device__ inline double minOf(double a, double b) {
  double m;
  asm("v_min_f64 %0, %1, %2" : "=v"(m) : "v"(a), "v"(b));
  return m;
}
__device__ inline double maxAbs(double a, double b) {
  double m;
  asm("v_max_f64 %0, %1, |%2|" : "=v"(m) : "v"(a), "v"(b));
  return m;
}

// orders the LDS accesses of one wavefront's lanes
__device__ inline void waveSync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
}

// One wavefront per workgroup takes E elements: it evaluates their 8 E Gauss points together, then condenses one element
// after the other. The points' data stay in LDS (4 KB per element); an element's K and R replace them on their way out.
// 96 x 96 x 48 elements, Neo-Hooke: 2.84 ms against 5.4 ms for the former kernel (one element per wavefront, sums by
// owned entries), whose 1,300 LDS accesses per element alone need 3.7 ms. With E = 4; 2: 3.1 ms; 8 elements in 2 or 4
// wavefronts: 2.9 and 3.1 ms; three wavefronts per SIMD at 168 registers: 3.3 ms with C in LDS, 4.3 ms with spills.
// What bounds it now: the matrix and vector pipes one after the other (per element 99 MFMAs of 64 cycles and 1,350
// vector instructions of 4: 2.3 ms); 3.8 GB are written (0.6 ms).
// Meshes that leave SIMDs idle take fewer elements per wavefront; assembly and update with E = 1 / 2 / 4, us:
//   512 elements 105 / 111 / 124, 2,048: 116 / 117 / 130, 9,216: 190 / 187 / 194, 18,432: 287 / 264 / 266,
//   98,304: 1,146 / 1,035 / 988.
constexpr int64_t kEasOne = 2048, kEasTwo = 16384;  // largest counts for E = 1 and 2
constexpr double kGaussX  = 2.0 * 0.28867513459481288225;  // |x| of a Gauss point

struct EasPoint {
  double C[22];     // C dV (packed upper; one entry of padding)
  double G[8][3];   // shape-function gradients g_a
  double F[9];
  double w;         // 1 / (detJ detJ0)
  double S[6];      // S dV
};
static_assert(sizeof(EasPoint) == 62 * 8, "62 doubles: the four points of a step lie in different LDS banks");
template <int E>
struct EasLds {
  union {
    struct {
      double X[24], U[24], alpha[NE + 1];
    } in;
    EasPoint pt[8];
    double out[36 * 9 + 24 + 4 + 64];  // K blocks, R, one slot per lane for entries that are not stored
  } u[E];
  double Ji0[E][10];  // inverse Jacobian at the centre
  int bad[E];
};

// Where the lanes of an element's wavefront put K and R into its output area, and find the blocks' entries there
struct EasTables {
  uint32_t put[6][64];  // positions of registers 2 m and 2 m + 1 of the tiles (1,1), (1,2), (2,2)
  uint32_t get[6][64];  // entry n = 64 m + lane of the 36 blocks: n % 9, block << 4, position << 10, transposed << 20
};
constexpr EasTables easTables() {
  EasTables t{};
  for (int lane = 0; lane < 64; ++lane)
    for (int m = 0; m < 6; ++m) {
      uint32_t w = 0;
      for (int h = 0; h < 2; ++h) {
        const int v = 2 * m + h, I = v < 8 ? 1 : 2, J = v < 4 ? 1 : 2;
        const int i = 16 * I + 4 * (v & 3) + lane / 16 - NE, j = 16 * J + lane % 16 - NE;
        uint32_t o = 352 + lane;  // not stored from there
        if (i >= 0 && i < 24 && j == 24) o = 324 + i;
        if (i >= 0 && i <= j && j < 24) o = 9 * upperBlock(i / 3, j / 3) + 3 * (i % 3) + j % 3;
        w |= o << (16 * h);
      }
      t.put[m][lane] = w;
      const int n = 64 * m + lane;
      if (n >= 324) continue;
      const int blk = n / 9, r = n % 9, rt = 3 * (r % 3) + r / 3;
      int src = r, srcT = rt;  // diagonal blocks: the lower triangle from the upper one
      for (int a = 0; a < 8; ++a)
        if (blk == upperBlock(a, a)) src = srcT = r < rt ? r : rt;
      t.get[m][lane] = r | blk << 4 | (9 * blk + src) << 10 | (9 * blk + srcT) << 20;
    }
  return t;
}
__constant__ const EasTables kEasTables = easTables();

// inverse of a 3x3 matrix of determinant 1 / id
__device__ inline void inv3(const double J[3][3], double id, double Ji[3][3]) {
  Ji[0][0] = (J[1][1] * J[2][2] - J[1][2] * J[2][1]) * id;
  Ji[0][1] = (J[0][2] * J[2][1] - J[0][1] * J[2][2]) * id;
  Ji[0][2] = (J[0][1] * J[1][2] - J[0][2] * J[1][1]) * id;
  Ji[1][0] = (J[1][2] * J[2][0] - J[1][0] * J[2][2]) * id;
  Ji[1][1] = (J[0][0] * J[2][2] - J[0][2] * J[2][0]) * id;
  Ji[1][2] = (J[0][2] * J[1][0] - J[0][0] * J[1][2]) * id;
  Ji[2][0] = (J[1][0] * J[2][1] - J[1][1] * J[2][0]) * id;
  Ji[2][1] = (J[0][1] * J[2][0] - J[0][0] * J[2][1]) * id;
  Ji[2][2] = (J[0][0] * J[1][1] - J[0][1] * J[1][0]) * id;
}

// S and C (Voigt) at the enhanced strain
template <int KIND>
__device__ inline bool material(double lam, double mu, const double Ev[6], double S[6], double Cp[21]) {
  if constexpr (KIND == IK_SVK) {
    const double tr = Ev[0] + Ev[1] + Ev[2];
    for (int i = 0; i < 3; ++i) S[i] = lam * tr + 2.0 * mu * Ev[i];
    for (int i = 3; i < 6; ++i) S[i] = mu * Ev[i];
    for (int i = 0; i < 21; ++i) Cp[i] = 0.0;
    for (int p = 0; p < 3; ++p)
      for (int q = p; q < 3; ++q) Cp[sym6(p, q)] = lam + (p == q ? 2.0 * mu : 0.0);
    for (int p = 3; p < 6; ++p) Cp[sym6(p, p)] = mu;
    return true;
  } else {
    double C[3][3];
    for (int v = 0; v < 6; ++v) {
      const int i = vI(v), j = vJ(v);
      const double e = v < 3 ? Ev[v] : 0.5 * Ev[v];
      C[i][j] = C[j][i] = 2.0 * e + (i == j ? 1.0 : 0.0);
    }
    const double detC = det3(C);
    if (!(detC > 0.0)) return false;
    const double id = 1.0 / detC;
    double Ci[3][3];
    inv3(C, id, Ci);
    const double lnJ = log(sqrt(detC));
    const double c2  = mu - lam * lnJ;
    for (int v = 0; v < 6; ++v) {
      const double ci = Ci[vI(v)][vJ(v)];
      S[v]            = mu * ((v < 3 ? 1.0 : 0.0) - ci) + lam * lnJ * ci;
    }
    for (int p = 0; p < 6; ++p)
      for (int q = p; q < 6; ++q) {
        const int I = vI(p), J = vJ(p), K = vI(q), L = vJ(q);
        Cp[sym6(p, q)] = lam * Ci[I][J] * Ci[K][L] + c2 * (Ci[I][K] * Ci[J][L] + Ci[I][L] * Ci[J][K]);
      }
    return true;
  }
}

// Phase 1 (lane (element, Gauss point)): kinematics, enhanced strain E + M alpha, material.
// Phase 2 (element by element): lane (c, q) = (lane % 16, lane / 16) forms columns c, 16 + c and 32 + c of N and CN at
// the points 2 q and 2 q + 1, whose 6 rows are the contraction steps: the values are the operands of
// v_mfma_f64_16x16x4 (A[i][k] and B[k][j] at lane 16 k + i or j) as they stand. Tile (I, J) of the sum holds entry
// (16 I + 4 v + q, 16 J + c) in its register v; columns 0-20 are the modes, 21-44 the displacements, 45 the residual.
// Phase 3: elimination of the mode rows, four at a time: register v of a tile row is the panel P (rows 4 v + q), again
// in operand layout; with the inverse of its 4 x 4 diagonal block (by 2 x 2 blocks; the reference inverts D by LU,
// enhancedassumedstrains.hh:243,294,344) What = P_pp^-1 P, and tiles -= P^T What. What remains at the displacement
// columns is K_uu - L^T D^-1 L and R_u - L^T D^-1 Rt. D is SPD while the material tangent is positive definite; a pivot
// that is not finite or vanishes against the largest entry of D makes the element singular (error flag word 1).
// Phase 4: the geometric part sum_g g_a . S dV g_b, diagonal blocks mirrored from their upper triangle, faces' loads.
template <int KIND, bool WANT_K, int E>
__global__ __launch_bounds__(64, 2) void easElement(const double* __restrict__ X, const double* __restrict__ U,
                                                          const int32_t* __restrict__ conn,
                                                          const double* __restrict__ alpha, int64_t e0, int64_t count,
                                                          double lam, double mu, const int32_t* __restrict__ dest,
                                                          const int32_t* __restrict__ rdest,
                                                          double* __restrict__ Kebe, double* __restrict__ Rebe,
                                                          const uint8_t* __restrict__ fbits, double3 trac,
                                                          double* __restrict__ cache,
                                                          unsigned long long* __restrict__ err) {
  __shared__ __attribute__((aligned(16))) EasLds<E> s;
  const int lane   = threadIdx.x;
  const int64_t i0 = (int64_t)blockIdx.x * E;  // first element of the workgroup, of `count` from e0
  const int nel    = count - i0 < E ? (int)(count - i0) : E;
  const int el0 = lane >> 3, gp = lane & 7;  // phase 1: the lane's element (el0 < nel) and Gauss point
  if (el0 < nel) {
    const int64_t nd = conn[(e0 + i0 + el0) * 8 + gp];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      s.u[el0].in.X[3 * gp + k] = X[nd * 3 + k];
      s.u[el0].in.U[3 * gp + k] = U[nd * 3 + k];
    }
  }
  for (int i = lane; i < nel * NE; i += 64) s.u[i / NE].in.alpha[i % NE] = alpha[(e0 + i0) * NE + i];
  if (lane < E) s.bad[lane] = 0;
  waveSync();
  if (el0 < nel) {
    const double d = 0.28867513459481288225;
    double xi[3], xm[3];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      xi[k] = ((gp >> k) & 1) ? 0.5 + d : 0.5 - d;
      xm[k] = 1.0 - xi[k];
    }
    // dN_a/dxi_k = +- f[k][m], m the corner's position in the other two directions
    double f[3][4];
#pragma unroll
    for (int m = 0; m < 4; ++m) {
      f[0][m] = ((m & 1) ? xi[1] : xm[1]) * ((m & 2) ? xi[2] : xm[2]);
      f[1][m] = ((m & 1) ? xi[0] : xm[0]) * ((m & 2) ? xi[2] : xm[2]);
      f[2][m] = ((m & 1) ? xi[0] : xm[0]) * ((m & 2) ? xi[1] : xm[1]);
    }
    // A[i][k] = sum_a Y_ai dN_a/dxi_k, and at the centre
    auto gradient = [&](const double* Y, double A[3][3], double (*A0)[3]) {
#pragma unroll
      for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int k = 0; k < 3; ++k) {
          double a = 0.0, a0 = 0.0;
#pragma unroll
          for (int m = 0; m < 4; ++m) {
            const int lo = k == 0 ? 2 * m : (k == 1 ? (m & 1) + 4 * (m >> 1) : m);
            const double y = Y[3 * (lo + (1 << k)) + i] - Y[3 * lo + i];
            a += y * f[k][m];
            a0 += y;
          }
          A[i][k] = a;
          if (A0) A0[i][k] = 0.25 * a0;
        }
    };
    double J[3][3], J0[3][3], Ji[3][3], Ji0[3][3], H[3][3], F[3][3];
    gradient(s.u[el0].in.X, J, J0);
    const double detJ = det3(J), dJ0 = det3(J0);
    inv3(J, 1.0 / detJ, Ji);
    inv3(J0, 1.0 / dJ0, Ji0);
    gradient(s.u[el0].in.U, H, nullptr);
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
      for (int j = 0; j < 3; ++j)
        F[i][j] = (i == j ? 1.0 : 0.0) + H[i][0] * Ji[0][j] + H[i][1] * Ji[1][j] + H[i][2] * Ji[2][j];
    // Mtilde alpha: one term per mode, in its row
    double wv[6] = {0, 0, 0, 0, 0, 0};
    const double sx[3] = {2.0 * xi[0] - 1.0, 2.0 * xi[1] - 1.0, 2.0 * xi[2] - 1.0};
#pragma unroll
    for (int c = 0; c < NE; ++c) {
      double fc = s.u[el0].in.alpha[c];
#pragma unroll
      for (int k = 0; k < 3; ++k)
        if ((monomialOf(c) >> k) & 1) fc *= sx[k];
      wv[kRowOf(c)] += fc;
    }
    waveSync();  // the points' data take the place of the element's inputs
    EasPoint& P = s.u[el0].pt[gp];
#pragma unroll
    for (int a = 0; a < 8; ++a) {
      const double d0 = (a & 1) ? f[0][a >> 1] : -f[0][a >> 1];
      const double d1 = (a & 2) ? f[1][(a & 1) + 2 * (a >> 2)] : -f[1][(a & 1) + 2 * (a >> 2)];
      const double d2 = (a & 4) ? f[2][a & 3] : -f[2][a & 3];
#pragma unroll
      for (int i = 0; i < 3; ++i) P.G[a][i] = Ji[0][i] * d0 + Ji[1][i] * d1 + Ji[2][i] * d2;
    }
    double Ev[6];
#pragma unroll
    for (int v = 0; v < 6; ++v) {
      const int I = vI(v), Jj = vJ(v);
      const double c = F[0][I] * F[0][Jj] + F[1][I] * F[1][Jj] + F[2][I] * F[2][Jj];
      Ev[v]          = v < 3 ? 0.5 * (c - 1.0) : c;  // engineering shear 2E_IJ = C_IJ
    }
    // E += M alpha = T0^-1 (Mtilde alpha) / detJ, T0^-1 w = Ji0^T w Ji0 / detJ0 on the strain tensor w (T(J)^-1 =
    // T(J^-1): the Voigt strain transformation represents the Jacobian, tensorutils.hh:440-465)
    const double w = 1.0 / (fabs(detJ) * fabs(dJ0));
    double T[3][3];
#pragma unroll
    for (int k = 0; k < 3; ++k)
#pragma unroll
      for (int b = 0; b < 3; ++b) {
        T[k][b] = 0.0;
#pragma unroll
        for (int l = 0; l < 3; ++l)
          T[k][b] += (k == l ? wv[k] : 0.5 * wv[k + l == 3 ? 3 : (k + l == 2 ? 4 : 5)]) * Ji0[l][b];
      }
#pragma unroll
    for (int v = 0; v < 6; ++v) {
      const int a = vI(v), b = vJ(v);
      const double m = Ji0[0][a] * T[0][b] + Ji0[1][a] * T[1][b] + Ji0[2][a] * T[2][b];
      Ev[v] += (v < 3 ? m : 2.0 * m) * w;
    }
    double Sv[6], Cp[21];
    if (!material<KIND>(lam, mu, Ev, Sv, Cp)) {
      atomicMin(err, (unsigned long long)(e0 + i0 + el0));
      s.bad[el0] = 1;
    }
    const double dV = fabs(detJ) * 0.125;
#pragma unroll
    for (int i = 0; i < 21; ++i) P.C[i] = Cp[i] * dV;
#pragma unroll
    for (int i = 0; i < 9; ++i) P.F[i] = F[i / 3][i % 3];
#pragma unroll
    for (int v = 0; v < 6; ++v) P.S[v] = Sv[v] * dV;
    P.w = w;
    if (gp == 0)
#pragma unroll
      for (int i = 0; i < 9; ++i) s.Ji0[el0][i] = Ji0[i / 3][i % 3];
  }
  __syncthreads();

  // the lane's columns: modes c and, for c < 5, 16 + c; displacements c - 5 (c >= 5, tile 1), 11 + c (c < 13, tile 2)
  const int c = lane & 15, q = lane >> 4;
  const bool mode1 = c < 5, rhs2 = c == 13;
  const int col1 = mode1 ? 0 : c - 5, col2 = c < 13 ? c + 11 : 23;
  const int b1 = col1 / 3, l1 = col1 - 3 * b1, b2 = col2 / 3, l2 = col2 - 3 * b2;
  // Voigt row and monomial of the lane's modes
  const int md1 = mode1 ? 16 + c : 16;
  const int row0 = (int)((packModes(true) >> (3 * c)) & 7), row1 = (int)((packModes(true) >> (3 * md1)) & 7);
  const int mono0 = (int)((packModes(false) >> (3 * c)) & 7), mono1 = (int)((packModes(false) >> (3 * md1)) & 7);
  // rows k, l of the centre's inverse Jacobian for them
  const int k0 = 3 * (row0 < 3 ? row0 : (row0 == 3 ? 1 : 0)), n0 = 3 * (row0 < 3 ? row0 : (row0 == 5 ? 1 : 2));
  const int k1 = 3 * (row1 < 3 ? row1 : (row1 == 3 ? 1 : 0)), n1 = 3 * (row1 < 3 ? row1 : (row1 == 5 ? 1 : 2));
  auto modeAt = [](int mono, int gp) {  // f_c at a Gauss point
    const double f = __popc(mono) == 1 ? kGaussX : kGaussX * kGaussX;
    return (__popc(mono & ~gp) & 1) ? -f : f;
  };
  const int ga = 4 * ((lane >> 3) & 1) + (lane & 3), gb = 4 * ((lane >> 2) & 1) + (lane & 3);  // geometric part: nodes
  const double unit[4] = {q == 0 ? 1.0 : 0.0, q == 1 ? 1.0 : 0.0, q == 2 ? 1.0 : 0.0, q == 3 ? 1.0 : 0.0};

  for (int el = 0; el < nel; ++el) {
    if (s.bad[el]) continue;  // uniform: the error flag is already set
    const int64_t e   = e0 + i0 + el;
    const EasPoint* points = s.u[el].pt;
    v4d t00 = {0, 0, 0, 0}, t01 = t00, t02 = t00, t11 = t00, t12 = t00, t22 = t00;
    double kg = 0.0;
    // columns of T0^-1 detJ0: the strain of directions (Jk, Jl), as a displacement column is that of (F_l, g_b)
    const double* Ji = s.Ji0[el];
#pragma unroll 1  // both points at once take more registers than two wavefronts per SIMD leave
    for (int p = 0; p < 2; ++p) {
      const EasPoint& P = points[2 * q + p];
      double C[21], S[6], N0[6], N1[6], N2[6], cn[6];
#pragma unroll
      for (int i = 0; i < 21; ++i) C[i] = P.C[i];
#pragma unroll
      for (int v = 0; v < 6; ++v) S[v] = P.S[v];
      auto strainColumn = [&](const double* A, const double* G, double f, double N[6]) {
        const double A0 = f * A[0], A1 = f * A[1], A2 = f * A[2], g0 = G[0], g1 = G[1], g2 = G[2];
        N[0] = A0 * g0;
        N[1] = A1 * g1;
        N[2] = A2 * g2;
        N[3] = A1 * g2 + A2 * g1;
        N[4] = A0 * g2 + A2 * g0;
        N[5] = A0 * g1 + A1 * g0;
      };
      auto times = [&](const double N[6], double y[6]) {
#pragma unroll
        for (int v = 0; v < 6; ++v) {
          double a = C[sym6(v, 0)] * N[0];
#pragma unroll
          for (int u = 1; u < 6; ++u) a += C[sym6(v, u)] * N[u];
          y[v] = a;
        }
      };
      const double w = P.w;
      // column by column of tiles, and no reordering across them: the registers of one column at a time
      strainColumn(Ji + k0, Ji + n0, modeAt(mono0, 2 * q + p) * w, N0);
      times(N0, cn);
#pragma unroll
      for (int v = 0; v < 6; ++v) t00 = __builtin_amdgcn_mfma_f64_16x16x4f64(N0[v], cn[v], t00, 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
      strainColumn(mode1 ? Ji + k1 : P.F + 3 * l1, mode1 ? Ji + n1 : P.G[b1],
                   mode1 ? modeAt(mono1, 2 * q + p) * w : 1.0, N1);
      times(N1, cn);
#pragma unroll
      for (int v = 0; v < 6; ++v) {
        t01 = __builtin_amdgcn_mfma_f64_16x16x4f64(N0[v], cn[v], t01, 0, 0, 0);
        t11 = __builtin_amdgcn_mfma_f64_16x16x4f64(N1[v], cn[v], t11, 0, 0, 0);
      }
      __builtin_amdgcn_sched_barrier(0);
      strainColumn(P.F + 3 * l2, P.G[b2], 1.0, N2);  // lanes 13-15: rows and columns that nothing reads
      times(N2, cn);
#pragma unroll
      for (int v = 0; v < 6; ++v) cn[v] = rhs2 ? S[v] : cn[v];
#pragma unroll
      for (int v = 0; v < 6; ++v) {
        t02 = __builtin_amdgcn_mfma_f64_16x16x4f64(N0[v], cn[v], t02, 0, 0, 0);
        t12 = __builtin_amdgcn_mfma_f64_16x16x4f64(N1[v], cn[v], t12, 0, 0, 0);
        t22 = __builtin_amdgcn_mfma_f64_16x16x4f64(N2[v], cn[v], t22, 0, 0, 0);
      }
      if constexpr (WANT_K) {
        double g[3], h[3];
#pragma unroll
        for (int i = 0; i < 3; ++i) {
          g[i] = P.G[ga][i];
          h[i] = P.G[gb][i];
        }
        kg = __builtin_amdgcn_mfma_f64_4x4x4f64(g[0], S[0] * h[0] + S[5] * h[1] + S[4] * h[2], kg, 0, 0, 0);
        kg = __builtin_amdgcn_mfma_f64_4x4x4f64(g[1], S[5] * h[0] + S[1] * h[1] + S[3] * h[2], kg, 0, 0, 0);
        kg = __builtin_amdgcn_mfma_f64_4x4x4f64(g[2], S[4] * h[0] + S[3] * h[1] + S[2] * h[2], kg, 0, 0, 0);
      }
    }

    // the lane's table entries and destinations, in flight during the elimination: ahead of the stores, whose
    // completion a load behind them waits for. (Loaded for each element, from a stand-in where there are none: held
    // over the loop above they would take its registers, and a branch would wait for them.)
    uint32_t put[6], get[6];
    int32_t code[6];
    int ln = lane;
    asm volatile("" : "+v"(ln));
    const int nd = ln < 24 ? ln / 3 : 7, kd = ln % 3;
    const int32_t* dfrom = dest ? dest + e * 36 : (const int32_t*)kEasTables.get;
    const int32_t* rfrom = (rdest ? rdest : conn) + e * 8;
    const uint8_t* ffrom = fbits ? fbits + e : (const uint8_t*)kEasTables.get;
#pragma unroll
    for (int m = 0; m < 6; ++m) {
      put[m]  = kEasTables.put[m][ln];
      get[m]  = kEasTables.get[m][ln];
      code[m] = dfrom[m < 5 || ln < 4 ? (ln + 64 * m) / 9 : 35];
    }
    const int32_t rcode = rfrom[nd];
    unsigned bits       = *ffrom;

    // the largest entry of D: all of tile (0, 0), columns 16-20 of (0, 1) and (1, 1) (rows 16-19 and 20)
    double dmax = 0.0;
#pragma unroll
    for (int v = 0; v < 4; ++v) dmax = maxAbs(maxAbs(dmax, t00[v]), mode1 ? t01[v] : 0.0);
    dmax = maxAbs(maxAbs(dmax, mode1 ? t11[0] : 0.0), mode1 && q == 0 ? t11[1] : 0.0);
    dmax = maxAbs(dmax, dppMove<0x111, 0xF>(dmax));  // over the wavefront, as waveSum
    dmax = maxAbs(dmax, dppMove<0x112, 0xF>(dmax));
    dmax = maxAbs(dmax, dppMove<0x114, 0xF>(dmax));
    dmax = maxAbs(dmax, dppMove<0x118, 0xF>(dmax));
    dmax = maxAbs(dmax, dppMove<0x142, 0xA>(dmax));
    dmax = maxAbs(dmax, dppMove<0x143, 0xC>(dmax));
    dmax = lane63(dmax);
    // The diagonal blocks are inverted times a power of two that brings D's largest entry to about 1: D scales with
    // mu h^-13 in the element's extent h, and the determinants with its square, which leaves the range of a double at
    // extents where D does not (mu = 8e10: h of 1e-11; without the scaling such elements were called singular). Exact,
    // so the results do not change: two multiplications per panel, the factor itself in scalar registers.
    const int dexp     = (int)(__builtin_bit_cast(unsigned long long, dmax) >> 52);  // dmax >= 0
    const double scale = __builtin_bit_cast(
        double, (unsigned long long)(2046 - (dexp < 1 ? 1 : (dexp > 2045 ? 2045 : dexp))) << 52);
    // Pivots against the threshold, per 2 x 2 block its first entry and its determinant over that. One that is not
    // finite makes all later ones NaN (its reciprocal is), so the last one shows it.
    const double limit = 1e-13 * dmax, limitS = limit * scale;
    double least = INFINITY, gap = INFINITY;
    auto block2 = [&](double a, double b, double c) {  // 1 / determinant
      const double det = a * c - b * b;
      least            = minAbs(least, a);
      gap              = minOf(gap, fma(-limitS, fabs(a), fabs(det)));
      return reciprocal(det);
    };
    double* cy = cache + e * kEasCache;
#pragma unroll
    for (int p = 0; p < 5; ++p) {
      const double P0 = p < 4 ? t00[p & 3] : 0.0, P1 = p < 4 ? t01[p & 3] : t11[0], P2 = p < 4 ? t02[p & 3] : t12[0];
      const double Pd = (p < 4 ? P0 : P1) * scale;
      const int lc    = p < 4 ? 4 * p : 0;
      auto a = [&](int k, int l) { return readLane(Pd, 16 * k + lc + l); };
      // scale D_pp = [A B; B^T C] by 2 x 2 blocks; x = column q of its inverse
      const double a00 = a(0, 0), a01 = a(0, 1), a11 = a(1, 1);
      const double b00 = a(0, 2), b01 = a(0, 3), b10 = a(1, 2), b11 = a(1, 3);
      const double ra = block2(a00, a01, a11);
      const double i00 = a11 * ra, i01 = -a01 * ra, i11 = a00 * ra;
      const double m00 = i00 * b00 + i01 * b10, m01 = i00 * b01 + i01 * b11;
      const double m10 = i01 * b00 + i11 * b10, m11 = i01 * b01 + i11 * b11;
      const double s00 = a(2, 2) - (b00 * m00 + b10 * m10), s01 = a(2, 3) - (b00 * m01 + b10 * m11);
      const double s11 = a(3, 3) - (b01 * m01 + b11 * m11);
      const double rs  = block2(s00, s01, s11);
      const double v0 = unit[2] - (m00 * unit[0] + m10 * unit[1]), v1 = unit[3] - (m01 * unit[0] + m11 * unit[1]);
      const double x2 = (s11 * v0 - s01 * v1) * rs, x3 = (s00 * v1 - s01 * v0) * rs;
      const double x0 = i00 * unit[0] + i01 * unit[1] - (m00 * x2 + m01 * x3);
      const double x1 = i01 * unit[0] + i11 * unit[1] - (m10 * x2 + m11 * x3);
      asm("" : : "v"(x0), "v"(x1), "v"(x2), "v"(x3));  // all four before the selection: no branches around them
      const double xr = ((lane & 2) ? ((lane & 1) ? x3 : x2) : ((lane & 1) ? x1 : x0)) * scale;
      const double W1 = __builtin_amdgcn_mfma_f64_4x4x4f64(xr, P1, 0.0, 0, 0, 0);
      const double W2 = __builtin_amdgcn_mfma_f64_4x4x4f64(xr, P2, 0.0, 0, 0, 0);
      if (p < 3) {
        const double W0 = __builtin_amdgcn_mfma_f64_4x4x4f64(xr, P0, 0.0, 0, 0, 0);
        t00             = __builtin_amdgcn_mfma_f64_16x16x4f64(-P0, W0, t00, 0, 0, 0);
        t01             = __builtin_amdgcn_mfma_f64_16x16x4f64(-P0, W1, t01, 0, 0, 0);
        t02             = __builtin_amdgcn_mfma_f64_16x16x4f64(-P0, W2, t02, 0, 0, 0);
        const int w = 12 - 4 * p;
        if (c >= 4 * (p + 1)) cy[cacheLow(p) + w * q + c - 4 * (p + 1)] = W0;
      }
      t11 = __builtin_amdgcn_mfma_f64_16x16x4f64(-P1, W1, t11, 0, 0, 0);
      t12 = __builtin_amdgcn_mfma_f64_16x16x4f64(-P1, W2, t12, 0, 0, 0);
      t22 = __builtin_amdgcn_mfma_f64_16x16x4f64(-P2, W2, t22, 0, 0, 0);
      cy[64 * p + lane] = W1;
      if (c < 14) cy[320 + 56 * p + 14 * q + c] = W2;
    }
    {  // row 20: register 1 of the tiles (1, J), lanes q = 0
      const double d20 = readLane(t11[1], 4), r20 = reciprocal(d20);
      if (!(least > limitS && gap > 0.0 && fabs(d20) > limit && fabs(d20) < INFINITY && dmax < INFINITY) && lane == 0)
        atomicMin(err + 1, (unsigned long long)e);
      const double P1 = q == 0 ? t11[1] : 0.0, P2 = q == 0 ? t12[1] : 0.0;
      const double W1 = P1 * r20, W2 = P2 * r20;
      t11 = __builtin_amdgcn_mfma_f64_16x16x4f64(-P1, W1, t11, 0, 0, 0);
      t12 = __builtin_amdgcn_mfma_f64_16x16x4f64(-P1, W2, t12, 0, 0, 0);
      t22 = __builtin_amdgcn_mfma_f64_16x16x4f64(-P2, W2, t22, 0, 0, 0);
      if (q == 0) {
        if (c >= 5) cy[696 + c - 5] = W1;
        if (c < 14) cy[696 + 11 + c] = W2;
      }
    }

    // K and R to LDS, over the element's points
    double* out = s.u[el].out;
    waveSync();
#pragma unroll
    for (int v = 0; v < 12; ++v) {
      const uint32_t o = (put[v / 2] >> (16 * (v & 1))) & 0xFFFF;
      out[o]           = v < 4 ? t11[v & 3] : (v < 8 ? t12[v & 3] : t22[v & 3]);
    }
    waveSync();
    if constexpr (WANT_K) {
      const int a = 4 * ((lane >> 3) & 1) + q;  // geometric entry (a, gb) of the lane
      if (a <= gb) {
        const int o = upperBlock(a, gb) * 9;
        const double d0 = out[o], d1 = out[o + 4], d2 = out[o + 8];
        out[o]     = d0 + kg;
        out[o + 4] = d1 + kg;
        out[o + 8] = d2 + kg;
      }
      waveSync();
#pragma unroll
      for (int m = 0; m < 6; ++m)
        if (lane + 64 * m < 324) {
          const int64_t pos = dest ? (int64_t)(code[m] >> 1) : e * 36 + ((get[m] >> 4) & 63);
          const bool turned = dest && (code[m] & 1);
          Kebe[pos * 9 + (get[m] & 15)] = out[turned ? get[m] >> 20 : (get[m] >> 10) & 1023];
        }
    }
    if (lane < 24) {
      double acc = out[324 + lane];
      if (fbits && bits)  // Traction skill, after the EAS element's condensed internal forces
        acc += faceLoad(X, conn, e, bits, nd, kd == 0 ? trac.x : (kd == 1 ? trac.y : trac.z));
      Rebe[rdest ? (int64_t)rcode * 3 + kd : e * 24 + lane] = acc;
    }
  }
}

// alpha_e -= D_e^-1 (Rt_e + L_e du_e) = Lb^-T (what_e + What_e du_e): 21 lanes per element, 3 elements per wavefront
// (lane 63 idle). The cache is read in one run per wavefront, into LDS. Lane i forms z_i = what_i + (What du)_i; the
// back substitution with Lb^T then runs from the last mode up, x_m = z_m reaching the lanes of earlier panels by a
// shuffle.
constexpr int kUpdElemsPerWave = 64 / NE, kUpdWaves = 4;
__global__ __launch_bounds__(64 * kUpdWaves) void easUpdateKernel(const double* __restrict__ cache,
                                                                  const int32_t* __restrict__ conn,
                                                                  const double* __restrict__ du, int64_t ne,
                                                                  double* __restrict__ alpha) {
  __shared__ v2d sw[kUpdWaves][kUpdElemsPerWave * kEasCache / 2];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, sub = lane / NE, i = lane - NE * sub;
  const int64_t ew  = ((int64_t)blockIdx.x * kUpdWaves + wave) * kUpdElemsPerWave, e = ew + sub;
  const bool active = sub < kUpdElemsPerWave && e < ne;
  const int64_t nw  = ne - ew < kUpdElemsPerWave ? (ne - ew > 0 ? ne - ew : 0) : kUpdElemsPerWave;
  constexpr int RUN = (kUpdElemsPerWave * kEasCache / 2 + 63) / 64;
  const int run     = (int)nw * (kEasCache / 2);
  const v2d* src = (const v2d*)(cache + ew * kEasCache);
  v2d v[RUN];
#pragma unroll
  for (int m = 0; m < RUN; ++m)
    if (lane + 64 * m < run) v[m] = src[lane + 64 * m];
  double d[24];
  if (active)
#pragma unroll
    for (int a = 0; a < 8; ++a) {
      const int64_t nd = conn[e * 8 + a];
#pragma unroll
      for (int k = 0; k < 3; ++k) d[3 * a + k] = du[nd * 3 + k];
    }
#pragma unroll
  for (int m = 0; m < RUN; ++m)
    if (lane + 64 * m < run) sw[wave][lane + 64 * m] = v[m];
  waveSync();
  const double* cy = (const double*)sw[wave] + (active ? sub : 0) * kEasCache;
  const int p = i >> 2, k = i & 3;
  const double* c1 = i < 20 ? cy + 64 * p + 16 * k - 16 : cy + 696 - NE;        // columns 16-31
  const double* c2 = i < 20 ? cy + 320 + 56 * p + 14 * k - 32 : cy + 696 - NE;  // columns 32-45
  double z         = 0.0;
  if (active) {
    z = c2[45];
#pragma unroll
    for (int j = 0; j < 24; ++j) z += (j < 11 ? c1 : c2)[NE + j] * d[j];
  }
  // every lane takes part in the shuffles; lanes of other elements and idle lanes read values they drop
  const double* c0 = cy + cacheLow(p) + (12 - 4 * p) * k - 4 * (p + 1);  // columns below 16 (panels 0-2)
#pragma unroll
  for (int m = NE - 1; m >= 4; --m) {
    const double xm = __shfl(z, NE * sub + m, 64);
    if (active && p < (m >> 2)) z -= (m < 16 ? c0 : c1)[m] * xm;
  }
  if (active) alpha[e * NE + i] -= z;
}

template <bool WK, int E>
void launchEasElems(ik_handle* h, int64_t e0, int64_t count, const int32_t* dest, const int32_t* rdest, double* Kebe) {
  auto launch = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3((unsigned)((count + E - 1) / E)), dim3(64), 0, h->stream, h->X.p, h->u.p,
                       h->conn.p, h->alpha.p, e0, count, h->lam, h->mu, dest, rdest, Kebe, h->ebeR.p, h->faceBits.p,
                       loadedTraction(h), h->easCache.p, h->errFlag.p);
  };
  if (h->material == IK_SVK)
    launch(easElement<IK_SVK, WK, E>);
  else
    launch(easElement<IK_NEOHOOKE, WK, E>);
}
template <bool WK>
void launchEas(ik_handle* h, int64_t e0, int64_t count, const int32_t* dest, const int32_t* rdest, double* Kebe) {
  (count <= kEasOne   ? launchEasElems<WK, 1>
   : count <= kEasTwo ? launchEasElems<WK, 2>
                      : launchEasElems<WK, 4>)(h, e0, count, dest, rdest, Kebe);
}

}  // namespace

void easStage(ik_handle* h, int64_t e0, int64_t count, bool wantK, const int32_t* dest, const int32_t* rdest) {
  h->easCache.ensure((size_t)h->ne * kEasCache);
  if (wantK)
    launchEas<true>(h, e0, count, dest, rdest, h->ebeK64.p);
  else
    launchEas<false>(h, e0, count, nullptr, rdest, nullptr);
}

void easUpdate(ik_handle* h, const double* duDev) {
  require(h->easCacheValid, IK_EINVAL, "EAS update needs D, L, Rt of the current state (assemble first)");
  const int64_t perBlock = kUpdWaves * kUpdElemsPerWave;
  hipLaunchKernelGGL(easUpdateKernel, dim3((unsigned)((h->ne + perBlock - 1) / perBlock)), dim3(64 * kUpdWaves), 0,
                     h->stream, h->easCache.p, h->conn.p, duDev, h->ne, h->alpha.p);
  h->easCacheValid = false;
}

}  // namespace ik

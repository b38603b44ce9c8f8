// mlp.hip — the learned load-step predictor: a per-node MLP 14 -> 128 -> 128 -> 128 -> 3 with SiLU
// activations, trained and evaluated on the GPU. No reference counterpart: it replaces the constant
// (loadcontrol.inl:55-57) / secant (pathfollowingfunctions.hh:188-195) displacement predictor, and
// NewtonRaphson still has to reach the same ||R|| tolerance from the predicted state.
//
// Products run on the BF16 matrix instructions: operands rounded to BF16 (round to nearest even), FP32 accumulation,
// parameters with an FP32 master copy updated by Adam. Training takes three launches per step: forward and backward of
// the activations (mlpRows), the weight and bias gradients per batch slice (mlpWeightGrad), and their sum over the
// slices with the Adam update (mlpFold). The prediction inside the load loop runs in one fused kernel (features, four
// layers, update of u).
//
// Features of node v for the step n -> n+1 (load increment dlam, velocities v_n = du_n / dlam):
//   [ X_v / L (3), t / 40 (3), lam_{n+1}, 40 dlam, v_n / 0.1 (3), v_{n-1} / 0.1 (3) ]
// Output y (3): v_{n+1} = v_n + 0.1 y, u_pred = u_n + dlam v_{n+1} (clamped DOFs keep u_n).
#include <cmath>
#include <mutex>

#include "ik_internal.hh"

namespace ik {

constexpr int kIn = 14, kHid = 128, kOut = 3;
constexpr int64_t kParams = kHid * kIn + kHid + 2 * (kHid * kHid + kHid) + kOut * kHid + kOut;
// parameter offsets
constexpr int64_t oW1 = 0, oB1 = oW1 + kHid * kIn, oW2 = oB1 + kHid, oB2 = oW2 + kHid * kHid, oW3 = oB2 + kHid,
                  oB3 = oW3 + kHid * kHid, oW4 = oB3 + kHid, oB4 = oW4 + kOut * kHid;
constexpr double kVelScale = 0.1, kTracScale = 1.0 / 40.0, kDlamScale = 40.0;

namespace {

typedef short bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

// FP32 -> BF16 bits, round to nearest even (NaN kept quiet): v_cvt_pk_bf16_f32
__device__ inline uint16_t toBf16(float f) { return __builtin_bit_cast(uint16_t, (__bf16)f); }

// logistic function and SiLU; the reciprocal is v_rcp_f32 (1 ulp), 1 + e^-z >= 1 so it never sees a denormal
__device__ inline float sigmoid(float z) { return __builtin_amdgcn_rcpf(1.f + __expf(-z)); }
__device__ inline float silu(float z) { return z * sigmoid(z); }

// ---- training and batched forward -----------------------------------------------------------------------------
// One wavefront = 16 rows at a time, weights in LDS as BF16, every activation and every
// pre-activation of a row in registers from the features to the loss gradient and back. Each layer is computed
// transposed, out^T (outputs x 16 rows) = W act^T, with W as the MFMA A operand: lane (n, kq) = (lane & 15,
// lane >> 4) then holds outputs 16 t + 4 kq + r of row n (C fragment of tile t), which is the B fragment of K step t
// of the next layer on v_mfma_f32_16x16x16bf16_1k, in the natural order of the inputs, so no value moves between
// lanes. The backward products dA^T = W^T dZ^T run the same way on a transposed copy of the weights. Operands are
// rounded to BF16 (nearest even), K runs in steps of 16 in increasing order with FP32 accumulation, then the bias.
// Bound: a batch of 8192 rows is 3.5 GFLOP over 512 wavefronts (half of one per SIMD), so latency (LDS fragment ->
// MFMA -> SiLU chains) and the staging of the weights, not the matrix rate. Layer by layer through memory, the
// forward and backward products, SiLU' and loss kernels of that batch took 11 launches and 116 us; this kernel takes
// 24 us (26 with 4 wavefronts per workgroup in training: 8 stage the 140 KB of parameters faster).
constexpr int kWr = kHid + 8;  // padded row of 128 BF16 values (68 dwords): the 16 rows of a fragment read spread over
                               // the banks
// LDS layout (BF16 values): W1 [128][16], W2, W3 [128][kWr], W4 [16][kWr] (rows past the 3 outputs zero), and for the
// backward pass W2^T, W3^T [128][kWr], W4^T [128][16] (columns past 3 zero)
constexpr int lW1 = 0, lW2 = lW1 + kHid * 16, lW3 = lW2 + kHid * kWr, lW4 = lW3 + kHid * kWr, lEndF = lW4 + 16 * kWr,
              lT2 = lEndF, lT3 = lT2 + kHid * kWr, lT4 = lT3 + kHid * kWr, lEndB = lT4 + kHid * 16;
static_assert(lEndB * 2 + (3 * kHid + 16) * 4 + 64 <= 160 * 1024, "weights and their transposes fit the LDS of a CU");

__device__ inline bf16x4 pack4(float a, float b, float c, float d) {
  return bf16x4{(short)toBf16(a), (short)toBf16(b), (short)toBf16(c), (short)toBf16(d)};
}
// four consecutive BF16 values of a weight row in LDS (8-byte aligned): a 16x16x16 A fragment
__device__ inline bf16x4 wfrag(const uint16_t* w) { return *reinterpret_cast<const bf16x4*>(w); }

// acc[t] = tile t of W act^T for T output tiles: W rows of `ld` values in LDS, KS steps of 16 inputs
template <int T, int KS>
__device__ inline void layerT(const uint16_t* W, int ld, int n, int kq, const bf16x4* act, f32x4* acc) {
  // keeps the fragment reads here (hoisted out of the row loop they would spill hundreds of registers)
  asm volatile("" ::: "memory");
#pragma unroll
  for (int t = 0; t < T; ++t) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int s = 0; s < KS; ++s)
#pragma unroll
    for (int t = 0; t < T; ++t)
      acc[t] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(wfrag(W + (16 * t + n) * ld + 16 * s + 4 * kq), act[s], acc[t],
                                                         0, 0, 0);
}

// BACK: the hidden activations A[l] and the gradients dZ[l] (n x 128) and dY (n x 3) go to memory for the weight
// gradients, with the workgroup's sum of (y - t)^2 in partial[blockIdx.x]. Otherwise only the outputs y (n x 3).
template <bool BACK>
__global__ __launch_bounds__(BACK ? 512 : 256) void mlpRows(const float* __restrict__ P, const float* __restrict__ X,
                                                             const float* __restrict__ Tg, int64_t n, float scale,
                                                             float* __restrict__ Y, float* __restrict__ A0,
                                                             float* __restrict__ A1, float* __restrict__ A2,
                                                             float* __restrict__ D0, float* __restrict__ D1,
                                                             float* __restrict__ D2, float* __restrict__ dY,
                                                             double* __restrict__ partial) {
  constexpr int BS = BACK ? 512 : 256;
  __shared__ __align__(16) uint16_t sW[BACK ? lEndB : lEndF];
  __shared__ float sB[3 * kHid + 16];
  __shared__ double red[BS / 64];
  const int tid = threadIdx.x;
  for (int i = tid; i < kHid * 16; i += BS) {
    const int j = i >> 4, k = i & 15;
    sW[lW1 + i] = toBf16(k < kIn ? P[oW1 + j * kIn + k] : 0.f);
    if constexpr (BACK) sW[lT4 + i] = toBf16(k < kOut ? P[oW4 + k * kHid + j] : 0.f);
  }
  for (int i = tid; i < 16 * kHid; i += BS) {
    const int j = i >> 7, k = i & 127;
    sW[lW4 + j * kWr + k] = toBf16(j < kOut ? P[oW4 + j * kHid + k] : 0.f);
  }
#pragma unroll 4
  for (int i = tid; i < kHid * kHid / 4; i += BS) {  // four inputs of one output at a time
    const int j = i >> 5, k = 4 * (i & 31);
    const float* w2 = P + oW2 + j * kHid + k;
    const float* w3 = P + oW3 + j * kHid + k;
    *reinterpret_cast<bf16x4*>(&sW[lW2 + j * kWr + k]) = pack4(w2[0], w2[1], w2[2], w2[3]);
    *reinterpret_cast<bf16x4*>(&sW[lW3 + j * kWr + k]) = pack4(w3[0], w3[1], w3[2], w3[3]);
  }
  if constexpr (BACK) {
#pragma unroll 4
    for (int i = tid; i < kHid * kHid / 4; i += BS) {  // four outputs of one input, for the transposes
      const int k = i & 127, j = 4 * (i >> 7);
      const float* w2 = P + oW2 + j * kHid + k;
      const float* w3 = P + oW3 + j * kHid + k;
      *reinterpret_cast<bf16x4*>(&sW[lT2 + k * kWr + j]) = pack4(w2[0], w2[kHid], w2[2 * kHid], w2[3 * kHid]);
      *reinterpret_cast<bf16x4*>(&sW[lT3 + k * kWr + j]) = pack4(w3[0], w3[kHid], w3[2 * kHid], w3[3 * kHid]);
    }
  }
  for (int i = tid; i < 3 * kHid + 16; i += BS) {
    float v = 0.f;
    if (i < kHid) v = P[oB1 + i];
    else if (i < 2 * kHid) v = P[oB2 + i - kHid];
    else if (i < 3 * kHid) v = P[oB3 + i - 2 * kHid];
    else if (i - 3 * kHid < kOut) v = P[oB4 + i - 3 * kHid];
    sB[i] = v;
  }
  __syncthreads();
  const int lane = tid & 63, nl = lane & 15, kq = lane >> 4;
  double sq = 0.0;
  for (int64_t r0 = ((int64_t)blockIdx.x + (int64_t)gridDim.x * (tid >> 6)) * 16; r0 < n;
       r0 += (int64_t)gridDim.x * (BS / 4)) {
    const int64_t v  = r0 + nl;
    const bool valid = v < n;
    float f[4] = {0.f, 0.f, 0.f, 0.f};
    if (valid)
#pragma unroll
      for (int q = 0; q < 4; ++q)
        if (4 * kq + q < kIn) f[q] = X[v * kIn + 4 * kq + q];
    bf16x4 act[8];
    f32x4 Z[3][8], acc[8];
    act[0] = pack4(f[0], f[1], f[2], f[3]);
    // pre-activation, SiLU, the next layer's B fragments (and the activations to memory)
    auto activate = [&](int l, float* Al) {
#pragma unroll
      for (int t = 0; t < 8; ++t) {
        f32x4 a;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          Z[l][t][r] = acc[t][r] + sB[l * kHid + 16 * t + 4 * kq + r];
          a[r]       = silu(Z[l][t][r]);
        }
        act[t] = pack4(a[0], a[1], a[2], a[3]);
        if constexpr (BACK)
          if (valid) *reinterpret_cast<f32x4*>(&Al[v * kHid + 16 * t + 4 * kq]) = a;
      }
    };
    layerT<8, 1>(sW + lW1, 16, nl, kq, act, acc);
    activate(0, A0);
    layerT<8, 8>(sW + lW2, kWr, nl, kq, act, acc);
    activate(1, A1);
    layerT<8, 8>(sW + lW3, kWr, nl, kq, act, acc);
    activate(2, A2);
    layerT<1, 8>(sW + lW4, kWr, nl, kq, act, acc);
    // lanes kq = 0 hold the outputs 0..2 of row n
    const bool out = valid && kq == 0;
    float g[3] = {0.f, 0.f, 0.f};
    if (out) {
#pragma unroll
      for (int k = 0; k < kOut; ++k) {
        const float y = acc[0][k] + sB[3 * kHid + k];
        if constexpr (BACK) {
          const float d = y - Tg[v * kOut + k];
          g[k]          = 2.f * d * scale;
          sq += (double)d * d;
          dY[v * kOut + k] = g[k];
        } else {
          Y[v * kOut + k] = y;
        }
      }
    }
    if constexpr (BACK) {
      act[0] = pack4(g[0], g[1], g[2], 0.f);
      // dZ = dA silu'(Z), the B fragments of the next product (and dZ to memory)
      auto gradient = [&](int l, float* Dl) {
#pragma unroll
        for (int t = 0; t < 8; ++t) {
          f32x4 d;
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const float z = Z[l][t][r], sg = sigmoid(z);
            d[r]          = acc[t][r] * sg * (1.f + z * (1.f - sg));
          }
          act[t] = pack4(d[0], d[1], d[2], d[3]);
          if (valid) *reinterpret_cast<f32x4*>(&Dl[v * kHid + 16 * t + 4 * kq]) = d;
        }
      };
      layerT<8, 1>(sW + lT4, 16, nl, kq, act, acc);
      gradient(2, D2);
      layerT<8, 8>(sW + lT3, kWr, nl, kq, act, acc);
      gradient(1, D1);
      layerT<8, 8>(sW + lT2, kWr, nl, kq, act, acc);
      gradient(0, D0);
    }
  }
  if constexpr (BACK) {
    for (int o = 32; o > 0; o >>= 1) sq += __shfl_xor(sq, o, 64);
    if (lane == 0) red[tid >> 6] = sq;
    __syncthreads();
    if (tid == 0) {
      double t = red[0];
#pragma unroll
      for (int w = 1; w < BS / 64; ++w) t += red[w];
      partial[blockIdx.x] = t;
    }
  }
}

// Weight and bias gradients of all four layers over one slice of the batch: dW_l = dZ_l^T A_{l-1}, db_l = column sums
// of dZ_l, into slice blockIdx.y of part (kParams values, laid out as the parameters). blockIdx.x = one 64 x 64 tile of
// one product (kGradTiles of them): 4 wavefronts of 32 x 32. kRowsStep rows of both operands (64 columns each) are
// loaded at once (lanes along the columns, four rows per thread and step), rounded to BF16 and stored row-packed, so
// that an MFMA fragment (four rows of one column) is one 8-byte LDS read. Bound by the latency of those loads: 12 x 32
// workgroups for 8192 rows, two load rounds each, 12 us for
// 8192 rows (27 with every load guarded; 318 for the products and column sums of one launch per layer before).
constexpr int kGradTiles = 12;    // 128x128 (W3, W2): 4 each; 3x128 (W4), 128x14 (W1): 2 each
constexpr int kRowsStep  = 128;
constexpr int kGs = kRowsStep + 4;  // padded column (66 dwords)
__global__ __launch_bounds__(256) void mlpWeightGrad(const float* __restrict__ X, const float* __restrict__ A0,
                                                     const float* __restrict__ A1, const float* __restrict__ A2,
                                                     const float* __restrict__ D0, const float* __restrict__ D1,
                                                     const float* __restrict__ D2, const float* __restrict__ dY,
                                                     int64_t n, int64_t chunk, float* __restrict__ part) {
  __shared__ __align__(16) uint16_t As[64 * kGs], Bs[64 * kGs];
  __shared__ float sb[4][64];
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int tile = blockIdx.x;
  const float *D, *A;
  int M, N, i0, j0;
  int64_t oW, oB;
  if (tile < 4) {
    D = D2, A = A1, M = kHid, N = kHid, i0 = 64 * (tile >> 1), j0 = 64 * (tile & 1), oW = oW3, oB = oB3;
  } else if (tile < 8) {
    D = D1, A = A0, M = kHid, N = kHid, i0 = 64 * ((tile - 4) >> 1), j0 = 64 * (tile & 1), oW = oW2, oB = oB2;
  } else if (tile < 10) {
    D = dY, A = A2, M = kOut, N = kHid, i0 = 0, j0 = 64 * (tile & 1), oW = oW4, oB = oB4;
  } else {
    D = D0, A = X, M = kHid, N = kIn, i0 = 64 * (tile & 1), j0 = 0, oW = oW1, oB = oB1;
  }
  const int64_t k0 = (int64_t)blockIdx.y * chunk, k1 = k0 + chunk < n ? k0 + chunk : n;
  const bool ci = i0 + lane < M, cj = j0 + lane < N;
  f32x4 acc[2][2];
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b) acc[a][b] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int wm = w >> 1, wn = w & 1;
  float bsum = 0.f;
  for (int64_t kb = k0; kb < k1; kb += kRowsStep) {
    // wavefront w loads rows 4 (4 q + w) .. + 3 of column `lane` of both operands
    float va[kRowsStep / 16][4], vb[kRowsStep / 16][4];
    const float* d = D + (kb + 4 * w) * M + i0 + lane;
    const float* a = A + (kb + 4 * w) * N + j0 + lane;
    auto load = [&](auto guarded) {
#pragma unroll
      for (int q = 0; q < kRowsStep / 16; ++q)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const bool in = !decltype(guarded)::value || kb + 4 * w + 16 * q + r < k1;
          va[q][r]      = (!decltype(guarded)::value || (ci && in)) ? d[(16 * q + r) * M] : 0.f;
          vb[q][r]      = (!decltype(guarded)::value || (cj && in)) ? a[(16 * q + r) * N] : 0.f;
        }
    };
    if (tile < 8 && kb + kRowsStep <= k1)  // whole tiles of the 128x128 products
      load(std::false_type{});
    else
      load(std::true_type{});
    if (kb > k0) __syncthreads();  // the previous step's fragments have been read
#pragma unroll
    for (int q = 0; q < kRowsStep / 16; ++q) {
      *reinterpret_cast<bf16x4*>(&As[lane * kGs + 4 * (4 * q + w)]) = pack4(va[q][0], va[q][1], va[q][2], va[q][3]);
      *reinterpret_cast<bf16x4*>(&Bs[lane * kGs + 4 * (4 * q + w)]) = pack4(vb[q][0], vb[q][1], vb[q][2], vb[q][3]);
      bsum += (va[q][0] + va[q][1]) + (va[q][2] + va[q][3]);
    }
    __syncthreads();
#pragma unroll
    for (int s = 0; s < kRowsStep / 16; ++s) {
      bf16x4 a[2], b[2];
#pragma unroll
      for (int m = 0; m < 2; ++m) {
        a[m] = wfrag(&As[(32 * wm + 16 * m + (lane & 15)) * kGs + 16 * s + 4 * (lane >> 4)]);
        b[m] = wfrag(&Bs[(32 * wn + 16 * m + (lane & 15)) * kGs + 16 * s + 4 * (lane >> 4)]);
      }
#pragma unroll
      for (int m = 0; m < 2; ++m)
#pragma unroll
        for (int q = 0; q < 2; ++q) acc[m][q] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a[m], b[q], acc[m][q], 0, 0, 0);
    }
  }
  float* out = part + (int64_t)blockIdx.y * kParams;
#pragma unroll
  for (int m = 0; m < 2; ++m)
#pragma unroll
    for (int q = 0; q < 2; ++q)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int i = i0 + 32 * wm + 16 * m + 4 * (lane >> 4) + r, j = j0 + 32 * wn + 16 * q + (lane & 15);
        if (i < M && j < N) out[oW + (int64_t)i * N + j] = acc[m][q][r];
      }
  if (j0 == 0) {  // the tiles of the first columns also own the bias gradient of their rows
    sb[w][lane] = bsum;
    __syncthreads();
    if (w == 0 && ci) out[oB + i0 + lane] = ((sb[0][lane] + sb[1][lane]) + sb[2][lane]) + sb[3][lane];
  }
}

// g[i] = sum over the slices z = 0 .. nz-1 of part[z * kParams + i], in that order (the gradients do not depend on
// scheduling); ADAM: then one Adam step on the parameters
template <bool ADAM>
__global__ __launch_bounds__(256) void mlpFold(const float* __restrict__ part, int nz, float* __restrict__ g,
                                               float* __restrict__ p, float* __restrict__ m, float* __restrict__ v,
                                               float lr, float b1, float b2, float eps, float c1, float c2) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= kParams) return;
  float gi = 0.f;
#pragma unroll 8
  for (int z = 0; z < nz; ++z) gi += part[(int64_t)z * kParams + i];
  g[i] = gi;
  if constexpr (ADAM) {
    const float mi = b1 * m[i] + (1.f - b1) * gi;
    const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
    m[i]           = mi;
    v[i]           = vi;
    p[i] -= lr * (mi * c1) / (sqrtf(vi * c2) + eps);
  }
}

__global__ void fillF(float* __restrict__ p, int64_t n, float v) {
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) p[i] = v;
}

// BF16 copy of the network for the fused predictor, row-major output by input: W1 [128][16] (inputs past 14
// zero), W2 and W3 [128][kWs], W4 [16][kWs] (rows past the 3 outputs zero). The rows of 128 inputs are padded to
// kWs = 136 values (68 dwords), so the 16 rows one MFMA A fragment reads start on 16 different bank quadruples
// instead of all on bank 0; the whole copy (kWbN values, 78 KB) is staged into LDS as it lies. Within each group
// of 32 inputs 32 s .. 32 s + 31 the columns are stored in the order the 16x16x32 MFMA consumes them: lane group
// g (lanes 16 g .. 16 g + 15) takes slots 8 g .. 8 g + 7 = inputs 32 s + 4 g + (0..3) and 32 s + 16 + 4 g + (0..3).
constexpr int kWs = kHid + 8;
constexpr int oWb1 = 0, oWb2 = oWb1 + kHid * 16, oWb3 = oWb2 + kHid * kWs, oWb4 = oWb3 + kHid * kWs,
              kWbN = oWb4 + 16 * kWs;
static_assert(kWbN % 8 == 0, "staged in 16-byte pieces");

__global__ void packBf16Weights(const float* __restrict__ P, uint16_t* __restrict__ Wb) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= kWbN) return;
  float v = 0.f;
  if (i < oWb2) {
    const int j = i / 16, k = i % 16;
    v = k < kIn ? P[oW1 + j * kIn + k] : 0.f;
  } else {
    const int l = i < oWb3 ? 0 : i < oWb4 ? 1 : 2;
    const int o = i - (l == 0 ? oWb2 : l == 1 ? oWb3 : oWb4);
    const int j = o / kWs, c = o % kWs;
    if (c < kHid && (l < 2 || j < kOut)) {
      const int g = (c % 32) / 8, q = c % 8;
      const int k = c / 32 * 32 + (q < 4 ? 4 * g + q : 16 + 4 * g + q - 4);
      v           = P[(l == 0 ? oW2 : l == 1 ? oW3 : oW4) + j * kHid + k];
    }
  }
  Wb[i] = toBf16(v);
}

// eight consecutive BF16 values of a weight row in LDS (16-byte aligned): a 16x16x32 A fragment
__device__ inline bf16x8 wfrag8(const uint16_t* w) { return *reinterpret_cast<const bf16x8*>(w); }
// the 16x16x32 B fragment of K step s: this lane's outputs of tiles 2 s and 2 s + 1
__device__ inline bf16x8 actPair(bf16x4 lo, bf16x4 hi) {
  return __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
}

// The in-solver prediction in one launch: the per-node features (file header; velocities from the two previous
// increments), the three SiLU layers, the output layer and u <- u + dlam (v_n + 0.1 y) on free DOFs, with the
// activations kept in registers. A wavefront takes 16 nodes at a time and computes each layer transposed,
// out^T (128 x 16) = W (128 x 128) act^T, with W as the MFMA A operand (from LDS) and the activations as the B
// operand. Lane (n, kq) = (lane & 15, lane >> 4) holds node n's outputs 16 t + 4 kq + r of output tile t (C
// fragment). Layer 1 (K = 16) runs on v_mfma_f32_16x16x16_bf16; layers 2-4 on v_mfma_f32_16x16x32_bf16, whose K
// step s takes from this lane exactly its outputs of tiles 2 s and 2 s + 1 (the weight columns are stored in
// that order): no data moves between lanes from layer to layer. The 8 output tiles of a layer are independent
// accumulation chains, interleaved per K step. Same operand rounding (BF16, round to nearest even), FP32
// accumulation, bias and SiLU as mlpRows (within a 32-input step the summation order differs).
__global__ __launch_bounds__(256) void mlpPredictFused(const uint16_t* __restrict__ Wb, const float* __restrict__ P,
                                                       const double* __restrict__ X, const double* __restrict__ duN,
                                                       const double* __restrict__ duN1, int64_t nn, double invL,
                                                       double t0, double t1, double t2, double lamNext, double dlam,
                                                       double dlamPrev, double dlamPrev2, double* __restrict__ u,
                                                       const uint8_t* __restrict__ fixed) {
  __shared__ __align__(16) uint16_t sW[kWbN];  // 78 KB
  __shared__ float sB[3 * kHid + 16];
  for (int i = threadIdx.x; i < kWbN / 8; i += 256)
    reinterpret_cast<uint4*>(sW)[i] = reinterpret_cast<const uint4*>(Wb)[i];
  for (int i = threadIdx.x; i < 3 * kHid + 16; i += 256) {
    float v = 0.f;
    if (i < kHid) v = P[oB1 + i];
    else if (i < 2 * kHid) v = P[oB2 + i - kHid];
    else if (i < 3 * kHid) v = P[oB3 + i - 2 * kHid];
    else if (i - 3 * kHid < kOut) v = P[oB4 + i - 3 * kHid];
    sB[i] = v;
  }
  __syncthreads();
  const int lane = threadIdx.x & 63, n = lane & 15, kq = lane >> 4;
  const int64_t nblk = (nn + 15) / 16;
  for (int64_t blk = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6); blk < nblk; blk += (int64_t)gridDim.x * 4) {
    const int64_t v = blk * 16 + n;
    const bool valid = v < nn;
    // input fragment: features 4 kq .. 4 kq + 3 of node v (as predictorFeatures)
    float f[4] = {0.f, 0.f, 0.f, 0.f};
    if (valid) {
      if (kq == 0) {
        f[0] = (float)(X[v * 3] * invL);
        f[1] = (float)(X[v * 3 + 1] * invL);
        f[2] = (float)(X[v * 3 + 2] * invL);
        f[3] = (float)(t0 * kTracScale);
      } else if (kq == 1) {
        f[0] = (float)(t1 * kTracScale);
        f[1] = (float)(t2 * kTracScale);
        f[2] = (float)lamNext;
        f[3] = (float)(dlam * kDlamScale);
      } else if (kq == 2) {
        for (int k = 0; k < 3; ++k) f[k] = dlamPrev > 0 ? (float)(duN[v * 3 + k] / dlamPrev / kVelScale) : 0.f;
        f[3] = dlamPrev2 > 0 ? (float)(duN1[v * 3] / dlamPrev2 / kVelScale) : 0.f;
      } else {
        for (int k = 0; k < 2; ++k) f[k] = dlamPrev2 > 0 ? (float)(duN1[v * 3 + 1 + k] / dlamPrev2 / kVelScale) : 0.f;
      }
    }
    bf16x4 act[8];
    act[0] = bf16x4{(short)toBf16(f[0]), (short)toBf16(f[1]), (short)toBf16(f[2]), (short)toBf16(f[3])};
    f32x4 acc[8];
    // layer 1: K = 16 (one step)
#pragma unroll
    for (int t = 0; t < 8; ++t) {
      const bf16x4 a = wfrag(sW + oWb1 + (16 * t + n) * 16 + 4 * kq);
      acc[t] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, act[0], f32x4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
    }
    // bias, SiLU, BF16: the next layer's B fragments
    auto activate = [&](const float* bias) {
#pragma unroll
      for (int t = 0; t < 8; ++t) {
        short q[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) q[r] = (short)toBf16(silu(acc[t][r] + bias[16 * t + 4 * kq + r]));
        act[t] = bf16x4{q[0], q[1], q[2], q[3]};
      }
    };
    activate(sB);
    // layers 2 and 3: 4 K steps of 32 x 8 independent output tiles
#pragma unroll
    for (int l = 0; l < 2; ++l) {
      const uint16_t* W = sW + (l == 0 ? oWb2 : oWb3);
#pragma unroll
      for (int t = 0; t < 8; ++t) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) {
        const bf16x8 b = actPair(act[2 * ks], act[2 * ks + 1]);
#pragma unroll
        for (int t = 0; t < 8; ++t)
          acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wfrag8(W + (16 * t + n) * kWs + 32 * ks + 8 * kq), b,
                                                           acc[t], 0, 0, 0);
      }
      activate(sB + (l + 1) * kHid);
    }
    // output layer: one tile (rows 0..2 of 16 used), 4 K steps of 32
    f32x4 y = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int ks = 0; ks < 4; ++ks)
      y = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wfrag8(sW + oWb4 + n * kWs + 32 * ks + 8 * kq),
                                                  actPair(act[2 * ks], act[2 * ks + 1]), y, 0, 0, 0);
    // lanes kq = 0 hold outputs 0..3 of node n: u <- u + dlam (v_n + 0.1 y) on free DOFs
    if (valid && kq == 0) {
#pragma unroll
      for (int k = 0; k < kOut; ++k) {
        const int64_t i = v * 3 + k;
        if (fixed[i]) continue;
        const float yk   = y[k] + sB[3 * kHid + k];
        const double vn  = dlamPrev > 0 ? duN[i] / dlamPrev : 0.0;
        u[i] += dlam * (vn + kVelScale * (double)yk);
      }
    }
  }
}

inline unsigned g1(int64_t n) { return (unsigned)std::min<int64_t>(std::max<int64_t>((n + 255) / 256, 1), 4096); }

}  // namespace

// ------------------------------------------------------------------------------------------------
// MLP context shared by the training entry points and the in-solver predictor
// ------------------------------------------------------------------------------------------------
struct Mlp {
  hipStream_t s = nullptr;
  DevBuf<float> P, G, Mo, Vo;      // params (fp32 master), grads, Adam moments
  DevBuf<float> Aa[3], dZ[3], Y, dY, Xin, Tin;
  DevBuf<float> Gpart;  // per-slice partial gradients, folded in a fixed order
  DevBuf<uint16_t> Wb;  // BF16 weights of the fused predictor (packed when the parameters are set)
  DevBuf<double> partial;
  double* hred = nullptr;
  int64_t step = 0;
  std::string err;

  // Buffers of a batch of n rows, for the pass that uses them. Each one checks its own size, so one that could not be
  // had is asked for again by the next call.
  void ensureForward(int64_t n, bool host) {
    Y.ensure(n * kOut);
    if (host) Xin.ensure(n * kIn);
  }
  void ensureTraining(int64_t n, bool host) {
    for (int l = 0; l < 3; ++l) {
      Aa[l].ensure(n * kHid);
      dZ[l].ensure(n * kHid);
    }
    dY.ensure(n * kOut);
    if (host) {
      Xin.ensure(n * kIn);
      Tin.ensure(n * kOut);
    }
  }

  // y (n x 3) = the network on x (n x 14); nothing is kept and nothing is allocated
  void forward(const float* x, int64_t n, float* y) {
    const unsigned grid = (unsigned)std::min<int64_t>((n + 63) / 64, 512);  // 2 workgroups of 80 KB LDS per CU
    hipLaunchKernelGGL((mlpRows<false>), dim3(grid), dim3(256), 0, s, P.p, x, nullptr, n, 0.f, y, nullptr, nullptr,
                       nullptr, nullptr, nullptr, nullptr, nullptr, nullptr);
  }

  // mean-squared-error loss and its gradient w.r.t. all parameters (into G); train: then one Adam step
  double lossGrad(const float* x, const float* t, int64_t n, bool train = false, float lr = 0.f) {
    const int nb = (int)std::min<int64_t>((n + 63) / 64, 256);  // one workgroup of 156 KB LDS per CU
    partial.ensure(256);
    hipLaunchKernelGGL((mlpRows<true>), dim3(nb), dim3(512), 0, s, P.p, x, t, n, (float)(1.0 / (double)(n * kOut)),
                       nullptr, Aa[0].p, Aa[1].p, Aa[2].p, dZ[0].p, dZ[1].p, dZ[2].p, dY.p, partial.p);
    // slices of 256 rows, at most 256 of them
    const int64_t split = std::max<int64_t>(1, std::min<int64_t>(n / 256, 256));
    const int64_t chunk = split > 1 ? ((n + split - 1) / split + 15) / 16 * 16 : n;
    const int nz        = (int)((n + chunk - 1) / chunk);
    Gpart.ensure((size_t)nz * kParams);
    hipLaunchKernelGGL(mlpWeightGrad, dim3(kGradTiles, nz), dim3(256), 0, s, x, Aa[0].p, Aa[1].p, Aa[2].p, dZ[0].p,
                       dZ[1].p, dZ[2].p, dY.p, n, chunk, Gpart.p);
    const dim3 gf((unsigned)((kParams + 255) / 256));
    if (train) {
      const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
      ++step;
      const float c1 = 1.f / (1.f - std::pow(b1, (float)step)), c2 = 1.f / (1.f - std::pow(b2, (float)step));
      hipLaunchKernelGGL((mlpFold<true>), gf, dim3(256), 0, s, Gpart.p, nz, G.p, P.p, Mo.p, Vo.p, lr, b1, b2, eps, c1,
                         c2);
    } else {
      hipLaunchKernelGGL((mlpFold<false>), gf, dim3(256), 0, s, Gpart.p, nz, G.p, nullptr, nullptr, nullptr, 0.f, 0.f,
                         0.f, 0.f, 0.f, 0.f);
    }
    IK_HIP(hipMemcpyAsync(hred, partial.p, nb * sizeof(double), hipMemcpyDeviceToHost, s));
    IK_HIP(hipStreamSynchronize(s));
    double sum = 0.0;
    for (int i = 0; i < nb; ++i) sum += hred[i];
    return sum / (double)(n * kOut);
  }
};

Mlp* mlpCreate(hipStream_t s) {
  auto* m = new Mlp;
  m->s    = s;
  m->P.ensure(kParams);
  m->G.ensure(kParams);
  m->Mo.ensure(kParams);
  m->Vo.ensure(kParams);
  hipLaunchKernelGGL(fillF, dim3(g1(kParams)), dim3(256), 0, s, m->Mo.p, kParams, 0.f);
  hipLaunchKernelGGL(fillF, dim3(g1(kParams)), dim3(256), 0, s, m->Vo.p, kParams, 0.f);
  IK_HIP(hipHostMalloc((void**)&m->hred, 256 * sizeof(double), hipHostMallocDefault));
  return m;
}

void mlpDestroy(Mlp* m) {
  if (!m) return;
  if (m->s) (void)hipStreamSynchronize(m->s);
  if (m->hred) (void)hipHostFree(m->hred);
  delete m;
}

int64_t mlpNumParams() { return kParams; }

void mlpSetParams(Mlp* m, const float* p, int where, hipStream_t s) {
  IK_HIP(hipMemcpyAsync(m->P.p, p, kParams * sizeof(float),
                        where == IK_DEVICE ? hipMemcpyDeviceToDevice : hipMemcpyHostToDevice, s));
  m->Wb.ensure(kWbN);
  hipLaunchKernelGGL(packBf16Weights, dim3((kWbN + 255) / 256), dim3(256), 0, s, m->P.p, m->Wb.p);
  IK_HIP(hipStreamSynchronize(s));
}

void mlpGetParams(Mlp* m, float* p, int where, hipStream_t s) {
  IK_HIP(hipMemcpyAsync(p, m->P.p, kParams * sizeof(float),
                        where == IK_DEVICE ? hipMemcpyDeviceToDevice : hipMemcpyDeviceToHost, s));
  IK_HIP(hipStreamSynchronize(s));
}

// in-solver prediction: u (device) <- MLP prediction for lamNext from the two previous increments
void mlpPredict(ik_handle* h, const double* duN, const double* duN1, double lamNext, double dlam, double dlamPrev,
                double dlamPrev2) {
  require(h->mlp != nullptr && h->mlpLoaded, IK_EINVAL, "MLP predictor selected but no parameters set");
  Mlp* m = h->mlp;
  m->s   = h->stream;
  ScopedKernelTimer t(h, KMLP);
  // one fused launch; 2 workgroups of 80 KB LDS per CU, each wavefront looping over blocks of 16 nodes
  const int64_t blocks = (h->nn + 63) / 64;
  const unsigned grid  = (unsigned)std::max<int64_t>(1, std::min<int64_t>(blocks, 512));
  hipLaunchKernelGGL(mlpPredictFused, dim3(grid), dim3(256), 0, h->stream, m->Wb.p, m->P.p, h->X.p, duN, duN1, h->nn,
                     1.0 / h->mlpCharLen, h->mlpTraction[0], h->mlpTraction[1], h->mlpTraction[2], lamNext, dlam,
                     dlamPrev, dlamPrev2, h->u.p, h->fixed.p);
}

}  // namespace ik

// ------------------------------------------------------------------------------------------------
// C ABI of the training context
// ------------------------------------------------------------------------------------------------
struct ik_mlp {
  ik::Mlp* m = nullptr;
  hipStream_t s = nullptr;
  int device = 0;            // the device current at ik_mlp_create: the context's stream and memory live there
  std::string err;
};

// Scratch of the allocation-free forward (ik_mlp_forward_noalloc): the outputs of a call whose y overlaps its x (the
// kernel's workgroups read x while others write y), IK_MLP_NOALLOC_MAX_ROWS x 3 FP32, one copy per device held until
// the process ends. Host code uses only the address hipGetSymbolAddress returns for the device (the array's name on the
// host is not a device address), resolved once per device at ik_mlp_create with that device current.
static __device__ __align__(256) float scratch[IK_MLP_NOALLOC_MAX_ROWS * ik::kOut];

namespace {
constexpr int kMaxDevices = 64;
std::mutex g_scratchMutex;
float* g_scratchPtr[kMaxDevices] = {};

float* resolveScratch(int device) {
  ik::require(device >= 0 && device < kMaxDevices, IK_EINVAL, "device index out of range");
  std::lock_guard<std::mutex> lock(g_scratchMutex);
  if (!g_scratchPtr[device]) {
    void* ptr = nullptr;
    IK_HIP(hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)));
    g_scratchPtr[device] = static_cast<float*>(ptr);
  }
  return g_scratchPtr[device];
}
}  // namespace

namespace {
template <class F>
int mguard(ik_mlp* m, F&& f) {
  try {
    f();
    if (m) m->err.clear();
    return IK_OK;
  } catch (const ik::Error& e) {
    if (m) m->err = e.msg;
    return e.code;
  } catch (const std::exception& e) {
    if (m) m->err = e.what();
    return IK_EINVAL;
  }
}
// He-uniform weights U(-sqrt(6/fan_in), +) from SplitMix64, zero biases, last layer scaled by 0.1
void initParams(std::vector<float>& p, uint64_t seed) {
  using namespace ik;
  p.assign(kParams, 0.f);
  uint64_t st = seed;
  auto uni = [&]() {
    uint64_t z = (st += 0x9E3779B97F4A7C15ULL);
    z          = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ULL;
    z          = (z ^ (z >> 27)) * 0x94D049BB133111EBULL;
    z ^= z >> 31;
    return (double)(z >> 11) * (1.0 / 9007199254740992.0);
  };
  auto fill = [&](int64_t off, int64_t count, int fanIn, double scale) {
    const double b = std::sqrt(6.0 / fanIn) * scale;
    for (int64_t i = 0; i < count; ++i) p[off + i] = (float)((2.0 * uni() - 1.0) * b);
  };
  fill(oW1, kHid * kIn, kIn, 1.0);
  fill(oW2, kHid * kHid, kHid, 1.0);
  fill(oW3, kHid * kHid, kHid, 1.0);
  fill(oW4, kOut * kHid, kHid, 0.1);
}
}  // namespace

extern "C" {

int ik_mlp_create(ik_mlp** out, uint64_t seed) {
  if (!out) return IK_EINVAL;
  auto* m = new ik_mlp;
  *out    = m;
  return mguard(m, [&] {
    IK_HIP(hipGetDevice(&m->device));
    (void)resolveScratch(m->device);  // the device's scratch address for ik_mlp_forward_noalloc
    IK_HIP(hipStreamCreateWithFlags(&m->s, hipStreamNonBlocking));
    m->m = ik::mlpCreate(m->s);
    std::vector<float> p;
    initParams(p, seed);
    IK_HIP(hipMemcpyAsync(m->m->P.p, p.data(), p.size() * sizeof(float), hipMemcpyHostToDevice, m->s));
    IK_HIP(hipStreamSynchronize(m->s));
  });
}

void ik_mlp_destroy(ik_mlp* m) {
  if (!m) return;
  ik::mlpDestroy(m->m);
  if (m->s) (void)hipStreamDestroy(m->s);
  delete m;
}

const char* ik_mlp_last_error(const ik_mlp* m) { return m ? m->err.c_str() : "null context"; }

int ik_mlp_params(ik_mlp* m, float* out, int where) {
  return mguard(m, [&] {
    IK_HIP(hipMemcpyAsync(out, m->m->P.p, ik::kParams * sizeof(float),
                          where == IK_DEVICE ? hipMemcpyDeviceToDevice : hipMemcpyDeviceToHost, m->s));
    IK_HIP(hipStreamSynchronize(m->s));
  });
}

int ik_mlp_load(ik_mlp* m, const float* p, int where) {
  return mguard(m, [&] {
    IK_HIP(hipMemcpyAsync(m->m->P.p, p, ik::kParams * sizeof(float),
                          where == IK_DEVICE ? hipMemcpyDeviceToDevice : hipMemcpyHostToDevice, m->s));
    IK_HIP(hipStreamSynchronize(m->s));
    m->m->step = 0;
  });
}

int ik_mlp_forward(ik_mlp* m, const float* x, int64_t n, float* y, int where) {
  return mguard(m, [&] {
    ik::require(n > 0, IK_EINVAL, "empty batch");
    m->m->ensureForward(n, where != IK_DEVICE);
    const float* xd = x;
    if (where != IK_DEVICE) {
      IK_HIP(hipMemcpyAsync(m->m->Xin.p, x, n * ik::kIn * sizeof(float), hipMemcpyHostToDevice, m->s));
      xd = m->m->Xin.p;
    }
    m->m->forward(xd, n, m->m->Y.p);
    IK_HIP(hipMemcpyAsync(y, m->m->Y.p, n * ik::kOut * sizeof(float),
                          where == IK_DEVICE ? hipMemcpyDeviceToDevice : hipMemcpyDeviceToHost, m->s));
    IK_HIP(hipStreamSynchronize(m->s));
  });
}

int ik_mlp_forward_noalloc(ik_mlp* m, const float* x, int64_t n, float* y) {
  return mguard(m, [&] {
    ik::require(x != nullptr && y != nullptr, IK_EINVAL, "null argument");
    ik::require(n > 0 && n <= IK_MLP_NOALLOC_MAX_ROWS, IK_EINVAL,
                "ik_mlp_forward_noalloc: the batch must have 1 to IK_MLP_NOALLOC_MAX_ROWS (8192) rows");
    float* s0 = g_scratchPtr[m->device];  // resolved at ik_mlp_create; never the array's host-side name
    ik::require(s0 != nullptr, IK_EINVAL, "ik_mlp_forward_noalloc: scratch not resolved for this device");
    const uintptr_t x0 = (uintptr_t)x, y0 = (uintptr_t)y;
    const bool overlap = y0 < x0 + n * ik::kIn * sizeof(float) && x0 < y0 + n * ik::kOut * sizeof(float);
    m->m->s            = m->s;
    m->m->forward(x, n, overlap ? s0 : y);
    if (overlap) IK_HIP(hipMemcpyAsync(y, s0, n * ik::kOut * sizeof(float), hipMemcpyDeviceToDevice, m->s));
    IK_HIP(hipStreamSynchronize(m->s));
  });
}

int ik_mlp_loss_grad(ik_mlp* m, const float* x, const float* t, int64_t n, double* loss, float* grad, int where) {
  return mguard(m, [&] {
    ik::require(n > 0, IK_EINVAL, "empty batch");
    m->m->ensureTraining(n, where != IK_DEVICE);
    const float *xd = x, *td = t;
    if (where != IK_DEVICE) {
      IK_HIP(hipMemcpyAsync(m->m->Xin.p, x, n * ik::kIn * sizeof(float), hipMemcpyHostToDevice, m->s));
      IK_HIP(hipMemcpyAsync(m->m->Tin.p, t, n * ik::kOut * sizeof(float), hipMemcpyHostToDevice, m->s));
      xd = m->m->Xin.p;
      td = m->m->Tin.p;
    }
    const double l = m->m->lossGrad(xd, td, n);
    if (loss) *loss = l;
    if (grad) {
      IK_HIP(hipMemcpyAsync(grad, m->m->G.p, ik::kParams * sizeof(float),
                            where == IK_DEVICE ? hipMemcpyDeviceToDevice : hipMemcpyDeviceToHost, m->s));
      IK_HIP(hipStreamSynchronize(m->s));
    }
  });
}

int ik_mlp_train_step(ik_mlp* m, const float* x, const float* t, int64_t n, float lr, double* loss, int where) {
  return mguard(m, [&] {
    ik::require(n > 0, IK_EINVAL, "empty batch");
    m->m->ensureTraining(n, where != IK_DEVICE);
    const float *xd = x, *td = t;
    if (where != IK_DEVICE) {
      IK_HIP(hipMemcpyAsync(m->m->Xin.p, x, n * ik::kIn * sizeof(float), hipMemcpyHostToDevice, m->s));
      IK_HIP(hipMemcpyAsync(m->m->Tin.p, t, n * ik::kOut * sizeof(float), hipMemcpyHostToDevice, m->s));
      xd = m->m->Xin.p;
      td = m->m->Tin.p;
    }
    const double l = m->m->lossGrad(xd, td, n, true, lr);
    if (loss) *loss = l;
  });
}

}  // extern "C"

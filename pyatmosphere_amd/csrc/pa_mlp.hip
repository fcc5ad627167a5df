// Kernels of the transmittance-PDT surrogate: a small MLP trained and evaluated
// on the device.  Training runs in float32 (float32 MFMA products, exact enough
// for gradient checks against a float64 host MLP); inference GEMMs run on bf16 MFMA with float32 accumulation and fused
// bias + activation.  Activation: SiLU, z * sigmoid(z).  Output head: NB
// logits (softmax PDT over NB transmittance bins) and one log-variance.
#include "pa_internal.h"

namespace pa {

typedef __bf16 b8 __attribute__((ext_vector_type(8)));
typedef float f4v __attribute__((ext_vector_type(4)));
typedef unsigned short us8 __attribute__((ext_vector_type(8)));

// ------------------------------------------------------------------ fp32 GEMM
// C[M][N] = op(A) op(B), row-major, op = transpose when t* is set: op(A) is M x K
// (A is M x K, or K x M when TA), op(B) is K x N (B is K x N, or N x K when TB).
//
// The training shapes (1024 x 384 x 384 and the like) are small: what bounds
// them is latency, not the 2 GFLOP of a step (13 us at the float32 matrix
// rate).  One block owns one 32 x 32 tile of C and its WK waves split K, so a
// 384-deep product is 12 loads deep per wave and a 384 x 384 weight gradient
// still gives 144 blocks of 16 waves; the waves' partial tiles are added in LDS
// in wave order (deterministic).  Operands go from L2 straight to registers
// on v_mfma_f32_32x32x2f32 (float32 products and sums): lane l supplies row
// (column) l % 32 at k = k0 + 4 (l / 32) + i for i = 0..3, so an operand whose
// K is contiguous is read as one float4 per lane and 8 k (VA / VB), and one
// whose rows are contiguous as four coalesced dwords.  Rows past M and columns
// past N repeat the last one (their results are not stored); k past the end
// is zero in both operands.
// Measured, a 1024-pair step of the 384-wide network (loss, gradients, Adam):
// 1856 us with 64 x 64 LDS tiles on the vector units (94 us a product, 36 to 96
// blocks), serial column sums for db (194 us) and a launch per pass and tensor;
// 91 us with these kernels (10-12 us a product, 20 us for all weight gradients;
// 8 waves a tile or other depths of loads in flight are 8 to 25% slower).
typedef float f16v __attribute__((ext_vector_type(16)));
constexpr int GT = 32;             // C tile
constexpr int GU = 4;              // groups of 8 k in flight per wave

template <bool T, bool VEC>
__device__ __forceinline__ void gemm_load(float (&x)[4], const float* __restrict__ P, int ld, int row, int k, int kend) {
  // T: element (row, k) at P[k ld + row], else P[row ld + k]
  if constexpr (!T && VEC) {
    const int kk = min(k, kend - 4);
    const f4v v = *reinterpret_cast<const f4v*>(P + (size_t)row * ld + kk);
#pragma unroll
    for (int i = 0; i < 4; ++i) x[i] = k < kend ? v[i] : 0.f;
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int kk = min(k + i, kend - 1);
      const float v = T ? P[(size_t)kk * ld + row] : P[(size_t)row * ld + kk];
      x[i] = k + i < kend ? v : 0.f;
    }
  }
}

// The sum of the tile at (m0, n0) over K into red[0 .. WK) (32 x 32 partial
// tiles, row stride 33).  With SUMA, rs[wave][row] receives the wave's sums of
// op(A)'s rows over K.  Ends with a barrier.
template <int WK, bool TA, bool TB, bool VA, bool VB, bool SUMA>
__device__ __forceinline__ void gemm_tile32(int M, int N, int K, int m0, int n0, const float* __restrict__ A, int lda,
                                            const float* __restrict__ B, int ldb, float* red, float* rs) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, r = lane & 31, h = lane >> 5;
  const int row = min(m0 + r, M - 1), col = min(n0 + r, N - 1);
  const int per = ((K + 7) / 8 + WK - 1) / WK * 8;       // k per wave, a multiple of 8
  const int kb = wave * per, ke = min(K, kb + per);
  f16v acc;
#pragma unroll
  for (int i = 0; i < 16; ++i) acc[i] = 0.f;
  float sum = 0.f;
  if (kb < ke) {
    float a[GU][4], b[GU][4];
    auto fetch = [&](int k0) {
#pragma unroll
      for (int u = 0; u < GU; ++u) {
        gemm_load<TA, VA>(a[u], A, lda, row, k0 + 8 * u + 4 * h, ke);
        gemm_load<!TB, VB>(b[u], B, ldb, col, k0 + 8 * u + 4 * h, ke);
      }
    };
    fetch(kb);
    for (int k0 = kb; k0 < ke; k0 += 8 * GU) {
      float ca[GU][4], cb[GU][4];
#pragma unroll
      for (int u = 0; u < GU; ++u)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          ca[u][i] = a[u][i];
          cb[u][i] = b[u][i];
        }
      if (k0 + 8 * GU < ke) fetch(k0 + 8 * GU);
#pragma unroll
      for (int u = 0; u < GU; ++u)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          acc = __builtin_amdgcn_mfma_f32_32x32x2f32(ca[u][i], cb[u][i], acc, 0, 0, 0);
          if constexpr (SUMA) sum += ca[u][i];
        }
    }
  }
#pragma unroll
  for (int v = 0; v < 16; ++v) red[wave * (GT * 33) + (8 * (v / 4) + 4 * h + v % 4) * 33 + r] = acc[v];
  if constexpr (SUMA) {
    sum += __shfl_xor(sum, 32, 64);
    if (h == 0) rs[wave * GT + r] = sum;
  }
  __syncthreads();
}

template <int WK>
__device__ __forceinline__ float gemm_sum(const float* red, int r, int c) {
  float s = 0.f;
#pragma unroll
  for (int w = 0; w < WK; ++w) s += red[w * (GT * 33) + r * 33 + c];
  return s;
}

constexpr int kGemmWaves = 4;
template <bool TA, bool TB, bool VA, bool VB>
__global__ void __launch_bounds__(64 * kGemmWaves)
k_gemm_f32(int M, int N, int K, const float* __restrict__ A, int lda, const float* __restrict__ B, int ldb,
           float* __restrict__ C, int ldc, float alpha, float beta) {
  __shared__ float red[kGemmWaves * GT * 33];
  const int m0 = blockIdx.y * GT, n0 = blockIdx.x * GT;
  gemm_tile32<kGemmWaves, TA, TB, VA, VB, false>(M, N, K, m0, n0, A, lda, B, ldb, red, nullptr);
  for (int e = threadIdx.x; e < GT * GT; e += 64 * kGemmWaves) {
    const int r = e / GT, c = e % GT;
    if (m0 + r >= M || n0 + c >= N) continue;
    float* o = C + (size_t)(m0 + r) * ldc + n0 + c;
    *o = alpha * gemm_sum<kGemmWaves>(red, r, c) + (beta != 0.f ? beta * *o : 0.f);
  }
}

// ------------------------------------------------------------------ elementwise
__device__ __forceinline__ float sigm(float z) { return 1.f / (1.f + expf(-z)); }

// Z += bias (row broadcast); Y = act(Z) when act != 0 else Y = Z.
__global__ void k_bias_act(int M, int N, float* __restrict__ Z, const float* __restrict__ bias,
                           float* __restrict__ Y, int act) {
  const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= (size_t)M * N) return;
  const float z = Z[i] + bias[i % N];
  Z[i] = z;
  Y[i] = act ? z * sigm(z) : z;
}

// dZ = dY * act'(Z)
__global__ void k_act_backward(int M, int N, const float* __restrict__ Z, const float* __restrict__ dY,
                               float* __restrict__ dZ) {
  const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= (size_t)M * N) return;
  const float z = Z[i], s = sigm(z);
  dZ[i] = dY[i] * s * (1.f + z * (1.f - s));
}

// db[n] = sum_m dZ[m][n] (fixed order per column)
__global__ void k_bias_grad(int M, int N, const float* __restrict__ dZ, float* __restrict__ db) {
  const int n = blockIdx.x * 256 + threadIdx.x;
  if (n >= N) return;
  float s = 0.f;
  for (int m = 0; m < M; ++m) s += dZ[(size_t)m * N + n];
  db[n] = s;
}

// Z = X W^T + bias and (Y non-null) Y = SiLU(Z) of one layer, X M x K, W N x K:
// the bias and the activation ride on the product's epilogue instead of two
// more passes over the M x N values.
template <bool VEC>
__global__ void __launch_bounds__(64 * kGemmWaves)
k_layer_forward(int M, int N, int K, const float* __restrict__ X, const float* __restrict__ W,
                const float* __restrict__ bias, float* __restrict__ Z, float* __restrict__ Y) {
  __shared__ float red[kGemmWaves * GT * 33];
  const int m0 = blockIdx.y * GT, n0 = blockIdx.x * GT;
  gemm_tile32<kGemmWaves, false, true, VEC, VEC, false>(M, N, K, m0, n0, X, K, W, K, red, nullptr);
  for (int e = threadIdx.x; e < GT * GT; e += 64 * kGemmWaves) {
    const int r = e / GT, c = e % GT;
    if (m0 + r >= M || n0 + c >= N) continue;
    const float z = gemm_sum<kGemmWaves>(red, r, c) + bias[n0 + c];
    const size_t o = (size_t)(m0 + r) * N + n0 + c;
    Z[o] = z;
    if (Y) Y[o] = z * sigm(z);
  }
}

// dZ = (D W) * SiLU'(Z) of the layer below: D M x K (this layer's dZ), W K x N,
// Z the lower layer's M x N pre-activations.
template <bool VEC>
__global__ void __launch_bounds__(64 * kGemmWaves)
k_layer_backward(int M, int N, int K, const float* __restrict__ D, const float* __restrict__ W,
                 const float* __restrict__ Z, float* __restrict__ dZ) {
  __shared__ float red[kGemmWaves * GT * 33];
  const int m0 = blockIdx.y * GT, n0 = blockIdx.x * GT;
  gemm_tile32<kGemmWaves, false, false, VEC, false, false>(M, N, K, m0, n0, D, K, W, N, red, nullptr);
  for (int e = threadIdx.x; e < GT * GT; e += 64 * kGemmWaves) {
    const int r = e / GT, c = e % GT;
    if (m0 + r >= M || n0 + c >= N) continue;
    const size_t o = (size_t)(m0 + r) * N + n0 + c;
    const float z = Z[o], s = sigm(z);
    dZ[o] = gemm_sum<kGemmWaves>(red, r, c) * s * (1.f + z * (1.f - s));
  }
}

// Every layer's dW = D^T H (fo x fi over K = M rows) and db = column sums of D
// in one launch, and the mean of the rows' losses in a block of its own (the
// last, mean non-null): the products do not depend on each other, and together they
// fill the chip (336 tiles of 16 waves for the 16-384-384-384-65 network).
constexpr int kGradLayers = 8;      // layers per launch
constexpr int kGradWaves = 16;
struct GradLayers {
  const float* d[kGradLayers];
  const float* h[kGradLayers];
  float* dw[kGradLayers];
  float* db[kGradLayers];
  int fo[kGradLayers], fi[kGradLayers], first[kGradLayers + 1];   // first: tiles before this layer
};
__global__ void __launch_bounds__(64 * kGradWaves)
k_weight_grads(int layers, int M, GradLayers g, const float* __restrict__ loss, float* __restrict__ mean) {
  __shared__ float red[kGradWaves * GT * 33];
  __shared__ float rs[kGradWaves * GT];
  if ((int)blockIdx.x == g.first[layers]) {
    float s = 0.f;
    for (int i = threadIdx.x; i < M; i += 64 * kGradWaves) s += loss[i];
    red[threadIdx.x] = s;
    for (int o = 32 * kGradWaves; o > 0; o >>= 1) {
      __syncthreads();
      if ((int)threadIdx.x < o) red[threadIdx.x] += red[threadIdx.x + o];
    }
    if (threadIdx.x == 0) *mean = red[0] / M;
    return;
  }
  int i = 0;
  while (i + 1 < layers && (int)blockIdx.x >= g.first[i + 1]) ++i;
  const int fo = g.fo[i], fi = g.fi[i], nx = (fi + GT - 1) / GT, tile = blockIdx.x - g.first[i];
  const int m0 = tile / nx * GT, n0 = tile % nx * GT;
  gemm_tile32<kGradWaves, true, false, false, false, true>(fo, fi, M, m0, n0, g.d[i], fo, g.h[i], fi, red, rs);
  const int r = threadIdx.x / GT, c = threadIdx.x % GT;
  if (m0 + r < fo && n0 + c < fi) g.dw[i][(size_t)(m0 + r) * fi + n0 + c] = gemm_sum<kGradWaves>(red, r, c);
  if (n0 == 0 && threadIdx.x < GT && m0 + (int)threadIdx.x < fo) {
    float s = 0.f;
#pragma unroll
    for (int w = 0; w < kGradWaves; ++w) s += rs[w * GT + threadIdx.x];
    g.db[i][m0 + threadIdx.x] = s;
  }
}
static_assert(GT * GT == 64 * kGradWaves, "one thread per element of the tile");

// Head: row m of out holds NB logits and one log-variance.  Loss per row:
//   -sum_j t_j log p_j + wc sum_j (P_j - T_j)^2 + wv (lv - tv)^2
// with p = softmax(logits), P and T the cumulative sums of p and t (a ranked
// probability score, the squared distance between the CDFs the KS metric
// compares).  Gradient (divided by M): with g_i = 2 wc sum_{j >= i} (P_j - T_j),
// dL/dl_i = p_i - t_i + p_i (g_i - sum_k p_k g_k); dL/dlv = 2 wv (lv - tv).
// One wave per row; NB <= 64 (one bin per lane).
__global__ void __launch_bounds__(64)
k_head_loss(int M, int NB, const float* __restrict__ out, const float* __restrict__ target,
            const float* __restrict__ tvar, float wv, float wc, float* __restrict__ loss, float* __restrict__ dout) {
  const int m = blockIdx.x;
  const int j = threadIdx.x;
  const bool on = j < NB;
  const float* l = out + (size_t)m * (NB + 1);
  const float lj = on ? l[j] : -3.4e38f;
  float mx = lj;
  for (int o = 32; o > 0; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o, 64));
  const float ej = on ? expf(lj - mx) : 0.f;
  float se = ej;
  for (int o = 32; o > 0; o >>= 1) se += __shfl_xor(se, o, 64);
  const float lse = mx + logf(se);
  const float pj = ej / se;
  const float tj = on ? target[(size_t)m * NB + j] : 0.f;
  // inclusive prefix sums of p and t over the lanes
  float P = pj, T = tj;
  for (int o = 1; o < 64; o <<= 1) {
    const float a = __shfl_up(P, o, 64), b = __shfl_up(T, o, 64);
    if (j >= o) {
      P += a;
      T += b;
    }
  }
  const float dcdf = on ? P - T : 0.f;
  // suffix sums of (P - T)
  float G = dcdf;
  for (int o = 1; o < 64; o <<= 1) {
    const float a = __shfl_down(G, o, 64);
    if (j + o < 64) G += a;
  }
  const float gj = 2.f * wc * G;
  float pg = pj * gj;
  for (int o = 32; o > 0; o >>= 1) pg += __shfl_xor(pg, o, 64);
  float part = (on ? -tj * (lj - lse) : 0.f) + wc * dcdf * dcdf;
  for (int o = 32; o > 0; o >>= 1) part += __shfl_xor(part, o, 64);
  if (on && dout) dout[(size_t)m * (NB + 1) + j] = (pj - tj + pj * (gj - pg)) / M;
  if (j == 0) {
    const float d = l[NB] - tvar[m];
    if (loss) loss[m] = part + wv * d * d;
    if (dout) dout[(size_t)m * (NB + 1) + NB] = 2.f * wv * d / M;
  }
}

// Adam with bias correction; w, m, v float32.
__device__ __forceinline__ void adam_update(int i, float* __restrict__ w, const float* __restrict__ g,
                                            float* __restrict__ m, float* __restrict__ v, float lr, float b1,
                                            float b2, float eps, float c1, float c2) {
  const float gi = g[i];
  const float mi = b1 * m[i] + (1.f - b1) * gi;
  const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
  m[i] = mi;
  v[i] = vi;
  w[i] -= lr * (mi / c1) / (sqrtf(vi / c2) + eps);
}

__global__ void k_adam(int n, float* __restrict__ w, const float* __restrict__ g, float* __restrict__ m,
                       float* __restrict__ v, float lr, float b1, float b2, float eps, float c1, float c2) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i < n) adam_update(i, w, g, m, v, lr, b1, b2, eps, c1, c2);
}

// The same update of several tensors in one launch (kAdamPer values per block).
constexpr int kAdamTensors = 16, kAdamPer = 1024;
struct AdamTensors {
  float* w[kAdamTensors];
  const float* g[kAdamTensors];
  float* m[kAdamTensors];
  float* v[kAdamTensors];
  int n[kAdamTensors], first[kAdamTensors];   // first: blocks before this tensor
};
__global__ void __launch_bounds__(256)
k_adam_multi(int count, AdamTensors a, float lr, float b1, float b2, float eps, float c1, float c2) {
  int t = 0;
  while (t + 1 < count && (int)blockIdx.x >= a.first[t + 1]) ++t;
  const int base = (blockIdx.x - a.first[t]) * kAdamPer + threadIdx.x;
  float *w = a.w[t], *m = a.m[t], *v = a.v[t];
  const float* g = a.g[t];
#pragma unroll
  for (int j = 0; j < kAdamPer / 256; ++j) {
    const int i = base + 256 * j;
    if (i < a.n[t]) adam_update(i, w, g, m, v, lr, b1, b2, eps, c1, c2);
  }
}

__device__ __forceinline__ unsigned short f2bf(float f) {
  unsigned int u = __float_as_uint(f);
  u += 0x7FFFu + ((u >> 16) & 1u);
  return (unsigned short)(u >> 16);
}

__global__ void k_to_bf16(size_t n, const float* __restrict__ x, unsigned short* __restrict__ y) {
  const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (i < n) y[i] = f2bf(x[i]);
}

// ------------------------------------------------------------------ bf16 MFMA inference layer
// Y[M][N] = act(X[M][K] W[N][K]^T + bias), X float32 (rounded to bf16 on load),
// W bf16, fp32 accumulation.  One wave per 32x32 output tile, 4 waves per block
// covering 32 rows x 128 columns; K multiple of 16, N multiple of 32 (padded by caller).
__global__ void __launch_bounds__(256)
k_layer_bf16(int M, int N, int K, const float* __restrict__ X, const unsigned short* __restrict__ W,
             const float* __restrict__ bias, float* __restrict__ Y, int act) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int m0 = blockIdx.y * 32, n0 = blockIdx.x * 128 + wave * 32;
  if (n0 >= N) return;
  f16v acc;
#pragma unroll
  for (int i = 0; i < 16; ++i) acc[i] = 0.f;
  const int row = m0 + (lane & 31);
  const int col = n0 + (lane & 31);
  for (int k0 = 0; k0 < K; k0 += 16) {
    const int kb = k0 + 8 * (lane >> 5);
    us8 a, b;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      a[j] = row < M ? f2bf(X[(size_t)row * K + kb + j]) : (unsigned short)0;
      b[j] = W[(size_t)col * K + kb + j];
    }
    acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(b8, a), __builtin_bit_cast(b8, b), acc,
                                                  0, 0, 0);
  }
#pragma unroll
  for (int v = 0; v < 16; ++v) {
    const int r = m0 + 8 * (v / 4) + 4 * (lane >> 5) + (v % 4);
    if (r >= M) continue;
    const float z = acc[v] + bias[col];
    Y[(size_t)r * N + col] = act ? z * sigm(z) : z;
  }
}

// ------------------------------------------------------------------ fused bf16 inference
// The whole network in one launch, for layers up to kInferWidth values wide.  A
// block takes 32 rows of one member through every layer; the activations stay
// in LDS as the bf16 values the next product reads, so nothing but the inputs,
// the weights (L2) and the outputs moves.  Weights are packed once per set of
// weights in the order the products read them (pack_bf16): the fragment of
// (32-column tile, 16-wide K chunk) is 1 KB, 16 bytes per lane, where rows of
// the plain matrix gave 32 scattered 32-byte pieces.  A wave owns a tile and
// walks K in groups of kInferAhead chunks, the next group's fragments loaded
// before the current one's products (a serial chain per tile, so the loads'
// latency bounds it); 12 waves cover a 384-wide layer at once, and two blocks
// share a CU.  Chunk order, operand roles and roundings are k_layer_bf16's,
// so the outputs are bit-equal to running the layers one by one.
// Measured, 4096 rows x 3 members of width 384: 720 us of layer launches before,
// 34 us now (55 with one guarded chunk at a time, which took 168 registers, one
// block per CU, and waited for every load).
constexpr int kInferRows = 32, kInferWaves = 12, kInferWidth = 512, kInferAhead = 4;
constexpr int kInferLayers = 16, kInferMembers = 8;
constexpr int kInferStride = kInferWidth + 8;   // bf16 per LDS row: 16-byte reads of 32 rows hit all banks

struct InferNet {
  const float* bias[kInferMembers];             // packed: every layer's biases, then the fragments
  int sizes[kInferLayers + 1];
};

static __host__ __device__ inline int tiles32(int n) { return (n + 31) / 32; }

__global__ void __launch_bounds__(64 * kInferWaves, 2 * kInferWaves / 4)
k_mlp_infer(int layers, int inputs, int M, const float* __restrict__ x, InferNet net, float* __restrict__ out) {
  __shared__ __attribute__((aligned(16))) unsigned short act[2][kInferRows * kInferStride];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, r = lane & 31, h = lane >> 5;
  const int m0 = blockIdx.x * kInferRows, member = blockIdx.y;
  const float* bias = net.bias[member];
  int nb = 0;
  for (int i = 0; i < layers; ++i) nb += 32 * tiles32(net.sizes[i + 1]);
  const unsigned short* w = reinterpret_cast<const unsigned short*>(bias + nb);
  for (int e = threadIdx.x; e < kInferRows * net.sizes[0]; e += 64 * kInferWaves) {
    const int rr = e / net.sizes[0], k = e % net.sizes[0];
    act[0][rr * kInferStride + k] = m0 + rr < M && k < inputs ? f2bf(x[(size_t)(m0 + rr) * inputs + k]) : 0;
  }
  for (int i = 0; i < layers; ++i) {
    __syncthreads();
    const unsigned short* cur = act[i & 1] + r * kInferStride + 8 * h;
    unsigned short* nxt = act[(i + 1) & 1];
    const int nc = net.sizes[i] / 16, fo = net.sizes[i + 1], nt = tiles32(fo);
    for (int t = wave; t < nt; t += kInferWaves) {
      const us8* f = reinterpret_cast<const us8*>(w) + (size_t)t * nc * 64 + lane;
      f16v acc;
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[v] = 0.f;
      auto mma = [&](int c, us8 bf) {
        const us8 a = *reinterpret_cast<const us8*>(cur + 16 * c);
        acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(b8, a), __builtin_bit_cast(b8, bf), acc, 0, 0, 0);
      };
      us8 q[kInferAhead];
#pragma unroll
      for (int u = 0; u < kInferAhead; ++u) q[u] = f[(size_t)min(u, nc - 1) * 64];
      int c0 = 0;
      for (; c0 + kInferAhead <= nc; c0 += kInferAhead) {
        us8 nq[kInferAhead];
#pragma unroll
        for (int u = 0; u < kInferAhead; ++u) nq[u] = f[(size_t)min(c0 + kInferAhead + u, nc - 1) * 64];
#pragma unroll
        for (int u = 0; u < kInferAhead; ++u) mma(c0 + u, q[u]);
#pragma unroll
        for (int u = 0; u < kInferAhead; ++u) q[u] = nq[u];
      }
#pragma unroll
      for (int u = 0; u < kInferAhead - 1; ++u)
        if (c0 + u < nc) mma(c0 + u, q[u]);
      // an opaque copy of the lane index: the epilogue's addresses are formed
      // here, not carried through the layers in registers
      int el = lane;
      asm volatile("" : "+v"(el));
      const int col = 32 * t + (el & 31), row = 4 * (el >> 5);
      const float bc = bias[col];
      if (i < layers - 1) {
        unsigned short* o = nxt + row * kInferStride + col;
#pragma unroll
        for (int v = 0; v < 16; ++v) {
          const float z = acc[v] + bc;
          o[(8 * (v / 4) + v % 4) * kInferStride] = f2bf(z * sigm(z));
        }
      } else if (col < fo) {
        float* o = out + ((size_t)member * M + m0 + row) * fo + col;
        const int left = M - m0 - row;
#pragma unroll
        for (int v = 0; v < 16; ++v) {
          const int rr = 8 * (v / 4) + v % 4;
          if (rr < left) o[rr * fo] = acc[v] + bc;
        }
      }
    }
    bias += 32 * nt;
    w += (size_t)nt * nc * 512;
  }
}

// One layer's weights W[fo][fi] and biases into the packed order.
__global__ void k_pack_bf16(int fo, int fi, const float* __restrict__ W, const float* __restrict__ b,
                            float* __restrict__ pb, unsigned short* __restrict__ pw) {
  const int nc = fi / 16, nt = tiles32(fo), i = blockIdx.x * 256 + threadIdx.x;
  if (i < 32 * nt) pb[i] = i < fo ? b[i] : 0.f;
  if (i >= nt * nc * 512) return;
  const int j = i & 7, l = (i >> 3) & 63, c = (i >> 9) % nc, t = (i >> 9) / nc;
  const int col = 32 * t + (l & 31), k = 16 * c + 8 * (l >> 5) + j;
  pw[i] = col < fo ? f2bf(W[(size_t)col * fi + k]) : 0;
}

// Softmax in float64 of every member's 64 logits, their mean, the mean of the
// log-variances and the members' spread: the largest |CDF difference| of a
// member and the mean (NaN where a logit is NaN, as numpy's max gives).  One
// wave per row, lane = bin.  out: mean [M][64], log-variance [M], spread [M].
__device__ __forceinline__ double nan_max(double a, double b) { return a != a ? a : b != b ? b : fmax(a, b); }
template <class F>
__device__ __forceinline__ double wave_fold(double v, F f) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v = f(v, __shfl_xor(v, o, 64));
  return v;
}
__device__ __forceinline__ double wave_cumsum(double v, int lane) {
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const double a = __shfl_up(v, o, 64);
    if (lane >= o) v += a;
  }
  return v;
}
__global__ void __launch_bounds__(256)
k_mlp_pdt(int members, int M, const float* __restrict__ logits, double* __restrict__ out) {
  const int lane = threadIdx.x & 63, row = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row >= M) return;
  double p[kInferMembers], mean = 0.0, lv = 0.0;
#pragma unroll
  for (int i = 0; i < kInferMembers; ++i) {
    p[i] = 0.0;
    if (i < members) {
      const float* l = logits + ((size_t)i * M + row) * 65;
      const double x = l[lane];
      const double e = exp(x - wave_fold(x, nan_max));
      p[i] = e / wave_fold(e, [](double a, double b) { return a + b; });
      mean += p[i];
      lv += (double)l[64];
    }
  }
  mean /= members;
  const double cm = wave_cumsum(mean, lane);
  double spread = 0.0;
#pragma unroll
  for (int i = 0; i < kInferMembers; ++i)
    if (i < members) spread = nan_max(spread, fabs(wave_cumsum(p[i], lane) - cm));
  spread = wave_fold(spread, nan_max);
  out[(size_t)row * 64 + lane] = mean;
  if (lane == 0) {
    out[(size_t)M * 64 + row] = lv / members;
    out[(size_t)M * 65 + row] = spread;
  }
}

// ------------------------------------------------------------------ launchers
// float4 reads of an operand whose K is contiguous need whole quads of k at 16-byte addresses
static bool quads(const float* p, int ld, int K) {
  return K % 4 == 0 && ld % 4 == 0 && reinterpret_cast<uintptr_t>(p) % 16 == 0;
}

// Row tiles lie on a grid axis of at most 65535 blocks: calls f(first row, rows) for
// as many launches as M rows take.
constexpr int kGridRows = 65535 * GT;
template <class F>
static void row_launches(int M, F f) {
  for (long long m = 0; m < M; m += kGridRows) f((size_t)m, (int)(M - m < kGridRows ? M - m : kGridRows));
}

int mlp_gemm_f32(int M, int N, int K, const float* A, int lda, int ta, const float* B, int ldb, int tb, float* C,
                 int ldc, float alpha, float beta, hipStream_t s) {
  const bool va = !ta && quads(A, lda, K), vb = tb && quads(B, ldb, K);
  row_launches(M, [&](size_t m, int rows) {
    const dim3 g((N + GT - 1) / GT, (rows + GT - 1) / GT);
    const float* a = A + (ta ? m : m * lda);
    float* c = C + m * ldc;
#define G_(TA, TB, VA, VB)                                                                                         \
  hipLaunchKernelGGL((k_gemm_f32<TA, TB, VA, VB>), g, dim3(64 * kGemmWaves), 0, s, rows, N, K, a, lda, B, ldb, c, \
                     ldc, alpha, beta)
    if (ta && tb) {
      if (vb) G_(true, true, false, true);
      else G_(true, true, false, false);
    } else if (ta) {
      G_(true, false, false, false);
    } else if (tb) {
      if (va && vb) G_(false, true, true, true);
      else G_(false, true, false, false);
    } else {
      if (va) G_(false, false, true, false);
      else G_(false, false, false, false);
    }
#undef G_
  });
  return check_launch("mlp_gemm_f32");
}

// Floats of scratch for mlp_loss_grads: per layer Z and dZ (M x fo), and Y for
// the hidden ones; each starts at a multiple of 4 floats.
static size_t padded(size_t n) { return (n + 3) / 4 * 4; }
long long mlp_loss_grads_scratch(int layers, const int* sizes, int M) {
  size_t n = 0;
  for (int i = 0; i < layers; ++i) n += (i < layers - 1 ? 3 : 2) * padded((size_t)M * sizes[i + 1]);
  return (long long)(n * sizeof(float));
}

int mlp_loss_grads(int layers, const int* sizes, int M, const float* X, const float* const* params,
                   const float* target, const float* tvar, float wv, float wc, float* loss, float* mean,
                   float* const* grads, float* scratch, hipStream_t s) {
  const int NB = sizes[layers] - 1;
  // scratch: every layer's Z, then every layer's dZ, then the hidden layers' Y
  size_t all = 0;
  for (int i = 0; i < layers; ++i) all += padded((size_t)M * sizes[i + 1]);
  const float* h = X;
  float *z = scratch, *d = scratch + all, *y = scratch + 2 * all;
  for (int i = 0; i < layers; ++i) {
    const int fi = sizes[i], fo = sizes[i + 1];
    const float *W = params[2 * i], *bias = params[2 * i + 1];
    float* Y = i < layers - 1 ? y : nullptr;
    const bool vec = quads(h, fi, fi) && quads(W, fi, fi);
    row_launches(M, [&](size_t m, int rows) {
      const dim3 g((fo + GT - 1) / GT, (rows + GT - 1) / GT);
      float* Ym = Y ? Y + m * fo : nullptr;
      if (vec)
        hipLaunchKernelGGL(k_layer_forward<true>, g, dim3(64 * kGemmWaves), 0, s, rows, fo, fi, h + m * fi, W, bias,
                           z + m * fo, Ym);
      else
        hipLaunchKernelGGL(k_layer_forward<false>, g, dim3(64 * kGemmWaves), 0, s, rows, fo, fi, h + m * fi, W, bias,
                           z + m * fo, Ym);
    });
    if (i < layers - 1) {
      h = y;
      y += padded((size_t)M * fo);
      z += padded((size_t)M * fo);
      d += padded((size_t)M * fo);
    }
  }
  // z, d: the last layer's
  hipLaunchKernelGGL(k_head_loss, dim3(M), dim3(64), 0, s, M, NB, z, target, tvar, wv, wc, loss, d);
  for (int i = layers - 1; i > 0; --i) {
    const int fi = sizes[i], fo = sizes[i + 1];
    z -= padded((size_t)M * fi);
    float* dn = d - padded((size_t)M * fi);
    const bool vec = quads(d, fo, fo);
    row_launches(M, [&](size_t m, int rows) {
      const dim3 g((fi + GT - 1) / GT, (rows + GT - 1) / GT);
      if (vec)
        hipLaunchKernelGGL(k_layer_backward<true>, g, dim3(64 * kGemmWaves), 0, s, rows, fi, fo, d + m * fo,
                           params[2 * i], z + m * fi, dn + m * fi);
      else
        hipLaunchKernelGGL(k_layer_backward<false>, g, dim3(64 * kGemmWaves), 0, s, rows, fi, fo, d + m * fo,
                           params[2 * i], z + m * fi, dn + m * fi);
    });
    d = dn;
  }
  // d: the first layer's; every layer's dZ and inputs follow one another
  y = scratch + 2 * all;
  h = X;
  for (int i0 = 0; i0 < layers; i0 += kGradLayers) {
    const int cnt = layers - i0 < kGradLayers ? layers - i0 : kGradLayers;
    GradLayers g = {};
    for (int j = 0; j < cnt; ++j) {
      const int fi = sizes[i0 + j], fo = sizes[i0 + j + 1];
      g.d[j] = d;
      g.h[j] = h;
      g.dw[j] = grads[2 * (i0 + j)];
      g.db[j] = grads[2 * (i0 + j) + 1];
      g.fo[j] = fo;
      g.fi[j] = fi;
      g.first[j + 1] = g.first[j] + ((fo + GT - 1) / GT) * ((fi + GT - 1) / GT);
      d += padded((size_t)M * fo);
      h = y;
      y += padded((size_t)M * fo);
    }
    const bool last = i0 + cnt == layers;
    hipLaunchKernelGGL(k_weight_grads, dim3(g.first[cnt] + (last && mean ? 1 : 0)), dim3(64 * kGradWaves), 0, s, cnt, M,
                       g, loss, mean);
  }
  return check_launch("mlp_loss_grads");
}

int mlp_adam_multi(int count, const int* n, float* const* w, const float* const* g, float* const* m,
                   float* const* v, float lr, float b1, float b2, float eps, int t, hipStream_t s) {
  const float c1 = 1.f - powf(b1, (float)t), c2 = 1.f - powf(b2, (float)t);
  for (int i0 = 0; i0 < count;) {
    AdamTensors a = {};
    int blocks = 0, cnt = 0;
    // a tensor that is there already (weights that layers share) is updated again
    // in the next launch, after the first update
    auto there = [&](int i) {
      for (int j = 0; j < cnt; ++j)
        if (a.w[j] == w[i] || a.m[j] == m[i] || a.v[j] == v[i]) return true;
      return false;
    };
    for (int i = i0; i < count && cnt < kAdamTensors && !there(i); ++i, ++cnt) {
      a.w[cnt] = w[i];
      a.g[cnt] = g[i];
      a.m[cnt] = m[i];
      a.v[cnt] = v[i];
      a.n[cnt] = n[i];
      a.first[cnt] = blocks;
      blocks += (n[i] + kAdamPer - 1) / kAdamPer;
    }
    i0 += cnt;
    hipLaunchKernelGGL(k_adam_multi, dim3(blocks), dim3(256), 0, s, cnt, a, lr, b1, b2, eps, c1, c2);
  }
  return check_launch("mlp_adam_multi");
}
int mlp_bias_act(int M, int N, float* Z, const float* bias, float* Y, int act, hipStream_t s) {
  hipLaunchKernelGGL(k_bias_act, dim3((unsigned)(((size_t)M * N + 255) / 256)), dim3(256), 0, s, M, N, Z, bias,
                     Y, act);
  return check_launch("mlp_bias_act");
}
int mlp_act_backward(int M, int N, const float* Z, const float* dY, float* dZ, hipStream_t s) {
  hipLaunchKernelGGL(k_act_backward, dim3((unsigned)(((size_t)M * N + 255) / 256)), dim3(256), 0, s, M, N, Z,
                     dY, dZ);
  return check_launch("mlp_act_backward");
}
int mlp_bias_grad(int M, int N, const float* dZ, float* db, hipStream_t s) {
  hipLaunchKernelGGL(k_bias_grad, dim3((N + 255) / 256), dim3(256), 0, s, M, N, dZ, db);
  return check_launch("mlp_bias_grad");
}
int mlp_head_loss(int M, int NB, const float* out, const float* target, const float* tvar, float wv, float wc,
                  float* loss, float* dout, hipStream_t s) {
  hipLaunchKernelGGL(k_head_loss, dim3(M), dim3(64), 0, s, M, NB, out, target, tvar, wv, wc, loss, dout);
  return check_launch("mlp_head_loss");
}
int mlp_adam(int n, float* w, const float* g, float* m, float* v, float lr, float b1, float b2, float eps,
             int t, hipStream_t s) {
  const float c1 = 1.f - powf(b1, (float)t), c2 = 1.f - powf(b2, (float)t);
  hipLaunchKernelGGL(k_adam, dim3((n + 255) / 256), dim3(256), 0, s, n, w, g, m, v, lr, b1, b2, eps, c1, c2);
  return check_launch("mlp_adam");
}
int mlp_to_bf16(long long n, const float* x, unsigned short* y, hipStream_t s) {
  hipLaunchKernelGGL(k_to_bf16, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, (size_t)n, x, y);
  return check_launch("mlp_to_bf16");
}
int mlp_layer_bf16(int M, int N, int K, const float* X, const unsigned short* W, const float* bias, float* Y,
                   int act, hipStream_t s) {
  dim3 g((N + 127) / 128, (M + 31) / 32);
  hipLaunchKernelGGL(k_layer_bf16, g, dim3(256), 0, s, M, N, K, X, W, bias, Y, act);
  return check_launch("mlp_layer_bf16");
}


bool mlp_infer_fits(int layers, const int* sizes) {
  if (layers > kInferLayers) return false;
  for (int i = 0; i < layers; ++i)
    if (sizes[i] % 16 || sizes[i] > kInferWidth) return false;
  return true;
}
long long mlp_pack_bytes(int layers, const int* sizes) {
  long long n = 0;
  for (int i = 0; i < layers; ++i) n += tiles32(sizes[i + 1]) * (128ll + (long long)sizes[i] / 16 * 1024);
  return n;
}
int mlp_pack_bf16(int layers, const int* sizes, const float* const* params, void* packed, hipStream_t s) {
  float* pb = reinterpret_cast<float*>(packed);
  int nb = 0;
  for (int i = 0; i < layers; ++i) nb += 32 * tiles32(sizes[i + 1]);
  unsigned short* pw = reinterpret_cast<unsigned short*>(pb + nb);
  for (int i = 0; i < layers; ++i) {
    const int fi = sizes[i], fo = sizes[i + 1], nt = tiles32(fo), n = nt * (fi / 16) * 512;
    hipLaunchKernelGGL(k_pack_bf16, dim3((n + 255) / 256), dim3(256), 0, s, fo, fi, params[2 * i], params[2 * i + 1], pb,
                       pw);
    pb += 32 * nt;
    pw += n;
  }
  return check_launch("mlp_pack_bf16");
}
int mlp_infer(int layers, const int* sizes, int inputs, int members, const void* const* packed, int M, const float* x,
              float* out, hipStream_t s) {
  for (int i0 = 0; i0 < members; i0 += kInferMembers) {
    const int cnt = members - i0 < kInferMembers ? members - i0 : kInferMembers;
    InferNet net = {};
    for (int j = 0; j < cnt; ++j) net.bias[j] = reinterpret_cast<const float*>(packed[i0 + j]);
    for (int i = 0; i <= layers; ++i) net.sizes[i] = sizes[i];
    hipLaunchKernelGGL(k_mlp_infer, dim3((M + kInferRows - 1) / kInferRows, cnt), dim3(64 * kInferWaves), 0, s, layers,
                       inputs, M, x, net, out + (size_t)i0 * M * sizes[layers]);
  }
  return check_launch("mlp_infer");
}
int mlp_pdt(int members, int M, const float* logits, double* out, hipStream_t s) {
  if (members > kInferMembers) return set_error(PA_ERR_ARG, "mlp_pdt: at most 8 members");
  hipLaunchKernelGGL(k_mlp_pdt, dim3((M + 3) / 4), dim3(256), 0, s, members, M, logits, out);
  return check_launch("mlp_pdt");
}

}  // namespace pa

// mlp.hip -- the learned warm start's network: 4 dense layers (n_in -> W ->
// W -> W -> n_out, ReLU between) trained and evaluated with hand-written
// BF16 MFMA kernels (v_mfma_f32_16x16x16_bf16, FP32 accumulation).
//
// No reference counterpart: the network replaces the linear extrapolation of
// Bead::initialGuess (Bead.hpp:202-217) as the first Broyden iterate.
//
// Numerics (mirrored by the CPU oracle oracle/mlp_oracle.py):
//   forward   x_n = (x - mu)/sigma rounded to BF16; weights rounded to BF16;
//             z_l = h_{l-1} W_l^T + b_l in FP32; h_l = BF16(relu(z_l));
//             y = tau * (h_3 W_3^T + b_3 + x_n S^T) with S an optional
//             fixed linear map set by the host (a ridge fit), BF16
//             (fs_mlp_set_skip); the layers then learn the residual
//   loss      mean over batch and outputs of (y_n - t/tau)^2, y_n the
//             normalised output
//   backward  g = BF16(dL/dz) feeds both MFMA products (dW = g^T h,
//             dh = g W); bias gradients from the FP32 dL/dz
//   inference in one launch up to 2 Mi weights (k_mlp_forward), the same
//             rounding points
//   optimiser Adam on FP32 master weights (beta 0.9/0.999, eps 1e-8)
#include <hip/hip_runtime.h>

#include <climits>
#include <cmath>
#include <cstdint>
#include <type_traits>
#include <vector>

#include "common.hpp"

namespace fs {

typedef short s4v __attribute__((ext_vector_type(4)));
typedef float f4v __attribute__((ext_vector_type(4)));
typedef __bf16 b8v __attribute__((ext_vector_type(8)));

__device__ __forceinline__ uint16_t f2bf(float f) {  // round to nearest even
  uint32_t u = __float_as_uint(f);
  u += 0x7FFFu + ((u >> 16) & 1u);
  return (uint16_t)(u >> 16);
}
__device__ __forceinline__ float bf2f(uint16_t b) {
  return __uint_as_float(((uint32_t)b) << 16);
}

enum { EPI_STORE = 0, EPI_HIDDEN = 1, EPI_OUT = 2, EPI_DRELU = 3, EPI_ADD = 4 };

// C(m,n) = sum_k A(m,k) B(k,n), A(m,k) = A[m*sam + k*sak], B(k,n) =
// B[k*sbk + n*sbn] (BF16). One workgroup per 32x32 output tile (2x2 MFMA
// 16x16 blocks): wavefront w takes the w-th quarter of the K steps of 16,
// and the four partial tiles are added through LDS in wavefront order
// before the epilogue (a fixed order: results do not depend on timing).
// MFMA 16x16x16 lane layout: lane l feeds A[l%16][4(l/16)..+3] and
// B[4(l/16)..+3][l%16] and receives D[4(l/16)+i][l%16], i < 4. AV / BV: A
// (B) is contiguous along k with 8-byte aligned rows (columns), so a lane's
// four k values are one 8-byte load.
// Epilogues: STORE  Cf = acc
//            HIDDEN Zf = acc + bias, Hb = BF16(relu(Zf))
//            OUT    Cf = acc + bias
//            DRELU  g = acc * (Zf > 0): Cf = g, Hb = BF16(g)
//            ADD    Cf += acc
// Bound by the latency of the loads: those of 4 steps go out together, what is
// left of a wavefront's steps by 2 and 1 (K = 64, one step a wavefront: 4.3 us;
// always 4 steps, with zeros past the end, 5.9 us).
template <bool AV, bool BV>
__global__ void __launch_bounds__(256)
    k_gemm_bf16(int M, int N, int K, const uint16_t *__restrict__ A, long sam,
                long sak, const uint16_t *__restrict__ B, long sbk, long sbn,
                int epi, const float *__restrict__ bias, float *__restrict__ Cf,
                long ldc, uint16_t *__restrict__ Hb, long ldh,
                const float *__restrict__ Zin, long ldz) {
  __shared__ float red[4][32 * 33];  // the waves' partial tiles
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int tilesN = (N + 31) / 32;
  const int tm = blockIdx.x / tilesN, tn = blockIdx.x - tm * tilesN;
  const int m0 = tm * 32, n0 = tn * 32;
  const int r = lane & 15, kq = (lane >> 4) * 4;
  const int ks = (K + 15) / 16;
  const int s0 = ks * wave / 4, s1 = ks * (wave + 1) / 4;
  f4v acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[i][j] = f4v{0.f, 0.f, 0.f, 0.f};
  // steps sb .. sb + AH - 1
  const auto steps = [&](auto ahead, int sb) {
    constexpr int AH = decltype(ahead)::value;
    s4v a[AH][2], b[AH][2];
#pragma unroll
    for (int u = 0; u < AH; ++u) {
      const int k = 16 * (sb + u) + kq;
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int m = m0 + 16 * i + r;
        if (AV && m < M && k + 4 <= K) {
          a[u][i] = *reinterpret_cast<const s4v *>(A + (long)m * sam + k);
        } else {
#pragma unroll
          for (int q = 0; q < 4; ++q)
            a[u][i][q] = (m < M && k + q < K)
                             ? (short)A[(long)m * sam + (long)(k + q) * sak]
                             : (short)0;
        }
      }
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const int n = n0 + 16 * j + r;
        if (BV && n < N && k + 4 <= K) {
          b[u][j] = *reinterpret_cast<const s4v *>(B + (long)n * sbn + k);
        } else {
#pragma unroll
          for (int q = 0; q < 4; ++q)
            b[u][j][q] = (n < N && k + q < K)
                             ? (short)B[(long)(k + q) * sbk + (long)n * sbn]
                             : (short)0;
        }
      }
    }
#pragma unroll
    for (int u = 0; u < AH; ++u)
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(
              a[u][i], b[u][j], acc[i][j], 0, 0, 0);
  };
  int s = s0;
  for (; s + 4 <= s1; s += 4) steps(std::integral_constant<int, 4>{}, s);
  if (s + 2 <= s1) {
    steps(std::integral_constant<int, 2>{}, s);
    s += 2;
  }
  if (s < s1) steps(std::integral_constant<int, 1>{}, s);
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int q = 0; q < 4; ++q)
        red[wave][(16 * i + kq + q) * 33 + 16 * j + r] = acc[i][j][q];
  __syncthreads();
  for (int e = threadIdx.x; e < 32 * 32; e += 256) {
    const int lm = e >> 5, ln = e & 31;
    const int m = m0 + lm, n = n0 + ln;
    if (m >= M || n >= N) continue;
    const int o = lm * 33 + ln;
    const float v = ((red[0][o] + red[1][o]) + red[2][o]) + red[3][o];
    if (epi == EPI_HIDDEN) {
      const float z = v + bias[n];
      Cf[(long)m * ldc + n] = z;
      Hb[(long)m * ldh + n] = f2bf(z > 0.f ? z : 0.f);
    } else if (epi == EPI_OUT) {
      Cf[(long)m * ldc + n] = v + bias[n];
    } else if (epi == EPI_ADD) {
      Cf[(long)m * ldc + n] += v;
    } else if (epi == EPI_DRELU) {
      const float g = Zin[(long)m * ldz + n] > 0.f ? v : 0.f;
      Cf[(long)m * ldc + n] = g;
      Hb[(long)m * ldh + n] = f2bf(g);
    } else {
      Cf[(long)m * ldc + n] = v;
    }
  }
}

// ---------------------------------------------------------------------
// The whole inference pass of 16 rows in one workgroup of 16 wavefronts:
// normalised inputs and activations stay in LDS as BF16, the weights are read
// from L2. Each wavefront makes 16 outputs of a layer (16 x 16 MFMA tile, all
// of K; further tiles 16 wavefronts on). Same roundings as the layers one by
// one (inputs, activations BF16, sums FP32, bias and skip term added in FP32).
// Bound by the latency and the rate at which a CU reads the weights: they are
// kept a second time in the order of the loads, 1 KB of a wavefront in one
// piece (as stored, a load's 16 rows of 64 bytes each are looked up one by
// one: 27 us instead of 16 us for 1,000 rows of 716-256-256-256-180 with a skip
// map, and 46 us layer by layer). 8,000 rows 147 -> 38 us.
// ---------------------------------------------------------------------
constexpr int kMlpRows = 16, kMlpWaves = 16, kMlpAhead = 8;

// LDS row of n BF16 values: whole steps of 32, and 16 bytes so that 16 rows
// fall on different banks.
__host__ __device__ constexpr int mlp_row(int n) { return (n + 31) / 32 * 32 + 8; }

// Place of element (n, k) of a matrix with K columns among its tiles of 16
// rows by 32 columns: lane l of a wavefront reads row l % 16, columns
// 8 (l / 16) .. + 7 of a tile as 16 bytes, the tiles of 16 rows in a row.
__host__ __device__ inline long mlp_packed(int K, int n, int k) {
  const long tile = (long)(n >> 4) * ((K + 31) / 32) + (k >> 5);
  return (tile * 64 + (n & 15) + 16 * ((k >> 3) & 3)) * 8 + (k & 7);
}
__host__ __device__ inline long mlp_packed_size(int K, int N) {
  return (long)((N + 15) / 16) * ((K + 31) / 32) * 512;
}

// Layers of the network: offsets of W_l and b_l in the parameters, of the
// packed W_l (l < 4) and skip map (l = 4) in packed (nullptr: not kept).
struct MlpNet {
  long woff[4], boff[4], poff[5];
  int dims[5];
  uint16_t *packed;
};

__device__ __forceinline__ void mlp_pack_param(const MlpNet &net, long i,
                                               uint16_t v) {
  if (!net.packed) return;
#pragma unroll
  for (int l = 0; l < 4; ++l)
    if (i >= net.woff[l] && i < net.boff[l]) {
      const uint32_t K = net.dims[l], r = (uint32_t)(i - net.woff[l]), n = r / K;
      net.packed[net.poff[l] + mlp_packed(K, n, r - n * K)] = v;
    }
}

__global__ void k_pack_skip(const uint16_t *__restrict__ S, MlpNet net) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  const int K = net.dims[0];
  if (i >= (long)K * net.dims[4]) return;
  const int n = (int)(i / K);
  net.packed[net.poff[4] + mlp_packed(K, n, (int)(i - (long)n * K))] = S[i];
}

// 16 x 16 tile sum_k A[m][k] W[n][k] over the LDS rows a (stride lda) and 16
// packed rows w of W. Lane l holds rows 4 (l / 16) + i of column l % 16.
__device__ __forceinline__ f4v mlp_tile(const uint16_t *a, int lda,
                                        const uint16_t *__restrict__ w, int K,
                                        int lane) {
  constexpr int P = kMlpAhead;
  const int steps = (K + 31) / 32;
  const b8v *wl = reinterpret_cast<const b8v *>(w) + lane;
  const uint16_t *ar = a + (lane & 15) * lda + 8 * (lane >> 4);
  f4v acc = {0.f, 0.f, 0.f, 0.f};
  for (int s = 0; s < steps; s += P) {
    b8v v[P];  // the last step's again past the end
#pragma unroll
    for (int j = 0; j < P; ++j) v[j] = wl[64 * min(s + j, steps - 1)];
#pragma unroll
    for (int j = 0; j < P; ++j)
      if (s + j < steps) {
        const b8v x = *reinterpret_cast<const b8v *>(ar + 32 * (s + j));
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(x, v[j], acc, 0, 0, 0);
      }
  }
  return acc;
}

// P: the FP32 parameters (biases).
__global__ void __launch_bounds__(64 * kMlpWaves)
    k_mlp_forward(int rows, MlpNet net, int skip, const float *__restrict__ mu,
                  const float *__restrict__ sig, const float *__restrict__ tau,
                  const float *__restrict__ P, const float *__restrict__ X,
                  float *__restrict__ Y) {
  extern __shared__ __align__(16) uint16_t s_mlp[];
  const int nin = net.dims[0], width = net.dims[1], nout = net.dims[4];
  const int ldx = mlp_row(nin), ldh = mlp_row(width);
  uint16_t *xn = s_mlp, *h0 = xn + kMlpRows * ldx, *h1 = h0 + kMlpRows * ldh;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int r0 = blockIdx.x * kMlpRows;
  // one wavefront a row; what pads K to whole steps is zero
  const bool row = r0 + wave < rows;
  for (int c = lane; c < ldx; c += 64) {
    float v = 0.f;
    if (row && c < nin) v = (X[(long)(r0 + wave) * nin + c] - mu[c]) / sig[c];
    xn[wave * ldx + c] = f2bf(v);
  }
  for (int c = width + lane; c < ldh; c += 64)
    h0[wave * ldh + c] = h1[wave * ldh + c] = 0;
  __syncthreads();
  const int n16 = lane & 15, m4 = 4 * (lane >> 4);
  const uint16_t *a = xn;
  int lda = ldx, K = nin;
  for (int l = 0; l < 3; ++l) {
    uint16_t *h = (l & 1) ? h1 : h0;
    for (int t = wave; 16 * t < width; t += kMlpWaves) {
      const int n = 16 * t + n16;
      const f4v acc = mlp_tile(
          a, lda, net.packed + net.poff[l] + mlp_packed(K, 16 * t, 0), K, lane);
      if (n < width) {
        const float b = P[net.boff[l] + n];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float z = acc[i] + b;
          h[(m4 + i) * ldh + n] = f2bf(z > 0.f ? z : 0.f);
        }
      }
    }
    __syncthreads();
    a = h;
    lda = ldh;
    K = width;
  }
  for (int t = wave; 16 * t < nout; t += kMlpWaves) {
    const int n = 16 * t + n16;
    const f4v acc = mlp_tile(
        a, lda, net.packed + net.poff[3] + mlp_packed(K, 16 * t, 0), K, lane);
    f4v sk = {0.f, 0.f, 0.f, 0.f};
    if (skip)
      sk = mlp_tile(xn, ldx,
                    net.packed + net.poff[4] + mlp_packed(nin, 16 * t, 0), nin,
                    lane);
    if (n < nout) {
      const float b = P[net.boff[3] + n], tn = tau[n];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        float y = acc[i] + b;
        if (skip) y += sk[i];
        if (r0 + m4 + i < rows) Y[(long)(r0 + m4 + i) * nout + n] = y * tn;
      }
    }
  }
}
static_assert(kMlpRows == kMlpWaves, "one wavefront normalises a row");

__global__ void k_to_bf16(const float *__restrict__ x, long n,
                          uint16_t *__restrict__ y) {
  long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) y[i] = f2bf(x[i]);
}

// BF16 parameters, as stored and packed
__global__ void k_quantise(const float *__restrict__ x, long n,
                           uint16_t *__restrict__ y, MlpNet net) {
  long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const uint16_t v = f2bf(x[i]);
  y[i] = v;
  mlp_pack_param(net, i, v);
}

// Column of element i of n elements in rows of cols: a 64-bit division only
// where 32 bits do not hold the elements.
__device__ __forceinline__ int column_of(long i, long n, int cols) {
  return n <= 0xFFFFFFFFl ? (int)((uint32_t)i % (uint32_t)cols) : (int)(i % cols);
}

// x_n = BF16((x - mu) / sigma) per column
__global__ void k_normalise_in(const float *__restrict__ x, int rows, int cols,
                               const float *__restrict__ mu,
                               const float *__restrict__ sig,
                               uint16_t *__restrict__ y) {
  long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= (long)rows * cols) return;
  const int c = column_of(i, (long)rows * cols, cols);
  y[i] = f2bf((x[i] - mu[c]) / sig[c]);
}

__global__ void k_scale_out(float *__restrict__ y, int rows, int cols,
                            const float *__restrict__ tau) {
  long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= (long)rows * cols) return;
  y[i] *= tau[column_of(i, (long)rows * cols, cols)];
}

// dL/dy_n for L = mean((y_n - t/tau)^2); partial loss sums per block.
__global__ void __launch_bounds__(256)
    k_mse_grad(const float *__restrict__ yn, const float *__restrict__ t,
               const float *__restrict__ tau, int rows, int cols,
               float *__restrict__ g, uint16_t *__restrict__ gb,
               float *__restrict__ partial) {
  __shared__ float red[256];
  long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  const long n = (long)rows * cols;
  float l = 0.f;
  if (i < n) {
    float d = yn[i] - t[i] / tau[column_of(i, n, cols)];
    float gi = 2.f * d / (float)n;
    g[i] = gi;
    gb[i] = f2bf(gi);
    l = d * d;
  }
  red[threadIdx.x] = l;
  __syncthreads();
  for (int off = 128; off > 0; off >>= 1) {
    if (threadIdx.x < off) red[threadIdx.x] += red[threadIdx.x + off];
    __syncthreads();
  }
  if (threadIdx.x == 0) partial[blockIdx.x] = red[0];
}

// column sums (bias gradients) in a fixed order: a workgroup of 16
// wavefronts per 64 columns, wavefront w adds the w-th contiguous sixteenth
// of the rows (one coalesced row segment per load), then the 16 partial
// sums are added in wavefront order. Few workgroups, so bound by the latency
// of the loads: 16 of them are in flight, of the last rows 8 (1,000 rows by 256
// 4.7 us; the last rows one by one 7.9 us).
__global__ void __launch_bounds__(1024)
    k_colsum(const float *__restrict__ g, int rows, int cols,
             float *__restrict__ out) {
  __shared__ float part[16][64];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int c = blockIdx.x * 64 + lane;
  const int per = (rows + 15) / 16, r0 = min(rows, w * per),
            r1 = min(rows, r0 + per);
  float s = 0.f;
  if (c < cols) {
    int r = r0;
    for (; r + 16 <= r1; r += 16) {
      float v[16];
#pragma unroll
      for (int j = 0; j < 16; ++j) v[j] = g[(long)(r + j) * cols + c];
#pragma unroll
      for (int j = 0; j < 16; ++j) s += v[j];
    }
    for (; r < r1; r += 8) {
      float v[8];  // the last row's again past the end
#pragma unroll
      for (int j = 0; j < 8; ++j) v[j] = g[(long)min(r + j, r1 - 1) * cols + c];
#pragma unroll
      for (int j = 0; j < 8; ++j)
        if (r + j < r1) s += v[j];
    }
  }
  part[w][lane] = s;
  __syncthreads();
  if (w == 0 && c < cols) {
    float t = 0.f;
#pragma unroll
    for (int k = 0; k < 16; ++k) t += part[k][lane];
    out[c] = t;
  }
}

// sum of n partials in a fixed order: thread t adds the t-th contiguous
// run of ceil(n / 256), then a tree over the 256 run sums
__global__ void __launch_bounds__(256)
    k_sum(const float *__restrict__ p, int n, float *__restrict__ out) {
  __shared__ float red[256];
  const int t = threadIdx.x, per = (n + 255) / 256;
  const int lo = min(n, t * per), hi = min(n, lo + per);
  float s = 0.f;
  for (int i = lo; i < hi; ++i) s += p[i];
  red[t] = s;
  __syncthreads();
  for (int off = 128; off > 0; off >>= 1) {
    if (t < off) red[t] += red[t + off];
    __syncthreads();
  }
  if (t == 0) *out = red[0];
}

__global__ void k_adam(float *__restrict__ w, const float *__restrict__ g,
                       float *__restrict__ m, float *__restrict__ v, long n,
                       float lr, float b1, float b2, float eps, float c1,
                       float c2, uint16_t *__restrict__ wb, MlpNet net) {
  long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  float gi = g[i];
  float mi = b1 * m[i] + (1.f - b1) * gi;
  float vi = b2 * v[i] + (1.f - b2) * gi * gi;
  m[i] = mi;
  v[i] = vi;
  float wi = w[i] - lr * (mi / c1) / (sqrtf(vi / c2) + eps);
  w[i] = wi;
  const uint16_t b = f2bf(wi);
  wb[i] = b;
  mlp_pack_param(net, i, b);
}

// Packed values up to which inference goes in one launch. One launch and layer
// by layer in us, 716 inputs and 180 outputs, 16 and 1,000 rows: 256 wide (0.5
// Mi values) 15 and 16, 36 and 46; 768 wide (2.0 Mi) 44 and 47, 47 and 85;
// 1,024 wide (3.0 Mi) 73 and 67, 52 and 115.
constexpr long kMlpFusedWeights = 2 << 20;
// Packed values in use below which many rows go layer by layer: a workgroup of
// 16 wavefronts has work for one to four of them in so narrow a net, so its time
// is the rows'. The line in rows follows the measured crossings, one launch and
// layer by layer in us: 28-16-16-16-12 (2 Ki values) 30,000 rows 24 and 25,
// 40,000 29 and 27, 200,000 130 and 81; with a skip map 60,000 42 and 48, 100,000
// 68 and 63; 28-64-64-64-12 (11 Ki) 60,000 54 and 62, 200,000 171 and 151;
// 92-64-64-64-24 (16 Ki) 200,000 193 and 199.
constexpr long kMlpNarrow = 14 << 10;
inline long mlp_fused_rows(long values, bool skip) {
  return values >= kMlpNarrow ? LONG_MAX
                              : 20480 + 8 * values + (skip ? 40960 : 0);
}

struct MlpImpl {
  int nin = 0, width = 0, nout = 0;
  int dims[5];
  long woff[5], boff[5];  // offsets of W_l (out x in) and b_l in params
  long nparams = 0;
  dbuf params, grads, adam_m, adam_v, wbf;  // fp32 master + bf16 copies
  dbuf norm;                                 // mu[nin], sigma[nin], tau[nout]
  dbuf skip;                                 // BF16 S[nout][nin] (optional)
  bool has_skip = false;
  MlpNet net{};                              // one-launch inference
  dbuf packed;
  dbuf act;                                  // activations / scratch
  long act_rows = 0;
  long step = 0;
  float *Zf[4];
  uint16_t *Hb[4];
  float *Y, *G, *Gtmp;
  uint16_t *Gb, *Gb2;
  float *partial, *lossd;
  hipStream_t st = nullptr;

  int init(int n_in, int w, int n_out, unsigned long long seed) {
    FS_CHECK(n_in >= 1 && w >= 16 && n_out >= 1 && n_in <= 65536 &&
                 w <= 4096 && n_out <= 65536,
             FS_ERR_ARG, "bad MLP sizes %d %d %d", n_in, w, n_out);
    nin = n_in;
    width = w;
    nout = n_out;
    dims[0] = n_in;
    dims[1] = dims[2] = dims[3] = w;
    dims[4] = n_out;
    long o = 0;
    for (int l = 0; l < 4; ++l) {
      woff[l] = o;
      o += (long)dims[l + 1] * dims[l];
      boff[l] = o;
      o += dims[l + 1];
    }
    nparams = o;
    FS_TRY(params.alloc(sizeof(float) * nparams));
    FS_TRY(grads.alloc(sizeof(float) * nparams));
    FS_TRY(adam_m.alloc(sizeof(float) * nparams));
    FS_TRY(adam_v.alloc(sizeof(float) * nparams));
    FS_TRY(wbf.alloc(sizeof(uint16_t) * nparams));
    FS_TRY(norm.alloc(sizeof(float) * (2 * nin + nout)));
    FS_TRY(init_packed());
    // He-uniform initialisation from a splitmix64 stream, zero biases
    std::vector<float> h(nparams, 0.f);
    uint64_t s = seed;
    auto next = [&]() {
      uint64_t z = (s += 0x9E3779B97F4A7C15ull);
      z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
      z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
      z ^= z >> 31;
      return (z >> 11) * (1.0 / 9007199254740992.0);
    };
    for (int l = 0; l < 4; ++l) {
      double lim = std::sqrt(6.0 / dims[l]) * (l == 3 ? 0.1 : 1.0);
      for (long i = 0; i < (long)dims[l + 1] * dims[l]; ++i)
        h[woff[l] + i] = (float)((2.0 * next() - 1.0) * lim);
    }
    FS_HIP(hipMemcpy(params.p, h.data(), sizeof(float) * nparams,
                     hipMemcpyHostToDevice));
    FS_HIP(hipMemset(adam_m.p, 0, sizeof(float) * nparams));
    FS_HIP(hipMemset(adam_v.p, 0, sizeof(float) * nparams));
    std::vector<float> nm(2 * nin + nout, 0.f);
    for (int i = 0; i < nin; ++i) nm[nin + i] = 1.f;
    for (int i = 0; i < nout; ++i) nm[2 * nin + i] = 1.f;
    FS_HIP(hipMemcpy(norm.p, nm.data(), sizeof(float) * nm.size(),
                     hipMemcpyHostToDevice));
    FS_TRY(requantise());
    FS_HIP(hipDeviceSynchronize());
    return FS_OK;
  }
  void release() {
    params.release();
    grads.release();
    adam_m.release();
    adam_v.release();
    wbf.release();
    norm.release();
    skip.release();
    packed.release();
    act.release();
  }
  int requantise() {
    hipLaunchKernelGGL(k_quantise, dim3(ceil_div(nparams, 256)), dim3(256), 0,
                       st, params.as<float>(), nparams, wbf.as<uint16_t>(), net);
    FS_LAUNCHED();
    return FS_OK;
  }
  int ensure(long rows) {
    if (rows <= act_rows) return FS_OK;
    long w = width, mx = std::max<long>(std::max<long>(nin, nout), width);
    // every piece starts on a 256-byte boundary: the allocation is the sum
    // of the rounded sizes
    auto r256 = [](size_t b) { return (b + 255) & ~size_t(255); };
    size_t bytes = 0;
    bytes += 4 * r256(rows * w * sizeof(float));      // Zf
    bytes += 4 * r256(rows * mx * sizeof(uint16_t));  // Hb (Hb[0] = x_n)
    bytes += 3 * r256(rows * mx * sizeof(float));     // Y, G, Gtmp
    bytes += 2 * r256(rows * mx * sizeof(uint16_t));  // Gb, Gb2
    bytes += r256((rows * mx / 256 + 4) * sizeof(float));  // partial
    bytes += r256(16);                                      // loss
    FS_TRY(act.alloc(bytes));
    char *p = (char *)act.p;
    auto take = [&](size_t b) {
      char *r = p;
      p += r256(b);
      return r;
    };
    for (int l = 0; l < 4; ++l) Zf[l] = (float *)take(rows * w * sizeof(float));
    for (int l = 0; l < 4; ++l) Hb[l] = (uint16_t *)take(rows * mx * 2);
    Y = (float *)take(rows * mx * sizeof(float));
    G = (float *)take(rows * mx * sizeof(float));
    Gtmp = (float *)take(rows * mx * sizeof(float));
    Gb = (uint16_t *)take(rows * mx * 2);
    Gb2 = (uint16_t *)take(rows * mx * 2);
    partial = (float *)take((rows * mx / 256 + 4) * sizeof(float));
    lossd = (float *)take(16);
    act_rows = rows;
    return FS_OK;
  }
  void gemm(int M, int N, int K, const uint16_t *A, long sam, long sak,
            const uint16_t *B, long sbk, long sbn, int epi, const float *bias,
            float *Cf, long ldc, uint16_t *Hbo, long ldh, const float *Z,
            long ldz) {
    const long tiles = (long)((M + 31) / 32) * ((N + 31) / 32);
    const bool av = sak == 1 && sam % 4 == 0 && ((uintptr_t)A & 7) == 0;
    const bool bv = sbk == 1 && sbn % 4 == 0 && ((uintptr_t)B & 7) == 0;
    auto go = [&](auto kern) {
      hipLaunchKernelGGL(kern, dim3(tiles), dim3(256), 0, st, M, N, K, A, sam,
                         sak, B, sbk, sbn, epi, bias, Cf, ldc, Hbo, ldh, Z, ldz);
    };
    if (av && bv) go(k_gemm_bf16<true, true>);
    else if (av) go(k_gemm_bf16<true, false>);
    else if (bv) go(k_gemm_bf16<false, true>);
    else go(k_gemm_bf16<false, false>);
  }
  const float *mu() { return norm.as<float>(); }
  const float *sig() { return norm.as<float>() + nin; }
  const float *tau() { return norm.as<float>() + 2 * nin; }
  // forward into Y (normalised output), activations kept for backward
  int forward_n(int B, const float *X) {
    FS_TRY(ensure(B));
    hipLaunchKernelGGL(k_normalise_in, dim3(ceil_div((long)B * nin, 256)),
                       dim3(256), 0, st, X, B, nin, mu(), sig(), Hb[0]);
    const uint16_t *W = wbf.as<uint16_t>();
    const float *P = params.as<float>();
    const uint16_t *h = Hb[0];
    long ldh = nin;
    for (int l = 0; l < 3; ++l) {
      // z = h W_l^T: B(k=in, n=out) = W_l[out][in]
      gemm(B, dims[l + 1], dims[l], h, ldh, 1, W + woff[l], 1, dims[l],
           EPI_HIDDEN, P + boff[l], Zf[l], width, Hb[l + 1], width, nullptr, 0);
      h = Hb[l + 1];
      ldh = width;
    }
    gemm(B, nout, width, h, width, 1, W + woff[3], 1, width, EPI_OUT,
         P + boff[3], Y, nout, nullptr, 0, nullptr, 0);
    if (has_skip)  // Y += x_n S^T: B(k=in, n=out) = S[out][in]
      gemm(B, nout, nin, Hb[0], nin, 1, skip.as<uint16_t>(), 1, nin, EPI_ADD,
           nullptr, Y, nout, nullptr, 0, nullptr, 0);
    FS_LAUNCHED();
    return FS_OK;
  }
  // Whether inference goes in one launch. Every workgroup reads all weights,
  // so nets beyond kMlpFusedWeights go layer by layer, where workgroups share
  // them out, and so do many rows of narrow nets. Its outputs must not lie over
  // inputs that another workgroup has yet to read.
  bool fused(int B, const float *X, const float *Yout) const {
    const uintptr_t x = (uintptr_t)X, y = (uintptr_t)Yout;
    const long values =
        net.poff[4] + (has_skip ? mlp_packed_size(nin, nout) : 0);
    return net.packed && B <= mlp_fused_rows(values, has_skip) &&
           (x + sizeof(float) * (size_t)B * nin <= y ||
            y + sizeof(float) * (size_t)B * nout <= x);
  }
  size_t fused_lds() const {
    return sizeof(uint16_t) * kMlpRows *
           ((size_t)mlp_row(nin) + 2 * (size_t)mlp_row(width));
  }
  int init_packed() {
    long o = 0;
    for (int l = 0; l < 5; ++l) {
      net.dims[l] = dims[l];
      if (l < 4) {
        net.woff[l] = woff[l];
        net.boff[l] = boff[l];
      }
      net.poff[l] = o;
      o += l < 4 ? mlp_packed_size(dims[l], dims[l + 1])
                 : mlp_packed_size(nin, nout);
    }
    net.packed = nullptr;
    if (o > kMlpFusedWeights || fused_lds() > 160 * 1024) return FS_OK;
    FS_TRY(packed.alloc(sizeof(uint16_t) * o));
    FS_HIP(hipMemset(packed.p, 0, sizeof(uint16_t) * o));
    FS_HIP(hipFuncSetAttribute((const void *)k_mlp_forward,
                               hipFuncAttributeMaxDynamicSharedMemorySize,
                               160 * 1024));
    net.packed = packed.as<uint16_t>();
    return FS_OK;
  }
  int forward(int B, const float *X, float *Yout) {
    if (fused(B, X, Yout)) {
      hipLaunchKernelGGL(k_mlp_forward, dim3(ceil_div(B, kMlpRows)),
                         dim3(64 * kMlpWaves), fused_lds(), st, B, net,
                         (int)has_skip, mu(), sig(), tau(), params.as<float>(),
                         X, Yout);
      FS_LAUNCHED();
      return FS_OK;
    }
    FS_TRY(forward_n(B, X));
    FS_HIP(hipMemcpyAsync(Yout, Y, sizeof(float) * B * nout,
                          hipMemcpyDeviceToDevice, st));
    hipLaunchKernelGGL(k_scale_out, dim3(ceil_div((long)B * nout, 256)),
                       dim3(256), 0, st, Yout, B, nout, tau());
    FS_LAUNCHED();
    return FS_OK;
  }
  // loss and gradients into grads
  int backward(int B, const float *X, const float *T, float *loss_host) {
    FS_TRY(forward_n(B, X));
    const long n = (long)B * nout;
    const int nblk = ceil_div(n, 256);
    hipLaunchKernelGGL(k_mse_grad, dim3(nblk), dim3(256), 0, st, Y, T, tau(),
                       B, nout, G, Gb, partial);
    if (loss_host)
      hipLaunchKernelGGL(k_sum, dim3(1), dim3(256), 0, st, partial, nblk, lossd);
    float *g = grads.as<float>();
    const uint16_t *W = wbf.as<uint16_t>();
    // layer 3: dW3 = Gb^T H3 (out x width), db3 = colsum(G), dH3 = Gb W3
    float *gcur = G;
    uint16_t *gb = Gb;
    int gcols = nout;
    for (int l = 3; l >= 0; --l) {
      const uint16_t *hin = Hb[l];
      const int in = dims[l], out = dims[l + 1];
      const long ldin = (l == 0) ? nin : width;
      // dW_l(o, i) = sum_b g(b, o) h(b, i)
      gemm(out, in, B, gb, 1, gcols, hin, ldin, 1, EPI_STORE, nullptr,
           g + woff[l], in, nullptr, 0, nullptr, 0);
      hipLaunchKernelGGL(k_colsum, dim3(ceil_div(out, 64)), dim3(1024), 0, st,
                         gcur, B, out, g + boff[l]);
      if (l > 0) {
        // dh(b, i) = sum_o g(b, o) W_l[o][i]; dz = dh * (z_{l-1} > 0)
        uint16_t *gb_next = (gb == Gb) ? Gb2 : Gb;
        float *g_next = (gcur == G) ? Gtmp : G;
        gemm(B, in, out, gb, gcols, 1, W + woff[l], in, 1, EPI_DRELU, nullptr,
             g_next, width, gb_next, width, Zf[l - 1], width);
        gcur = g_next;
        gb = gb_next;
        gcols = width;
      }
    }
    FS_LAUNCHED();
    if (loss_host) {
      float lv;
      FS_HIP(hipMemcpyAsync(&lv, lossd, sizeof(float), hipMemcpyDeviceToHost,
                            st));
      FS_HIP(hipStreamSynchronize(st));
      *loss_host = lv / (float)n;
    }
    return FS_OK;
  }
  int adam(float lr) {
    ++step;
    const float b1 = 0.9f, b2 = 0.999f;
    float c1 = 1.f - std::pow(b1, (float)step), c2 = 1.f - std::pow(b2, (float)step);
    hipLaunchKernelGGL(k_adam, dim3(ceil_div(nparams, 256)), dim3(256), 0, st,
                       params.as<float>(), grads.as<float>(), adam_m.as<float>(),
                       adam_v.as<float>(), nparams, lr, b1, b2, 1e-8f, c1, c2,
                       wbf.as<uint16_t>(), net);
    FS_LAUNCHED();
    return FS_OK;
  }
};

}  // namespace fs

using fs::MlpImpl;

struct fs_mlp {
  MlpImpl impl;
};

namespace fs {
MlpImpl *mlp_impl(fs_mlp *h) { return h ? &h->impl : nullptr; }
int mlp_forward(MlpImpl *m, int B, const float *X, float *Y, hipStream_t st) {
  m->st = st;
  return m->forward(B, X, Y);
}
int mlp_dims(MlpImpl *m, int *nin, int *nout) {
  *nin = m->nin;
  *nout = m->nout;
  return FS_OK;
}
}  // namespace fs

extern "C" int fs_mlp_create(int n_in, int width, int n_out,
                             unsigned long long seed, fs_mlp **out) {
  FS_CHECK(out, FS_ERR_ARG, "null argument");
  *out = nullptr;
  fs_mlp *h = new fs_mlp();
  int rc = h->impl.init(n_in, width, n_out, seed);
  if (rc != FS_OK) {
    h->impl.release();
    delete h;
    return rc;
  }
  *out = h;
  return FS_OK;
}

extern "C" int fs_mlp_destroy(fs_mlp *h) {
  if (!h) return FS_OK;
  (void)hipDeviceSynchronize();
  h->impl.release();
  delete h;
  return FS_OK;
}

extern "C" int fs_mlp_num_params(fs_mlp *h, int *n) {
  FS_CHECK(h && n, FS_ERR_ARG, "null argument");
  *n = (int)h->impl.nparams;
  return FS_OK;
}

extern "C" int fs_mlp_forward(fs_mlp *h, int batch, const float *X, float *Y,
                              void *stream) {
  FS_CHECK(h && X && Y && batch >= 1, FS_ERR_ARG, "bad argument");
  h->impl.st = (hipStream_t)stream;
  return h->impl.forward(batch, X, Y);
}

extern "C" int fs_mlp_train_step(fs_mlp *h, int batch, const float *X,
                                 const float *T, float lr, float *loss,
                                 void *stream) {
  FS_CHECK(h && X && T && batch >= 1 && lr > 0, FS_ERR_ARG, "bad argument");
  h->impl.st = (hipStream_t)stream;
  FS_TRY(h->impl.backward(batch, X, T, loss));
  return h->impl.adam(lr);
}

extern "C" int fs_mlp_gradients(fs_mlp *h, int batch, const float *X,
                                const float *T, float *grad, int n_grad,
                                float *loss) {
  FS_CHECK(h && X && T && grad && batch >= 1, FS_ERR_ARG, "bad argument");
  FS_CHECK(n_grad == h->impl.nparams, FS_ERR_SIZE, "n_grad %d != %ld", n_grad,
           h->impl.nparams);
  h->impl.st = nullptr;
  FS_TRY(h->impl.backward(batch, X, T, loss));
  FS_HIP(hipMemcpy(grad, h->impl.grads.p, sizeof(float) * n_grad,
                   hipMemcpyDeviceToHost));
  return FS_OK;
}

extern "C" int fs_mlp_get_params(fs_mlp *h, float *p, int n) {
  FS_CHECK(h && p && n == h->impl.nparams, FS_ERR_ARG, "bad argument");
  FS_HIP(hipDeviceSynchronize());
  FS_HIP(hipMemcpy(p, h->impl.params.p, sizeof(float) * n,
                   hipMemcpyDeviceToHost));
  return FS_OK;
}

extern "C" int fs_mlp_set_params(fs_mlp *h, const float *p, int n) {
  FS_CHECK(h && p && n == h->impl.nparams, FS_ERR_ARG, "bad argument");
  FS_HIP(hipMemcpy(h->impl.params.p, p, sizeof(float) * n,
                   hipMemcpyHostToDevice));
  h->impl.st = nullptr;
  FS_TRY(h->impl.requantise());
  FS_HIP(hipDeviceSynchronize());
  return FS_OK;
}

extern "C" int fs_mlp_set_skip(fs_mlp *h, const float *S) {
  FS_CHECK(h, FS_ERR_ARG, "null handle");
  MlpImpl &m = h->impl;
  if (!S) {
    m.has_skip = false;
    return FS_OK;
  }
  const long n = (long)m.nout * m.nin;
  fs::dbuf tmp;
  FS_TRY(tmp.alloc(sizeof(float) * n));
  FS_TRY(m.skip.alloc(sizeof(uint16_t) * n));
  int rc = FS_OK;
  if (hipMemcpy(tmp.p, S, sizeof(float) * n, hipMemcpyHostToDevice) !=
      hipSuccess) {
    fs::set_error("copy of the skip map failed");
    rc = FS_ERR_HIP;
  }
  if (rc == FS_OK) {
    hipLaunchKernelGGL(fs::k_to_bf16, dim3(fs::ceil_div(n, 256)), dim3(256), 0,
                       nullptr, tmp.as<float>(), n, m.skip.as<uint16_t>());
    if (m.net.packed)
      hipLaunchKernelGGL(fs::k_pack_skip, dim3(fs::ceil_div(n, 256)), dim3(256), 0,
                         nullptr, m.skip.as<uint16_t>(), m.net);
    if (hipDeviceSynchronize() != hipSuccess) {
      fs::set_error("conversion of the skip map failed");
      rc = FS_ERR_HIP;
    }
  }
  tmp.release();
  if (rc == FS_OK) m.has_skip = true;
  return rc;
}

extern "C" int fs_mlp_set_norm(fs_mlp *h, const float *mu, const float *sigma,
                               const float *tau) {
  FS_CHECK(h && mu && sigma && tau, FS_ERR_ARG, "null argument");
  const int nin = h->impl.nin, nout = h->impl.nout;
  for (int i = 0; i < nin; ++i)
    FS_CHECK(sigma[i] > 0, FS_ERR_ARG, "sigma[%d] must be > 0", i);
  for (int i = 0; i < nout; ++i)
    FS_CHECK(tau[i] > 0, FS_ERR_ARG, "tau[%d] must be > 0", i);
  float *d = h->impl.norm.as<float>();
  FS_HIP(hipMemcpy(d, mu, sizeof(float) * nin, hipMemcpyHostToDevice));
  FS_HIP(hipMemcpy(d + nin, sigma, sizeof(float) * nin, hipMemcpyHostToDevice));
  FS_HIP(hipMemcpy(d + 2 * nin, tau, sizeof(float) * nout,
                   hipMemcpyHostToDevice));
  return FS_OK;
}

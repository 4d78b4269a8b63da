// Kernels of the MLP angle proposer (fp32): forward and backward of dense
// layers, ReLU, mean-squared-error loss and Adam.  No reference counterpart:
// the reference has no learned component; the proposer warm-starts the QAOA
// optimizer of examples/qaoa_maxcut.py:37-87.
//
// Dense layer y = relu(x W^T + b), x [B, in], W [out, in] (row-major).
// All products go through one matrix-core GEMM with strided operand access:
//   C[m][n] = sum_k A(m, k) B(k, n),  A(m, k) = A[m*sam + k*sak],
//                                     B(k, n) = B[k*sbk + n*sbn]
// forward: (x, W^T); input gradient: (dz, W), masked by the layer below's
// ReLU; weight gradient: (dz^T, x), whose row sums of A are the bias gradient.
// Every output element is summed in a fixed order, so results are bitwise
// reproducible.
#include "qfx_common.h"

namespace {

typedef float v16f __attribute__((ext_vector_type(16)));
typedef float v4f __attribute__((ext_vector_type(4)));

constexpr int kTile = 32;                 // C tile per workgroup: 32 x 32
constexpr int kWaves = 8;                 // k blocks are dealt to 8 waves in turn
constexpr int kThreads = 64 * kWaves;
constexpr int kKb = 8;                    // k block: 4 MFMAs of 32x32x2
constexpr int kBatchKb = 4;               // k blocks loaded before the first MFMA

// One k block of one operand: lane (i = l % 32, h = l / 32) holds its row's
// k = 8 kb + 4 h + j, j < 4; MFMA j then sums k = 8 kb + j and 8 kb + 4 + j.
// VEC: the four are one 16-byte load.
template <bool VEC>
__device__ __forceinline__ void load_kb(float (&r)[4], const float* __restrict__ p, long sk,
                                        int k) {
  if constexpr (VEC) {
    const v4f q = *reinterpret_cast<const v4f*>(p + k);
#pragma unroll
    for (int j = 0; j < 4; ++j) r[j] = q[j];
  } else {
#pragma unroll
    for (int j = 0; j < 4; ++j) r[j] = p[(long)(k + j) * sk];
  }
}

// The products of a 256-wide network are far too small to fill the chip (a
// 512 x 256 x 256 product is 67 MFLOP, 0.5 us of matrix work): latency bounds
// them, so a tile is small (128 workgroups there), its K loop is split over
// the workgroup's eight waves with every load of a wave's share in flight,
// and operands come straight from L2 (no staging barrier); the waves' partial
// tiles meet once in LDS.  512 x 256 x 256: 5.6 us, against 45 us with
// 64 x 64 tiles walking K in 16-wide LDS stages (32 workgroups).
template <bool VA, bool VB>
__global__ __launch_bounds__(kThreads) void gemm_kernel(
    float* __restrict__ C, const float* __restrict__ A, const float* __restrict__ Bm, int M,
    int N, int K, long sam, long sak, long sbk, long sbn, const float* __restrict__ bias,
    int relu, const float* __restrict__ mask, float* __restrict__ rowsum) {
  __shared__ float part[kWaves][kTile * (kTile + 1)];
  __shared__ float rpart[kWaves][kTile];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int i = lane & 31, h = lane >> 5;
  const int m0 = blockIdx.y * kTile, n0 = blockIdx.x * kTile;
  // rows and columns past the edge re-read the last one: they only reach
  // outputs that are not stored
  const float* ap = A + (long)(m0 + i < M ? m0 + i : M - 1) * sam;
  const float* bp = Bm + (long)(n0 + i < N ? n0 + i : N - 1) * sbn;
  const int nkb = (K + kKb - 1) / kKb, full = K / kKb;
  v16f acc;
#pragma unroll
  for (int r = 0; r < 16; ++r) acc[r] = 0.0f;
  float rs = 0.0f;
  int kb = w;
  for (; kb + (kBatchKb - 1) * kWaves < full; kb += kBatchKb * kWaves) {
    float a[kBatchKb][4], b[kBatchKb][4];
#pragma unroll
    for (int u = 0; u < kBatchKb; ++u) {
      const int k = (kb + u * kWaves) * kKb + 4 * h;
      load_kb<VA>(a[u], ap, sak, k);
      load_kb<VB>(b[u], bp, sbk, k);
    }
#pragma unroll
    for (int u = 0; u < kBatchKb; ++u)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        rs += a[u][j];
        acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a[u][j], b[u][j], acc, 0, 0, 0);
      }
  }
  for (; kb < nkb; kb += kWaves) {
    const int k = kb * kKb + 4 * h;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const bool in = k + j < K;
      const float a = in ? ap[(long)(k + j) * sak] : 0.0f;
      const float b = in ? bp[(long)(k + j) * sbk] : 0.0f;
      rs += a;
      acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, acc, 0, 0, 0);
    }
  }
  // register r of lane (i, h) is row 8 (r / 4) + 4 h + r % 4 of column i
#pragma unroll
  for (int r = 0; r < 16; ++r)
    part[w][(8 * (r >> 2) + 4 * h + (r & 3)) * (kTile + 1) + i] = acc[r];
  rs += __shfl_xor(rs, 32, 64);
  if (h == 0) rpart[w][i] = rs;
  __syncthreads();
  const int nw = nkb < kWaves ? nkb : kWaves;
  const int col = threadIdx.x & 31, n = n0 + col;
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    const int row = (threadIdx.x >> 5) + 16 * q, m = m0 + row;
    if (m >= M || n >= N) continue;
    float v = 0.0f;
    for (int p = 0; p < nw; ++p) v += part[p][row * (kTile + 1) + col];
    if (bias) v += bias[n];
    if (relu) v = v > 0.0f ? v : 0.0f;
    if (mask) v = mask[(long)m * N + n] > 0.0f ? v : 0.0f;
    C[(long)m * N + n] = v;
  }
  if (rowsum && blockIdx.x == 0 && threadIdx.x < kTile && m0 + (int)threadIdx.x < M) {
    float v = 0.0f;
    for (int p = 0; p < nw; ++p) v += rpart[p][threadIdx.x];
    rowsum[m0 + threadIdx.x] = v;
  }
}

// dz = dy * (y > 0)
__global__ void relu_bwd_kernel(float* __restrict__ dz, const float* __restrict__ dy,
                                const float* __restrict__ y, long len) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < len) dz[i] = y[i] > 0.0f ? dy[i] : 0.0f;
}

// out[n] = sum_b x[b][n], one lane per column, rows in order
__global__ void colsum_kernel(float* __restrict__ out, const float* __restrict__ x, int B, int N) {
  const int n = blockIdx.x * blockDim.x + threadIdx.x;
  if (n >= N) return;
  float s = 0.0f;
  for (int b = 0; b < B; ++b) s += x[(long)b * N + n];
  out[n] = s;
}

// dy = 2 (y - t) / (B N); per-block partial sums of (y - t)^2 / (B N)
__global__ void mse_kernel(float* __restrict__ dy, float* __restrict__ partial,
                           const float* __restrict__ y, const float* __restrict__ t, long len,
                           float scale) {
  __shared__ float red[4];
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  float sq = 0.0f;
  if (i < len) {
    const float d = y[i] - t[i];
    dy[i] = 2.0f * d * scale;
    sq = d * d * scale;
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) sq += __shfl_down(sq, off, 64);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = sq;
  __syncthreads();
  if (threadIdx.x == 0) partial[blockIdx.x] = ((red[0] + red[1]) + red[2]) + red[3];
}

__global__ void sum_kernel(float* __restrict__ out, const float* __restrict__ x, int len) {
  if (threadIdx.x == 0 && blockIdx.x == 0) {
    float s = 0.0f;
    for (int i = 0; i < len; ++i) s += x[i];
    out[0] = s;
  }
}

// The same in one workgroup, up to 32 values a lane: 2.7 us for 512 x 8
// outputs, where two launches took 8.3 us of GPU time.
constexpr int kMseBlock = 1024;
constexpr long kMseOneBlock = 32768;

__global__ __launch_bounds__(kMseBlock) void mse_one_kernel(float* __restrict__ dy,
                                                            float* __restrict__ loss,
                                                            const float* __restrict__ y,
                                                            const float* __restrict__ t, int len,
                                                            float scale) {
  __shared__ float red[kMseBlock / 64];
  float sq = 0.0f;
  for (int i = threadIdx.x; i < len; i += kMseBlock) {
    const float d = y[i] - t[i];
    dy[i] = 2.0f * d * scale;
    sq += d * d * scale;
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) sq += __shfl_down(sq, off, 64);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = sq;
  __syncthreads();
  if (threadIdx.x == 0) {
    float s = 0.0f;
    for (int w = 0; w < kMseBlock / 64; ++w) s += red[w];
    loss[0] = s;
  }
}

__global__ void adam_kernel(float* __restrict__ p, const float* __restrict__ g,
                            float* __restrict__ m, float* __restrict__ v, long len, float lr,
                            float b1, float b2, float eps, float c1, float c2, float wd) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= len) return;
  const float gi = g[i] + wd * p[i];
  const float mi = b1 * m[i] + (1.0f - b1) * gi;
  const float vi = b2 * v[i] + (1.0f - b2) * gi * gi;
  m[i] = mi;
  v[i] = vi;
  p[i] -= lr * (mi / c1) / (sqrtf(vi / c2) + eps);
}

int grid1(long len, int bs) { return (int)((len + bs - 1) / bs); }

}  // namespace

extern "C" {

int qfx_mlp_gemm_fused(void* stream, void* C, const void* A, const void* B, int M, int N, int K,
                       int64_t sam, int64_t sak, int64_t sbk, int64_t sbn, const void* bias,
                       int relu, const void* mask, void* rowsum) {
  if (!C || !A || !B) return qfx::set_error(QFX_EINVAL, "qfx_mlp_gemm: null pointer");
  if (M < 1 || N < 1 || K < 1) return qfx::set_error(QFX_ERANGE, "qfx_mlp_gemm: empty product");
  const dim3 grid((N + kTile - 1) / kTile, (M + kTile - 1) / kTile);
  // four k of a row in one 16-byte load: k contiguous, every row 16-byte
  // aligned
  const bool va = sak == 1 && sam % 4 == 0 && reinterpret_cast<uintptr_t>(A) % 16 == 0;
  const bool vb = sbk == 1 && sbn % 4 == 0 && reinterpret_cast<uintptr_t>(B) % 16 == 0;
  auto kernel = va ? (vb ? gemm_kernel<true, true> : gemm_kernel<true, false>)
                   : (vb ? gemm_kernel<false, true> : gemm_kernel<false, false>);
  hipLaunchKernelGGL(kernel, grid, dim3(kThreads), 0, qfx::as_stream(stream),
                     static_cast<float*>(C), static_cast<const float*>(A),
                     static_cast<const float*>(B), M, N, K, (long)sam, (long)sak, (long)sbk,
                     (long)sbn, static_cast<const float*>(bias), relu,
                     static_cast<const float*>(mask), static_cast<float*>(rowsum));
  return qfx::check_launch("qfx_mlp_gemm");
}

int qfx_mlp_gemm(void* stream, void* C, const void* A, const void* B, int M, int N, int K,
                 int64_t sam, int64_t sak, int64_t sbk, int64_t sbn, const void* bias, int relu) {
  return qfx_mlp_gemm_fused(stream, C, A, B, M, N, K, sam, sak, sbk, sbn, bias, relu, nullptr,
                            nullptr);
}

int qfx_mlp_relu_bwd(void* stream, void* dz, const void* dy, const void* y, int64_t len) {
  if (!dz || !dy || !y) return qfx::set_error(QFX_EINVAL, "qfx_mlp_relu_bwd: null pointer");
  if (len < 1) return QFX_OK;
  hipLaunchKernelGGL(relu_bwd_kernel, dim3(grid1(len, 256)), dim3(256), 0, qfx::as_stream(stream),
                     static_cast<float*>(dz), static_cast<const float*>(dy),
                     static_cast<const float*>(y), (long)len);
  return qfx::check_launch("qfx_mlp_relu_bwd");
}

int qfx_mlp_colsum(void* stream, void* out, const void* x, int B, int N) {
  if (!out || !x) return qfx::set_error(QFX_EINVAL, "qfx_mlp_colsum: null pointer");
  if (B < 1 || N < 1) return qfx::set_error(QFX_ERANGE, "qfx_mlp_colsum: empty input");
  hipLaunchKernelGGL(colsum_kernel, dim3(grid1(N, 256)), dim3(256), 0, qfx::as_stream(stream),
                     static_cast<float*>(out), static_cast<const float*>(x), B, N);
  return qfx::check_launch("qfx_mlp_colsum");
}

int64_t qfx_mlp_mse_workspace(int64_t len) { return ((len + 255) / 256) * (int64_t)sizeof(float); }

int qfx_mlp_mse(void* stream, void* dy, void* loss, const void* y, const void* t, int64_t len,
                void* workspace) {
  if (!dy || !loss || !y || !t || !workspace)
    return qfx::set_error(QFX_EINVAL, "qfx_mlp_mse: null pointer");
  if (len < 1) return qfx::set_error(QFX_ERANGE, "qfx_mlp_mse: empty input");
  hipStream_t s = qfx::as_stream(stream);
  if (len <= kMseOneBlock) {
    hipLaunchKernelGGL(mse_one_kernel, dim3(1), dim3(kMseBlock), 0, s, static_cast<float*>(dy),
                       static_cast<float*>(loss), static_cast<const float*>(y),
                       static_cast<const float*>(t), (int)len, 1.0f / (float)len);
    return qfx::check_launch("qfx_mlp_mse");
  }
  const int nb = grid1(len, 256);
  hipLaunchKernelGGL(mse_kernel, dim3(nb), dim3(256), 0, s, static_cast<float*>(dy),
                     static_cast<float*>(workspace), static_cast<const float*>(y),
                     static_cast<const float*>(t), (long)len, 1.0f / (float)len);
  int rc = qfx::check_launch("qfx_mlp_mse");
  if (rc) return rc;
  hipLaunchKernelGGL(sum_kernel, dim3(1), dim3(64), 0, s, static_cast<float*>(loss),
                     static_cast<const float*>(workspace), nb);
  return qfx::check_launch("qfx_mlp_mse");
}

int qfx_mlp_adam(void* stream, void* params, const void* grads, void* m, void* v, int64_t len,
                 float lr, float beta1, float beta2, float eps, int step, float weight_decay) {
  if (!params || !grads || !m || !v) return qfx::set_error(QFX_EINVAL, "qfx_mlp_adam: null pointer");
  if (step < 1) return qfx::set_error(QFX_EINVAL, "qfx_mlp_adam: step counts from 1");
  if (len < 1) return QFX_OK;
  const float c1 = 1.0f - powf(beta1, (float)step), c2 = 1.0f - powf(beta2, (float)step);
  hipLaunchKernelGGL(adam_kernel, dim3(grid1(len, 256)), dim3(256), 0, qfx::as_stream(stream),
                     static_cast<float*>(params), static_cast<const float*>(grads),
                     static_cast<float*>(m), static_cast<float*>(v), (long)len, lr, beta1, beta2,
                     eps, c1, c2, weight_decay);
  return qfx::check_launch("qfx_mlp_adam");
}

}  // extern "C"

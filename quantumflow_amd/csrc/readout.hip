// Readout kernels: inner product, |psi|, |psi|^2, diagonal expectation,
// all-qubit <Z>, squared norm.
//
// Replace numpybk.inner (quantumflow/backend/numpybk.py:125-128),
// State.probabilities (quantumflow/states.py:113-119), State.expectation
// (quantumflow/states.py:131-147) and QubitVector.norm
// (quantumflow/qubits.py:180-182).  Reductions run in two stages with a fixed
// work assignment (block partials, then one block in a fixed order), so a
// result is bitwise reproducible for a given length.
#include <mutex>
#include <string>

#include "permute_tile.h"
#include "qfx_common.h"

namespace {

constexpr int kBlock = 256;
constexpr int kMaxRedBlocks = 1024;
constexpr int kZChunkBits = 16;  // most bits of a <Z> block's chunk

// Sum `v` over the block; the result is valid in thread 0.
template <int NV>
__device__ __forceinline__ void block_sum(double (&v)[NV], double* lds /*NV*4*/) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
  for (int j = 0; j < NV; ++j) v[j] = wave_sum(v[j]);
  __syncthreads();
  if (lane == 0) {
#pragma unroll
    for (int j = 0; j < NV; ++j) lds[j * 4 + wave] = v[j];
  }
  __syncthreads();
  if (threadIdx.x == 0) {
#pragma unroll
    for (int j = 0; j < NV; ++j) v[j] = ((lds[j * 4] + lds[j * 4 + 1]) + lds[j * 4 + 2]) + lds[j * 4 + 3];
  }
}

int red_blocks(uint64_t len) {
  uint64_t b = (len + kBlock * 4 - 1) / (kBlock * 4);
  if (b > (uint64_t)kMaxRedBlocks) b = kMaxRedBlocks;
  if (b < 1) b = 1;
  return (int)b;
}

// mode 0: sum conj(a) b (complex); 1: sum |a|^2 diag; 2: sum |a|^2
// Bound by the read.  A block takes kRedPer * 256 consecutive elements at a
// time, so that the grid walks memory in order (each lane's loads a grid
// apart instead, a power of two of megabytes, met in the same channels):
// 26 qubits: norm 207 -> 174 us (6.2 TB/s), inner product 456 -> 345 us.
constexpr int kRedPer = 4;

template <int MODE>
__device__ __forceinline__ void red_add(double (&acc)[2], const double2 x, const double2 y) {
  if (MODE == 0) {
    acc[0] = fma(x.x, y.x, acc[0]);
    acc[0] = fma(x.y, y.y, acc[0]);
    acc[1] = fma(x.x, y.y, acc[1]);
    acc[1] = fma(-x.y, y.x, acc[1]);
  } else if (MODE == 1) {
    acc[0] = fma(fma(x.x, x.x, x.y * x.y), y.x, acc[0]);
  } else {
    acc[0] = fma(x.x, x.x, fma(x.y, x.y, acc[0]));
  }
}

template <int MODE>
__global__ __launch_bounds__(kBlock) void reduce_stage1(const double2* __restrict__ a,
                                                       const void* __restrict__ b, uint64_t len,
                                                       double2* __restrict__ partial) {
  __shared__ double lds[2 * 4];
  double acc[2] = {0.0, 0.0};
  auto other = [&](uint64_t i) {
    if (MODE == 0) return static_cast<const double2*>(b)[i];
    if (MODE == 1) return make_double2(static_cast<const double*>(b)[i], 0.0);
    return make_double2(0.0, 0.0);
  };
  constexpr uint64_t kStep = kRedPer * kBlock;
  uint64_t i0 = (uint64_t)blockIdx.x * kStep;
  for (; i0 + kStep <= len; i0 += (uint64_t)gridDim.x * kStep) {
    double2 x[kRedPer], y[kRedPer];
#pragma unroll
    for (int u = 0; u < kRedPer; ++u) x[u] = a[i0 + threadIdx.x + u * kBlock];
#pragma unroll
    for (int u = 0; u < kRedPer; ++u) y[u] = other(i0 + threadIdx.x + u * kBlock);
#pragma unroll
    for (int u = 0; u < kRedPer; ++u) red_add<MODE>(acc, x[u], y[u]);
  }
  for (uint64_t i = i0 + threadIdx.x; i < len && i < i0 + kStep; i += kBlock)
    red_add<MODE>(acc, a[i], other(i));
  block_sum<2>(acc, lds);
  if (threadIdx.x == 0) partial[blockIdx.x] = make_double2(acc[0], acc[1]);
}

// sum conj(a[i]) b[j], bit src[b] of j = bit b of i: the inner product with a
// state whose qubits are ordered otherwise, without writing that state in the
// other order.  Tiles of b are read in its own order and turned in LDS, as by
// permute_tile_kernel.  26 qubits in a random order: 374 us (5.7 TB/s);
// permuting (415 us) and then multiplying (345 us) moves the state twice more.
__global__ __launch_bounds__(kPermBlock) void inner_permuted_stage1(
    const double2* __restrict__ a, const double2* __restrict__ b, uint64_t ntiles,
    double2* __restrict__ partial, PermTile p) {
  __shared__ v2d tile_lds[1 << kPermT];
  __shared__ double lds[2 * 4];
  double acc[2] = {0.0, 0.0};
  const PermLane q = perm_lane(p);
  for (uint64_t tile = blockIdx.x; tile < ntiles; tile += gridDim.x) {
    uint64_t bi, bo;
    perm_bases(p, tile, &bi, &bo);
    v2d y[kPermPer];
    double2 x[kPermPer];
    const v2d* src = reinterpret_cast<const v2d*>(b) + bi + q.in_lane;
#pragma unroll
    for (int u = 0; u < kPermPer; ++u) y[u] = ld_stream(src + q.in_u[u]);
#pragma unroll
    for (int u = 0; u < kPermPer; ++u) x[u] = ld_stream(a + bo + q.out_lane + q.out_u[u]);
#pragma unroll
    for (int u = 0; u < kPermPer; ++u) tile_lds[q.lds_in[u]] = y[u];
    __syncthreads();
#pragma unroll
    for (int u = 0; u < kPermPer; ++u) {
      const v2d z = tile_lds[perm_swz(threadIdx.x + kPermBlock * u)];
      red_add<0>(acc, x[u], make_double2(z.x, z.y));
    }
    __syncthreads();
  }
  block_sum<2>(acc, lds);
  if (threadIdx.x == 0) partial[blockIdx.x] = make_double2(acc[0], acc[1]);
}

// Sums `nparts` partials in a fixed order; writes complex (MODE 0) or real.
template <int MODE>
__global__ __launch_bounds__(kBlock) void reduce_stage2(const double2* __restrict__ partial,
                                                       int nparts, void* __restrict__ result) {
  __shared__ double lds[2 * 4];
  double acc[2] = {0.0, 0.0};
  for (int j = threadIdx.x; j < nparts; j += kBlock) {
    acc[0] += partial[j].x;
    acc[1] += partial[j].y;
  }
  block_sum<2>(acc, lds);
  if (threadIdx.x == 0) {
    if (MODE == 0)
      static_cast<double2*>(result)[0] = make_double2(acc[0], acc[1]);
    else
      static_cast<double*>(result)[0] = acc[0];
  }
}

// partial[blk] = {sum |psi_i|^2 with bit b of i clear, ... with it set}
__global__ __launch_bounds__(kBlock) void bit_prob_stage1(const double2* __restrict__ a,
                                                         uint64_t len, int b,
                                                         double2* __restrict__ partial) {
  __shared__ double lds[2 * 4];
  double acc[2] = {0.0, 0.0};
  const uint64_t stride = (uint64_t)gridDim.x * kBlock;
  for (uint64_t i = (uint64_t)blockIdx.x * kBlock + threadIdx.x; i < len; i += stride) {
    const double2 x = a[i];
    const double p = fma(x.x, x.x, x.y * x.y);
    if ((i >> b) & 1) acc[1] += p;
    else acc[0] += p;
  }
  block_sum<2>(acc, lds);
  if (threadIdx.x == 0) partial[blockIdx.x] = make_double2(acc[0], acc[1]);
}

__global__ __launch_bounds__(kBlock) void abs_kernel(double* __restrict__ out,
                                                    const double2* __restrict__ in, uint64_t len,
                                                    int squared) {
  const uint64_t i = (uint64_t)blockIdx.x * kBlock + threadIdx.x;
  if (i >= len) return;
  const double2 z = in[i];
  out[i] = squared ? fma(z.x, z.x, z.y * z.y) : hypot(z.x, z.y);
}

// <Z> stage 1: block `blk` sums chunk [blk << c, (blk+1) << c).  Element
// i = base + tid + 256 m; bits 0..7 of i are those of tid, bits 8..c-1 those
// of m.  Writes column blk of partial ([1 + kZChunkBits][nblk]): the total and
// S_0 .. S_{c-1}, S_b = sum |psi_i|^2 bit_b(i) over the chunk.  Bound by the
// read: eight elements a lane in flight, whose three bits of m cost a few adds.
// 26 qubits 180 us, 5.9 TB/s (256 us with one load in flight); 20 qubits 20 us with both stages against 73 us, when its
// 16 chunks of 2^16 left the chip idle.
constexpr int kZPer = 8;

__global__ __launch_bounds__(kBlock) void z_stage1(const double2* __restrict__ psi, int c,
                                                  double* __restrict__ partial) {
  __shared__ double lds[(1 + 8 + 8) * 4];
  const uint64_t base = (uint64_t)blockIdx.x << c;
  const int tid = threadIdx.x;
  const int chunk = 1 << c;
  const int mcount = chunk > kBlock ? chunk / kBlock : 1;
  double tot = 0.0;
  double accm[8] = {0, 0, 0, 0, 0, 0, 0, 0};
  for (int m0 = 0; m0 < mcount; m0 += kZPer) {
    double2 z[kZPer];
#pragma unroll
    for (int u = 0; u < kZPer; ++u) {
      const int e = tid + (m0 + u) * kBlock;
      z[u] = e < chunk ? psi[base + e] : make_double2(0.0, 0.0);
    }
    double p[kZPer];
#pragma unroll
    for (int u = 0; u < kZPer; ++u) p[u] = fma(z[u].x, z[u].x, z[u].y * z[u].y);
    const double s13 = p[1] + p[3], s57 = p[5] + p[7], s26 = p[2] + p[6];
    const double odd = s13 + s57;
    const double sum = ((p[0] + p[4]) + s26) + odd;
    tot += sum;
    accm[0] += odd;
    accm[1] += s26 + (p[3] + p[7]);
    accm[2] += (p[4] + p[6]) + s57;
#pragma unroll
    for (int j = 3; j < 8; ++j)
      if ((m0 >> j) & 1) accm[j] += sum;
  }
  double v[17];
  v[0] = tot;
#pragma unroll
  for (int j = 0; j < 8; ++j) v[1 + j] = ((tid >> j) & 1) ? tot : 0.0;
#pragma unroll
  for (int j = 0; j < 8; ++j) v[9 + j] = accm[j];
  block_sum<17>(v, lds);
  if (tid == 0) {
#pragma unroll
    for (int b = 0; b <= kZChunkBits; ++b) partial[(uint64_t)b * gridDim.x + blockIdx.x] = v[b];
  }
}

// <Z> stage 2: block b writes out[n-1-b] = total - 2 S_b; high bits (>= c)
// come from the block index.  Fixed summation order, the same total in every
// block.  26 qubits: 5 us; one block walking the bits in turn took 37 us.
__global__ __launch_bounds__(kBlock) void z_stage2(const double* __restrict__ partial, int nblk,
                                                  int n, int c, double* __restrict__ out) {
  __shared__ double lds[2 * 4];
  const int b = blockIdx.x;
  const double* sb = partial + (uint64_t)(1 + b) * nblk;
  double acc[2] = {0.0, 0.0};
  for (int j = threadIdx.x; j < nblk; j += kBlock) {
    const double t = partial[j];
    acc[0] += t;
    if (b < c) acc[1] += sb[j];
    else if ((j >> (b - c)) & 1) acc[1] += t;
  }
  block_sum<2>(acc, lds);
  if (threadIdx.x == 0) out[n - 1 - b] = acc[0] - 2.0 * acc[1];
}

// Chunk bits of an n-qubit state: about 1024 chunks (four workgroups a CU)
// of 2^11 (eight elements a lane) to 2^16 amplitudes.
int z_chunk_bits(int n) {
  int c = n - 10;
  if (c < 11) c = 11;
  if (c > kZChunkBits) c = kZChunkBits;
  return c < n ? c : n;
}

template <int MODE>
int run_reduce(hipStream_t s, void* result, const void* a, const void* b, int64_t len,
               void* ws, const char* fn) {
  if (!result || !a || !ws || (MODE != 2 && !b))
    return qfx::set_error(QFX_EINVAL, std::string(fn) + ": null pointer");
  if (len < 1) return qfx::set_error(QFX_ERANGE, std::string(fn) + ": empty input");
  const int nb = red_blocks((uint64_t)len);
  auto* part = static_cast<double2*>(ws);
  hipLaunchKernelGGL(reduce_stage1<MODE>, dim3(nb), dim3(kBlock), 0, s,
                     static_cast<const double2*>(a), b, (uint64_t)len, part);
  int rc = qfx::check_launch(fn);
  if (rc) return rc;
  hipLaunchKernelGGL(reduce_stage2<MODE>, dim3(1), dim3(kBlock), 0, s, part, nb, result);
  return qfx::check_launch(fn);
}

}  // namespace

// ---- expectation without a caller workspace --------------------------------
// The block partials of qfx_expect_diag_noalloc live in this file-scope
// device array (16 KiB: one double2 per stage-1 block, at most
// kMaxRedBlocks), which every GPU holds once for the life of the process.
// Host code never passes the array's name to a kernel: in host code it is a
// stand-in, not a device address.  Its address on each device comes from
// hipGetSymbolAddress, taken once per device with that device current.
// Every slot stage 2 reads is written by stage 1 of the same call, so the
// array needs no clearing; calls that overlap on one GPU share it and race.
static __device__ __align__(256) double2 scratch[kMaxRedBlocks];

namespace {

constexpr int kMaxScratchDevices = 64;
std::mutex g_scratch_mu;
void* g_scratch_ptr[kMaxScratchDevices] = {};

int scratch_on_current_device(void** out, const char* fn) {
  int dev = 0;
  int rc = qfx::check_hip(hipGetDevice(&dev), "hipGetDevice");
  if (rc) return rc;
  if (dev < 0 || dev >= kMaxScratchDevices)
    return qfx::set_error(QFX_ERANGE, std::string(fn) + ": device index out of range");
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (!g_scratch_ptr[dev]) {
    void* p = nullptr;
    rc = qfx::check_hip(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)), "hipGetSymbolAddress");
    if (rc) return rc;
    if (!p) return qfx::set_error(QFX_EHIP, std::string(fn) + ": no address for scratch");
    g_scratch_ptr[dev] = p;
  }
  *out = g_scratch_ptr[dev];
  return QFX_OK;
}

}  // namespace

extern "C" {

int qfx_expect_diag_noalloc(void* stream, void* result, const void* psi, const void* diag,
                            int64_t len) {
  if (len > ((int64_t)1 << QFX_MAX_QUBITS))
    return qfx::set_error(QFX_ERANGE,
                          "qfx_expect_diag_noalloc: len exceeds the maximum of 2^34 elements");
  if (!result || !psi || !diag)
    return qfx::set_error(QFX_EINVAL, "qfx_expect_diag_noalloc: null pointer");
  if (len < 1) return qfx::set_error(QFX_ERANGE, "qfx_expect_diag_noalloc: empty input");
  static_assert(sizeof(scratch) == (size_t)kMaxRedBlocks * sizeof(double2),
                "scratch holds one partial per stage-1 block");
  void* ws = nullptr;
  int rc = scratch_on_current_device(&ws, "qfx_expect_diag_noalloc");
  if (rc) return rc;
  return run_reduce<1>(qfx::as_stream(stream), result, psi, diag, len, ws,
                       "qfx_expect_diag_noalloc");
}

int64_t qfx_reduce_workspace_bytes(int64_t len) {
  int64_t z = 16;
  if (len > 1) {
    int n = 0;
    while (((int64_t)1 << n) < len) ++n;
    const int c = z_chunk_bits(n);
    z = ((int64_t)1 << (n - c)) * (1 + kZChunkBits) * (int64_t)sizeof(double);
  }
  const int64_t r = (int64_t)kMaxRedBlocks * (int64_t)sizeof(double2);
  return z > r ? z : r;
}

int qfx_inner(void* stream, void* result, const void* a, const void* b, int64_t len,
              void* workspace) {
  return run_reduce<0>(qfx::as_stream(stream), result, a, b, len, workspace, "qfx_inner");
}

int qfx_inner_permuted(void* stream, void* result, const void* a, const void* b, int n,
                       const int* src_bit, void* workspace) {
  const char* fn = "qfx_inner_permuted";
  if (!result || !a || !b || !src_bit || !workspace)
    return qfx::set_error(QFX_EINVAL, std::string(fn) + ": null pointer");
  if (n < kPermT || n > QFX_MAX_QUBITS)
    return qfx::set_error(QFX_ERANGE, std::string(fn) + ": n out of range");
  int rc = qfx::check_permutation(n, src_bit, fn);
  if (rc) return rc;
  hipStream_t s = qfx::as_stream(stream);
  const uint64_t ntiles = (uint64_t)1 << (n - kPermT);
  const int nb = ntiles < (uint64_t)kMaxRedBlocks ? (int)ntiles : kMaxRedBlocks;
  auto* part = static_cast<double2*>(workspace);
  hipLaunchKernelGGL(inner_permuted_stage1, dim3(nb), dim3(kPermBlock), 0, s,
                     static_cast<const double2*>(a), static_cast<const double2*>(b), ntiles, part,
                     make_perm_tile(n, src_bit));
  rc = qfx::check_launch(fn);
  if (rc) return rc;
  hipLaunchKernelGGL(reduce_stage2<0>, dim3(1), dim3(kBlock), 0, s, part, nb, result);
  return qfx::check_launch(fn);
}

int qfx_expect_diag(void* stream, void* result, const void* psi, const void* diag, int64_t len,
                    void* workspace) {
  return run_reduce<1>(qfx::as_stream(stream), result, psi, diag, len, workspace,
                       "qfx_expect_diag");
}

int qfx_norm2(void* stream, void* result, const void* psi, int64_t len, void* workspace) {
  return run_reduce<2>(qfx::as_stream(stream), result, psi, nullptr, len, workspace, "qfx_norm2");
}

int qfx_qubit_probs(void* stream, void* out, const void* psi, int n, int axis, void* workspace) {
  if (!out || !psi || !workspace) return qfx::set_error(QFX_EINVAL, "qfx_qubit_probs: null pointer");
  if (n < 1 || n > QFX_MAX_QUBITS) return qfx::set_error(QFX_ERANGE, "qfx_qubit_probs: n out of range");
  if (axis < 0 || axis >= n) return qfx::set_error(QFX_EINVAL, "qfx_qubit_probs: axis out of range");
  hipStream_t s = qfx::as_stream(stream);
  const uint64_t len = (uint64_t)1 << n;
  const int nb = red_blocks(len);
  auto* part = static_cast<double2*>(workspace);
  hipLaunchKernelGGL(bit_prob_stage1, dim3(nb), dim3(kBlock), 0, s,
                     static_cast<const double2*>(psi), len, n - 1 - axis, part);
  int rc = qfx::check_launch("qfx_qubit_probs");
  if (rc) return rc;
  hipLaunchKernelGGL(reduce_stage2<0>, dim3(1), dim3(kBlock), 0, s, part, nb, out);
  return qfx::check_launch("qfx_qubit_probs");
}

int qfx_abs(void* stream, void* out, const void* in, int64_t len) {
  if (!out || !in) return qfx::set_error(QFX_EINVAL, "qfx_abs: null pointer");
  if (len < 1) return QFX_OK;
  hipLaunchKernelGGL(abs_kernel, dim3((unsigned)((len + kBlock - 1) / kBlock)), dim3(kBlock), 0,
                     qfx::as_stream(stream), static_cast<double*>(out),
                     static_cast<const double2*>(in), (uint64_t)len, 0);
  return qfx::check_launch("qfx_abs");
}

int qfx_abs2(void* stream, void* out, const void* in, int64_t len) {
  if (!out || !in) return qfx::set_error(QFX_EINVAL, "qfx_abs2: null pointer");
  if (len < 1) return QFX_OK;
  hipLaunchKernelGGL(abs_kernel, dim3((unsigned)((len + kBlock - 1) / kBlock)), dim3(kBlock), 0,
                     qfx::as_stream(stream), static_cast<double*>(out),
                     static_cast<const double2*>(in), (uint64_t)len, 1);
  return qfx::check_launch("qfx_abs2");
}

int qfx_expect_z(void* stream, void* out, const void* psi, int n, void* workspace) {
  if (!out || !psi || !workspace) return qfx::set_error(QFX_EINVAL, "qfx_expect_z: null pointer");
  if (n < 1 || n > QFX_MAX_QUBITS) return qfx::set_error(QFX_ERANGE, "qfx_expect_z: n out of range");
  hipStream_t s = qfx::as_stream(stream);
  const int c = z_chunk_bits(n);
  const uint64_t nblk = (uint64_t)1 << (n - c);
  auto* part = static_cast<double*>(workspace);
  hipLaunchKernelGGL(z_stage1, dim3((unsigned)nblk), dim3(kBlock), 0, s,
                     static_cast<const double2*>(psi), c, part);
  int rc = qfx::check_launch("qfx_expect_z");
  if (rc) return rc;
  hipLaunchKernelGGL(z_stage2, dim3(n), dim3(kBlock), 0, s, part, (int)nblk, n, c,
                     static_cast<double*>(out));
  return qfx::check_launch("qfx_expect_z");
}

}  // extern "C"

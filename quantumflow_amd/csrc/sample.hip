// Sampling the computational basis from |psi|^2 on the device.
//
// Replaces the host-side numpy draws of State.sample / State.measure
// (quantumflow/states.py:121-129 and :149-160), which copy all 2^n probabilities
// to the host: here the probabilities never leave HBM.
//
//   1. chunk sums: S_c = sum of |psi_i|^2 over chunk c (2^cb amplitudes,
//      cb = min(10, n)), in a fixed order;
//   2. exclusive prefix P_c over the chunk sums, P_nchunks = total, in a
//      fixed order (segments of 1024 chunks, then the segments in turn);
//   3. per sample t: u = U(seed, t) * total with U a SplitMix64 stream
//      (Steele, Lea, Flood, "Fast splittable pseudorandom number generators",
//      OOPSLA 2014) mapped to [0, 1); binary search for the chunk with
//      P_c <= u < P_c+1, then for the first index of the chunk whose running
//      sum exceeds u - P_c: the chunk is 64 segments of up to 16 amplitudes,
//      R_l the prefix of the segment sums (a wave-wide scan) and the running
//      sum inside segment l starts at R_(l-1).  Indices with probability 0
//      are never drawn.
// Step 3 has two forms with the same arithmetic, hence the same draws: few
// draws scan their own chunk, one wave each (sample_kernel); many draws share
// a table of every R_l that step 1 writes on the way (sample_table_kernel).
// Results depend only on (psi, seed, trials): bitwise reproducible.
#include "qfx_common.h"

namespace {

constexpr int kMaxChunkBits = 10;
constexpr int kScanBlock = 1024;

__device__ __forceinline__ double uniform01(uint64_t seed, uint64_t t) {
  uint64_t z = seed + (t + 1) * 0x9E3779B97F4A7C15ull;
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  z ^= z >> 31;
  return (double)(z >> 11) * 0x1.0p-53;
}

// Inclusive prefix over the wave's 64 lanes; segment l covers [previous
// lane's prefix, own prefix), so the segments tile the chunk with no gap or
// overlap.
__device__ __forceinline__ double segment_prefix(double mine, int lane) {
  double incl = mine;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const double o = __shfl_up(incl, d, 64);
    if (lane >= d) incl += o;
  }
  return incl;
}

// |psi|^2 sums of chunks of 2^cb <= 1024 amplitudes, one wave per chunk (the
// order of a 256-lane sum: four strided accumulators a lane, summed over the
// wave and then across the four).  With TAB also the chunk's segment prefixes
// R_0..R_63 into tab: 8 bytes per 16 amplitudes, 1/32 of what is read.
// Bound by the read of psi: a wave holds a whole chunk in flight (16 loads a
// lane) and meets no barrier.  One draw in all (this kernel and the prefix) at
// 28 qubits, 4 GiB: 711 us, 6.0 TB/s (1255 us with a 256-lane workgroup and
// two barriers per chunk and a one-workgroup prefix); TAB adds 71 us there
// and 3 us at 24 qubits.
constexpr int kSumWaves = 4;
constexpr int kSegs = 64;                       // segments per chunk
constexpr int kSegMax = 16;                     // amplitudes per segment
constexpr int kSegPad = kSegMax + 1;            // LDS stride: lanes on different banks

template <bool TAB>
__global__ __launch_bounds__(64 * kSumWaves) void chunk_sum_kernel(double* __restrict__ sums,
                                                                  double* __restrict__ tab,
                                                                  const double2* __restrict__ psi,
                                                                  int cb, uint64_t nchunks) {
  __shared__ double q_lds[TAB ? kSumWaves : 1][TAB ? kSegs * kSegPad : 1];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const uint64_t c = (uint64_t)blockIdx.x * kSumWaves + wave;
  if (c >= nchunks) return;                     // whole waves; no barrier below
  const int len = 1 << cb;
  const int sh = cb > 6 ? cb - 6 : 0;           // log2 amplitudes per segment
  const double2* p = psi + (c << cb);
  double2 v[16];
#pragma unroll
  for (int j = 0; j < 16; ++j) {
    const int i = lane + 64 * j;
    v[j] = i < len ? p[i] : make_double2(0.0, 0.0);
  }
  double acc[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
  for (int j = 0; j < 16; ++j)                  // element 64 (w + 4 m) + lane
    acc[j & 3] = fma(v[j].x, v[j].x, fma(v[j].y, v[j].y, acc[j & 3]));
#pragma unroll
  for (int w = 0; w < 4; ++w) acc[w] = wave_sum(acc[w]);
  if (lane == 0) sums[c] = (acc[0] + acc[1]) + (acc[2] + acc[3]);
  if constexpr (TAB) {
    double* q = q_lds[wave];
#pragma unroll
    for (int j = 0; j < 16; ++j) {
      const int i = lane + 64 * j;
      if (i < len)
        q[(i >> sh) * kSegPad + (i & ((1 << sh) - 1))] = fma(v[j].x, v[j].x, v[j].y * v[j].y);
    }
    // the wave's own LDS writes, read by other lanes of the same wave
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    double mine = 0.0;
#pragma unroll
    for (int k = 0; k < kSegMax; ++k)
      if (k < (1 << sh) && (lane << sh) + k < len) mine += q[lane * kSegPad + k];
    tab[c * kSegs + lane] = segment_prefix(mine, lane);
  }
}

// Prefix of the chunk sums in segments of kScanBlock chunks: each segment's
// inclusive scan (Hillis-Steele in LDS, two buffers, one barrier a step) into
// pre[1 ..], its total into seg.
__global__ __launch_bounds__(kScanBlock) void prefix_segments_kernel(
    double* __restrict__ pre, double* __restrict__ seg, const double* __restrict__ sums,
    uint64_t nchunks) {
  __shared__ double buf[2][kScanBlock];
  const int t = threadIdx.x;
  const uint64_t i = (uint64_t)blockIdx.x * kScanBlock + t;
  buf[0][t] = i < nchunks ? sums[i] : 0.0;
  __syncthreads();
  int cur = 0;
  for (int d = 1; d < kScanBlock; d <<= 1) {
    buf[cur ^ 1][t] = t >= d ? buf[cur][t] + buf[cur][t - d] : buf[cur][t];
    cur ^= 1;
    __syncthreads();
  }
  if (i < nchunks) pre[i + 1] = buf[cur][t];
  if (i == 0) pre[0] = 0.0;
  if (t == kScanBlock - 1) seg[blockIdx.x] = buf[cur][t];
}

// Adds to segment b the totals of the segments before it, summed in order
// (a serial chain of b adds, at most 2^14, out of LDS).
__global__ __launch_bounds__(kScanBlock) void prefix_carry_kernel(double* __restrict__ pre,
                                                                  const double* __restrict__ seg,
                                                                  uint64_t nchunks) {
  __shared__ double part[kScanBlock];
  __shared__ double carry;
  const unsigned nb = blockIdx.x;
  if (threadIdx.x == 0) carry = 0.0;
  for (unsigned s0 = 0; s0 < nb; s0 += kScanBlock) {
    __syncthreads();
    if (s0 + threadIdx.x < nb) part[threadIdx.x] = seg[s0 + threadIdx.x];
    __syncthreads();
    if (threadIdx.x == 0) {
      double c = carry;
      const unsigned m = nb - s0 < (unsigned)kScanBlock ? nb - s0 : (unsigned)kScanBlock;
      for (unsigned j = 0; j < m; ++j) c += part[j];
      carry = c;
    }
  }
  __syncthreads();
  const uint64_t i = (uint64_t)nb * kScanBlock + threadIdx.x;
  if (i < nchunks) pre[i + 1] = carry + pre[i + 1];
}

// u of draw t and the largest chunk c in [0, nchunks) with pre[c] <= u.
__device__ __forceinline__ uint64_t draw_chunk(const double* __restrict__ pre, uint64_t nchunks,
                                               uint64_t seed, int64_t t, double* target) {
  const double total = pre[nchunks];
  double u = uniform01(seed, (uint64_t)t) * total;
  if (u >= total) u = nextafter(total, 0.0);
  uint64_t lo = 0, hi = nchunks - 1;
  while (lo < hi) {
    const uint64_t mid = (lo + hi + 1) >> 1;
    if (pre[mid] <= u) lo = mid;
    else hi = mid - 1;
  }
  *target = u - pre[lo];
  return lo;
}

// one wave per sample, 4 samples per workgroup
__global__ __launch_bounds__(256) void sample_kernel(int64_t* __restrict__ out,
                                                     const double2* __restrict__ psi,
                                                     const double* __restrict__ pre,
                                                     uint64_t nchunks, int cb, int64_t trials,
                                                     uint64_t seed) {
  const int lane = threadIdx.x & 63;
  const int64_t t = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (t >= trials) return;   // uniform per wave
  double target;
  const uint64_t lo = draw_chunk(pre, nchunks, seed, t, &target);
  const int len = 1 << cb;
  const int per = len >= 64 ? len / 64 : 1;      // contiguous amplitudes per lane
  const double2* p = psi + (lo << cb);
  double pr[16];
  double mine = 0.0;
#pragma unroll
  for (int k = 0; k < 16; ++k) {
    const int i = lane * per + k;
    double q = 0.0;
    if (k < per && i < len) {
      const double2 v = p[i];
      q = fma(v.x, v.x, v.y * v.y);
    }
    pr[k] = q;
    mine += q;
  }
  const double incl = segment_prefix(mine, lane);
  double excl = __shfl_up(incl, 1, 64);
  if (lane == 0) excl = 0.0;
  // the one lane whose interval holds the target claims the first index
  // whose running sum passes it (its last nonzero index if rounding leaves
  // the running sum short of the target)
  int found = -1;
  if (mine > 0.0 && excl <= target && target < incl) {
    double run = excl;
    int last = -1;
#pragma unroll
    for (int k = 0; k < 16; ++k) {
      if (k < per && pr[k] > 0.0) {
        run += pr[k];
        last = lane * per + k;
        if (found < 0 && run > target) found = last;
      }
    }
    if (found < 0) found = last;
  }
  unsigned long long claim = found >= 0 ? (unsigned long long)found : ~0ull;
  for (int d = 32; d > 0; d >>= 1) {
    const unsigned long long o = __shfl_xor(claim, d, 64);
    claim = o < claim ? o : claim;
  }
  // no claim: the target lies at or above the wave's own chunk total
  // (rounding between the two summation orders); take the chunk's last
  // nonzero index
  if (claim == ~0ull) {
    long long last = -1;
#pragma unroll
    for (int k = 0; k < 16; ++k)
      if (k < per && pr[k] > 0.0) last = lane * per + k;
    for (int d = 32; d > 0; d >>= 1) {
      const long long o = __shfl_xor(last, d, 64);
      last = o > last ? o : last;
    }
    claim = (unsigned long long)(last >= 0 ? last : 0);
  }
  if (lane == 0) out[t] = (int64_t)((lo << cb) | claim);
}

// A draw whose segment cannot be had by bisection alone: its target lies at
// or above the chunk's last prefix, or in a gap that rounding left in front of
// a segment without amplitudes.  Takes the first segment that holds the
// target and an amplitude, else the chunk's last amplitude (as sample_kernel).
__device__ __noinline__ int draw_slow(const double2* p, const double* r, double target, int len,
                                      int per) {
  double excl = 0.0;
  for (int l = 0; l < kSegs && l * per < len; ++l) {
    const double incl = r[l];
    if (excl <= target && target < incl) {
      double run = excl;
      int last = -1;
      for (int k = l * per; k < (l + 1) * per; ++k) {
        const double2 v = p[k];
        const double q = fma(v.x, v.x, v.y * v.y);
        if (!(q > 0.0)) continue;
        run += q;
        last = k;
        if (run > target) return k;
      }
      if (last >= 0) return last;
    }
    excl = incl;
  }
  for (int k = len - 1; k > 0; --k) {
    const double2 v = p[k];
    if (fma(v.x, v.x, v.y * v.y) > 0.0) return k;
  }
  return 0;
}

// Draws from the table of segment prefixes: one draw per lane bisects the
// chunks (pre) and its chunk's 64 prefixes (tab), then each quarter wave in
// turn fetches a draw's segment (256 contiguous bytes) and leaves its
// |psi|^2 in LDS, where the draw's own lane walks them.  A draw reads about
// 1 KiB instead of its 16 KiB chunk, and 64 draws share a wave's latency:
// 2^20 draws of 24 qubits take 115 us (one wave per draw: 4657 us).
__global__ __launch_bounds__(64) void sample_table_kernel(int64_t* __restrict__ out,
                                                          const double2* __restrict__ psi,
                                                          const double* __restrict__ pre,
                                                          const double* __restrict__ tab,
                                                          uint64_t nchunks, int cb,
                                                          int64_t trials, uint64_t seed) {
  __shared__ double q_lds[64 * kSegPad];
  const int lane = threadIdx.x;
  const int64_t t = (int64_t)blockIdx.x * 64 + lane;
  const bool live = t < trials;
  const int len = 1 << cb;
  const int sh = cb > 6 ? cb - 6 : 0, per = 1 << sh;
  double target = 0.0;
  // lanes past the last draw follow draw 0: no lane leaves the fetch below
  const uint64_t c = draw_chunk(pre, nchunks, seed, live ? t : 0, &target);
  const double* r = tab + c * kSegs;
  // first prefix above the target: r[lo] <= target < r[hi]
  int lo = -1, hi = kSegs - 1;
  const bool above = !(target < r[hi]);
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (target < r[mid]) hi = mid;
    else lo = mid;
  }
  double run = hi > 0 ? r[hi - 1] : 0.0;
  // segments past a short chunk's end hold nothing; slow below, but in range
  const int seg = (hi << sh) < len ? hi : 0;
  const uint64_t first = (c << cb) + ((uint64_t)seg << sh);
  const int g = lane >> 4, k = lane & 15;
  double2 v[16];
#pragma unroll
  for (int it = 0; it < 16; ++it) {
    const uint64_t f = __shfl((unsigned long long)first, it * 4 + g, 64);
    v[it] = k < per ? psi[f + k] : make_double2(0.0, 0.0);
  }
#pragma unroll
  for (int it = 0; it < 16; ++it)
    q_lds[(it * 4 + g) * kSegPad + k] = fma(v[it].x, v[it].x, v[it].y * v[it].y);
  __syncthreads();
  if (!live) return;
  int found = -1, last = -1;
#pragma unroll
  for (int j = 0; j < kSegMax; ++j) {
    const double q = q_lds[lane * kSegPad + j];
    if (q > 0.0) {
      run += q;
      last = j;
      if (found < 0 && run > target) found = j;
    }
  }
  if (found < 0) found = last;
  if (above || found < 0 || seg != hi)
    out[t] = (int64_t)((c << cb) | (uint64_t)draw_slow(psi + (c << cb), r, target, len, per));
  else
    out[t] = (int64_t)(first + (uint64_t)found);
}

__global__ __launch_bounds__(256) void histogram_kernel(unsigned long long* __restrict__ counts,
                                                        const int64_t* __restrict__ idx,
                                                        int64_t m) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i < m) atomicAdd(counts + idx[i], 1ull);
}

int chunk_bits(int n) { return n < kMaxChunkBits ? n : kMaxChunkBits; }

uint64_t scan_segments(uint64_t nchunks) { return (nchunks + kScanBlock - 1) / kScanBlock; }

// The segment table: 2^(n-1) bytes (512 MiB at 30 qubits, the largest size
// that keeps one).
constexpr int kMaxTableQubits = 30;

// Draws from which the table pays.  Filling it adds a write of 2^(n-1) bytes
// to the sums (3, 15 and 71 us at 24, 26 and 28 qubits); without it each draw
// reads its 16 KiB chunk (2048 draws +8 us at 24 qubits, 4096 +26 us at 26,
// 8192 +112 us at 28).  Below 24 qubits the two are level up to about 2000
// draws.
int64_t table_trials(int n) { return n > 25 ? (int64_t)1 << (n - 15) : 1024; }

bool uses_table(int n, int64_t trials) {
  return n <= kMaxTableQubits && trials >= table_trials(n);
}

}  // namespace

extern "C" {

int64_t qfx_sample_workspace_bytes_for(int n, int64_t trials) {
  if (n < 1 || n > QFX_MAX_QUBITS) return 0;
  const uint64_t nchunks = (uint64_t)1 << (n - chunk_bits(n));
  const uint64_t table = uses_table(n, trials) ? nchunks * kSegs : 0;
  return (int64_t)(sizeof(double) * (2 * nchunks + 1 + scan_segments(nchunks) + table));
}

int64_t qfx_sample_workspace_bytes(int n) {
  return qfx_sample_workspace_bytes_for(n, INT64_MAX);
}

int qfx_sample(void* stream, int64_t* out, const void* psi, int n, int64_t trials,
               uint64_t seed, void* ws) {
  if (n < 1 || n > QFX_MAX_QUBITS) return qfx::set_error(QFX_ERANGE, "qfx_sample: n out of range");
  if (trials < 0) return qfx::set_error(QFX_EINVAL, "qfx_sample: negative trials");
  if (trials == 0) return QFX_OK;
  if (!out || !psi || !ws) return qfx::set_error(QFX_EINVAL, "qfx_sample: null pointer");
  hipStream_t s = qfx::as_stream(stream);
  const int cb = chunk_bits(n);
  const uint64_t nchunks = (uint64_t)1 << (n - cb);
  const uint64_t nseg = scan_segments(nchunks);
  double* sums = static_cast<double*>(ws);
  double* pre = sums + nchunks;
  double* seg = pre + nchunks + 1;
  double* tab = seg + nseg;
  const bool table = uses_table(n, trials);
  auto* st = static_cast<const double2*>(psi);
  const dim3 sgrid((unsigned)((nchunks + kSumWaves - 1) / kSumWaves)), sblock(64 * kSumWaves);
  if (table)
    hipLaunchKernelGGL(chunk_sum_kernel<true>, sgrid, sblock, 0, s, sums, tab, st, cb, nchunks);
  else
    hipLaunchKernelGGL(chunk_sum_kernel<false>, sgrid, sblock, 0, s, sums, tab, st, cb, nchunks);
  int rc = qfx::check_launch("chunk_sum_kernel");
  if (rc) return rc;
  hipLaunchKernelGGL(prefix_segments_kernel, dim3((unsigned)nseg), dim3(kScanBlock), 0, s, pre,
                     seg, sums, nchunks);
  rc = qfx::check_launch("prefix_segments_kernel");
  if (rc) return rc;
  if (nseg > 1) {
    hipLaunchKernelGGL(prefix_carry_kernel, dim3((unsigned)nseg), dim3(kScanBlock), 0, s, pre, seg,
                       nchunks);
    rc = qfx::check_launch("prefix_carry_kernel");
    if (rc) return rc;
  }
  if (table) {
    const uint64_t blocks = ((uint64_t)trials + 63) / 64;
    hipLaunchKernelGGL(sample_table_kernel, dim3((unsigned)blocks), dim3(64), 0, s, out, st, pre,
                       tab, nchunks, cb, trials, seed);
    return qfx::check_launch("sample_table_kernel");
  }
  const uint64_t blocks = ((uint64_t)trials + 3) / 4;
  hipLaunchKernelGGL(sample_kernel, dim3((unsigned)blocks), dim3(256), 0, s, out, st, pre, nchunks,
                     cb, trials, seed);
  return qfx::check_launch("sample_kernel");
}

int qfx_histogram(void* stream, int64_t* counts, const int64_t* idx, int64_t m, int n) {
  if (n < 1 || n > QFX_MAX_QUBITS) return qfx::set_error(QFX_ERANGE, "qfx_histogram: n out of range");
  if (m < 0) return qfx::set_error(QFX_EINVAL, "qfx_histogram: negative count");
  if (m == 0) return QFX_OK;
  if (!counts || !idx) return qfx::set_error(QFX_EINVAL, "qfx_histogram: null pointer");
  hipStream_t s = qfx::as_stream(stream);
  const uint64_t blocks = ((uint64_t)m + 255) / 256;
  hipLaunchKernelGGL(histogram_kernel, dim3((unsigned)blocks), dim3(256), 0, s,
                     reinterpret_cast<unsigned long long*>(counts), idx, m);
  return qfx::check_launch("histogram_kernel");
}

}  // extern "C"

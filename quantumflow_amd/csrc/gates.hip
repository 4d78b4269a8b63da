// Per-gate state-vector kernels (the plain, one-launch-per-gate path).
//
// Replaces numpybk.tensormul (quantumflow/backend/numpybk.py:159-214) as
// called from Gate.run (quantumflow/ops.py:161-166): out = G applied to the
// axes `targets` of in.  Every kernel assigns one amplitude group (the 2^k
// amplitudes that differ only in the target bits) to one work item, so the
// 16-byte complex128 loads of consecutive lanes are consecutive in memory
// whenever the lowest index bits are not targets, and out == in is safe.
// Amplitudes are streamed with nontemporal loads and stores (each is
// touched once per gate), except where a target lies inside a 128-byte line
// (below).
#include <cmath>
#include <cstring>

#include "permute_tile.h"
#include "qfx_common.h"

namespace {

constexpr int kBlock = 256;
constexpr int kCus = 256;

template <int K>
struct DenseArg {
  double2 m[1 << (2 * K)];   // row-major, row = output
  uint64_t off[1 << K];      // address offset of gate-local index r
  int sorted[K];             // target bits ascending
};

// groups per thread: keep ~8 amplitude loads in flight per lane
template <int K>
constexpr int groups_per_thread() { return K == 1 ? 4 : (K == 2 ? 2 : 1); }

// A target below bit 3 leaves each load and store instruction a part of its
// 128-byte lines (8 amplitudes); the rest follows in the lane's next ones.
// Nontemporal, every part moved its line to and from memory again; through
// the caches the parts meet there.  26 qubits (2 GiB read and written): RX on
// bit 0 3.34 -> 5.54 TB/s, X 2.82 -> 5.54, CNOT on bits 0 and 1 1.15 -> 4.66;
// from bit 3 up nontemporal streams 6.0-6.4 TB/s.
constexpr int kLineBits = 3;

template <bool NT>
__device__ __forceinline__ double2 ld_amp(const double2* p) {
  if constexpr (NT) return ld_stream(p);
  else return *p;
}
template <bool NT>
__device__ __forceinline__ void st_amp(double2* p, double2 v) {
  if constexpr (NT) st_stream(p, v);
  else *p = v;
}

template <int K, int G, bool NT>
__global__ __launch_bounds__(kBlock) void dense_kernel(double2* out, const double2* in,
                                                      uint64_t ngroups, DenseArg<K> a) {
  constexpr int D = 1 << K;
  const uint64_t g0 = (uint64_t)blockIdx.x * (kBlock * G) + threadIdx.x;
  double2 v[G][D];
  uint64_t base[G];
#pragma unroll
  for (int u = 0; u < G; ++u) {
    const uint64_t g = g0 + (uint64_t)u * kBlock;
    base[u] = insert_zeros<K>(g, a.sorted);
    if (g < ngroups) {
#pragma unroll
      for (int r = 0; r < D; ++r) v[u][r] = ld_amp<NT>(in + base[u] + a.off[r]);
    }
  }
#pragma unroll
  for (int u = 0; u < G; ++u) {
    const uint64_t g = g0 + (uint64_t)u * kBlock;
    if (g < ngroups) {
#pragma unroll
      for (int r = 0; r < D; ++r) {
        double2 acc = make_double2(0.0, 0.0);
#pragma unroll
        for (int c = 0; c < D; ++c) cmac(acc, a.m[r * D + c], v[u][c]);
        st_amp<NT>(out + base[u] + a.off[r], acc);
      }
    }
  }
}

// Rows of a diagonal or monomial gate: out row r <- phase[r] * in row src[r].
struct SparseArg {
  uint64_t off[32];     // address offset of output row r
  uint64_t srcoff[32];  // address offset of the source row of r
  double2 ph[32];       // phase of row r
  uint32_t active;      // rows written (all rows out of place)
  uint32_t has_phase;   // rows whose phase is not exactly 1
  int sorted[5];
};

// ALL: every row is written (out of place), so the loads are issued together
// (CCNOT at 25 qubits 493 -> 292 us on bit 0); else the rows of `active`
// alone, each behind a uniform branch.
template <int K, int G, bool ALL, bool NT>
__global__ __launch_bounds__(kBlock) void sparse_kernel(double2* out, const double2* in,
                                                       uint64_t ngroups, SparseArg a) {
  constexpr int D = 1 << K;
  const uint64_t g0 = (uint64_t)blockIdx.x * (kBlock * G) + threadIdx.x;
  double2 v[G][D];
  uint64_t base[G];
#pragma unroll
  for (int u = 0; u < G; ++u) {
    const uint64_t g = g0 + (uint64_t)u * kBlock;
    base[u] = insert_zeros<K>(g, a.sorted);
    if (g < ngroups) {
#pragma unroll
      for (int r = 0; r < D; ++r)
        if (ALL || (a.active & (1u << r))) v[u][r] = ld_amp<NT>(in + base[u] + a.srcoff[r]);
    }
  }
#pragma unroll
  for (int u = 0; u < G; ++u) {
    const uint64_t g = g0 + (uint64_t)u * kBlock;
    if (g < ngroups) {
#pragma unroll
      for (int r = 0; r < D; ++r) {
        if (ALL || (a.active & (1u << r))) {
          const double2 x = (a.has_phase & (1u << r)) ? cmul_fma(a.ph[r], v[u][r]) : v[u][r];
          st_amp<NT>(out + base[u] + a.off[r], x);
        }
      }
    }
  }
}

// Dense gate of up to 3 qubits with the matrix in device memory; one output
// amplitude per lane.  Needs out != in.  The 2^k column offsets are built in LDS.
struct DevTargets {
  int t[QFX_MAX_DENSE_K];  // bit of gate qubit j (MSB first)
};

__global__ __launch_bounds__(kBlock) void dense_dev_kernel(double2* __restrict__ out,
                                                          const double2* __restrict__ in,
                                                          uint64_t len, int k, DevTargets tg,
                                                          const double2* __restrict__ m) {
  extern __shared__ uint64_t s_off[];
  const int D = 1 << k;
  uint64_t tmask = 0;
  for (int j = 0; j < k; ++j) tmask |= (uint64_t)1 << tg.t[j];
  for (int c = threadIdx.x; c < D; c += kBlock) {
    uint64_t off = 0;
    for (int j = 0; j < k; ++j)
      if ((c >> (k - 1 - j)) & 1) off |= (uint64_t)1 << tg.t[j];
    s_off[c] = off;
  }
  __syncthreads();
  const uint64_t i = (uint64_t)blockIdx.x * kBlock + threadIdx.x;
  if (i >= len) return;
  unsigned r = 0;
  for (int j = 0; j < k; ++j) r = (r << 1) | (unsigned)((i >> tg.t[j]) & 1);
  const uint64_t base = i & ~tmask;
  double2 acc = make_double2(0.0, 0.0);
  const double2* row = m + (uint64_t)r * D;
  for (int c = 0; c < D; ++c) cmac(acc, row[c], in[base + s_off[c]]);
  out[i] = acc;
}

// Dense gates of 4 to 12 qubits on the matrix cores: Y = M X with X the
// 2^k x 2^(n-k) matrix of the state's amplitude groups, in complex products of
// four v_mfma_f64_16x16x4f64 each (operand layout: lane l holds A[l%16][l/16],
// B[l/16][l%16] and, in register j, D[4j + l/16][l%16]).
//
// A workgroup computes R gate rows of C groups (R = 2^k up to 64, so gates of
// up to 6 qubits read the state once) and walks the gate's columns 16 at a
// time; the chunk of X and M for the next step is in flight while the current
// one is multiplied out of LDS.  Both matrices are indexed with the targets in
// ascending order, so that a chunk holds the four lowest targets together
// with the C lowest groups: its loads run over contiguous memory whichever
// bits those are (M's rows and columns are permuted to match).  Arithmetic is
// 8 2^k flops an amplitude: memory bounds gates of 4 and 5 qubits, the matrix
// cores those from 7 on.  8 qubits of 20: 54 us, 39 TFLOP/s (one output
// amplitude a lane: 250 us on high bits, 564 us on low ones); 10 of 24 qubits
// 2.3 ms, 60 TFLOP/s (21.3 ms); 4 of 24 qubits 107-133 us, 4.0-5.0 TB/s
// (383-653 us).
struct GemmArg {
  int k;
  int epos[11];               // chunk element bit t -> state index bit
  int eslot[11];              //                     -> bit of (c << log2 C | g)
  unsigned einvalid;          // element bits past the state's groups
  int gbits;                  // group bits inside a tile (log2 C unless n-k is less)
  int gpos[7];                // their index bits
  int sorted[QFX_MAX_DENSE_K];   // targets ascending
  int mbit[QFX_MAX_DENSE_K];     // bit j of the ascending order -> matrix index bit
  int nrest;
  int rest[QFX_MAX_QUBITS];   // index bits of the tile number
};

typedef double v4d __attribute__((ext_vector_type(4)));
constexpr int kKc = 16;       // gate columns per step

template <int R, int C>
__global__ __launch_bounds__(kBlock) void dense_mfma_kernel(double2* __restrict__ out,
                                                           const double2* __restrict__ in,
                                                           unsigned ntiles, GemmArg a,
                                                           const double2* __restrict__ m) {
  constexpr int kLc = C == 128 ? 7 : 6;
  constexpr int NX = kKc * C / kBlock, NM = kKc * R / kBlock;
  constexpr int WR = R < 32 ? R : 32, kRowWaves = R / WR;
  constexpr int WC = C * kRowWaves / 4;               // one wave: WR x WC
  constexpr int RB = WR / 16, CB = WC / 16;
  __shared__ v2d xs[kKc * C], ms[kKc * R];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int q = lane >> 4, col = lane & 15;
  const int D = 1 << a.k, nrt = D / R;
  // tiles that share their groups follow each other on one XCD (blocks are
  // dealt to the 8 XCDs in turn)
  unsigned ct, rt;
  if ((ntiles & 7u) == 0) {
    ct = (blockIdx.x / (8u * nrt)) * 8u + (blockIdx.x & 7u);
    rt = (blockIdx.x >> 3) % nrt;
  } else {
    ct = blockIdx.x / nrt;
    rt = blockIdx.x % nrt;
  }
  uint64_t base = 0;
  for (int b = 0; b < a.nrest; ++b) base |= (uint64_t)((ct >> b) & 1u) << a.rest[b];
  // this lane's chunk elements tid + 256 u: state offsets and LDS slots
  uint64_t xoff[NX];
  int xslot[NX];
  bool xin[NX];
#pragma unroll
  for (int u = 0; u < NX; ++u) {
    const unsigned e = tid + kBlock * u;
    uint64_t o = 0;
    unsigned sl = 0;
#pragma unroll
    for (int t = 0; t < 4 + kLc; ++t) {
      const unsigned bit = (e >> t) & 1u;
      o |= (uint64_t)bit << a.epos[t];
      sl |= bit << a.eslot[t];
    }
    xin[u] = (e & a.einvalid) == 0;
    xoff[u] = xin[u] ? o : 0;
    const unsigned c = sl >> kLc, g = sl & (C - 1);
    xslot[u] = (int)(c * C + (g ^ c));   // lanes differing in c on different banks
  }
  auto mat_index = [&](unsigned v, int lo) {
    unsigned r = 0;
    for (int j = lo; j < a.k; ++j) r |= ((v >> j) & 1u) << a.mbit[j];
    return r;
  };
  uint64_t moff[NM];
  int mslot[NM];
#pragma unroll
  for (int u = 0; u < NM; ++u) {
    const unsigned c = tid & 15u, r = (tid >> 4) + 16u * u;
    moff[u] = (uint64_t)mat_index(rt * R + r, 0) * D + mat_index(c, 0);
    mslot[u] = (int)(c * R + (r ^ c));
  }
  v2d x[NX], mm[NM];
  auto fetch = [&](unsigned chunk) {
    uint64_t co = 0;
    for (int j = 4; j < a.k; ++j) co |= (uint64_t)((chunk >> (j - 4)) & 1u) << a.sorted[j];
    const v2d* p = reinterpret_cast<const v2d*>(in) + base + co;
    const v2d* pm = reinterpret_cast<const v2d*>(m) + mat_index(chunk << 4, 4);
#pragma unroll
    for (int u = 0; u < NX; ++u) x[u] = xin[u] ? p[xoff[u]] : v2d{0.0, 0.0};
#pragma unroll
    for (int u = 0; u < NM; ++u) mm[u] = pm[moff[u]];
  };
  const int wr = (wave % kRowWaves) * WR, wc = (wave / kRowWaves) * WC;
  v4d re[RB][CB], im[RB][CB];
#pragma unroll
  for (int i = 0; i < RB; ++i)
#pragma unroll
    for (int j = 0; j < CB; ++j) re[i][j] = im[i][j] = v4d{0.0, 0.0, 0.0, 0.0};
  const unsigned nchunk = (unsigned)D / kKc;
  fetch(0);
  for (unsigned ch = 0; ch < nchunk; ++ch) {
#pragma unroll
    for (int u = 0; u < NX; ++u) xs[xslot[u]] = x[u];
#pragma unroll
    for (int u = 0; u < NM; ++u) ms[mslot[u]] = mm[u];
    __syncthreads();
    if (ch + 1 < nchunk) fetch(ch + 1);
#pragma unroll
    for (int ks = 0; ks < kKc / 4; ++ks) {
      const int c = 4 * ks + q;
      v2d av[RB], bv[CB];
#pragma unroll
      for (int i = 0; i < RB; ++i) av[i] = ms[c * R + ((wr + 16 * i + col) ^ c)];
#pragma unroll
      for (int j = 0; j < CB; ++j) bv[j] = xs[c * C + ((wc + 16 * j + col) ^ c)];
#pragma unroll
      for (int i = 0; i < RB; ++i)
#pragma unroll
        for (int j = 0; j < CB; ++j) {
          re[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(av[i].x, bv[j].x, re[i][j], 0, 0, 0);
          im[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(av[i].x, bv[j].y, im[i][j], 0, 0, 0);
          re[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(-av[i].y, bv[j].y, re[i][j], 0, 0, 0);
          im[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(av[i].y, bv[j].x, im[i][j], 0, 0, 0);
        }
    }
    __syncthreads();
  }
  // row wr + 16 i + 4 j + q, group wc + 16 cb + col
  const uint64_t qoff = ((uint64_t)(q & 1) << a.sorted[0]) | ((uint64_t)(q >> 1) << a.sorted[1]);
#pragma unroll
  for (int cb = 0; cb < CB; ++cb) {
    const unsigned g = wc + 16 * cb + col;
    if (g >> a.gbits) continue;
    uint64_t go = base | qoff;
    for (int t = 0; t < a.gbits; ++t) go |= (uint64_t)((g >> t) & 1u) << a.gpos[t];
#pragma unroll
    for (int i = 0; i < RB; ++i) {
      const unsigned r = rt * R + wr + 16 * i;
      uint64_t ro = 0;
      for (int t = 4; t < a.k; ++t) ro |= (uint64_t)((r >> t) & 1u) << a.sorted[t];
      v2d* p = reinterpret_cast<v2d*>(out) + (go | ro);
#pragma unroll
      for (int j = 0; j < 4; ++j)
        p[((uint64_t)(j & 1) << a.sorted[2]) | ((uint64_t)(j >> 1) << a.sorted[3])] =
            v2d{re[i][cb][j], im[i][cb][j]};
    }
  }
}

// out[i] = in[j] where bit src[b] of j equals bit b of i (a relabelling of
// the index bits), by tiles that read and write contiguous runs.
// 26 qubits, 2 GiB moved: a random order 415 us (5.2 TB/s), the reversed order
// 401 us; by gathering 1096 and 2122 us.
__global__ __launch_bounds__(kPermBlock) void permute_tile_kernel(double2* __restrict__ out,
                                                                 const double2* __restrict__ in,
                                                                 uint64_t ntiles, PermTile p) {
  __shared__ v2d lds[1 << kPermT];
  const PermLane q = perm_lane(p);
  for (uint64_t tile = blockIdx.x; tile < ntiles; tile += gridDim.x) {
    uint64_t bi, bo;
    perm_bases(p, tile, &bi, &bo);
    v2d v[kPermPer];
    const v2d* src = reinterpret_cast<const v2d*>(in) + bi + q.in_lane;
#pragma unroll
    for (int u = 0; u < kPermPer; ++u) v[u] = ld_stream(src + q.in_u[u]);
#pragma unroll
    for (int u = 0; u < kPermPer; ++u) lds[q.lds_in[u]] = v[u];
    __syncthreads();
    v2d* dst = reinterpret_cast<v2d*>(out) + bo + q.out_lane;
#pragma unroll
    for (int u = 0; u < kPermPer; ++u)
      st_stream(dst + q.out_u[u], lds[perm_swz(threadIdx.x + kPermBlock * u)]);
    __syncthreads();
  }
}

// The same for states smaller than a tile.
struct PermArg {
  int src[QFX_MAX_QUBITS];
};

__global__ __launch_bounds__(kBlock) void permute_bits_kernel(double2* __restrict__ out,
                                                             const double2* __restrict__ in,
                                                             uint64_t len, int n, PermArg a) {
  const uint64_t i = (uint64_t)blockIdx.x * kBlock + threadIdx.x;
  if (i >= len) return;
  uint64_t j = 0;
  for (int b = 0; b < n; ++b) j |= ((i >> b) & 1) << a.src[b];
  out[i] = in[j];
}

__global__ __launch_bounds__(kBlock) void fill_kernel(double2* psi, uint64_t len, double2 first,
                                                     double2 rest) {
  const uint64_t i = (uint64_t)blockIdx.x * kBlock + threadIdx.x;
  if (i < len) psi[i] = (i == 0) ? first : rest;
}

template <int K>
int launch_dense(hipStream_t s, double2* out, const double2* in, int n, const int* targets,
                 const qfx_c128* matrix) {
  DenseArg<K> a;
  constexpr int D = 1 << K;
  for (int i = 0; i < D * D; ++i) a.m[i] = make_double2(matrix[i].re, matrix[i].im);
  for (unsigned r = 0; r < (unsigned)D; ++r) a.off[r] = qfx::local_offset(K, targets, r);
  qfx::sort_bits(K, targets, a.sorted);
  constexpr int G = groups_per_thread<K>();
  const uint64_t ngroups = (uint64_t)1 << (n - K);
  const uint64_t blocks = (ngroups + kBlock * G - 1) / (kBlock * G);
  auto kernel = a.sorted[0] < kLineBits ? dense_kernel<K, G, false> : dense_kernel<K, G, true>;
  hipLaunchKernelGGL(kernel, dim3((unsigned)blocks), dim3(kBlock), 0, s, out, in, ngroups, a);
  return qfx::check_launch("dense_kernel");
}

template <int K>
int launch_sparse_k(hipStream_t s, double2* out, const double2* in, int n, const SparseArg& a) {
  const uint64_t ngroups = (uint64_t)1 << (n - K);
  if (out != in) {
    constexpr int G = K == 1 ? 4 : (K == 2 ? 2 : 1);
    const uint64_t blocks = (ngroups + kBlock * G - 1) / (kBlock * G);
    auto kernel = a.sorted[0] < kLineBits ? sparse_kernel<K, G, true, false>
                                          : sparse_kernel<K, G, true, true>;
    hipLaunchKernelGGL(kernel, dim3((unsigned)blocks), dim3(kBlock), 0, s, out, in, ngroups, a);
    return qfx::check_launch("sparse_kernel");
  }
  constexpr int G = K == 1 ? 4 : ((K == 2 || K == 4) ? 2 : 1);
  const uint64_t blocks = (ngroups + kBlock * G - 1) / (kBlock * G);
  auto kernel = a.sorted[0] < kLineBits ? sparse_kernel<K, G, false, false>
                                        : sparse_kernel<K, G, false, true>;
  hipLaunchKernelGGL(kernel, dim3((unsigned)blocks), dim3(kBlock), 0, s, out, in, ngroups, a);
  return qfx::check_launch("sparse_kernel");
}

int launch_sparse(hipStream_t s, double2* out, const double2* in, int n, int k,
                  const SparseArg& a) {
  switch (k) {
    case 1: return launch_sparse_k<1>(s, out, in, n, a);
    case 2: return launch_sparse_k<2>(s, out, in, n, a);
    case 3: return launch_sparse_k<3>(s, out, in, n, a);
    case 4: return launch_sparse_k<4>(s, out, in, n, a);
    case 5: return launch_sparse_k<5>(s, out, in, n, a);
  }
  return qfx::set_error(QFX_ERANGE, "sparse gate width out of range");
}

template <int R, int C>
int launch_mfma(hipStream_t s, double2* out, const double2* in, int n, int k, const int* targets,
                const double2* m) {
  constexpr int kLc = C == 128 ? 7 : 6;
  GemmArg a;
  std::memset(&a, 0, sizeof(a));
  a.k = k;
  qfx::sort_bits(k, targets, a.sorted);
  for (int j = 0; j < k; ++j)
    for (int t = 0; t < k; ++t)
      if (targets[t] == a.sorted[j]) a.mbit[j] = k - 1 - t;   // gate qubit 0 is the MSB
  uint64_t tmask = 0;
  for (int j = 0; j < k; ++j) tmask |= (uint64_t)1 << targets[j];
  for (int b = 0; b < n; ++b) {
    if ((tmask >> b) & 1) continue;
    if (a.gbits < kLc) a.gpos[a.gbits++] = b;
    else a.rest[a.nrest++] = b;
  }
  // chunk elements in address order: columns 0..3 of the gate and the groups
  int t = 0;
  for (int b = 0; b < n; ++b) {
    for (int j = 0; j < 4; ++j)
      if (a.sorted[j] == b) { a.epos[t] = b; a.eslot[t++] = kLc + j; }
    for (int j = 0; j < a.gbits; ++j)
      if (a.gpos[j] == b) { a.epos[t] = b; a.eslot[t++] = j; }
  }
  for (int j = a.gbits; j < kLc; ++j) {      // groups that the state does not have
    a.einvalid |= 1u << t;
    a.epos[t] = 0;
    a.eslot[t++] = j;
  }
  const unsigned ntiles = 1u << a.nrest;
  const unsigned blocks = ntiles * (unsigned)((1 << k) / R);
  hipLaunchKernelGGL((dense_mfma_kernel<R, C>), dim3(blocks), dim3(kBlock), 0, s, out, in, ntiles,
                     a, m);
  return qfx::check_launch("dense_mfma_kernel");
}

// The largest tile whose grid still covers the 256 CUs, else 16 x 64, whose
// step is a quarter as long and whose grid is larger (8 qubits of 16: 47 us
// with 16 workgroups of 64 x 64, 22 us with 64 of 16 x 64; 10 of 18: 179 and
// 87 us, 64 and 256 workgroups).
int launch_wide(hipStream_t s, double2* out, const double2* in, int n, int k, const int* targets,
                const double2* m) {
  const int gb = n - k;
  auto blocks = [&](int row_bits, int col_bits) {
    return (int64_t)1 << ((k > row_bits ? k - row_bits : 0) + (gb > col_bits ? gb - col_bits : 0));
  };
  if (k >= 6 && blocks(6, 6) >= kCus) return launch_mfma<64, 64>(s, out, in, n, k, targets, m);
  if (k == 5 && blocks(5, 7) >= kCus) return launch_mfma<32, 128>(s, out, in, n, k, targets, m);
  if (k == 4 && blocks(4, 7) >= kCus) return launch_mfma<16, 128>(s, out, in, n, k, targets, m);
  return launch_mfma<16, 64>(s, out, in, n, k, targets, m);
}

bool is_one(const qfx_c128& z) { return z.re == 1.0 && z.im == 0.0; }

// Build SparseArg for a diagonal (src == NULL) or monomial gate.
int build_sparse(int n, int k, const int* targets, const int* src, const qfx_c128* ph,
                 bool inplace, SparseArg* a, const char* fn) {
  int rc = qfx::check_targets(n, k, targets, 5, fn);
  if (rc) return rc;
  const int D = 1 << k;
  std::memset(a, 0, sizeof(*a));
  uint32_t seen = 0;
  for (int r = 0; r < D; ++r) {
    const int sr = src ? src[r] : r;
    if (sr < 0 || sr >= D) return qfx::set_error(QFX_EINVAL, std::string(fn) + ": bad source row");
    if (seen & (1u << sr))
      return qfx::set_error(QFX_EINVAL, std::string(fn) + ": source rows are not a permutation");
    seen |= 1u << sr;
    a->off[r] = qfx::local_offset(k, targets, r);
    a->srcoff[r] = qfx::local_offset(k, targets, sr);
    const qfx_c128 z = ph ? ph[r] : qfx_c128{1.0, 0.0};
    a->ph[r] = make_double2(z.re, z.im);
    const bool one = is_one(z);
    if (!one) a->has_phase |= 1u << r;
    if (!inplace || !one || sr != r) a->active |= 1u << r;
  }
  qfx::sort_bits(k, targets, a->sorted);
  return QFX_OK;
}

}  // namespace

extern "C" {

int qfx_apply_matrix(void* stream, void* out, const void* in, int n, int k, const int* targets,
                     const qfx_c128* matrix) {
  int rc = qfx::check_targets(n, k, targets, 3, "qfx_apply_matrix");
  if (rc) return rc;
  if (!out || !in || !matrix) return qfx::set_error(QFX_EINVAL, "qfx_apply_matrix: null pointer");
  hipStream_t s = qfx::as_stream(stream);
  auto* o = static_cast<double2*>(out);
  auto* i = static_cast<const double2*>(in);
  switch (k) {
    case 1: return launch_dense<1>(s, o, i, n, targets, matrix);
    case 2: return launch_dense<2>(s, o, i, n, targets, matrix);
    case 3: return launch_dense<3>(s, o, i, n, targets, matrix);
  }
  return qfx::set_error(QFX_ERANGE, "qfx_apply_matrix: k > 3 needs qfx_apply_matrix_dev");
}

int qfx_apply_matrix_dev(void* stream, void* out, const void* in, int n, int k,
                         const int* targets, const void* matrix) {
  int rc = qfx::check_targets(n, k, targets, QFX_MAX_DENSE_K, "qfx_apply_matrix_dev");
  if (rc) return rc;
  if (!out || !in || !matrix)
    return qfx::set_error(QFX_EINVAL, "qfx_apply_matrix_dev: null pointer");
  if (out == in) return qfx::set_error(QFX_EINVAL, "qfx_apply_matrix_dev: out must not alias in");
  if (k >= 4)
    return launch_wide(qfx::as_stream(stream), static_cast<double2*>(out),
                       static_cast<const double2*>(in), n, k, targets,
                       static_cast<const double2*>(matrix));
  DevTargets tg;
  std::memset(&tg, 0, sizeof(tg));
  for (int j = 0; j < k; ++j) tg.t[j] = targets[j];
  const uint64_t len = (uint64_t)1 << n;
  const uint64_t blocks = (len + kBlock - 1) / kBlock;
  hipLaunchKernelGGL(dense_dev_kernel, dim3((unsigned)blocks), dim3(kBlock),
                     sizeof(uint64_t) << k, qfx::as_stream(stream), static_cast<double2*>(out),
                     static_cast<const double2*>(in), len, k, tg,
                     static_cast<const double2*>(matrix));
  return qfx::check_launch("dense_dev_kernel");
}

int qfx_apply_diagonal(void* stream, void* out, const void* in, int n, int k, const int* targets,
                       const qfx_c128* diag) {
  if (!out || !in || !diag) return qfx::set_error(QFX_EINVAL, "qfx_apply_diagonal: null pointer");
  SparseArg a;
  int rc = build_sparse(n, k, targets, nullptr, diag, false, &a, "qfx_apply_diagonal");
  if (rc) return rc;
  return launch_sparse(qfx::as_stream(stream), static_cast<double2*>(out),
                       static_cast<const double2*>(in), n, k, a);
}

int qfx_apply_monomial(void* stream, void* out, const void* in, int n, int k, const int* targets,
                       const int* src, const qfx_c128* phase) {
  if (!out || !in || !src) return qfx::set_error(QFX_EINVAL, "qfx_apply_monomial: null pointer");
  SparseArg a;
  int rc = build_sparse(n, k, targets, src, phase, false, &a, "qfx_apply_monomial");
  if (rc) return rc;
  return launch_sparse(qfx::as_stream(stream), static_cast<double2*>(out),
                       static_cast<const double2*>(in), n, k, a);
}

int qfx_apply_diagonal_inplace(void* stream, void* state, int n, int k, const int* targets,
                               const qfx_c128* diag) {
  if (!state || !diag)
    return qfx::set_error(QFX_EINVAL, "qfx_apply_diagonal_inplace: null pointer");
  SparseArg a;
  int rc = build_sparse(n, k, targets, nullptr, diag, true, &a, "qfx_apply_diagonal_inplace");
  if (rc) return rc;
  if (!a.active) return QFX_OK;
  auto* p = static_cast<double2*>(state);
  return launch_sparse(qfx::as_stream(stream), p, p, n, k, a);
}

int qfx_apply_monomial_inplace(void* stream, void* state, int n, int k, const int* targets,
                               const int* src, const qfx_c128* phase) {
  if (!state || !src)
    return qfx::set_error(QFX_EINVAL, "qfx_apply_monomial_inplace: null pointer");
  SparseArg a;
  int rc = build_sparse(n, k, targets, src, phase, true, &a, "qfx_apply_monomial_inplace");
  if (rc) return rc;
  if (!a.active) return QFX_OK;
  auto* p = static_cast<double2*>(state);
  return launch_sparse(qfx::as_stream(stream), p, p, n, k, a);
}

int qfx_permute_qubits(void* stream, void* out, const void* in, int n, const int* src_bit) {
  if (!out || !in || !src_bit) return qfx::set_error(QFX_EINVAL, "qfx_permute_qubits: null pointer");
  if (out == in) return qfx::set_error(QFX_EINVAL, "qfx_permute_qubits: out must not alias in");
  if (n < 1 || n > QFX_MAX_QUBITS)
    return qfx::set_error(QFX_ERANGE, "qfx_permute_qubits: n out of range");
  int rc = qfx::check_permutation(n, src_bit, "qfx_permute_qubits");
  if (rc) return rc;
  const uint64_t len = (uint64_t)1 << n;
  if (n >= kPermT) {
    const uint64_t ntiles = len >> kPermT;
    hipLaunchKernelGGL(permute_tile_kernel, dim3((unsigned)(ntiles < (1u << 20) ? ntiles : 1u << 20)),
                       dim3(kPermBlock), 0, qfx::as_stream(stream), static_cast<double2*>(out),
                       static_cast<const double2*>(in), ntiles, make_perm_tile(n, src_bit));
    return qfx::check_launch("permute_tile_kernel");
  }
  PermArg a;
  std::memset(&a, 0, sizeof(a));
  for (int b = 0; b < n; ++b) a.src[b] = src_bit[b];
  hipLaunchKernelGGL(permute_bits_kernel, dim3((unsigned)((len + kBlock - 1) / kBlock)),
                     dim3(kBlock), 0, qfx::as_stream(stream), static_cast<double2*>(out),
                     static_cast<const double2*>(in), len, n, a);
  return qfx::check_launch("permute_bits_kernel");
}

int qfx_zero_state(void* stream, void* psi, int n) {
  if (!psi) return qfx::set_error(QFX_EINVAL, "qfx_zero_state: null pointer");
  if (n < 0 || n > QFX_MAX_QUBITS) return qfx::set_error(QFX_ERANGE, "qfx_zero_state: n out of range");
  const uint64_t len = (uint64_t)1 << n;
  hipLaunchKernelGGL(fill_kernel, dim3((unsigned)((len + kBlock - 1) / kBlock)), dim3(kBlock), 0,
                     qfx::as_stream(stream), static_cast<double2*>(psi), len,
                     make_double2(1.0, 0.0), make_double2(0.0, 0.0));
  return qfx::check_launch("fill_kernel");
}

int qfx_plus_state(void* stream, void* psi, int n) {
  if (!psi) return qfx::set_error(QFX_EINVAL, "qfx_plus_state: null pointer");
  if (n < 0 || n > QFX_MAX_QUBITS) return qfx::set_error(QFX_ERANGE, "qfx_plus_state: n out of range");
  const uint64_t len = (uint64_t)1 << n;
  const double a = std::ldexp(1.0, -n / 2) * ((n & 1) ? 0.70710678118654752440 : 1.0);
  hipLaunchKernelGGL(fill_kernel, dim3((unsigned)((len + kBlock - 1) / kBlock)), dim3(kBlock), 0,
                     qfx::as_stream(stream), static_cast<double2*>(psi), len, make_double2(a, 0.0),
                     make_double2(a, 0.0));
  return qfx::check_launch("fill_kernel");
}

}  // extern "C"

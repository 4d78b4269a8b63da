// Runs of gates on small states and on a few bits of large ones: many gates a
// launch, planned in native code as the call is made.
//
// Circuit.run below the fused executor's sizes, Circuit.evolve on densities and
// Circuit.asgate apply their gates in order (quantumflow/circuits.py:87-127),
// one launch each on the per-gate path: about 20 us of host work for 2-4 us of
// GPU work at 12 qubits, one HBM pass per gate at 24.  Here a launch loads
// every 2^T-amplitude tile into LDS, applies up to a few dozen gates to it and
// writes it back.  The gates travel by value in the kernel arguments (4 KB), so
// a call copies nothing, keeps nothing and may be captured.
//
//   n <= 13   the whole state is one tile, the gates run in order;
//   n >  13   a pass collects gates greedily, in order, while their bits fit
//             the tile with the kLowBits lowest bits (contiguous runs); a gate
//             may pass one that is left behind if they share no bit.  A pass
//             of one gate runs on the per-gate kernels.
#include <algorithm>
#include <cstddef>
#include <cstring>
#include <new>
#include <string>
#include <vector>

#include "qfx_common.h"

namespace {

constexpr int kWholeBits = 13;         // largest state held in one tile (128 KiB)
constexpr int kTileBits = 12;          // tile of larger states: two per CU
constexpr int kLowBits = 3;            // 128-byte runs
constexpr int kMaxOpK = 4;             // sparse gates; dense ones up to 3
constexpr unsigned kGrid = 512;        // workgroups of a tiled pass: two per CU
constexpr int kUnits = 248;            // 16-byte units of ops and their data
constexpr int kAhead = 4;              // units read ahead of an op, past the last as well

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

enum ListKind : unsigned { LK_DENSE = 0, LK_ROWS = 1, LK_MULTI = 2 };

// One op.  Its k bits split the tile into groups; element r of a group sits at
// the group's slot XOR an offset.  A dense gate has 4^k coefficients.  A
// diagonal or monomial gate lists the rows it changes, 2^lr of them (a CNOT 2
// of 4, a CZ 1; filled up with rows it leaves alone): offsets to | from << 16,
// four a unit, then 2^lr phases if any row has one (bit of `phased`).  Two or
// three dense or diagonal 1-qubit gates in a row on different bits are one op
// of that many bits: 4 coefficients or 2 phases each, and 4 bits of `phased`
// (diagonal; which of its phases differ from 1).
struct ListOp {
  uint8_t form;                        // kind | k << 2 | lr << 5
  uint8_t data;                        // unit of the op's data
  uint16_t phased;
  uint16_t off[4];                     // slot offset of gate qubit j (MSB first)
  uint8_t sorted[4];                   // tile bits ascending, 31 past the k-th
};
static_assert(sizeof(ListOp) == 16, "an op is one unit");

struct ListArgs {
  u32x4 units[kUnits];                // ops from the front, data from the back
  v2d* out;
  const v2d* in;
  unsigned ntiles;
  int T, nops, stream;
  uint8_t pos[kWholeBits + 3];         // state bit of tile bit j, ascending
};
static_assert(sizeof(ListArgs) <= 4096 && offsetof(ListArgs, units) == 0, "kernel arguments");

// The arguments' units where they lie (ListArgs is the kernels' only
// parameter): a by-value array indexed at run time would be copied to scratch.
typedef const __attribute__((address_space(4))) u32x4* unit_ptr;

__device__ __forceinline__ unit_ptr arg_units() {
  return (unit_ptr)__builtin_amdgcn_kernarg_segment_ptr();
}

// Slot of tile element e: higher bits folded into the lowest three, so that
// strided groups spread over the LDS banks.  XOR-linear.
__host__ __device__ __forceinline__ unsigned lsw(unsigned e) {
  return e ^ (((e >> 3) ^ (e >> 6) ^ (e >> 9) ^ (e >> 12)) & 7u);
}

// A unit every lane read from the same LDS address, in scalar registers.
__device__ __forceinline__ u32x4 uniform(u32x4 w) {
#pragma unroll
  for (int i = 0; i < 4; ++i) w[i] = (uint32_t)__builtin_amdgcn_readfirstlane((int)w[i]);
  return w;
}

// The kernel declares no static LDS, so its dynamic LDS starts at address 0
// and a slot's byte offset is its address.
typedef __attribute__((address_space(3))) v2d v2d_lds;
__device__ __forceinline__ v2d_lds* at(unsigned byte) { return (v2d_lds*)(size_t)byte; }

// LDS address of group g: zeros inserted at K bits (bit 31 inserts none).
// Linear in g, so group lane + u BS sits at the lane's address XOR u's, which
// is scalar.
template <int K>
__device__ __forceinline__ unsigned group_addr(unsigned g, unsigned sorted) {
#pragma unroll
  for (int j = 0; j < K; ++j) g += g & ~((1u << ((sorted >> (8 * j)) & 255u)) - 1u);
  return lsw(g) << 4;
}

// Calls f(addresses of G groups) for the lane's groups: lanes are dealt groups
// in turn, G at a time where each has that many.
template <int K, int BS, int G, typename F>
__device__ __forceinline__ void for_groups(int ngroups, int tid, unsigned sorted, F&& f) {
  if (tid >= ngroups) return;
  const unsigned mine = group_addr<K>((unsigned)tid, sorted);
  const int nu = ngroups > BS ? ngroups / BS : 1;
  int u = 0;
  if constexpr (G > 1) {
    for (; u + G <= nu; u += G) {
      unsigned ad[G];
#pragma unroll
      for (int i = 0; i < G; ++i) ad[i] = mine ^ group_addr<K>((unsigned)(u + i) * BS, sorted);
      f(ad);
    }
  }
  for (; u < nu; ++u) {
    const unsigned ad[1] = {mine ^ group_addr<K>((unsigned)u * BS, sorted)};
    f(ad);
  }
}

// `p`: the op's first four data units, read ahead.
template <int K, int BS>
__device__ __forceinline__ void list_dense(int T, int tid, const u32x4 w, const v2d (&p)[kAhead],
                                           const v2d* m) {
  constexpr int D = 1 << K, G = K == 1 ? 4 : (K == 2 ? 2 : 1);
  const unsigned o[4] = {(w.y & 65535u) << 4, (w.y >> 16) << 4, (w.z & 65535u) << 4,
                         (w.z >> 16) << 4};
  unsigned off[D];
#pragma unroll
  for (int r = 0; r < D; ++r) {
    off[r] = 0;
#pragma unroll
    for (int j = 0; j < K; ++j) off[r] ^= ((r >> (K - 1 - j)) & 1) ? o[j] : 0u;
  }
  for_groups<K, BS, G>(1 << (T - K), tid, w.w, [&](const auto& ad) {
    constexpr int N = sizeof(ad) / sizeof(unsigned);
    v2d v[N][D];
#pragma unroll
    for (int u = 0; u < N; ++u)
#pragma unroll
      for (int r = 0; r < D; ++r) v[u][r] = *at(ad[u] ^ off[r]);
#pragma unroll
    for (int r = 0; r < D; ++r) {
      v2d acc[N];
#pragma unroll
      for (int u = 0; u < N; ++u) acc[u] = v2d{0.0, 0.0};
#pragma unroll
      for (int q = 0; q < D; ++q) {
        const v2d x = r * D + q < kAhead ? p[(r * D + q) % kAhead] : m[r * D + q];
#pragma unroll
        for (int u = 0; u < N; ++u) cmac(acc[u], x, v[u][q]);
      }
#pragma unroll
      for (int u = 0; u < N; ++u) *at(ad[u] ^ off[r]) = acc[u];
      if constexpr (K > 2) __builtin_amdgcn_sched_barrier(0);   // one row in registers
    }
  });
}

// NB 1-qubit gates on different bits, gate j on qubit j's bit, in one sweep;
// those in DIAG are diagonal.  Compile-time, since a branch between the two
// would keep the amplitudes twice over at its end.
template <int NB, int DIAG, int BS>
__device__ __forceinline__ void list_multi(int T, int tid, const u32x4 w, const v2d (&p)[kAhead],
                                           const v2d* m) {
  constexpr int D = 1 << NB;
  const unsigned o[3] = {(w.y & 65535u) << 4, (w.y >> 16) << 4, (w.z & 65535u) << 4};
  const unsigned kinds = w.x >> 16;
  v2d c[NB][4];
#pragma unroll
  for (int j = 0; j < NB; ++j) {
    const int n = ((DIAG >> j) & 1) ? 2 : 4;
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (i < n) c[j][i] = j == 0 ? p[i] : m[i];
    m += n;
  }
  for_groups<NB, BS, 1>(1 << (T - NB), tid, w.w, [&](const auto& ad) {
    v2d v[D];                           // bit j of the index: qubit j
    auto addr = [&](int r) {
      unsigned x = ad[0];
#pragma unroll
      for (int j = 0; j < NB; ++j) x ^= ((r >> j) & 1) ? o[j] : 0u;
      return x;
    };
#pragma unroll
    for (int r = 0; r < D; ++r) v[r] = *at(addr(r));
#pragma unroll
    for (int j = 0; j < NB; ++j) {
      if ((DIAG >> j) & 1) {
#pragma unroll
        for (int r = 0; r < D; ++r) {
          // a phase of exactly 1 leaves the amplitude as it is
          const int h = (r >> j) & 1;
          const bool on = (kinds >> (4 * j)) & (2u << h);
          const v2d x = cmul_fma(c[j][h], v[r]);
          v[r].x = on ? x.x : v[r].x;
          v[r].y = on ? x.y : v[r].y;
        }
      } else {
#pragma unroll
        for (int r = 0; r < D; ++r) {
          if ((r >> j) & 1) continue;
          const v2d x = v[r], y = v[r | (1 << j)];
          v2d s = {0.0, 0.0}, t = {0.0, 0.0};
          cmac(s, c[j][0], x);
          cmac(s, c[j][1], y);
          cmac(t, c[j][2], x);
          cmac(t, c[j][3], y);
          v[r] = s;
          v[r | (1 << j)] = t;
        }
      }
    }
#pragma unroll
    for (int r = 0; r < D; ++r) *at(addr(r)) = v[r];
  });
}

template <int NB, int BS>
__device__ __forceinline__ void list_multi_any(int T, int tid, const u32x4 w,
                                               const v2d (&p)[kAhead], const v2d* m) {
  const unsigned kinds = w.x >> 16;
  switch ((kinds & 1u) | ((kinds >> 3) & 2u) | ((kinds >> 6) & 4u)) {
    case 0: list_multi<NB, 0, BS>(T, tid, w, p, m); break;
    case 1: list_multi<NB, 1, BS>(T, tid, w, p, m); break;
    case 2: list_multi<NB, 2, BS>(T, tid, w, p, m); break;
    case 3: list_multi<NB, 3, BS>(T, tid, w, p, m); break;
    case 4: if constexpr (NB > 2) list_multi<NB, 4, BS>(T, tid, w, p, m); break;
    case 5: if constexpr (NB > 2) list_multi<NB, 5, BS>(T, tid, w, p, m); break;
    case 6: if constexpr (NB > 2) list_multi<NB, 6, BS>(T, tid, w, p, m); break;
    case 7: if constexpr (NB > 2) list_multi<NB, 7, BS>(T, tid, w, p, m); break;
  }
}

template <int R, int BS>
__device__ __forceinline__ void list_rows(int T, int tid, const u32x4 w, const v2d (&p)[kAhead],
                                          const v2d* d) {
  constexpr int G = R >= 8 ? 1 : (R == 4 ? 2 : 4), U = R > 4 ? R / 4 : 1;
  const unsigned phased = w.x >> 16;
  unsigned to[R], from[R];
#pragma unroll
  for (int q = 0; q < U; ++q) {
    const u32x4 x = uniform(__builtin_bit_cast(u32x4, p[q]));
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (4 * q + i < R) {
        to[4 * q + i] = (x[i] & 65535u) << 4;
        from[4 * q + i] = (x[i] >> 16) << 4;
      }
  }
  v2d ph[R <= 4 ? R : 1];
  if constexpr (R <= 4) {
#pragma unroll
    for (int r = 0; r < R; ++r) ph[r] = U + r < 4 ? p[U + r < 4 ? U + r : 0] : d[U + r];
  }
  for_groups<kMaxOpK, BS, G>(1 << (T - ((w.x >> 2) & 7u)), tid, w.w, [&](const auto& ad) {
    constexpr int N = sizeof(ad) / sizeof(unsigned);
    v2d v[N][R];
#pragma unroll
    for (int u = 0; u < N; ++u)
#pragma unroll
      for (int r = 0; r < R; ++r) v[u][r] = *at(ad[u] ^ from[r]);
#pragma unroll
    for (int r = 0; r < R; ++r) {
      if (phased & (1u << r)) {
        v2d x;
        if constexpr (R <= 4) x = ph[r];
        else x = d[U + r];
#pragma unroll
        for (int u = 0; u < N; ++u) v[u][r] = cmul_fma(x, v[u][r]);
      }
#pragma unroll
      for (int u = 0; u < N; ++u) *at(ad[u] ^ to[r]) = v[u][r];
    }
  });
}

// What bounds it.  A small state: the latency of each op (record, coefficients,
// amplitudes, barrier), 0.4-0.5 us up to 10 bits; so records and first data
// units are read an op ahead, and lane addresses are one deposit per op and a
// scalar XOR per access.  A large tile: LDS, about 0.8 us of a CU per sweep of
// 2^12 amplitudes (65 bytes a clock), which hides the arithmetic; so rotations
// in a row share a sweep and sparse gates move only the rows they change.  The
// ops are staged behind the tile once per workgroup: fetched from the argument
// memory as they came, each waited about a microsecond (40 us instead of 20
// for 28 gates at 9 qubits).
// 360 gates, 12 qubits: 242 us in 5 launches (one launch a gate: 7.4 ms, of
// which 1.1 ms on the GPU).  24 index bits: 100 us a pass and 13-16 us a gate,
// where a gate of its own takes 90-100 us.
template <int BS>
__global__ __launch_bounds__(BS) __attribute__((amdgpu_waves_per_eu(4))) void gate_list_kernel(
    ListArgs a) {
  extern __shared__ v2d lds[];
  constexpr int kLb = __builtin_ctz(BS);
  const int T = a.T;
  const unsigned tsize = 1u << T;
  v2d* data = lds + tsize;
  {
    unit_ptr units = arg_units();
    for (int i = threadIdx.x; i < kUnits; i += BS)
      reinterpret_cast<u32x4*>(data)[i] = units[i];
  }
  // The lane's offset, and the mask and first bit of the element bits above
  // the lane's, which step by carry-add (and wrap to 0 past the last one).  A
  // tile's base steps likewise by the deposited grid stride.
  uint64_t lane_off = 0, hm = 0, h0 = 0, tmask = 0;
  uint64_t base = blockIdx.x, step = gridDim.x;
#pragma unroll
  for (int j = 0; j < kWholeBits; ++j)
    if (j < T) {
      const uint64_t bit = (uint64_t)1 << a.pos[j];
      base = ((base & ~(bit - 1)) << 1) | (base & (bit - 1));
      step = ((step & ~(bit - 1)) << 1) | (step & (bit - 1));
      tmask |= bit;
      if (j < kLb) lane_off |= ((threadIdx.x >> j) & 1u) ? bit : 0;
      else hm |= bit;
      if (j == kLb) h0 = bit;
    }
  constexpr int kIo = 8;
  const int nk = tsize > (unsigned)BS ? (int)(tsize / BS) : 1;
  for (unsigned tile = blockIdx.x; tile < a.ntiles;
       tile += gridDim.x, base = ((base | tmask) + step) & ~tmask) {
    // opaque per tile (and op, below): the lane arithmetic of every element
    // and op would otherwise be hoisted out of the loops and spilled
    uint64_t zl = base | lane_off;
    unsigned me = threadIdx.x;
    __asm__ volatile("" : "+v"(zl), "+v"(me));
    uint64_t zh = 0;
    // A lane loads and stores the same elements, so its slots of the tile
    // before are its own to overwrite.  Lanes and steps past the tile's end
    // load an element again.
    for (int k0 = 0; k0 < nk; k0 += kIo) {
      v2d v[kIo];
#pragma unroll
      for (int i = 0; i < kIo; ++i) {
        v[i] = a.stream ? ld_stream(a.in + (zl | zh)) : a.in[zl | zh];
        zh = ((zh | ~hm) + h0) & hm;
      }
#pragma unroll
      for (int i = 0; i < kIo; ++i)
        if (k0 + i < nk && me < tsize) lds[lsw(me + (unsigned)(k0 + i) * BS)] = v[i];
    }
    __syncthreads();
    // op i's record and first data units are read while op i - 1 runs
    u32x4 next = reinterpret_cast<const u32x4*>(data)[0];
    v2d p[kAhead];
    auto read_ahead = [&](unsigned form) {
      const v2d* d = data + ((form >> 8) & 255u);
#pragma unroll
      for (int j = 0; j < kAhead; ++j) p[j] = d[j];
    };
    u32x4 w = uniform(next);
    read_ahead(w.x);
    for (int i = 0; i < a.nops; ++i) {
      int tid = threadIdx.x;
      __asm__ volatile("" : "+v"(tid));
      next = reinterpret_cast<const u32x4*>(data)[i + 1 < a.nops ? i + 1 : i];
      const unsigned kind = w.x & 3u, k = (w.x >> 2) & 7u, lr = (w.x >> 5) & 7u;
      const v2d* d = data + ((w.x >> 8) & 255u);
      if (kind == LK_MULTI) {
        if (k == 3) list_multi_any<3, BS>(T, tid, w, p, d);
        else list_multi_any<2, BS>(T, tid, w, p, d);
      } else if (kind == LK_DENSE) {
        switch (k) {
          case 1: list_dense<1, BS>(T, tid, w, p, d); break;
          case 2: list_dense<2, BS>(T, tid, w, p, d); break;
          case 3: list_dense<3, BS>(T, tid, w, p, d); break;
        }
      } else {
        switch (lr) {
          case 0: list_rows<1, BS>(T, tid, w, p, d); break;
          case 1: list_rows<2, BS>(T, tid, w, p, d); break;
          case 2: list_rows<4, BS>(T, tid, w, p, d); break;
          case 3: list_rows<8, BS>(T, tid, w, p, d); break;
          case 4: list_rows<16, BS>(T, tid, w, p, d); break;
        }
      }
      w = uniform(next);
      read_ahead(w.x);
      __syncthreads();
    }
    zh = 0;
    __asm__ volatile("" : "+v"(zl), "+v"(me));
    for (int k0 = 0; k0 < nk; k0 += kIo) {
      v2d v[kIo];
#pragma unroll
      for (int i = 0; i < kIo; ++i)
        v[i] = lds[lsw((me + (unsigned)(k0 + i) * BS) & (tsize - 1u))];
#pragma unroll
      for (int i = 0; i < kIo; ++i) {
        if (k0 + i < nk && me < tsize) {
          if (a.stream) st_stream(a.out + (zl | zh), v[i]);
          else a.out[zl | zh] = v[i];
        }
        zh = ((zh | ~hm) + h0) & hm;
      }
    }
  }
}

// ---- host: packing and planning ---------------------------------------------

struct Item {
  const qfx_gate* g;
  const int* bits;
  uint64_t mask;
  int units;                            // as an op of its own (item_units)
};

bool is_one(const qfx_c128& z) { return z.re == 1.0 && z.im == 0.0; }

// The rows a diagonal or monomial gate changes, filled up to a power of two
// with rows it leaves alone.
struct Rows {
  int lr;                               // log2 of the count; -1: the identity
  uint8_t row[16];
  uint16_t phased;                      // bit i: row[i] has a phase
};

Rows changed_rows(const qfx_gate& g) {
  const int D = 1 << g.k;
  Rows c;
  c.phased = 0;
  int m = 0;
  uint32_t used = 0;
  for (int r = 0; r < D; ++r) {
    const bool one = !g.coef || is_one(g.coef[r]);
    const bool moved = g.kind == QFX_GATE_MONOMIAL && g.src[r] != r;
    if (one && !moved) continue;
    if (!one) c.phased |= (uint16_t)(1u << m);
    used |= 1u << r;
    c.row[m++] = (uint8_t)r;
  }
  c.lr = m ? 0 : -1;
  while (m && (1 << c.lr) < m) ++c.lr;
  for (int r = 0; m && m < (1 << c.lr); ++r)
    if (!((used >> r) & 1u)) c.row[m++] = (uint8_t)r;
  return c;
}

// 16-byte units an item takes as an op of its own.
int item_units(const qfx_gate& g) {
  if (g.kind == QFX_GATE_DENSE) return 1 + (1 << (2 * g.k));
  const Rows c = changed_rows(g);
  if (c.lr < 0) return 0;
  const int n = 1 << c.lr;
  return 1 + (n + 3) / 4 + (c.phased ? n : 0);
}

struct Packer {
  ListArgs a;
  int top;                              // first data unit
  // the 1-qubit gates of the last op, if it can take more of them
  int nopen, open_top, open_bit[3];
  const qfx_gate* open[3];

  Packer() { clear(); }
  void clear() {
    a.nops = 0;
    top = kUnits;
    nopen = 0;
  }
  bool fits(int units) const { return a.nops + units <= top; }

  // tile_bit[b]: tile bit of state bit b
  void add(const Item& it, const int* tile_bit) {
    const qfx_gate& g = *it.g;
    int t[4] = {0, 0, 0, 0};
    for (int j = 0; j < g.k; ++j) t[j] = tile_bit[it.bits[j]];
    if (g.kind != QFX_GATE_DENSE && changed_rows(g).lr < 0) return;   // the identity
    if (g.k == 1 && g.kind != QFX_GATE_MONOMIAL) {
      bool join = nopen > 0 && nopen < 3;
      for (int j = 0; j < nopen; ++j) join = join && open_bit[j] != t[0];
      if (join) {                       // the op is packed again with one gate more
        --a.nops;
        top = open_top;
      } else {
        nopen = 0;
        open_top = top;
      }
      open[nopen] = &g;
      open_bit[nopen++] = t[0];
      if (nopen > 1) {
        add_multi();
        return;
      }
    } else {
      nopen = 0;
    }
    ListOp op;
    std::memset(&op, 0, sizeof(op));
    set_bits(&op, g.k, t);
    if (g.kind == QFX_GATE_DENSE) {
      op.form = (uint8_t)(LK_DENSE | g.k << 2);
      push(g.coef, 1 << (2 * g.k));
    } else {
      const Rows c = changed_rows(g);
      const int n = 1 << c.lr;
      op.form = (uint8_t)(LK_ROWS | g.k << 2 | c.lr << 5);
      op.phased = c.phased;
      auto offset = [&](int r) {
        unsigned o = 0;
        for (int j = 0; j < g.k; ++j)
          if ((r >> (g.k - 1 - j)) & 1) o |= 1u << t[j];
        return lsw(o);
      };
      uint32_t rows[16] = {};
      for (int i = 0; i < n; ++i) {
        const int r = c.row[i];
        rows[i] = offset(r) | offset(g.kind == QFX_GATE_MONOMIAL ? g.src[r] : r) << 16;
      }
      for (int i = n - 1; c.phased && i >= 0; --i) push(&g.coef[c.row[i]], 1);
      push(rows, (n + 3) / 4);
    }
    finish(op);
  }

 private:
  void push(const void* data, int units) {
    top -= units;
    std::memcpy(&a.units[top], data, 16 * (size_t)units);
  }
  void finish(ListOp& op) {
    op.data = (uint8_t)top;
    std::memcpy(&a.units[a.nops++], &op, sizeof(op));
  }
  void add_multi() {
    ListOp op;
    std::memset(&op, 0, sizeof(op));
    set_bits(&op, nopen, open_bit);
    op.form = (uint8_t)(LK_MULTI | nopen << 2);
    for (int j = nopen - 1; j >= 0; --j) {
      const qfx_gate& g = *open[j];
      const bool diag = g.kind == QFX_GATE_DIAGONAL;
      if (diag)
        op.phased |= (uint16_t)((1u | (is_one(g.coef[0]) ? 0u : 2u) | (is_one(g.coef[1]) ? 0u : 4u))
                                << (4 * j));
      push(g.coef, diag ? 2 : 4);
    }
    finish(op);
  }
  void set_bits(ListOp* op, int k, const int* t) {
    int sorted[4];
    qfx::sort_bits(k, t, sorted);
    for (int j = 0; j < 4; ++j) {
      op->off[j] = j < k ? (uint16_t)lsw(1u << t[j]) : 0;
      op->sorted[j] = j < k ? (uint8_t)sorted[j] : 31;
    }
  }
};

template <int BS>
int launch_list_bs(hipStream_t s, const ListArgs& a) {
  const size_t lds = sizeof(v2d) * (((size_t)1 << a.T) + kUnits + kAhead);
  if (lds > 65536) {
    const int rc = qfx::check_hip(
        hipFuncSetAttribute(reinterpret_cast<const void*>(gate_list_kernel<BS>),
                            hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds),
        "hipFuncSetAttribute");
    if (rc) return rc;
  }
  const unsigned grid = a.ntiles < kGrid ? a.ntiles : kGrid;
  hipLaunchKernelGGL(gate_list_kernel<BS>, dim3(grid), dim3(BS), lds, s, a);
  return qfx::check_launch("gate_list_kernel");
}

int launch_list(hipStream_t s, ListArgs& a, int n) {
  a.ntiles = 1u << (n - a.T);
  // four amplitudes a lane, eight from 12 bits on: at 9, 10, 11, 12 and 13 bits
  // 360 gates took 232, 256, 286, 373 and 547 us with these and 243, 259, 324,
  // 412 and 559 us with the next best (before gates shared sweeps)
  if (n > kWholeBits) return launch_list_bs<512>(s, a);
  if (a.T <= 9) return launch_list_bs<128>(s, a);
  if (a.T <= 11) return launch_list_bs<256>(s, a);
  if (a.T == 12) return launch_list_bs<512>(s, a);
  return launch_list_bs<1024>(s, a);
}

int run_single(void* stream, void* out, const void* in, int n, const Item& it) {
  const qfx_gate& g = *it.g;
  if (g.kind == QFX_GATE_DENSE) return qfx_apply_matrix(stream, out, in, n, g.k, it.bits, g.coef);
  if (g.kind == QFX_GATE_DIAGONAL)
    return out == in ? qfx_apply_diagonal_inplace(stream, out, n, g.k, it.bits, g.coef)
                     : qfx_apply_diagonal(stream, out, in, n, g.k, it.bits, g.coef);
  return out == in ? qfx_apply_monomial_inplace(stream, out, n, g.k, it.bits, g.src, g.coef)
                   : qfx_apply_monomial(stream, out, in, n, g.k, it.bits, g.src, g.coef);
}

int apply_gates(void* stream, void* out, const void* in, int n, int ngates,
                const qfx_gate* const* gates, const int* bits) {
  const char* fn = "qfx_apply_gates";
  if (!out || !in || !gates || !bits)
    return qfx::set_error(QFX_EINVAL, std::string(fn) + ": null pointer");
  if (ngates < 1) return qfx::set_error(QFX_ERANGE, std::string(fn) + ": no gates");
  std::vector<Item> items((size_t)ngates);
  for (int i = 0; i < ngates; ++i) {
    const qfx_gate* g = gates[i];
    if (!g) return qfx::set_error(QFX_EINVAL, std::string(fn) + ": null gate");
    const bool dense = g->kind == QFX_GATE_DENSE;
    if (g->kind < QFX_GATE_DENSE || g->kind > QFX_GATE_MONOMIAL ||
        (g->kind != QFX_GATE_MONOMIAL && !g->coef) || (g->kind == QFX_GATE_MONOMIAL && !g->src))
      return qfx::set_error(QFX_EINVAL, std::string(fn) + ": bad gate");
    int rc = qfx::check_targets(n, g->k, bits, dense ? 3 : kMaxOpK, fn);
    if (rc) return rc;
    if (g->kind == QFX_GATE_MONOMIAL) {
      unsigned seen = 0;
      for (int r = 0; r < (1 << g->k); ++r) {
        if (g->src[r] < 0 || g->src[r] >= (1 << g->k) || ((seen >> g->src[r]) & 1u))
          return qfx::set_error(QFX_EINVAL,
                                std::string(fn) + ": source rows are not a permutation");
        seen |= 1u << g->src[r];
      }
    }
    items[i] = Item{g, bits, 0, item_units(*g)};
    for (int j = 0; j < g->k; ++j) items[i].mask |= (uint64_t)1 << bits[j];
    bits += g->k;
  }
  hipStream_t s = qfx::as_stream(stream);
  const void* src = in;
  Packer p;
  int tile_bit[QFX_MAX_QUBITS];
  auto flush = [&]() {
    p.a.out = static_cast<v2d*>(out);
    p.a.in = static_cast<const v2d*>(src);
    const int rc = launch_list(s, p.a, n);
    src = out;
    p.clear();
    return rc;
  };
  auto set_tile = [&](uint64_t tile) {
    p.a.T = 0;
    for (int b = 0; b < n; ++b)
      if ((tile >> b) & 1) {
        tile_bit[b] = p.a.T;
        p.a.pos[p.a.T++] = (uint8_t)b;
      }
  };
  p.a.stream = 0;
  if (n <= kWholeBits) {
    set_tile(((uint64_t)1 << n) - 1);
    for (const Item& it : items) {
      if (!p.fits(it.units)) {
        const int rc = flush();
        if (rc) return rc;
      }
      p.add(it, tile_bit);
    }
    return flush();
  }
  // A pass looks at the gates that earlier ones passed over, left[head ..],
  // then at those from `next` on, until none can join it any more: so far and
  // no further, or a list of many passes would cost the square of its length.
  const uint64_t low = ((uint64_t)1 << kLowBits) - 1, all = ((uint64_t)1 << n) - 1;
  std::vector<int> left, over, take;
  size_t head = 0, next = 0;
  while (head < left.size() || next < items.size()) {
    uint64_t tile = low, blocked = 0;
    int units = 0;
    over.clear();
    take.clear();
    // takes gate i or passes over it; false once no later gate can be taken
    auto offer = [&](int i) {
      const Item& it = items[i];
      if (!(it.mask & blocked) && __builtin_popcountll(tile | it.mask) <= kTileBits) {
        if (units + it.units <= kUnits) {
          tile |= it.mask;
          units += it.units;
          take.push_back(i);
          return true;
        }
        over.push_back(i);
        return false;
      }
      blocked |= it.mask;
      over.push_back(i);
      return blocked != all && (__builtin_popcountll(tile) < kTileBits || (tile & ~blocked) != 0);
    };
    bool open = true;
    size_t at = head;
    while (open && at < left.size()) open = offer(left[at++]);
    if (open) {
      while (open && next < items.size()) open = offer((int)next++);
      left.swap(over);
      head = 0;
    } else {
      head = at - over.size();
      std::copy(over.begin(), over.end(), left.begin() + (ptrdiff_t)head);
    }
    if (take.size() == 1) {
      const int rc = run_single(stream, out, src, n, items[take[0]]);
      if (rc) return rc;
      src = out;
      continue;
    }
    for (int b = 0; __builtin_popcountll(tile) < kTileBits; ++b) tile |= (uint64_t)1 << b;
    set_tile(tile);
    for (int i : take) p.add(items[i], tile_bit);
    const int rc = flush();
    if (rc) return rc;
  }
  return QFX_OK;
}

}  // namespace

extern "C" {

int qfx_apply_gates(void* stream, void* out, const void* in, int n, int ngates,
                    const qfx_gate* const* gates, const int* bits) {
  try {
    return apply_gates(stream, out, in, n, ngates, gates, bits);
  } catch (const std::bad_alloc&) {      // the list's own vectors
    return qfx::set_error(QFX_EHIP, "qfx_apply_gates: out of host memory");
  }
}

}  // extern "C"

// Batched QAOA MaxCut engine: expectation values and adjoint gradients of
// many instances (graphs of different sizes) in one persistent launch.
//
// Replaces, for a whole batch at once, the reference's per-instance chain
//   qubo_circuit (quantumflow/qaoa.py:22-64) -> Circuit.run
//   (quantumflow/circuits.py:87-99) -> State.expectation(graph_cuts)
//   (quantumflow/states.py:131-147, quantumflow/qaoa.py:68-81)
// and the TensorFlow autograd gradient of examples/qaoa_maxcut.py:53-64.
//
// Per instance the state is |+>^n, then per layer l the cost layer
// prod_e ZZ(-w gamma_l / pi) = exp(i gamma_l (W/2 - C(z))) (W = sum of edge
// weights, C(z) the cut value) and the mixer RX(beta_l) on every qubit.
//
// Execution: every instance has a host-built program of passes.  A pass
// names a tile bit set S (|S| = T <= 13) and a list of stages; each of its
// 2^(n-T) tiles is one work item.  An item of pass k waits for the instance's
// items of pass k-1 and for nothing else; a launch without the workspace for
// that puts a grid barrier between the passes.  Instances with n <= T run as
// one item from start to end.
//
// A tile lives in registers: a workgroup of 512 lanes holds 2^R = 2^(T-9)
// amplitudes a lane (tiles below 2^9 leave lanes idle).  Tile bits 0-5 are the
// lane's, 6-8 the wave's and 9-12 the register's; a mixer stage pairs
// amplitudes of one lane on register bits, takes the partner from another lane
// by DPP on lane bits 0-3, exchanges lane bits 4 and 5 with a register bit by
// permlane swaps, and the three wave bits with three register bits through LDS
// (once per stage: the next stage starts from the exchanged order).  The cost
// layer is a table lookup of exp(i gamma (W/2 - c)) by integer cut count c.
// Adjoint backward (mode QFX_QAOA_BACKWARD): starting from the stored final
// state psi and lambda = C psi, the stages are undone in reverse order; the
// gradient of <C> is
//   d/d beta_l  = Im sum_j <lambda|X_j|psi>          (any point of mixer l)
//   d/d gamma_l = 2 Im <lambda|C|psi> - W Im <lambda|psi>   (after cost l)
// with lambda, psi carried back by RX(-beta) and the conjugate phases.
#include <cmath>
#include <cstring>
#include <mutex>
#include <type_traits>

#include "qfx_common.h"

namespace {

enum Stage : int {
  ST_INIT = 1,         // tile <- 2^(-n/2)
  ST_COST = 2,         // psi *= exp(i g (W/2 - C))
  ST_RX = 3,           // RX(beta) on the tile bits in mask
  ST_EXPECT = 4,       // acc += sum |psi|^2 C
  ST_MAKE_LAMBDA = 5,  // lambda <- C psi
  ST_RX_ADJ = 6,       // grad_beta += Im sum <lam|X_j|psi>; RX(-beta) on psi, lam
  ST_COST_ADJ = 7,     // grad_gamma += 2 Im <lam|C|psi> - W Im <lam|psi>; conj phases
  ST_COST_RX = 8,      // ST_COST then ST_RX of the same layer
  ST_RX_LOAD = 10,     // ST_RX as the first stage of a pass that loads
  ST_RX_STORE = 11,    // ST_RX as the last stage of a pass that stores
};

enum PassFlags : int { PF_LOAD_PSI = 1, PF_LOAD_LAM = 2, PF_STORE_PSI = 4, PF_STORE_LAM = 8 };

constexpr int kMaxT = 13;
constexpr int kMaxPLayers = QFX_QAOA_MAX_LAYERS;
constexpr int kAccum = 1 + 2 * kMaxPLayers;  // value, d/dbeta, d/dgamma
constexpr int kMaxEdgesTab = 512;  // cut counts 0..kMaxEdgesTab-1 tabulated
// A wait gives up after kBarrierSeconds of wall-clock time.  One
// phase of the largest program qfx_qaoa_check accepts (n <= 30: a 16 GiB
// state read and written once) streams in well under 0.1 s, so a timeout
// means workgroups that never arrive, not a slow phase.
constexpr int kBarrierSeconds = 10;
constexpr int kMaxDevices = 64;

constexpr int kThreads = 512;
constexpr int kWaves = kThreads / 64;
constexpr int kLaneBits = 6, kWaveBits = 3, kBaseBits = kLaneBits + kWaveBits;
// exchange buffer: 8 amplitudes a lane
constexpr int kExchange = kThreads * 8;

__device__ __forceinline__ double uniform_d(double x) {
  const uint64_t u = __builtin_bit_cast(uint64_t, x);
  const uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)u);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(u >> 32));
  return __builtin_bit_cast(double, ((uint64_t)hi << 32) | lo);
}

// sincos while a lane holds a tile: the library's takes some fifty registers
// for arguments of any size.  x / pi in two parts p + e, sincospi of p (which
// reduces exactly), and e by the angle sum; e is at most half an ulp of p, so
// below |x| = 2^30 its sine and cosine are pi e and 1.
__device__ __forceinline__ void sincos_held(double x, double* sn, double* cs) {
  constexpr double kInvPi = 0x1.45f306dc9c883p-2, kInvPiLow = -0x1.6b01ec5417056p-56;
  constexpr double kPi = 3.14159265358979323846;
  const double p = x * kInvPi;
  const double e = fma(x, kInvPiLow, fma(x, kInvPi, -p));
  double s, c;
  sincospi(p, &s, &c);
  if (fabs(x) < 0x1p30) {
    const double d = kPi * e;
    *sn = fma(c, d, s);
    *cs = fma(-s, d, c);
  } else {
    double se, ce;
    sincospi(e, &se, &ce);
    *sn = fma(s, ce, c * se);
    *cs = fma(c, ce, -s * se);
  }
}

// ---- amplitudes across lanes ------------------------------------------------

template <int CTRL>
__device__ __forceinline__ double dpp_d(double x) {
  const uint64_t u = __builtin_bit_cast(uint64_t, x);
  const uint32_t lo = (uint32_t)__builtin_amdgcn_mov_dpp((int)(uint32_t)u, CTRL, 15, 15, true);
  const uint32_t hi =
      (uint32_t)__builtin_amdgcn_mov_dpp((int)(uint32_t)(u >> 32), CTRL, 15, 15, true);
  return __builtin_bit_cast(double, ((uint64_t)hi << 32) | lo);
}

// The value of the lane that differs in the B-th lane bit of the tile index:
// lane ^ 1, 2, 7, 8, 16, 32 (tile_lane; for lane ^ 4 there is no single DPP
// form).
template <int B>
__device__ __forceinline__ double from_lane(double x) {
  if constexpr (B == 0) return dpp_d<0xB1>(x);                  // quad_perm [1,0,3,2]
  else if constexpr (B == 1) return dpp_d<0x4E>(x);             // quad_perm [2,3,0,1]
  else if constexpr (B == 2) return dpp_d<0x141>(x);            // row_half_mirror
  else if constexpr (B == 3) return dpp_d<0x128>(x);            // row_ror:8
  else return __shfl_xor(x, 1 << B, 64);
}


__device__ __forceinline__ unsigned tile_lane(unsigned lane) {
  return lane ^ ((lane & 4u) ? 3u : 0u);
}

// Exchanges lane bit B (4 or 5) with the choice of register: afterwards every
// lane holds in x and y the two amplitudes that differed in that lane bit, 0 in
// x.  Its own inverse.
template <int B>
__device__ __forceinline__ void swap_lane_bit(double& x, double& y) {
  const uint64_t u = __builtin_bit_cast(uint64_t, x), w = __builtin_bit_cast(uint64_t, y);
  uint32_t a[2] = {(uint32_t)u, (uint32_t)(u >> 32)}, b[2] = {(uint32_t)w, (uint32_t)(w >> 32)};
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    if constexpr (B == 4) {
      const auto r = __builtin_amdgcn_permlane16_swap(a[i], b[i], false, false);
      a[i] = r[0];
      b[i] = r[1];
    } else {
      const auto r = __builtin_amdgcn_permlane32_swap(a[i], b[i], false, false);
      a[i] = r[0];
      b[i] = r[1];
    }
  }
  x = __builtin_bit_cast(double, ((uint64_t)a[1] << 32) | a[0]);
  y = __builtin_bit_cast(double, ((uint64_t)b[1] << 32) | b[0]);
}

// ---- RX(theta): new_x = c x - i s y, c = cos(theta/2), s = sin(theta/2) -------
// As c (x - i t y), t = s / c, one fused operation a component instead of a
// product and one; the c of all bits of a stage are applied at its end.  Where
// |c| < |s| the bits are flipped besides, new_x = -i s (y - i t x) with
// t = -c / s, so |t| <= 1: the flip only changes which index a lane's amplitudes
// belong to, and -i, common to all of them, is dropped.
//
// In all updates of held amplitudes the products that read the old values come
// before the first new one: an update is then in place, where a new value
// beside the old one would be copied back at the next join of two branches (all
// amplitudes at once: 750 spilled registers).

__device__ __forceinline__ void rx_half(double& xr, double& xi, double yr, double yi, double t) {
  xr = fma(t, yi, xr);
  xi = fma(-t, yr, xi);
}

__device__ __forceinline__ void rx_pair(double& xr, double& xi, double& yr, double& yi, double t) {
  const double a = t * yi, b = t * yr;
  yr = fma(t, xi, yr);
  yi = fma(-t, xr, yi);
  xr = xr + a;
  xi = xi - b;
}

// One layer's mixer: t, whether it flips, and the factors of k = 0..kMaxT
// bits, (1 + t^2)^(-k/2), which keep the norm where c^k with a rounded c is off
// the same way at every layer (and so is a power of one rounded factor: they
// carry their error along).  Against 80-bit floats, 8 to 16 qubits and 2 to 8
// layers, values are 0.9e-15 off and gradients 2.6e-15 (rms, relative), where
// c x - i s y left 1.7e-15 and 3.4e-15.
struct Mixer {
  double t, flip, scale[kMaxT + 1];
};
constexpr int kMixerEntries = sizeof(Mixer) / sizeof(v2d);
static_assert(sizeof(Mixer) % sizeof(v2d) == 0, "whole complex entries");

__device__ __forceinline__ void make_mixer(double sn, double cs, v2d* to) {
  Mixer& m = *reinterpret_cast<Mixer*>(to);
  const bool flip = fabs(cs) < fabs(sn);
  const double t = flip ? -cs / sn : sn / cs;
  m.t = t;
  m.flip = flip ? 1.0 : 0.0;
  const double q = fma(t, t, 1.0), ql = fma(t, t, 1.0 - q);
  const double r = 1.0 / sqrt(q), r2 = r * r, r2l = fma(r, r, -r2);
  const double rl = -0.5 * r * (fma(r2, q, -1.0) + fma(r2l, q, r2 * ql));
  double h = 1.0, l = 0.0;
  for (int k = 0; k <= kMaxT; ++k) {
    m.scale[k] = h;
    const double x = h * r, e = fma(h, r, -x) + fma(h, rl, l * r);
    h = x + e;
    l = e - (h - x);
  }
}

__device__ __forceinline__ void scale_by(double& xr, double& xi, const v2d ph) {
  const double a = ph.y * xi, b = ph.y * xr;
  xr = fma(ph.x, xr, -a);
  xi = fma(ph.x, xi, b);
}

// A scheduling fence after every N-th step of an unrolled loop over a lane's
// amplitudes, which would otherwise keep the temporaries of all of them.
template <int N>
__device__ __forceinline__ void fence_every(int i) {
  if (i % N == N - 1) __builtin_amdgcn_sched_barrier(0);
}

// Im conj(l) p: half of a pair's term of the beta gradient
__device__ __forceinline__ double im_dot(double lr, double li, double pr, double pi, double g) {
  return fma(lr, pi, fma(-li, pr, g));
}

// The amplitudes a lane holds of its tile, psi and (BWD) lambda, their real
// and imaginary parts apart: as 2-vectors every update built a new register
// tuple.
template <int R, bool BWD>
struct Tile {
  static constexpr int N = 1 << R;
  double vr[N], vi[N];
  double lr[BWD ? N : 1], li[BWD ? N : 1];
};

// RX on register bit J, and its terms of the gradient (LAM).
template <int J, bool LAM, int R, bool BWD>
__device__ __forceinline__ void rx_reg(Tile<R, BWD>& t, double tn, double q, double& g) {
#pragma unroll
  for (int r = 0; r < (1 << R); ++r) {
    if (r & (1 << J)) continue;
    const int o = r | (1 << J);
    if constexpr (LAM) {
      g = im_dot(t.lr[r], t.li[r], t.vr[o], t.vi[o],
                 im_dot(t.lr[o], t.li[o], t.vr[r], t.vi[r], g));
      rx_pair(t.lr[r], t.li[r], t.lr[o], t.li[o], tn);
    }
    rx_pair(t.vr[r], t.vi[r], t.vr[o], t.vi[o], tn);
    fence_every<2>(r);
  }
  g *= q;
}

// RX on the register bits of `mask`; bit j is tile bit j + first (kBaseBits and
// up, or the wave bits in their place).
template <bool LAM, int R, bool BWD>
__device__ __forceinline__ void rx_regs(Tile<R, BWD>& t, unsigned mask, double tn, double q,
                                        double& g) {
  if constexpr (R >= 1) if (mask & 1u) rx_reg<0, LAM>(t, tn, q, g);      // uniform
  if constexpr (R >= 2) if (mask & 2u) rx_reg<1, LAM>(t, tn, q, g);
  if constexpr (R >= 3) if (mask & 4u) rx_reg<2, LAM>(t, tn, q, g);
  if constexpr (R >= 4) if (mask & 8u) rx_reg<3, LAM>(t, tn, q, g);
}

// RX on lane bit B, partners by lane exchange.
template <int B, bool LAM, int R, bool BWD>
__device__ __forceinline__ void rx_lane(Tile<R, BWD>& t, double tn, double q, double& g) {
#pragma unroll
  for (int r = 0; r < (1 << R); ++r) {
    const double yr = from_lane<B>(t.vr[r]), yi = from_lane<B>(t.vi[r]);
    if constexpr (LAM) {
      const double mr = from_lane<B>(t.lr[r]), mi = from_lane<B>(t.li[r]);
      g = im_dot(t.lr[r], t.li[r], yr, yi, g);
      rx_half(t.lr[r], t.li[r], mr, mi, tn);
    }
    rx_half(t.vr[r], t.vi[r], yr, yi, tn);
    fence_every<4>(r);
  }
  g *= q;
}

// Exchanges lane bit B (4 or 5) with register bit 0.
template <int B, bool LAM, int R, bool BWD>
__device__ __forceinline__ void swap_lane_reg(Tile<R, BWD>& t) {
#pragma unroll
  for (int r = 0; r < (1 << R); r += 2) {
    swap_lane_bit<B>(t.vr[r], t.vr[r + 1]);
    swap_lane_bit<B>(t.vi[r], t.vi[r + 1]);
    if constexpr (LAM) {
      swap_lane_bit<B>(t.lr[r], t.lr[r + 1]);
      swap_lane_bit<B>(t.li[r], t.li[r + 1]);
    }
    fence_every<4>(r / 2);
  }
}

// Exchanges the wave bits with register bits 0-2: an 8 x 8 transpose of
// 64-lane rows through LDS, 8 amplitudes a lane at a time.
template <int R>
__device__ __forceinline__ void exchange(double (&vr)[1 << R], double (&vi)[1 << R], v2d* buf,
                                         unsigned wave, unsigned lane) {
#pragma unroll
  for (int h = 0; h < (1 << R); h += 8) {
    __syncthreads();
#pragma unroll
    for (int q = 0; q < 8; ++q) buf[(q * kWaves + wave) * 64 + lane] = v2d{vr[h + q], vi[h + q]};
    __syncthreads();
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      const v2d x = buf[(wave * kWaves + q) * 64 + lane];
      vr[h + q] = x.x;
      vi[h + q] = x.y;
    }
  }
}

// RX on wave bit i of a tile too small for the exchange: partners by LDS.
template <bool LAM, int R, bool BWD>
__device__ __forceinline__ void rx_wave(Tile<R, BWD>& t, int i, double tn, double q, double& g,
                                        v2d* buf) {
  constexpr int N = 1 << R;
  static_assert(N * (BWD ? 2 : 1) <= 8, "fits the exchange buffer");
  const unsigned me = threadIdx.x, other = me ^ (64u << i);
  __syncthreads();
#pragma unroll
  for (int r = 0; r < N; ++r) {
    buf[r * kThreads + me] = v2d{t.vr[r], t.vi[r]};
    if constexpr (LAM) buf[(N + r) * kThreads + me] = v2d{t.lr[r], t.li[r]};
  }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < N; ++r) {
    const v2d y = buf[r * kThreads + other];
    if constexpr (LAM) {
      const v2d m = buf[(N + r) * kThreads + other];
      g = im_dot(t.lr[r], t.li[r], y.x, y.y, g);
      rx_half(t.lr[r], t.li[r], m.x, m.y, tn);
    }
    rx_half(t.vr[r], t.vi[r], y.x, y.y, tn);
  }
  g *= q;
}

// Where the tile bits sit: `waves` while the wave bits and register bits 0-2
// are exchanged, `lanes` while register bit 0, lane bit 5 and lane bit 4 are
// rotated (register 0 holds lane bit 5, lane bit 5 holds 4, lane bit 4 holds
// register 0).
struct Order {
  unsigned waves = 0, lanes = 0;
};

// RX on the tile bits of `mask`, without the factor of its bits.  LAM: on
// lambda too, and returns the lane's gradient terms in units of the factors
// squared: <lambda|X|psi> of one bit is the same before and after RX on
// another, so each is taken on the way, and g *= q = 1 + t^2 brings the earlier
// ones to the unit of the next.
template <bool LAM, int R, bool BWD>
__device__ __forceinline__ double rx_mask(Tile<R, BWD>& t, unsigned mask, double tn, double q,
                                          Order& o, v2d* buf) {
  double g = 0.0;
  if (mask & 1u) rx_lane<0, LAM>(t, tn, q, g);
  if (mask & 2u) rx_lane<1, LAM>(t, tn, q, g);
  if (mask & 4u) rx_lane<2, LAM>(t, tn, q, g);
  if (mask & 8u) rx_lane<3, LAM>(t, tn, q, g);
  const unsigned mid = (mask >> kLaneBits) & 7u, high = mask >> kBaseBits;
  unsigned l45 = mask & 48u;
  if constexpr (R == 0) {
    if (l45 & 16u) rx_lane<4, LAM>(t, tn, q, g);
    if (l45 & 32u) rx_lane<5, LAM>(t, tn, q, g);
  } else if (o.lanes && (mask >> 4)) {
    if (l45 & 32u) rx_reg<0, LAM>(t, tn, q, g);
    swap_lane_reg<5, LAM>(t);
    if (l45 & 16u) rx_reg<0, LAM>(t, tn, q, g);
    swap_lane_reg<4, LAM>(t);
    o.lanes = l45 = 0;
  }
  if constexpr (R >= 3) {
    // the three bits now in registers 0-2, the three now across waves; bit 12
    // (register bit 3) goes with the first
    unsigned here = o.waves ? mid | (high & 8u) : high;
    const unsigned there = o.waves ? high & 7u : mid;
    for (int half = 0;; ++half) {
      rx_regs<LAM>(t, here, tn, q, g);
      if (half || !there) break;
      const unsigned wave = threadIdx.x >> 6, lane = threadIdx.x & 63u;
      exchange<R>(t.vr, t.vi, buf, wave, lane);
      if constexpr (LAM) exchange<R>(t.lr, t.li, buf, wave, lane);
      o.waves ^= 1u;
      here = there;
    }
  } else {
    rx_regs<LAM>(t, high, tn, q, g);
    for (int i = 0; i < kWaveBits; ++i)
      if ((mid >> i) & 1u) rx_wave<LAM>(t, i, tn, q, g, buf);
  }
  if constexpr (R > 0) {
    if (l45) {
      swap_lane_reg<4, LAM>(t);
      if (l45 & 16u) rx_reg<0, LAM>(t, tn, q, g);
      swap_lane_reg<5, LAM>(t);
      if (l45 & 32u) rx_reg<0, LAM>(t, tn, q, g);
      o.lanes = 1;
    }
  }
  return g;
}

// RX with its factor; returns the lane's gradient terms (LAM).
template <bool LAM, int R, bool BWD>
__device__ __forceinline__ double mix(Tile<R, BWD>& t, unsigned mask, double tn, double scale,
                                      Order& o, v2d* buf) {
  const double g = rx_mask<LAM>(t, mask, tn, fma(tn, tn, 1.0), o, buf);
#pragma unroll
  for (int r = 0; r < (1 << R); ++r) {
    t.vr[r] *= scale;
    t.vi[r] *= scale;
    if constexpr (LAM) {
      t.lr[r] *= scale;
      t.li[r] *= scale;
    }
    fence_every<4>(r);
  }
  return g * scale * scale;
}

// exp(i g (W/2 - c)), c = 0..ncut, into tab (conjugated for the way back)
__device__ __forceinline__ void phase_table(v2d* tab, int ncut, double g, double wsum, bool conj) {
  for (int c = threadIdx.x; c <= ncut; c += kThreads) {
    double sn, cs;
    sincos_held(g * (0.5 * wsum - (double)c), &sn, &cs);
    tab[c] = v2d{cs, conj ? -sn : sn};
  }
}

// Indices of a lane's amplitudes in the current order: element r sits at
// at(r), kept at stored(at(r)).
struct Index {
  uint32_t lane[2];          // the share of lane bits 0-3 and the wave bits, by Order::waves
  uint32_t reg[2][4];        // index bit of register bit j, by Order::waves
  uint32_t bit4, bit5;       // index bits of lane bits 4 and 5
  uint32_t mmask;            // mirror instances: all n index bits; else 0
  int mshift;                // mirror instances: n - 1

  // Where the amplitude of full-state index z is kept: a mirror instance keeps
  // only the indices with bit n-1 clear, and one with it set is the
  // complementary index (MaxCut states are symmetric under flipping every
  // bit); other instances keep z itself.
  __device__ __forceinline__ uint32_t stored(uint32_t z) const {
    return z ^ (mmask & (0u - ((z >> mshift) & 1u)));
  }

  // element 0 and the bits of the others
  template <int R>
  __device__ __forceinline__ uint32_t share(const Order& o, uint32_t (&h)[4]) const {
#pragma unroll
    for (int j = 0; j < R; ++j) h[j] = o.waves ? reg[1][j] : reg[0][j];
    uint32_t at4 = bit4, at5 = bit5;
    if constexpr (R > 0)
      if (o.lanes) {
        at4 = h[0];
        at5 = bit4;
        h[0] = bit5;
      }
    uint32_t z = o.waves ? lane[1] : lane[0];
    if (threadIdx.x & 16u) z ^= at4;
    if (threadIdx.x & 32u) z ^= at5;
    return z;
  }
};

template <int R>
__device__ __forceinline__ uint32_t elem_at(const Index& ix, const Order& o, int r) {
  uint32_t h[4];
  uint32_t z = ix.share<R>(o, h);
#pragma unroll
  for (int j = 0; j < R; ++j)
    if ((r >> j) & 1) z ^= h[j];
  return ix.stored(z);
}

template <int R, int FENCE, typename F>
__device__ __forceinline__ void for_elems(const Index& ix, const Order& o, F&& f) {
  uint32_t h[4];
  const uint32_t z0 = ix.share<R>(o, h);
#pragma unroll
  for (int r = 0; r < (1 << R); ++r) {
    uint32_t x = 0;
#pragma unroll
    for (int j = 0; j < R; ++j) x |= ((r >> j) & 1) ? h[j] : 0u;
    f(r, ix.stored(z0 ^ x));
    fence_every<FENCE>(r);
  }
}

__device__ __forceinline__ bool is_cost(int type) {
  return type == ST_COST || type == ST_COST_RX || type == ST_COST_ADJ;
}

__device__ __forceinline__ bool is_mixer(int type) {
  return type == ST_RX || type == ST_COST_RX || type == ST_RX_LOAD || type == ST_RX_STORE ||
         type == ST_RX_ADJ;
}

// Amplitudes of an instance in a pool.  FLOW: other workgroups' stores of
// this launch are read without a cache flush in between, so loads and stores
// go to memory at agent scope (sc1: past this XCD's L2 where another XCD may
// hold newer data); 16 bytes a lane as the buffer forms take, which is why the
// pool of one instance stays under 2^31 bytes.
// No release or acquire fence is needed beside them: at agent scope these
// write the L2 back and drop its lines, for accesses that stop there, and the
// pools' do not.  What is needed is order.  A workgroup's stores have reached
// memory before it counts its item (stores_done, then the barrier, then one
// lane's atomic, itself at agent scope); a workgroup loads only after the count
// was seen (one lane polls, then the barrier, which the compiler moves no
// access across).  The pools are all that passes between workgroups of a
// launch: tables come from the kernel before, partial sums go to the one after.
template <bool FLOW>
struct Pool;

template <>
struct Pool<false> {
  v2d* p;
  __device__ __forceinline__ Pool(v2d* base, uint64_t) : p(base) {}
  __device__ __forceinline__ v2d load(uint32_t z) const { return p[z]; }
  __device__ __forceinline__ void store(uint32_t z, v2d x) const { p[z] = x; }
};

template <>
struct Pool<true> {
  static constexpr int kRaw = 0x00020000, kAgent = 16;
  typedef unsigned v4u __attribute__((ext_vector_type(4)));
  __amdgpu_buffer_rsrc_t r;
  __device__ __forceinline__ Pool(v2d* base, uint64_t len)
      : r(__builtin_amdgcn_make_buffer_rsrc(base, 0, (uint32_t)(len * sizeof(v2d)), kRaw)) {}
  __device__ __forceinline__ v2d load(uint32_t z) const {
    return __builtin_bit_cast(v2d, __builtin_amdgcn_raw_buffer_load_b128(r, (int)(z << 4), 0, kAgent));
  }
  __device__ __forceinline__ void store(uint32_t z, v2d x) const {
    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(v4u, x), r, (int)(z << 4), 0, kAgent);
  }
};

// Waits until this wave's stores have been taken; a workgroup barrier alone
// does not.
__device__ __forceinline__ void stores_done() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

// The launch's counters at the head of its tables: items taken from each
// XCD's share, then items finished of each instance.
constexpr int kXcds = 8;
constexpr int kWorkStride = 16;        // 64 bytes apart
constexpr int kDoneAt = kXcds * kWorkStride, kDoneStride = 4;

// The item after `now`: FLOW takes the next of the workgroup's XCD's.
template <bool FLOW>
__device__ __forceinline__ int next_item(unsigned* work, int now) {
  if constexpr (!FLOW) return now + (int)gridDim.x;
  if (gridDim.x % kXcds) return (int)atomicAdd(work, 1u);
  const unsigned x = blockIdx.x % kXcds;
  return (int)(x + kXcds * atomicAdd(work + kWorkStride * x, 1u));
}

// One work item.  BWD selects the kernel of a mode: the forward kernel holds
// no adjoint stages.
template <int R, bool BWD, bool FLOW, bool WTD>
__device__ __forceinline__ void run_item(const qfx_qaoa_inst& in, const qfx_qaoa_pass& ps,
                                         uint32_t tile, const double* __restrict__ angles,
                                         v2d* __restrict__ psi_pool, v2d* __restrict__ lam_pool,
                                         const uint16_t* __restrict__ cnt_pool,
                                         const double* __restrict__ val_pool,
                                         double* __restrict__ partial, int width, v2d* buf,
                                         double* acc, v2d* tab, v2d* mixers,
                                         const v2d* __restrict__ made, unsigned* work,
                                         int* next) {
  const int T = R ? kBaseBits + R : ps.T;
  const int p = in.p;
  const double* beta = angles + in.angle_off;
  const double* gamma = beta + p;
  const bool unit = !WTD || !in.weighted;
  const uint16_t* cnt = cnt_pool + in.cut_off;
  const double* cval = val_pool + in.cut_off;
  const uint64_t kept = (uint64_t)1 << (in.n - in.mirror);
  const Pool<FLOW> psi(psi_pool + in.psi_off, kept);
  const Pool<FLOW> lam(BWD ? lam_pool + in.lam_off : psi_pool, kept);
  const unsigned lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;

  Index ix;
  ix.mmask = in.mirror ? (uint32_t)(((uint64_t)1 << in.n) - 1) : 0u;
  ix.mshift = in.mirror ? in.n - 1 : 0;
  uint32_t base = tile;
#pragma unroll
  for (int j = 0; j < kMaxT; ++j)
    if (j < T) {
      const uint32_t low = (1u << ps.pos[j]) - 1u;
      base = ((base & ~low) << 1) | (base & low);
    }
  uint32_t zl = base, wa = 0, wb = 0;
  const unsigned tl = tile_lane(lane);
#pragma unroll
  for (int j = 0; j < 4; ++j)
    if (j < T) zl |= ((tl >> j) & 1u) << ps.pos[j];
  ix.bit4 = 4 < T ? 1u << ps.pos[4] : 0u;
  ix.bit5 = 5 < T ? 1u << ps.pos[5] : 0u;
#pragma unroll
  for (int j = 0; j < kWaveBits; ++j) {
    if (kLaneBits + j < T) wa |= ((wave >> j) & 1u) << ps.pos[kLaneBits + j];
    if constexpr (R >= 3) wb |= ((wave >> j) & 1u) << ps.pos[kBaseBits + j];
  }
  ix.lane[0] = zl | wa;
  ix.lane[1] = zl | wb;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    ix.reg[0][j] = j < R ? 1u << ps.pos[kBaseBits + j] : 0u;
    ix.reg[1][j] = j < R ? 1u << ps.pos[j < 3 ? kLaneBits + j : kBaseBits + j] : 0u;
  }
  const bool live = R > 0 || threadIdx.x < (1u << T);

  bool sums = false;
  for (int si = 0; si < ps.nstage; ++si) {
    const int ty = ps.stage[si][0];
    sums |= ty == ST_EXPECT || ty == ST_RX_ADJ || ty == ST_COST_ADJ;
  }
  int ncost = 0;
  for (int si = 0; si < ps.nstage; ++si) ncost += is_cost(ps.stage[si][0]);
  Tile<R, BWD> t;
  Order order;
  if ((ps.flags & PF_LOAD_PSI) && live)
    for_elems<R, 4>(ix, order, [&](int r, uint32_t z) {
      const v2d x = psi.load(z);
      t.vr[r] = x.x;
      t.vi[r] = x.y;
    });
  else
#pragma unroll
    for (int r = 0; r < (1 << R); ++r) t.vr[r] = t.vi[r] = 0.0;
  bool with_lam = BWD && (ps.flags & PF_LOAD_LAM);
  if constexpr (BWD) {
    if ((ps.flags & PF_LOAD_LAM) && live)
      for_elems<R, 4>(ix, order, [&](int r, uint32_t z) {
        const v2d x = lam.load(z);
        t.lr[r] = x.x;
        t.li[r] = x.y;
      });
    else
#pragma unroll
      for (int r = 0; r < (1 << R); ++r) t.lr[r] = t.li[r] = 0.0;
  }
  // Angles and phase tables of the pass's layers: copied from the launch's
  // tables or, without them, made here.  A pass with more cost layers than fit
  // takes each table when it comes to it.
  const int tabsize = in.nedges + 1;
  const bool ahead = unit && ncost * tabsize <= kMaxEdgesTab;
  const int made_stride = kMixerEntries + (unit ? tabsize : 0);
  auto table = [&](v2d* to, int layer, bool conj) {
    if constexpr (FLOW) {
      for (int c = threadIdx.x; c < tabsize; c += kThreads) {
        const v2d x = made[layer * made_stride + kMixerEntries + c];
        to[c] = v2d{x.x, conj ? -x.y : x.y};
      }
    } else {
      phase_table(to, in.nedges, gamma[layer], in.wsum, conj);
    }
  };
  __syncthreads();
  if (ahead && ncost) {
    int c = 0;
    for (int si = 0; si < ps.nstage; ++si) {
      const int ty = ps.stage[si][0];
      if (is_cost(ty)) table(tab + c++ * tabsize, ps.stage[si][1], ty == ST_COST_ADJ);
    }
  }
  if constexpr (FLOW) {
    for (int c = threadIdx.x; c < p * kMixerEntries; c += kThreads)
      mixers[c] = made[c / kMixerEntries * made_stride + c % kMixerEntries];
  } else {
    if ((int)threadIdx.x >= kThreads - 64 && (int)lane < p) {
      double sn, cs;
      sincos_held(0.5 * beta[lane], &sn, &cs);
      make_mixer(sn, cs, mixers + lane * kMixerEntries);
    }
  }
  __syncthreads();
  int ci = 0;                // cost layers so far

  // acc[j * kWaves + wave]: each wave's sums, its own to clear and to add to
  if (lane < kAccum) acc[lane * kWaves + wave] = 0.0;
  auto add = [&](int j, double v) {
    v = wave_sum(v);
    if (lane == 0) acc[j * kWaves + wave] += v;
  };

  for (int si = 0; si < ps.nstage; ++si) {
    const int type = ps.stage[si][0], layer = ps.stage[si][1];
    const unsigned mask = (unsigned)ps.stage[si][2];
    if (type == ST_COST || type == ST_COST_RX || (BWD && type == ST_COST_ADJ)) {
      const double g = gamma[layer];
      const bool adj = BWD && type == ST_COST_ADJ;
      const v2d* tb = ahead ? tab + ci * tabsize : tab;
      ++ci;
      if (unit && !ahead) {
        __syncthreads();
        table(tab, layer, adj);
        __syncthreads();
      }
      double sum = 0.0;
      auto cost = [&](int r, const v2d ph, double cz) {
        if constexpr (BWD) {
          if (adj) {
            const double ip = im_dot(t.lr[r], t.li[r], t.vr[r], t.vi[r], 0.0);  // conj(l) psi
            sum += 2.0 * cz * ip - in.wsum * ip;
            scale_by(t.lr[r], t.li[r], ph);
          }
        }
        scale_by(t.vr[r], t.vi[r], ph);
      };
      if (unit) {
        // all counts in flight before the first phase is looked up
        int kc[1 << R];
        for_elems<R, 4>(ix, order, [&](int r, uint32_t z) { kc[r] = live ? cnt[z] : 0; });
#pragma unroll
        for (int r = 0; r < (1 << R); ++r) {
          cost(r, tb[kc[r]], (double)kc[r]);
          fence_every<4>(r);
        }
      } else if constexpr (WTD) {
        // phases into the lane's own slots of the exchange buffer, one sincos
        // at a time
        constexpr int N = 1 << R, kPart = N < 8 ? N : 8;
#pragma unroll
        for (int h = 0; h < N; h += kPart) {
          __syncthreads();
#pragma unroll 1
          for (int q = 0; live && q < kPart; ++q) {
            double sn, cs;
            sincos_held(g * (0.5 * in.wsum - cval[elem_at<R>(ix, order, h + q)]), &sn, &cs);
            buf[q * kThreads + threadIdx.x] = v2d{cs, adj ? -sn : sn};
          }
          if (live) {
#pragma unroll
            for (int q = 0; q < kPart; ++q)
              cost(h + q, buf[q * kThreads + threadIdx.x], cval[elem_at<R>(ix, order, h + q)]);
          }
        }
      }
      if (adj) add(1 + p + layer, sum);
    }
    if (is_mixer(type)) {
      const bool adj = BWD && type == ST_RX_ADJ;
      const Mixer& mx = *reinterpret_cast<const Mixer*>(mixers + layer * kMixerEntries);
      const double tn = uniform_d(adj ? -mx.t : mx.t);
      const double scale = uniform_d(mx.scale[__popc(mask)]);
      if (__builtin_amdgcn_readfirstlane((int)mx.flip)) {
        uint32_t flip = 0;
        for (int j = 0; j < T; ++j) flip |= ((mask >> j) & 1u) << ps.pos[j];
        ix.lane[0] ^= flip;
        ix.lane[1] ^= flip;
      }
      double g = 0.0;
      if constexpr (BWD) {
        if (with_lam || adj) g = mix<true>(t, mask, tn, scale, order, buf);
        else mix<false>(t, mask, tn, scale, order, buf);
      } else {
        mix<false>(t, mask, tn, scale, order, buf);
      }
      if (adj) add(1 + layer, g);
    }
    if (type == ST_INIT) {
      const double a = ldexp(1.0, -(in.n / 2)) * ((in.n & 1) ? 0.70710678118654752440 : 1.0);
#pragma unroll
      for (int r = 0; r < (1 << R); ++r) {
        t.vr[r] = live ? a : 0.0;
        t.vi[r] = 0.0;
      }
    }
    if (type == ST_EXPECT || (BWD && type == ST_MAKE_LAMBDA)) {
      double sum = 0.0;
      double cut[1 << R];
      for_elems<R, 4>(ix, order, [&](int r, uint32_t z) {
        if constexpr (WTD) cut[r] = !live ? 0.0 : (unit ? (double)cnt[z] : cval[z]);
        else cut[r] = live ? (double)cnt[z] : 0.0;
      });
#pragma unroll
      for (int r = 0; r < (1 << R); ++r) {
        const double cz = cut[r];
        if (type == ST_EXPECT) sum += fma(t.vr[r], t.vr[r], t.vi[r] * t.vi[r]) * cz;
        if constexpr (BWD)
          if (type == ST_MAKE_LAMBDA) {
            t.lr[r] = cz * t.vr[r];
            t.li[r] = cz * t.vi[r];
          }
        fence_every<4>(r);
      }
      if (type == ST_EXPECT) add(0, sum);
      if (BWD && type == ST_MAKE_LAMBDA) with_lam = true;
    }
  }
  if (threadIdx.x == 0) *next = next_item<FLOW>(work, *next);
  if ((ps.flags & PF_STORE_PSI) && live)
    for_elems<R, 4>(ix, order, [&](int r, uint32_t z) { psi.store(z, v2d{t.vr[r], t.vi[r]}); });
  if constexpr (BWD) {
    if ((ps.flags & PF_STORE_LAM) && live)
      for_elems<R, 4>(ix, order, [&](int r, uint32_t z) { lam.store(z, v2d{t.lr[r], t.li[r]}); });
  }
  if (sums) {
    __syncthreads();
    if ((int)threadIdx.x < width) {
      double v = 0.0;
      for (int w = 0; w < kWaves; ++w) v += acc[threadIdx.x * kWaves + w];
      partial[threadIdx.x] = v;
    }
  } else if ((int)threadIdx.x < width) {
    partial[threadIdx.x] = 0.0;
  }
  stores_done();
  __syncthreads();
}

// Waits for *counter to reach target, bounded by the device's constant-rate
// wall clock (limit_ticks); on timeout it sets this launch's error flag
// (err[0], which makes every waiting workgroup leave too) and the sticky flag
// (err[1], cleared only by the batch's owner), and returns false.  Relaxed
// polls: an acquiring one drops the XCD's L2 contents each time, under the
// workgroups still at work.
__device__ bool wait_for(const unsigned* counter, unsigned target, int* err,
                         uint64_t limit_ticks) {
  const uint64_t t0 = wall_clock64();
  while (__hip_atomic_load(counter, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < target) {
    __builtin_amdgcn_s_sleep(8);
    if (__hip_atomic_load(err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) ||
        wall_clock64() - t0 > limit_ticks) {
      atomicExch(err, 1);
      atomicOr(err + 1, 1);
      return false;
    }
  }
  return true;
}

// Grid barrier on a monotone counter.
__device__ bool grid_barrier(unsigned* counter, unsigned target, int* err,
                             uint64_t limit_ticks) {
  stores_done();
  __syncthreads();
  __shared__ int s_ok;
  if (threadIdx.x == 0) {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
    __hip_atomic_fetch_add(counter, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    s_ok = wait_for(counter, target, err, limit_ticks);
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
  }
  __syncthreads();
  return s_ok != 0;
}

// The persistent kernel.  FLOW: workgroups take items off the list (the next
// of their XCD's share, so that items which share lines share an L2) and wait
// for what an item needs by its instance's count of finished items; no cache
// is flushed, as the state's loads and stores pass the L2 at agent scope
// (Pool).  An item needs only items before it on the list, each taken by a
// workgroup that runs (the first one as well: where another launch holds part
// of the CUs, an item named by blockIdx would wait for a workgroup that has
// not started), so the first unfinished one can always go on.  Else:
// items in turn, and a grid barrier with a cache flush after each pass.  WTD:
// the launch may hold weighted instances, whose phases are made in place.
// WIDE: 256 registers a lane and one workgroup a CU, for 13-bit tiles of psi
// and lambda, and for 12-bit ones where phases are made in place (in 128
// registers 81 were spilled, into the sincos loop: 8 weighted instances of 12
// qubits and 4 layers 165 us, now 86; 512 of 14 978, now 571); all else fits 128
// registers and two.
//
// What bounds it: with its tile in registers an item of 13 bits backward takes
// 25 us a layer on the way there and 45 us back on its CU, of which the mixer's
// arithmetic is 5.5 and 13 us (512 lanes; 17 us each with the two products a
// component and lambda carried along all the way), loads and stores through
// the memory system 10-15 us each way, the cost layer 4.  The same with tiles
// in LDS, four bits to a sweep of it, and one grid barrier a pass: 104
// forward instances of 10 to 22 qubits and 4 layers 2615 us, now 860; 15
// backward of 16 to 24 and 8 layers 21.7 ms, now 12.0.  Of that the registers
// gave 2615 -> 1750 and 21.7 -> 17.0, polls of the barrier that leave the L2
// alone 1500 and 15.2, items instead of barriers 1190 (and for 64 instances
// of 16 qubits backward 1.29 -> 0.55 ms), t the rest.
template <bool BWD, bool FLOW, bool WTD, bool WIDE>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(BWD && WIDE ? 2 : 4)))
void qaoa_kernel(
    const qfx_qaoa_inst* __restrict__ insts, const qfx_qaoa_pass* __restrict__ passes,
    const qfx_qaoa_item* __restrict__ items, const int* __restrict__ kstart, int nk,
    const double* __restrict__ angles, v2d* __restrict__ psi_pool, v2d* __restrict__ lam_pool,
    const uint16_t* __restrict__ cnt_pool, const double* __restrict__ val_pool,
    double* __restrict__ partials, int width, unsigned* sync, int* err, uint64_t limit_ticks,
    uint64_t* __restrict__ timing, int64_t timing_len, v2d* tables,
    const int64_t* __restrict__ table_off, const int* __restrict__ item_need) {
  extern __shared__ v2d buf[];
  __shared__ double acc[kAccum * kWaves];
  __shared__ v2d tab[kMaxEdgesTab], mixers[kMaxPLayers * kMixerEntries];
  __shared__ int s_next, s_ok;
  unsigned* work = reinterpret_cast<unsigned*>(tables);
  // one pass: no item waits, and the first one is named by blockIdx (600 values
  // of 10 qubits: 29.3 us, else 30.1)
  int next = blockIdx.x;
  if (threadIdx.x == 0) s_next = !FLOW || nk == 1 ? next : next_item<FLOW>(work, next);
  if (FLOW && nk > 1) {
    __syncthreads();
    next = __builtin_amdgcn_readfirstlane(s_next);
  }
  for (int k = 0; k < nk; ++k) {
    const int64_t tslot = 2 * ((int64_t)k * gridDim.x + blockIdx.x);
    const bool timed = timing != nullptr && tslot + 1 < timing_len && threadIdx.x == 0;
    if (timed) timing[tslot] = wall_clock64();
    for (const int end = kstart[k + 1]; next < end;) {
      const qfx_qaoa_item item = items[next];
      if constexpr (FLOW) {
        const int need = item_need[next];
        if (need > 0) {
          if (threadIdx.x == 0)
            s_ok = wait_for(work + kDoneAt + kDoneStride * item.inst, (unsigned)need, err,
                            limit_ticks);
          __syncthreads();
          if (!s_ok) return;
        }
      }
      const qfx_qaoa_inst& in = insts[item.inst];
      const qfx_qaoa_pass& ps = passes[item.pass];
      double* part = partials + (uint64_t)item.partial * width;
      const v2d* made = FLOW ? tables + table_off[item.inst] : nullptr;
      auto run = [&](auto r) {
        run_item<decltype(r)::value, BWD, FLOW, WTD>(in, ps, (uint32_t)item.tile, angles, psi_pool, lam_pool,
                                          cnt_pool, val_pool, part, width, buf, acc, tab, mixers, made,
                                          work, &s_next);
      };
      switch (ps.T) {
        case 13: if constexpr (!BWD || WIDE) run(std::integral_constant<int, 4>{}); break;
        case 12: if constexpr (!BWD || WIDE || !WTD) run(std::integral_constant<int, 3>{}); break;
        case 11: run(std::integral_constant<int, 2>{}); break;
        case 10: run(std::integral_constant<int, 1>{}); break;
        default: run(std::integral_constant<int, 0>{}); break;
      }
      next = __builtin_amdgcn_readfirstlane(s_next);
      if (FLOW && threadIdx.x == 0)
        __hip_atomic_fetch_add(work + kDoneAt + kDoneStride * item.inst, 1u, __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_AGENT);
    }
    if (timed) timing[tslot + 1] = wall_clock64();
    if (!FLOW && k + 1 < nk && !grid_barrier(sync, (unsigned)(k + 1) * gridDim.x, err, limit_ticks))
      return;
  }
}

// out[i * width + j] = sum of the instance's partial slots: one workgroup
// per output, a fixed strided split over its threads and a fixed-order tree
// (bitwise reproducible).
constexpr int kReduceBlock = 256;

__global__ __launch_bounds__(kReduceBlock) void qaoa_reduce_kernel(
    const qfx_qaoa_inst* __restrict__ insts, int ninst, const double* __restrict__ partials,
    int width, double* __restrict__ out) {
  const int i = blockIdx.x;
  const int inst = i / width, j = i % width;
  const qfx_qaoa_inst& in = insts[inst];
  double s = 0.0;
  for (int q = threadIdx.x; q < in.nslots; q += kReduceBlock)
    s += partials[(uint64_t)(in.slot0 + q) * width + j];
  __shared__ double red[kReduceBlock / 64];
  s = wave_sum(s);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
  __syncthreads();
  // a mirror instance's items each stand for their tile and its complement
  if (threadIdx.x == 0) out[i] = ((red[0] + red[1]) + (red[2] + red[3])) * (in.mirror ? 2.0 : 1.0);
}

// Resets the barrier (workgroup 0) and makes the launch's tables, one
// instance and layer a workgroup: {cos, sin}(beta/2), then (unit weights)
// exp(i gamma (W/2 - c)) for every cut count c.  Made by each item for itself,
// they cost it a sincos and two barriers before its first load.
constexpr int kPrepBlock = 256;

__global__ __launch_bounds__(kPrepBlock) void prepare_kernel(
    unsigned* sync, int* err, const qfx_qaoa_inst* __restrict__ insts,
    const double* __restrict__ angles, v2d* __restrict__ tables,
    const int64_t* __restrict__ table_off, unsigned taken) {
  if (blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x == 0) {
    sync[0] = 0u;
    err[0] = 0;
  }
  if (!tables) return;
  unsigned* work = reinterpret_cast<unsigned*>(tables);
  if (blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x < kXcds)
    work[kWorkStride * threadIdx.x] = taken;
  if (blockIdx.y == 0 && threadIdx.x == 0) work[kDoneAt + kDoneStride * blockIdx.x] = 0u;
  const qfx_qaoa_inst& in = insts[blockIdx.x];
  const int layer = blockIdx.y;
  if (layer >= in.p) return;
  const int n = in.weighted ? 0 : in.nedges + 1;
  v2d* to = tables + table_off[blockIdx.x] + (int64_t)layer * (kMixerEntries + n);
  const double g = angles[in.angle_off + in.p + layer], b = angles[in.angle_off + layer];
  for (int c = (int)threadIdx.x - 1; c < n; c += kPrepBlock) {
    double sn, cs;
    sincos(c < 0 ? 0.5 * b : g * (0.5 * in.wsum - (double)c), &sn, &cs);
    if (c < 0) make_mixer(sn, cs, to);
    else to[kMixerEntries + c] = v2d{cs, sn};
  }
}

// Persistent grid of one instantiation on one device: every workgroup that
// fits the device at once (occupancy x CUs for this mode), so all of them are
// resident together and the grid barrier cannot wait on a workgroup that has
// not started.  Made once per device; other threads wait until it is whole.
struct Grid {
  int grid = 0;
  uint64_t limit_ticks = 0;
};

int make_grid(const void* fn, size_t lds, int dev, Grid* to) {
  int rc = qfx::check_hip(
      hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds),
      "hipFuncSetAttribute");
  if (rc) return rc;
  int per_cu = 0, cus = 0, rate_khz = 0;
  rc = qfx::check_hip(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, fn, kThreads, lds),
                      "hipOccupancyMaxActiveBlocksPerMultiprocessor");
  if (rc) return rc;
  if (per_cu < 1) return qfx::set_error(QFX_ERANGE, "qfx_qaoa_run: kernel does not fit a CU");
  rc = qfx::check_hip(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev),
                      "hipDeviceGetAttribute");
  if (rc) return rc;
  rc = qfx::check_hip(hipDeviceGetAttribute(&rate_khz, hipDeviceAttributeWallClockRate, dev),
                      "hipDeviceGetAttribute");
  if (rc) return rc;
  if (rate_khz <= 0) return qfx::set_error(QFX_EKERNEL, "qfx_qaoa_run: no wall-clock rate");
  to->grid = per_cu * cus;
  to->limit_ticks = (uint64_t)rate_khz * 1000u * kBarrierSeconds;
  return QFX_OK;
}

template <bool BWD, bool FLOW, bool WTD, bool WIDE>
int launch_qaoa(hipStream_t s, const qfx_qaoa_args& a) {
  const size_t lds = sizeof(v2d) * kExchange;
  static std::mutex mu;
  static Grid made[kMaxDevices];
  int dev = 0;
  int rc = qfx::check_hip(hipGetDevice(&dev), "hipGetDevice");
  if (rc) return rc;
  if (dev < 0 || dev >= kMaxDevices)
    return qfx::set_error(QFX_ERANGE, "qfx_qaoa_run: device index out of range");
  Grid gc;
  {
    std::lock_guard<std::mutex> lock(mu);
    if (made[dev].grid == 0) {
      rc = make_grid((const void*)qaoa_kernel<BWD, FLOW, WTD, WIDE>, lds, dev, &made[dev]);
      if (rc) return rc;
    }
    gc = made[dev];
  }
  int g = gc.grid;
  if (a.max_items_per_k > 0 && a.max_items_per_k < g) g = a.max_items_per_k;
  auto* sync = static_cast<unsigned*>(a.sync);
  auto* err = reinterpret_cast<int*>(sync + 1);
  // items taken before the launch: in one pass, each workgroup's first
  const unsigned taken = a.nk > 1 ? 0u : (unsigned)(g % kXcds ? g : g / kXcds);
  hipLaunchKernelGGL(prepare_kernel, FLOW ? dim3(a.ninst, kMaxPLayers) : dim3(1),
                     dim3(kPrepBlock), 0, s, sync, err,
                     static_cast<const qfx_qaoa_inst*>(a.insts),
                     static_cast<const double*>(a.angles),
                     FLOW ? static_cast<v2d*>(a.tables) : nullptr,
                     static_cast<const int64_t*>(a.table_off), taken);
  rc = qfx::check_launch("prepare_kernel");
  if (rc) return rc;
  hipLaunchKernelGGL((qaoa_kernel<BWD, FLOW, WTD, WIDE>), dim3(g), dim3(kThreads), lds, s,
                     static_cast<const qfx_qaoa_inst*>(a.insts),
                     static_cast<const qfx_qaoa_pass*>(a.passes),
                     static_cast<const qfx_qaoa_item*>(a.items), static_cast<const int*>(a.kstart),
                     a.nk, static_cast<const double*>(a.angles), static_cast<v2d*>(a.psi_pool),
                     static_cast<v2d*>(a.lam_pool), static_cast<const uint16_t*>(a.cnt_pool),
                     static_cast<const double*>(a.val_pool), static_cast<double*>(a.partials),
                     a.width, sync, err, gc.limit_ticks, static_cast<uint64_t*>(a.timing),
                     a.timing ? a.timing_len : (int64_t)0, static_cast<v2d*>(a.tables),
                     static_cast<const int64_t*>(a.table_off),
                     static_cast<const int*>(a.item_need));
  rc = qfx::check_launch("qaoa_kernel");
  if (rc) return rc;
  const int nout = a.ninst * a.width;
  hipLaunchKernelGGL(qaoa_reduce_kernel, dim3(nout), dim3(kReduceBlock), 0, s,
                     static_cast<const qfx_qaoa_inst*>(a.insts), a.ninst,
                     static_cast<const double*>(a.partials), a.width,
                     static_cast<double*>(a.out));
  return qfx::check_launch("qaoa_reduce_kernel");
}

}  // namespace

extern "C" {

int qfx_qaoa_check(const qfx_qaoa_inst* insts, int ninst, const qfx_qaoa_pass* passes,
                   int npasses, const qfx_qaoa_item* items, const int* kstart, int nk, int width,
                   int64_t psi_pool_len, int64_t lam_pool_len, int64_t cnt_pool_len,
                   int64_t val_pool_len, int64_t npartial, int mode, int tile_bits) {
  if (tile_bits < 0 || tile_bits > (mode == QFX_QAOA_BACKWARD ? kMaxT - 1 : kMaxT))
    return qfx::set_error(QFX_ERANGE, "qfx_qaoa_check: tile_bits out of range");
  const int tmax = tile_bits ? tile_bits : kMaxT;
  for (int i = 0; i < ninst; ++i) {
    const qfx_qaoa_inst& in = insts[i];
    if (in.n < 1 || in.n > 30 || in.p < 1 || in.p > kMaxPLayers)
      return qfx::set_error(QFX_ERANGE, "qfx_qaoa_check: n or p out of range");
    const int64_t len = (int64_t)1 << in.n;
    if (in.weighted) {
      if (in.cut_off < 0 || in.cut_off + len > val_pool_len)
        return qfx::set_error(QFX_EINVAL, "qfx_qaoa_check: cut values out of range");
    } else {
      if (in.cut_off < 0 || in.cut_off + len > cnt_pool_len)
        return qfx::set_error(QFX_EINVAL, "qfx_qaoa_check: cut counts out of range");
      if (in.nedges < 0 || in.nedges >= kMaxEdgesTab)
        return qfx::set_error(QFX_ERANGE, "qfx_qaoa_check: too many edges for the phase table");
    }
    if (in.mirror != 0 && in.mirror != 1)
      return qfx::set_error(QFX_EINVAL, "qfx_qaoa_check: mirror must be 0 or 1");
    const int64_t slen = in.mirror ? len / 2 : len;   // amplitudes kept
    if (in.psi_off < 0 || in.psi_off + slen > psi_pool_len)
      return qfx::set_error(QFX_EINVAL, "qfx_qaoa_check: state out of range");
    if (mode == QFX_QAOA_BACKWARD && (in.lam_off < 0 || in.lam_off + slen > lam_pool_len))
      return qfx::set_error(QFX_EINVAL, "qfx_qaoa_check: lambda out of range");
    if (in.slot0 < 0 || in.nslots < 0 || in.slot0 + in.nslots > npartial)
      return qfx::set_error(QFX_EINVAL, "qfx_qaoa_check: partial slots out of range");
  }
  if (width < 1 || width > kAccum)
    return qfx::set_error(QFX_ERANGE, "qfx_qaoa_check: width out of range");
  for (int q = 0; q < npasses; ++q) {
    const qfx_qaoa_pass& ps = passes[q];
    if (ps.T < 1 || ps.T > tmax || ps.nstage < 0 || ps.nstage > QFX_QAOA_MAX_STAGES)
      return qfx::set_error(QFX_ERANGE, "qfx_qaoa_check: pass tile or stage count out of range");
    if (mode != QFX_QAOA_BACKWARD && (ps.flags & (PF_LOAD_LAM | PF_STORE_LAM)))
      return qfx::set_error(QFX_EINVAL, "qfx_qaoa_check: lambda traffic in a forward program");
    for (int j = 0; j < ps.T; ++j)
      if (ps.pos[j] < 0 || ps.pos[j] > 30 || (j && ps.pos[j] <= ps.pos[j - 1]))
        return qfx::set_error(QFX_EINVAL, "qfx_qaoa_check: tile positions not ascending");
    for (int si = 0; si < ps.nstage; ++si) {
      const int ty = ps.stage[si][0], l = ps.stage[si][1];
      const unsigned mask = (unsigned)ps.stage[si][2];
      if (ty < ST_INIT || (ty > ST_COST_RX && ty != ST_RX_LOAD && ty != ST_RX_STORE) || l < 0 ||
          l >= kMaxPLayers)
        return qfx::set_error(QFX_EINVAL, "qfx_qaoa_check: bad stage");
      const bool io = ty == ST_RX_LOAD || ty == ST_RX_STORE;
      const bool rx = ty == ST_RX || ty == ST_RX_ADJ || ty == ST_COST_RX || io;
      if (io && (mode == QFX_QAOA_BACKWARD || mask == 0))
        return qfx::set_error(QFX_EINVAL, "qfx_qaoa_check: bad load/store RX stage");
      if (ty == ST_RX_LOAD && (si != 0 || !(ps.flags & PF_LOAD_PSI)))
        return qfx::set_error(QFX_EINVAL, "qfx_qaoa_check: load RX stage not first or no load");
      if (ty == ST_RX_STORE && (si != ps.nstage - 1 || !(ps.flags & PF_STORE_PSI)))
        return qfx::set_error(QFX_EINVAL, "qfx_qaoa_check: store RX stage not last or no store");
      if (rx && (mask >> ps.T))
        return qfx::set_error(QFX_EINVAL, "qfx_qaoa_check: RX mask outside the tile");
      if (ty == ST_COST_RX && mask == 0)
        return qfx::set_error(QFX_EINVAL, "qfx_qaoa_check: fused cost stage without RX bits");
      if (ty == ST_COST_RX && mode == QFX_QAOA_BACKWARD)
        return qfx::set_error(QFX_EINVAL, "qfx_qaoa_check: fused cost stage in a backward program");
      if (mode != QFX_QAOA_BACKWARD &&
          (ty == ST_MAKE_LAMBDA || ty == ST_RX_ADJ || ty == ST_COST_ADJ))
        return qfx::set_error(QFX_EINVAL, "qfx_qaoa_check: backward stage in a forward program");
    }
  }
  if (nk < 0 || kstart[0] != 0)
    return qfx::set_error(QFX_EINVAL, "qfx_qaoa_check: bad pass index table");
  for (int k = 0; k < nk; ++k)
    if (kstart[k + 1] < kstart[k]) return qfx::set_error(QFX_EINVAL, "qfx_qaoa_check: kstart");
  for (int it = 0; it < kstart[nk]; ++it) {
    const qfx_qaoa_item& item = items[it];
    if (item.inst < 0 || item.inst >= ninst || item.pass < 0 || item.pass >= npasses ||
        item.partial < 0 || item.partial >= npartial)
      return qfx::set_error(QFX_EINVAL, "qfx_qaoa_check: item out of range");
    const qfx_qaoa_inst& in = insts[item.inst];
    const qfx_qaoa_pass& ps = passes[item.pass];
    if (ps.T > in.n || item.tile < 0 || ((int64_t)item.tile >> (in.n - ps.T)) != 0)
      return qfx::set_error(QFX_EINVAL, "qfx_qaoa_check: tile out of range");
    // mirror: bit n-1 is the pass's highest tile bit, the tile's highest
    // non-tile bit is clear (so its complement tile is not an item)
    if (in.mirror && (ps.T < 1 || ps.pos[ps.T - 1] != in.n - 1 || in.n - ps.T < 1 ||
                      ((int64_t)item.tile >> (in.n - ps.T - 1)) != 0))
      return qfx::set_error(QFX_EINVAL, "qfx_qaoa_check: mirror pass or tile out of range");
    for (int j = 0; j < ps.T; ++j)
      if (ps.pos[j] >= in.n) return qfx::set_error(QFX_EINVAL, "qfx_qaoa_check: tile bit >= n");
    for (int si = 0; si < ps.nstage; ++si)
      if (ps.stage[si][1] >= in.p) return qfx::set_error(QFX_EINVAL, "qfx_qaoa_check: layer >= p");
  }
  return QFX_OK;
}

int qfx_qaoa_run(void* stream, const qfx_qaoa_args* args) {
  if (!args) return qfx::set_error(QFX_EINVAL, "qfx_qaoa_run: null args");
  const qfx_qaoa_args& a = *args;
  if (!a.insts || !a.passes || !a.items || !a.kstart || !a.angles || !a.psi_pool ||
      !a.partials || !a.out || !a.sync || (!a.cnt_pool && !a.val_pool))
    return qfx::set_error(QFX_EINVAL, "qfx_qaoa_run: null pointer");
  if (a.mode == QFX_QAOA_BACKWARD && !a.lam_pool)
    return qfx::set_error(QFX_EINVAL, "qfx_qaoa_run: backward needs lam_pool");
  if (a.width < 1 || a.width > kAccum || a.ninst < 1 || a.nk < 1)
    return qfx::set_error(QFX_ERANGE, "qfx_qaoa_run: sizes out of range");
  if (a.tile_bits < 0 || a.tile_bits > (a.mode == QFX_QAOA_BACKWARD ? kMaxT - 1 : kMaxT))
    return qfx::set_error(QFX_ERANGE, "qfx_qaoa_run: tile_bits out of range");
  if (a.block != 256 && a.block != 512 && a.block != 1024)
    return qfx::set_error(QFX_EINVAL, "qfx_qaoa_run: block must be 256, 512 or 1024");
  hipStream_t s = qfx::as_stream(stream);
  // programs without cut values hold no weighted instance
  const bool flow = a.tables && a.table_off && a.item_need, weighted = a.val_pool;
  // in-place phases (weighted instances; every launch with barriers) leave no
  // registers for 12-bit tiles at two workgroups a CU
  const bool wide = a.tile_bits == 0 || (a.tile_bits == 12 && (!flow || weighted));
  if (a.mode == QFX_QAOA_BACKWARD && wide)
    return !flow      ? launch_qaoa<true, false, true, true>(s, a)
           : weighted ? launch_qaoa<true, true, true, true>(s, a)
                      : launch_qaoa<true, true, false, true>(s, a);
  if (a.mode == QFX_QAOA_BACKWARD)
    return !flow      ? launch_qaoa<true, false, true, false>(s, a)
           : weighted ? launch_qaoa<true, true, true, false>(s, a)
                      : launch_qaoa<true, true, false, false>(s, a);
  return !flow      ? launch_qaoa<false, false, true, true>(s, a)
         : weighted ? launch_qaoa<false, true, true, true>(s, a)
                    : launch_qaoa<false, true, false, true>(s, a);
}

int qfx_qaoa_status(const void* sync, int* failed) {
  if (!sync || !failed) return qfx::set_error(QFX_EINVAL, "qfx_qaoa_status: null pointer");
  int e[2] = {0, 0};
  int rc = qfx::check_hip(hipMemcpy(e, static_cast<const unsigned*>(sync) + 1, sizeof(e),
                                    hipMemcpyDeviceToHost),
                          "hipMemcpy");
  if (rc) return rc;
  *failed = (e[0] | e[1]) != 0;
  return QFX_OK;
}

}  // extern "C"

// Tiles of a qubit relabelling out[i] = in[j], bit src[b] of j = bit b of i.
//
// A plain gather writes whole lines but reads 16-byte pieces wherever a low
// source bit sits at a high output bit.  A tile here spans kPermT output bits
// chosen so that both its reads and its writes run over contiguous memory:
// alternately the lowest output bits and the output bits fed by the lowest
// source bits, i.e. at least the five lowest of each (512-byte runs).  The
// tile is loaded in source order and turned to output order in LDS.
#pragma once

#include "qfx_common.h"

constexpr int kPermT = 10;                       // 1024 amplitudes, 16 KiB of LDS
constexpr int kPermBlock = 256;
constexpr int kPermLb = 8;                       // log2 kPermBlock
constexpr int kPermPer = 1 << (kPermT - kPermLb);

struct PermTile {
  int outpos[kPermT];                            // tile bits of i, ascending
  int inpos[kPermT];                             // tile bits of j, ascending
  int rank[kPermT];                              // tile bit of i that inpos[t] feeds
  int rest_out[QFX_MAX_QUBITS];                  // the other bits of i and their
  int rest_in[QFX_MAX_QUBITS];                   // source bits
  int nrest;
};

// src_bit must be a permutation of 0..n-1, n >= kPermT.
inline PermTile make_perm_tile(int n, const int* src_bit) {
  PermTile p;
  int out_of[QFX_MAX_QUBITS];
  bool in_tile[QFX_MAX_QUBITS] = {};
  for (int b = 0; b < n; ++b) out_of[src_bit[b]] = b;
  int count = 0;
  for (int l = 0; count < kPermT; ++l) {
    for (int b : {l, out_of[l]})
      if (count < kPermT && !in_tile[b]) {
        in_tile[b] = true;
        ++count;
      }
  }
  int t = 0;
  p.nrest = 0;
  for (int b = 0; b < n; ++b) {
    if (in_tile[b]) {
      p.outpos[t++] = b;
    } else {
      p.rest_out[p.nrest] = b;
      p.rest_in[p.nrest++] = src_bit[b];
    }
  }
  t = 0;
  for (int s = 0; s < n; ++s)
    if (in_tile[out_of[s]]) {
      p.inpos[t] = s;
      for (int r = 0; r < kPermT; ++r)
        if (p.outpos[r] == out_of[s]) p.rank[t] = r;
      ++t;
    }
  return p;
}

__device__ __forceinline__ unsigned perm_swz(unsigned e) {
  return e ^ (((e >> 3) ^ (e >> 6) ^ (e >> 9)) & 7u);
}

// One lane's share of every tile: elements lane + 256 u in either order.
struct PermLane {
  uint64_t in_lane, out_lane, in_u[kPermPer], out_u[kPermPer];
  unsigned lds_in[kPermPer];                     // slot of the u-th element read
};

__device__ __forceinline__ PermLane perm_lane(const PermTile& p) {
  PermLane q;
  q.in_lane = q.out_lane = 0;
  unsigned slot = 0;
#pragma unroll
  for (int t = 0; t < kPermLb; ++t) {
    const uint64_t bit = (threadIdx.x >> t) & 1u;
    q.in_lane |= bit << p.inpos[t];
    q.out_lane |= bit << p.outpos[t];
    slot |= (unsigned)bit << p.rank[t];
  }
#pragma unroll
  for (int u = 0; u < kPermPer; ++u) {
    q.in_u[u] = q.out_u[u] = 0;
    unsigned su = slot;
#pragma unroll
    for (int t = kPermLb; t < kPermT; ++t) {
      const uint64_t bit = (u >> (t - kPermLb)) & 1;
      q.in_u[u] |= bit << p.inpos[t];
      q.out_u[u] |= bit << p.outpos[t];
      su |= (unsigned)bit << p.rank[t];
    }
    q.lds_in[u] = perm_swz(su);
  }
  return q;
}

__device__ __forceinline__ void perm_bases(const PermTile& p, uint64_t tile, uint64_t* in,
                                           uint64_t* out) {
  uint64_t bi = 0, bo = 0;
  for (int k = 0; k < p.nrest; ++k) {
    const uint64_t bit = (tile >> k) & 1;
    bi |= bit << p.rest_in[k];
    bo |= bit << p.rest_out[k];
  }
  *in = bi;
  *out = bo;
}

// Device-side step engine for gfx950, shared by the grid-wide step kernels and the
// batched persistent executor.
//
// A step (ts_step, include/tensorsat_prog.h) computes for every out index o
//     acc(o) = sum_c lhs[L(o, c)] * rhs[R(o, c)]
// where L/R scatter the bits of o and of the summed index c to operand bit positions.
// L(o, c) = Lo(o) + Lc(c) with both parts linear in the bits, evaluated with byte-chunk
// lookup tables held in LDS: Lo(o) = T0[o & 255] + T1[(o >> 8) & 255] + ...
// Out indices are walked in blocks of 256 consecutive values, one per thread, so the
// low chunk is a per-thread constant and the higher chunks are workgroup-uniform
// (LDS broadcast); stores are byte-coalesced.
//
// Paths:
//  * sum_rank == 0: product (or copy for unary steps);
//  * TS_STEP_KINNER: the summed bits are the lowest bits of both operands in the same
//    order, so each operand's 2^sum_rank terms are contiguous: 2/4/8/16-byte vector
//    loads and popcount(lhs & rhs) on 0/1 bytes;
//  * otherwise: loop over c with LDS tables for Lc/Rc.
// Epilogues: GT0 (acc > 0) and MOD256 ((acc mod 256) != 0) for 0/1 bytes; exact uint64
// with overflow detection for the counting semiring.

#pragma once

#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

#include "../../include/tensorsat_amd.h"

namespace tsd {

constexpr int WG = 256;

// NQ byte chunks per table: 4 cover every rank up to 27 bits (TS_MAX_BITS); 2 suffice
// when every tensor has at most 16 bits (LDS-resident arenas).
template <int NQ>
struct LutT {
  uint32_t ol[NQ][256];
  uint32_t orr[NQ][256];
  uint32_t cl[NQ][256];
  uint32_t cr[NQ][256];
};
using Lut = LutT<4>;

__device__ __forceinline__ int nchunks(int bits) { return (bits + 7) >> 3; }

// 8 bytes of a record from byte `off` on (a constant), from its aligned dwords.
__device__ __forceinline__ uint2 rec8(const uint32_t* w, size_t off) {
  const int q = (int)(off >> 2), r = (int)(off & 3);
  if (r == 0) return make_uint2(w[q], w[q + 1]);
  return make_uint2(__builtin_amdgcn_alignbyte(w[q + 1], w[q], r), __builtin_amdgcn_alignbyte(w[q + 2], w[q + 1], r));
}

// The low 8 bits of v at the positions in pos (one byte each); set bits of v beyond the ones
// that exist are the caller's to clear.  TS_NOPOS shifts its bit to position 31; positions
// are below TS_MAX_BITS, so bit 31 is cleared at the end.  Three 32-bit instructions per bit
// (64-bit shifts of the position list were most of a small step).
__device__ __forceinline__ uint32_t place8(uint32_t v, uint2 pos) {
  uint32_t off = 0;
#pragma unroll
  for (int i = 0; i < 8; ++i) off |= ((v >> i) & 1u) << (((i < 4 ? pos.x : pos.y) >> (8 * (i & 3))) & 31u);
  return off & 0x7fffffffu;
}

// Build the chunk tables of one step (all threads of the workgroup participate; the
// caller synchronises afterwards).
template <int NQ>
__device__ inline void build_lut(const ts_step& st, LutT<NQ>& L, bool need_c, int tid) {
  const int ro = st.out_rank;
  // Chunk 0 is always built: a scalar step (out_rank 0) reads entry [0][0], which must
  // be 0 and not a value left in LDS by an earlier step.
  int nqo = nchunks(ro) > 0 ? nchunks(ro) : 1;
  nqo = nqo < NQ ? nqo : NQ;  // callers keep ranks within the table (16 bits for NQ = 2)
  const uint32_t* w = reinterpret_cast<const uint32_t*>(&st);
  for (int e = tid; e < nqo * 256; e += WG) {
    const int q = e >> 8, left = ro - 8 * q;
    const uint32_t v = (uint32_t)e & (left < 8 ? (1u << left) - 1u : 255u);  // left >= 0
    L.ol[q][e & 255] = place8(v, rec8(w + 2 * q, offsetof(ts_step, o_lpos)));
    L.orr[q][e & 255] = place8(v, rec8(w + 2 * q, offsetof(ts_step, o_rpos)));
  }
  if (need_c) {
    const int nc = st.sum_rank;
    int nqc = nchunks(nc) > 0 ? nchunks(nc) : 1;
    nqc = nqc < NQ ? nqc : NQ;
    for (int e = tid; e < nqc * 256; e += WG) {
      const int q = e >> 8, v = e & 255;
      uint32_t al = 0, ar = 0;
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const int j = q * 8 + i;
        if (j < nc && ((v >> i) & 1)) {
          const uint8_t pl = st.c_lpos[j], pr = st.c_rpos[j];
          if (pl != TS_NOPOS) al |= 1u << pl;
          if (pr != TS_NOPOS) ar |= 1u << pr;
        }
      }
      L.cl[q][v] = al;
      L.cr[q][v] = ar;
    }
  }
}

// High-chunk part of an out offset (o >> 8), workgroup-uniform in the block loops.
template <int NQ>
__device__ __forceinline__ uint32_t hi_off(const uint32_t (*T)[256], uint32_t hi, int nq) {
  uint32_t r = 0;
  if (nq > 1) r += T[1][hi & 255];
  if (NQ > 2 && nq > 2) r += T[NQ > 2 ? 2 : 0][(hi >> 8) & 255];
  if (NQ > 3 && nq > 3) r += T[NQ > 3 ? 3 : 0][hi >> 16];
  return r;
}

template <int NQ>
__device__ __forceinline__ uint32_t c_off(const uint32_t (*T)[256], uint32_t c, int nq) {
  uint32_t r = T[0][c & 255];
  if (nq > 1) r += T[1][(c >> 8) & 255];
  if (NQ > 2 && nq > 2) r += T[NQ > 2 ? 2 : 0][(c >> 16) & 255];
  if (NQ > 3 && nq > 3) r += T[NQ > 3 ? 3 : 0][c >> 24];
  return r;
}

__device__ __forceinline__ uint32_t popc_and(const uint8_t* a, const uint8_t* b, int nc,
                                             bool norhs) {
  // 2^nc contiguous 0/1 bytes in each operand, aligned to min(16, 2^nc).
  switch (nc) {
    case 1: {
      uint32_t x = *reinterpret_cast<const uint16_t*>(a);
      if (!norhs) x &= *reinterpret_cast<const uint16_t*>(b);
      return __popc(x);
    }
    case 2: {
      uint32_t x = *reinterpret_cast<const uint32_t*>(a);
      if (!norhs) x &= *reinterpret_cast<const uint32_t*>(b);
      return __popc(x);
    }
    case 3: {
      uint64_t x = *reinterpret_cast<const uint64_t*>(a);
      if (!norhs) x &= *reinterpret_cast<const uint64_t*>(b);
      return __popcll(x);
    }
    default: {
      uint32_t acc = 0;
      const int n16 = 1 << (nc - 4);
      for (int i = 0; i < n16; ++i) {
        uint4 x = reinterpret_cast<const uint4*>(a)[i];
        if (!norhs) {
          const uint4 y = reinterpret_cast<const uint4*>(b)[i];
          x.x &= y.x;
          x.y &= y.y;
          x.z &= y.z;
          x.w &= y.w;
        }
        acc += __popc(x.x) + __popc(x.y) + __popc(x.z) + __popc(x.w);
      }
      return acc;
    }
  }
}

// The 2^nc contiguous bytes of one row, nc = 2 or 3, as an integer (aligned to 2^nc).
__device__ __forceinline__ uint64_t load_row(const uint8_t* p, int nc) {
  return nc == 2 ? *reinterpret_cast<const uint32_t*>(p) : *reinterpret_cast<const uint64_t*>(p);
}

// ---- vector path for short rows ------------------------------------------------------
//
// Rows of 1..8 bytes (at most 3 summed bits, innermost).  Where each operand holds the T
// lowest out bits right above its summed bits in order (or not at all), the rows of 2^T
// consecutive outputs are one run of at most 32 bytes; T = 2 for every layout of the compiler,
// T = 1 only for operands that come in other orders.  A lane computes 16 consecutive outputs
// as groups of 2^T: the other low out bits just move the run's address, so all its loads go
// out at once, and the rows are combined a dword at a time (v_perm picks the bytes of one term
// of four outputs; rows of 4 and 8 bytes are whole dwords).  Counts are at most 64, so both
// epilogues reduce to "any bit of the AND set".
// Bound by HBM and, on many workgroups, by their tables: 16 jobs of 2^23 outputs on 65536
// workgroups took 336 us with each output's row picked out of a chunk held in 64-bit words
// (40 vector instructions per output), 288 us with dwords (6), and 75 us once 8192 workgroups
// shared the work.  T = 1, 2^18 outputs of 4-byte rows: 5.3 us picked out of chunks, 6.8 us one
// output per lane, 3.9 us so.

// T of a step (2 or 1), 0 if it has no such runs.
__host__ __device__ inline int run_bits(const ts_step& st) {
  const int nc = st.sum_rank;
  if (nc > 3 || !(nc == 0 || (st.flags & TS_STEP_KINNER)) || st.out_rank < 4) return 0;
  const bool norhs = st.flags & TS_STEP_NORHS;
  int hl = 0, hr = 0;
  for (int j = 0; j < 2; ++j) {
    if (st.o_lpos[j] != TS_NOPOS && st.o_lpos[j] != nc + hl++) return j;
    if (!norhs && st.o_rpos[j] != TS_NOPOS && st.o_rpos[j] != nc + hr++) return j;
  }
  return 2;
}

// 2^LG bytes (LG <= 5) as dwords.
template <int LG>
struct Run {
  uint32_t w[LG < 4 ? 2 : 1 << (LG - 2)];
};
template <int LG>
__device__ __forceinline__ Run<LG> load_run(const uint8_t* p) {
  Run<LG> r;
  if constexpr (LG <= 2) {
    r.w[1] = 0;
    if constexpr (LG == 0) r.w[0] = *p;
    else if constexpr (LG == 1) r.w[0] = *reinterpret_cast<const uint16_t*>(p);
    else r.w[0] = *reinterpret_cast<const uint32_t*>(p);
  } else if constexpr (LG == 3) {
    const uint2 v = *reinterpret_cast<const uint2*>(p);
    r.w[0] = v.x;
    r.w[1] = v.y;
  } else {
#pragma unroll
    for (int h = 0; h < (1 << (LG - 4)); ++h) {
      const uint4 v = reinterpret_cast<const uint4*>(p)[h];
      r.w[4 * h] = v.x;
      r.w[4 * h + 1] = v.y;
      r.w[4 * h + 2] = v.z;
      r.w[4 * h + 3] = v.w;
    }
  }
  return r;
}

// Index of output i's row in an operand that holds H of the T lowest out bits (H = 1 of 2: bit
// `one` of them).
template <int T, int H>
__device__ __forceinline__ uint32_t run_row(int i, int one) {
  return H == 0 ? 0u : H == T ? (uint32_t)i : (uint32_t)(i >> one) & 1u;
}

// Byte c of the rows of outputs 4d .. 4d + 3 (K <= 1): of one run (T = 2), or of two runs of at
// most a dword each, side by side (T = 1).
template <int T, class R>
__device__ __forceinline__ uint32_t run_bytes(const R* r, int d, uint32_t sel, int c) {
  const uint32_t lo = T == 2 ? r[d].w[0] : r[2 * d].w[0], hi = T == 2 ? r[d].w[1] : r[2 * d + 1].w[0];
  return __builtin_amdgcn_perm(hi, lo, sel + 0x01010101u * (uint32_t)c);
}

// Dword d of output i's row within its run (K >= 2).
template <int T, int K, int H>
__device__ __forceinline__ uint32_t run_word(const Run<K + H>& r, int i, int d, int one) {
  constexpr int D = 1 << (K - 2);
  if constexpr (H == 1 && T == 2) return one ? r.w[(i >> 1) * D + d] : r.w[(i & 1) * D + d];
  else return r.w[(H == 0 ? 0 : i) * D + d];
}

template <int T, int K, int HL, int HR, int NQ>
__device__ void step_runs_kh(const ts_step& st, const LutT<NQ>& L, const uint8_t* __restrict__ lhs,
                             const uint8_t* __restrict__ rhs, uint8_t* __restrict__ out, uint64_t first,
                             uint64_t stride) {
  constexpr int G = 16 >> T, B = 4 - T;  // runs per operand, out bits that tell them apart
  const bool norhs = st.flags & TS_STEP_NORHS;
  const int nqo = nchunks(st.out_rank);
  const uint64_t n = 1ull << (st.out_rank - 4);
  if (first >= n) return;
  const int one_l = st.o_lpos[0] == TS_NOPOS, one_r = norhs || st.o_rpos[0] == TS_NOPOS;
  uint32_t dl[B], dr[B];  // what out bits T .. 3 add to the offsets
#pragma unroll
  for (int j = 0; j < B; ++j) {
    dl[j] = st.o_lpos[T + j] != TS_NOPOS ? 1u << st.o_lpos[T + j] : 0u;
    dr[j] = !norhs && st.o_rpos[T + j] != TS_NOPOS ? 1u << st.o_rpos[T + j] : 0u;
  }
  uint32_t sl = 0, sr = 0;  // byte selectors of term 0 (K <= 1)
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const uint32_t run = T == 2 ? 0u : 4u * (uint32_t)(i >> 1);
    const int k = i & ((1 << T) - 1);
    sl |= (run + (run_row<T, HL>(k, one_l) << K)) << (8 * i);
    sr |= (run + (run_row<T, HR>(k, one_r) << K)) << (8 * i);
  }
  const uint32_t lo = (uint32_t)((first << 4) & 255);  // the same for every trip of this lane
  const uint32_t lo_l = L.ol[0][lo], lo_r = L.orr[0][lo];
  for (uint64_t q = first; q < n; q += stride) {
    const uint64_t o = q << 4;
    const uint32_t hi = (uint32_t)(o >> 8);
    const uint8_t* pl = lhs + lo_l + hi_off<NQ>(L.ol, hi, nqo);
    const uint8_t* pr = rhs + lo_r + hi_off<NQ>(L.orr, hi, nqo);
    Run<K + HL> a[G];
    Run<K + HR> b[G];
#pragma unroll
    for (int g = 0; g < G; ++g) {
      uint32_t off = 0;
#pragma unroll
      for (int j = 0; j < B; ++j) off += (g >> j) & 1 ? dl[j] : 0u;
      a[g] = load_run<K + HL>(pl + off);
    }
    if (!norhs) {
#pragma unroll
      for (int g = 0; g < G; ++g) {
        uint32_t off = 0;
#pragma unroll
        for (int j = 0; j < B; ++j) off += (g >> j) & 1 ? dr[j] : 0u;
        b[g] = load_run<K + HR>(pr + off);
      }
    } else {
#pragma unroll
      for (int g = 0; g < G; ++g)
#pragma unroll
        for (uint32_t& w : b[g].w) w = ~0u;
    }
    uint32_t res[4];
#pragma unroll
    for (int d = 0; d < 4; ++d) {
      if constexpr (K <= 1) {
        uint32_t x = run_bytes<T>(a, d, sl, 0) & run_bytes<T>(b, d, sr, 0);
        if constexpr (K == 1) x |= run_bytes<T>(a, d, sl, 1) & run_bytes<T>(b, d, sr, 1);
        res[d] = ((((x & 0x7F7F7F7Fu) + 0x7F7F7F7Fu) | x) >> 7) & 0x01010101u;
      } else {
        res[d] = 0;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int g = (4 * d + i) >> T, k = i & ((1 << T) - 1);
          uint32_t x = run_word<T, K, HL>(a[g], k, 0, one_l) & run_word<T, K, HR>(b[g], k, 0, one_r);
          if constexpr (K == 3) x |= run_word<T, K, HL>(a[g], k, 1, one_l) & run_word<T, K, HR>(b[g], k, 1, one_r);
          res[d] |= (x < 1u ? x : 1u) << (8 * i);
        }
      }
    }
    *reinterpret_cast<uint4*>(out + o) = make_uint4(res[0], res[1], res[2], res[3]);
  }
}

template <int T, int K, int HL, int NQ>
__device__ __forceinline__ void step_runs_k(const ts_step& st, int hr, const LutT<NQ>& L, const uint8_t* lhs,
                                            const uint8_t* rhs, uint8_t* out, uint64_t first, uint64_t stride) {
  if (hr == 0) step_runs_kh<T, K, HL, 0, NQ>(st, L, lhs, rhs, out, first, stride);
  else if (hr == 1) step_runs_kh<T, K, HL, 1, NQ>(st, L, lhs, rhs, out, first, stride);
  else if constexpr (T == 2) step_runs_kh<T, K, HL, 2, NQ>(st, L, lhs, rhs, out, first, stride);
}

template <int T, int K, int NQ>
__device__ __forceinline__ void step_runs_l(const ts_step& st, int hl, int hr, const LutT<NQ>& L, const uint8_t* lhs,
                                            const uint8_t* rhs, uint8_t* out, uint64_t first, uint64_t stride) {
  if (hl == 0) step_runs_k<T, K, 0, NQ>(st, hr, L, lhs, rhs, out, first, stride);
  else if (hl == 1) step_runs_k<T, K, 1, NQ>(st, hr, L, lhs, rhs, out, first, stride);
  else if constexpr (T == 2) step_runs_k<T, K, 2, NQ>(st, hr, L, lhs, rhs, out, first, stride);
}

template <int T, int NQ>
__device__ __forceinline__ void step_runs_t(const ts_step& st, const LutT<NQ>& L, const uint8_t* lhs,
                                            const uint8_t* rhs, uint8_t* out, uint64_t first, uint64_t stride) {
  const bool norhs = st.flags & TS_STEP_NORHS;
  int hl = 0, hr = 0;  // low out bits that each operand holds
  for (int j = 0; j < T; ++j) {
    hl += st.o_lpos[j] != TS_NOPOS;
    hr += !norhs && st.o_rpos[j] != TS_NOPOS;
  }
  if (st.sum_rank == 0) step_runs_l<T, 0, NQ>(st, hl, hr, L, lhs, rhs, out, first, stride);
  else if (st.sum_rank == 1) step_runs_l<T, 1, NQ>(st, hl, hr, L, lhs, rhs, out, first, stride);
  else if (st.sum_rank == 2) step_runs_l<T, 2, NQ>(st, hl, hr, L, lhs, rhs, out, first, stride);
  else step_runs_l<T, 3, NQ>(st, hl, hr, L, lhs, rhs, out, first, stride);
}

// Grid-stride over groups of 16 outputs of a step with t = run_bits(st) > 0 (first / stride as
// for step_u8).
template <int NQ>
__device__ inline void step_runs(int t, const ts_step& st, const LutT<NQ>& L, const uint8_t* __restrict__ lhs,
                                 const uint8_t* __restrict__ rhs, uint8_t* __restrict__ out, uint64_t first,
                                 uint64_t stride) {
  if (t == 2) step_runs_t<2, NQ>(st, L, lhs, rhs, out, first, stride);
  else step_runs_t<1, NQ>(st, L, lhs, rhs, out, first, stride);
}

// Boolean step over out indices o = first + k * stride (first = block * 256 + tid and
// stride = blocks * 256: the callers' grid-stride launch shape).
template <int NQ>
__device__ inline void step_u8(const ts_step& st, const LutT<NQ>& L, const uint8_t* __restrict__ lhs,
                               const uint8_t* __restrict__ rhs, uint8_t* __restrict__ out,
                               uint64_t first, uint64_t stride, int mode) {
  const int ro = st.out_rank, nc = st.sum_rank;
  const bool norhs = st.flags & TS_STEP_NORHS;
  const bool kinner = st.flags & TS_STEP_KINNER;
  const uint64_t n = 1ull << ro;
  const int nqo = nchunks(ro), nqc = nchunks(nc);
  if (first >= n) return;
  const uint32_t lo_l = L.ol[0][first & 255];
  const uint32_t lo_r = L.orr[0][first & 255];
  if (kinner && (nc == 2 || nc == 3)) {
    // Rows of 4 or 8 bytes: the workgroup takes U adjacent blocks of 256 outputs per
    // trip (thread t: output t of each), every load of the trip issued before any is
    // used -- U row pairs in flight per thread, all in one neighbourhood of memory
    // (measured faster than one output per trip for these rows, slower for 1-2 bytes).
    constexpr int U = 8;
    const uint64_t lane = first % WG, blk = first / WG, nblk = stride / WG;
    const uint64_t nb = (n + WG - 1) / WG;
    for (uint64_t b0 = blk * U; b0 < nb; b0 += nblk * U) {
      uint64_t a[U], b[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const uint64_t o = (b0 + u) * WG + lane;
        a[u] = 0;
        b[u] = ~0ull;
        if (o < n) {
          const uint32_t hi = (uint32_t)(o >> 8);
          a[u] = load_row(lhs + lo_l + hi_off<NQ>(L.ol, hi, nqo), nc);
          if (!norhs) b[u] = load_row(rhs + lo_r + hi_off<NQ>(L.orr, hi, nqo), nc);
        }
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const uint64_t o = (b0 + u) * WG + lane;
        if (o < n) out[o] = (uint8_t)((a[u] & b[u]) != 0);  // at most 8 terms: both epilogues agree
      }
    }
    return;
  }
  for (uint64_t o = first; o < n; o += stride) {
    const uint32_t hi = (uint32_t)(o >> 8);
    const uint32_t offl = lo_l + hi_off<NQ>(L.ol, hi, nqo);
    const uint32_t offr = lo_r + hi_off<NQ>(L.orr, hi, nqo);
    uint32_t acc;
    if (nc == 0) {
      acc = lhs[offl];
      if (!norhs) acc &= rhs[offr];
    } else if (kinner) {
      acc = popc_and(lhs + offl, rhs + offr, nc, norhs);
    } else {
      acc = 0;
      const uint32_t nterm = 1u << nc;
      for (uint32_t c = 0; c < nterm; ++c) {
        const uint8_t a = lhs[offl + c_off<NQ>(L.cl, c, nqc)];
        const uint8_t b = norhs ? (uint8_t)1 : rhs[offr + c_off<NQ>(L.cr, c, nqc)];
        acc += a & b;
      }
    }
    out[o] = (uint8_t)(mode == TS_MODE_MOD256 ? ((acc & 255u) != 0) : (acc != 0));
  }
}

// Counting step (uint64 exact); returns true if any value of this thread overflowed.
__device__ inline bool step_u64(const ts_step& st, const Lut& L, const uint64_t* __restrict__ lhs,
                                const uint64_t* __restrict__ rhs, uint64_t* __restrict__ out,
                                uint64_t first, uint64_t stride) {
  const int ro = st.out_rank, nc = st.sum_rank;
  const bool norhs = st.flags & TS_STEP_NORHS;
  const bool kinner = st.flags & TS_STEP_KINNER;
  const uint64_t n = 1ull << ro;
  const int nqo = nchunks(ro), nqc = nchunks(nc);
  bool ovf = false;
  if (first >= n) return false;
  const uint32_t lo_l = L.ol[0][first & 255];
  const uint32_t lo_r = L.orr[0][first & 255];
  for (uint64_t o = first; o < n; o += stride) {
    const uint32_t hi = (uint32_t)(o >> 8);
    const uint32_t offl = lo_l + hi_off<4>(L.ol, hi, nqo);
    const uint32_t offr = lo_r + hi_off<4>(L.orr, hi, nqo);
    uint64_t acc = 0;
    const uint32_t nterm = 1u << nc;
    for (uint32_t c = 0; c < nterm; ++c) {
      const uint32_t cl = kinner ? c : c_off<4>(L.cl, c, nqc);
      const uint32_t cr = kinner ? c : c_off<4>(L.cr, c, nqc);
      const uint64_t a = lhs[offl + cl];
      const uint64_t b = norhs ? 1ull : rhs[offr + cr];
      uint64_t p;
      ovf |= __builtin_mul_overflow(a, b, &p);
      ovf |= __builtin_add_overflow(acc, p, &acc);
    }
    out[o] = acc;
  }
  return ovf;
}

}  // namespace tsd

// Kernels of the learned planner's message-passing network (gfx950): bf16 operands,
// fp32 accumulation.
//
//  * k_gemm: C = A x B (+ bias) (ReLU) with arbitrary strides, so one kernel covers the
//    forward product X W and the backward products dX = dZ W^T and dW = X^T dZ.
//    64x64 block tiles, 4 waves each computing 32x32 with 2x2 v_mfma_f32_16x16x32_bf16,
//    K in steps of 32 staged through LDS with 16-byte loads along whichever index is
//    contiguous.  Output fp32 or bf16, optionally accumulated.
//  * k_panel: the same product with all of B in LDS, for k-contiguous A and 128 columns at a
//    time: the state updates X W and the input gradients dZ W^T.
//  * k_wgrad, k_wgrad_sum: dW += X^T dZ over blocks of rows, partial sums through scratch.
//  * k_segsum16, k_segsum_row, k_segsum: out[r, off + f] = sum over incidences e of row r of |w[e]| X[col[e], f],
//    positive and negative literals (the sign of w[e]) into separate column blocks: the
//    normalised signed neighbour sums of the clause-variable incidence graph.  The edge
//    weights are symmetric (1/sqrt(deg(c) deg(v))), so the transpose incidence with the
//    same weights runs the backward pass.
//  * elementwise: bias-gradient column sums, ReLU masks, the squared-error loss and its
//    gradient, Adam updates on fp32 master weights with a bf16 copy.
//
// There is no counterpart in the reference (the north star adds the learned planner).

#include <hip/hip_runtime.h>
#include <hip/hip_bf16.h>
#include <stdint.h>

#include <algorithm>
#include <cmath>

#include "../../include/tensorsat_amd.h"

namespace {

typedef __bf16 bf8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf4 __attribute__((ext_vector_type(4)));
typedef float f4 __attribute__((ext_vector_type(4)));

constexpr int TM = 64, TN = 64, TK = 32;

__device__ __forceinline__ float bf2f(__bf16 x) { return (float)x; }
__device__ __forceinline__ __bf16 f2bf(float x) { return (__bf16)x; }

// Staging of one 64 x 32 operand tile into LDS, dst[row][k] = src[row * s_row + k * s_k]
// (zero outside rows < nrows, k < ke): 16-byte loads of 8 elements along the contiguous
// index when it is k (vec 1: one 16-byte LDS store) or the row (vec 2: eight 2-byte LDS
// stores, transposing), element loads otherwise and for ragged edges.
__device__ __forceinline__ int vec_mode(const __bf16* p, int64_t s_row, int64_t s_k) {
  if (reinterpret_cast<uintptr_t>(p) & 15) return 0;
  if (s_k == 1 && (s_row & 7) == 0) return 1;
  if (s_row == 1 && (s_k & 7) == 0) return 2;
  return 0;
}

__device__ __forceinline__ void stage_tile(__bf16 (*dst)[TK + 8], const __bf16* __restrict__ src, int64_t s_row,
                                           int64_t s_k, int row0, int nrows, int k0, int ke, int vec, int tid) {
  if (vec == 1) {  // 64 rows x 4 vectors of 8 k
    const int r = tid >> 2, c = (tid & 3) * 8;
    const int m = row0 + r, k = k0 + c;
    if (m < nrows && k + 8 <= ke) {
      *reinterpret_cast<uint4*>(&dst[r][c]) = *reinterpret_cast<const uint4*>(src + (int64_t)m * s_row + k);
    } else {
#pragma unroll
      for (int t = 0; t < 8; ++t)
        dst[r][c + t] = (m < nrows && k + t < ke) ? src[(int64_t)m * s_row + k + t] : f2bf(0.f);
    }
    return;
  }
  if (vec == 2) {  // 32 k x 8 vectors of 8 rows
    const int c = tid >> 3, r = (tid & 7) * 8;
    const int m = row0 + r, k = k0 + c;
    if (k < ke && m + 8 <= nrows) {
      const uint4 v = *reinterpret_cast<const uint4*>(src + m + (int64_t)k * s_k);
      const __bf16* e = reinterpret_cast<const __bf16*>(&v);
#pragma unroll
      for (int t = 0; t < 8; ++t) dst[r + t][c] = e[t];
    } else {
#pragma unroll
      for (int t = 0; t < 8; ++t)
        dst[r + t][c] = (k < ke && m + t < nrows) ? src[m + t + (int64_t)k * s_k] : f2bf(0.f);
    }
    return;
  }
  const bool kfast = s_k == 1;  // coalesce along the contiguous index
  for (int e = tid; e < 64 * TK; e += 256) {
    const int r = kfast ? e / TK : e % 64, c = kfast ? e % TK : e / 64;
    const int m = row0 + r, k = k0 + c;
    dst[r][c] = (m < nrows && k < ke) ? src[(int64_t)m * s_row + (int64_t)k * s_k] : f2bf(0.f);
  }
}

// The vector modes split into a global load (the thread's 8 elements, zero outside the
// bounds) and an LDS store, so that the next K tile's loads are in flight while the
// current tile's MFMAs run.
__device__ __forceinline__ uint4 load_vec(const __bf16* __restrict__ src, int64_t s_row, int64_t s_k, int row0,
                                          int nrows, int k0, int ke, int vec, int tid) {
  bf8 x;
  if (vec == 1) {
    const int r = tid >> 2, c = (tid & 3) * 8;
    const int m = row0 + r, k = k0 + c;
    if (m < nrows && k + 8 <= ke) return *reinterpret_cast<const uint4*>(src + (int64_t)m * s_row + k);
#pragma unroll
    for (int t = 0; t < 8; ++t) x[t] = (m < nrows && k + t < ke) ? src[(int64_t)m * s_row + k + t] : f2bf(0.f);
  } else {
    const int c = tid >> 3, r = (tid & 7) * 8;
    const int m = row0 + r, k = k0 + c;
    if (k < ke && m + 8 <= nrows) return *reinterpret_cast<const uint4*>(src + m + (int64_t)k * s_k);
#pragma unroll
    for (int t = 0; t < 8; ++t) x[t] = (k < ke && m + t < nrows) ? src[m + t + (int64_t)k * s_k] : f2bf(0.f);
  }
  return __builtin_bit_cast(uint4, x);
}

__device__ __forceinline__ void store_vec(__bf16 (*dst)[TK + 8], uint4 v, int vec, int tid) {
  if (vec == 1) {
    *reinterpret_cast<uint4*>(&dst[tid >> 2][(tid & 3) * 8]) = v;
    return;
  }
  const bf8 x = __builtin_bit_cast(bf8, v);
  const int c = tid >> 3, r = (tid & 7) * 8;
#pragma unroll
  for (int t = 0; t < 8; ++t) dst[r + t][c] = x[t];
}

// C[m, n] (+)= sum_k A(m, k) B(k, n); A(m,k) = A[m*sam + k*sak], B(k,n) = B[k*sbk + n*sbn],
// C at C[m*ldc + n].  Bounds are checked per element.
__global__ __launch_bounds__(256) void k_gemm(const __bf16* __restrict__ A, int64_t sam, int64_t sak,
                                              const __bf16* __restrict__ B, int64_t sbk, int64_t sbn,
                                              void* __restrict__ C, int64_t ldc, int M, int N, int K,
                                              const float* __restrict__ bias, int relu, int out_bf16,
                                              int accumulate, int kchunk) {
  __shared__ __bf16 sA[TM][TK + 8];
  __shared__ __bf16 sB[TN][TK + 8];  // stored transposed: sB[n][k]
  const int tid = threadIdx.x;
  const int wave = tid >> 6, lane = tid & 63;
  const int m0 = blockIdx.y * TM, n0 = blockIdx.x * TN;
  const int wm = (wave >> 1) * 32, wn = (wave & 1) * 32;
  // Split-K: block z covers k in [kb, ke); partial sums are added atomically (fp32 C).
  const int kb = blockIdx.z * kchunk;
  const int ke = min(K, kb + kchunk);
  const int vec_a = vec_mode(A, sam, sak), vec_b = vec_mode(B, sbn, sbk);
  f4 acc[2][2];
  for (int i = 0; i < 2; ++i)
    for (int j = 0; j < 2; ++j) acc[i][j] = (f4){0.f, 0.f, 0.f, 0.f};
  // Lane l of a 16x16x32 tile holds row/col (l % 16) and k = 8*(l/16) .. +7 of both.
  const int rr = lane & 15, kk = (lane >> 4) * 8;
  auto mfma_tile = [&]() {
    bf8 a[2], b[2];
    for (int i = 0; i < 2; ++i)
      for (int t = 0; t < 8; ++t) a[i][t] = sA[wm + 16 * i + rr][kk + t];
    for (int j = 0; j < 2; ++j)
      for (int t = 0; t < 8; ++t) b[j][t] = sB[wn + 16 * j + rr][kk + t];
    for (int i = 0; i < 2; ++i)
      for (int j = 0; j < 2; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i], b[j], acc[i][j], 0, 0, 0);
  };
  if (vec_a && vec_b) {
    uint4 ra = load_vec(A, sam, sak, m0, M, kb, ke, vec_a, tid);
    uint4 rb = load_vec(B, sbn, sbk, n0, N, kb, ke, vec_b, tid);
    for (int k0 = kb; k0 < ke; k0 += TK) {
      store_vec(sA, ra, vec_a, tid);
      store_vec(sB, rb, vec_b, tid);
      __syncthreads();
      if (k0 + TK < ke) {
        ra = load_vec(A, sam, sak, m0, M, k0 + TK, ke, vec_a, tid);
        rb = load_vec(B, sbn, sbk, n0, N, k0 + TK, ke, vec_b, tid);
      }
      mfma_tile();
      __syncthreads();
    }
  } else {
    for (int k0 = kb; k0 < ke; k0 += TK) {
      stage_tile(sA, A, sam, sak, m0, M, k0, ke, vec_a, tid);
      stage_tile(sB, B, sbn, sbk, n0, N, k0, ke, vec_b, tid);
      __syncthreads();
      mfma_tile();
      __syncthreads();
    }
  }
  // Accumulator layout: lane l holds rows 4*(l/16) + t (t = 0..3), column l % 16.
  for (int i = 0; i < 2; ++i)
    for (int j = 0; j < 2; ++j)
      for (int t = 0; t < 4; ++t) {
        const int m = m0 + wm + 16 * i + 4 * (lane >> 4) + t;
        const int n = n0 + wn + 16 * j + (lane & 15);
        if (m >= M || n >= N) continue;
        float v = acc[i][j][t];
        if (gridDim.z > 1) {  // split-K partial sum (fp32 output, no bias/ReLU)
          atomicAdd(reinterpret_cast<float*>(C) + (int64_t)m * ldc + n, v);
          continue;
        }
        if (bias) v += bias[n];
        if (relu) v = v > 0.f ? v : 0.f;
        if (out_bf16) {
          __bf16* c = reinterpret_cast<__bf16*>(C) + (int64_t)m * ldc + n;
          *c = f2bf(accumulate ? bf2f(*c) + v : v);
        } else {
          float* c = reinterpret_cast<float*>(C) + (int64_t)m * ldc + n;
          *c = accumulate ? *c + v : v;
        }
      }
}

// Four rows of four bf16 (r[i] = elements i0 .. i0 + 3 of row i) transposed: out[c] = column c.
__device__ __forceinline__ void transpose4(const uint2 (&r)[4], uint2 (&c)[4]) {
  // v_perm selectors: low or high halves of two dwords
  constexpr uint32_t LO = 0x05040100u, HI = 0x07060302u;
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const uint32_t a = h ? r[0].y : r[0].x, b = h ? r[1].y : r[1].x, d = h ? r[2].y : r[2].x, e = h ? r[3].y : r[3].x;
    c[2 * h] = make_uint2(__builtin_amdgcn_perm(b, a, LO), __builtin_amdgcn_perm(e, d, LO));
    c[2 * h + 1] = make_uint2(__builtin_amdgcn_perm(b, a, HI), __builtin_amdgcn_perm(e, d, HI));
  }
}

// C[m, n] (+)= sum_k A[m * lda + k] B(k, n) for 128 columns n, K = 32 KS: the network's state
// updates and input gradients, 10^4..10^5 rows against one weight matrix.  Bound by reading A
// and writing C once, so B (at most 384 x 128) is transposed into LDS once per workgroup,
// rows padded by 16 bytes (16 lanes read 16 rows without a bank conflict), and each wave
// streams 16-row tiles of A from memory into registers, a whole tile's loads in flight while
// the one before is multiplied.  The MFMA computes C^T, so a lane ends with 4 consecutive
// columns of one row: 8- or 16-byte stores.  74356 x 384 by 384 x 128: 47 us in 64 x 64
// tiles staged through LDS, 27 us here.
constexpr int PTHREADS = 512, PN = 128;

template <int KS>
__global__ __launch_bounds__(PTHREADS) void k_panel(const __bf16* __restrict__ A, int64_t lda,
                                                    const __bf16* __restrict__ B, int64_t sbk, int64_t sbn,
                                                    void* __restrict__ C, int64_t ldc, int M,
                                                    const float* __restrict__ bias, int relu, int out_bf16,
                                                    int accumulate) {
  constexpr int K = 32 * KS, PITCH = K + 8;
  __shared__ __attribute__((aligned(16))) __bf16 sB[PN * PITCH];
  const int tid = threadIdx.x, lane = tid & 63;
  const int n0 = blockIdx.y * PN;
  if (sbk == 1) {  // rows n are contiguous in k
    for (int u = tid; u < PN * (K / 8); u += PTHREADS) {
      const int n = u / (K / 8), k = (u % (K / 8)) * 8;
      *reinterpret_cast<uint4*>(&sB[n * PITCH + k]) = *reinterpret_cast<const uint4*>(B + (int64_t)(n0 + n) * sbn + k);
    }
  } else {  // rows k are contiguous in n: 4 x 4 blocks transposed in registers
    for (int u = tid; u < (K / 4) * (PN / 4); u += PTHREADS) {
      const int k = (u / (PN / 4)) * 4, n = (u % (PN / 4)) * 4;
      uint2 r[4], c[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) r[i] = *reinterpret_cast<const uint2*>(B + (int64_t)(k + i) * sbk + n0 + n);
      transpose4(r, c);
#pragma unroll
      for (int i = 0; i < 4; ++i) *reinterpret_cast<uint2*>(&sB[(n + i) * PITCH + k]) = c[i];
    }
  }
  __syncthreads();
  const int ntiles = (M + 15) / 16, nwaves = gridDim.x * (PTHREADS / 64);
  const int rr = lane & 15, kk = (lane >> 4) * 8;
  int t = blockIdx.x * (PTHREADS / 64) + (tid >> 6);
  if (t >= ntiles) return;
  bf8 a[KS], next[KS];
  auto load = [&](bf8 (&x)[KS], int tile) {
    const __bf16* p = A + (int64_t)min(tile * 16 + rr, M - 1) * lda + kk;
#pragma unroll
    for (int s = 0; s < KS; ++s) x[s] = *reinterpret_cast<const bf8*>(p + 32 * s);
  };
  load(a, t);
  for (; t < ntiles; t += nwaves) {
    if (t + nwaves < ntiles) load(next, t + nwaves);
    f4 acc[PN / 16];
#pragma unroll
    for (int j = 0; j < PN / 16; ++j) acc[j] = (f4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      asm volatile("" ::: "memory");  // the panel is the same for every tile: keep its reads here, not in registers
#pragma unroll
      for (int j = 0; j < PN / 16; ++j) {
        const bf8 b = *reinterpret_cast<const bf8*>(&sB[(16 * j + rr) * PITCH + 32 * s + kk]);
        acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b, a[s], acc[j], 0, 0, 0);
      }
    }
    const int m = t * 16 + rr;
    if (m < M) {
#pragma unroll
      for (int j = 0; j < PN / 16; ++j) {
        const int n = n0 + 16 * j + 4 * (lane >> 4);
        f4 v = acc[j];
        if (bias) v += *reinterpret_cast<const f4*>(bias + n);
        if (relu)
#pragma unroll
          for (int i = 0; i < 4; ++i) v[i] = v[i] > 0.f ? v[i] : 0.f;
        if (out_bf16) {
          bf4* c = reinterpret_cast<bf4*>(reinterpret_cast<__bf16*>(C) + (int64_t)m * ldc + n);
          if (accumulate) {
            const bf4 o = *c;
#pragma unroll
            for (int i = 0; i < 4; ++i) v[i] += bf2f(o[i]);
          }
          bf4 o;
#pragma unroll
          for (int i = 0; i < 4; ++i) o[i] = f2bf(v[i]);
          *c = o;
        } else {
          f4* c = reinterpret_cast<f4*>(reinterpret_cast<float*>(C) + (int64_t)m * ldc + n);
          *c = accumulate ? *c + v : v;
        }
      }
    }
#pragma unroll
    for (int s = 0; s < KS; ++s) a[s] = next[s];
  }
}

// Weight gradients dW[m, n] += sum_r X[r, m] dZ[r, n], n < 128: the contraction runs over the
// 10^4..10^5 rows.  A workgroup takes 128 columns of X and a block of rows, 64 rows at a
// time: both operands are row-contiguous, so 4 x 4 blocks are transposed in registers on the
// way into LDS (16-byte segments XOR-swizzled by the row, so the stores of a wave spread
// over the banks), the next rows' loads in flight during the MFMAs.  Each block of rows
// writes its partial tile to scratch and k_wgrad_sum adds them up: one pass over X, no
// atomics between XCDs.  74356 rows, 384 x 128: 124 us with split-K and atomics, 28 us and 4 for the sum.
constexpr int WK = 64, WM = 128;

__device__ __forceinline__ int wgrad_at(int row, int seg) { return row * WK + ((seg ^ (row >> 2)) & 7) * 8; }

__global__ __launch_bounds__(256) void k_wgrad(const __bf16* __restrict__ X, int64_t ldx,
                                               const __bf16* __restrict__ Z, int64_t ldz, int M, int rows, int per,
                                               float* __restrict__ part) {
  __shared__ __attribute__((aligned(16))) __bf16 sX[WM * WK], sZ[WM * WK];
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int m0 = blockIdx.x * WM;
  const int r0 = blockIdx.y * per, r1 = min(rows, r0 + per);
  // Unit u of a stage: columns 4 (u % 32) .. + 3, rows 4 (u / 32) .. + 3; two per thread.
  const int col = (tid & 31) * 4, rq = (tid >> 5) * 4;
  const bool xin = m0 + col < M;
  uint2 x[2][4], z[2][4];
  auto load = [&](int r) {
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int row = r + rq + 32 * h + i;
        x[h][i] = z[h][i] = make_uint2(0, 0);
        if (row < r1) {
          if (xin) x[h][i] = *reinterpret_cast<const uint2*>(X + (int64_t)row * ldx + m0 + col);
          z[h][i] = *reinterpret_cast<const uint2*>(Z + (int64_t)row * ldz + col);
        }
      }
  };
  auto store = [&](__bf16* dst, const uint2 (&v)[2][4]) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      uint2 c[4];
      transpose4(v[h], c);
      const int k = rq + 32 * h;
#pragma unroll
      for (int i = 0; i < 4; ++i) *reinterpret_cast<uint2*>(&dst[wgrad_at(col + i, k >> 3) + (k & 4)]) = c[i];
    }
  };
  f4 acc[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = (f4){0.f, 0.f, 0.f, 0.f};
  const int wm = (wave >> 1) * 64, wn = (wave & 1) * 64, rr = lane & 15, seg = lane >> 4;
  load(r0);
  for (int r = r0; r < r1; r += WK) {
    store(sX, x);
    store(sZ, z);
    __syncthreads();
    if (r + WK < r1) load(r + WK);
#pragma unroll
    for (int s = 0; s < WK / 32; ++s) {
      bf8 a[4], b[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) a[i] = *reinterpret_cast<const bf8*>(&sX[wgrad_at(wm + 16 * i + rr, 4 * s + seg)]);
#pragma unroll
      for (int j = 0; j < 4; ++j) b[j] = *reinterpret_cast<const bf8*>(&sZ[wgrad_at(wn + 16 * j + rr, 4 * s + seg)]);
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b[j], a[i], acc[i][j], 0, 0, 0);
    }
    __syncthreads();
  }
  // acc[i][j]: rows n = 4 (lane / 16) + t of tile j, column m = lane % 16 of tile i.
  float* out = part + ((int64_t)blockIdx.y * gridDim.x + blockIdx.x) * WM * WM;
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j)
      *reinterpret_cast<f4*>(out + (wm + 16 * i + rr) * WM + wn + 16 * j + 4 * seg) = acc[i][j];
}

// dW[m, n .. n + 3] += the sum of the partial tiles: 64 outputs of four and 4 shares of the
// blocks per workgroup.
__global__ __launch_bounds__(256) void k_wgrad_sum(const float* __restrict__ part, int M, int mtiles, int blocks,
                                                   float* __restrict__ dW, int64_t ldw) {
  __shared__ f4 red[256];
  const int tid = threadIdx.x, q = blockIdx.x * 64 + (tid & 63);
  const int m = q / (WM / 4), n = (q % (WM / 4)) * 4;
  const float* p = part + (int64_t)(m / WM) * WM * WM + (m % WM) * WM + n;
  f4 s = (f4){0.f, 0.f, 0.f, 0.f};
  if (m < M)
#pragma unroll 4
    for (int b = tid >> 6; b < blocks; b += 4) s += *reinterpret_cast<const f4*>(p + (int64_t)b * mtiles * WM * WM);
  red[tid] = s;
  __syncthreads();
  if (tid < 64 && m < M) {
    f4* d = reinterpret_cast<f4*>(dW + (int64_t)m * ldw + n);
    *d += (red[tid] + red[tid + 64]) + (red[tid + 128] + red[tid + 192]);
  }
}

// Signed neighbour sums for 128 features, 16-byte aligned rows.  Bound by the gathers: what
// counts is how many are in flight and how long a row's chain of them is.  A row's
// incidences are added in their order in every kernel.
//  * k_segsum16 (many rows with a few incidences each: clauses): a lane holds 8 consecutive
//    features, so 16 lanes read a whole neighbour row and a load moves four times what a
//    feature pair per lane does; four incidences in flight.  74356 rows: 37 us -> 16.
//  * k_segsum_row (few rows with many incidences: variables): a wave per row; 64 columns and
//    weights are read at once, one per lane, and SEG_FEW neighbour rows are in flight, so a
//    row of 100 incidences waits for memory a few times, not for two loads per four of them.
//    7185 rows of 46 on average: 70 us -> 33.
constexpr int SEG_FEW = 16;

template <bool XF32>
__device__ __forceinline__ void load8(float (&v)[8], const void* X, int64_t at) {
  if constexpr (XF32) {
    const f4* p = reinterpret_cast<const f4*>(reinterpret_cast<const float*>(X) + at);
    const f4 a = p[0], b = p[1];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      v[i] = a[i];
      v[4 + i] = b[i];
    }
  } else {
    const bf8 a = *reinterpret_cast<const bf8*>(reinterpret_cast<const __bf16*>(X) + at);
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = bf2f(a[i]);
  }
}

template <bool XF32, bool ACC>
__global__ __launch_bounds__(256) void k_segsum16(const int32_t* __restrict__ rowptr, const int32_t* __restrict__ col,
                                                  const float* __restrict__ weight, int nrows,
                                                  const void* __restrict__ X, int64_t ldx, int xoff_pos, int xoff_neg,
                                                  void* __restrict__ out, int64_t ldo, int off_pos, int off_neg) {
  constexpr int U = 4;
  const int r = (blockIdx.x * 256 + threadIdx.x) >> 4, f = (threadIdx.x & 15) * 8;
  if (r >= nrows) return;
  float p[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f}, q[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  const int end = rowptr[r + 1];
  for (int e = rowptr[r]; e < end; e += U) {
    float w[U], v[U][8];
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (e + u < end) {
        w[u] = weight[e + u];
        load8<XF32>(v[u], X, (int64_t)col[e + u] * ldx + (w[u] > 0.f ? xoff_pos : xoff_neg) + f);
      }
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (e + u < end) {
        const float aw = fabsf(w[u]);
        if (w[u] > 0.f) {
#pragma unroll
          for (int i = 0; i < 8; ++i) p[i] = __builtin_fmaf(aw, v[u][i], p[i]);
        } else {
#pragma unroll
          for (int i = 0; i < 8; ++i) q[i] = __builtin_fmaf(aw, v[u][i], q[i]);
        }
      }
  }
  if constexpr (ACC) {
    f4* o = reinterpret_cast<f4*>(reinterpret_cast<float*>(out) + (int64_t)r * ldo + off_pos + f);
    f4 a = o[0], b = o[1];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      a[i] = a[i] + p[i] + q[i];
      b[i] = b[i] + p[4 + i] + q[4 + i];
    }
    o[0] = a;
    o[1] = b;
  } else {
    __bf16* o = reinterpret_cast<__bf16*>(out) + (int64_t)r * ldo + f;
    bf8 a, b;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      a[i] = f2bf(p[i]);
      b[i] = f2bf(q[i]);
    }
    *reinterpret_cast<bf8*>(o + off_pos) = a;
    *reinterpret_cast<bf8*>(o + off_neg) = b;
  }
}

template <bool XF32, bool ACC>
__global__ __launch_bounds__(256) void k_segsum_row(const int32_t* __restrict__ rowptr, const int32_t* __restrict__ col,
                                                    const float* __restrict__ weight, int nrows,
                                                    const void* __restrict__ X, int64_t ldx, int xoff_pos, int xoff_neg,
                                                    void* __restrict__ out, int64_t ldo, int off_pos, int off_neg) {
  const int r = __builtin_amdgcn_readfirstlane((blockIdx.x * 256 + threadIdx.x) >> 6), lane = threadIdx.x & 63;
  if (r >= nrows) return;
  const int begin = rowptr[r], end = rowptr[r + 1];
  float p0 = 0.f, p1 = 0.f, q0 = 0.f, q1 = 0.f;  // features 2 lane, 2 lane + 1
  for (int e = begin; e < end; e += 64) {
    const int cnt = min(64, end - e);
    int c = 0, wbits = 0;
    if (lane < cnt) {
      c = col[e + lane];
      wbits = __builtin_bit_cast(int, weight[e + lane]);
    }
    for (int i = 0; i < cnt; i += SEG_FEW) {
      uint32_t v0[SEG_FEW], v1[SEG_FEW];
      float w[SEG_FEW];
#pragma unroll
      for (int u = 0; u < SEG_FEW; ++u) {
        const int l = min(i + u, cnt - 1);  // past the end: the last row again, not added
        w[u] = __builtin_bit_cast(float, __builtin_amdgcn_readlane(wbits, l));
        const int64_t at = (int64_t)__builtin_amdgcn_readlane(c, l) * ldx + (w[u] > 0.f ? xoff_pos : xoff_neg);
        if constexpr (XF32) {
          const uint2 x = reinterpret_cast<const uint2*>(reinterpret_cast<const float*>(X) + at)[lane];
          v0[u] = x.x;
          v1[u] = x.y;
        } else {
          v0[u] = reinterpret_cast<const uint32_t*>(reinterpret_cast<const __bf16*>(X) + at)[lane];
        }
      }
#pragma unroll
      for (int u = 0; u < SEG_FEW; ++u)
        if (i + u < cnt) {
          const float aw = fabsf(w[u]);
          const float x0 = __builtin_bit_cast(float, XF32 ? v0[u] : v0[u] << 16);
          const float x1 = __builtin_bit_cast(float, XF32 ? v1[u] : v0[u] & 0xFFFF0000u);
          if (w[u] > 0.f) {
            p0 = __builtin_fmaf(aw, x0, p0);
            p1 = __builtin_fmaf(aw, x1, p1);
          } else {
            q0 = __builtin_fmaf(aw, x0, q0);
            q1 = __builtin_fmaf(aw, x1, q1);
          }
        }
    }
  }
  if constexpr (ACC) {
    float2* o = reinterpret_cast<float2*>(reinterpret_cast<float*>(out) + (int64_t)r * ldo + off_pos) + lane;
    const float2 v = *o;
    *o = make_float2(v.x + p0 + q0, v.y + p1 + q1);
  } else {
    const auto pack = [](float a, float b) {
      return (uint32_t)__builtin_bit_cast(uint16_t, f2bf(a)) | ((uint32_t)__builtin_bit_cast(uint16_t, f2bf(b)) << 16);
    };
    __bf16* o = reinterpret_cast<__bf16*>(out) + (int64_t)r * ldo;
    reinterpret_cast<uint32_t*>(o + off_pos)[lane] = pack(p0, p1);
    reinterpret_cast<uint32_t*>(o + off_neg)[lane] = pack(q0, q1);
  }
}

// One wave per row: lanes cover the F features (F <= 128, two per lane).  Positive and
// negative incidences go to column blocks off_pos / off_neg of the row.
__global__ __launch_bounds__(256) void k_segsum(const int32_t* __restrict__ rowptr, const int32_t* __restrict__ col,
                                                const float* __restrict__ weight, int nrows,
                                                const void* __restrict__ X, int64_t ldx, int xoff_pos,
                                                int xoff_neg, int x_f32, void* __restrict__ out, int64_t ldo,
                                                int off_pos, int off_neg, int F, int out_f32_accumulate,
                                                int pairs) {
  const int wave = (blockIdx.x * blockDim.x + threadIdx.x) >> 6;
  const int lane = threadIdx.x & 63;
  if (wave >= nrows) return;
  const int r = wave;
  float p0 = 0.f, p1 = 0.f, q0 = 0.f, q1 = 0.f;
  // pairs: lane l holds features 2l and 2l + 1 (one 4- or 8-byte load per incidence, a
  // wave reading one contiguous row); otherwise features l and l + 64.
  const int f0 = pairs ? 2 * lane : lane, f1 = pairs ? 2 * lane + 1 : lane + 64;
  auto load = [&](int e, float& v0, float& v1, float& w) {
    w = weight[e];
    const int64_t base = (int64_t)col[e] * ldx + (w > 0.f ? xoff_pos : xoff_neg);
    v0 = v1 = 0.f;
    if (x_f32) {
      const float* x = reinterpret_cast<const float*>(X) + base;
      if (pairs && f1 < F) {
        const float2 v = *reinterpret_cast<const float2*>(x + f0);
        v0 = v.x;
        v1 = v.y;
      } else {
        if (f0 < F) v0 = x[f0];
        if (f1 < F) v1 = x[f1];
      }
    } else {
      const __bf16* x = reinterpret_cast<const __bf16*>(X) + base;
      if (pairs && f1 < F) {
        const uint32_t u = *reinterpret_cast<const uint32_t*>(x + f0);
        v0 = bf2f(__builtin_bit_cast(__bf16, (uint16_t)(u & 0xFFFFu)));
        v1 = bf2f(__builtin_bit_cast(__bf16, (uint16_t)(u >> 16)));
      } else {
        if (f0 < F) v0 = bf2f(x[f0]);
        if (f1 < F) v1 = bf2f(x[f1]);
      }
    }
  };
  auto add = [&](float v0, float v1, float w) {
    const float aw = fabsf(w);
    if (w > 0.f) {
      p0 += aw * v0;
      p1 += aw * v1;
    } else {
      q0 += aw * v0;
      q1 += aw * v1;
    }
  };
  // Four incidences per trip, their rows loaded before any is added (four row gathers in
  // flight per wave instead of one).
  int e = rowptr[r];
  const int end = rowptr[r + 1];
  for (; e + 4 <= end; e += 4) {
    float v0[4], v1[4], w[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) load(e + u, v0[u], v1[u], w[u]);
#pragma unroll
    for (int u = 0; u < 4; ++u) add(v0[u], v1[u], w[u]);
  }
  for (; e < end; ++e) {
    float v0, v1, w;
    load(e, v0, v1, w);
    add(v0, v1, w);
  }
  if (out_f32_accumulate) {
    float* o = reinterpret_cast<float*>(out) + (int64_t)r * ldo;
    if (pairs && f1 < F) {
      float2* d = reinterpret_cast<float2*>(o + off_pos + f0);
      const float2 v = *d;
      *d = make_float2(v.x + p0 + q0, v.y + p1 + q1);
    } else {
      if (f0 < F) o[off_pos + f0] += p0 + q0;
      if (f1 < F) o[off_pos + f1] += p1 + q1;
    }
  } else {
    __bf16* o = reinterpret_cast<__bf16*>(out) + (int64_t)r * ldo;
    if (pairs && f1 < F) {
      const auto pack = [](float a, float b) {
        return (uint32_t)__builtin_bit_cast(uint16_t, f2bf(a)) | ((uint32_t)__builtin_bit_cast(uint16_t, f2bf(b)) << 16);
      };
      *reinterpret_cast<uint32_t*>(o + off_pos + f0) = pack(p0, p1);
      *reinterpret_cast<uint32_t*>(o + off_neg + f0) = pack(q0, q1);
    } else {
      if (f0 < F) {
        o[off_pos + f0] = f2bf(p0);
        o[off_neg + f0] = f2bf(q0);
      }
      if (f1 < F) {
        o[off_pos + f1] = f2bf(p1);
        o[off_neg + f1] = f2bf(q1);
      }
    }
  }
}

// dZ = dH * (H > 0) (ReLU backward), written as bf16 for the next products, and fp32 column
// sums added into db: one add per column and workgroup, so few large workgroups (adds from
// different XCDs to one line queue up at memory).
//  * k_relu_back8: 128 features, 8 per thread (32-, 16- and 16-byte accesses).  74356 rows:
//    71 us with one feature per thread and one add per 128 threads, 17 us here.
//  * k_relu_back: any other width or alignment.
constexpr int RTHREADS = 512;

__global__ __launch_bounds__(RTHREADS) void k_relu_back8(const float* __restrict__ dH, int64_t ldd,
                                                         const __bf16* __restrict__ H, int64_t ldh, int rows,
                                                         __bf16* __restrict__ dZ, int64_t ldz,
                                                         float* __restrict__ db) {
  constexpr int RPB = RTHREADS / 16;  // rows per pass of a workgroup
  __shared__ float red[RPB][128 + 4];
  const int tid = threadIdx.x, f = (tid & 15) * 8;
  float s[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  for (int r = blockIdx.x * RPB + (tid >> 4); r < rows; r += gridDim.x * RPB) {
    const f4* d = reinterpret_cast<const f4*>(dH + (int64_t)r * ldd + f);
    const f4 a = d[0], b = d[1];
    const bf8 h = *reinterpret_cast<const bf8*>(H + (int64_t)r * ldh + f);
    bf8 z;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const float g = bf2f(h[i]) > 0.f ? (i < 4 ? a[i & 3] : b[i & 3]) : 0.f;
      z[i] = f2bf(g);
      s[i] += g;
    }
    *reinterpret_cast<bf8*>(dZ + (int64_t)r * ldz + f) = z;
  }
  if (!db) return;
#pragma unroll
  for (int i = 0; i < 8; ++i) red[tid >> 4][f + i] = s[i];
  __syncthreads();
  if (tid < 128) {
    float t = 0.f;
    for (int k = 0; k < RPB; ++k) t += red[k][tid];
    atomicAdd(&db[tid], t);
  }
}

__global__ __launch_bounds__(256) void k_relu_back(const float* __restrict__ dH, int64_t ldd,
                                                   const __bf16* __restrict__ H, int64_t ldh, int rows, int F,
                                                   __bf16* __restrict__ dZ, int64_t ldz, float* __restrict__ db) {
  const int f = threadIdx.x % 128;
  const int rgroup = (blockIdx.x * blockDim.x + threadIdx.x) / 128;
  const int ngroups = (gridDim.x * blockDim.x) / 128;
  float s = 0.f;
  if (f < F) {
    for (int r = rgroup; r < rows; r += ngroups) {
      const float g = bf2f(H[(int64_t)r * ldh + f]) > 0.f ? dH[(int64_t)r * ldd + f] : 0.f;
      dZ[(int64_t)r * ldz + f] = f2bf(g);
      s += g;
    }
    if (db) atomicAdd(&db[f], s);
  }
}

// y[r] = sum_f H[r, f] w[f] + b ; loss = sum_r mask[r] (y[r]-t[r])^2 / count ;
// dy[r] = 2 mask[r] (y[r]-t[r]) / count ; dH[r, f] = dy[r] w[f] ; dw[f] += sum_r dy[r] H[r, f].
// One wave per row, features l and 64 + l on lane l; a workgroup adds its share of dw, db and
// the loss once.  7185 rows: 31 us with a workgroup and seven barriers per row, 18 us here.
__global__ __launch_bounds__(256) void k_head(const __bf16* __restrict__ H, int64_t ldh, int rows,
                                              const float* __restrict__ w, const float* __restrict__ b,
                                              const float* __restrict__ target, const float* __restrict__ mask,
                                              float inv_count, float* __restrict__ y, float* __restrict__ loss,
                                              float* __restrict__ dH, float* __restrict__ dw, float* __restrict__ db,
                                              int F, int train) {
  __shared__ float red[4][128 + 2];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int f0 = lane, f1 = lane + 64;
  const float w0 = f0 < F ? w[f0] : 0.f, w1 = f1 < F ? w[f1] : 0.f, b0 = b[0];
  float dw0 = 0.f, dw1 = 0.f, db_acc = 0.f, loss_acc = 0.f;  // this wave's rows
  for (int r = blockIdx.x * 4 + wave; r < rows; r += gridDim.x * 4) {
    const float h0 = f0 < F ? bf2f(H[(int64_t)r * ldh + f0]) : 0.f, h1 = f1 < F ? bf2f(H[(int64_t)r * ldh + f1]) : 0.f;
    float s = h0 * w0 + h1 * w1;
    for (int m = 32; m > 0; m >>= 1) s += __shfl_xor(s, m);
    const float yr = s + b0;
    if (lane == 0) y[r] = yr;
    if (train) {
      const float m = mask ? mask[r] : 1.f;
      const float d = yr - target[r];
      const float g = 2.f * m * d * inv_count;
      loss_acc += m * d * d * inv_count;
      db_acc += g;
      if (f0 < F) dH[(int64_t)r * F + f0] = g * w0;
      if (f1 < F) dH[(int64_t)r * F + f1] = g * w1;
      dw0 += g * h0;
      dw1 += g * h1;
    }
  }
  if (!train) return;
  red[wave][f0] = dw0;
  red[wave][f1] = dw1;
  if (lane == 0) {
    red[wave][128] = db_acc;
    red[wave][129] = loss_acc;
  }
  __syncthreads();
  const int t = threadIdx.x;
  if (t < F) atomicAdd(&dw[t], (red[0][t] + red[1][t]) + (red[2][t] + red[3][t]));
  if (t == 128) atomicAdd(db, (red[0][t] + red[1][t]) + (red[2][t] + red[3][t]));
  if (t == 129) atomicAdd(loss, (red[0][t] + red[1][t]) + (red[2][t] + red[3][t]));
}

__global__ __launch_bounds__(256) void k_adam(float* __restrict__ p, const float* __restrict__ g,
                                              float* __restrict__ m, float* __restrict__ v,
                                              __bf16* __restrict__ pbf, int64_t n, float lr, float b1, float b2,
                                              float eps, float c1, float c2, float wd) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
    const float gi = g[i] + wd * p[i];
    const float mi = b1 * m[i] + (1.f - b1) * gi;
    const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    const float upd = lr * (mi / c1) / (sqrtf(vi / c2) + eps);
    p[i] -= upd;
    if (pbf) pbf[i] = f2bf(p[i]);
  }
}

__global__ __launch_bounds__(256) void k_cast_bf16(const float* __restrict__ x, __bf16* __restrict__ y, int64_t n) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
    y[i] = f2bf(x[i]);
}

inline uintptr_t at(const void* p) { return reinterpret_cast<uintptr_t>(p); }

// k_panel takes whole multiples of 128 columns, K of 32, 128, 256 or 384 (the network's
// widths) and 16-byte aligned rows of A, B and C (bias included).  Below 1024 rows the
// 64 x 64 tiles of k_gemm fill as many CUs without a panel to stage.
inline bool panel_fits(const void* A, int64_t sam, int64_t sak, const void* B, int64_t sbk, int64_t sbn, const void* C,
                       int64_t ldc, int M, int N, int K, const float* bias, int out_bf16) {
  if (M < 1024 || N % PN || (K != 32 && K != 128 && K != 256 && K != 384)) return false;
  if (sak != 1 || (sam & 7) || ((at(A) | at(B) | at(bias)) & 15)) return false;
  if (!(sbk == 1 && (sbn & 7) == 0) && !(sbn == 1 && (sbk & 7) == 0)) return false;
  return (ldc & 3) == 0 && (at(C) & (out_bf16 ? 7 : 15)) == 0;
}

template <int KS>
int launch_panel(const void* A, int64_t lda, const void* B, int64_t sbk, int64_t sbn, void* C, int64_t ldc, int M, int N,
                 const float* bias, int relu, int out_bf16, int accumulate, ts_stream stream) {
  // As many workgroups as fit the 256 CUs at once (their panels in 160 KiB of LDS, at most
  // four), at most one per eight tiles.
  constexpr int per_cu = std::min(4, (160 * 1024) / (PN * (32 * KS + 8) * 2));
  const int tiles = (M + 15) / 16;
  const dim3 grid(std::min((tiles + 7) / 8, 256 * per_cu), N / PN);
  hipLaunchKernelGGL((k_panel<KS>), grid, dim3(PTHREADS), 0, reinterpret_cast<hipStream_t>(stream),
                     reinterpret_cast<const __bf16*>(A), lda, reinterpret_cast<const __bf16*>(B), sbk, sbn, C, ldc, M,
                     bias, relu, out_bf16, accumulate);
  return hipGetLastError() == hipSuccess ? TS_OK : TS_EHIP;
}

// Blocks of rows of a weight gradient: one per 256 rows, up to a workgroup per CU.
inline int wgrad_blocks(int M, int rows) {
  const int mtiles = std::max(1, (M + WM - 1) / WM);
  return std::max(1, std::min((rows + 255) / 256, 256 / mtiles));
}

inline int blocks_for(int64_t n, int per) { return (int)std::min<int64_t>((n + per - 1) / per, 65535); }

}  // namespace

extern "C" {

int ts_gnn_gemm(const void* A, int64_t sam, int64_t sak, const void* B, int64_t sbk, int64_t sbn, void* C,
                int64_t ldc, int32_t M, int32_t N, int32_t K, const float* bias, int32_t relu, int32_t out_bf16,
                int32_t accumulate, ts_stream stream) {
  if (!A || !B || !C || M < 0 || N < 0 || K < 0) return TS_EINVAL;
  if (M == 0 || N == 0) return TS_OK;
  if (panel_fits(A, sam, sak, B, sbk, sbn, C, ldc, M, N, K, bias, out_bf16)) {
    switch (K / 32) {
      case 1: return launch_panel<1>(A, sam, B, sbk, sbn, C, ldc, M, N, bias, relu, out_bf16, accumulate, stream);
      case 4: return launch_panel<4>(A, sam, B, sbk, sbn, C, ldc, M, N, bias, relu, out_bf16, accumulate, stream);
      case 8: return launch_panel<8>(A, sam, B, sbk, sbn, C, ldc, M, N, bias, relu, out_bf16, accumulate, stream);
      default: return launch_panel<12>(A, sam, B, sbk, sbn, C, ldc, M, N, bias, relu, out_bf16, accumulate, stream);
    }
  }
  dim3 grid((N + TN - 1) / TN, (M + TM - 1) / TM, 1);
  if (grid.y > 65535) return TS_EUNSUPPORTED;
  // Few output tiles over a long K (weight gradients X^T dZ): split K across blocks and
  // add fp32 partial sums into C, which the caller has zeroed (requires accumulate).
  int kchunk = K > 0 ? K : 1;
  const int tiles = (int)(grid.x * grid.y);
  if (tiles < 256 && K >= 4096 && !out_bf16 && accumulate && !bias && !relu) {
    int splits = std::min(256 / tiles + 1, (K + 2047) / 2048);
    kchunk = ((K + splits - 1) / splits + TK - 1) / TK * TK;
    grid.z = (K + kchunk - 1) / kchunk;
  }
  hipLaunchKernelGGL(k_gemm, grid, dim3(256), 0, reinterpret_cast<hipStream_t>(stream),
                     reinterpret_cast<const __bf16*>(A), sam, sak, reinterpret_cast<const __bf16*>(B), sbk, sbn, C,
                     ldc, M, N, K, bias, relu, out_bf16, accumulate, kchunk);
  return hipGetLastError() == hipSuccess ? TS_OK : TS_EHIP;
}

int ts_gnn_wgrad_scratch(int32_t M, int32_t rows, int64_t* bytes) {
  if (!bytes || M < 0 || rows < 0 || M > 256 * WM) return TS_EINVAL;
  *bytes = (int64_t)wgrad_blocks(M, rows) * ((M + WM - 1) / WM) * WM * WM * 4;
  return TS_OK;
}

int ts_gnn_wgrad(const void* X, int64_t ldx, const void* dZ, int64_t ldz, int32_t M, int32_t N, int32_t rows, float* dW,
                 int64_t ldw, void* scratch, int64_t scratch_bytes, ts_stream stream) {
  if (!X || !dZ || !dW || M < 0 || N < 0 || rows < 0) return TS_EINVAL;
  if (M == 0 || N == 0 || rows == 0) return TS_OK;
  int64_t need = 0;
  const bool fits = N == WM && M % 4 == 0 && M <= 256 * WM && ((ldx | ldz | ldw) & 3) == 0 &&
                    ((at(X) | at(dZ)) & 7) == 0 && ((at(dW) | at(scratch)) & 15) == 0 && scratch &&
                    ts_gnn_wgrad_scratch(M, rows, &need) == TS_OK && need <= scratch_bytes;
  if (!fits) return ts_gnn_gemm(X, 1, ldx, dZ, ldz, 1, dW, ldw, M, N, rows, nullptr, 0, 0, 1, stream);
  const int mtiles = (M + WM - 1) / WM, blocks = wgrad_blocks(M, rows);
  const int per = ((rows + blocks - 1) / blocks + WK - 1) / WK * WK;
  const int used = (rows + per - 1) / per;
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  float* part = reinterpret_cast<float*>(scratch);
  hipLaunchKernelGGL(k_wgrad, dim3(mtiles, used), dim3(256), 0, s, reinterpret_cast<const __bf16*>(X), ldx,
                     reinterpret_cast<const __bf16*>(dZ), ldz, M, rows, per, part);
  hipLaunchKernelGGL(k_wgrad_sum, dim3((M * (WM / 4) + 63) / 64), dim3(256), 0, s, part, M, mtiles, used, dW, ldw);
  return hipGetLastError() == hipSuccess ? TS_OK : TS_EHIP;
}

int ts_gnn_segsum(const int32_t* rowptr, const int32_t* col, const float* weight, int32_t nrows, const void* X,
                  int64_t ldx, int32_t xoff_pos, int32_t xoff_neg, int32_t x_f32, void* out, int64_t ldo,
                  int32_t off_pos, int32_t off_neg, int32_t F, int32_t out_f32_accumulate, ts_stream stream) {
  if (nrows < 0 || F < 0 || F > 128) return TS_EINVAL;
  if (nrows == 0) return TS_OK;
  if (!rowptr || !col || !weight || !X || !out) return TS_EINVAL;
  const int threads = 256;
  const int64_t waves = nrows;
  // 128 features that start at 16-byte boundaries: a wave per row below 16384 rows (16 lanes
  // per row would leave CUs without a wave: 7185 rows 73 us), else 16 lanes per row.
  const int el = x_f32 ? 3 : 7, eo = out_f32_accumulate ? 3 : 7;
  if (F == 128 && ((at(X) | at(out)) & 15) == 0 && ((ldx | xoff_pos | xoff_neg) & el) == 0 &&
      ((ldo | off_pos | (out_f32_accumulate ? 0 : off_neg)) & eo) == 0 && nrows < (1 << 27)) {
    const bool few = nrows < 16384;
    const int per = few ? 4 : 16;  // rows per workgroup
    auto go = [&](auto kernel) {
      hipLaunchKernelGGL(kernel, dim3((nrows + per - 1) / per), dim3(threads), 0, reinterpret_cast<hipStream_t>(stream),
                         rowptr, col, weight, nrows, X, ldx, xoff_pos, xoff_neg, out, ldo, off_pos, off_neg);
      return hipGetLastError() == hipSuccess ? TS_OK : TS_EHIP;
    };
    if (x_f32 && out_f32_accumulate) return few ? go(k_segsum_row<true, true>) : go(k_segsum16<true, true>);
    if (!x_f32 && !out_f32_accumulate) return few ? go(k_segsum_row<false, false>) : go(k_segsum16<false, false>);
    if (x_f32) return few ? go(k_segsum_row<true, false>) : go(k_segsum16<true, false>);
    return few ? go(k_segsum_row<false, true>) : go(k_segsum16<false, true>);
  }
  // Feature pairs need every pair's first element at an even element offset (8- or
  // 4-byte aligned pair loads and stores).
  const int pairs = ((reinterpret_cast<uintptr_t>(X) | reinterpret_cast<uintptr_t>(out)) & 7) == 0 &&
                    ((ldx | xoff_pos | xoff_neg | ldo | off_pos | off_neg) & 1) == 0;
  hipLaunchKernelGGL(k_segsum, dim3(blocks_for(waves * 64, threads)), dim3(threads), 0,
                     reinterpret_cast<hipStream_t>(stream), rowptr, col, weight, nrows, X, ldx, xoff_pos, xoff_neg,
                     x_f32, out, ldo, off_pos, off_neg, F, out_f32_accumulate, pairs);
  return hipGetLastError() == hipSuccess ? TS_OK : TS_EHIP;
}

int ts_gnn_relu_back(const float* dH, int64_t ldd, const void* H, int64_t ldh, int32_t rows, int32_t F, void* dZ,
                     int64_t ldz, float* db, ts_stream stream) {
  if (!dH || !H || !dZ || rows < 0 || F < 0 || F > 128) return TS_EINVAL;
  if (rows == 0) return TS_OK;
  if (F == 128 && ((at(dH) | at(H) | at(dZ)) & 15) == 0 && (ldd & 3) == 0 && ((ldh | ldz) & 7) == 0) {
    const int rpb = RTHREADS / 16;
    hipLaunchKernelGGL(k_relu_back8, dim3(std::min(256, (rows + rpb - 1) / rpb)), dim3(RTHREADS), 0,
                       reinterpret_cast<hipStream_t>(stream), dH, ldd, reinterpret_cast<const __bf16*>(H), ldh, rows,
                       reinterpret_cast<__bf16*>(dZ), ldz, db);
    return hipGetLastError() == hipSuccess ? TS_OK : TS_EHIP;
  }
  const int grid = std::min(1024, std::max(1, rows / 16));
  hipLaunchKernelGGL(k_relu_back, dim3(grid), dim3(256), 0, reinterpret_cast<hipStream_t>(stream), dH, ldd,
                     reinterpret_cast<const __bf16*>(H), ldh, rows, F, reinterpret_cast<__bf16*>(dZ), ldz, db);
  return hipGetLastError() == hipSuccess ? TS_OK : TS_EHIP;
}

int ts_gnn_head(const void* H, int64_t ldh, int32_t rows, const float* w, const float* b, const float* target,
                const float* mask, float inv_count, float* y, float* loss, float* dH, float* dw, float* db,
                int32_t F, int32_t train, ts_stream stream) {
  if (!H || !w || !b || !y || rows < 0 || F < 0 || F > 128) return TS_EINVAL;
  if (train && (!target || !loss || !dH || !dw || !db)) return TS_EINVAL;
  if (rows == 0) return TS_OK;
  hipLaunchKernelGGL(k_head, dim3(std::min((rows + 3) / 4, 512)), dim3(256), 0, reinterpret_cast<hipStream_t>(stream),
                     reinterpret_cast<const __bf16*>(H), ldh, rows, w, b, target, mask, inv_count, y, loss, dH, dw,
                     db, F, train);
  return hipGetLastError() == hipSuccess ? TS_OK : TS_EHIP;
}

int ts_gnn_adam(float* p, const float* g, float* m, float* v, void* pbf, int64_t n, float lr, float b1, float b2,
                float eps, int32_t step, float wd, ts_stream stream) {
  if (!p || !g || !m || !v || n < 0 || step < 1) return TS_EINVAL;
  if (n == 0) return TS_OK;
  const float c1 = 1.f - powf(b1, (float)step), c2 = 1.f - powf(b2, (float)step);
  hipLaunchKernelGGL(k_adam, dim3(blocks_for(n, 256)), dim3(256), 0, reinterpret_cast<hipStream_t>(stream), p, g, m,
                     v, reinterpret_cast<__bf16*>(pbf), n, lr, b1, b2, eps, c1, c2, wd);
  return hipGetLastError() == hipSuccess ? TS_OK : TS_EHIP;
}

int ts_gnn_cast_bf16(const float* x, void* y, int64_t n, ts_stream stream) {
  if (!x || !y || n < 0) return TS_EINVAL;
  if (n == 0) return TS_OK;
  hipLaunchKernelGGL(k_cast_bf16, dim3(blocks_for(n, 256)), dim3(256), 0, reinterpret_cast<hipStream_t>(stream), x,
                     reinterpret_cast<__bf16*>(y), n);
  return hipGetLastError() == hipSuccess ? TS_OK : TS_EHIP;
}

}  // extern "C"

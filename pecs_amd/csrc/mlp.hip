// Learned warm start: a network trained on steady states produced by the
// time stepper.  A fully connected encoder (nin inputs -> nlayers hidden
// ReLU layers) feeds either nout linear outputs (a plain MLP) or a
// convolutional decoder: the encoder's last layer (ReLU) is read as a
// c0 x g0 x g0 feature map, and each decoder stage is an optional nearest
// x2 upsampling followed by a 3x3 convolution (zero padding), ReLU after all
// but the last stage.  Training is FP32 (forward, backward, Adam); inference
// is FP32 or BF16 storage with FP32 accumulation, all in the kernels of this
// file; the C-ABI (include/pecs_abi.h, pecs_mlp_*) moves host arrays in and
// out.
//
// Every matrix product runs on the matrix cores: v_mfma_f32_16x16x4f32 for
// FP32, v_mfma_f32_16x16x16bf16_1k for BF16.  MFMA operand layout (both): lane
// l holds A[l%16][k], B[k][l%16] with k = l/16 (FP32) or 4(l/16)..4(l/16)+3
// (BF16); accumulator lane l, register r holds C[4(l/16)+r][l%16].
//   k_dense    the dense layers and their gradients, one 16 x 16 tile per wave
//   k_conv     the convolutions and their input gradients as implicit GEMMs on
//              input strips staged in LDS
//   k_conv_dw  their weight and bias gradients on the same strips
//   k_mm       64 x 64 tiles staged in LDS: dense products that fill the chip
//              with them, and any of the convolution products, im2col gathered
//              element by element, on maps that do not divide into strips of
//              whole rows
// Every product adds its k terms in ascending order in groups of 4 (FP32) or
// 16 (BF16), whichever kernel runs it: the forward pass is the same bit by bit.
//
// Parameters are one FP32 array: per dense layer W (n_in x n_out, row-major)
// then b (n_out); per convolution W (cout x cin x 3 x 3) then b (cout).
// Feature maps are NCHW per sample.  Loss: mean squared error over the batch
// and outputs.
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdint>
#include <cstring>
#include <memory>
#include <random>
#include <stdexcept>
#include <string>
#include <type_traits>
#include <vector>

#include "../../include/pecs_abi.h"

namespace {

thread_local std::string g_mlp_error;

#define MCHECK(x)                                                                                 \
  do {                                                                                            \
    hipError_t e_ = (x);                                                                          \
    if (e_ != hipSuccess) throw std::runtime_error(std::string(#x) + ": " + hipGetErrorString(e_)); \
  } while (0)

typedef float v4f __attribute__((ext_vector_type(4)));
typedef short v4s __attribute__((ext_vector_type(4)));

__device__ __forceinline__ float bf16_to_f32(uint16_t h) {
  uint32_t u = (uint32_t)h << 16;
  float f;
  memcpy(&f, &u, 4);
  return f;
}

// Round to nearest even (NaN not expected here).
__host__ __device__ __forceinline__ uint16_t f32_to_bf16(float f) {
  uint32_t u;
  memcpy(&u, &f, 4);
  u += 0x7fffu + ((u >> 16) & 1u);
  return (uint16_t)(u >> 16);
}

template <class T>
__device__ __forceinline__ float ldv(const T* p, int64_t i);
template <>
__device__ __forceinline__ float ldv<float>(const float* p, int64_t i) {
  return p[i];
}
template <>
__device__ __forceinline__ float ldv<uint16_t>(const uint16_t* p, int64_t i) {
  return bf16_to_f32(p[i]);
}

// An operand matrix of k_mm, read element by element while staging tiles.
enum OpKind {
  OP_ROW = 0,     // (r, c) = p[r ld + c]
  OP_TRANS = 1,   // (r, c) = p[c ld + r]
  OP_IM2COL = 2,  // (ci 9 + t, b R^2 + px): input pixel under tap t of output pixel px (conv forward B)
  OP_IM2COL_T = 3,  // its transpose (weight gradient B)
  OP_CHAN = 4,    // (ch, b R^2 + px) of a C x R x R map per sample (weight gradient A)
  OP_WT = 5,      // (ci, co 9 + t) of W[co][ci][t], C = cin (input gradient A)
  OP_DCOL = 6     // (co 9 + t, b R^2 + px): output gradient at px - offset(t) (input gradient B)
};

struct Opnd {
  const void* p;
  int kind;
  int ld;  // OP_ROW / OP_TRANS
  int C;   // channels of the map read (OP_WT: cin)
  int R;   // side of the convolution's output (and upsampled input)
  int up;  // OP_IM2COL*: the input map is R/2 x R/2, upsampled by 2 (nearest)
};

template <class T>
__device__ __forceinline__ float opnd(const Opnd& o, int r, int c) {
  const T* p = static_cast<const T*>(o.p);
  switch (o.kind) {
    case OP_ROW:
      return ldv(p, (int64_t)r * o.ld + c);
    case OP_TRANS:
      return ldv(p, (int64_t)c * o.ld + r);
    case OP_IM2COL:
    case OP_IM2COL_T: {
      const int k = o.kind == OP_IM2COL ? r : c, n = o.kind == OP_IM2COL ? c : r;
      const int R2 = o.R * o.R;
      const int ci = k / 9, t = k - 9 * ci;
      const int b = n / R2, px = n - b * R2;
      const int y = px / o.R + t / 3 - 1, x = px % o.R + t % 3 - 1;
      if (y < 0 || y >= o.R || x < 0 || x >= o.R) return 0.f;
      const int Ri = o.R >> o.up;
      return ldv(p, (((int64_t)b * o.C + ci) * Ri + (y >> o.up)) * Ri + (x >> o.up));
    }
    case OP_CHAN: {
      const int R2 = o.R * o.R;
      const int b = c / R2, px = c - b * R2;
      return ldv(p, ((int64_t)b * o.C + r) * R2 + px);
    }
    case OP_WT: {
      const int co = c / 9, t = c - 9 * co;
      return ldv(p, ((int64_t)co * o.C + r) * 9 + t);
    }
    default: {  // OP_DCOL
      const int R2 = o.R * o.R;
      const int co = r / 9, t = r - 9 * co;
      const int b = c / R2, px = c - b * R2;
      const int y = px / o.R - (t / 3 - 1), x = px % o.R - (t % 3 - 1);
      if (y < 0 || y >= o.R || x < 0 || x >= o.R) return 0.f;
      return ldv(p, (((int64_t)b * o.C + co) * o.R + y) * o.R + x);
    }
  }
}

// Where k_mm writes C[m][n]: row-major (ld), or as channel m of the maps
// (n = b R^2 + px).  Bias per column (dense) or per row (convolution).
struct Dst {
  void* p;
  int chan;  // 0: p[m ld + n]; 1: p[(b C + m) R^2 + px]
  int ld, C, R;
  const float* bias;
  int bias_row;
  int relu;
  int bf16;  // store BF16 (hidden activations of BF16 inference)
  const float* mask;  // ReLU backward: zero where mask (the layer's output, indexed as p) is not positive
};

constexpr int TM = 64, TN = 64, TK = 16;  // tile: 64 x 64 outputs, 16-deep k steps, 4 waves of 32 x 32

// Epilogue of C[m][n] = v: bias, ReLU, store (row-major or as map channel m).
__device__ __forceinline__ void mm_store(const Dst& D, int m, int n, float v) {
  if (D.bias) v += D.bias_row ? D.bias[m] : D.bias[n];
  if (D.relu && v < 0.f) v = 0.f;
  int64_t o;
  if (D.chan) {
    const int R2 = D.R * D.R;
    const int b = n / R2, px = n - b * R2;
    o = ((int64_t)b * D.C + m) * R2 + px;
  } else {
    o = (int64_t)m * D.ld + n;
  }
  if (D.mask && D.mask[o] <= 0.f) v = 0.f;
  if (D.bf16) static_cast<uint16_t*>(D.p)[o] = f32_to_bf16(v);
  else static_cast<float*>(D.p)[o] = v;
}

// C[M x N] = A[M x K] B[K x N] on the matrix cores.  T: FP32 (MFMA 16x16x4
// f32) or BF16 (MFMA 16x16x16 bf16, operands as stored, FP32 accumulation).
// The k loop runs in a fixed order: results are reproducible.
// Split k: block z of gridDim.z covers k in [z kchunk, (z + 1) kchunk) and
// writes its raw sums to part[(z M + m) N + n]; k_mm_reduce adds the slices
// in order (deterministic) and applies the epilogue.  Used where M x N has
// few tiles and K is long (the weight gradients, K = batch x pixels).
template <class T>
__global__ __launch_bounds__(256) void k_mm(Opnd A, Opnd B, Dst D, int M, int N, int K, int kchunk,
                                            float* __restrict__ part) {
  constexpr bool BF = sizeof(T) == 2;
  // BF16 rows padded by 4 halves (8-byte aligned 4-wide reads), FP32 by 1
  __shared__ T As[TM][TK + (BF ? 4 : 1)];
  __shared__ T Bs[TK][TN + (BF ? 4 : 1)];
  const int m0 = blockIdx.y * TM, n0 = blockIdx.x * TN;
  const int w = threadIdx.x >> 6, l = threadIdx.x & 63;
  const int wm = (w & 1) * 32, wn = (w >> 1) * 32;
  const int li = l & 15, lq = l >> 4;
  v4f acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[i][j] = v4f{0.f, 0.f, 0.f, 0.f};
  const int kbeg = blockIdx.z * kchunk, kend = min(K, kbeg + kchunk);
  for (int k0 = kbeg; k0 < kend; k0 += TK) {
    for (int e = threadIdx.x; e < TM * TK; e += 256) {
      const int r = e / TK, kk = e % TK;
      const int gm = m0 + r, gk = k0 + kk;
      const float v = (gm < M && gk < kend) ? opnd<T>(A, gm, gk) : 0.f;
      if constexpr (BF) As[r][kk] = f32_to_bf16(v);
      else As[r][kk] = v;
    }
    for (int e = threadIdx.x; e < TK * TN; e += 256) {
      const int kk = e / TN, c = e % TN;
      const int gn = n0 + c, gk = k0 + kk;
      const float v = (gn < N && gk < kend) ? opnd<T>(B, gk, gn) : 0.f;
      if constexpr (BF) Bs[kk][c] = f32_to_bf16(v);
      else Bs[kk][c] = v;
    }
    __syncthreads();
    if constexpr (BF) {
      v4s a[2], b[2];
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          a[i][e] = (short)As[wm + 16 * i + li][4 * lq + e];
          b[i][e] = (short)Bs[4 * lq + e][wn + 16 * i + li];
        }
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a[i], b[j], acc[i][j], 0, 0, 0);
    } else {
#pragma unroll
      for (int ks = 0; ks < TK; ks += 4) {
        float a[2], b[2];
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          a[i] = As[wm + 16 * i + li][ks + lq];
          b[i] = Bs[ks + lq][wn + 16 * i + li];
        }
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
          for (int j = 0; j < 2; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i], b[j], acc[i][j], 0, 0, 0);
      }
    }
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int m = m0 + wm + 16 * i + 4 * lq + r, n = n0 + wn + 16 * j + li;
        if (m >= M || n >= N) continue;
        if (part) part[((int64_t)blockIdx.z * M + m) * N + n] = acc[i][j][r];
        else mm_store(D, m, n, acc[i][j][r]);
      }
}

__global__ __launch_bounds__(256) void k_mm_reduce(const float* __restrict__ part, int splits, Dst D, int M, int N) {
  const int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (e >= (int64_t)M * N) return;
  float v = 0.f;
  for (int z = 0; z < splits; ++z) v += part[(int64_t)z * M * N + e];
  mm_store(D, (int)(e / N), (int)(e % N), v);
}

// ---- dense products ---------------------------------------------------------
// C[m][n] = sum_k a[m am + k ak] b[k bk + n bn], one 16 x 16 tile per wave, the
// operands straight from L2 into registers (no LDS, no barriers), two groups of
// DU steps in turn so that one's loads run under the other's MFMAs.  With the
// few rows of a minibatch the 64 x 64 tiles of k_mm left 4 to 64 workgroups
// with a barrier and a load latency per 16 k (42 us at 32 x 256 x 256, 449 us
// at 32 x 256 x 4096).  blockIdx.z: k slice of kchunk (a multiple of 16), raw
// sums to part.
template <class T>
__global__ __launch_bounds__(256) void k_dense(const T* __restrict__ a, int am, int ak, const T* __restrict__ b, int bk,
                                               int bn, Dst D, int M, int N, int K, int kchunk,
                                               float* __restrict__ part) {
  constexpr bool BF = sizeof(T) == 2;
  constexpr int KS = BF ? 16 : 4, E = BF ? 4 : 1, DU = BF ? 4 : 8;  // k per MFMA, entries per lane, steps per group
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int n0 = (blockIdx.x * 4 + wave) * 16, m0 = blockIdx.y * 16;
  if (n0 >= N) return;
  const int li = lane & 15, lq = lane >> 4;
  const int m = min(m0 + li, M - 1), n = min(n0 + li, N - 1);  // (rows and columns past the end are not stored)
  const T* __restrict__ pa = a + (int64_t)m * am;
  const T* __restrict__ pb = b + (int64_t)n * bn;
  const int kbeg = blockIdx.z * kchunk, kend = min(K, kbeg + kchunk);
  v4f acc = {0.f, 0.f, 0.f, 0.f};
  T A[2][DU][E], B[2][DU][E];
  auto load = [&](int k0, T (&x)[DU][E], T (&y)[DU][E]) {
#pragma unroll
    for (int u = 0; u < DU; ++u)
#pragma unroll
      for (int e = 0; e < E; ++e) {
        const int k = k0 + u * KS + lq * E + e, kc = min(k, kend - 1);
        const T va = pa[(int64_t)kc * ak], vb = pb[(int64_t)kc * bk];
        x[u][e] = k < kend ? va : T(0);
        y[u][e] = k < kend ? vb : T(0);
      }
  };
  auto mma = [&](const T (&x)[DU][E], const T (&y)[DU][E]) {
#pragma unroll
    for (int u = 0; u < DU; ++u) {
      if constexpr (BF) {
        v4s xa, yb;
#pragma unroll
        for (int e = 0; e < E; ++e) {
          xa[e] = (short)x[u][e];
          yb[e] = (short)y[u][e];
        }
        acc = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(xa, yb, acc, 0, 0, 0);
      } else {
        acc = __builtin_amdgcn_mfma_f32_16x16x4f32(x[u][0], y[u][0], acc, 0, 0, 0);
      }
    }
  };
  load(kbeg, A[0], B[0]);
  for (int k0 = kbeg; k0 < kend; k0 += 2 * DU * KS) {
    if (k0 + DU * KS < kend) load(k0 + DU * KS, A[1], B[1]);
    mma(A[0], B[0]);
    if (k0 + DU * KS >= kend) break;
    if (k0 + 2 * DU * KS < kend) load(k0 + 2 * DU * KS, A[0], B[0]);
    mma(A[1], B[1]);
  }
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int mm = m0 + 4 * lq + r, nn = n0 + li;
    if (mm >= M || nn >= N) continue;
    if (part) part[((int64_t)blockIdx.z * M + mm) * N + nn] = acc[r];
    else mm_store(D, mm, nn, acc[r]);
  }
}

// ---- convolutions on staged strips ------------------------------------------
// A strip is P consecutive output pixels of one sample, whole rows; its input
// (all channels, a border of one pixel, zeros outside the map, upsampled if the
// stage upsamples) is staged in LDS once, so that the operand of tap (ci, t) at
// a pixel is at (pixel offset) + (tap offset): two table look-ups per MFMA
// instead of k_mm's divisions, bounds checks and loads per element.
struct Conv {
  int C;     // channels of the staged map
  int R;     // side of the output (and of the upsampled input)
  int up;    // the map read is R/2 x R/2
  int P;     // output pixels per strip
  int M, K;  // output channels, C * 9
  int rows() const { return P / R; }
  int ch() const { return (P / R + 2) * (R + 2); }  // staged entries per channel
};

// The rows of the strip and one above and below, all channels, 8 loads per
// thread in flight (one row per wave at a time, W entries in passes of 64, cost
// a load latency per row: 32 channels at R = 64 staged for longer than they
// were multiplied).  R is a power of two (it divides P); the border columns are
// zero by themselves.
template <class T>
__device__ __forceinline__ void conv_stage(const Conv& c, const T* __restrict__ in, int smp, int y0, T* sIn) {
  const int W = c.R + 2, rows = c.P / c.R + 2, Ri = c.R >> c.up, nrow = c.C * rows;
  const int sh = 31 - __clz(c.R), n = nrow << sh;
  const uint32_t inv = 0xffffffffu / (uint32_t)rows + 1;  // q / rows = umulhi(q, inv) for q < 2^16 (rows >= 3)
  const T* src = in + (int64_t)smp * c.C * Ri * Ri;
  for (int q = threadIdx.x; q < nrow; q += 256) sIn[q * W] = sIn[q * W + W - 1] = T(0);
  constexpr int U = 8;
  for (int e0 = threadIdx.x; e0 < n; e0 += 256 * U) {
    T v[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int e = min(e0 + 256 * u, n - 1), x = e & (c.R - 1), q = e >> sh;
      const int ci = (int)__umulhi((uint32_t)q, inv), y = y0 + q - ci * rows - 1;
      const T t = src[(ci * Ri + (min(max(y, 0), c.R - 1) >> c.up)) * Ri + (x >> c.up)];
      v[u] = y >= 0 && y < c.R ? t : T(0);
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int e = e0 + 256 * u;
      if (e < n) sIn[(e >> sh) * W + (e & (c.R - 1)) + 1] = v[u];
    }
  }
}

// Forward (FLIP 0): out[m][px] = sum over (ci, t) of w[m][ci][t] in[ci][px + off(t)];
// input gradient (FLIP 1): the staged map is the output gradient (C = the
// stage's output channels), out[m][px] = sum over (co, t) of w[co][m][t]
// in[co][px - off(t)].  MW waves of 16 output channels, 4 / MW groups of NC
// 16-pixel blocks.
template <class T, int FLIP, int MW, int NC>
__global__ __launch_bounds__(256) void k_conv(Conv c, const T* __restrict__ in, const T* __restrict__ w, Dst D) {
  constexpr bool BF = sizeof(T) == 2;
  constexpr int KS = BF ? 16 : 4, E = BF ? 4 : 1, DU = BF ? 2 : 8;
  extern __shared__ __align__(16) char smem[];
  int2* sK = reinterpret_cast<int2*>(smem);        // per k: tap offset in the strip, weight offset
  T* sIn = reinterpret_cast<T*>(smem + (size_t)c.K * sizeof(int2));
  const int W = c.R + 2, R2 = c.R * c.R, CH = (c.P / c.R + 2) * W;
  const int64_t n0 = (int64_t)blockIdx.x * c.P;
  const int smp = (int)(n0 / R2), px0 = (int)(n0 - (int64_t)smp * R2);
  for (int k = threadIdx.x; k < c.K; k += 256) {
    const int ci = k / 9, t = k - 9 * ci, ty = t / 3, tx = t - 3 * ty;
    sK[k] = FLIP ? make_int2(ci * CH + (2 - ty) * W + 2 - tx, ci * c.M * 9 + t) : make_int2(ci * CH + ty * W + tx, k);
  }
  conv_stage(c, in, smp, px0 / c.R, sIn);
  __syncthreads();
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int li = lane & 15, lq = lane >> 4;
  const int m0 = (blockIdx.y * MW + wave % MW) * 16;
  if (m0 >= c.M) return;
  const T* __restrict__ wm = w + (int64_t)min(m0 + li, c.M - 1) * (FLIP ? 9 : c.K);
  int px[NC], po[NC];
#pragma unroll
  for (int j = 0; j < NC; ++j) {
    px[j] = ((wave / MW) * NC + j) * 16 + li;
    const int y = px[j] / c.R;
    po[j] = y * W + px[j] - y * c.R;
  }
  v4f acc[NC];
#pragma unroll
  for (int j = 0; j < NC; ++j) acc[j] = v4f{0.f, 0.f, 0.f, 0.f};
  T A[2][DU][E];
  int O[2][DU][E];
  auto load = [&](int k0, T (&x)[DU][E], int (&o)[DU][E]) {
    if (BF && !FLIP && k0 + DU * KS <= c.K) {  // a lane's 4 weights are consecutive: one load of 8 bytes
#pragma unroll
      for (int u = 0; u < DU; ++u) {
        const int k = k0 + u * KS + lq * E;
        memcpy(x[u], wm + k, E * sizeof(T));
#pragma unroll
        for (int e = 0; e < E; ++e) o[u][e] = sK[k + e].x;
      }
      return;
    }
#pragma unroll
    for (int u = 0; u < DU; ++u)
#pragma unroll
      for (int e = 0; e < E; ++e) {
        const int k = k0 + u * KS + lq * E + e;
        const int2 ko = sK[min(k, c.K - 1)];
        const T v = wm[ko.y];
        x[u][e] = k < c.K ? v : T(0);
        o[u][e] = k < c.K ? ko.x : -1;
      }
  };
  auto mma = [&](const T (&x)[DU][E], const int (&o)[DU][E], auto tail) {  // tail: some k past the end
#pragma unroll
    for (int u = 0; u < DU; ++u)
#pragma unroll
      for (int j = 0; j < NC; ++j) {
        T b[E];
#pragma unroll
        for (int e = 0; e < E; ++e) {
          if constexpr (decltype(tail)::value) {
            const T v = sIn[max(o[u][e], 0) + po[j]];
            b[e] = o[u][e] >= 0 ? v : T(0);
          } else {
            b[e] = sIn[o[u][e] + po[j]];
          }
        }
        if constexpr (BF) {
          v4s xa, yb;
#pragma unroll
          for (int e = 0; e < E; ++e) {
            xa[e] = (short)x[u][e];
            yb[e] = (short)b[e];
          }
          acc[j] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(xa, yb, acc[j], 0, 0, 0);
        } else {
          acc[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(x[u][0], b[0], acc[j], 0, 0, 0);
        }
      }
  };
  constexpr int KG = DU * KS;
  auto group = [&](int k0, int h) {
    if (k0 + KG <= c.K) mma(A[h], O[h], std::false_type{});
    else mma(A[h], O[h], std::true_type{});
  };
  load(0, A[0], O[0]);
  for (int k0 = 0; k0 < c.K; k0 += 2 * KG) {
    if (k0 + KG < c.K) load(k0 + KG, A[1], O[1]);
    group(k0, 0);
    if (k0 + KG >= c.K) break;
    if (k0 + 2 * KG < c.K) load(k0 + 2 * KG, A[0], O[0]);
    group(k0 + KG, 1);
  }
  // mm_store of channel m, pixel px0 + px[j] of sample smp
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int m = m0 + 4 * lq + r;
    if (m >= c.M) continue;
    const float bias = D.bias ? D.bias[m] : 0.f;
    const int64_t o0 = ((int64_t)smp * D.C + m) * R2 + px0;
#pragma unroll
    for (int j = 0; j < NC; ++j) {
      float v = acc[j][r];
      if (D.bias) v += bias;
      if (D.relu && v < 0.f) v = 0.f;
      if (D.mask && D.mask[o0 + px[j]] <= 0.f) v = 0.f;
      if (D.bf16) static_cast<uint16_t*>(D.p)[o0 + px[j]] = f32_to_bf16(v);
      else static_cast<float*>(D.p)[o0 + px[j]] = v;
    }
  }
}

// dW[co][ci t] = sum over pixels of dOut[co][px] in[ci][px + off(t)], and the
// bias gradient sum of dOut[co] as one more column block against ones.  A
// workgroup takes every gridDim.x-th strip, keeps all of dW in registers (the
// column blocks dealt to its 4 waves, NT per wave, MB row blocks each) and
// writes raw sums to part; k_conv_dw_reduce adds the workgroups in order.
// Split products over K = batch x pixels with k_mm read each element of both
// operands through the im2col switch (187 to 247 us per stage at batch 32) and
// summed the bias gradient over one workgroup per channel (up to 170 us).
template <int MB, int NT>
__global__ __launch_bounds__(256) void k_conv_dw(Conv c, const float* __restrict__ in, const float* __restrict__ dout,
                                                 int strips, float* __restrict__ part) {
  extern __shared__ __align__(16) char smem[];
  float* sIn = reinterpret_cast<float*>(smem);
  const int W = c.R + 2, R2 = c.R * c.R, CH = (c.P / c.R + 2) * W, lda = c.P + 4;
  float* sA = sIn + c.C * CH;  // output gradient of the strip: [co][pixel]
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int li = lane & 15, lq = lane >> 4;
  const int ncol = c.K + 1;  // column K: ones
  const int sh = 31 - __clz(c.R);
  constexpr int G = 4;  // groups of 4 pixels whose LDS reads go out together (P is a multiple of 16)
  int off[NT];  // tap offset of this lane's column; -1: ones, -2: none
#pragma unroll
  for (int j = 0; j < NT; ++j) {
    const int n = (wave + 4 * j) * 16 + li;
    const int ci = n / 9, t = n - 9 * ci, ty = t / 3;
    off[j] = n < c.K ? ci * CH + ty * W + t - 3 * ty : n == c.K ? -1 : -2;
  }
  v4f acc[MB][NT];
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j) acc[i][j] = v4f{0.f, 0.f, 0.f, 0.f};
  for (int st = blockIdx.x; st < strips; st += gridDim.x) {
    const int64_t n0 = (int64_t)st * c.P;
    const int smp = (int)(n0 / R2), px0 = (int)(n0 - (int64_t)smp * R2);
    __syncthreads();  // the previous strip has been read
    conv_stage(c, in, smp, px0 / c.R, sIn);
    for (int m = wave; m < 16 * MB; m += 4)
      for (int x = lane; x < c.P; x += 64)
        sA[m * lda + x] = m < c.M ? dout[((int64_t)smp * c.M + m) * R2 + px0 + x] : 0.f;
    __syncthreads();
    for (int g = 0; g < c.P; g += 4 * G) {
      float a[G][MB], b[G][NT];
#pragma unroll
      for (int u = 0; u < G; ++u) {
        const int x = g + 4 * u + lq, po = (x >> sh) * W + (x & (c.R - 1));
#pragma unroll
        for (int i = 0; i < MB; ++i) a[u][i] = sA[(16 * i + li) * lda + x];
#pragma unroll
        for (int j = 0; j < NT; ++j) b[u][j] = sIn[max(off[j], 0) + po];
      }
#pragma unroll
      for (int u = 0; u < G; ++u)
#pragma unroll
        for (int j = 0; j < NT; ++j) {
          const float v = off[j] >= 0 ? b[u][j] : off[j] == -1 ? 1.f : 0.f;
#pragma unroll
          for (int i = 0; i < MB; ++i) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[u][i], v, acc[i][j], 0, 0, 0);
        }
    }
  }
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int m = 16 * i + 4 * lq + r, n = (wave + 4 * j) * 16 + li;
        if (m < c.M && n < ncol) part[((int64_t)blockIdx.x * c.M + m) * ncol + n] = acc[i][j][r];
      }
}

// The sum over the workgroups' parts: 16 threads per entry, each every 16th
// part, their sums added in order (one thread per entry went through 256 parts
// in 15 us).
__global__ __launch_bounds__(256) void k_conv_dw_reduce(const float* __restrict__ part, int slices, int M, int K,
                                                        float* __restrict__ dw, float* __restrict__ db) {
  __shared__ float sv[16][17];
  const int x = threadIdx.x & 15, g = threadIdx.x >> 4;
  const int ncol = K + 1, n = M * ncol, e = blockIdx.x * 16 + x;
  float v = 0.f;
  if (e < n)
    for (int z0 = g; z0 < slices; z0 += 16 * 8) {  // 8 loads in flight, added in order
      float q[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) q[u] = z0 + 16 * u < slices ? part[(int64_t)(z0 + 16 * u) * n + e] : 0.f;
#pragma unroll
      for (int u = 0; u < 8; ++u) v += q[u];
    }
  sv[g][x] = v;
  __syncthreads();
  if (g || e >= n) return;
  v = 0.f;
#pragma unroll
  for (int u = 0; u < 16; ++u) v += sv[u][x];
  const int m = e / ncol, c = e - m * ncol;
  if (c < K) dw[m * K + c] = v;
  else db[m] = v;
}

// db[c] = sum over rows of dZ[r][c] (in order, 8 loads in flight)
__global__ __launch_bounds__(256) void k_colsum(const float* __restrict__ dZ, float* __restrict__ db, int m, int n) {
  const int c = blockIdx.x * 256 + threadIdx.x;
  if (c >= n) return;
  float s = 0.f;
  for (int r0 = 0; r0 < m; r0 += 8) {
    float q[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) q[u] = r0 + u < m ? dZ[(int64_t)(r0 + u) * n + c] : 0.f;
#pragma unroll
    for (int u = 0; u < 8; ++u) s += q[u];
  }
  db[c] = s;
}

// db[ch] = sum over samples and pixels of dZ[b][ch][px] (one block per
// channel, fixed-order tree reduction)
__global__ __launch_bounds__(256) void k_chansum(const float* __restrict__ dZ, float* __restrict__ db, int batch,
                                                 int C, int R2) {
  __shared__ float s[256];
  const int ch = blockIdx.x;
  float acc = 0.f;
  const int64_t n = (int64_t)batch * R2;
  for (int64_t e = threadIdx.x; e < n; e += 256) {
    const int64_t b = e / R2, px = e - b * R2;
    acc += dZ[(b * C + ch) * R2 + px];
  }
  s[threadIdx.x] = acc;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) s[threadIdx.x] += s[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) db[ch] = s[0];
}

// gradient of a nearest x2 upsampling, then of the ReLU before it: each input
// pixel sums its 2 x 2 block, zero where A (that layer's output) is not positive
__global__ __launch_bounds__(256) void k_down2_relu(const float* __restrict__ dUp, const float* __restrict__ A,
                                                    float* __restrict__ dIn, int64_t maps, int Ri) {
  const int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (e >= maps * Ri * Ri) return;
  const int64_t mp = e / ((int64_t)Ri * Ri);
  const int px = (int)(e - mp * Ri * Ri), Y = px / Ri, X = px % Ri;
  const int R = 2 * Ri;
  const float* u = dUp + mp * R * R + (int64_t)(2 * Y) * R + 2 * X;
  const float v = (u[0] + u[1]) + (u[R] + u[R + 1]);
  dIn[e] = A[e] <= 0.f ? 0.f : v;
}

// dY = 2 (Y - T) / count; per-block partial sums of (Y - T)^2 into part
__global__ __launch_bounds__(256) void k_mse(const float* __restrict__ Y, const float* __restrict__ T,
                                             float* __restrict__ dY, float* __restrict__ part, int64_t n) {
  __shared__ float s[256];
  float acc = 0.f;
  const float sc = 2.f / (float)n;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) {
    const float d = Y[i] - T[i];
    dY[i] = sc * d;
    acc += d * d;
  }
  s[threadIdx.x] = acc;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) s[threadIdx.x] += s[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) part[blockIdx.x] = s[0];
}

__global__ __launch_bounds__(256) void k_adam(float* __restrict__ p, const float* __restrict__ g, float* __restrict__ m,
                                              float* __restrict__ v, int64_t n, float lr, float b1, float b2,
                                              float c1, float c2, float eps) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  const float gi = g[i];
  const float mi = b1 * m[i] + (1.f - b1) * gi;
  const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
  m[i] = mi;
  v[i] = vi;
  p[i] -= lr * (mi / c1) / (sqrtf(vi / c2) + eps);
}

__global__ __launch_bounds__(256) void k_to_bf16(const float* __restrict__ a, uint16_t* __restrict__ b, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i < n) b[i] = f32_to_bf16(a[i]);
}

inline unsigned nblk(int64_t n, int b) { return (unsigned)((n + b - 1) / b); }

Opnd op_row(const void* p, int ld) { return Opnd{p, OP_ROW, ld, 0, 0, 0}; }
Opnd op_trans(const void* p, int ld) { return Opnd{p, OP_TRANS, ld, 0, 0, 0}; }

// k slices for an M x N x K product: enough workgroups to fill the chip
// when the output has few tiles, slices of at least 1024 deep (a multiple
// of TK), at most MAX_SPLIT
constexpr int MAX_SPLIT = 256;
inline int mm_splits(int M, int N, int K) {
  const int64_t tiles = (int64_t)nblk(N, TN) * nblk(M, TM);
  if (tiles >= 256 || K < 2048) return 1;
  int s = (int)std::min<int64_t>(512 / tiles, K / 1024);
  return std::max(1, std::min(s, MAX_SPLIT));
}

template <class T>
void mm(const Opnd& A, const Opnd& B, const Dst& D, int M, int N, int K, hipStream_t s, float* part = nullptr,
        int64_t part_cap = 0) {
  int splits = part ? mm_splits(M, N, K) : 1;
  if ((int64_t)splits * M * N > part_cap) splits = 1;
  const int kchunk = splits > 1 ? (((K + splits - 1) / splits + TK - 1) / TK) * TK : K;
  if (splits > 1) splits = (K + kchunk - 1) / kchunk;
  dim3 grid(nblk(N, TN), nblk(M, TM), splits);
  k_mm<T><<<grid, 256, 0, s>>>(A, B, D, M, N, K, kchunk, splits > 1 ? part : nullptr);
  MCHECK(hipGetLastError());
  if (splits > 1) {
    k_mm_reduce<<<nblk((int64_t)M * N, 256), 256, 0, s>>>(part, splits, D, M, N);
    MCHECK(hipGetLastError());
  }
}

// Dense product.  k slices (where a scratch array is given) until about 512
// waves are at work, each slice at least 128 deep, and never fewer than k_mm
// takes: a weight gradient over many rows is not one chain of sums (256 x 256
// weights in us, with the sum of the slices: 8192 rows 150 -> 33, 32768 593 ->
// 115; k_mm 190 and 228).
// With enough whole 64 x 64 tiles k_mm is faster, whose tiles read an operand
// entry once per 64 outputs instead of 16: from 512 tiles on (two workgroups
// per CU), or 256 where b is read across its rows, 64 bytes of each per step
// here (the input gradients).  256 x 256 weights, k_mm against k_dense, in us:
// forward 2048 rows 50 / 19, 4096 50 / 34, 8192 54 / 72 (BF16 45 / 65), 32768
// 123 / 252; input gradients 2048 rows 38 / 31, 4096 40 / 61, 8192 51 / 117.
// 256 x 4096 weights, forward: 512 rows 54 / 72, 4096 197 / 503.  Where a is
// read across its rows (the weight gradients) k_dense is faster throughout:
// 256 x 4096 weights, 4096 rows 694 / 188.
template <class T>
void dense(const T* a, int am, int ak, const T* b, int bk, int bn, const Dst& D, int M, int N, int K, hipStream_t s,
           float* part = nullptr, int64_t part_cap = 0) {
  if (ak == 1 && (int64_t)(M / TM) * (N / TN) >= (bn == 1 ? 512 : 256)) {
    mm<T>(op_row(a, am), bn == 1 ? op_row(b, bk) : op_trans(b, bn), D, M, N, K, s);
    return;
  }
  const int64_t waves = (int64_t)nblk(N, 16) * nblk(M, 16);
  int splits = part ? (int)std::max<int64_t>(mm_splits(M, N, K), std::min<int64_t>(512 / waves, K / 128)) : 1;
  splits = (int)std::max<int64_t>(1, std::min<int64_t>(splits, part_cap / ((int64_t)M * N)));
  const int kchunk = splits > 1 ? ((K + splits - 1) / splits + 15) / 16 * 16 : K;
  if (splits > 1) splits = (K + kchunk - 1) / kchunk;
  k_dense<T><<<dim3(nblk(N, 64), nblk(M, 16), splits), 256, 0, s>>>(a, am, ak, b, bk, bn, D, M, N, K, kchunk,
                                                                    splits > 1 ? part : nullptr);
  MCHECK(hipGetLastError());
  if (splits > 1) {
    k_mm_reduce<<<nblk((int64_t)M * N, 256), 256, 0, s>>>(part, splits, D, M, N);
    MCHECK(hipGetLastError());
  }
}

// A stage's strips: P = 16 NC 4 / MW pixels, whole rows of one sample, the
// largest NC of 4, 2, 1 that divides the map so and fits in 64 KB of LDS.
constexpr size_t CONV_LDS = 64 << 10;
inline int conv_mw(int M) { return M > 32 ? 4 : M > 16 ? 2 : 1; }
inline bool conv_strip(Conv& c, int px, size_t per_entry, size_t extra) {
  c.P = px;
  return px % c.R == 0 && c.R * c.R % px == 0 && (size_t)c.C * c.ch() * per_entry + extra <= CONV_LDS;
}

// The convolution product on staged strips; false if the map does not divide.
template <class T, int FLIP>
bool conv(const T* in, int C, int R, int up, const T* w, int M, int batch, const Dst& D, hipStream_t s) {
  const int mw = conv_mw(M);
  Conv c{C, R, up, 0, M, C * 9};
  int nc = 4;
  while (nc && !conv_strip(c, 16 * nc * (4 / mw), sizeof(T), (size_t)c.K * sizeof(int2))) nc /= 2;
  if (!nc) return false;
  const size_t lds = (size_t)c.K * sizeof(int2) + (size_t)C * c.ch() * sizeof(T);
  const dim3 g((unsigned)((int64_t)batch * R * R / c.P), nblk(M, 16 * mw));
#define MLP_CONV(WW, NN)                                       \
  if (mw == WW && nc == NN) {                                  \
    k_conv<T, FLIP, WW, NN><<<g, 256, lds, s>>>(c, in, w, D);  \
    MCHECK(hipGetLastError());                                 \
    return true;                                               \
  }
  MLP_CONV(4, 4) MLP_CONV(4, 2) MLP_CONV(4, 1) MLP_CONV(2, 4) MLP_CONV(2, 2) MLP_CONV(2, 1)
  MLP_CONV(1, 4) MLP_CONV(1, 2) MLP_CONV(1, 1)
#undef MLP_CONV
  return false;
}

// Weight and bias gradients of a convolution on staged strips; false if the
// map does not divide, or dW does not fit in registers or its slices in part.
inline bool conv_dw(const float* in, int C, int R, int up, const float* dout, int M, int batch, float* dw, float* db,
                    float* part, int64_t part_cap, hipStream_t s) {
  Conv c{C, R, up, 0, M, C * 9};
  // (three row blocks take the variant of four, whose last one is zero)
  const int mb = M > 32 && M <= 48 ? 4 : nblk(M, 16), nt = nblk(nblk(c.K + 1, 16), 4);
  if (R % 4 || mb > 4 || nt > 10) return false;
  // the largest strip with which 512 workgroups have work, else the smallest
  // that is there: 256 workgroups, one wave per SIMD, waited on every LDS read
  int best = 0;
  for (int px = 256; px >= 16; px /= 2) {
    if (!conv_strip(c, px, 4, (size_t)16 * mb * (px + 4) * 4)) continue;
    best = px;
    if ((int64_t)batch * R * R / px >= 512) break;
  }
  if (!best) return false;
  c.P = best;
  const size_t lds = ((size_t)C * c.ch() + (size_t)16 * mb * (c.P + 4)) * 4;
  const int64_t strips = (int64_t)batch * R * R / c.P, cells = (int64_t)M * (c.K + 1);
  const int slices = (int)std::min<int64_t>(std::min<int64_t>(strips, 512), part_cap / cells);
  if (slices < 1 || strips > (1 << 30)) return false;
#define MLP_DW(BB, NN)                                                                        \
  if (mb == BB && nt <= NN) {                                                                 \
    k_conv_dw<BB, NN><<<slices, 256, lds, s>>>(c, in, dout, (int)strips, part);               \
    MCHECK(hipGetLastError());                                                                \
    k_conv_dw_reduce<<<nblk(cells, 16), 256, 0, s>>>(part, slices, M, c.K, dw, db);          \
    MCHECK(hipGetLastError());                                                                \
    return true;                                                                              \
  }
  MLP_DW(1, 3) MLP_DW(1, 5) MLP_DW(1, 10) MLP_DW(2, 5) MLP_DW(2, 10) MLP_DW(4, 5) MLP_DW(4, 10)
#undef MLP_DW
  return false;
}

Dst dst_row(void* p, int ld, const float* bias, bool relu, bool bf16) {
  return Dst{p, 0, ld, 0, 0, bias, 0, relu ? 1 : 0, bf16 ? 1 : 0, nullptr};
}
Dst dst_chan(void* p, int C, int R, const float* bias, bool relu, bool bf16) {
  return Dst{p, 1, 0, C, R, bias, 1, relu ? 1 : 0, bf16 ? 1 : 0, nullptr};
}

struct Layer {
  bool conv = false;
  int nin = 0, nout = 0;             // dense: widths
  int cin = 0, cout = 0, R = 0, up = 0;  // convolution: channels, output side, upsampled input
  int64_t woff = 0, boff = 0;
  int64_t in_size() const { return conv ? (int64_t)cin * (R >> up) * (R >> up) : nin; }
  int64_t out_size() const { return conv ? (int64_t)cout * R * R : nout; }
};

}  // namespace

struct pecs_mlp {
  std::vector<Layer> layers;
  int nin = 0, nout = 0;
  int64_t np = 0;
  float *p = nullptr, *g = nullptr, *m = nullptr, *v = nullptr;  // parameters, gradients, Adam moments
  uint16_t* pb = nullptr;                                        // BF16 copy of the parameters (inference)
  bool pb_valid = false;
  int64_t t = 0;  // Adam step count
  // work buffers, sized for cap rows
  int cap = 0;
  std::vector<float*> act;  // act[l]: cap x size of layer l's input (act[L] = output)
  std::vector<float*> dact;
  std::vector<uint16_t*> actb;
  float* dup = nullptr;  // input gradient of an upsampling convolution at the upsampled size
  float* kpart = nullptr;  // split-k partial sums of the weight gradients
  int64_t kpart_cap = 0;
  float *target = nullptr, *part = nullptr;
  float* hpart = nullptr;  // pinned host copy of the loss's partial sums, from the first gradient call on
  hipStream_t s = nullptr;
  ~pecs_mlp() {
    if (s) (void)hipStreamSynchronize(s);
    auto f = [](void* q) {
      if (q) (void)hipFree(q);
    };
    f(p), f(g), f(m), f(v), f(pb), f(target), f(part), f(dup), f(kpart);
    for (float* a : act) f(a);
    for (float* a : dact) f(a);
    for (uint16_t* a : actb) f(a);
    if (hpart) (void)hipHostFree(hpart);
    if (s) (void)hipStreamDestroy(s);
  }
  int L() const { return (int)layers.size(); }
  int64_t size(int l) const { return l == 0 ? nin : layers[l - 1].out_size(); }
  void ensure(int rows) {
    if (rows <= cap) return;
    (void)hipStreamSynchronize(s);
    for (float* a : act) (void)hipFree(a);
    for (float* a : dact) (void)hipFree(a);
    for (uint16_t* a : actb) (void)hipFree(a);
    if (target) (void)hipFree(target);
    if (dup) (void)hipFree(dup);
    dup = nullptr;
    act.assign(L() + 1, nullptr);
    dact.assign(L() + 1, nullptr);
    actb.assign(L() + 1, nullptr);
    for (int l = 0; l <= L(); ++l) {
      MCHECK(hipMalloc(&act[l], (size_t)rows * size(l) * sizeof(float)));
      MCHECK(hipMalloc(&dact[l], (size_t)rows * size(l) * sizeof(float)));
      MCHECK(hipMalloc(&actb[l], (size_t)rows * size(l) * sizeof(uint16_t)));
    }
    int64_t dmax = 0;
    for (const Layer& y : layers)
      if (y.conv && y.up) dmax = std::max(dmax, (int64_t)y.cin * y.R * y.R);
    if (dmax) MCHECK(hipMalloc(&dup, (size_t)rows * dmax * sizeof(float)));
    MCHECK(hipMalloc(&target, (size_t)rows * nout * sizeof(float)));
    cap = rows;
  }
  // layer l (1-based) from act[l-1] (or actb) to act[l] (or actb)
  template <class T>
  void layer_fwd(int l, int rows, const T* in, void* out, const T* w, bool bf16out) {
    const Layer& y = layers[l - 1];
    const bool relu = l < L();
    const float* bias = p + y.boff;
    if (!y.conv) {
      dense<T>(in, y.nin, 1, w + y.woff, y.nout, 1, dst_row(out, y.nout, bias, relu, bf16out), rows, y.nout, y.nin, s);
    } else if (!conv<T, 0>(in, y.cin, y.R, y.up, w + y.woff, y.cout, rows,
                           dst_chan(out, y.cout, y.R, bias, relu, bf16out), s)) {
      const Opnd B{in, OP_IM2COL, 0, y.cin, y.R, y.up};
      mm<T>(op_row(w + y.woff, y.cin * 9), B, dst_chan(out, y.cout, y.R, bias, relu, bf16out), y.cout,
            rows * y.R * y.R, y.cin * 9, s);
    }
  }
  void forward(int rows) {
    for (int l = 1; l <= L(); ++l) layer_fwd<float>(l, rows, act[l - 1], act[l], p, false);
  }
  // loss gradient in dact[L], its partial sums to hpart (on the stream)
  void loss_grad(int rows) {
    const int64_t n = (int64_t)rows * nout;
    if (!hpart) MCHECK(hipHostMalloc((void**)&hpart, 256 * sizeof(float), hipHostMallocDefault));
    k_mse<<<256, 256, 0, s>>>(act[L()], target, dact[L()], part, n);
    MCHECK(hipGetLastError());
    MCHECK(hipMemcpyAsync(hpart, part, 256 * sizeof(float), hipMemcpyDeviceToHost, s));
  }
  float loss(int rows) const {  // once the stream has drained
    double acc = 0.0;
    for (int i = 0; i < 256; ++i) acc += hpart[i];
    return (float)(acc / (double)((int64_t)rows * nout));
  }
  void backward(int rows) {
    for (int l = L(); l >= 1; --l) {
      const Layer& y = layers[l - 1];
      // (every layer but the last ends in a ReLU: the input gradients are
      // masked by the layer's output below)
      const float* below = act[l - 1];
      if (!y.conv) {
        // dW = act[l-1]^T dact[l]; db = colsum(dact[l]); dact[l-1] = dact[l] W^T
        dense<float>(act[l - 1], 1, y.nin, dact[l], y.nout, 1, dst_row(g + y.woff, y.nout, nullptr, false, false), y.nin,
                     y.nout, rows, s, kpart, kpart_cap);
        k_colsum<<<nblk(y.nout, 256), 256, 0, s>>>(dact[l], g + y.boff, rows, y.nout);
        MCHECK(hipGetLastError());
        if (l > 1) {
          Dst d = dst_row(dact[l - 1], y.nin, nullptr, false, false);
          d.mask = below;
          dense<float>(dact[l], y.nout, 1, p + y.woff, 1, y.nout, d, rows, y.nin, y.nout, s, kpart, kpart_cap);
        }
      } else {
        const int R2 = y.R * y.R;
        // dW[co][ci t] = sum over (b, px) of dOut[b][co][px] im2col(in)[ci t][b px]
        if (!conv_dw(act[l - 1], y.cin, y.R, y.up, dact[l], y.cout, rows, g + y.woff, g + y.boff, kpart, kpart_cap, s)) {
          mm<float>(Opnd{dact[l], OP_CHAN, 0, y.cout, y.R, 0}, Opnd{act[l - 1], OP_IM2COL_T, 0, y.cin, y.R, y.up},
                    dst_row(g + y.woff, y.cin * 9, nullptr, false, false), y.cout, y.cin * 9, rows * R2, s, kpart,
                    kpart_cap);
          k_chansum<<<y.cout, 256, 0, s>>>(dact[l], g + y.boff, rows, y.cout, R2);
          MCHECK(hipGetLastError());
        }
        if (l > 1) {
          // d(upsampled input)[ci][b px] = sum over (co, t) of W[co][ci][t] dOut[b][co][px - offset(t)]
          Dst d = dst_chan(y.up ? dup : dact[l - 1], y.cin, y.R, nullptr, false, false);
          if (!y.up) d.mask = below;
          if (!conv<float, 1>(dact[l], y.cout, y.R, 0, p + y.woff, y.cin, rows, d, s))
            mm<float>(Opnd{p + y.woff, OP_WT, 0, y.cin, 0, 0}, Opnd{dact[l], OP_DCOL, 0, y.cout, y.R, 0}, d, y.cin,
                      rows * R2, y.cout * 9, s);
          if (y.up) {
            const int Ri = y.R / 2;
            const int64_t n = (int64_t)rows * y.cin * Ri * Ri;
            k_down2_relu<<<nblk(n, 256), 256, 0, s>>>(dup, below, dact[l - 1], (int64_t)rows * y.cin, Ri);
            MCHECK(hipGetLastError());
          }
        }
      }
    }
  }
};

namespace {

int mlp_fail(const std::exception& e) {
  g_mlp_error = e.what();
  return -1;
}

// parameter offsets, He-uniform weights for the ReLU layers, Glorot-uniform
// for the output layer, zero biases; device arrays and the stream
void mlp_init(pecs_mlp* net, unsigned seed) {
  int64_t off = 0;
  for (Layer& y : net->layers) {
    y.woff = off;
    off += y.conv ? (int64_t)y.cout * y.cin * 9 : (int64_t)y.nin * y.nout;
    y.boff = off;
    off += y.conv ? y.cout : y.nout;
  }
  net->np = off;
  int64_t wmax = 0;
  for (const Layer& y : net->layers) wmax = std::max(wmax, y.boff - y.woff + (y.conv ? y.cout : y.nout));
  net->kpart_cap = std::min<int64_t>((int64_t)MAX_SPLIT * wmax, (int64_t)1 << 24);  // larger products do not split
  MCHECK(hipMalloc(&net->kpart, net->kpart_cap * sizeof(float)));
  std::vector<float> h(off, 0.f);
  std::mt19937_64 rng(seed);
  for (int l = 1; l <= net->L(); ++l) {
    const Layer& y = net->layers[l - 1];
    const double fi = y.conv ? 9.0 * y.cin : y.nin, fo = y.conv ? 9.0 * y.cout : y.nout;
    const double a = l < net->L() ? std::sqrt(6.0 / fi) : std::sqrt(6.0 / (fi + fo));
    std::uniform_real_distribution<double> U(-a, a);
    for (int64_t i = y.woff; i < y.boff; ++i) h[i] = (float)U(rng);
  }
  MCHECK(hipStreamCreateWithFlags(&net->s, hipStreamNonBlocking));
  MCHECK(hipMalloc(&net->p, off * sizeof(float)));
  MCHECK(hipMalloc(&net->g, off * sizeof(float)));
  MCHECK(hipMalloc(&net->m, off * sizeof(float)));
  MCHECK(hipMalloc(&net->v, off * sizeof(float)));
  MCHECK(hipMalloc(&net->pb, off * sizeof(uint16_t)));
  MCHECK(hipMalloc(&net->part, 256 * sizeof(float)));
  MCHECK(hipMemcpy(net->p, h.data(), off * sizeof(float), hipMemcpyHostToDevice));
  MCHECK(hipMemset(net->m, 0, off * sizeof(float)));
  MCHECK(hipMemset(net->v, 0, off * sizeof(float)));
  MCHECK(hipMemset(net->g, 0, off * sizeof(float)));
}

}  // namespace

extern "C" {

const char* pecs_mlp_last_error(void) { return g_mlp_error.c_str(); }

int pecs_mlp_create(int nin, int nhidden, int nlayers, int nout, unsigned seed, pecs_mlp** out) {
  if (!out) return -1;
  *out = nullptr;
  try {
    if (nin < 1 || nhidden < 1 || nlayers < 1 || nlayers > 8 || nout < 1)
      throw std::runtime_error("pecs_mlp_create: sizes must be positive (1..8 hidden layers)");
    auto net = std::make_unique<pecs_mlp>();
    net->nin = nin;
    net->nout = nout;
    int prev = nin;
    for (int l = 0; l <= nlayers; ++l) {
      Layer y;
      y.nin = prev;
      y.nout = l < nlayers ? nhidden : nout;
      net->layers.push_back(y);
      prev = y.nout;
    }
    mlp_init(net.get(), seed);
    *out = net.release();
  } catch (const std::exception& e) {
    return mlp_fail(e);
  }
  return 0;
}

int pecs_mlp_create_decoder(int nin, int nhidden, int nlayers, int c0, int g0, int nconv, const int* conv_cout,
                            const int* conv_up, unsigned seed, pecs_mlp** out) {
  if (!out) return -1;
  *out = nullptr;
  try {
    if (nin < 1 || nhidden < 1 || nlayers < 1 || nlayers > 8 || c0 < 1 || g0 < 1 || nconv < 1 || nconv > 8 ||
        !conv_cout || !conv_up)
      throw std::runtime_error("pecs_mlp_create_decoder: sizes must be positive (1..8 hidden layers, 1..8 stages)");
    auto net = std::make_unique<pecs_mlp>();
    net->nin = nin;
    int prev = nin;
    for (int l = 0; l <= nlayers; ++l) {  // the last dense layer is the c0 x g0 x g0 feature map
      Layer y;
      y.nin = prev;
      y.nout = l < nlayers ? nhidden : c0 * g0 * g0;
      net->layers.push_back(y);
      prev = y.nout;
    }
    int cin = c0, side = g0;
    for (int j = 0; j < nconv; ++j) {
      if (conv_cout[j] < 1 || (conv_up[j] != 0 && conv_up[j] != 1))
        throw std::runtime_error("pecs_mlp_create_decoder: stage channels must be positive and up 0 or 1");
      Layer y;
      y.conv = true;
      y.cin = cin;
      y.cout = conv_cout[j];
      y.up = conv_up[j];
      y.R = side << y.up;
      if ((int64_t)y.R * y.R > (1 << 20)) throw std::runtime_error("pecs_mlp_create_decoder: maps above 1024 x 1024");
      net->layers.push_back(y);
      cin = y.cout;
      side = y.R;
    }
    net->nout = cin * side * side;
    mlp_init(net.get(), seed);
    *out = net.release();
  } catch (const std::exception& e) {
    return mlp_fail(e);
  }
  return 0;
}

int pecs_mlp_destroy(pecs_mlp* net) {
  if (!net) return -1;
  delete net;
  return 0;
}

int64_t pecs_mlp_num_params(pecs_mlp* net) { return net ? net->np : -1; }

int64_t pecs_mlp_num_outputs(pecs_mlp* net) { return net ? net->nout : -1; }

int pecs_mlp_get_params(pecs_mlp* net, float* params) {
  if (!net || !params) return -1;
  try {
    MCHECK(hipStreamSynchronize(net->s));
    MCHECK(hipMemcpy(params, net->p, net->np * sizeof(float), hipMemcpyDeviceToHost));
  } catch (const std::exception& e) {
    return mlp_fail(e);
  }
  return 0;
}

int pecs_mlp_set_params(pecs_mlp* net, const float* params) {
  if (!net || !params) return -1;
  try {
    MCHECK(hipStreamSynchronize(net->s));
    MCHECK(hipMemcpy(net->p, params, net->np * sizeof(float), hipMemcpyHostToDevice));
    net->pb_valid = false;
  } catch (const std::exception& e) {
    return mlp_fail(e);
  }
  return 0;
}

int pecs_mlp_gradients(pecs_mlp* net, const float* x, const float* y, int batch, float* grads, float* loss) {
  if (!net || !x || !y || batch < 1) return -1;
  try {
    net->ensure(batch);
    MCHECK(hipMemcpyAsync(net->act[0], x, (size_t)batch * net->nin * sizeof(float), hipMemcpyHostToDevice, net->s));
    MCHECK(hipMemcpyAsync(net->target, y, (size_t)batch * net->nout * sizeof(float), hipMemcpyHostToDevice, net->s));
    net->forward(batch);
    net->loss_grad(batch);
    net->backward(batch);
    if (grads) MCHECK(hipMemcpyAsync(grads, net->g, net->np * sizeof(float), hipMemcpyDeviceToHost, net->s));
    MCHECK(hipStreamSynchronize(net->s));
    if (loss) *loss = net->loss(batch);
  } catch (const std::exception& e) {
    return mlp_fail(e);
  }
  return 0;
}

int pecs_mlp_train_step(pecs_mlp* net, const float* x, const float* y, int batch, float lr, float* loss) {
  if (!net || !x || !y || batch < 1 || !(lr > 0)) return -1;
  try {
    float l = 0.f;
    if (pecs_mlp_gradients(net, x, y, batch, nullptr, &l) != 0) throw std::runtime_error(g_mlp_error);
    net->t += 1;
    const float b1 = 0.9f, b2 = 0.999f;
    const float c1 = 1.f - std::pow(b1, (float)net->t), c2 = 1.f - std::pow(b2, (float)net->t);
    k_adam<<<nblk(net->np, 256), 256, 0, net->s>>>(net->p, net->g, net->m, net->v, net->np, lr, b1, b2, c1, c2,
                                                   1e-8f);
    MCHECK(hipGetLastError());
    net->pb_valid = false;
    if (loss) *loss = l;
  } catch (const std::exception& e) {
    return mlp_fail(e);
  }
  return 0;
}

int pecs_mlp_predict(pecs_mlp* net, const float* x, int batch, float* y, int bf16) {
  if (!net || !x || !y || batch < 1) return -1;
  try {
    net->ensure(batch);
    MCHECK(hipMemcpyAsync(net->act[0], x, (size_t)batch * net->nin * sizeof(float), hipMemcpyHostToDevice, net->s));
    const int L = net->L();
    if (!bf16) {
      net->forward(batch);
    } else {
      if (!net->pb_valid) {
        k_to_bf16<<<nblk(net->np, 256), 256, 0, net->s>>>(net->p, net->pb, net->np);
        MCHECK(hipGetLastError());
        net->pb_valid = true;
      }
      const int64_t n0 = (int64_t)batch * net->nin;
      k_to_bf16<<<nblk(n0, 256), 256, 0, net->s>>>(net->act[0], net->actb[0], n0);
      MCHECK(hipGetLastError());
      // BF16 weights and activations, FP32 accumulation and biases; hidden
      // outputs rounded to BF16, the last layer's output kept in FP32
      for (int l = 1; l <= L; ++l) {
        if (l < L) net->layer_fwd<uint16_t>(l, batch, net->actb[l - 1], net->actb[l], net->pb, true);
        else net->layer_fwd<uint16_t>(l, batch, net->actb[l - 1], net->act[l], net->pb, false);
      }
    }
    MCHECK(hipMemcpyAsync(y, net->act[L], (size_t)batch * net->nout * sizeof(float), hipMemcpyDeviceToHost, net->s));
    MCHECK(hipStreamSynchronize(net->s));
  } catch (const std::exception& e) {
    return mlp_fail(e);
  }
  return 0;
}

}  // extern "C"

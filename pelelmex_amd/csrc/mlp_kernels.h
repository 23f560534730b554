// Surrogate MLP kernels for gfx950: BF16 operands on the matrix cores (v_mfma_f32_16x16x32_bf16),
// FP32 accumulation, fused bias / GELU epilogues, and the elementwise kernels of training
// (GELU backward, bias gradients, MSE loss, Adam). No counterpart in the reference: the learned
// dt_react map is an addition in front of the BDF (cells it cannot vouch for go to the BDF).
//
// Layouts: activations are row-major [rows x features] (features fastest), weights row-major
// [in x out]. The GEMM takes element strides for both operands, so the forward product
// (X W), the data gradient (dZ W^T) and the weight gradient (X^T dZ) all use the one kernel.
#ifndef PR_MLP_KERNELS_H
#define PR_MLP_KERNELS_H
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace prk {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

enum { EPI_NONE = 0, EPI_GELU = 1 };

struct GemmParams {
  int M, N, K;
  const __bf16* A;  // element (m, k) at A[m * sam + k * sak]
  long sam, sak;
  const __bf16* B;  // element (k, n) at B[k * sbk + n * sbn]
  long sbk, sbn;
  const float* bias;  // [N] or null
  int epi;            // EPI_NONE / EPI_GELU
  float* C;           // fp32 result after the epilogue [M x ldc] or null
  long ldc;
  __bf16* Cb;         // bf16 copy of the result or null
  long ldcb;
  float* Z;           // pre-activation (bias added, before GELU) or null
  long ldz;
  int accumulate;     // C += result (fp32 only, no epilogue), for gradient accumulation
};

__device__ __forceinline__ float gelu_f(float z) { return 0.5f * z * (1.0f + erff(z * 0.70710678118654752f)); }

// d gelu / dz = Phi(z) + z phi(z)
__device__ __forceinline__ float gelu_grad_f(float z) {
  const float cdf = 0.5f * (1.0f + erff(z * 0.70710678118654752f));
  const float pdf = 0.39894228040143268f * expf(-0.5f * z * z);
  return cdf + z * pdf;
}

// Products with operands in any layout. A wave forms a 32 x 32 tile as 2 x 2 MFMA 16 x 16 x 32
// tiles, its operands going from memory straight into the MFMA registers: the matrices are small
// (they sit in L2) and a K step's loads are issued one step ahead, so staging through LDS would
// only add two barriers a step. MFMA lane layout: lane l supplies A row l % 16 and B column l % 16
// with k = 8 (l / 16) .. 8 (l / 16) + 7, and receives D rows 4 (l / 16) .. + 3 of column l % 16.
// How an operand is read (x: its row m or column n):
//   LD_K     k contiguous, 16-byte aligned rows: one 16-byte load per tile
//   LD_PAIR  x contiguous, 4-byte aligned, even extent: one 4-byte load per k gives rows 2 r and
//            2 r + 1, which go to the wave's two tiles (tile i holds rows 2 r + i)
//   LD_ROW   k contiguous at any alignment: one 16-byte load per tile, or where a row may begin between
//            4-byte words the words and both ends (load8_odd); the last k of a row that do not fill one
//            by single elements (nothing past the row is read)
//   LD_ANY   x contiguous: one 2-byte load per element, neighbouring lanes on neighbouring elements
// Blocks: KS == 1: 4 waves cover 64 x 64 (2 x 2), each over the whole K. KS > 1: KS waves share one
// 32 x 32 tile, wave w taking the K steps w, w + KS, ..; their partial tiles are added in wave order
// through LDS. The split is for products with a long K and a small result (weight gradients: K is
// the batch, 16 tiles of 64 x 64 for a 256 x 256 layer on 256 CUs). What bounds both is the latency
// of the loads, not the matrix cores. Products of a
// training step (batch 4096, 4 layers of 256), 14 in all: 2790 us with operands staged element by
// element through LDS and no split, 188 us now (a weight gradient 530 -> 16, a forward layer 36 ->
// 16, a data gradient 25 -> 9). Rows at any alignment by single elements were slower than through LDS
// on large products, where each 2-byte load of a wavefront touches 16 rows (through LDS / by elements /
// one unaligned 16-byte load / LD_ROW, us): 262144 x 256 x 23 (the features' layer over a 64^3 box) 162 / 197 /
// 126 / 137, 4096 x 4095 x 4097 2019 / 2732 / 1862 / 1216 and with B by rows too 1921 / 4474 / 3113 / 1611.
constexpr int GT_K = 32, G_PITCH = 40;
enum { LD_K = 0, LD_PAIR = 1, LD_ROW = 2, LD_ANY = 3 };
constexpr int kSplitWaves = 16;

// Eight elements from an address that may be off a 4-byte word by one element, where a 16-byte load is slow
// (4096^3 by rows: 920 us at even pitches, 3110 at an odd one, 1610 so): the whole words and the
// elements at both ends.
__device__ __forceinline__ bf16x8 load8_odd(const __bf16* q) {
  const bool off = (reinterpret_cast<uintptr_t>(q) & 2) != 0;
  uint32_t d[3], w[4];
  uint16_t e0, e6, e7;
  __builtin_memcpy(d, __builtin_assume_aligned(q + (off ? 1 : 0), 4), 12);
  __builtin_memcpy(&e0, q, 2);
  __builtin_memcpy(&e6, q + 6, 2);
  __builtin_memcpy(&e7, q + 7, 2);
  w[0] = off ? e0 | d[0] << 16 : d[0];
  w[1] = off ? d[0] >> 16 | d[1] << 16 : d[1];
  w[2] = off ? d[1] >> 16 | d[2] << 16 : d[2];
  w[3] = (off ? d[2] >> 16 : (uint32_t)e6) | (uint32_t)e7 << 16;
  bf16x8 f;
  __builtin_memcpy(&f, w, 16);
  return f;
}

// Fragments of the wave's two tiles from operand X (element (x, k) at p[x * sx + k * sk]), rows
// x0 .. x0 + 31, k0 .. k0 + 31. Rows past nx read row nx - 1 (their results are not stored), k past
// K is zero in both operands.
template <int LD>
__device__ __forceinline__ void load_frags(const __bf16* __restrict__ p, long sx, long sk, int x0, int nx, int k0,
                                           int K, int l, bf16x8 (&f)[2]) {
  const int r = l % 16, k = k0 + 8 * (l / 16);
  const __bf16 zero = (__bf16)0.0f;
  if constexpr (LD == LD_K) {  // K is a multiple of 8: a chunk of 8 is inside or outside
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int x = x0 + 16 * i + r;
      f[i] = *reinterpret_cast<const bf16x8*>(p + (long)(x < nx ? x : nx - 1) * sx + (k < K ? k : 0));
    }
    if (k >= K)
#pragma unroll
      for (int j = 0; j < 8; ++j) f[0][j] = f[1][j] = zero;
  } else if constexpr (LD == LD_PAIR) {
    typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
    const int x = x0 + 2 * r;
    const __bf16* q = p + (x < nx ? x : nx - 2);
    bf16x2 v[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = *reinterpret_cast<const bf16x2*>(q + (long)(k + j < K ? k + j : 0) * sk);
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      f[0][j] = k + j < K ? v[j][0] : zero;
      f[1][j] = k + j < K ? v[j][1] : zero;
    }
  } else if constexpr (LD == LD_ROW) {
    const __bf16* q[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int x = x0 + 16 * i + r;
      q[i] = p + (long)(x < nx ? x : nx - 1) * sx + k;
    }
    if (k + 8 <= K) {
      if (((sx | (long)(reinterpret_cast<uintptr_t>(p) >> 1)) & 1) == 0) {  // every row 4-byte aligned
#pragma unroll
        for (int i = 0; i < 2; ++i) __builtin_memcpy(&f[i], __builtin_assume_aligned(q[i], 4), sizeof(bf16x8));
      } else {
#pragma unroll
        for (int i = 0; i < 2; ++i) f[i] = load8_odd(q[i]);
      }
    } else {
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          f[i][j] = zero;
          if (k + j < K) f[i][j] = q[i][j];
        }
    }
  } else {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int x = x0 + 16 * i + r;
      const __bf16* q = p + (long)(x < nx ? x : nx - 1) * sx;
      __bf16 v[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) v[j] = q[(long)(k + j < K ? k + j : 0) * sk];
#pragma unroll
      for (int j = 0; j < 8; ++j) f[i][j] = k + j < K ? v[j] : zero;
    }
  }
}

// Row (or column) of the operand that tile i's row r holds.
template <int LD>
__device__ __forceinline__ int frag_row(int i, int r) {
  return LD == LD_PAIR ? 2 * r + i : 16 * i + r;
}

__device__ __forceinline__ void gemm_store(const GemmParams& P, int gm, int gn, float v) {
  if (gm >= P.M || gn >= P.N) return;
  if (P.accumulate) {
    P.C[(long)gm * P.ldc + gn] += v;
    return;
  }
  if (P.bias) v += P.bias[gn];
  if (P.Z) P.Z[(long)gm * P.ldz + gn] = v;
  if (P.epi == EPI_GELU) v = gelu_f(v);
  if (P.C) P.C[(long)gm * P.ldc + gn] = v;
  if (P.Cb) P.Cb[(long)gm * P.ldcb + gn] = (__bf16)v;
}

template <int LA, int LB, int KS>
__global__ void __launch_bounds__(KS == 1 ? 256 : 64 * KS) gemm_bf16_kernel(GemmParams P) {
  const int wave = threadIdx.x / 64, l = threadIdx.x % 64;
  const int m0 = KS == 1 ? blockIdx.y * 64 + (wave / 2) * 32 : blockIdx.y * 32;
  const int n0 = KS == 1 ? blockIdx.x * 64 + (wave % 2) * 32 : blockIdx.x * 32;
  if (KS == 1 && (m0 >= P.M || n0 >= P.N)) return;  // no barrier on this path
  f32x4 acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int step = GT_K * KS;
  int k0 = KS == 1 ? 0 : GT_K * wave;
  bf16x8 a[2], b[2];
  if (k0 < P.K) {
    load_frags<LA>(P.A, P.sam, P.sak, m0, P.M, k0, P.K, l, a);
    load_frags<LB>(P.B, P.sbn, P.sbk, n0, P.N, k0, P.K, l, b);
  }
  for (; k0 < P.K; k0 += step) {
    bf16x8 an[2], bn[2];  // the next step's operands (past the end: zeros, not used)
    load_frags<LA>(P.A, P.sam, P.sak, m0, P.M, k0 + step, P.K, l, an);
    load_frags<LB>(P.B, P.sbn, P.sbk, n0, P.N, k0 + step, P.K, l, bn);
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i], b[j], acc[i][j], 0, 0, 0);
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      a[i] = an[i];
      b[i] = bn[i];
    }
  }
  if constexpr (KS == 1) {
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          gemm_store(P, m0 + frag_row<LA>(i, 4 * (l / 16) + r), n0 + frag_row<LB>(j, l % 16), acc[i][j][r]);
  } else {
    __shared__ float part[KS][32 * 33];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          part[wave][frag_row<LA>(i, 4 * (l / 16) + r) * 33 + frag_row<LB>(j, l % 16)] = acc[i][j][r];
    __syncthreads();
    for (int e = threadIdx.x; e < 1024; e += 64 * KS) {
      const int m = e / 32, n = e % 32;
      float v = 0.f;
#pragma unroll
      for (int w = 0; w < KS; ++w) v += part[w][m * 33 + n];
      gemm_store(P, m0 + m, n0 + n, v);
    }
  }
}

// Forward product of a hidden layer on the inference path: A [M x K] row-major (k fastest, lda =
// K), Bt = W^T [N x K] row-major (k fastest), K % 32 == 0, N % 128 == 0. Block tile 128 x 128,
// 256 threads = 4 waves of 64 x 64 (4 x 4 MFMA 16 x 16 x 32 tiles); operand tiles move as 16-byte
// vectors into double-buffered LDS (pitch 40 bf16), the next K step's loads in flight while the
// current one multiplies. Per output element the K steps and the MFMA are those of
// gemm_bf16_kernel, so the two give the same bits. Epilogue: bias, GELU (epi), bf16 store.
constexpr int FT_M = 128, FT_N = 128;

__global__ void __launch_bounds__(256) gemm_bf16_fwd_kernel(int M, int N, int K, const __bf16* __restrict__ A,
                                                            const __bf16* __restrict__ Bt,
                                                            const float* __restrict__ bias, int epi,
                                                            __bf16* __restrict__ Cb, long ldcb) {
  __shared__ __align__(16) __bf16 As[2][FT_M * G_PITCH];
  __shared__ __align__(16) __bf16 Bs[2][FT_N * G_PITCH];
  const int t = threadIdx.x;
  const int wave = t / 64, l = t % 64;
  const int m0 = blockIdx.y * FT_M, n0 = blockIdx.x * FT_N;
  const int wm = (wave / 2) * 64, wn = (wave % 2) * 64;
  // staging: 512 16-byte chunks per operand tile (128 rows x 4 chunks of 8 k); thread t moves
  // chunks t and t + 256 of each operand: row (c / 4), k offset 8 (c % 4)
  int arow[2], brow[2], kc[2];
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    const int c = t + 256 * u;
    const int r = c / 4;
    kc[u] = 8 * (c % 4);
    const int gm = m0 + r;
    arow[u] = gm < M ? gm : M - 1;  // rows past M read a valid row; their results are not stored
    brow[u] = n0 + r;
  }
  bf16x8 ra[2], rb[2];
  auto gload = [&](int k0) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      ra[u] = *reinterpret_cast<const bf16x8*>(A + (long)arow[u] * K + k0 + kc[u]);
      rb[u] = *reinterpret_cast<const bf16x8*>(Bt + (long)brow[u] * K + k0 + kc[u]);
    }
  };
  auto sstore = [&](int buf) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int r = (t + 256 * u) / 4;
      *reinterpret_cast<bf16x8*>(&As[buf][r * G_PITCH + kc[u]]) = ra[u];
      *reinterpret_cast<bf16x8*>(&Bs[buf][r * G_PITCH + kc[u]]) = rb[u];
    }
  };
  f32x4 acc[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  gload(0);
  sstore(0);
  __syncthreads();
  int buf = 0;
  for (int k0 = 0; k0 < K; k0 += GT_K) {
    const bool more = k0 + GT_K < K;
    if (more) gload(k0 + GT_K);
    bf16x8 a[4], b[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) a[i] = *reinterpret_cast<const bf16x8*>(&As[buf][(wm + 16 * i + l % 16) * G_PITCH + 8 * (l / 16)]);
#pragma unroll
    for (int j = 0; j < 4; ++j) b[j] = *reinterpret_cast<const bf16x8*>(&Bs[buf][(wn + 16 * j + l % 16) * G_PITCH + 8 * (l / 16)]);
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i], b[j], acc[i][j], 0, 0, 0);
    if (more) sstore(buf ^ 1);  // the other buffer: its last readers passed the previous barrier
    __syncthreads();
    buf ^= 1;
  }
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int gn = n0 + wn + 16 * j + l % 16;
    const float bj = bias ? bias[gn] : 0.f;
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int gm = m0 + wm + 16 * i + 4 * (l / 16) + r;
        if (gm >= M) continue;
        float v = acc[i][j][r];
        if (bias) v += bj;
        if (epi == EPI_GELU) v = gelu_f(v);
        Cb[(long)gm * ldcb + gn] = (__bf16)v;
      }
  }
}

// dZ = dA * gelu'(Z) (elementwise over rows x cols, row pitches given), as bf16 for the next
// products, optionally also fp32.
__global__ void gelu_bwd_kernel(long rows, int cols, const float* dA, long lda, const float* Z, long ldz,
                                __bf16* dZb, long ldb, float* dZ, long ldd) {
  const long e = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= rows * cols) return;
  const long r = e / cols;
  const int c = (int)(e % cols);
  const float g = dA[r * lda + c] * gelu_grad_f(Z[r * ldz + c]);
  dZb[r * ldb + c] = (__bf16)g;
  if (dZ) dZ[r * ldd + c] = g;
}

// db[c] = sum over rows of d[r, c]: four partial sums of the rows r, r + 4, .., each in row order (the
// first Adam step divides a bias gradient by its own magnitude, so its rounding is part of the
// result), then (0 + 1) + (2 + 3). 16 columns per block; 512 threads stage 512 rows in LDS, the next
// tile's loads in flight while one wavefront adds. What bounds it is the latency of those loads on a
// few CUs (two smaller tiles in flight 18 us): 4096 rows of 256 columns 240 us with the adding threads
// reading memory themselves (64 columns per block), 16 us now (9 us with a tree over 64 partial sums, whose rounding shifted the
// first steps of biases with gradients near Adam's epsilon).
constexpr int kSumCols = 16, kSumRows = 512;
__global__ void __launch_bounds__(512) col_sum_kernel(long rows, int cols, const float* d, long ld, float* out,
                                                      int accumulate) {
  __shared__ float tile[kSumRows * kSumCols];
  __shared__ float part[4][kSumCols];
  const int t = threadIdx.x, cl = t % kSumCols;
  const int c = blockIdx.x * kSumCols + cl;
  constexpr int NL = kSumCols;  // rows a thread stages: t / 16 + 32 j
  float v[NL];
  auto load = [&](long r0) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < NL; ++j) {
      const long r = r0 + t / kSumCols + (long)(kSumRows / NL) * j;
      v[j] = (c < cols && r < rows) ? d[r * ld + c] : 0.f;
    }
  };
  const int rg = t / kSumCols;  // partial sum of the adding threads (t < 64)
  float s = 0.f;
  load(0);
  for (long r0 = 0; r0 < rows; r0 += kSumRows) {
#pragma unroll
    for (int j = 0; j < NL; ++j) tile[t + kSumRows * j] = v[j];
    __syncthreads();
    if (r0 + kSumRows < rows) load(r0 + kSumRows);
    if (t < 4 * kSumCols) {
      const int m = (int)(rows - r0 < kSumRows ? rows - r0 : kSumRows);
      if (m == kSumRows) {
#pragma unroll 32
        for (int i = 0; i < kSumRows / 4; ++i) s += tile[(4 * i + rg) * kSumCols + cl];
      } else {
        for (int r = rg; r < m; r += 4) s += tile[r * kSumCols + cl];
      }
    }
    __syncthreads();
  }
  if (t < 4 * kSumCols) part[rg][cl] = s;
  __syncthreads();
  if (t < kSumCols && c < cols) {
    const float w = (part[0][t] + part[1][t]) + (part[2][t] + part[3][t]);
    out[c] = accumulate ? out[c] + w : w;
  }
}

// Mean-squared error over the first `cols` outputs: dY = 2 (Y - T) / (rows cols) (fp32, row
// pitch ldy) and the loss summed into *loss (one atomic per block).
__global__ void __launch_bounds__(256) mse_kernel(long rows, int cols, const float* Y, long ldy, const float* T,
                                                  long ldt, float* dY, float* loss) {
  __shared__ float red[256];
  const long e = (long)blockIdx.x * blockDim.x + threadIdx.x;
  float l = 0.f;
  if (e < rows * cols) {
    const long r = e / cols;
    const int c = (int)(e % cols);
    const float d = Y[r * ldy + c] - T[r * ldt + c];
    dY[r * ldy + c] = 2.0f * d / (float)(rows * cols);
    l = d * d / (float)(rows * cols);
  }
  red[threadIdx.x] = l;
  __syncthreads();
  for (int s = 128; s > 0; s >>= 1) {
    if (threadIdx.x < s) red[threadIdx.x] += red[threadIdx.x + s];
    __syncthreads();
  }
  if (threadIdx.x == 0) atomicAdd(loss, red[0]);
}

// Adam (Kingma & Ba 2015) on fp32 master parameters, with the bf16 copy the products read.
__global__ void adam_kernel(long n, float* p, const float* g, float* m, float* v, __bf16* pb, float lr, float b1,
                            float b2, float eps, float bc1, float bc2) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const float gi = g[i];
  const float mi = b1 * m[i] + (1.0f - b1) * gi;
  const float vi = b2 * v[i] + (1.0f - b2) * gi * gi;
  m[i] = mi;
  v[i] = vi;
  const float pi = p[i] - lr * (mi / bc1) / (sqrtf(vi / bc2) + eps);
  p[i] = pi;
  if (pb) pb[i] = (__bf16)pi;
}

__global__ void f32_to_bf16_kernel(long n, const float* a, __bf16* b) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) b[i] = (__bf16)a[i];
}

}  // namespace prk
#endif

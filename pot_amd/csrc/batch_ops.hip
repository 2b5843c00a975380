// Batched dense operations of the ot.batch API that are not Sinkhorn sweeps:
//
// * pairwise_kernel: the Minkowski and KL cost matrices of
//   ot.batch.dist_lp_batch (ot/batch/_linear.py:20-51) and dist_kl_batch
//   (:88-120), one 64 x 64 output tile per workgroup with the two point
//   tiles staged through LDS (the squared Euclidean cost lives in dist.hip);
// * gemm_batched_kernel: C_b = alpha op(A_b) op(B_b) + beta C_b with
//   arbitrary element strides, fp32 / fp64 accumulation in the input dtype.
//   It carries the Gromov-Wasserstein tensor product (hC1 T hC2^T per
//   feature channel, ot/batch/_quadratic.py:535-572, whose channel-last
//   layout is read in place through the strides) and the backward pass of
//   the squared Euclidean cost.
//
// Both are small next to the Sinkhorn sweeps (they run once per solve or
// once per outer Gromov step): pairwise_kernel has 256 threads with 4 x 4
// outputs each, gemm_batched_kernel a short chain on the matrix cores.
#include <algorithm>

#include "../../include/pot_amd.h"
#include "host.h"
#include "internal.h"

namespace potamd {

namespace {

constexpr int kTile = 64;
constexpr int kChunk = 16;

template <typename T>
__device__ inline T abs_pow(T x, T p) {
  x = x < (T)0 ? -x : x;
  if (p == (T)2) return x * x;
  if (p == (T)1) return x;
  return x == (T)0 ? (T)0 : (T)pow(x, p);
}

// metric 0: (sum_d |x - y|^p)^(q / p); 1: sum_d y log(y + eps) - y log(x + eps);
// 2: sum_d y log(y + eps) - y x (x holds logits).
template <typename T, int METRIC>
__global__ __launch_bounds__(256) void pairwise_kernel(const T* __restrict__ X,
                                                       const T* __restrict__ Y, int B, int n,
                                                       int m, int d, T p, T q, T eps,
                                                       T* __restrict__ M) {
  __shared__ T xs[kChunk][kTile + 1];
  __shared__ T ys[kChunk][kTile + 1];
  __shared__ T yl[kChunk][kTile + 1];  // y log(y + eps) (KL only)
  const int i0 = blockIdx.y * kTile, j0 = blockIdx.x * kTile;
  const int tx = threadIdx.x % 16, ty = threadIdx.x / 16;
  for (int b = blockIdx.z; b < B; b += gridDim.z) {
    const T* Xb = X + (int64_t)b * n * d;
    const T* Yb = Y + (int64_t)b * m * d;
    T acc[4][4] = {}, ent[4] = {};
    for (int k0 = 0; k0 < d; k0 += kChunk) {
      for (int e = threadIdx.x; e < kChunk * kTile; e += 256) {
        const int r = e / kChunk, k = e % kChunk;
        const int i = i0 + r, j = j0 + r, kk = k0 + k;
        T xv = (i < n && kk < d) ? Xb[(int64_t)i * d + kk] : (T)0;
        T yv = (j < m && kk < d) ? Yb[(int64_t)j * d + kk] : (T)0;
        if (METRIC == 1) xv = (T)log(xv + eps);
        xs[k][r] = xv;
        ys[k][r] = yv;
        if (METRIC != 0) yl[k][r] = yv * (T)log(yv + eps);
      }
      __syncthreads();
      const int kn = min(kChunk, d - k0);
      for (int k = 0; k < kn; ++k) {
        T xv[4], yv[4];
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          xv[t] = xs[k][ty + 16 * t];
          yv[t] = ys[k][tx + 16 * t];
          if (METRIC != 0) ent[t] += yl[k][tx + 16 * t];
        }
#pragma unroll
        for (int r = 0; r < 4; ++r)
#pragma unroll
          for (int c = 0; c < 4; ++c) {
            if (METRIC == 0) {
              acc[r][c] += abs_pow(xv[r] - yv[c], p);
            } else {
              // rounded product, then the add, in the order of the entropy
              // sum: KL(y || x) of a row with itself is then exactly 0
#pragma clang fp contract(off)
              acc[r][c] = acc[r][c] + yv[c] * xv[r];
            }
          }
      }
      __syncthreads();
    }
    T* Mb = M + (int64_t)b * n * m;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int i = i0 + ty + 16 * r;
      if (i >= n) continue;
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const int j = j0 + tx + 16 * c;
        if (j >= m) continue;
        T val;
        if (METRIC == 0)
          val = (q == p) ? acc[r][c] : (T)pow(acc[r][c], q / p);
        else
          val = ent[c] - acc[r][c];
        Mb[(int64_t)i * m + j] = val;
      }
    }
  }
}

struct GemmBatchArgs {
  int B, M, N, K;
  const void* A;
  int64_t sA, rsA, csA;  // element (i, k) of op(A_b) at A + b sA + i rsA + k csA
  const void* Bm;
  int64_t sB, rsB, csB;  // element (k, j) of op(B_b) at B + b sB + k rsB + j csB
  void* C;
  int64_t sC, ldc;       // element (i, j) of C_b at C + b sC + i ldc + j
  double alpha, beta;
};

// One 16 x 16 x 4 step of the matrix core: a = A[lane % 16][lane / 16],
// b = B[lane / 16][lane % 16]; value i of c is column lane % 16 and row
// out_row(i) of the product.
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef double f64x4 __attribute__((ext_vector_type(4)));
template <typename T> struct Mma;
template <> struct Mma<float> {
  using Acc = f32x4;
  static __device__ __forceinline__ f32x4 step(float a, float b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ int out_row(int lane, int i) { return 4 * (lane / 16) + i; }
};
template <> struct Mma<double> {
  using Acc = f64x4;
  static __device__ __forceinline__ f64x4 step(double a, double b, f64x4 c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ int out_row(int lane, int i) { return lane / 16 + 4 * i; }
};

// A workgroup of four waves forms a TS x TS tile of C_b, KC of K at a time
// through LDS, the next chunk's loads issued before the products of this one.
// These products are small (K of 40 to a few hundred), so the time is their
// chain: launch, loads, products, store.  One chunk covers K <= 64 with the
// tile of 32, which also gives four times the workgroups of the tile of 64.
template <typename T, int TS, int KC>
__global__ __launch_bounds__(256) void gemm_batched_kernel(GemmBatchArgs g) {
  __shared__ T as[KC][TS + 1];
  __shared__ T bs[KC][TS + 1];
  constexpr int L = TS * KC / 256;  // elements a thread loads of each operand
  constexpr int SUB = TS / 32;      // 16 x 16 products a side of a wave's quarter
  const int i0 = blockIdx.y * TS, j0 = blockIdx.x * TS;
  const int tid = threadIdx.x, lane = tid % kWave, wave = tid / kWave;
  const int wi = wave / 2 * (TS / 2), wj = wave % 2 * (TS / 2);
  const T* A = static_cast<const T*>(g.A);
  const T* Bm = static_cast<const T*>(g.Bm);
  T* C = static_cast<T*>(g.C);
  // Thread-to-element maps that keep the loads coalesced: along k when k is
  // the contiguous index of the operand, along the row (column) otherwise.
  const bool a_k_fast = g.csA == 1;
  const bool b_j_fast = g.csB == 1;
  for (int b = blockIdx.z; b < g.B; b += gridDim.z) {
    const T* Ab = A + (int64_t)b * g.sA;
    const T* Bb = Bm + (int64_t)b * g.sB;
    T ra[L], rb[L];
    auto load = [&](int k0) {
#pragma unroll
      for (int e = 0; e < L; ++e) {
        const int q = tid + 256 * e;
        const int r = a_k_fast ? q / KC : q % TS, k = k0 + (a_k_fast ? q % KC : q / TS);
        const int i = i0 + r;
        ra[e] = (i < g.M && k < g.K) ? Ab[(int64_t)i * g.rsA + (int64_t)k * g.csA] : (T)0;
      }
#pragma unroll
      for (int e = 0; e < L; ++e) {
        const int q = tid + 256 * e;
        const int c = b_j_fast ? q % TS : q / KC, k = k0 + (b_j_fast ? q / TS : q % KC);
        const int j = j0 + c;
        rb[e] = (j < g.N && k < g.K) ? Bb[(int64_t)k * g.rsB + (int64_t)j * g.csB] : (T)0;
      }
    };
    typename Mma<T>::Acc acc[SUB][SUB] = {};
    load(0);
    for (int k0 = 0; k0 < g.K; k0 += KC) {
#pragma unroll
      for (int e = 0; e < L; ++e) {
        const int q = tid + 256 * e;
        as[a_k_fast ? q % KC : q / TS][a_k_fast ? q / KC : q % TS] = ra[e];
        bs[b_j_fast ? q / TS : q % KC][b_j_fast ? q % TS : q / KC] = rb[e];
      }
      __syncthreads();
      if (k0 + KC < g.K) load(k0 + KC);
      const int kn = min(KC, g.K - k0);
      for (int k = 0; k < kn; k += 4) {  // (rows past K are zero)
        T av[SUB], bv[SUB];
#pragma unroll
        for (int t = 0; t < SUB; ++t) {
          av[t] = as[k + lane / 16][wi + 16 * t + lane % 16];
          bv[t] = bs[k + lane / 16][wj + 16 * t + lane % 16];
        }
#pragma unroll
        for (int r = 0; r < SUB; ++r)
#pragma unroll
          for (int c = 0; c < SUB; ++c) acc[r][c] = Mma<T>::step(av[r], bv[c], acc[r][c]);
      }
      __syncthreads();
    }
    T* Cb = C + (int64_t)b * g.sC;
    const T alpha = (T)g.alpha, beta = (T)g.beta;
#pragma unroll
    for (int r = 0; r < SUB; ++r)
#pragma unroll
      for (int c = 0; c < SUB; ++c) {
        const int j = j0 + wj + 16 * c + lane % 16;
        if (j >= g.N) continue;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int i = i0 + wi + 16 * r + Mma<T>::out_row(lane, q);
          if (i >= g.M) continue;
          T* dst = Cb + (int64_t)i * g.ldc + j;
          // beta == 0 never reads C, so an uninitialised C stays harmless
          *dst = beta == (T)0 ? alpha * acc[r][c][q] : fma(alpha, acc[r][c][q], beta * *dst);
        }
      }
  }
}

dim3 tile_grid(int rows, int cols, int B, int tile = kTile) {
  return dim3((cols + tile - 1) / tile, (rows + tile - 1) / tile, B < 65535 ? B : 65535);
}

// The tile of 64 (half the loads an output) where its workgroups fill the chip,
// unless the whole product fits the tile of 32.  us with 64 / 32: 256 float64
// products of 64^3 8.3 / 11.7 (16 before, with vector instructions), 64 float32
// of 180 x 8 x 200 (192 tiles of 64) 12.7 / 9.6 (33), 8 float64 of 200^3 (128)
// 17 / 12 (41), 16 float64 of 48 x 40 x 48 6.4 / 3.7 (10), 4000 float32 of 20^3
// 28 / 19 (21).
template <typename T>
void launch_gemm(const GemmBatchArgs& g, hipStream_t s) {
  const int64_t wide = (int64_t)((g.M + 63) / 64) * ((g.N + 63) / 64) * g.B;
  if (wide >= 256 && std::max(g.M, g.N) > 32)
    hipLaunchKernelGGL((gemm_batched_kernel<T, 64, 32>), tile_grid(g.M, g.N, g.B, 64), dim3(256), 0,
                       s, g);
  else
    hipLaunchKernelGGL((gemm_batched_kernel<T, 32, 64>), tile_grid(g.M, g.N, g.B, 32), dim3(256), 0,
                       s, g);
}

}  // namespace

}  // namespace potamd

using namespace potamd;

extern "C" int potamd_pairwise_batch(int dtype, int metric, const void* X, const void* Y,
                                     int batch, int n, int m, int d, double p, double q,
                                     double eps, void* M, void* stream) {
  if ((dtype != POTAMD_F32 && dtype != POTAMD_F64) || metric < 0 || metric > 2 || !X || !Y ||
      !M || batch < 1 || n < 1 || m < 1 || d < 1)
    return POTAMD_EINVAL;
  if (metric == 0 && !(p > 0.0 && q > 0.0)) return POTAMD_EINVAL;
  if (metric != 0 && !(eps >= 0.0)) return POTAMD_EINVAL;
  hipStream_t s = static_cast<hipStream_t>(stream);
  const dim3 grid = tile_grid(n, m, batch);
#define POTAMD_PAIRWISE(T, MET)                                                               \
  hipLaunchKernelGGL((pairwise_kernel<T, MET>), grid, dim3(256), 0, s,                        \
                     static_cast<const T*>(X), static_cast<const T*>(Y), batch, n, m, d,      \
                     (T)p, (T)q, (T)eps, static_cast<T*>(M))
  if (dtype == POTAMD_F32) {
    if (metric == 0) POTAMD_PAIRWISE(float, 0);
    else if (metric == 1) POTAMD_PAIRWISE(float, 1);
    else POTAMD_PAIRWISE(float, 2);
  } else {
    if (metric == 0) POTAMD_PAIRWISE(double, 0);
    else if (metric == 1) POTAMD_PAIRWISE(double, 1);
    else POTAMD_PAIRWISE(double, 2);
  }
#undef POTAMD_PAIRWISE
  HIP_TRY(hipGetLastError());
  return 0;
}

extern "C" int potamd_gemm_batched(int dtype, int batch, int M, int N, int K, double alpha,
                                   const void* A, int64_t sA, int64_t rsA, int64_t csA,
                                   const void* B, int64_t sB, int64_t rsB, int64_t csB,
                                   double beta, void* C, int64_t sC, int64_t ldc, void* stream) {
  if ((dtype != POTAMD_F32 && dtype != POTAMD_F64) || !A || !B || !C || batch < 1 || M < 1 ||
      N < 1 || K < 1 || ldc < N)
    return POTAMD_EINVAL;
  GemmBatchArgs g{batch, M, N, K, A, sA, rsA, csA, B, sB, rsB, csB, C, sC, ldc, alpha, beta};
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (dtype == POTAMD_F32)
    launch_gemm<float>(g, s);
  else
    launch_gemm<double>(g, s);
  HIP_TRY(hipGetLastError());
  return 0;
}

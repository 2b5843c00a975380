// Transport plan, its cost and entropy terms from converged potentials.
//
// P_ij = exp(-M_ij / reg + u_i + v_j) (log domain, ot/bregman/_sinkhorn.py:915-918,
// ot/batch/_utils.py:286-290) or P_ij = u_i K_ij v_j (scaling domain,
// _sinkhorn.py:683-687, _utils.py:160).  Every element is formed in fp64 from
// the fp64 potentials and the input cost, then stored in the cost's dtype;
// the per-problem sums are fp64 with a fixed reduction order:
//   sums[0] = sum M * P                  (sinkhorn2 loss, value_linear)
//   sums[1] = sum P * log(P + 1e-16)     (-entropy_batch, _utils.py:4-22)
//   sums[2] = sum P * log(P / (a b) + 1e-16)  (KL value, _linear.py:342-345)
//   sums[3] = sum P
// A plan has the same bits whether sums are asked for or not.
// Bound: the plan alone reads the cost and writes P (16384^2 float32: 2.1 GB);
// the sums are bound by the fp64 exponential and logarithms, so a logarithm is
// taken only where its sum is asked for.
#include <algorithm>

#include "host.h"
#include "internal.h"

namespace potamd {

constexpr int kPlanThreads = 256;
constexpr int kPlanSums = 4;

// (aligned as its elements: rows of any width and stride move 16 bytes at a
// time; an element at a time, a 5000 x 4999 float32 plan took 82 us, 53 to 59
// now, of which the fp64 exponential is 5)
template <typename TM, int VEC>
struct PlanVec {
  TM x[VEC];
};

// A thread owns VEC adjacent columns, whose v stays in registers, and walks
// down the block's rows, four at a time in flight: 1 << A.tx column threads by
// 256 >> A.tx row threads.  (A row at a time over 256 column threads left 3 of
// 4 threads idle at 64 columns, read v anew for every row and waited for each
// load: 512 plans of 64^2 took 51 us, 16384^2 float32 1464 us.)
template <typename TM, int VEC, bool SUMS>
__global__ __launch_bounds__(kPlanThreads) void plan_kernel(PlanArgs A) {
  using V = PlanVec<TM, VEC>;
  const int p = blockIdx.y;
  const int n = A.n, m = A.m;
  const int TX = 1 << A.tx, TY = kPlanThreads >> A.tx;
  const int tx = threadIdx.x & (TX - 1), ty = threadIdx.x >> A.tx;
  const TM* Mp = static_cast<const TM*>(A.M) + (int64_t)p * A.bstride;
  const double* u = A.u + (int64_t)p * n;
  const double* v = A.v + (int64_t)p * m;
  TM* P = A.P ? static_cast<TM*>(A.P) + (int64_t)p * A.pstride : nullptr;
  TM* L = A.logP ? static_cast<TM*>(A.logP) + (int64_t)p * A.pstride : nullptr;
  const double inv_reg = A.kernel_given ? 0.0 : 1.0 / A.reg;
  const bool logd = A.domain == kLog, given = A.kernel_given;
  const bool ent = SUMS && A.which & 2, kl = SUMS && A.which & 4;
  double s_cost = 0, s_ent = 0, s_kl = 0, s_mass = 0;
  const int r0 = (blockIdx.x / A.csplit) * A.rpb, r1 = min(n, r0 + A.rpb);
  for (int jt = ((blockIdx.x % A.csplit) * TX + tx) * VEC; jt < m; jt += A.csplit * TX * VEC) {
    // The last vector ends with the row; the columns it shares with its
    // neighbour get the same values twice and count in the neighbour's sums.
    const int j0 = min(jt, m - VEC), skip = jt - j0;
    double vj[VEC], bj[VEC];
#pragma unroll
    for (int c = 0; c < VEC; ++c) {
      vj[c] = v[j0 + c];
      bj[c] = kl ? A.b[(int64_t)p * m + j0 + c] : 1.0;
    }
    constexpr int Q = 4;
    for (int i0 = r0 + ty; i0 < r1; i0 += Q * TY) {
      V x[Q];
      double ui[Q];
#pragma unroll
      for (int q = 0; q < Q; ++q) {
        const int i = min(i0 + q * TY, r1 - 1);
        x[q] = *reinterpret_cast<const V*>(Mp + (int64_t)i * A.ldm + j0);
        ui[q] = u[i];
      }
#pragma unroll
      for (int q = 0; q < Q; ++q) {
        const int i = i0 + q * TY;
        if (i >= r1) break;
        V out, lout;
        const double ai = kl ? A.a[(int64_t)p * n + i] : 1.0;
#pragma unroll
        for (int c = 0; c < VEC; ++c) {
          const double mij = (double)x[q].x[c];
          double pij, xij = 0.0;
          if (logd) {
            xij = (given ? mij : -mij * inv_reg) + ui[q] + vj[c];
            pij = exp(xij);
          } else {
            const double kij = given ? mij : exp(-mij * inv_reg);
            pij = ui[q] * kij * vj[c];
          }
          out.x[c] = (TM)pij;
          lout.x[c] = (TM)xij;
          if (SUMS && c >= skip) {
            s_cost += mij * pij;
            if (ent) s_ent += pij * log(pij + 1e-16);
            if (kl) s_kl += pij * log(pij / (ai * bj[c]) + 1e-16);
            s_mass += pij;
          }
        }
        if (P) *reinterpret_cast<V*>(P + (int64_t)i * m + j0) = out;
        if (L) *reinterpret_cast<V*>(L + (int64_t)i * m + j0) = lout;
      }
    }
  }
  if (!SUMS) return;
  __shared__ double red[kPlanSums][kPlanThreads / kWave];
  const double vals[kPlanSums] = {s_cost, s_ent, s_kl, s_mass};
#pragma unroll
  for (int q = 0; q < kPlanSums; ++q) {
    const double w = wave_sum_dpp_d(vals[q]);
    if ((threadIdx.x & (kWave - 1)) == 0) red[q][threadIdx.x / kWave] = w;
  }
  __syncthreads();
  if (threadIdx.x < kPlanSums) {
    double t = 0;
    for (int w = 0; w < kPlanThreads / kWave; ++w) t += red[threadIdx.x][w];
    A.partial[((int64_t)p * gridDim.x + blockIdx.x) * kPlanSums + threadIdx.x] = t;
  }
}

// Adds a problem's block partials: 64 strided sums for each of the four, then
// the sums of a wave in a fixed order.  (One thread over 2048 blocks, a load
// at a time, took 270 us.)
__global__ __launch_bounds__(kPlanThreads) void plan_sums_kernel(int nblk, const double* partial,
                                                                 double* sums) {
  const int p = blockIdx.x;
  const int lane = threadIdx.x & (kWave - 1), q = threadIdx.x / kWave;
  const double* src = partial + (int64_t)p * nblk * kPlanSums + q;
  double t = 0;
#pragma unroll 4
  for (int b = lane; b < nblk; b += kWave) t += src[(int64_t)b * kPlanSums];
  t = wave_sum_dpp_d(t);
  if (lane == 0) sums[(int64_t)p * kPlanSums + q] = t;
}

// Most blocks of a problem's plan (the partials of its sums).
int plan_blocks(int n) { return (n + 7) / 8 + 8; }

hipError_t launch_plan(int dtype, PlanArgs a, int B, double* sums, hipStream_t s) {
  const int wide = dtype == 0 ? 4 : 2;
  // A plan written over its cost takes an element at a time where rows do not
  // end with a vector: the last one would read columns that its neighbour's
  // thread may have written.
  const bool over = a.P == a.M || a.logP == a.M;
  const bool vec = a.m >= wide && !(over && a.m % wide != 0);
  const int v = vec ? wide : 1;
  a.tx = 3;
  while (a.tx < 8 && (v << a.tx) < a.m) ++a.tx;
  const int ty = kPlanThreads >> a.tx;
  const int chunks = (a.m + (v << a.tx) - 1) / (v << a.tx);
  // Rows of a block: 16 for each row thread, fewer while that leaves the chip
  // (256 CUs, 8 blocks each) without work; then the column chunks are split.
  int rows = 16 * ty;
  auto blocks = [&](int r) { return (a.n + r - 1) / r; };
  while (rows > 4 * ty && (int64_t)B * blocks(rows) * chunks < 2048) rows -= 4 * ty;
  rows = std::max(rows, 8);
  a.rpb = rows;
  const int nrow = blocks(rows);
  a.csplit = std::max(1, std::min(chunks, plan_blocks(a.n) / nrow));
  const int nblk = nrow * a.csplit;
  dim3 grid(nblk, B);
#define POTAMD_PLAN(TM, VEC)                                                              \
  if (sums)                                                                               \
    hipLaunchKernelGGL((plan_kernel<TM, VEC, true>), grid, dim3(kPlanThreads), 0, s, a);  \
  else                                                                                    \
    hipLaunchKernelGGL((plan_kernel<TM, VEC, false>), grid, dim3(kPlanThreads), 0, s, a);
  if (dtype == 0) {
    if (vec) {
      POTAMD_PLAN(float, 4)
    } else {
      POTAMD_PLAN(float, 1)
    }
  } else {
    if (vec) {
      POTAMD_PLAN(double, 2)
    } else {
      POTAMD_PLAN(double, 1)
    }
  }
#undef POTAMD_PLAN
  hipError_t e = hipGetLastError();
  if (e != hipSuccess || !sums) return e;
  hipLaunchKernelGGL(plan_sums_kernel, dim3(B), dim3(kPlanThreads), 0, s, nblk, a.partial, sums);
  return hipGetLastError();
}

}  // namespace potamd

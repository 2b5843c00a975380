// Kernel of the dense-cost Sinkhorn with the cost resident on the chip: the
// whole solve in one launch (or one launch per check interval, see `segment`).
//
// The row-sweep solver (dense.hip) reads the cost from memory once per
// iteration and needs three launches for it.  Where the problem (or the
// batch) fits the register files, that is launch and memory latency and
// little else: 2048^2 float64 took 37 us an iteration (17 us of sweep, 12 of
// merge, 4 of decision, the gaps), 100 x 120 took 12 us, for 1 us of
// arithmetic.  Here a problem is cut into R x C blocks, one workgroup each,
// and every thread keeps its ER x EC elements of
//     K_ij = 2^(M_ij s2 + Ur_i + Vr_j)
// in registers.  The log domain runs on K with plain scalings
//     f_i = a_i / sum_j K_ij g_j,   g_j = b_j / sum_i K_ij f_i,
// relative to the references (Ur, Vr), which are potentials of an earlier
// iterate: U = Ur + log2 f, V = Vr + log2 g.  So an iteration is two multiply-
// adds per element and no exponential.  K's rows sum to 1 at the reference; a
// scaling that leaves [2^-L, 2^L] becomes part of its reference and K is
// formed again from M (exponents in fp64), so nothing that counts underflows.
// A row whose sum leaves the representable range altogether is redone as an
// exact log-sum-exp, as are the first column and row updates.  The scaling
// domain (sinkhorn_knopp) has no references: K and the scalings are the
// caller's.
//
// Row sums meet in 16-lane DPP butterflies (a wave owns 4 row threads x 16
// column threads), column sums in lane swaps and one LDS step.  Blocks of one
// problem exchange their partial sums through memory: every value travels as
// 32-bit halves, each in an 8-byte word beside the number of the exchange, so
// a reader that sees the number has the value and no flag, fence or cache
// flush is needed (device-scope relaxed accesses bypass the caches that are
// not coherent).  Two slots alternate: a member can be at most one exchange
// ahead of the slowest.  The members add the parts in the same order, so they
// all hold the same sums and take the same decisions.
//
// Workgroups that wait for each other have to be resident together: the host
// launches at most what fits the GPU, several solves at a time only where they
// fit together, and every wait is bounded (then the solve is abandoned and
// repeated by dense.hip, as it is where a scaling is not finite or a column
// mass falls below the trusted range, whose outcome dense.hip reports).
//
// The stabilised solver (sinkhorn_stabilized) is the scaling domain on
// K = exp((alpha + beta - M) / reg) in fp64, kept in the cost's type, with
// alpha and beta as references that move as the reference's do: where a
// scaling exceeded tau, alpha += reg log u, beta += reg log v, u and v start
// again at 1 / dim.  Whether one did is known to all blocks an exchange later:
// the column sums that followed are then thrown away.
#pragma once

#include <type_traits>

#include "host.h"
#include "internal.h"

// (10 x 20: all of a CU's registers for K, 320 x 320 a workgroup, so that
// 5120^2 float32 fits the chip; the rest spills, 0.2 to 0.3 KB a thread.
// 5000 x 4999: 12.3 us an iteration in the scaling domain and 36 in the log
// domain, against 49 on the row sweep.)
#define POTAMD_TILES_F32(X) \
  X(4, 2, 4) X(4, 4, 4) X(8, 4, 8) X(4, 8, 8) X(8, 8, 8) X(8, 4, 16) X(8, 8, 16) X(8, 10, 20)
#define POTAMD_TILES_F64(X) X(4, 2, 4) X(4, 4, 4) X(8, 2, 8) X(8, 4, 8) X(4, 8, 8) X(8, 8, 8) X(8, 4, 16)

namespace potamd {
namespace {

// Longest wait, in ticks of the 100 MHz clock: 20 ms.  The members of an exchange
// are some microseconds apart (a member that forms K again tens), so a wait that
// lasts is for a workgroup that another process or a long kernel keeps off the GPU.
constexpr long long kWaitTicks = 2000000;
// Ctrl::counter of a solve that was given up: by its numbers, or by a wait.
constexpr unsigned kGivenUp = 1, kWaitedOut = 2;

typedef unsigned long long word_t;

// Cache policy of device-scope reads and writes (sc1).
constexpr int kAgent = 16;
typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
typedef __amdgpu_buffer_rsrc_t rsrc_t;
__device__ __forceinline__ rsrc_t slot_at(word_t* w, int words) {
  return __builtin_amdgcn_make_buffer_rsrc(w, 0, words * 8, 0x00027000);
}
__device__ __forceinline__ void value_put(rsrc_t r, int idx, float x, unsigned tag) {
  __builtin_amdgcn_raw_buffer_store_b64(u32x2{__float_as_uint(x), tag}, r, idx * 8, 0, kAgent);
}
__device__ __forceinline__ void value_put(rsrc_t r, int idx, double x, unsigned tag) {
  const word_t b = (word_t)__double_as_longlong(x);
  __builtin_amdgcn_raw_buffer_store_b128(u32x4{(unsigned)b, tag, (unsigned)(b >> 32), tag}, r,
                                         idx * 16, 0, kAgent);
}

// Sum or maximum over the 16 lanes of a DPP row, in every lane.
template <bool MAX>
__device__ __forceinline__ float op2(float x, float y) { return MAX ? fmaxf(x, y) : x + y; }
template <bool MAX>
__device__ __forceinline__ double op2(double x, double y) { return MAX ? fmax(x, y) : x + y; }
template <int CTRL> __device__ __forceinline__ float dpp(float x) { return dpp_f<CTRL>(x); }
template <int CTRL> __device__ __forceinline__ double dpp(double x) { return dpp_d<CTRL>(x); }
template <bool MAX, typename R>
__device__ __forceinline__ R row16(R x) {
  x = op2<MAX>(x, dpp<0xB1>(x));
  x = op2<MAX>(x, dpp<0x4E>(x));
  x = op2<MAX>(x, dpp<0x141>(x));
  return op2<MAX>(x, dpp<0x140>(x));
}

// a of lanes 0-31 (0-15, 32-47) with its partner lanes' a, b likewise in the
// other lanes.
template <bool MAX>
__device__ __forceinline__ float fold32(float a, float b) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false,
                                                  false);
  return op2<MAX>(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
template <bool MAX>
__device__ __forceinline__ float fold16(float a, float b) {
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false,
                                                  false);
  return op2<MAX>(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
template <bool MAX>
__device__ __forceinline__ double fold32(double a, double b) {
  const word_t x = (word_t)__double_as_longlong(a), y = (word_t)__double_as_longlong(b);
  const auto l = __builtin_amdgcn_permlane32_swap((unsigned)x, (unsigned)y, false, false);
  const auto h = __builtin_amdgcn_permlane32_swap((unsigned)(x >> 32), (unsigned)(y >> 32), false,
                                                  false);
  return op2<MAX>(__longlong_as_double((long long)(((word_t)h[0] << 32) | l[0])),
                  __longlong_as_double((long long)(((word_t)h[1] << 32) | l[1])));
}
template <bool MAX>
__device__ __forceinline__ double fold16(double a, double b) {
  const word_t x = (word_t)__double_as_longlong(a), y = (word_t)__double_as_longlong(b);
  const auto l = __builtin_amdgcn_permlane16_swap((unsigned)x, (unsigned)y, false, false);
  const auto h = __builtin_amdgcn_permlane16_swap((unsigned)(x >> 32), (unsigned)(y >> 32), false,
                                                  false);
  return op2<MAX>(__longlong_as_double((long long)(((word_t)h[0] << 32) | l[0])),
                  __longlong_as_double((long long)(((word_t)h[1] << 32) | l[1])));
}

// Lane E of each 16-lane row, in every lane of the row (row_newbcast).
template <int E, int N, typename R>
__device__ __forceinline__ void row_spread(R x, R* out) {
  if constexpr (E < N) {
    out[E] = dpp<0x150 + E>(x);
    row_spread<E + 1, N>(x, out);
  }
}

__device__ __forceinline__ float fma_r(float x, float y, float z) {
  return __builtin_fmaf(x, y, z);
}
__device__ __forceinline__ double fma_r(double x, double y, double z) {
  return __builtin_fma(x, y, z);
}

// 2^x of an fp64 exponent in the element type: the fraction is rounded once.
__device__ __forceinline__ double exp2_of(double x, double) { return exp2(x); }
__device__ __forceinline__ float exp2_of(double x, float) {
  x = x < -1000.0 ? -1000.0 : x;  // -inf; a NaN stays
  const double k = rint(x);
  return ldexpf(exp2_fast((float)(x - k)), (int)k);
}

// Scaling domain, log domain, stabilised (see above).
enum ResidentMode { kResScaling, kResLog, kResStab };

// (Two waves a SIMD: eight waves need that, and of the tiles of four, two
// workgroups of the largest then share a CU.  Without it the float64 log solve
// of 128 x 128 took 258 registers: 257 problems of 100^2 293 us, 236 with two.)
template <typename TM, typename R, int W, int ER, int EC, int MODE, bool BLK>
__global__ __launch_bounds__(64 * W, 2) void resident_kernel(ResidentArgs A) {
  constexpr bool LOG = MODE == kResLog, STAB = MODE == kResStab;
  constexpr int T = 64 * W, TR = 4 * W, RB = TR * ER, CB = 16 * EC;
  static_assert(ER <= 16 && EC % 4 == 0 && CB <= T, "tile");
  constexpr int kDrift = sizeof(R) == 4 ? 32 : 200;  // log2
  constexpr double kSafe = sizeof(R) == 4 ? 1.152921504606847e18 : 1e250;  // 2^60
  constexpr double kFloor = sizeof(R) == 4 ? 1e-36 : 1e-300;

  extern __shared__ double lds[];
  double* part = lds;              // W x CB column partials
  double* vr = part + W * CB;      // column references
  double* cmx = vr + CB;           // exact column pass: maxima
  double* ursh = cmx + CB;         // row references
  R* gsh = reinterpret_cast<R*>(ursh + RB);
  double* xs = ursh + RB + CB;     // exchanged values
  __shared__ double red[W];
  __shared__ int dead;    // a wait ended: 1 another workgroup gave up, 2 too long
  // Of the column update: 1 references move, 2 abandon.  Stabilised: a scaling
  // over tau, of columns 4 and 16 in turn (a wave may be a column update ahead
  // of one that reads the last one's), of rows 8.
  __shared__ int events;
  __shared__ int weird_rows;  // a row sum off the type's range

  const int tid = threadIdx.x, lane = tid & 63;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lc = lane & 15, lr = lane >> 4;
  const int n = A.n, m = A.m, GR = BLK ? A.R : 1, GC = BLK ? A.C : 1;
  const int p = BLK ? blockIdx.x / (GR * GC) : blockIdx.x, rem = BLK ? blockIdx.x % (GR * GC) : 0;
  const int I = BLK ? rem / GC : 0, J = BLK ? rem % GC : 0;
  const int row0 = I * A.rbs, nr = min(A.rbs, n - row0);
  const int col0 = J * A.cbs, nc = min(A.cbs, m - col0);
  const TM* Mp = static_cast<const TM*>(A.M) + (int64_t)p * A.bstride + (int64_t)row0 * A.ldm + col0;
  const bool row_first = A.row_first;
  const double s2 = A.s2;

  if (A.segment && A.ctrl->done) return;
  if (tid == 0) {
    dead = 0;
    events = 0;
    weird_rows = 0;
  }

  // Row owner: lane lc < ER holds row lc of its wave's ER rows per row thread.
  const int rl = wv * 4 + lr + TR * lc;
  const bool rown = lc < ER && rl < nr;
  const int64_t ri = (int64_t)p * n + row0 + rl;
  const double a_l = rown ? A.a[ri] : 0.0;
  // Column owner: thread t < nc.
  const bool cown = tid < nc;
  const int64_t ci = (int64_t)p * m + col0 + tid;
  const double b_t = cown ? A.b[ci] : 0.0;

  double f_l = 0.0, Ur_l = 0.0, g_t = 0.0, Vr_t = 0.0;
  const double unit = LOG && !A.resume ? kLog2e : 1.0;
  if (rown) Ur_l = A.u_in[ri] * unit;
  if (cown) Vr_t = A.v_in[ci] * unit;
  const double la_l = rown && LOG ? log2(a_l) : 0.0;

  unsigned tag_r = 0, tag_c = 0, tag_e = 0;
  word_t* const xrow = A.words + (int64_t)(p * GR + I) * 2 * A.row_slot;
  word_t* const xcol = A.words + A.col_base + (int64_t)(p * GC + J) * 2 * A.col_slot;
  word_t* const xerr = A.words + A.err_base;

  // Polls units tagged entries of BYTES each until all carry the tag: entry w
  // lies at byte at(w) of the slot, and take(w, entry) keeps a complete one.
  // Entries are read past the caches that are not coherent.  `pause`: 512
  // clocks first: the entries of members that left the last
  // exchange with this one are then there at the first read, which otherwise
  // comes back too early and costs a second one (2048^2 float64 8.0 -> 7.0 us
  // an iteration; single float words arrive sooner and do without).
  auto poll = [&](auto bytes, rsrc_t rsrc, int units, bool pause, unsigned tag, auto at, auto take) {
    constexpr int Q = ER == 10 ? 5 : 4;  // reads of a thread in flight
    using V = typename std::conditional<decltype(bytes)::value == 16, u32x4, u32x2>::type;
    if (A.wait_ticks < 0 && tag >= 3) {  // (as potamd_resident_wait_limit asked)
      dead = 2;
      return;
    }
    if (pause) __builtin_amdgcn_s_sleep(8);
    for (int w0 = tid; w0 < units; w0 += Q * T) {
      V v[Q];
      unsigned pend = 0;
#pragma unroll
      for (int q = 0; q < Q; ++q) pend |= (w0 + q * T < units ? 1u : 0u) << q;
      long long since = 0;
      for (int spin = 0; pend; ++spin) {
        asm volatile("" ::: "memory");  // read anew each time
#pragma unroll
        for (int q = 0; q < Q; ++q)
          if (pend >> q & 1) {
            if constexpr (sizeof(V) == 16)
              v[q] = __builtin_amdgcn_raw_buffer_load_b128(rsrc, at(w0 + q * T), 0, kAgent);
            else
              v[q] = __builtin_amdgcn_raw_buffer_load_b64(rsrc, at(w0 + q * T), 0, kAgent);
          }
#pragma unroll
        for (int q = 0; q < Q; ++q)
          if (pend >> q & 1 && take(w0 + q * T, v[q])) pend &= ~(1u << q);
        if (pend) {
          __builtin_amdgcn_s_sleep(1);
          if ((spin & 63) == 63) {
            const long long now = wall_clock64();
            if (since == 0) since = now;
            const bool told = dead || __hip_atomic_load(&A.ctrl->counter, __ATOMIC_RELAXED,
                                                        __HIP_MEMORY_SCOPE_AGENT);
            if (told || now - since > A.wait_ticks) {
              if (!dead) dead = told ? 1 : 2;
              break;
            }
          }
        }
      }
    }
  };
  using Bytes8 = std::integral_constant<int, 8>;
  using Bytes16 = std::integral_constant<int, 16>;
  auto as_double = [](u32x4 v) {
    return __longlong_as_double((long long)(((word_t)v[2] << 32) | v[0]));
  };
  // Reads N = G x L tagged values into LDS; value w, entry w % L of member
  // w / L, lands at (w % L) * GS + w / L.  A lane reads 16 bytes, two tagged
  // words (one double or two floats).
  auto gather = [&](auto* dst, word_t* src, int N, int L, int GS, unsigned tag) {
    using P = typename std::remove_pointer<decltype(dst)>::type;
    constexpr int PER = 2 / (sizeof(P) / 4);  // values a read
    const int units = (N + PER - 1) / PER;
    poll(Bytes16(), slot_at(src, units * 2), units, sizeof(P) == 8 || units > T, tag,
         [&](int w) { return w * 16; },
         [&](int u, u32x4 v) {
           const int w = u * PER;
           const bool second = sizeof(P) == 8 || w + 1 < N;
           if (v[1] != tag || (second && v[3] != tag)) return false;
           if constexpr (sizeof(P) == 8) {
             dst[(w % L) * GS + w / L] = as_double(v);
           } else {
             dst[(w % L) * GS + w / L] = __uint_as_float(v[0]);
             if (second) dst[((w + 1) % L) * GS + (w + 1) / L] = __uint_as_float(v[2]);
           }
           return true;
         });
  };
  // Sum or maximum of x over the G members of this block's row or column
  // group, for the owner of entry idx < L; every thread takes part.
  // (Stabilised: with one more entry, the member's flag; `raised` says whether
  // one of the members did.)
  bool raised = false;
  constexpr bool TWO = BLK && !STAB && ER * EC >= 64;  // (smaller blocks have fewer values)
  auto exchange = [&](auto x, bool own, int idx, int L, int G, int me, word_t* slots, int slot,
                      int room, unsigned& tag, auto maxop, bool flag) -> double {
    if (STAB) ++L;
    using P = decltype(x);
    constexpr bool MAX = decltype(maxop)::value;
    ++tag;
    word_t* base = slots + (int64_t)(tag & 1) * slot;
    if (own) value_put(slot_at(base, slot), me * L + idx, x, tag);
    if (STAB && tid == 0) value_put(slot_at(base, slot), me * L + L - 1, (P)(flag ? 1 : 0), tag);
    P* dst = reinterpret_cast<P*>(xs);
    const int GS = G | 1;
    if constexpr (TWO) if (G * L * (int)sizeof(P) > 64 * T) {
      // Many values: each member reads and adds a G-th of the entries and the
      // totals are exchanged again: two waits of a read or two a thread in
      // place of one of more than eight (all members read all G x L values).
      // 2800^2 float64 (22 members, 255 rows) 11.7 -> 8.1 us an iteration;
      // 5000 x 800 (20 members, 115 columns) 8.8 this way and 7.8 the other.
      const int S = (L + G - 1) / G, s0 = min(me * S, L), cnt = min(S, L - s0);
      constexpr int VB = 2 * sizeof(P);
      poll(std::integral_constant<int, VB>(), slot_at(base, slot), G * cnt, sizeof(P) == 8, tag,
           [&](int w) { return (w / cnt * L + s0 + w % cnt) * VB; },
           [&](int w, auto v) {
             bool all = v[1] == tag;
             if constexpr (VB == 16) all = all && v[3] == tag;
             if (!all) return false;
             if constexpr (VB == 16)
               dst[w % cnt * GS + w / cnt] = as_double(v);
             else
               dst[w % cnt * GS + w / cnt] = __uint_as_float(v[0]);
             return true;
           });
      __syncthreads();
      const rsrc_t totals = slot_at(base + slot - 2 * room, 2 * room);
      if (tid < cnt) {
        double s = (double)dst[tid * GS];
        for (int k = 1; k < G; ++k) s = op2<MAX>(s, (double)dst[tid * GS + k]);
        value_put(totals, s0 + tid, s, tag);
      }
      double* tot = xs + (S * GS * sizeof(P) + 7) / 8;
      poll(Bytes16(), totals, L, true, tag, [&](int w) { return w * 16; },
           [&](int w, u32x4 v) {
             if (v[1] != tag || v[3] != tag) return false;
             tot[w] = as_double(v);
             return true;
           });
      __syncthreads();
      return own ? tot[idx] : 0.0;
    }
    gather(dst, base, L * G, L, GS, tag);
    __syncthreads();
    if (STAB) raised = __any(lane < G && dst[(L - 1) * GS + lane] != (P)0);
    double s = 0.0;
    if (own) {
      s = (double)dst[idx * GS];
      for (int k = 1; k < G; ++k) s = op2<MAX>(s, (double)dst[idx * GS + k]);
    }
    return s;
  };
  using Sum = std::false_type;
  using Max = std::true_type;
  auto rows_of = [&](auto x, auto maxop, bool flag = false) -> double {  // row owners
    return exchange(x, rown, rl, nr, GC, J, xrow, A.row_slot, A.rbs + 1, tag_r, maxop, flag);
  };
  auto cols_of = [&](auto x, auto maxop, bool flag = false) -> double {  // column owners
    return exchange(x, cown, tid, nc, GR, I, xcol, A.col_slot, A.cbs + 1, tag_c, maxop, flag);
  };
  auto abandon = [&]() {
    if (tid == 0) {
      if (dead != 1) {  // (else the cause stands there)
        const unsigned why = dead == 2 ? kWaitedOut : kGivenUp;
        __hip_atomic_store(&A.ctrl->counter, why, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (A.host) A.host->counter = why;
      }
      if (A.segment) A.ctrl->done = 1;
    }
  };

  // Column reduction: EC per-thread values over the block's rows; the column
  // owner gets its column's.  One barrier.
  auto cols_reduce = [&](auto* acc, auto maxop) -> double {
    using P = typename std::remove_pointer<decltype(acc)>::type;
    constexpr bool MAX = decltype(maxop)::value;
#pragma unroll
    for (int q = 0; q < EC / 2; ++q) acc[q] = fold32<MAX>(acc[q], acc[q + EC / 2]);
#pragma unroll
    for (int q = 0; q < EC / 4; ++q) acc[q] = fold16<MAX>(acc[q], acc[q + EC / 4]);
    P* dst = reinterpret_cast<P*>(part) + wv * CB + lc + 16 * ((lr & 1) * (EC / 4) + (lr >> 1) * (EC / 2));
#pragma unroll
    for (int q = 0; q < EC / 4; ++q) dst[16 * q] = acc[q];
    __syncthreads();
    double s = MAX ? -__builtin_inf() : 0.0;
    if (tid < CB) {
      const P* src = reinterpret_cast<const P*>(part) + tid;
#pragma unroll
      for (int w = 0; w < W; ++w) s = op2<MAX>(s, (double)src[w * CB]);
    }
    return s;
  };

  R K[ER][EC];
  // Lane position that the compiler takes for a new value: the addresses and
  // masks built from it are formed where they are used, not kept in registers
  // over the iterations.
  auto here = [&](int x) {
    asm volatile("" : "+v"(x));
    return x;
  };
  // K at the references; a wave's rows only, so no barrier.
  auto build = [&]() {
    const int l = here(lane), c0 = l & 15, r0 = wv * 4 + (l >> 4);
    if (c0 < ER) ursh[r0 + TR * c0] = rown ? Ur_l : -__builtin_inf();
    __builtin_amdgcn_wave_barrier();
    const float s_hi = A.s_hi, s_lo = A.s_lo;
#pragma unroll
    for (int e = 0; e < ER; ++e) {
      const int r = r0 + TR * e;
      const double ur = ursh[r];
      const TM* row = Mp + (int64_t)min(r, nr - 1) * A.ldm;
#pragma unroll
      for (int k = 0; k < EC; ++k) K[e][k] = (R)row[min(c0 + 16 * k, nc - 1)];
      if constexpr (STAB) {
#pragma unroll
        for (int k = 0; k < EC; ++k)
          K[e][k] = (R)(TM)exp(((ur - (double)K[e][k]) + vr[c0 + 16 * k]) * A.inv_reg);
      } else if constexpr (LOG) {
#pragma unroll
        for (int k = 0; k < EC; ++k)
          K[e][k] = exp2_of(fma((double)K[e][k], s2, ur + vr[c0 + 16 * k]), R());
      } else if (!A.kernel_given) {
#pragma unroll
        for (int k = 0; k < EC; ++k) {
          if constexpr (sizeof(R) == 4)
            K[e][k] = exp2_fast(scaled_exponent(K[e][k], s_hi, s_lo, (R)0));
          else
            K[e][k] = exp2_of(K[e][k] * s2, R());
        }
      }
      if (r >= nr) {
#pragma unroll
        for (int k = 0; k < EC; ++k) K[e][k] = (R)0;
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    if (nc < CB) {
#pragma unroll
      for (int k = 0; k < EC; ++k) {
        const bool ok = c0 + 16 * k < nc;
#pragma unroll
        for (int e = 0; e < ER; ++e) K[e][k] = ok ? K[e][k] : (R)0;
      }
    }
  };
  // U = log a - LSE_j(M s2 + V) of the wave's rows, into Ur (less log a).
  // A row with weight and no finite potential makes K, and so every column
  // sum, no number.
  auto exact_rows = [&]() {
    const int l = here(lane), c0 = l & 15, r0 = wv * 4 + (l >> 4);
    auto exponents = [&](int k, auto use) {
      const int c = c0 + 16 * k;
      const double vk = vr[c] + log2((double)gsh[c]);
#pragma unroll
      for (int e = 0; e < ER; ++e)
        use(e, fma((double)Mp[(int64_t)min(r0 + TR * e, nr - 1) * A.ldm + min(c, nc - 1)], s2, vk));
    };
    double mx[ER], sm[ER];
#pragma unroll
    for (int e = 0; e < ER; ++e) mx[e] = -__builtin_inf();
#pragma unroll 1
    for (int k = 0; k < EC; ++k) exponents(k, [&](int e, double x) { mx[e] = fmax(mx[e], x); });
    double mine = 0.0;
#pragma unroll
    for (int e = 0; e < ER; ++e) {
      mx[e] = row16<true>(mx[e]);
      mine = lc == e ? mx[e] : mine;
    }
    if (GC > 1) {
      mine = rows_of(mine, Max());
      __syncthreads();
    }
    if (!(mine > -1e300)) mine = 0.0;  // a row of nothing
    row_spread<0, ER>(mine, mx);
#pragma unroll
    for (int e = 0; e < ER; ++e) sm[e] = 0.0;
#pragma unroll 1
    for (int k = 0; k < EC; ++k)
      exponents(k, [&](int e, double x) { sm[e] += (double)exp2_of(x - mx[e], R()); });
    double tot = 0.0;
#pragma unroll
    for (int e = 0; e < ER; ++e) {
      sm[e] = row16<false>(sm[e]);
      tot = lc == e ? sm[e] : tot;
    }
    if (GC > 1) {
      tot = rows_of(tot, Sum());
      __syncthreads();
    }
    f_l = a_l;
    Ur_l = a_l > 0.0 ? -mine - log2(tot) : -__builtin_inf();
    if (rown && a_l != 0.0 && !__builtin_isfinite(Ur_l)) Ur_l = __builtin_nan("");
  };

  // ---- start ----
  bool skip_rows = false;  // the loop starts with the column half
  bool exact_now = false;  // the first row half is the exact log-sum-exp
  if (STAB) {
    f_l = rown ? A.u_start : 0.0;  // (Ur, Vr: alpha, beta)
    g_t = cown ? A.v_start : 0.0;
  } else if (A.resume || !LOG) {
    if (LOG) {
      Ur_l = a_l > 0.0 ? Ur_l - la_l : -__builtin_inf();
      f_l = a_l;
      g_t = b_t != 0.0 ? 1.0 : 0.0;
      if (!row_first && b_t == 0.0) Vr_t = -__builtin_inf();
    } else {
      f_l = Ur_l;
      g_t = Vr_t;
      Ur_l = 0.0;
      Vr_t = 0.0;
    }
    skip_rows = A.resume && !row_first;
  } else {
    exact_now = true;
    g_t = cown ? 1.0 : 0.0;
  }
  if (tid < CB) {
    vr[tid] = cown ? Vr_t : -__builtin_inf();
    gsh[tid] = (R)g_t;
  }
  __syncthreads();
  if (LOG && !A.resume && !row_first) {
    // v_1 = log b - LSE_i(M s2 + u_0), in fp64 for either type.
    const int l = here(lane), c0 = l & 15, r0 = wv * 4 + (l >> 4);
    if (c0 < ER) ursh[r0 + TR * c0] = rown ? Ur_l : -__builtin_inf();
    __builtin_amdgcn_wave_barrier();
    double acc[EC];
    auto exponents = [&](int e, auto use) {
      const int r = r0 + TR * e;
      const double ur = ursh[r];
      const TM* row = Mp + (int64_t)min(r, nr - 1) * A.ldm;
#pragma unroll
      for (int k = 0; k < EC; ++k) use(k, fma((double)row[min(c0 + 16 * k, nc - 1)], s2, ur));
    };
#pragma unroll
    for (int k = 0; k < EC; ++k) acc[k] = -__builtin_inf();
#pragma unroll 1
    for (int e = 0; e < ER; ++e) exponents(e, [&](int k, double x) { acc[k] = fmax(acc[k], x); });
    double mx = cols_reduce(acc, Max());
    if (GR > 1) mx = cols_of(mx, Max());
    if (!(mx > -1e300)) mx = 0.0;
    if (tid < CB) cmx[tid] = mx;
    __syncthreads();
#pragma unroll
    for (int k = 0; k < EC; ++k) acc[k] = 0.0;
#pragma unroll 1
    for (int e = 0; e < ER; ++e)
      exponents(e, [&](int k, double x) { acc[k] += exp2(x - cmx[c0 + 16 * k]); });
    double sm = cols_reduce(acc, Sum());
    if (GR > 1) sm = cols_of(sm, Sum());
    if (cown) {
      Vr_t = b_t != 0.0 ? log2(b_t) - mx - log2(sm) : -__builtin_inf();
      if (b_t != 0.0 && !__builtin_isfinite(Vr_t)) events = 2;
      g_t = b_t != 0.0 ? 1.0 : 0.0;
    }
    if (tid < CB) {
      vr[tid] = cown ? Vr_t : -__builtin_inf();
      gsh[tid] = (R)g_t;
    }
    __syncthreads();
    if (events || (BLK && dead)) return abandon();
  }
  bool need_build = !exact_now;
  bool check_cols = !row_first && !skip_rows;  // not where a segment resumes
  bool knopp_start = !LOG && !A.resume && !row_first;  // v_1 = b / (K^T u_0) first
  if (knopp_start) {
    skip_rows = true;
    check_cols = false;
  }

  int it = A.it0;
  int next_check = row_first ? (it <= 1 && !A.resume ? 1 : it + 10) : (check_cols || knopp_start ? 0 : it + 10);
  int n_err = 0, status = kMaxIter, niter = 0;
  int over_last = 16;  // the flag that the last column update may have raised
  double last_err = 1.0;  // stabilised: the reference's, kept between checks
  double g_prev = g_t;
  const bool live = rown && a_l != 0.0;
  // Whether a positive double lies outside [2^-kDrift, 2^kDrift] (or is no
  // number), from its exponent.
  auto off_range = [](double x) {
    const unsigned hi = (unsigned)((unsigned long long)__double_as_longlong(x) >> 32);
    return hi - ((1023u - kDrift) << 20) > ((2u * kDrift) << 20);
  };

  // Whether this thread's column cannot be updated from its sum c: no number, a
  // mass below the trusted range, or a scaling that the row sweep reports.
  auto no_update = [&](double c) -> bool {
    if (!cown) return false;
    const double g = b_t / c;
    if (LOG)
      return b_t == 0.0 ? c != c : !(g_t * c >= kFloor) || !__builtin_isfinite(g) || !(g > 0.0);
    return c == 0.0 || !__builtin_isfinite(c) || !__builtin_isfinite(g);
  };

  // Square root of the problems' summed squared errors, joint over the batch.
  // Returns -1 where the launch ends here (segment) or the wait gave up.
  auto joint_error = [&](double e2, int parts, bool publish, int me) -> double {
    const double s = wave_sum_dpp_d(e2);
    if (lane == 0) red[wv] = s;
    __syncthreads();
    double tot = 0.0;
#pragma unroll
    for (int w = 0; w < W; ++w) tot += red[w];
    if (A.segment) {
      if (tid == 0) A.errpart[p] = tot;
      return -1.0;
    }
    const int nprob = A.each ? 1 : A.B;
    if (nprob * parts == 1) return sqrt(tot);
    ++tag_e;
    word_t* base = xerr + (int64_t)(tag_e & 1) * A.err_slot;
    if (publish && tid == 0)
      value_put(slot_at(base, (int)A.err_slot), p * parts + me, tot, tag_e);
    const int N = nprob * parts;
    gather(xs, base + (A.each ? (int64_t)p * parts * 2 : 0), N, N, 1, tag_e);
    __syncthreads();
    double e = 0.0;
    for (int q = tid; q < nprob; q += T) {
      double t = 0.0;
      for (int k = 0; k < parts; ++k) t += xs[q * parts + k];
      e = A.err_norm == 1 ? e + t : fmax(e, sqrt(t));
      if (__builtin_isnan(t)) e = t;
    }
    if (A.err_norm == 1) {
      e = wave_sum_dpp_d(e);
    } else {
      const bool nan = __any(__builtin_isnan(e));
      e = nan ? __builtin_nan("") : wave_max(e);
    }
    __syncthreads();  // red and xs are read above
    if (lane == 0) red[wv] = e;
    __syncthreads();
    e = red[0];
#pragma unroll
    for (int w = 1; w < W; ++w) {
      if (A.err_norm == 1)
        e += red[w];
      else
        e = (red[w] > e || __builtin_isnan(red[w])) ? red[w] : e;
    }
    return A.err_norm == 1 ? sqrt(e) : e;
  };

  for (;;) {
    if (need_build) build();
    need_build = false;
    // ---- row half: f = a / (K g) ----
    if (!skip_rows) {
      bool slow = exact_now;
      double S = 0.0;
      if (!exact_now) {
        R s[ER];
#pragma unroll
        for (int e = 0; e < ER; ++e) s[e] = 0;
#pragma unroll
        for (int k = 0; k < EC; ++k) {
          const R g = gsh[lc + 16 * k];
#pragma unroll
          for (int e = 0; e < ER; ++e) s[e] = fma_r(K[e][k], g, s[e]);
        }
        R mine = 0;
#pragma unroll
        for (int e = 0; e < ER; ++e) {
          s[e] = row16<false>(s[e]);
          mine = lc == e ? s[e] : mine;
        }
        S = (double)mine;
        if (GC > 1) {
          S = rows_of(mine, Sum(), STAB && (events & over_last));
          if (STAB && raised && tid == 0) atomicOr(&events, over_last);
          if (dead) return abandon();
        }
        if (row_first && it == next_check) {
          const double d = f_l * S - a_l;
          const double err = joint_error(live ? d * d : 0.0, GR, J == 0, I);
          if (A.segment) break;
          if (dead) return abandon();
          if (!A.each && blockIdx.x == 0 && tid == 0 && n_err < A.err_cap) A.err_hist[n_err] = err;
          ++n_err;
          next_check += 10;
          if (err < A.stop_thr) {
            status = kConverged;
            niter = it - 1;
            break;
          }
        }
        f_l = rown ? a_l / S : 0.0;
        // (One lane of a wave raises the flag: where most scalings pass tau, an
        // atomic of each took 1 us an iteration.  1000 x 900 float64 with an
        // absorption in every one 12.6 us, 11.9 now; 1524 x 661 15.8 and 14.1.)
        if (STAB && __any(fabs(f_l) > A.tau) && lane == 0) atomicOr(&events, 8);
        if (LOG) {
          if (!live) f_l = 0.0;
          slow = __any(live && off_range(S));  // (a wave has its rows to itself)
        }
      }
      if (LOG && slow) {
        // A row sum off the range: its scaling goes into the reference; off
        // the type's range, or in the first iteration, the exact sum.  (Where
        // the row's blocks have to meet for that, the whole workgroup does it
        // after its next barrier.)
        const bool weird = live && !(S >= 1.0 / kSafe && S <= kSafe);
        if (exact_now || (GC == 1 && __any(weird))) {
          exact_rows();
        } else if (weird) {
          weird_rows = 1;
        } else if (live && off_range(S)) {
          Ur_l -= log2(S);
          f_l = a_l;
        }
        exact_now = false;
        need_build = skip_rows = true;  // K again, then on with the column half
        continue;
      }
    }
    skip_rows = false;

    // ---- column half: g = b / (K^T f) ----
    double c;
    {
      R fe[ER];
      row_spread<0, ER>((R)f_l, fe);
      R acc[EC];
#pragma unroll
      for (int k = 0; k < EC; ++k) {
        acc[k] = K[0][k] * fe[0];
#pragma unroll
        for (int e = 1; e < ER; ++e) acc[k] = fma_r(K[e][k], fe[e], acc[k]);
      }
      c = cols_reduce(acc, Sum());
    }
    if (LOG && GC > 1 && weird_rows) {
      __syncthreads();
      if (tid == 0) weird_rows = 0;
      exact_rows();
      need_build = skip_rows = true;
      continue;
    }
    bool absorb = false;
    if (STAB) absorb = (events & (8 | over_last)) != 0;
    if (GR > 1) {
      c = cols_of((R)c, Sum(), STAB && (events & 8));
      if (STAB) absorb = raised || (events & over_last);
    }
    if (STAB && absorb) {
      // A scaling exceeded tau in the iteration that these sums follow: they
      // are of the unabsorbed pair.  Every block learns it here, columns'
      // scalings through the row exchange, rows' through this one.
      __syncthreads();
      if (tid == 0) events = 0;
      if (BLK && dead) return abandon();
      if (rown) Ur_l += A.reg * log(f_l);
      if (cown) vr[tid] = Vr_t += A.reg * log(g_t);
      f_l = rown ? A.u_start : 0.0;
      g_t = cown ? A.v_start : 0.0;
      if (cown) gsh[tid] = (R)g_t;
      __syncthreads();
      need_build = skip_rows = true;
      continue;
    }
    if (STAB && !knopp_start) {
      if (it == next_check) {
        const double d = g_t * c - b_t;
        last_err = joint_error(cown ? d * d : 0.0, GC, I == 0, J);
        if (dead) return abandon();
        if (blockIdx.x == 0 && tid == 0 && n_err < A.err_cap) A.err_hist[n_err] = last_err;
        ++n_err;
        next_check += A.period;
      }
      const bool stop = last_err <= A.stop_thr;
      if (stop || it >= A.max_iter - 1) {
        // (a row scaling that is no number makes every column sum so; the pair
        // before it is the outcome then)
        if (__syncthreads_or(cown && c != c)) return abandon();
        if (stop) status = kConverged;
        niter = it;
        break;
      }
    }
    if (!STAB && check_cols && it == next_check) {
      const double d = g_t * c - b_t;
      const double err = joint_error(cown ? d * d : 0.0, GC, I == 0, J);
      // (the update that follows decides first: what it gives up on is neither
      // converged nor the last state)
      if (A.segment) {
        if (__syncthreads_or(no_update(c))) return abandon();
        break;
      }
      if (dead) return abandon();
      if (!A.each && blockIdx.x == 0 && tid == 0 && n_err < A.err_cap) A.err_hist[n_err] = err;
      ++n_err;
      next_check += 10;
      if (err < A.stop_thr) {
        if (__syncthreads_or(no_update(c))) return abandon();
        status = kConverged;
        niter = it;
        break;
      }
    }
    check_cols = !row_first;
    g_prev = g_t;
    if (cown) {
      const bool none = no_update(c);  // (a row scaling that is not finite makes every c so)
      g_t = LOG && b_t == 0.0 ? 0.0 : b_t / c;
      if (none)
        atomicOr(&events, 2);
      else if (LOG && b_t != 0.0 && off_range(g_t))
        atomicOr(&events, 1);
      gsh[tid] = (R)g_t;
    }
    if (STAB && __any(cown && __builtin_isfinite(c) && fabs(g_t) > A.tau) && lane == 0)
      atomicOr(&events, 20 - over_last);
    __syncthreads();
    over_last = 20 - over_last;
    if ((STAB ? events & 2 : events) | (BLK ? dead : 0)) {
      // Uniform in the workgroup; references move in the whole column group,
      // whose members have the same sums.
      if ((events & 2) || (BLK && dead)) return abandon();
      if (it < A.max_iter - 1) {
        __syncthreads();
        if (tid == 0) events = 0;
        if (cown && g_t > 0.0) {
          Vr_t += log2(g_t);
          g_t = 1.0;
          vr[tid] = Vr_t;
          gsh[tid] = (R)1;
        }
        __syncthreads();
        need_build = true;
      }
    }
    if (knopp_start) {
      knopp_start = false;
      continue;  // the first iteration proper follows
    }
    if (!STAB && it >= A.max_iter - 1) {
      niter = it;
      if (!row_first) g_t = g_prev;
      break;
    }
    ++it;
  }

  // ---- results ----
  // (a segment's state stays in base 2; the host converts the last one)
  const double back = LOG && !A.segment ? kLn2 : 1.0;
  if (rown && J == 0)
    A.u_out[ri] = LOG ? (a_l > 0.0 ? (Ur_l + log2(f_l)) * back : -__builtin_inf()) : f_l;
  if (cown && I == 0)
    A.v_out[ci] = LOG ? (g_t > 0.0 ? (Vr_t + log2(g_t)) * back : -__builtin_inf()) : g_t;
  if (STAB) {
    if (rown && J == 0) A.alpha_out[ri] = Ur_l;
    if (cown && I == 0) A.beta_out[ci] = Vr_t;
  }
  if (tid == 0 && !A.segment) {
    if (A.each && rem == 0) {
      A.niters[p] = niter;
      A.statuses[p] = status;
    }
    Ctrl* q = A.host ? A.host : A.ctrl;
    if (gridDim.x == 1) q->counter = 0;  // no launch has cleared it
    if (A.each && A.B > 1) {
      atomicMax(&q->niter, niter);  // the last problem's stop
    } else if (blockIdx.x == 0) {
      q->done = 1;
      q->status = status;
      q->niter = niter;
      q->bad_iter = -1;
      q->n_err = A.each ? 0 : n_err;
    }
  }
}

// Launches the kernel, or only asks how many workgroups fit a CU.
template <typename TM, typename R, int W, int ER, int EC, int MODE, bool BLK>
hipError_t on_kernel(const ResidentArgs& a, int grid, size_t lds, hipStream_t s, int* per_cu) {
  const auto k = resident_kernel<TM, R, W, ER, EC, MODE, BLK>;
  if (per_cu) return hipOccupancyMaxActiveBlocksPerMultiprocessor(per_cu, k, 64 * W, lds);
  if (lds > 65536) {
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(k),
                                       hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return e;
  }
  hipLaunchKernelGGL(k, dim3(grid), dim3(64 * W), lds, s, a);
  return hipGetLastError();
}
template <typename TM, typename R, int MODE>
hipError_t on_tile(const ResidentTile& t, const ResidentArgs& a, int grid, size_t lds,
                   hipStream_t s, int* per_cu) {
  const bool blk = a.R * a.C > 1;
#define POTAMD_TILE(w_, er, ec)                                                            \
  if (t.W == w_ && t.ER == er && t.EC == ec)                                               \
    return blk ? on_kernel<TM, R, w_, er, ec, MODE, true>(a, grid, lds, s, per_cu)         \
               : on_kernel<TM, R, w_, er, ec, MODE, false>(a, grid, lds, s, per_cu);
  if constexpr (sizeof(R) == 4) {
    POTAMD_TILES_F32(POTAMD_TILE)
  } else {
    POTAMD_TILES_F64(POTAMD_TILE)
  }
#undef POTAMD_TILE
  return hipErrorInvalidConfiguration;
}

}  // namespace
}  // namespace potamd

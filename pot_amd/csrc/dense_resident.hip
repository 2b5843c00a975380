// Host side of the register-resident dense solve (resident.h): choice of the
// tile, the exchange workspace, and the launches.
#include <string.h>

#include <algorithm>
#include <atomic>
#include <chrono>
#include <condition_variable>
#include <mutex>
#include <thread>

#include "../../include/pot_amd.h"
#include "host.h"
#include "internal.h"
#include "resident.h"

namespace potamd {
namespace {

// Clears the exchange words and the control block and keeps the caller's
// start, which an abandoned solve begins from again.
__global__ __launch_bounds__(256) void resident_init_kernel(word_t* words, int64_t count, Ctrl* c,
                                                            const double* u, double* u_keep,
                                                            int64_t nu, const double* v,
                                                            double* v_keep, int64_t nv) {
  const int64_t i0 = (int64_t)blockIdx.x * 256 + threadIdx.x, step = (int64_t)gridDim.x * 256;
  for (int64_t i = i0; i < count; i += step) words[i] = 0;
  for (int64_t i = i0; i < nu; i += step) u_keep[i] = u[i];
  for (int64_t i = i0; i < nv; i += step) v_keep[i] = v[i];
  if (i0 == 0) {
    c->done = 0;
    c->status = kMaxIter;
    c->niter = -1;
    c->bad_iter = -1;
    c->counter = 0;
    c->n_err = 0;
    c->need_exact = 0;
    c->err = 0.0;
  }
}

// Stop decision between two segments: the batch's largest error (or its
// Frobenius norm) at the check iteration `it` that the segment ended with.
__global__ __launch_bounds__(256) void resident_decide_kernel(const double* errpart, int B,
                                                              int err_norm, int it, int last,
                                                              int checked, double stop_thr,
                                                              double* err_hist, int err_cap,
                                                              Ctrl* c) {
  if (c->done) return;
  const int tid = threadIdx.x;
  __shared__ double red[256];
  double e = 0.0;
  if (checked)
    for (int q = tid; q < B; q += 256) {
      const double t = errpart[q];
      e = err_norm == 1 ? e + t : fmax(e, sqrt(t));
      if (__builtin_isnan(t)) e = t;
    }
  red[tid] = e;
  __syncthreads();
  if (tid != 0) return;
  e = 0.0;
  for (int k = 0; k < 256; ++k) {
    if (err_norm == 1)
      e += red[k];
    else
      e = (red[k] > e || __builtin_isnan(red[k])) ? red[k] : e;
  }
  if (err_norm == 1) e = sqrt(e);
  if (checked) {
    if (c->n_err < err_cap) err_hist[c->n_err] = e;
    c->n_err += 1;
    c->err = e;
    if (e < stop_thr) {
      c->done = 1;
      c->status = kConverged;
      c->niter = it;
      return;
    }
  }
  if (last) {
    c->done = 1;
    c->status = kMaxIter;
    c->niter = it;
  }
}

using Tile = ResidentTile;

size_t lds_bytes(const Tile& t, int R, int C, int nerr) {
  const size_t rb = t.rows(), cb = t.cols();
  size_t x = 0;
  if (C > 1) x = (rb + 1) * (C | 1);
  if (R > 1) x = std::max(x, (cb + 1) * (R | 1));
  x = std::max(x, (size_t)nerr);
  return 8 * (t.W * cb + 2 * cb + rb + cb + x);
}

#define POTAMD_TILE_ENTRY(w, er, ec) {w, er, ec},
const Tile kTilesF32[] = {POTAMD_TILES_F32(POTAMD_TILE_ENTRY)};
const Tile kTilesF64[] = {POTAMD_TILES_F64(POTAMD_TILE_ENTRY)};
#undef POTAMD_TILE_ENTRY

// Tile and blocks of a problem.  Blocks that wait for each other must all be
// resident: one workgroup a CU is always possible, so at most 256 of them.
struct Choice {
  int tile = -1;
  int R = 1, C = 1;
};

// The cheapest tile by the clocks of an iteration: two multiply-adds an
// element on the resident workgroups of a CU (4 clocks each), about 1100
// clocks of reductions, divisions and barriers, and 3000 to 6000 clocks for an
// exchange, more with more members (measured a whole iteration, 2.4 GHz: one
// workgroup 1.1 us at 64 x 64, 1.8 at 100 x 120 and 2.3 at 200 x 120 in the
// float64 log domain; blocked 4.9 us at 300^2 (3 x 3), 5.4 at 1000 x 900, 6.8 at
// 2048^2 (16 x 16); the row sweep took 13, 13, 14, 15, 22 and 37 us).  So a problem
// that fits one workgroup stays in one.
// Of two tiles of one size (128 x 128 by eight waves or by four of twice the
// elements) the fewer waves where there are more problems than CUs, as more such
// workgroups are resident at once (300 problems of 110 x 90 7.2 us an iteration
// in segments, 2.5 so; float32 5.5, 1.8), and for a float64 problem in the log
// domain, whose waves each have their own checks (64 of 100^2 1.88, 1.73; the
// scaling domain 1.41, 1.48; float32 1.31, 1.41).  Both have the same exchange
// words.
Choice choose(int dtype, int B, int n, int m, bool logd = false) {
  Choice best;
  const bool f32 = dtype == 0;
  const Tile* tab = f32 ? kTilesF32 : kTilesF64;
  const int cnt = f32 ? sizeof(kTilesF32) / sizeof(Tile) : sizeof(kTilesF64) / sizeof(Tile);
  constexpr int kCus = 256;
  double best_cost = 0.0;
  for (int q = 0; q < cnt; ++q) {
    const Tile& t = tab[q];
    const int R = (n + t.rows() - 1) / t.rows(), C = (m + t.cols() - 1) / t.cols();
    const int64_t total = (int64_t)B * R * C;
    if (R > 64 || C > 64 || (R * C > 1 && total > kCus)) continue;
    const double share = std::max(1.0, (double)total / kCus);
    double cost = 1100.0 + 2.0 * t.ER * t.EC * t.W * share;
    if (C > 1) cost += 3000.0 + 3.0 * t.rows() * C / t.W;
    if (R > 1) cost += 3000.0 + 3.0 * t.cols() * R / t.W;
    const bool fewer = R * C == 1 && (total > kCus || (logd && !f32));
    if (best.tile < 0 || cost < best_cost || (fewer && cost == best_cost)) {
      best.tile = q;
      best.R = R;
      best.C = C;
      best_cost = cost;
    }
  }
  return best;
}

struct Words {
  int64_t row_slot, col_slot, err_slot, col_base, err_base, total;
};
Words words_of(int B, int n, int m, const Choice& c) {
  const int rbs = (n + c.R - 1) / c.R, cbs = (m + c.C - 1) / c.C;
  Words w;
  // Each member's values (and a flag), and the totals.
  w.row_slot = c.C > 1 ? (int64_t)(rbs + 1) * (c.C + 1) * 2 : 0;
  w.col_slot = c.R > 1 ? (int64_t)(cbs + 1) * (c.R + 1) * 2 : 0;
  w.err_slot = (int64_t)B * std::max(c.R, c.C) * 2;
  w.col_base = (int64_t)B * c.R * 2 * w.row_slot;
  w.err_base = w.col_base + (int64_t)B * c.C * 2 * w.col_slot;
  w.total = w.err_base + 2 * w.err_slot;
  return w;
}

// Solves whose workgroups wait for each other, of all threads of the process on
// one device: together they have at most a workgroup a CU, so that each finds a
// CU that none of the others holds and all are resident (workgroups go to the
// eight XCDs in turn, so a solve counts as a multiple of eight).  Other kernels
// end by themselves.
class WaitingSolves {
  using Clock = std::chrono::steady_clock;

 public:
  // Notes a solve of this thread; whether another thread had one in the last second.
  bool arrive() {
    std::lock_guard<std::mutex> lock(mutex_);
    const auto me = std::this_thread::get_id();
    if (me != last_) others_at_ = last_at_;
    last_ = me;
    last_at_ = Clock::now();
    return last_at_ - others_at_ < std::chrono::seconds(1);
  }
  // False where the CUs are not free for a second: the holders' streams share a
  // hardware queue with longer work.
  bool enter(int cus, int of) {
    std::unique_lock<std::mutex> lock(mutex_);
    if (!freed_.wait_for(lock, std::chrono::seconds(1),
                         [&] { return used_ == 0 || used_ + cus <= of; }))
      return false;
    used_ += cus;
    return true;
  }
  // Whether solves that wait are left out now: after a wait that ran out, for half
  // a second (what keeps workgroups off the GPU may do so at each call, and each
  // would lose those 20 ms).
  bool paused() {
    std::lock_guard<std::mutex> lock(mutex_);
    return Clock::now() < paused_until_;
  }
  void pause(std::chrono::milliseconds time) {
    std::lock_guard<std::mutex> lock(mutex_);
    paused_until_ = Clock::now() + time;
  }
  void leave(int cus) {
    {
      std::lock_guard<std::mutex> lock(mutex_);
      used_ -= cus;
    }
    freed_.notify_all();
  }
  static WaitingSolves& on(int dev) {
    static WaitingSolves* all = new WaitingSolves[64];  // (outlives every thread)
    return all[dev & 63];
  }

 private:
  std::mutex mutex_;
  std::condition_variable freed_;
  int used_ = 0;
  std::thread::id last_;  // the last solve's thread, and when; the last of another one
  Clock::time_point last_at_ = Clock::time_point() - std::chrono::hours(1);
  Clock::time_point others_at_ = last_at_;
  Clock::time_point paused_until_ = last_at_;
};

// The CUs of one solve, until it has ended.
struct CuShare {
  WaitingSolves* of = nullptr;
  int cus = 0;
  ~CuShare() {
    if (of) of->leave(cus);
  }
};

thread_local long long wait_ticks = kWaitTicks;

}  // namespace

bool resident_fits(int dtype, int B, int n, int m) { return choose(dtype, B, n, m).tile >= 0; }

size_t resident_workspace(int dtype, int B, int n, int m) {
  const Choice c = choose(dtype, B, n, m);
  return c.tile >= 0 ? (size_t)words_of(B, n, m, c).total * 8 : 0;
}

// 0: solved (info in *out), 1: not taken or abandoned (u and v are as they
// were), other: a HIP error.
int resident_solve(int dtype, ResidentArgs a, double* u_keep, double* v_keep, Ctrl* host_ctrl,
                   hipStream_t s, Ctrl* out) {
  const Choice c = choose(a.stab ? 1 : dtype, a.B, a.n, a.m, a.logd && !a.stab);
  if (c.tile < 0) return 1;
  const bool f32 = dtype == 0 && !a.stab;  // (stabilised: fp64 elements)
  const Tile t = f32 ? kTilesF32[c.tile] : kTilesF64[c.tile];
  a.R = c.R;
  a.C = c.C;
  a.rbs = (a.n + c.R - 1) / c.R;
  a.cbs = (a.m + c.C - 1) / c.C;
  const Words w = words_of(a.B, a.n, a.m, c);
  a.row_slot = (int)w.row_slot;
  a.col_slot = (int)w.col_slot;
  a.err_slot = w.err_slot;
  a.col_base = w.col_base;
  a.err_base = w.err_base;
  const int grid = a.B * c.R * c.C;
  const int parts = a.row_first ? c.R : c.C;
  const bool lone = grid == 1;
  // Workgroups that wait for each other: the blocks of a problem, and the
  // problems of a batch with one stop, unless there are more than fit.
  const bool blocked = c.R * c.C > 1, joint = a.B > 1 && !a.each;
  bool segment = false, waits = blocked || joint;
  a.wait_ticks = wait_ticks;
  size_t lds = lds_bytes(t, c.R, c.C, waits ? (a.each ? 1 : a.B) * parts : 0);
  auto launch = [&](const ResidentArgs& x, int* per_cu) -> hipError_t {
    if (x.stab) return resident_launch_stab(dtype == 0, t, x, grid, lds, s, per_cu);
    return f32 ? resident_launch_f32(t, x, grid, lds, s, per_cu)
               : resident_launch_f64(t, x, grid, lds, s, per_cu);
  };
  int dev = 0;
  if (waits) {
    if (hipGetDevice(&dev) != hipSuccess) return 1;
    int per_cu = 0;
    const bool fits = !WaitingSolves::on(dev).paused() && lds <= 160 * 1024 &&
                      launch(a, &per_cu) == hipSuccess &&
                      (int64_t)grid <= (int64_t)per_cu * device_cus();
    if (!fits) {
      if (blocked) return 1;
      segment = true;
      waits = false;
      lds = lds_bytes(t, c.R, c.C, 0);
    }
  }
  const int64_t Bn = (int64_t)a.B * a.n, Bm = (int64_t)a.B * a.m;
  Ctrl local;
  Ctrl* hc = host_ctrl ? host_ctrl : &local;

  CuShare share;
  if (waits) {
    WaitingSolves& solves = WaitingSolves::on(dev);
    // Where several threads solve, the CUs are held for the solve alone, not for
    // work queued before it (another thread's solve would wait for that).  A
    // program of one thread queues the solve behind that work: 2048^2 float64
    // 451 us a call, 494 with the wait.
    if (solves.arrive() && hipStreamSynchronize(s) != hipSuccess) return -1;
    const int cus = std::min(device_cus(), (grid + 7) / 8 * 8);
    if (!solves.enter(cus, device_cus())) return 1;
    share.of = &solves;
    share.cus = cus;
  }
  if (!lone) {
    const int64_t words = waits ? w.total : 0;
    const int64_t most = std::max(words, std::max(Bn, Bm));
    const int blocks = (int)std::min<int64_t>(1024, (most + 255) / 256);
    hipLaunchKernelGGL(resident_init_kernel, dim3(blocks), dim3(256), 0, s, a.words, words, a.ctrl,
                       a.u_in, u_keep, Bn, a.v_in, v_keep, Bm);
    if (hipGetLastError() != hipSuccess) return -1;
  }
  if (!segment) {
    a.segment = 0;
    a.resume = 0;
    a.it0 = 0;
    // The kernel writes its outcome where the host reads it (a copy of it was a
    // launch and its wait: 100 x 120 float64 93.2 us a call, 90.9 without), but for a
    // batch whose problems all add to it.
    a.host = nullptr;
    void* seen = nullptr;
    if (host_ctrl && !(a.each && a.B > 1)) {
      if (hipHostGetDevicePointer(&seen, host_ctrl, 0) == hipSuccess)
        a.host = static_cast<Ctrl*>(seen);
      else
        (void)hipGetLastError();
    }
    if (a.host) {
      memset(hc, 0, sizeof(Ctrl));
      std::atomic_thread_fence(std::memory_order_seq_cst);
    }
    if (launch(a, nullptr) != hipSuccess) return -1;
    if ((!a.host &&
         hipMemcpyAsync(hc, a.ctrl, sizeof(Ctrl), hipMemcpyDeviceToHost, s) != hipSuccess) ||
        hipStreamSynchronize(s) != hipSuccess)
      return -1;
    if (a.host && !hc->done && !hc->counter) hc->counter = kGivenUp;
  } else {
    // One launch per check interval; the state travels in u and v themselves
    // (base 2), and at most two intervals are queued past an unread decision.
    a.segment = 1;
    constexpr int kAhead = 2;
    hipEvent_t ev[kAhead];
    for (int k = 0; k < kAhead; ++k)
      if (hipEventCreateWithFlags(&ev[k], hipEventDisableTiming) != hipSuccess) return -1;
    Ctrl snap[kAhead];
    Ctrl* ring = host_ctrl ? host_ctrl : snap;
    bool ok = true, stop = false;
    int seg = 0;
    double* const u = a.u_out;
    double* const v = a.v_out;
    for (; ok && !stop; ++seg) {
      if (seg >= kAhead) {
        ok = hipEventSynchronize(ev[seg % kAhead]) == hipSuccess;
        if (!ok || ring[seg % kAhead].done) break;
      }
      // The check of this segment: iteration 10 seg (seen one iteration later
      // in the row-first order).
      const int chk = 10 * seg;
      const bool reach = a.row_first ? chk + 1 <= a.max_iter - 1 : chk <= a.max_iter - 1;
      a.resume = seg > 0;
      a.it0 = seg == 0 ? 0 : (a.row_first ? chk - 9 : chk - 10);
      a.u_in = u;
      a.v_in = v;
      ok = launch(a, nullptr) == hipSuccess;
      const bool last = !reach || (!a.row_first && chk == a.max_iter - 1);
      hipLaunchKernelGGL(resident_decide_kernel, dim3(1), dim3(256), 0, s, a.errpart, a.B,
                         a.err_norm, reach ? chk : a.max_iter - 1, last ? 1 : 0, reach ? 1 : 0,
                         a.stop_thr, a.err_hist, a.err_cap, a.ctrl);
      ok = ok && hipGetLastError() == hipSuccess &&
           hipMemcpyAsync(&ring[seg % kAhead], a.ctrl, sizeof(Ctrl), hipMemcpyDeviceToHost, s) ==
               hipSuccess &&
           hipEventRecord(ev[seg % kAhead], s) == hipSuccess;
      if (last) stop = true;
    }
    ok = ok && hipMemcpyAsync(hc, a.ctrl, sizeof(Ctrl), hipMemcpyDeviceToHost, s) == hipSuccess &&
         hipStreamSynchronize(s) == hipSuccess;
    for (int k = 0; k < kAhead; ++k) (void)hipEventDestroy(ev[k]);
    if (!ok) return -1;
    if (!hc->counter && a.logd) {
      if (launch_scale_copy(Bn, u, kLn2, u, s) != hipSuccess ||
          launch_scale_copy(Bm, v, kLn2, v, s) != hipSuccess)
        return -1;
    }
  }
  *out = *hc;
  if (a.each) out->status = out->niter >= a.max_iter - 1 ? kMaxIter : kConverged;
  if (!out->counter) return 0;
  if (out->counter == kWaitedOut && waits)
    WaitingSolves::on(dev).pause(std::chrono::milliseconds(500));
  // (the stabilised solve starts from alpha and beta, the others from u and v)
  double* const u_back = a.stab ? a.alpha_out : a.u_out;
  double* const v_back = a.stab ? a.beta_out : a.v_out;
  if (!lone && (launch_scale_copy(Bn, u_keep, 1.0, u_back, s) != hipSuccess ||
                launch_scale_copy(Bm, v_keep, 1.0, v_back, s) != hipSuccess))
    return -1;
  return 1;
}

}  // namespace potamd

using namespace potamd;

extern "C" int potamd_resident_wait_limit(int us) {
  wait_ticks = us == 0 ? kWaitTicks : us < 0 ? -1 : 100ll * us;
  int dev = 0;
  HIP_TRY(hipGetDevice(&dev));
  WaitingSolves::on(dev).pause(std::chrono::milliseconds(0));
  return 0;
}

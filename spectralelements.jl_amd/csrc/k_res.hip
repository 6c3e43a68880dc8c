// Tile plan and dispatch of the resident PCG (k_res.h) over P; the kernels are
// instantiated per P in k_res_inst.hip.
#include <algorithm>
#include <condition_variable>
#include <mutex>

#include "sem_common.h"

namespace sem {
namespace res {
template <typename T, int P>
int launch_res_p(hipStream_t st, const ResLaunch& l);
#define SEM_RES_EXTERN(P)                                                \
  extern template int launch_res_p<double, P>(hipStream_t, const ResLaunch&); \
  extern template int launch_res_p<float, P>(hipStream_t, const ResLaunch&);
SEM_RES_EXTERN(2) SEM_RES_EXTERN(3) SEM_RES_EXTERN(4) SEM_RES_EXTERN(5) SEM_RES_EXTERN(6)
SEM_RES_EXTERN(7) SEM_RES_EXTERN(8) SEM_RES_EXTERN(9) SEM_RES_EXTERN(10) SEM_RES_EXTERN(11)
SEM_RES_EXTERN(12) SEM_RES_EXTERN(13) SEM_RES_EXTERN(14) SEM_RES_EXTERN(15) SEM_RES_EXTERN(16)
#undef SEM_RES_EXTERN
}  // namespace res

// Tiles of at most max_waves waves of 64 / P elements each, at most one per CU.
// The cost in microseconds per iteration, from sweeps over tiles (P = 4 to 16, 20x20
// to 128x128 elements):
// - the two exchanges, by their form and the workgroups that take part; on one XCD
//   they are 0.6 (2 workgroups) to 0.8 (32) cheaper than spread over the chip;
// - a second wave per SIMD: 0.5 while the coefficients fit the scalar registers (FP64
//   up to P = 8), 1.2 beyond, in FP32 0.3 and 1.0 (fewer than four waves bring nothing);
// - each round of the waves other than the first over the tile's edge entries: 0.4.
// 64x64 elements, N = 9: 208 workgroups of 5x4 elements 7.7 us, 176 of 4x6 8.2 (a second
// round of the edges), 121 of 6x6 (6 waves) 9.5; 40x40, N = 7: 30 workgroups of 8x7 on
// one XCD 5.75, 56 of 5x6 6.1, 50 of 4x8 6.5.
ResPlan res_plan(const Layout& g, int elem_bytes, int ncu) {
  const int epw = 64 / g.P, max_waves = elem_bytes * g.P <= 80 ? 8 : 4;
  const int max_wg = std::min(ncu, 256);
  ResPlan best{};
  if ((long)g.L * g.NC >= (1L << 31) / 4) return best;
  double best_cost = 0.0;
  for (int TX = 1; TX <= std::min(g.Ex, max_waves * epw); ++TX) {
    const int ntx = (g.Ex + TX - 1) / TX;
    if ((g.Ex + ntx - 1) / ntx != TX) continue;   // the narrowest tile of this count
    for (int RY = 1; RY <= std::min(g.Ey, max_waves * epw / TX); ++RY) {
      const int nty = (g.Ey + RY - 1) / RY;
      if ((g.Ey + nty - 1) / nty != RY || (long)ntx * nty > max_wg) continue;
      ResPlan pl{TX, RY, ntx, nty, ntx * nty, (TX * RY + epw - 1) / epw, 0};
      pl.near = res_near(pl.nwg, ncu);
      const double second = elem_bytes == 4 ? (g.P <= 12 ? 0.3 : 1.0) : g.P <= 8 ? 0.5 : 1.2;
      const double exchange = pl.nwg == 1    ? -3.0
                              : pl.near == 1 ? -0.6 + 0.003 * pl.nwg
                              : pl.near == 2 ? 0.86 + 0.001 * (pl.nwg - 120)
                                             : 0.01 * std::min(pl.nwg, 64) +
                                                   0.004 * std::max(pl.nwg - 64, 0);
      const int edges = 2 * (TX * g.P + 2) + 2 * RY * g.P, movers = 64 * std::max(pl.nw - 1, 1);
      const double cost = exchange + (pl.nw > 4 ? second : 0.0) +
                          0.4 * ((edges + movers - 1) / movers) + 0.0005 * g.P * (TX + RY);
      if (best.nwg == 0 || cost < best_cost) {
        best = pl;
        best_cost = cost;
      }
    }
  }
  return best;
}

size_t res_mail_bytes(const Layout& g, int elem_bytes, const ResPlan& pl) {
  const size_t words = 2 * (256 + 8) * 8 +   // the exchanged lines (a fixed place), then the edges
                       (size_t)(elem_bytes / 4) * 2 * ((size_t)pl.nty * g.L + (size_t)pl.ntx * g.NC);
  return (8 * words + 255) / 256 * 256;
}

template <typename T>
int launch_pcg_res(hipStream_t st, const ResLaunch& l) {
  switch (l.g.P) {
#define SEM_RES_CASE(P) case P: return res::launch_res_p<T, P>(st, l);
    SEM_RES_CASE(2) SEM_RES_CASE(3) SEM_RES_CASE(4) SEM_RES_CASE(5) SEM_RES_CASE(6)
    SEM_RES_CASE(7) SEM_RES_CASE(8) SEM_RES_CASE(9) SEM_RES_CASE(10) SEM_RES_CASE(11)
    SEM_RES_CASE(12) SEM_RES_CASE(13) SEM_RES_CASE(14) SEM_RES_CASE(15) SEM_RES_CASE(16)
#undef SEM_RES_CASE
    default:
      set_error("resident PCG supports 2 <= nr == ns <= 16 (got %d)", l.g.P);
      return SEM_ERR_UNSUPPORTED;
  }
}
template int launch_pcg_res<double>(hipStream_t, const ResLaunch&);
template int launch_pcg_res<float>(hipStream_t, const ResLaunch&);

// The compute units that the process's resident solves hold on a device: a launch waits,
// in turn, until it fits beside those that run, since two that do not fit together could
// each hold a part of the CUs and call each other off. Small solves of several contexts
// run side by side so.
namespace {
struct Units {
  std::mutex mu;
  std::condition_variable cv;
  int used = 0;
  unsigned next = 0, turn = 0;
};
struct HeldUnits {
  Units& u;
  const int n;
  HeldUnits(Units& u_, int n_, int all) : u(u_), n(n_) {
    std::unique_lock<std::mutex> lk(u.mu);
    const unsigned mine = u.next++;
    u.cv.wait(lk, [&] { return u.turn == mine && u.used + n <= all; });
    ++u.turn;
    u.used += n;
    u.cv.notify_all();   // (the next one may fit too)
  }
  ~HeldUnits() {
    std::lock_guard<std::mutex> lk(u.mu);
    u.used -= n;
    u.cv.notify_all();
  }
};
constexpr int kDevices = 64;
Units g_units[kDevices];
}  // namespace

int run_resident(sem_ctx* ctx, const sem_operator* op, ResLaunch& l,
                 int (*launch)(hipStream_t, const ResLaunch&), size_t clear_mail, const void* b,
                 int* k_start, PcgHost* hh, hipEvent_t ev_end, bool* called_off) {
  SEM_ARG(reinterpret_cast<uintptr_t>(l.mail) % kMailAlign == 0, "resident PCG: misaligned mail");
  // workgroups go round the XCDs in turn; on one XCD alone they take that one's CUs only,
  // but the next launch may come to the same one
  const int cus = std::min(ctx->ncu, l.plan.near == 1 ? 8 * l.plan.nwg : (l.plan.nwg + 7) / 8 * 8);
  hipStream_t st = ctx->stream;
  // a launch holds the CUs for at most kResIters iterations (about 40 ms)
  constexpr int kResIters = 4096, kResTags = kResIters + 2;
  static_assert(kResTags < 65536, "16-bit tags within a launch");
  l.max_its = kResIters;
  // With the context's own mail the launches take turns with its two blocks of
  // control words, each clearing the other's, and write what the host reads to its
  // pinned memory; else (a caller's workspace) a fill before and a copy after.
  const bool own = clear_mail == 0;
  auto clear_ctl = [&]() -> int {
    SEM_HIP(hipMemsetAsync(ctx->mail_ctl, 0, kMailCtlBytes, st));
    SEM_HIP(hipStreamSynchronize(st));
    return SEM_OK;
  };
  for (;;) {
    const HeldUnits held(g_units[ctx->device % kDevices], cus, ctx->ncu);
    l.b = b;
    l.k_start = *k_start;
    if (own) {
      SEM_TRY(next_mail_tags(ctx, kResTags, &l.tag0));
      auto ctl = [&](unsigned turn) {
        return reinterpret_cast<ResCtl*>(static_cast<char*>(ctx->mail_ctl) +
                                         (turn & 1) * (kMailCtlBytes / 2));
      };
      l.ctl = ctl(ctx->mail_turn);
      l.ctl_next = ctl(++ctx->mail_turn);
      l.host = hh;
      *hh = PcgHost{};
    } else {
      SEM_HIP(hipMemsetAsync(l.mail, 0, clear_mail, st));
      l.tag0 = 0;
      if (l.plan.nwg > 1) SEM_HIP(hipMemsetAsync(l.ctl, 0, sizeof(ResCtl), st));
    }
    if (l.plan.nwg > 1) {
      // test hook: the launch finds itself called off
      if (op->resident == 2 || op->resident == 4 || (op->resident == 5 && !b))
        SEM_HIP(hipMemsetAsync(&l.ctl->decision, 2, 1, st));
      if (op->resident == 3)   // test hook: a group of workgroups on two XCDs
        SEM_HIP(hipMemsetAsync(&l.ctl->xcds[0], 3, 1, st));
    }
    const int ls = launch(st, l);
    if (ls != SEM_OK) {
      if (own) (void)clear_ctl();
      return ls;
    }
    if (ev_end) SEM_HIP(hipEventRecord(ev_end, st));
    if (!own) SEM_HIP(hipMemcpyAsync(hh, l.state, sizeof(PcgHost), hipMemcpyDeviceToHost, st));
    SEM_HIP(hipStreamSynchronize(st));
    if (l.plan.nwg > 1 && hh->ctl.decision != 1) {
      if (own) SEM_TRY(clear_ctl());
      if (op->resident != 2 && op->resident != 5)
        ctx->res_rest = std::chrono::steady_clock::now() + kResRest;
      *called_off = true;
      return SEM_OK;
    }
    if (l.plan.nwg > 1 && hh->ctl.failed) {
      if (own) SEM_TRY(clear_ctl());
      set_error("pcg: a workgroup of the resident solve stopped answering");
      return SEM_ERR_HIP;
    }
    if (hh->state.done) return SEM_OK;
    *k_start = hh->state.iters + 1;
    b = nullptr;
  }
}

}  // namespace sem

// Dispatch of the fused apply over P (2..16); the kernels are instantiated
// per P in k_ax_inst.hip.
#include "k_ax_impl.h"

namespace sem {
namespace ax {
#define SEM_AX_EXTERN(P)                                                                        \
  extern template int launch_apply_p<double, P>(hipStream_t, const Layout&, const ApplyArgs&, \
                                                const PcgLaunch*);                            \
  extern template int launch_apply_p<float, P>(hipStream_t, const Layout&, const ApplyArgs&,  \
                                               const PcgLaunch*);
SEM_AX_EXTERN(2) SEM_AX_EXTERN(3) SEM_AX_EXTERN(4) SEM_AX_EXTERN(5) SEM_AX_EXTERN(6)
SEM_AX_EXTERN(7) SEM_AX_EXTERN(8) SEM_AX_EXTERN(9) SEM_AX_EXTERN(10) SEM_AX_EXTERN(11)
SEM_AX_EXTERN(12) SEM_AX_EXTERN(13) SEM_AX_EXTERN(14) SEM_AX_EXTERN(15) SEM_AX_EXTERN(16)
#undef SEM_AX_EXTERN

template <typename T>
int dispatch(hipStream_t st, const Layout& g, const ApplyArgs& a, const PcgLaunch* pc) {
  switch (g.P) {
    case 2: return launch_apply_p<T, 2>(st, g, a, pc);
    case 3: return launch_apply_p<T, 3>(st, g, a, pc);
    case 4: return launch_apply_p<T, 4>(st, g, a, pc);
    case 5: return launch_apply_p<T, 5>(st, g, a, pc);
    case 6: return launch_apply_p<T, 6>(st, g, a, pc);
    case 7: return launch_apply_p<T, 7>(st, g, a, pc);
    case 8: return launch_apply_p<T, 8>(st, g, a, pc);
    case 9: return launch_apply_p<T, 9>(st, g, a, pc);
    case 10: return launch_apply_p<T, 10>(st, g, a, pc);
    case 11: return launch_apply_p<T, 11>(st, g, a, pc);
    case 12: return launch_apply_p<T, 12>(st, g, a, pc);
    case 13: return launch_apply_p<T, 13>(st, g, a, pc);
    case 14: return launch_apply_p<T, 14>(st, g, a, pc);
    case 15: return launch_apply_p<T, 15>(st, g, a, pc);
    case 16: return launch_apply_p<T, 16>(st, g, a, pc);
    default:
      set_error("fused apply supports 2 <= nr == ns <= 16 (got %d)", g.P);
      return SEM_ERR_UNSUPPORTED;
  }
}

}  // namespace ax

AxPlan make_plan(const Layout& g, bool assemble, bool pcg, int rows, int halo, bool wide,
                 int odd, bool always) {
  AxPlan pl{};
  const int cx = SEM_AX_THREADS / g.P;
  pl.S = assemble ? ax::rows_per_segment(g, cx, pcg, rows) : 1;
  // The assembled FMA apply (P < 16; 16 runs the MFMA forms) takes two
  // element rows side by side where one-row workgroups would be used, the
  // PCG iteration where a two-row sweep would be (it also runs three waves
  // per SIMD there instead of two), strips of odd width up to order odd (not in PCG
  // mode). rows < 0 forces RY = -rows (test hook: 2 or 4; 2 in PCG mode).
  pl.RY = 1;
  if (assemble && g.P < 16) {
    if (rows < 0) {
      const int ry = -rows;
      if ((ry == 2 || (ry == 4 && !pcg)) && cx % ry == 0) pl.RY = ry;
    } else if (rows == 0 && pl.S == (pcg ? 2 : 1) && (cx % 2 == 0 || (!pcg && g.P <= odd)) &&
               g.Ey >= 2) {
      pl.RY = 2;
    }
  }
  if (pl.RY > 1) pl.S = pl.RY;
  pl.CX = cx / pl.RY;
  pl.nstrips = (g.Ex + pl.CX - 1) / pl.CX;
  pl.nsegs = (g.Ey + pl.S - 1) / pl.S;
  pl.nk1 = pl.nstrips * pl.nsegs;
  if (assemble) {
    const int nxs = pl.nstrips - 1 + (g.per_x ? 1 : 0);
    const int nys = pl.nsegs - 1 + (g.per_y ? 1 : 0);
    pl.nxitems = (long)nxs * g.NC;
    pl.total = pl.nxitems + (long)nys * g.L;
    pl.nk2 = (int)((pl.total + 255) / 256);
  }
  // With a halo the workgroups are more (each writes 2 rows of its four, or 6 of eight,
  // and two elements less a row) but their apply is the only launch. While all of them are
  // resident at once it takes little longer: 64x64 elements, P = 4, 160 workgroups,
  // 6.6 -> 3.7 us; 30x30, P = 12, 150 workgroups, 11.1 -> 8.8. Beyond, the repeated
  // work costs more than the seam pass: P = 9, 416 workgroups, 10.2 against 11.0.
  // (One strip and segment need no seams either way: 16 points, 3x1 elements 9.1 us with,
  // 6.6 without.)
  if (assemble && !pcg && rows == 0 && halo > 0 && (pl.total > 0 || always)) {
    const int out = halo_cx(g.P, 4) / 4 - 2, strips = (g.Ex + out - 1) / out;
    for (int ry = 4; ry <= (wide ? 8 : 4); ry += 4) {
      const long groups = (long)strips * ((g.Ey + ry - 3) / (ry - 2));
      if (groups > (ry == 4 ? halo : 256)) continue;
      pl = AxPlan{};
      pl.halo = true;
      pl.CX = out;
      pl.RY = ry;
      pl.S = ry - 2;
      pl.nstrips = strips;
      pl.nsegs = (g.Ey + pl.S - 1) / pl.S;
      pl.nk1 = pl.nstrips * pl.nsegs;
      return pl;
    }
  }
  return pl;
}

template <typename T>
int launch_apply(hipStream_t st, const Layout& g, const ApplyArgs& a) {
  return ax::dispatch<T>(st, g, a, nullptr);
}

template <typename T>
int launch_apply_pcg(hipStream_t st, const Layout& g, const ApplyArgs& a, const PcgLaunch& pc) {
  return ax::dispatch<T>(st, g, a, &pc);
}

template int launch_apply<double>(hipStream_t, const Layout&, const ApplyArgs&);
template int launch_apply<float>(hipStream_t, const Layout&, const ApplyArgs&);
template int launch_apply_pcg<double>(hipStream_t, const Layout&, const ApplyArgs&,
                                      const PcgLaunch&);
template int launch_apply_pcg<float>(hipStream_t, const Layout&, const ApplyArgs&,
                                     const PcgLaunch&);

}  // namespace sem

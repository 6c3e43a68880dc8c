// Instantiates the resident PCG kernels for one P (-DSEM_P=<P>), FP64 and FP32.
#include "k_res.h"

#if !defined(SEM_P)
#error "compile with -DSEM_P=<points per direction>"
#endif

namespace sem {
namespace res {

template <typename T, int P>
int launch_res_p(hipStream_t st, const ResLaunch& l) {
  ResP<T> q{};
  const ApplyArgs& a = *l.a;
  q.b = static_cast<const T*>(l.b);
  q.x = static_cast<T*>(l.x);
  q.r = static_cast<T*>(l.r);
  q.p = static_cast<T*>(l.p);
  q.d = static_cast<const T*>(l.d);
  q.G11 = static_cast<const T*>(a.G11);
  q.G12 = static_cast<const T*>(a.G12);
  q.G22 = static_cast<const T*>(a.G22);
  q.B = static_cast<const T*>(a.B);
  q.nu_f = static_cast<const T*>(a.nu_f);
  q.k_f = static_cast<const T*>(a.k_f);
  q.nu = T(a.nu);
  q.k = T(a.k);
  q.has_mass = a.has_mass;
  q.Ex = l.g.Ex;
  q.Ey = l.g.Ey;
  q.TX = l.plan.TX;
  q.RY = l.plan.RY;
  q.ntx = l.plan.ntx;
  q.nty = l.plan.nty;
  q.per_x = l.g.per_x;
  q.per_y = l.g.per_y;
  q.bc = a.bc;
  u64* m = static_cast<u64*>(l.mail);
  q.slots = m;
  q.ymail = m + kSlotArea;
  q.xmail = q.ymail + Wire<T>::N * 2L * l.plan.nty * l.g.L;
  q.nwg = l.plan.nwg;
  q.near = l.plan.near;
  q.tag0 = l.tag0;
  q.ctl = l.ctl;
  q.ctl_next = l.ctl_next;
  q.host = l.host;
  q.state = l.state;
  q.tol = l.tol;
  q.maxiter = l.maxiter;
  q.k_start = l.k_start;
  q.max_its = l.max_its;
  q.keep = l.keep;
  const dim3 block(64 * l.plan.nw);
  if (l.plan.near == kFlat)
    hipLaunchKernelGGL((k_pcg_res<T, P, false>), dim3(l.plan.nwg), block, 0, st, q);
  else
    hipLaunchKernelGGL((k_pcg_res<T, P, true>),
                       dim3(l.plan.near == kNear ? kGroups * l.plan.nwg : l.plan.nwg), block, 0, st,
                       q);
  SEM_HIP(hipGetLastError());
  return SEM_OK;
}

template int launch_res_p<double, SEM_P>(hipStream_t, const ResLaunch&);
template int launch_res_p<float, SEM_P>(hipStream_t, const ResLaunch&);

}  // namespace res
}  // namespace sem

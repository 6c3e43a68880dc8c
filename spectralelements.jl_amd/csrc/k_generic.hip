// Element operators for any nr x ns blocks (the reference's Mesh(nr, ns, ...)
// takes any order in each direction, mesh.jl:66-133), where the fused strip
// kernels need nr == ns <= 16: one workgroup per element with the block, the
// fluxes and Dr, Ds in LDS, then QQ' and the mask through the sorted map. And
// PCG with such an operator (pcg.jl:16-60; host-driven, device vectors).
#include <algorithm>
#include <cmath>

#include "sem_device.h"

namespace sem {
namespace {

inline int nblk(long n, int bs = 256) { return (int)((n + bs - 1) / bs); }

constexpr int kGenThreads = 256;

// H = nu [Dr'(G11 ur + G12 us) + (G12 ur + G22 us) Ds] + k B u per element
// (laplace, lapl.jl:70-81; hlmz.jl:12-19): ur = Dr u, us = u Ds'.
__global__ void __launch_bounds__(kGenThreads)
k_ax_generic(const double* __restrict__ u, double* __restrict__ y,
             const double* __restrict__ G11, const double* __restrict__ G12,
             const double* __restrict__ G22, const double* __restrict__ B,
             const double* __restrict__ Dr, const double* __restrict__ Ds, double nu,
             const double* __restrict__ nu_f, double kc, const double* __restrict__ k_f,
             int has_mass, int nr, int ns, int Ex, int L) {
  extern __shared__ double sh[];
  const int ne = nr * ns;
  double* su = sh;               // u block (a + nr b)
  double* swr = su + ne;         // wr
  double* sws = swr + ne;        // ws
  double* sdr = sws + ne;        // Dr (nr x nr, column-major)
  double* sds = sdr + nr * nr;   // Ds (ns x ns)
  const int e = blockIdx.x;
  const int ex = e % Ex, ey = e / Ex;
  const long base = (long)ex * nr + (long)L * ((long)ey * ns);
  for (int q = threadIdx.x; q < nr * nr; q += kGenThreads) sdr[q] = Dr[q];
  for (int q = threadIdx.x; q < ns * ns; q += kGenThreads) sds[q] = Ds[q];
  for (int q = threadIdx.x; q < ne; q += kGenThreads) {
    const int a = q % nr, b = q / nr;
    su[q] = u[base + a + (long)L * b];
  }
  __syncthreads();
  for (int q = threadIdx.x; q < ne; q += kGenThreads) {
    const int a = q % nr, b = q / nr;
    double ur = 0.0, us = 0.0;
    for (int k = 0; k < nr; ++k) ur += sdr[a + nr * k] * su[k + nr * b];
    for (int k = 0; k < ns; ++k) us += su[a + nr * k] * sds[b + ns * k];
    const long t = base + a + (long)L * b;
    swr[q] = G11[t] * ur + G12[t] * us;
    sws[q] = G12[t] * ur + G22[t] * us;
  }
  __syncthreads();
  for (int q = threadIdx.x; q < ne; q += kGenThreads) {
    const int a = q % nr, b = q / nr;
    double p1 = 0.0, p2 = 0.0;
    for (int k = 0; k < nr; ++k) p1 += sdr[k + nr * a] * swr[k + nr * b];
    for (int k = 0; k < ns; ++k) p2 += sws[a + nr * k] * sds[k + ns * b];
    const long t = base + a + (long)L * b;
    double h = (nu_f ? nu_f[t] : nu) * (p1 + p2);
    if (has_mass) h = h + (k_f ? k_f[t] : kc) * (B[t] * su[q]);
    y[t] = h;
  }
}

// The same for ns <= kRowMax: a thread holds row a of an element in registers, all
// ns columns of it, and a workgroup takes as many elements as it has rows for. The
// s-direction runs in registers with coefficients from scalar loads; the
// r-direction reads the element's rows from LDS, one read per multiply-add and
// broadcast to the element's threads. Bound by memory and the latency of the phases.
// The form above, an element per workgroup and two LDS reads per multiply-add, has
// the shorter chain while all elements are resident at once, and is left for longer
// rows, whose registers hold this one to a wave per SIMD. hlmz, us, above / here: 4x7
// points, 160x160 elements 39.9 / 6.9; 12x9, 90x90 20.8 / 11.6, 30x30 6.0 / 6.9; 7x14,
// 90x90 22.0 / 14.0, 45x45 7.2 / 10.2; 17x17, 64x64 28.8 / 36.7.
constexpr int kRowMax = 16;
typedef const double __attribute__((address_space(4)))* ConstD;   // scalar loads
struct RowP {
  const double *u, *G11, *G12, *G22, *B, *Dr, *Ds, *nu_f, *k_f;
  double* y;
  double nu, k;
  int has_mass, nr, Ex, E, ne;
};

template <int NS>
__global__ void __launch_bounds__(kGenThreads) k_ax_rows(const RowP q) {
  extern __shared__ double sh[];
  const int nr = q.nr, ne = q.ne, Ex = q.Ex, tid = threadIdx.x;
  const int RS = (ne * nr) | 1;
  double* const sdr = sh + NS * RS;
  const long L = (long)nr * Ex;
  const int e = tid / nr, a = tid - e * nr;
  const int g = blockIdx.x * ne + e;
  const bool act = g < q.E;
  const int g1 = act ? g : q.E - 1;   // (loads without branches)
  const long base = (long)(g1 % Ex) * nr + a + L * ((long)(g1 / Ex) * NS);
  ConstD Ds = (ConstD)(unsigned long long)q.Ds;
  double u[NS], us[NS], g11[NS], g12[NS], g22[NS];
#pragma unroll
  for (int b = 0; b < NS; ++b) u[b] = q.u[base + L * b];
#pragma unroll
  for (int b = 0; b < NS; ++b) {
    g11[b] = q.G11[base + L * b];
    g12[b] = q.G12[base + L * b];
    g22[b] = q.G22[base + L * b];
  }
  for (int t = tid; t < nr * nr; t += blockDim.x) sdr[t] = q.Dr[t];
#pragma unroll
  for (int b = 0; b < NS; ++b) sh[b * RS + tid] = u[b];
#pragma unroll
  for (int b = 0; b < NS; ++b) us[b] = 0.0;
#pragma unroll
  for (int k = 0; k < NS; ++k)
#pragma unroll
    for (int b = 0; b < NS; ++b) us[b] += u[k] * Ds[b + NS * k];
  __syncthreads();
  const double* const row = sh + e * nr;   // the element's rows, column by column
  double h[NS];
#pragma unroll
  for (int b = 0; b < NS; ++b) h[b] = 0.0;
  for (int k = 0; k < nr; ++k) {
    const double d = sdr[a + nr * k];
#pragma unroll
    for (int b = 0; b < NS; ++b) h[b] += d * row[b * RS + k];
  }
  __syncthreads();
#pragma unroll
  for (int b = 0; b < NS; ++b) {
    sh[b * RS + tid] = g11[b] * h[b] + g12[b] * us[b];
    us[b] = g12[b] * h[b] + g22[b] * us[b];
  }
  // mass and coefficients on their way (a missing field reads G11)
  const double* const bs = q.has_mass ? q.B : q.G11;
  double bm[NS], nf[NS], kf[NS];
#pragma unroll
  for (int b = 0; b < NS; ++b) bm[b] = bs[base + L * b];
  if (q.nu_f) {
#pragma unroll
    for (int b = 0; b < NS; ++b) nf[b] = q.nu_f[base + L * b];
  }
  if (q.k_f) {
#pragma unroll
    for (int b = 0; b < NS; ++b) kf[b] = q.k_f[base + L * b];
  }
#pragma unroll
  for (int b = 0; b < NS; ++b) h[b] = us[0] * Ds[NS * b];
#pragma unroll
  for (int k = 1; k < NS; ++k)
#pragma unroll
    for (int b = 0; b < NS; ++b) h[b] += us[k] * Ds[k + NS * b];
  __syncthreads();
  for (int k = 0; k < nr; ++k) {
    const double d = sdr[k + nr * a];
#pragma unroll
    for (int b = 0; b < NS; ++b) h[b] += d * row[b * RS + k];
  }
  if (!act) return;
#pragma unroll
  for (int b = 0; b < NS; ++b) {
    double v = (q.nu_f ? nf[b] : q.nu) * h[b];
    if (q.has_mass) v = v + (q.k_f ? kf[b] : q.k) * (bm[b] * u[b]);
    q.y[base + L * b] = v;
  }
}

// Where it is taken, from sweeps over nr = 2 to 30, ns = 2 to 16 and 12 to 14400 elements:
// with few elements the one above takes 4.4 to 5 us whatever the block, this one as long only
// for the smallest. The line lies at 1600 to 2000 elements for rows of up to 8, for more
// at 2000 to 4000 as they grow longer, and at 900 to 1500 with 16 and more rows (above / here,
// us: 24x8 points, 100 elements 5.2 / 8.9, 1980 16.1 / 9.3; 12x8, 100 4.5 / 6.2, 4096 11.5 /
// 6.8; 4x12, 1980 5.2 / 7.2, 4096 9.4 / 7.5). Rows of 16 leave a workgroup a CU: in several
// rounds of them the last is to be at least three quarters of the CUs or so (12x16, 6320
// elements in 301 workgroups 25.0 / 30.5, 14400 in 686 50.2 / 44.4).
inline bool rows_better(int nr, int ns, long E) {
  if (ns <= 6 && nr * ns <= 40) return true;
  if (E < (nr >= 16 ? 1400 : ns <= 8 ? 2048 : 256 * ns)) return false;
  const long wgs = (E + kGenThreads / nr - 1) / (kGenThreads / nr), rounds = (wgs + 255) / 256;
  return ns < 16 || rounds == 1 || 4 * wgs >= 3 * 256 * rounds;
}

template <int NS>
void launch_rows(hipStream_t st, int ns, const RowP& q, size_t lds) {
  if constexpr (NS >= 2) {
    if (ns == NS)
      hipLaunchKernelGGL(k_ax_rows<NS>, dim3((q.E + q.ne - 1) / q.ne), dim3(q.ne * q.nr), lds, st, q);
    else
      launch_rows<NS - 1>(st, ns, q, lds);
  }
}

__global__ void k_copy_scale(const double* __restrict__ a, const double* __restrict__ d,
                             double* __restrict__ z, long n) {
  const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t < n) z[t] = d ? d[t] * a[t] : a[t];
}

// x += alpha p, r -= alpha w
__global__ void k_gen_xr(double* __restrict__ x, double* __restrict__ r,
                         const double* __restrict__ p, const double* __restrict__ w, double alpha,
                         long n) {
  const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t < n) {
    x[t] = x[t] + alpha * p[t];
    r[t] = r[t] - alpha * w[t];
  }
}

}  // namespace

int launch_apply_generic(hipStream_t st, const sem_mesh* m, const double* u, double* y,
                         const double* G11, const double* G12, const double* G22,
                         const double* B, double nu, const double* nu_f, double k,
                         const double* k_f, int has_mass, int assemble, int bits) {
  const int nr = m->nr, ns = m->ns;
  const size_t lds = sizeof(double) * (3 * (size_t)nr * ns + (size_t)nr * nr + (size_t)ns * ns);
  if (lds > 64 * 1024) {
    set_error("element operators support nr * ns blocks up to 64 KiB of LDS (got %d x %d)", nr,
              ns);
    return SEM_ERR_UNSUPPORTED;
  }
  if (ns >= 2 && ns <= kRowMax && nr <= kGenThreads &&
      rows_better(nr, ns, (long)m->Ex * m->Ey)) {
    RowP q{u, G11, G12, G22, B, m->Dr, m->Ds, nu_f, k_f, y, nu, k, has_mass, nr, m->Ex,
           m->Ex * m->Ey, kGenThreads / nr};
    const size_t rows = sizeof(double) * ((size_t)ns * ((q.ne * nr) | 1) + (size_t)nr * nr);
    if (rows <= 65536) {
      launch_rows<kRowMax>(st, ns, q, rows);
      if (assemble) SEM_TRY(launch_gsmap_masked(st, m->map, m->layout(), bits, y, y));
      SEM_HIP(hipGetLastError());
      return SEM_OK;
    }
  }
  hipLaunchKernelGGL(k_ax_generic, dim3(m->Ex * m->Ey), dim3(kGenThreads), lds, st, u, y, G11,
                     G12, G22, B, m->Dr, m->Ds, nu, nu_f, k, k_f, has_mass, nr, ns, m->Ex, m->L);
  SEM_HIP(hipGetLastError());
  if (assemble) SEM_TRY(launch_gsmap_masked(st, m->map, m->layout(), bits, y, y));
  return SEM_OK;
}

// pcg.jl:16-60 with a generic operator: x0 = 0, stop when norm(r, Inf) <= tol,
// inner products weighted by the mesh's mult, z = d .* r (or r): in one launch
// where the mesh fits the chip's registers, else with the scalars read on the
// host every iteration.
int pcg_generic(sem_ctx* ctx, const sem_operator* op, const double* d, const double* b, double* x,
                double tol, int maxiter, sem_pcg_info* info) {
  SEM_ARG(op->precision == SEM_F64, "pcg: meshes with nr != ns or nr > %d need SEM_F64", kMaxP);
  const sem_mesh* m = op->mesh;
  const long n = (long)m->nl;
  hipStream_t st = ctx->stream;
  const size_t vb = ((sizeof(double) * n + 255) / 256) * 256;
  constexpr int kParts = 256;
  SEM_TRY(ensure_ws(ctx, 4 * vb + sizeof(double) * (kParts + 1) + 512));
  SEM_TRY(ensure_pinned(ctx, 256));
  char* w0 = static_cast<char*>(ctx->ws);
  double* r = reinterpret_cast<double*>(w0);
  double* p = reinterpret_cast<double*>(w0 + vb);
  double* w = reinterpret_cast<double*>(w0 + 2 * vb);
  double* z = reinterpret_cast<double*>(w0 + 3 * vb);
  double* part = reinterpret_cast<double*>(w0 + 4 * vb);
  double* hv = reinterpret_cast<double*>(static_cast<char*>(ctx->pinned) + 64);
  const double* mult = m->f[SEM_MULT];
  auto fetch = [&](double* out) -> int {
    SEM_HIP(hipMemcpyAsync(hv, part + kParts, sizeof(double), hipMemcpyDeviceToHost, st));
    SEM_HIP(hipStreamSynchronize(st));
    *out = *hv;
    return SEM_OK;
  };
  auto dot = [&](const double* a, const double* c, double* out) -> int {
    SEM_TRY(launch_dot(st, n, a, c, mult, part, kParts, part + kParts));
    return fetch(out);
  };
  auto norm = [&](const double* a, double* out) -> int {
    SEM_TRY(launch_norm_inf(st, n, a, part, kParts, part + kParts));
    return fetch(out);
  };
  SEM_HIP(hipEventRecord(ctx->ev0, st));
  int k = 0;
  double res = 0.0, t = 0.0, t_prev = 1.0;
  // the whole solve in one launch where the mesh fits (k_res_gen.hip)
  ResPlan rp = may_be_resident(ctx, op) ? res_gen_plan(m->layout(), m->nr, m->ns, ctx->ncu) : ResPlan{};
  // (no memory for the mail: the steps below need none)
  if (rp.nwg > 0 &&
      ensure_mail(ctx, res_mail_bytes(m->layout(), (int)sizeof(double), rp)) != SEM_OK) {
    (void)hipGetLastError();
    rp = ResPlan{};
  }
  if (rp.nwg > 0) {
    ApplyArgs aa = args_of(op, nullptr, nullptr);
    aa.bc = op->desc.bc_bits;
    PcgHost* hh = static_cast<PcgHost*>(ctx->pinned);
    ResLaunch l{};
    l.g = m->layout();
    l.mesh = m;
    l.plan = rp;
    l.a = &aa;
    l.x = x;
    l.r = r;
    l.p = p;
    l.d = d;
    l.mail = ctx->mail;
    l.state = reinterpret_cast<PcgState*>(w0 + 4 * vb + ((sizeof(double) * (kParts + 1) + 255) / 256) * 256);
    l.ctl = reinterpret_cast<ResCtl*>(l.state + 1);
    l.tol = tol;
    l.maxiter = maxiter;
    int k_start = 1;
    bool called_off = false;
    SEM_TRY(run_resident(ctx, op, l, launch_pcg_res_gen, 0, b, &k_start, hh, ctx->ev1, &called_off));
    // a solve whose launch was called off goes on from there with the steps below
    if (called_off && k_start > 1) {
      PcgState s;
      SEM_HIP(hipMemcpyAsync(&s, l.state, sizeof(s), hipMemcpyDeviceToHost, st));
      SEM_HIP(hipStreamSynchronize(st));
      k = k_start - 1;
      t_prev = s.t[k & 1];
      tol = s.tol_eff;
    }
    if (!called_off) {
      float ms = 0.f;
      SEM_HIP(hipEventElapsedTime(&ms, ctx->ev0, ctx->ev1));
      const PcgState& s = hh->state;
      if (info) {
        info->iters = s.iters;
        info->converged = s.converged;
        info->res = s.res;
        info->elapsed_ms = ms;
        info->outer = 0;
        info->inner_total = s.iters;
      }
      if (!std::isfinite(s.res)) {
        set_error("pcg: residual is not finite after %d iterations", s.iters);
        return SEM_ERR_NONFINITE;
      }
      return s.converged ? SEM_OK : SEM_WARN_MAXITER;
    }
  }
  if (k == 0) {
    SEM_HIP(hipMemsetAsync(x, 0, sizeof(double) * n, st));
    SEM_HIP(hipMemcpyAsync(r, b, sizeof(double) * n, hipMemcpyDeviceToDevice, st));
  }
  SEM_TRY(norm(r, &res));
  if (tol < 0.0) tol = -tol * res;   // relative stop test
  bool conv = true;
  while (res > tol) {
    if (k == maxiter) {
      conv = false;
      break;
    }
    ++k;
    hipLaunchKernelGGL(k_copy_scale, dim3(nblk(n)), dim3(256), 0, st, r, d, z, n);
    SEM_TRY(dot(r, z, &t));
    if (k == 1) {
      SEM_HIP(hipMemcpyAsync(p, z, sizeof(double) * n, hipMemcpyDeviceToDevice, st));
    } else {
      SEM_TRY(launch_axpby(st, n, 1.0, z, t / t_prev, p, p));
    }
    SEM_TRY(sem_operator_apply(ctx, op, p, w));
    double pw = 0.0;
    SEM_TRY(dot(p, w, &pw));
    hipLaunchKernelGGL(k_gen_xr, dim3(nblk(n)), dim3(256), 0, st, x, r, p, w, t / pw, n);
    SEM_HIP(hipGetLastError());
    SEM_TRY(norm(r, &res));
    t_prev = t;
    if (!std::isfinite(res)) break;
  }
  SEM_HIP(hipEventRecord(ctx->ev1, st));
  SEM_HIP(hipEventSynchronize(ctx->ev1));
  float ms = 0.f;
  SEM_HIP(hipEventElapsedTime(&ms, ctx->ev0, ctx->ev1));
  if (info) {
    info->iters = k;
    info->converged = conv && res <= tol;
    info->res = res;
    info->elapsed_ms = ms;
    info->outer = 0;
    info->inner_total = k;
  }
  if (!std::isfinite(res)) {
    set_error("pcg: residual is not finite after %d iterations", k);
    return SEM_ERR_NONFINITE;
  }
  return (conv && res <= tol) ? SEM_OK : SEM_WARN_MAXITER;
}

}  // namespace sem

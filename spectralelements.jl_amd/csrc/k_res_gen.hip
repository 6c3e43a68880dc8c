// Resident PCG for element blocks of any nr x ns (the meshes the strip kernels do
// not take) and for diagonals that differ between the copies of a node: the
// scheme of k_res.h with the block sizes at run time. A workgroup owns a tile of
// whole elements; thread t holds nodes t, t + NT, ... of the tile in registers, and
// the contractions read the tile's u, wr and ws and the two derivative matrices from
// LDS. (With three or four nodes a thread, 36 to 39 of 256 registers are spilled to
// scratch, some 25 loads of them in an iteration.) <p, A p> is formed on the
// assembled A p (pcg.jl:50), so the edges travel first and the sum after them: three
// exchanges in a row instead of two.
//
// Why: the host-driven recurrence took 11 launches and 3 host waits per
// iteration, 73 us at 20x14 elements of 12x9 points, of which the device
// worked 24.
#include <algorithm>
#include <type_traits>

#include "k_res.h"

namespace sem {
namespace res {

constexpr int kGenThreads = 512;
constexpr int kGenMaxNodes = 4;      // nodes per thread
constexpr size_t kGenLds = 63 * 1024;   // (and the static part)

struct GenP {
  const double* __restrict__ b;
  double* __restrict__ x;
  double* __restrict__ r;
  double* __restrict__ p;
  const double* __restrict__ d;
  const double* __restrict__ G11;
  const double* __restrict__ G12;
  const double* __restrict__ G22;
  const double* __restrict__ B;
  const double* __restrict__ nu_f;
  const double* __restrict__ k_f;
  const double* __restrict__ Dr;
  const double* __restrict__ Ds;
  double nu, k;
  int has_mass, nr, ns;
  int Ex, Ey, TX, RY, ntx, nty, per_x, per_y, bc;
  u64* ymail;
  u64* xmail;
  u64* slots;
  int nwg, near;
  unsigned tag0;
  ResCtl *ctl, *ctl_next;
  PcgState* state;
  PcgHost* host;
  double tol;
  int maxiter, k_start, max_its;
};

// doubles of LDS for a tile of TX x RY elements: u (then H), wr, ws, Dr, Ds, the
// lines of the neighbouring tiles (y-lines with their end rows), a zero
__host__ __device__ constexpr int gen_lds_doubles(int nr, int ns, int TX, int RY) {
  return 3 * TX * RY * nr * ns + nr * nr + ns * ns + 2 * (TX * nr + 2) + 2 * RY * ns + 1;
}

__device__ __forceinline__ double await_word(const u64* s, int plane, unsigned tag, int* lost) {
  Wire<double> w;
  int n = 0;
  do w.load(s, plane);
  while (!w.ok(tag) && ++n < kResPolls);
  if (!w.ok(tag)) *lost = 1;
  return w.value();
}

template <int K, bool NEAR>   // NEAR: as in k_pcg_res
__global__ void __launch_bounds__(kGenThreads) k_pcg_res_gen(const GenP prm) {
  extern __shared__ double lds[];
  constexpr int NW = kGenThreads / 64;
  __shared__ double red[2][NW], bc[3];
  __shared__ int go, lost;
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, NT = blockDim.x;
  if (NEAR && prm.near == kNear && blockIdx.x % kGroups) return;
  const int nwg = prm.nwg, wg = NEAR && prm.near == kNear ? blockIdx.x / kGroups : blockIdx.x;
  if (tid == 0) lost = 0;
  if (nwg > 1) arrive(prm.ctl, prm.slots, prm.tag0, nwg, wg, NEAR ? prm.near : (int)kFlat);

  const int nr = prm.nr, ns = prm.ns, ne = nr * ns;
  const int Ex = prm.Ex, Ey = prm.Ey, ntx = prm.ntx, nty = prm.nty;
  const int L = nr * Ex, NC = ns * Ey;
  const int tx = wg % ntx, ty = wg / ntx;
  const int nex = min(prm.TX, Ex - tx * prm.TX), ney = min(prm.RY, Ey - ty * prm.RY);
  const int nt = nex * ney * ne;          // the tile's nodes
  const int wy = nex * nr, wx = ney * ns; // lengths of its edges
  double* const su = lds;
  double* const swr = su + nt;
  double* const sws = swr + nt;
  double* const sdr = sws + nt;
  double* const sds = sdr + nr * nr;
  const int oHY = 3 * nt + nr * nr + ns * ns, oHX = oHY + 2 * (wy + 2), oZ = oHX + 2 * wx;
  for (int q = tid; q < nr * nr; q += NT) sdr[q] = prm.Dr[q];
  for (int q = tid; q < ns * ns; q += NT) sds[q] = prm.Ds[q];
  if (tid == 0) lds[oZ] = 0.0;

  // this thread's nodes: their fields, weights, and the places in LDS of the
  // partner copies across x, across y and across both (the zero where none)
  double r[K], p[K], x[K], d[K], g11[K], g12[K], g22[K], bm[K], nv[K], kv[K], mw[K], on[K];
  int qn[K], ix[K], iy[K], ic[K];
#pragma unroll
  for (int j = 0; j < K; ++j) {
    const int q = tid + j * NT;
    const bool act = q < nt;
    const int qq = act ? q : 0;
    qn[j] = act ? q : -1;
    const int el = qq / ne, w = qq - el * ne;
    const int hh = el / nex, e = el - hh * nex, b = w / nr, a = w - b * nr;
    const int ex = tx * prm.TX + e, ey = ty * prm.RY + hh;
    const int i = ex * nr + a, jj = ey * ns + b, t = i + L * jj;
    g11[j] = prm.G11[t];
    g12[j] = prm.G12[t];
    g22[j] = prm.G22[t];
    bm[j] = prm.has_mass ? prm.B[t] : 0.0;
    nv[j] = prm.nu_f ? prm.nu_f[t] : prm.nu;
    kv[j] = prm.k_f ? prm.k_f[t] : prm.k;
    d[j] = prm.d ? prm.d[t] : 1.0;
    r[j] = prm.b ? prm.b[t] : prm.r[t];
    x[j] = prm.b ? 0.0 : prm.x[t];
    p[j] = prm.k_start > 1 ? prm.p[t] : 0.0;
    // partners: element and node across x (exn, an), across y (eyn, bn)
    int exn = -1, eyn = -1, an = a, bn = b;
    if (a == 0 && (ex > 0 || prm.per_x)) exn = ex > 0 ? ex - 1 : Ex - 1, an = nr - 1;
    if (a == nr - 1 && (ex < Ex - 1 || prm.per_x)) exn = ex < Ex - 1 ? ex + 1 : 0, an = 0;
    if (b == 0 && (ey > 0 || prm.per_y)) eyn = ey > 0 ? ey - 1 : Ey - 1, bn = ns - 1;
    if (b == ns - 1 && (ey < Ey - 1 || prm.per_y)) eyn = ey < Ey - 1 ? ey + 1 : 0, bn = 0;
    const int sx = a == 0 ? 0 : 1, sy = b == 0 ? 0 : 1;   // the side a partner lies on
    const bool xin = exn >= 0 && exn / prm.TX == tx, yin = eyn >= 0 && eyn / prm.RY == ty;
    const int en = xin ? exn - tx * prm.TX : 0, hn = yin ? eyn - ty * prm.RY : 0;
    auto node = [&](int e_, int h_, int a_, int b_) { return (e_ + nex * h_) * ne + a_ + nr * b_; };
    ix[j] = iy[j] = ic[j] = oZ;
    if (exn >= 0) ix[j] = xin ? node(en, hh, an, b) : oHX + sx * wx + hh * ns + b;
    if (eyn >= 0) iy[j] = yin ? node(e, hn, a, bn) : oHY + sy * (wy + 2) + e * nr + a + 1;
    if (exn >= 0 && eyn >= 0)
      ic[j] = yin ? (xin ? node(en, hn, an, bn) : oHX + sx * wx + hn * ns + bn)
                  : oHY + sy * (wy + 2) + (xin ? en * nr + an + 1 : sx == 0 ? 0 : wy + 1);
    mw[j] = act ? (exn >= 0 ? 0.5 : 1.0) * (eyn >= 0 ? 0.5 : 1.0) : 0.0;
    on[j] = act && mask_on(i, jj, L, NC, prm.bc) ? 1.0 : 0.0;
    if (!act) r[j] = x[j] = p[j] = 0.0;
  }

  int mode = kFlat;
  if (nwg > 1) {
    const int m = decide(prm.ctl, NEAR ? prm.near : (int)kFlat, &go);
    if (m < 0) return;
    if (NEAR) mode = m;
  }
  auto total = [&](double* v, bool two) {   // wave 0: the workgroup's sum (and maximum)
    const bool in = lane < (NT >> 6);
    v[0] = sum_first8(in ? red[0][lane & (NW - 1)] : 0.0);
    if (two) v[1] = max_first8(in ? red[1][lane & (NW - 1)] : 0.0);
  };
  auto reduce_r = [&](unsigned tag, double* t, double* res) {
    double rho = 0.0, m = 0.0;
#pragma unroll
    for (int j = 0; j < K; ++j) {
      rho += r[j] * (d[j] * r[j]) * mw[j];
      m = fmax(m, fabs(r[j]));
    }
    rho = sum_wave(rho);
    m = max_wave(m);
    if (lane == 0) {
      red[0][wv] = rho;
      red[1][wv] = m;
    }
    __syncthreads();
    if (wv == 0) {
      double v[2];
      total(v, true);
      bool ok = true;
      if (nwg > 1) {
        u64* const s = prm.slots + kMaxWg * kSlotWords;
        exch_post<2>(s + line_of(wg, mode) * kSlotWords, lane, tag, v, stays(mode));
        ok = exch_wait<2>(s, s + (kMaxWg + kGroups) * kSlotWords, nwg, wg, mode, lane, tag, v);
      }
      if (lane == 0) {
        bc[1] = v[0];
        bc[2] = v[0] != v[0] ? v[0] : v[1];
        if (!ok) lost = 1;
      }
    }
    __syncthreads();
    *t = uniform(bc[1]);
    *res = uniform(bc[2]);
  };

  const int yplane = 2 * nty * L, xplane = 2 * ntx * NC;
  unsigned tag = prm.tag0 + 1;
  double t, res, t_prev = 1.0;
  reduce_r(tag, &t, &res);
  int k = prm.k_start;
  double tol = prm.tol;
  if (tol < 0.0) tol = k == 1 ? -tol * res : uniform(prm.state->tol_eff);
  if (k > 1) t_prev = uniform(prm.state->t[(k - 1) & 1]);
  bool done = false;
  for (;;) {
    done = !(res > tol) || k - 1 == prm.maxiter;
    if (done || k - prm.k_start == prm.max_its || __builtin_amdgcn_readfirstlane(lost)) break;
    ++tag;
    const double beta = k == 1 ? 0.0 : uniform(t / t_prev);
#pragma unroll
    for (int j = 0; j < K; ++j) {
      p[j] = d[j] * r[j] + beta * p[j];
      if (qn[j] >= 0) su[qn[j]] = p[j];
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < K; ++j)
      if (qn[j] >= 0) {
        const int el = qn[j] / ne, w = qn[j] - el * ne, b = w / nr, a = w - b * nr;
        const double* u = su + el * ne;
        double ur = 0.0, us = 0.0;
#pragma unroll 4
        for (int q = 0; q < nr; ++q) ur += sdr[a + nr * q] * u[q + nr * b];
#pragma unroll 4
        for (int q = 0; q < ns; ++q) us += u[a + nr * q] * sds[b + ns * q];
        swr[qn[j]] = g11[j] * ur + g12[j] * us;
        sws[qn[j]] = g12[j] * ur + g22[j] * us;
      }
    __syncthreads();
    double h[K];
#pragma unroll
    for (int j = 0; j < K; ++j) {
      h[j] = 0.0;
      if (qn[j] >= 0) {
        const int el = qn[j] / ne, w = qn[j] - el * ne, b = w / nr, a = w - b * nr;
        const double* ur = swr + el * ne;
        const double* us = sws + el * ne;
        double p1 = 0.0, p2 = 0.0;
#pragma unroll 4
        for (int q = 0; q < nr; ++q) p1 += sdr[q + nr * a] * ur[q + nr * b];
#pragma unroll 4
        for (int q = 0; q < ns; ++q) p2 += us[a + nr * q] * sds[q + ns * b];
        h[j] = nv[j] * (p1 + p2);
        if (prm.has_mass) h[j] = h[j] + kv[j] * (bm[j] * p[j]);
        su[qn[j]] = h[j];   // (p's copies there are no longer read)
      }
    }
    __syncthreads();
    // edges out and in
    if (nwg > 1) {
      for (int q = tid; q < 2 * (wy + wx); q += NT) {
        int m = q;
        const bool isy = m < 2 * wy;
        if (!isy) m -= 2 * wy;
        const int w = isy ? wy : wx;
        const int up = m >= w ? 1 : 0;
        m -= up * w;
        if (isy ? nty == 1 : ntx == 1) continue;
        if (isy) {
          const int e = m / nr, a = m - e * nr;
          post<double>(prm.ymail + ((2 * ty + up) * L + tx * prm.TX * nr + m), yplane, tag,
                       su[(e + (up ? nex * (ney - 1) : 0)) * ne + a + (up ? nr * (ns - 1) : 0)],
                       mode == kNear);
        } else {
          const int hh = m / ns, b = m - hh * ns;
          post<double>(prm.xmail + ((2 * tx + up) * NC + ty * prm.RY * ns + m), xplane, tag,
                       su[((up ? nex - 1 : 0) + nex * hh) * ne + (up ? nr - 1 : 0) + nr * b],
                       mode == kNear);
        }
      }
      for (int q = tid; q < 2 * (wy + 2 + wx); q += NT) {
        int m = q;
        const bool isy = m < 2 * (wy + 2);
        if (!isy) m -= 2 * (wy + 2);
        const int w = isy ? wy + 2 : wx;
        const int up = m >= w ? 1 : 0;
        m -= up * w;
        if (isy ? nty == 1 : ntx == 1) continue;
        if (isy) {
          int s = up ? ty + 1 : ty - 1, pos = tx * prm.TX * nr + m - 1;
          if (!prm.per_y && (s < 0 || s >= nty)) continue;
          if (!prm.per_x && (pos < 0 || pos >= L)) continue;
          s = s < 0 ? nty - 1 : s >= nty ? 0 : s;
          pos = pos < 0 ? L - 1 : pos >= L ? 0 : pos;
          lds[oHY + up * (wy + 2) + m] =
              await_word(prm.ymail + ((2 * s + 1 - up) * L + pos), yplane, tag, &lost);
        } else {
          int s = up ? tx + 1 : tx - 1;
          if (!prm.per_x && (s < 0 || s >= ntx)) continue;
          s = s < 0 ? ntx - 1 : s >= ntx ? 0 : s;
          lds[oHX + up * wx + m] = await_word(
              prm.xmail + ((2 * s + 1 - up) * NC + ty * prm.RY * ns + m), xplane, tag, &lost);
        }
      }
      __syncthreads();
    }
    // QQ' (x-pairs, then y-pairs), the mask, and <p, A p>_mult
    double dot = 0.0;
#pragma unroll
    for (int j = 0; j < K; ++j) {
      h[j] = ((h[j] + lds[ix[j]]) + (lds[iy[j]] + lds[ic[j]])) * on[j];
      dot += p[j] * h[j] * mw[j];
    }
    dot = sum_wave(dot);
    if (lane == 0) red[0][wv] = dot;
    __syncthreads();
    if (wv == 0) {
      double v[1];
      total(v, false);
      bool ok = true;
      if (nwg > 1) {
        exch_post<1>(prm.slots + line_of(wg, mode) * kSlotWords, lane, tag, v,
                     stays(mode));
        ok = exch_wait<1>(prm.slots, prm.slots + 2 * kMaxWg * kSlotWords, nwg, wg, mode, lane,
                          tag, v);
      }
      if (lane == 0) {
        bc[0] = v[0];
        if (!ok) lost = 1;
      }
    }
    __syncthreads();
    const double alpha = uniform(t / bc[0]);
#pragma unroll
    for (int j = 0; j < K; ++j) {
      x[j] = x[j] + alpha * p[j];
      r[j] = r[j] - alpha * h[j];
    }
    t_prev = t;
    reduce_r(tag, &t, &res);
    ++k;
  }
  const bool failed = lost != 0;
#pragma unroll
  for (int j = 0; j < K; ++j)
    if (qn[j] >= 0) {
      const int el = qn[j] / ne, w = qn[j] - el * ne;
      const int hh = el / nex, e = el - hh * nex, b = w / nr, a = w - b * nr;
      const int q = (tx * prm.TX + e) * nr + a + L * ((ty * prm.RY + hh) * ns + b);
      prm.x[q] = x[j];
      if (!done) {
        prm.r[q] = r[j];
        prm.p[q] = p[j];
      }
    }
  if (wg == 0) {
    PcgState* st = prm.state;
    if (tid == 0) {
      st->iters = k - 1;
      st->converged = done && res <= tol ? 1 : 0;
      st->res = res;
      if (k > prm.k_start) st->t[(k - 1) & 1] = t_prev;
      st->tol_eff = tol;
      st->done = done && !failed ? 1 : 0;
    }
    report(prm.host, prm.ctl_next, st, tid);
  }
  if (failed && tid == 0) {
    atomicExch(&prm.ctl->failed, 1);
    if (prm.host) prm.host->ctl.failed = 1;
  }
}

}  // namespace res

// Tiles of whole elements with at most four nodes per thread and 63 KiB of LDS,
// one workgroup per CU. The contractions cost nodes per thread times (nr + ns); the
// exchanges of an iteration are 1.3 us dearer over 256 workgroups than over 128.
ResPlan res_gen_plan(const Layout& g, int nr, int ns, int ncu) {
  const int ne = nr * ns, max_wg = std::min(ncu, res::kMaxWg);
  ResPlan best{};
  if ((long)g.L * g.NC >= (1L << 31) / 4) return best;
  double best_cost = 0.0;
  for (int TX = 1; TX <= g.Ex; ++TX) {
    if (TX * ne > res::kGenThreads * res::kGenMaxNodes) break;
    const int ntx = (g.Ex + TX - 1) / TX;
    if ((g.Ex + ntx - 1) / ntx != TX) continue;
    for (int RY = 1; RY <= g.Ey && TX * RY * ne <= res::kGenThreads * res::kGenMaxNodes; ++RY) {
      const int nty = (g.Ey + RY - 1) / RY;
      if ((g.Ey + nty - 1) / nty != RY || (long)ntx * nty > max_wg) continue;
      if (sizeof(double) * res::gen_lds_doubles(nr, ns, TX, RY) > res::kGenLds) continue;
      const int nt = TX * RY * ne, nw = std::min((nt + 63) / 64, res::kGenThreads / 64);
      const int K = (nt + 64 * nw - 1) / (64 * nw);
      ResPlan pl{TX, RY, ntx, nty, ntx * nty, nw, 0};
      pl.near = res_near(pl.nwg, ncu);
      const double cost = (pl.nwg == 1 ? 0.0 : (pl.near == 1 ? 3.8 : 5.0) + 0.004 * pl.nwg +
                                               (pl.nwg > 128 ? 0.8 : 0.0)) +
                          0.03 * (nr + ns) * K * (nw > 4 ? 1.5 : 1.0) + 0.001 * (TX * nr + RY * ns);
      if (best.nwg == 0 || cost < best_cost) {
        best = pl;
        best_cost = cost;
      }
    }
  }
  return best;
}

int launch_pcg_res_gen(hipStream_t st, const ResLaunch& l) {
  const sem_mesh* m = l.mesh;
  const ApplyArgs& a = *l.a;
  res::GenP q{};
  q.b = static_cast<const double*>(l.b);
  q.x = static_cast<double*>(l.x);
  q.r = static_cast<double*>(l.r);
  q.p = static_cast<double*>(l.p);
  q.d = static_cast<const double*>(l.d);
  q.G11 = static_cast<const double*>(a.G11);
  q.G12 = static_cast<const double*>(a.G12);
  q.G22 = static_cast<const double*>(a.G22);
  q.B = static_cast<const double*>(a.B);
  q.nu_f = static_cast<const double*>(a.nu_f);
  q.k_f = static_cast<const double*>(a.k_f);
  q.Dr = m->Dr;
  q.Ds = m->Ds;
  q.nu = a.nu;
  q.k = a.k;
  q.has_mass = a.has_mass;
  q.nr = m->nr;
  q.ns = m->ns;
  q.Ex = m->Ex;
  q.Ey = m->Ey;
  q.TX = l.plan.TX;
  q.RY = l.plan.RY;
  q.ntx = l.plan.ntx;
  q.nty = l.plan.nty;
  q.per_x = m->per_x;
  q.per_y = m->per_y;
  q.bc = a.bc;
  q.slots = static_cast<res::u64*>(l.mail);
  q.ymail = q.slots + res::kSlotArea;
  q.xmail = q.ymail + 2 * 2L * l.plan.nty * m->L;
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
  const int nt = l.plan.TX * l.plan.RY * m->nr * m->ns, NT = 64 * l.plan.nw;
  const int K = (nt + NT - 1) / NT;
  const size_t lds = sizeof(double) * res::gen_lds_doubles(m->nr, m->ns, l.plan.TX, l.plan.RY);
  if (K > res::kGenMaxNodes || lds > res::kGenLds) {
    set_error("resident PCG: a tile of %d nodes does not fit a workgroup", nt);
    return SEM_ERR_UNSUPPORTED;
  }
  const dim3 grid(l.plan.near == res::kNear ? res::kGroups * l.plan.nwg : l.plan.nwg), block(NT);
  auto go = [&](auto near) {
    constexpr bool N = decltype(near)::value;
    if (K == 1) hipLaunchKernelGGL((res::k_pcg_res_gen<1, N>), grid, block, lds, st, q);
    else if (K == 2) hipLaunchKernelGGL((res::k_pcg_res_gen<2, N>), grid, block, lds, st, q);
    else hipLaunchKernelGGL((res::k_pcg_res_gen<4, N>), grid, block, lds, st, q);
  };
  if (l.plan.near == res::kFlat) go(std::false_type());
  else go(std::true_type());
  SEM_HIP(hipGetLastError());
  return SEM_OK;
}

}  // namespace sem

// Multigrid preconditioner for the fused SEM operator and PCG with the
// V-cycle as opM (pcg.jl:16-60 with a stronger preconditioner than the
// identity / Jacobi of diffusion.jl:47-49; the reference's own next step is
// the commented element fast-diagonalisation sketch of lapl.jl:105-118).
//
// Hierarchy: p-multigrid on the element grid (N -> N/2 -> ... -> 1), then
// h-multigrid on bilinear elements (2 x 2 elements -> 1). Every level is a
// library mesh + fused operator (k_ax + k_seams), rediscretised with the same
// scalar nu, k and Dirichlet bits on nodes that sample the fine geometry.
// Smoother: Chebyshev-Jacobi (Saad, Iterative Methods for Sparse Linear
// Systems, Alg. 12.1) with host-side coefficients, fused into the level's
// apply (P < 16); transfers: a thread a row of an element, its interpolation rows
// from a small table. The bilinear levels' visits run as nine-point stencils
// (sem_mgs.h: several steps a launch, the smallest levels in one workgroup).
#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <cstring>
#include <new>
#include <vector>

#include "sem_device.h"
#include "sem_l0.h"
#include "sem_mgs.h"

namespace sem {
namespace {

inline int nblk(long n, int bs = 256) { return (int)((n + bs - 1) / bs); }

// The V-cycle's vector kernels are typed by the cycle's precision T (FP64,
// or FP32 for the FP32 cycle); the coefficients come in FP64 from the host.

// Chebyshev start: d = dinv .* r / theta; x = d (x0 = 0, and r = b copied
// from b) or x += d.
template <typename T>
__global__ void k_cheb_start(const T* __restrict__ b, T* __restrict__ r,
                             const T* __restrict__ dinv, T* __restrict__ d, T* __restrict__ x,
                             double theta, int from_zero, long n) {
  const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n) return;
  T rv;
  if (from_zero) {
    rv = b[t];
    r[t] = rv;
  } else {
    rv = r[t];
  }
  const T dv = dinv[t] * rv / T(theta);
  d[t] = dv;
  x[t] = from_zero ? dv : x[t] + dv;
}

// the start from zero without r and x, which the first fused step takes from b and d
template <typename T>
__global__ void k_cheb_dir(const T* __restrict__ b, const T* __restrict__ dinv, T* __restrict__ d,
                           double theta, long n) {
  const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t < n) d[t] = dinv[t] * b[t] / T(theta);
}

// One Chebyshev step after w = A d: r -= w; d = c1 d + c2 dinv .* r; x += d
template <typename T>
__global__ void k_cheb_step(const T* __restrict__ w, T* __restrict__ r,
                            const T* __restrict__ dinv, T* __restrict__ d, T* __restrict__ x,
                            double c1, double c2, long n) {
  const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n) return;
  const T rv = r[t] - w[t];
  r[t] = rv;
  const T dv = cheb_dir(T(c1), d[t], T(c2), dinv[t], rv);
  d[t] = dv;
  x[t] = x[t] + dv;
}

template <typename T>
__global__ void k_sub(T* __restrict__ r, const T* __restrict__ w, long n) {
  const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t < n) r[t] = r[t] - w[t];
}

// Transfer geometry: fine element ef = (ec << h) + sub; J holds nsub
// row-major (pf x pc) blocks for x, then for y.
struct Xfer {
  int pf, pc, hx, hy;
  int Lf, NCf, Lc, NCc;
  int per_x, per_y;
};

// e = P xc (per fine element: Jx xc Jy'), x += e (x NULL: the residual update adds e).
// Row owner: thread i of
// grid row eyf holds fine row i of fine element row eyf; it forms the
// x-contraction s(bb) = sum_aa Jx(a, aa) xc(aa, bb) once and then every
// column b of the element, so each coarse value is loaded pc / pf times per
// fine node and there is one integer division per thread. Same operation
// order as the one-node-per-thread form: v = sum_bb Jy(b, bb) s(bb).
constexpr int kXferMaxP = 16;
template <typename T>
__global__ void __launch_bounds__(256) k_prolong(const T* __restrict__ xc, const T* __restrict__ J,
                                                  T* __restrict__ e, T* __restrict__ x, Xfer g) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= g.Lf) return;
  const int eyf = blockIdx.y;
  const int exf = i / g.pf, a = i - exf * g.pf;
  const int sx = exf & g.hx, sy = eyf & g.hy;
  const int exc = exf >> g.hx, eyc = eyf >> g.hy;
  const int blk = g.pf * g.pc;
  const T* jx = J + sx * blk + a * g.pc;
  const T* jy = J + (g.hx ? 2 : 1) * blk + sy * blk;
  const long c0 = (long)exc * g.pc + (long)g.Lc * ((long)eyc * g.pc);
  T sv[kXferMaxP];
#pragma unroll
  for (int bb = 0; bb < kXferMaxP; ++bb) {
    if (bb < g.pc) {
      T sacc = T(0);
      for (int aa = 0; aa < g.pc; ++aa) sacc += jx[aa] * xc[c0 + aa + (long)g.Lc * bb];
      sv[bb] = sacc;
    }
  }
  const long f0 = i + (long)g.Lf * ((long)eyf * g.pf);
  for (int b = 0; b < g.pf; ++b) {
    T v = T(0);
#pragma unroll
    for (int bb = 0; bb < kXferMaxP; ++bb)
      if (bb < g.pc) v += jy[b * g.pc + bb] * sv[bb];
    const long t = f0 + (long)g.Lf * b;
    e[t] = v;
    if (x) x[t] = x[t] + v;
  }
}

// rc (element-local) = Jx' (mult_f .* rf) Jy summed over the fine nodes of
// the coarse element; assembled and masked afterwards by the coarse QQ'.
// A workgroup takes one coarse element row (grid row) and the fine rows of
// ce whole coarse elements: it stages those rows of the element row's fine
// columns in LDS with the x multiplicity applied (coalesced loads; the
// multiplicities are 1 or 1/2, so the product is exact), then forms the
// x-contractions s(a, c) = sum_(sx, af) Jx(af, a) rf(af, c) once per coarse
// row and fine column, and each coarse node v = sum_c wy(c, b) s(a, c) with
// wy = Jy my: the operation order of the one-node-per-thread form, so the
// bits are the same.
template <typename T>
__global__ void __launch_bounds__(256) k_restrict(const T* __restrict__ rf, const T* __restrict__ J,
                                                   T* __restrict__ rc, Xfer g) {
  extern __shared__ unsigned char xfer_lds[];
  const int nsx = g.hx ? 2 : 1, nsy = g.hy ? 2 : 1;
  const int fw = nsx * g.pf;          // fine rows per coarse element
  const int ce = 256 / fw;            // coarse elements per workgroup
  const int FR = ce * fw;             // fine rows staged
  const int nfc = nsy * g.pf;         // fine columns of the coarse element row
  const int rows = ce * g.pc;         // coarse rows of the workgroup
  const int blk = g.pf * g.pc;
  T* tile = reinterpret_cast<T*>(xfer_lds);   // [nfc][FR]
  T* sx_ = tile + FR * nfc;                   // [nfc][rows]
  T* jx = sx_ + rows * nfc;                   // [nsx * blk]: J's x blocks
  T* wy = jx + nsx * blk;                     // [nfc][pc]: Jy times the y multiplicity
  const int eyc = blockIdx.y;
  const int i0 = blockIdx.x * FR;
  const int jf0 = eyc * nfc;
  for (int q = threadIdx.x; q < FR * nfc; q += blockDim.x) {
    const int c = q / FR, r = q - c * FR;
    const int ifn = i0 + r;
    T v = T(0);
    if (ifn < g.Lf) v = T(mult1(ifn, g.pf, g.Lf, g.per_x)) * rf[ifn + (long)g.Lf * (jf0 + c)];
    tile[c * FR + r] = v;
  }
  for (int q = threadIdx.x; q < nsx * blk; q += blockDim.x) jx[q] = J[q];
  for (int q = threadIdx.x; q < nfc * g.pc; q += blockDim.x) {
    const int c = q / g.pc, b = q - c * g.pc;
    const int sy = c / g.pf, bf = c - sy * g.pf;
    const int jf = ((eyc << g.hy) + sy) * g.pf + bf;
    wy[q] = J[nsx * blk + sy * blk + bf * g.pc + b] * T(mult1(jf, g.pf, g.NCf, g.per_y));
  }
  __syncthreads();
  for (int q = threadIdx.x; q < rows * nfc; q += blockDim.x) {
    const int c = q / rows, rl = q - c * rows;
    const int exl = rl / g.pc, a = rl - exl * g.pc;
    const T* trow = tile + c * FR + exl * fw;
    T sacc = T(0);
    for (int sx = 0; sx < nsx; ++sx)
      for (int af = 0; af < g.pf; ++af) sacc += jx[sx * blk + af * g.pc + a] * trow[sx * g.pf + af];
    sx_[c * rows + rl] = sacc;
  }
  __syncthreads();
  const int exc0 = i0 / fw;
  for (int o = threadIdx.x; o < rows * g.pc; o += blockDim.x) {
    const int b = o / rows, rl = o - b * rows;
    const int ic = exc0 * g.pc + rl;
    if (ic >= g.Lc) continue;
    T v = T(0);
    for (int c = 0; c < nfc; ++c) v += wy[c * g.pc + b] * sx_[c * rows + rl];
    rc[ic + (long)g.Lc * (eyc * g.pc + b)] = v;
  }
}

// The transfers between orders (h = 0) with the sizes at compile time. A thread holds
// a fine row of an element in registers, its loads or stores all in flight together,
// and a workgroup the rows of 256 / PF elements; the y-direction runs in registers
// with coefficients from scalar loads, the x-direction over the coarse rows in LDS.
// Bound by memory: 256x256 elements, 8 and 4 points, restriction 21.5 -> 7.7 us,
// prolongation 17.2 -> 9.
template <typename T>
using ConstT = const T __attribute__((address_space(4)))*;   // scalar loads

template <typename T, int PF>
__global__ void __launch_bounds__(256) k_restrict_p(const T* __restrict__ rf,
                                                    const T* __restrict__ J, T* __restrict__ rc,
                                                    Xfer g) {
  constexpr int PC = (PF - 1) / 2 + 1, NE = 256 / PF, RS = NE * PF + 1;
  __shared__ T st[PC * RS];
  const int tid = threadIdx.x, ey = blockIdx.y, e0 = blockIdx.x * NE;
  const int i = e0 * PF + tid, ic = min(i, g.Lf - 1);
  ConstT<T> Jy = (ConstT<T>)(unsigned long long)(J + PF * PC);
  T r[PF], t[PC];
#pragma unroll
  for (int b = 0; b < PF; ++b) r[b] = rf[ic + (long)g.Lf * (ey * PF + b)];
  r[0] *= T(mult1(ey * PF, PF, g.NCf, g.per_y));
  r[PF - 1] *= T(mult1(ey * PF + PF - 1, PF, g.NCf, g.per_y));
#pragma unroll
  for (int c = 0; c < PC; ++c) t[c] = Jy[c] * r[0];
#pragma unroll
  for (int b = 1; b < PF; ++b)
#pragma unroll
    for (int c = 0; c < PC; ++c) t[c] += Jy[b * PC + c] * r[b];
  const T mx = T(mult1(ic, PF, g.Lf, g.per_x));
  if (tid < NE * PF) {
#pragma unroll
    for (int c = 0; c < PC; ++c) st[c * RS + tid] = mx * t[c];
  }
  __syncthreads();
  const int e = tid / PC, a = tid - e * PC;   // coarse row
  const int oc = e0 * PC + tid;
  if (tid >= NE * PC || oc >= g.Lc) return;
  T jx[PF];
#pragma unroll
  for (int k = 0; k < PF; ++k) jx[k] = J[k * PC + a];
#pragma unroll
  for (int c = 0; c < PC; ++c) {
    T v = jx[0] * st[c * RS + e * PF];
#pragma unroll
    for (int k = 1; k < PF; ++k) v += jx[k] * st[c * RS + e * PF + k];
    rc[oc + (long)g.Lc * (ey * PC + c)] = v;
  }
}

template <typename T, int PF>
__global__ void __launch_bounds__(256) k_prolong_p(const T* __restrict__ xc, const T* __restrict__ J,
                                                   T* __restrict__ e_, T* __restrict__ x, Xfer g) {
  constexpr int PC = (PF - 1) / 2 + 1, NE = 256 / PF, RS = NE * PC;
  __shared__ T st[PC * RS];
  const int tid = threadIdx.x, ey = blockIdx.y, e0 = blockIdx.x * NE;
  ConstT<T> Jy = (ConstT<T>)(unsigned long long)(J + PF * PC);
  if (tid < RS) {
    const int oc = min(e0 * PC + tid, g.Lc - 1);
#pragma unroll
    for (int c = 0; c < PC; ++c) st[c * RS + tid] = xc[oc + (long)g.Lc * (ey * PC + c)];
  }
  __syncthreads();
  const int e = tid / PF, a = tid - e * PF;
  const int i = e0 * PF + tid;
  if (tid >= NE * PF || i >= g.Lf) return;
  T jx[PC], s[PC];
#pragma unroll
  for (int k = 0; k < PC; ++k) jx[k] = J[a * PC + k];
#pragma unroll
  for (int c = 0; c < PC; ++c) {
    s[c] = jx[0] * st[c * RS + e * PC];
#pragma unroll
    for (int k = 1; k < PC; ++k) s[c] += jx[k] * st[c * RS + e * PC + k];
  }
  const long f0 = i + (long)g.Lf * (ey * PF);
  T v[PF];
#pragma unroll
  for (int b = 0; b < PF; ++b) {
    v[b] = Jy[b * PC] * s[0];
#pragma unroll
    for (int c = 1; c < PC; ++c) v[b] += Jy[b * PC + c] * s[c];
  }
#pragma unroll
  for (int b = 0; b < PF; ++b) e_[f0 + (long)g.Lf * b] = v[b];
  if (x) {
#pragma unroll
    for (int b = 0; b < PF; ++b) x[f0 + (long)g.Lf * b] = x[f0 + (long)g.Lf * b] + v[b];
  }
}

// The coarse right-hand side assembled and masked, x-pairs first as everywhere, and
// (d given) the start of the smoothing from zero on it, d = dinv .* b / theta. From
// one buffer to another, so that every copy is its own thread: reads and writes are
// coalesced and there is no map. 256x256 elements, 4 points, with d: 15.5 us as the map's
// gather-scatter and a pass, 9.4 so.
template <typename T>
__global__ void __launch_bounds__(256) k_assemble(const T* __restrict__ w, T* __restrict__ b,
                                                  const T* __restrict__ dinv, T* __restrict__ d,
                                                  double theta, int P, int L, int NC, int per_x,
                                                  int per_y, int bc) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= L) return;
  const int a = i % P;
  const bool hx = a == 0 ? i > 0 || per_x : a == P - 1 && (i < L - 1 || per_x);
  // left and right, lower and upper copies (the node's own where there is one)
  const int il = hx && a == 0 ? (i > 0 ? i - 1 : L - 1) : i;
  const int ir = hx && a != 0 ? (i < L - 1 ? i + 1 : 0) : i;
  for (int j = blockIdx.y; j < NC; j += gridDim.y) {
    const int c = j % P;
    const bool hy = c == 0 ? j > 0 || per_y : c == P - 1 && (j < NC - 1 || per_y);
    const int jl = hy && c == 0 ? (j > 0 ? j - 1 : NC - 1) : j;
    const int ju = hy && c != 0 ? (j < NC - 1 ? j + 1 : 0) : j;
    const T ll = w[il + (long)L * jl], rl = w[ir + (long)L * jl];
    const T lu = w[il + (long)L * ju], ru = w[ir + (long)L * ju];
    const T lo = hx ? ll + rl : ll, up = hx ? lu + ru : lu;
    const T s = (hy ? lo + up : lo) * mval<T>(i, j, L, NC, bc);
    const long t = i + (long)L * j;
    b[t] = s;
    if (d) d[t] = dinv[t] * s / T(theta);
  }
}

// coarse coordinates: the fine field interpolated at the coarse nodes; Jc is
// (pc x pf) row-major, node a of a coarse element lies in fine sub-element
// (subbits >> a) & 1 (h-merge only)
__global__ void k_coarse_coords(const double* __restrict__ xf, const double* __restrict__ Jc,
                                int subbits, double* __restrict__ xc, Xfer g, long n) {
  const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n) return;
  const int i = (int)(t % g.Lc), j = (int)(t / g.Lc);
  const int exc = i / g.pc, a = i - exc * g.pc;
  const int eyc = j / g.pc, b = j - eyc * g.pc;
  const int exf = (exc << g.hx) + (g.hx ? (subbits >> a) & 1 : 0);
  const int eyf = (eyc << g.hy) + (g.hy ? (subbits >> b) & 1 : 0);
  const long f0 = (long)exf * g.pf + (long)g.Lf * ((long)eyf * g.pf);
  double v = 0.0;
  for (int bf = 0; bf < g.pf; ++bf) {
    double s = 0.0;
    for (int af = 0; af < g.pf; ++af) s += Jc[a * g.pf + af] * xf[f0 + af + (long)g.Lf * bf];
    v += Jc[b * g.pf + bf] * s;
  }
  xc[t] = v;
}

// hashed start vector of the power iteration: M .* (h(g) / 2^32 - 1/2),
// h(g) = (g * 2654435761 + 12345) mod 2^32 of the global node id
__global__ void k_hash_start(const int32_t* __restrict__ l2g, double* __restrict__ v, int L,
                             int NC, int bc, long n) {
  const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n) return;
  const uint32_t h = (uint32_t)l2g[t] * 2654435761u + 12345u;
  const int i = (int)(t % L), j = (int)(t / L);
  v[t] = mask_on(i, j, L, NC, bc) ? (double)h / 4294967296.0 - 0.5 : 0.0;
}

__global__ void k_mul2(const double* __restrict__ a, const double* __restrict__ b,
                       double* __restrict__ y, long n) {
  const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t < n) y[t] = a[t] * b[t];
}

__global__ void k_div_scalar(const double* __restrict__ a, const double* __restrict__ s,
                             double* __restrict__ y, long n) {
  const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t < n) y[t] = a[t] / s[0];
}

// v .* D (D = 1 ./ dinv where dinv != 0, else 0): the diagonal weight of the
// Rayleigh quotient's denominator
__global__ void k_times_diag(const double* __restrict__ v, const double* __restrict__ dinv,
                             double* __restrict__ y, long n) {
  const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t < n) {
    const double di = dinv[t];
    y[t] = di != 0.0 ? v[t] * (1.0 / di) : 0.0;
  }
}

// The solver's vector passes. Each block first adds the parts of the inner products
// that it needs (kParts of them, in the same order in every block), so that no
// launch stands between a product and its use.
constexpr int kParts = 256;   // and threads per block
__device__ __forceinline__ double sum_parts(const double* __restrict__ part, double* sh) {
  const double v = wave_sum(part[threadIdx.x]);
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = v;
  __syncthreads();
  const double s = (sh[0] + sh[1]) + (sh[2] + sh[3]);
  __syncthreads();
  return s;
}

// x += alpha p, r -= alpha w with alpha = <z, r> / <p, A p> (pcg.jl:50-52), the old r
// to q when given, and the block's part of norm(r, Inf) (NaN if any is) to host
// memory: the convergence test reads it after the loop's one wait. With d the next
// cycle's start on the new r, d = dinv .* r / theta.
__global__ void __launch_bounds__(kParts)
k_xr(double* __restrict__ x, double* __restrict__ r, const double* __restrict__ p,
     const double* __restrict__ w, const double* __restrict__ tz, const double* __restrict__ tpw,
     double* __restrict__ q, double* __restrict__ res, const double* __restrict__ dinv,
     double* __restrict__ d, double theta, long n) {
  __shared__ double sh[4];
  const double t = sum_parts(tz, sh), alpha = t / sum_parts(tpw, sh);
  double m = 0.0;
  for (long i = (long)blockIdx.x * kParts + threadIdx.x; i < n; i += (long)gridDim.x * kParts) {
    x[i] = x[i] + alpha * p[i];
    const double ro = r[i], rv = ro - alpha * w[i];
    if (q) q[i] = ro;
    r[i] = rv;
    if (d) d[i] = dinv[i] * rv / theta;
    m = nanmax(m, fabs(rv));
  }
  m = wave_max(m);
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = m;
  __syncthreads();
  if (threadIdx.x == 0) res[blockIdx.x] = nanmax(nanmax(sh[0], sh[1]), nanmax(sh[2], sh[3]));
}

// p = z + beta p with beta = t / t_prev, or (t - s) / t_prev when s is given (the
// flexible form of the FP32 cycle), pcg.jl:49; p = z in the first iteration (tprev NULL)
__global__ void __launch_bounds__(kParts)
k_pdir(const double* __restrict__ z, double* p, const double* __restrict__ tz,
       const double* __restrict__ tprev, const double* __restrict__ s, long n) {
  __shared__ double sh[4];
  double beta = 0.0;
  if (tprev) {
    const double t = sum_parts(tz, sh), sv = s ? sum_parts(s, sh) : 0.0;
    beta = (s ? t - sv : t) / sum_parts(tprev, sh);
  }
  for (long i = (long)blockIdx.x * kParts + threadIdx.x; i < n; i += (long)gridDim.x * kParts)
    p[i] = tprev ? z[i] + beta * p[i] : z[i];
}
// blocks of these passes: eight a CU, each with several nodes a thread
inline int pass_blocks(long n) { return (int)std::min<long>(2048, nblk(n, 2 * kParts)); }

// Interpolation matrix rows with exact unit rows where an output point equals
// an input point (so copies of a shared node interpolate to identical bits).
std::vector<double> interp_rows(int no, const double* xo, int ni, const double* xi) {
  std::vector<double> Jc((size_t)no * ni), J((size_t)no * ni);
  interpmat(no, xo, ni, xi, Jc.data());   // column-major
  for (int i = 0; i < no; ++i)
    for (int j = 0; j < ni; ++j) J[(size_t)i * ni + j] = Jc[i + (size_t)no * j];
  for (int i = 0; i < no; ++i)
    for (int j = 0; j < ni; ++j)
      if (xo[i] == xi[j]) {
        for (int q = 0; q < ni; ++q) J[(size_t)i * ni + q] = q == j ? 1.0 : 0.0;
        break;
      }
  return J;
}

}  // namespace
}  // namespace sem

using namespace sem;

struct sem_mg {
  struct Level {
    sem_mesh* mesh = nullptr;
    bool own_mesh = false;
    const sem_operator* op = nullptr;
    bool own_op = false;
    double* dinv = nullptr;
    double lmax = 0.0;
    int h = 0;            // the next level merges this level's elements 2 x 2
    double* J = nullptr;  // transfer rows from the next level onto this one
    Xfer xf{};
    long nJ = 0;
    double *x = nullptr, *b = nullptr, *r = nullptr, *d = nullptr, *w = nullptr, *e = nullptr;
    // the FP32 cycle: the level operator in FP32 and FP32 copies of the above
    const sem_operator* op32 = nullptr;
    float *fx = nullptr, *fb = nullptr, *fr = nullptr, *fd = nullptr, *fw = nullptr,
          *fe = nullptr, *fdinv = nullptr, *fJ = nullptr;
    // the level's applies carry the smoother's vector updates as a fused
    // epilogue (FP64 / FP32 cycle)
    bool fuse64 = false, fuse32 = false;
    // the device blocks the level vectors above live in (one allocation per
    // precision)
    double* blk64 = nullptr;
    float* blk32 = nullptr;
    // a bilinear level cycled on its global nodes: its stencil in the cycle's
    // precision (lc's allocation holds those of all levels below it too)
    StenLevel sl{};
    void* sten = nullptr;
    bool own_sten = false;
  };
  sem_mg_params prm{};
  int device = 0;
  const sem_operator* op = nullptr;
  bool f32 = false;
  // smoother updates fused into the level applies (SEM_MG_FUSE=0 at
  // creation turns it off: a test hook)
  bool fuse = true;
  // the bilinear levels ls .. last work on global nodes, lc .. last of them in one
  // workgroup (< 0: none; SEM_MG_BLOCK=0 at creation turns both off)
  int ls = -1, lc = -1;
  bool block = true;
  std::vector<Level> lv;
  // PCG vectors on the fine level (pq: the previous residual of the flexible
  // recurrence), reduction partials and the scalar slot
  double *pr = nullptr, *pp = nullptr, *pw = nullptr, *pz = nullptr, *pq = nullptr,
         *part = nullptr;
};

namespace {

// the parts of the inner products: [0] setup's reductions, [1], [2] <z, r> of the even
// and odd PCG iterations, [3] <p, A p>, [4] the flexible beta's s; then a result
constexpr int kProducts = 5;

void mg_free(sem_mg* mg) {
  if (!mg) return;
  (void)hipDeviceSynchronize();
  for (auto& L : mg->lv) {
    double* bufs[] = {L.blk64, L.J};
    for (double* p : bufs)
      if (p) (void)hipFree(p);
    float* fbufs[] = {L.blk32, L.fJ};
    for (float* p : fbufs)
      if (p) (void)hipFree(p);
    if (L.sten && L.own_sten) (void)hipFree(L.sten);
    if (L.op32) sem_operator_destroy(const_cast<sem_operator*>(L.op32));
    if (L.own_op) sem_operator_destroy(const_cast<sem_operator*>(L.op));
    if (L.own_mesh) sem_mesh_destroy(L.mesh);
  }
  double* bufs[] = {mg->pr, mg->pp, mg->pw, mg->pz, mg->pq, mg->part};
  for (double* p : bufs)
    if (p) (void)hipFree(p);
  delete mg;
}

template <typename T>
int dalloc(T** p, long n) {
  SEM_HIP(hipMalloc(p, sizeof(T) * std::max<long>(n, 1)));
  return SEM_OK;
}

// a level's buffers and operator in the cycle's precision
template <typename T>
struct LvBuf {
  T *x, *b, *r, *d, *w, *e, *dinv, *J;
  const sem_operator* op;
  bool fuse;
};
template <typename T>
LvBuf<T> bufs(sem_mg::Level& L);
template <>
LvBuf<double> bufs<double>(sem_mg::Level& L) {
  return {L.x, L.b, L.r, L.d, L.w, L.e, L.dinv, L.J, L.op, L.fuse64};
}
template <>
LvBuf<float> bufs<float>(sem_mg::Level& L) {
  return {L.fx, L.fb, L.fr, L.fd, L.fw, L.fe, L.fdinv, L.fJ, L.op32, L.fuse32};
}
// the fused Chebyshev step leaves the new direction in w: the two buffers
// trade roles
template <typename T>
void swap_dw(sem_mg::Level& L);
template <>
void swap_dw<double>(sem_mg::Level& L) {
  std::swap(L.d, L.w);
}
template <>
void swap_dw<float>(sem_mg::Level& L) {
  std::swap(L.fd, L.fw);
}

// host value of a device reduction result
int fetch(sem_ctx* ctx, const double* dev, double* out) {
  SEM_TRY(ensure_pinned(ctx, 128));
  double* h = reinterpret_cast<double*>(static_cast<char*>(ctx->pinned) + 64);
  SEM_HIP(hipMemcpyAsync(h, dev, sizeof(double), hipMemcpyDeviceToHost, ctx->stream));
  SEM_HIP(hipStreamSynchronize(ctx->stream));
  *out = *h;
  return SEM_OK;
}

int wdot_host(sem_ctx* ctx, sem_mg* mg, const Layout& g, const double* a, const double* b,
              double* out) {
  SEM_TRY(launch_wdot(ctx->stream, g, a, b, mg->part, kParts, mg->part + kProducts * kParts));
  return fetch(ctx, mg->part + kProducts * kParts, out);
}

int norm_host(sem_ctx* ctx, sem_mg* mg, long n, const double* a, double* out) {
  SEM_TRY(launch_norm_inf(ctx->stream, n, a, mg->part, kParts, mg->part + kProducts * kParts));
  return fetch(ctx, mg->part + kProducts * kParts, out);
}

int apply(sem_ctx* ctx, const sem_operator* op, const void* u, void* y) {
  return sem_operator_apply(ctx, op, u, y);
}

// r -= A v (fused into the apply's final writes where the level allows;
// w is scratch either way); with start_theta the fused form also starts the
// Chebyshev smoother from the new r (d = dinv .* r / theta; x += d) and
// returns *started = true
template <typename T>
int residual_update(sem_ctx* ctx, const LvBuf<T>& L, const T* v, const double* start_theta = nullptr,
                    bool* started = nullptr, bool more = true) {
  if (started) *started = false;
  if (L.fuse) {
    ApplyEpi e;
    e.kind = start_theta ? 3 : 2;
    e.r = L.r;
    if (start_theta) {
      e.x = L.x;
      e.dinv = L.dinv;
      e.d = L.d;
      e.theta = *start_theta;
      e.flags = kEpiXIn | kEpiXU | kEpiXOut | (more ? kEpiROut | kEpiDOut : 0);
    }
    SEM_TRY(operator_apply_epi(ctx, L.op, v, L.w, e));
    if (started) *started = start_theta != nullptr;
    return SEM_OK;
  }
  SEM_TRY(apply(ctx, L.op, v, L.w));
  const long n = (long)L.op->mesh->nl;
  hipLaunchKernelGGL((k_sub<T>), dim3(nblk(n)), dim3(256), 0, ctx->stream, L.r, L.w, n);
  SEM_HIP(hipGetLastError());
  return SEM_OK;
}

// The smoother's coefficients on [lmax / ratio, lmax]: the start's divisor, and
// those of steps 1 .. nstep (c1[0] is step 1's).
struct ChebIter {
  double theta, delta, sigma, rho;
  ChebIter(double lmax, double ratio) {
    const double lmin = lmax / ratio;
    theta = 0.5 * (lmax + lmin);
    delta = 0.5 * (lmax - lmin);
    sigma = theta / delta;
    rho = 1.0 / sigma;
  }
  void next(double* c1, double* c2) {
    const double rho_n = 1.0 / (2.0 * sigma - rho);
    *c1 = rho_n * rho;
    *c2 = 2.0 * rho_n / delta;
    rho = rho_n;
  }
};

// Chebyshev iteration of degree deg for D^-1 A on [lmax / ratio, lmax]; from
// zero (x = 0, r = b) or from (x, r). With want_r the residual of the final
// x is formed in r (one more apply).
template <typename T>
int cheby(sem_ctx* ctx, sem_mg* mg, sem_mg::Level& Lv, const T* b, int from_zero, int deg,
          bool want_r, bool started = false, bool dir_ready = false) {
  hipStream_t st = ctx->stream;
  LvBuf<T> L = bufs<T>(Lv);
  const long n = (long)Lv.mesh->nl;
  ChebIter ch(Lv.lmax, mg->prm.ratio);
  // fused steps: the first takes r from b and x from d; x is advanced every second
  // step, by both directions (the same sums); what nothing reads is not written
  const bool light = from_zero && L.fuse && deg > 1;
  if (light && dir_ready) {
    // (formed with the right-hand side)
  } else if (light) {
    hipLaunchKernelGGL((k_cheb_dir<T>), dim3(nblk(n)), dim3(256), 0, st, b, L.dinv, L.d, ch.theta,
                       n);
    SEM_HIP(hipGetLastError());
  } else if (!started) {   // else the residual update formed d and advanced x
    hipLaunchKernelGGL((k_cheb_start<T>), dim3(nblk(n)), dim3(256), 0, st, b, L.r, L.dinv, L.d,
                       L.x, ch.theta, from_zero, n);
    SEM_HIP(hipGetLastError());
  }
  bool pending = light;   // the direction at hand is not in x yet
  for (int i = 1; i < deg; ++i) {
    double c1, c2;
    ch.next(&c1, &c2);
    if (L.fuse) {
      // w = A d with r -= w; d' = c1 d + c2 dinv .* r; x += d' fused into
      // its final writes (d' lands in w, which becomes the direction)
      ApplyEpi e;
      e.kind = 1;
      e.r = L.r;
      e.x = L.x;
      e.dinv = L.dinv;
      e.c1 = c1;
      e.c2 = c2;
      const bool end = i == deg - 1, first = light && i == 1;
      if (first) e.r_in = b;
      e.flags = (first ? 0 : kEpiXIn) | (pending ? kEpiXU : 0) |
                (pending || end ? kEpiXOut : 0) | (end && !want_r ? 0 : kEpiROut | kEpiDOut);
      pending = !pending && !end;
      SEM_TRY(operator_apply_epi(ctx, L.op, L.d, L.w, e));
      swap_dw<T>(Lv);
      L = bufs<T>(Lv);
    } else {
      SEM_TRY(apply(ctx, L.op, L.d, L.w));
      hipLaunchKernelGGL((k_cheb_step<T>), dim3(nblk(n)), dim3(256), 0, st, L.w, L.r, L.dinv,
                         L.d, L.x, c1, c2, n);
      SEM_HIP(hipGetLastError());
    }
  }
  if (want_r) SEM_TRY(residual_update<T>(ctx, L, L.d));
  return SEM_OK;
}

// the transfers between orders of this hierarchy; false: another transfer
template <typename T, int PF>
bool launch_prolong_p(hipStream_t st, const T* xc, const T* J, T* e, T* x, const Xfer& g) {
  if constexpr (PF < 3) return false;
  else {
    if (g.pf != PF) return launch_prolong_p<T, PF - 1>(st, xc, J, e, x, g);
    if (g.hx || g.hy || g.pc != (PF - 1) / 2 + 1) return false;
    hipLaunchKernelGGL((k_prolong_p<T, PF>), dim3((g.Lf / PF + 256 / PF - 1) / (256 / PF), g.NCf / PF),
                       dim3(256), 0, st, xc, J, e, x, g);
    return true;
  }
}
template <typename T, int PF>
bool launch_restrict_p(hipStream_t st, const T* rf, const T* J, T* rc, const Xfer& g) {
  if constexpr (PF < 3) return false;
  else {
    if (g.pf != PF) return launch_restrict_p<T, PF - 1>(st, rf, J, rc, g);
    if (g.hx || g.hy || g.pc != (PF - 1) / 2 + 1) return false;
    hipLaunchKernelGGL((k_restrict_p<T, PF>), dim3((g.Lf / PF + 256 / PF - 1) / (256 / PF), g.NCf / PF),
                       dim3(256), 0, st, rf, J, rc, g);
    return true;
  }
}

// transfer launches; the geometry is checked against the kernels' limits
template <typename T>
int launch_prolong(hipStream_t st, const T* xc, const T* J, T* e, T* x, const Xfer& g) {
  if (g.pc > kXferMaxP || g.pf > kXferMaxP || g.NCf % g.pf != 0) {
    set_error("multigrid prolongation: unsupported transfer (%d -> %d points)", g.pc, g.pf);
    return SEM_ERR_UNSUPPORTED;
  }
  if (!launch_prolong_p<T, kXferMaxP>(st, xc, J, e, x, g))
    hipLaunchKernelGGL((k_prolong<T>), dim3(nblk(g.Lf), g.NCf / g.pf), dim3(256), 0, st, xc, J, e,
                       x, g);
  SEM_HIP(hipGetLastError());
  return SEM_OK;
}
template <typename T>
int launch_restrict(hipStream_t st, const T* rf, const T* J, T* rc, const Xfer& g) {
  const int fw = (g.hx ? 2 : 1) * g.pf, nfc = (g.hy ? 2 : 1) * g.pf;
  if (fw > 256 || g.pc > kXferMaxP || g.NCc % g.pc != 0) {
    set_error("multigrid restriction: unsupported transfer (%d -> %d points)", g.pf, g.pc);
    return SEM_ERR_UNSUPPORTED;
  }
  const int FR = (256 / fw) * fw, rows = (256 / fw) * g.pc;
  const int nsx = g.hx ? 2 : 1;
  const size_t lds =
      sizeof(T) * ((size_t)FR * nfc + (size_t)rows * nfc + (size_t)nsx * g.pf * g.pc + (size_t)nfc * g.pc);
  if (lds > 65536) {
    set_error("multigrid restriction: %zu bytes of LDS for %d -> %d points", lds, g.pf, g.pc);
    return SEM_ERR_UNSUPPORTED;
  }
  if (!launch_restrict_p<T, kXferMaxP>(st, rf, J, rc, g))
    hipLaunchKernelGGL((k_restrict<T>), dim3((g.Lf + FR - 1) / FR, g.NCc / g.pc), dim3(256), lds,
                       st, rf, J, rc, g);
  SEM_HIP(hipGetLastError());
  return SEM_OK;
}

// Smoothing on a stencil level: from zero (r = b), or from the coarse level's x
// with residual *r; steps after the start. With to_coarse the residual of the
// final x comes back in *r and, restricted, in the coarse right-hand side. One
// launch while its applies fit a tile's halo, else the state (residual and
// direction) passes through memory, between buffers read and written in turn.
template <typename T>
int sten_smooth(sem_ctx* ctx, sem_mg* mg, int l, int from, int steps, bool to_coarse,
                const T** r) {
  sem_mg::Level& Lv = mg->lv[l];
  const LvBuf<T> L = bufs<T>(Lv);
  StenArgs<T> q{};
  q.V = Lv.sl;
  q.c = static_cast<const T*>(Lv.sten);
  q.x = L.x;
  if (l + 1 < (int)mg->lv.size()) {
    const LvBuf<T> C = bufs<T>(mg->lv[l + 1]);
    q.xc = C.x;
    q.bc = C.b;
    q.nxc = mg->lv[l + 1].sl.nx;
    q.nyc = mg->lv[l + 1].sl.ny;
  }
  ChebIter ch(Lv.lmax, mg->prm.ratio);
  q.theta = T(ch.theta);
  q.from = from;
  q.rin = from == kFromZero ? L.b : *r;
  for (int left = steps;;) {
    const int pre = q.from == kFromCoarse ? 1 : 0;
    const bool all = pre + left + (to_coarse ? 2 : 0) <= kStenHalo;
    q.nstep = all ? left : std::min(left, kStenHalo - pre);
    q.out = !all ? kOutState : to_coarse ? kOutRestrict : kOutX;
    q.H = pre + q.nstep + (q.out == kOutRestrict ? 2 : 0);
    for (int i = 0; i < q.nstep; ++i) {
      double c1, c2;
      ch.next(&c1, &c2);
      q.c1[i] = T(c1);
      q.c2[i] = T(c2);
    }
    const bool w = q.rin != L.w;
    q.rout = w ? L.w : L.r;
    q.dout = w ? L.e : L.d;
    SEM_TRY(launch_sten<T>(ctx->stream, q));
    if (r) *r = q.rout;
    if (all) return SEM_OK;
    left -= q.nstep;
    q.from = kFromState;
    q.rin = q.rout;
    q.din = q.dout;
  }
}

// the V-cycle from stencil level l on: x = V(b) in the level buffers
template <typename T>
int sten_cycle(sem_ctx* ctx, sem_mg* mg, int l) {
  const int last = (int)mg->lv.size() - 1;
  if (l == mg->lc) {
    CycleArgs<T> q{};
    const LvBuf<T> L = bufs<T>(mg->lv[l]);
    q.c = static_cast<const T*>(mg->lv[l].sten);
    q.b = L.b;
    q.x = L.x;
    for (int i = l; i <= last; ++i) {
      sem_mg::Level& Lv = mg->lv[i];
      CycleLevel<T>& V = q.lv[q.nlev++];
      V.V = Lv.sl;
      V.off = q.nodes;
      V.wave = q.waves;
      V.inv = (unsigned)(((1ull << 32) + Lv.sl.nx - 1) / Lv.sl.nx);
      q.nodes += Lv.sl.nx * Lv.sl.ny;
      q.waves += (Lv.sl.nx * Lv.sl.ny + 63) / 64;
      V.nstep = (i == last ? mg->prm.degree_coarse : mg->prm.degree) - 1;
      ChebIter ch(Lv.lmax, mg->prm.ratio);
      V.theta = T(ch.theta);
      for (int k = 0; k < V.nstep; ++k) {
        double c1, c2;
        ch.next(&c1, &c2);
        V.c1[k] = T(c1);
        V.c2[k] = T(c2);
      }
    }
    return launch_sten_cycle<T>(ctx->stream, q);
  }
  if (l == last)
    return sten_smooth<T>(ctx, mg, l, kFromZero, mg->prm.degree_coarse - 1, false, nullptr);
  const T* r = nullptr;
  SEM_TRY(sten_smooth<T>(ctx, mg, l, kFromZero, mg->prm.degree - 1, true, &r));
  SEM_TRY(sten_cycle<T>(ctx, mg, l + 1));
  return sten_smooth<T>(ctx, mg, l, kFromCoarse, mg->prm.degree - 1, false, &r);
}

// V-cycle on level l: x = V(b) in the level buffers of precision T
template <typename T>
int vcycle(sem_ctx* ctx, sem_mg* mg, int l, bool dir_ready = false) {
  hipStream_t st = ctx->stream;
  if (l == mg->ls) return sten_cycle<T>(ctx, mg, l);
  sem_mg::Level& Lv = mg->lv[l];
  LvBuf<T> L = bufs<T>(Lv);
  const int last = (int)mg->lv.size() - 1;
  if (l == last)
    return cheby<T>(ctx, mg, Lv, L.b, 1, mg->prm.degree_coarse, false, false, dir_ready);
  SEM_TRY(cheby<T>(ctx, mg, Lv, L.b, 1, mg->prm.degree, true, false, dir_ready));
  L = bufs<T>(Lv);   // the smoother may have swapped d and w
  sem_mg::Level& Cv = mg->lv[l + 1];
  const LvBuf<T> C = bufs<T>(Cv);
  SEM_TRY(launch_restrict<T>(st, L.r, L.J, C.w, Lv.xf));
  const int cdeg = l + 1 == last ? mg->prm.degree_coarse : mg->prm.degree;
  const bool dir = C.fuse && cdeg > 1 && l + 1 != mg->ls;
  const sem_mesh* mc = Cv.mesh;
  hipLaunchKernelGGL((k_assemble<T>), dim3(nblk(mc->L), std::min(mc->NC, 32768)), dim3(256), 0, st, C.w,
                     C.b, C.dinv,
                     dir ? C.d : nullptr, ChebIter(Cv.lmax, mg->prm.ratio).theta, mc->nr, mc->L,
                     mc->NC, mc->per_x, mc->per_y, Cv.op->desc.bc_bits);
  SEM_HIP(hipGetLastError());
  SEM_TRY(vcycle<T>(ctx, mg, l + 1, dir));
  SEM_TRY(launch_prolong<T>(st, C.x, L.J, L.e, L.fuse ? nullptr : L.x, Lv.xf));
  // the post-smoother's start (from r) rides on the residual update
  const double theta = 0.5 * (Lv.lmax + Lv.lmax / mg->prm.ratio);
  bool started = false;
  SEM_TRY(residual_update<T>(ctx, L, L.e, &theta, &started, mg->prm.degree > 1));
  return cheby<T>(ctx, mg, Lv, L.b, 0, mg->prm.degree, false, started);
}

// lmax = safety x Rayleigh quotient after npow power steps of D^-1 A
int estimate_lmax(sem_ctx* ctx, sem_mg* mg, sem_mg::Level& L) {
  hipStream_t st = ctx->stream;
  const sem_mesh* m = L.mesh;
  const long n = (long)m->nl;
  const Layout g = m->layout();
  double* v = L.d;
  double* w = L.w;
  double* e = L.e;
  hipLaunchKernelGGL(k_hash_start, dim3(nblk(n)), dim3(256), 0, st, m->l2g, v, m->L, m->NC,
                     L.op->desc.bc_bits, n);
  SEM_HIP(hipGetLastError());
  // v <- D^-1 A v; the Rayleigh quotient is scale-free, so the iterate is
  // rescaled by its max norm only every kRenorm steps (|lambda| < 4 keeps the
  // growth in between far from overflow), which saves the reduction and the
  // division launches of the other steps
  constexpr int kRenorm = 8;
  for (int it = 0; it < mg->prm.npow; ++it) {
    SEM_TRY(apply(ctx, L.op, v, w));
    hipLaunchKernelGGL(k_mul2, dim3(nblk(n)), dim3(256), 0, st, L.dinv, w, e, n);
    if ((it + 1) % kRenorm == 0) {
      SEM_TRY(launch_norm_inf(st, n, e, mg->part, kParts, mg->part + kProducts * kParts));
      hipLaunchKernelGGL(k_div_scalar, dim3(nblk(n)), dim3(256), 0, st, e, mg->part + kProducts * kParts, v,
                         n);
    } else {
      std::swap(v, e);
    }
    SEM_HIP(hipGetLastError());
  }
  double num = 0.0, den = 0.0;
  SEM_TRY(apply(ctx, L.op, v, w));
  SEM_TRY(wdot_host(ctx, mg, g, v, w, &num));
  hipLaunchKernelGGL(k_times_diag, dim3(nblk(n)), dim3(256), 0, st, v, L.dinv, e, n);
  SEM_TRY(wdot_host(ctx, mg, g, v, e, &den));
  if (!(den > 0.0) || !(num > 0.0) || !std::isfinite(num / den)) {
    set_error("sem_mg_create: eigenvalue estimate failed on a level with p = %d, %d x %d "
              "elements (Rayleigh quotient %g / %g)", m->nr, m->Ex, m->Ey, num, den);
    return SEM_ERR_BREAKDOWN;
  }
  L.lmax = mg->prm.safety * num / den;
  return SEM_OK;
}

// the level's vectors (x and b only below the finest level) in one block,
// each starting on a 512-byte boundary
int level_buffers(sem_mg::Level& L, bool own_xb) {
  const long n = (long)L.mesh->nl;
  const long sz = (n + 63) / 64 * 64;
  SEM_TRY(dalloc(&L.blk64, sz * (own_xb ? 7 : 5)));
  double* p = L.blk64;
  L.dinv = p;
  L.r = p + sz;
  L.d = p + 2 * sz;
  L.w = p + 3 * sz;
  L.e = p + 4 * sz;
  if (own_xb) {
    L.x = p + 5 * sz;
    L.b = p + 6 * sz;
  }
  return SEM_OK;
}

// the levels cycled on global nodes (ls: the first below the finest that is
// bilinear, then all are) and in one workgroup (lc)
void plan_sten(sem_mg* mg) {
  const int nl = (int)mg->lv.size();
  if (!mg->block) return;
  for (int l = nl - 1; l >= 1; --l) {
    sem_mg::Level& L = mg->lv[l];
    const sem_mesh* m = L.mesh;
    const int bc = L.op->desc.bc_bits;
    // (Dirichlet bits on a periodic direction mask copies one by one: not a
    // function of the node)
    if (m->nr != 2 || m->ns != 2 || (m->per_x && (bc & (SEM_BC_XMIN | SEM_BC_XMAX))) ||
        (m->per_y && (bc & (SEM_BC_YMIN | SEM_BC_YMAX))))
      break;
    L.sl = StenLevel{m->Ex + (m->per_x ? 0 : 1), m->Ey + (m->per_y ? 0 : 1), m->Ex, m->Ey,
                     m->per_x, m->per_y, bc, 0};
    mg->ls = l;
  }
  if (mg->ls < 0) return;
  mg->lv[mg->ls].sl.loc = 1;
  if (mg->prm.degree > kBlkMaxDeg || mg->prm.degree_coarse > kBlkMaxDeg) return;
  size_t nodes = 0, waves = 0;
  for (int l = nl - 1; l >= mg->ls && nl - l <= kBlkMaxLevels; --l) {
    const size_t n = (size_t)mg->lv[l].sl.nx * mg->lv[l].sl.ny;
    nodes += n;
    waves += (n + 63) / 64;
    if (n > (size_t)kBlkNodes || waves > (size_t)kBlkWaves ||
        sizeof(double) * 2 * (nodes + n) > (size_t)kBlkLds)
      break;
    mg->lc = l;
  }
}

template <typename T>
int build_sten(sem_ctx* ctx, sem_mg* mg) {
  auto f = [](const void* p) { return static_cast<const double*>(p); };
  T* next = nullptr;
  for (int l = mg->ls; l >= 0 && l < (int)mg->lv.size(); ++l) {
    sem_mg::Level& L = mg->lv[l];
    const StenLevel& V = L.sl;
    auto size = [](const sem_mg::Level& Q) { return 6L * Q.sl.nx * Q.sl.ny; };
    if (mg->lc < 0 || l <= mg->lc) {
      long n = size(L);
      if (l == mg->lc)
        for (size_t q = l + 1; q < mg->lv.size(); ++q) n += size(mg->lv[q]);
      SEM_TRY(dalloc(&next, n));
      L.own_sten = true;
    }
    L.sten = next;
    const sem_operator* op = L.op;   // FP64: the FP32 cycle's entries are rounded once
    SEM_TRY(launch_sten_build<T>(ctx->stream, V, f(op->G11), f(op->G12), f(op->G22),
                                 op->has_mass ? f(op->B) : nullptr, L.dinv, op->desc.nu,
                                 op->desc.k, next));
    next += size(L);
  }
  return SEM_OK;
}

int build(sem_ctx* ctx, sem_mg* mg) {
  hipStream_t st = ctx->stream;
  const sem_operator* op0 = mg->op;
  {
    sem_mg::Level L0;
    L0.mesh = const_cast<sem_mesh*>(op0->mesh);
    L0.op = op0;
    mg->lv.push_back(L0);
  }
  while ((int)mg->lv.size() < mg->prm.max_levels) {
    sem_mg::Level& F = mg->lv.back();
    const sem_mesh* mf = F.mesh;
    const int N = mf->nr - 1;
    int pc, h;
    if (N > 1) {
      pc = N / 2 + 1;
      h = 0;
    } else if (mf->Ex % 2 == 0 && mf->Ey % 2 == 0 && mf->Ex >= 4 && mf->Ey >= 4) {
      pc = 2;
      h = 1;
    } else {
      break;
    }
    const int pf = mf->nr;
    std::vector<double> zc(pc), wc(pc);
    gll(pc, zc.data(), wc.data());
    sem_mesh* mc = nullptr;
    SEM_TRY(sem_mesh_create(ctx, pc, pc, mf->Ex >> h, mf->Ey >> h, mf->per_x, mf->per_y,
                            SEM_DEFORM_NONE, 0.0, &mc));
    sem_mg::Level C;
    C.mesh = mc;
    C.own_mesh = true;
    mg->lv.push_back(C);
    sem_mg::Level& Fl = mg->lv[mg->lv.size() - 2];
    Fl.h = h;
    Xfer xf{};
    xf.pf = pf;
    xf.pc = pc;
    xf.hx = h;
    xf.hy = h;
    xf.Lf = mf->L;
    xf.NCf = mf->NC;
    xf.Lc = mc->L;
    xf.NCc = mc->NC;
    xf.per_x = mf->per_x;
    xf.per_y = mf->per_y;
    Fl.xf = xf;
    // transfer rows: fine GLL nodes of each sub-element in the coarse
    // reference coordinate, for x then y (square elements: identical)
    const std::vector<double>& zf = mf->hzr;
    std::vector<double> Jall;
    for (int dir = 0; dir < 2; ++dir)
      for (int s = 0; s < (h ? 2 : 1); ++s) {
        std::vector<double> xo(pf);
        for (int i = 0; i < pf; ++i) xo[i] = h ? (zf[i] + 2.0 * s - 1.0) / 2.0 : zf[i];
        std::vector<double> J = interp_rows(pf, xo.data(), pc, zc.data());
        Jall.insert(Jall.end(), J.begin(), J.end());
      }
    Fl.nJ = (long)Jall.size();
    SEM_TRY(dalloc(&Fl.J, (long)Jall.size()));
    SEM_HIP(hipMemcpy(Fl.J, Jall.data(), sizeof(double) * Jall.size(), hipMemcpyHostToDevice));
    // coarse coordinates: the fine geometry at the coarse nodes
    int subbits = 0;
    std::vector<double> xo(pc);
    for (int a = 0; a < pc; ++a) {
      const int sub = (h && zc[a] > 0.0) ? 1 : 0;
      subbits |= sub << a;
      xo[a] = h ? 2.0 * zc[a] + 1.0 - 2.0 * sub : zc[a];
    }
    std::vector<double> Jc = interp_rows(pc, xo.data(), pf, zf.data());
    double* dJc = nullptr;
    SEM_TRY(dalloc(&dJc, (long)Jc.size()));
    SEM_HIP(hipMemcpy(dJc, Jc.data(), sizeof(double) * Jc.size(), hipMemcpyHostToDevice));
    const long nc = (long)mc->nl;
    hipLaunchKernelGGL(k_coarse_coords, dim3(nblk(nc)), dim3(256), 0, st, mf->f[SEM_X], dJc,
                       subbits, mc->f[SEM_X], xf, nc);
    hipLaunchKernelGGL(k_coarse_coords, dim3(nblk(nc)), dim3(256), 0, st, mf->f[SEM_Y], dJc,
                       subbits, mc->f[SEM_Y], xf, nc);
    const hipError_t e = hipGetLastError();
    (void)hipStreamSynchronize(st);
    (void)hipFree(dJc);
    SEM_HIP(e);
    SEM_TRY(sem_mesh_set_coords(ctx, mc, mc->f[SEM_X], mc->f[SEM_Y]));
  }
  // operators, diagonals, buffers, eigenvalue estimates
  for (size_t l = 0; l < mg->lv.size(); ++l) {
    sem_mg::Level& L = mg->lv[l];
    if (l > 0) {
      sem_op_desc d{};
      d.nu = op0->desc.nu;
      d.k = op0->desc.k;
      d.bc_bits = op0->desc.bc_bits;
      d.assemble = 1;
      sem_operator* oc = nullptr;
      SEM_TRY(sem_operator_create(ctx, L.mesh, &d, SEM_F64, &oc));
      L.op = oc;
      L.own_op = true;
    }
    SEM_TRY(level_buffers(L, l > 0));
    SEM_TRY(sem_operator_jacobi(ctx, L.op, L.dinv));
    SEM_TRY(estimate_lmax(ctx, mg, L));   // uses the level's d, w, e only
    L.fuse64 = mg->fuse && operator_epi_ok(L.op);
  }
  plan_sten(mg);
  // the FP32 cycle: the operators of the levels that apply them rebuilt in FP32
  // and FP32 copies of the diagonals and transfer rows (the eigenvalue bounds are
  // the FP64 ones)
  if (mg->f32) {
    for (size_t l = 0; l < mg->lv.size(); ++l) {
      sem_mg::Level& L = mg->lv[l];
      const long n = (long)L.mesh->nl;
      if (mg->ls < 0 || (int)l < mg->ls) {
        sem_op_desc d{};
        d.nu = op0->desc.nu;
        d.k = op0->desc.k;
        d.bc_bits = op0->desc.bc_bits;
        d.assemble = 1;
        sem_operator* o32 = nullptr;
        SEM_TRY(sem_operator_create(ctx, L.mesh, &d, SEM_F32, &o32));
        L.op32 = o32;
        L.fuse32 = mg->fuse && operator_epi_ok(o32);
      }
      const long sz = (n + 127) / 128 * 128;
      float** fb[] = {&L.fx, &L.fb, &L.fr, &L.fd, &L.fw, &L.fe, &L.fdinv};
      SEM_TRY(dalloc(&L.blk32, sz * 7));
      for (int q = 0; q < 7; ++q) *fb[q] = L.blk32 + q * sz;
      SEM_TRY(launch_convert_f64_f32(st, n, L.dinv, L.fdinv));
      if (L.nJ > 0) {
        SEM_TRY(dalloc(&L.fJ, L.nJ));
        SEM_TRY(launch_convert_f64_f32(st, L.nJ, L.J, L.fJ));
      }
    }
  }
  const long n0 = (long)op0->mesh->nl;
  SEM_TRY(dalloc(&mg->pr, n0));
  SEM_TRY(dalloc(&mg->pp, n0));
  SEM_TRY(dalloc(&mg->pw, n0));
  SEM_TRY(dalloc(&mg->pz, n0));
  if (mg->f32) SEM_TRY(dalloc(&mg->pq, n0));
  SEM_TRY(mg->f32 ? build_sten<float>(ctx, mg) : build_sten<double>(ctx, mg));
  SEM_HIP(hipStreamSynchronize(st));
  return SEM_OK;
}

int check_op(const sem_operator* op) {
  SEM_ARG(op->precision == SEM_F64, "multigrid: the operator must be SEM_F64");
  if (op->generic) {
    set_error("multigrid: needs nr == ns <= %d", kMaxP);
    return SEM_ERR_UNSUPPORTED;
  }
  SEM_ARG(op->desc.assemble, "multigrid: the operator must assemble (desc.assemble = 1)");
  if (op->desc.nu_f || op->desc.k_f || op->desc.G11 || op->desc.G12 || op->desc.G22 ||
      op->desc.B) {
    set_error("multigrid: field nu/k and factor overrides are not supported (scalar nu, k only)");
    return SEM_ERR_UNSUPPORTED;
  }
  return SEM_OK;
}

// z = V(r); dir_ready: the finest level's first direction lies in its d (FP64 cycle)
int vcycle_of(sem_ctx* ctx, sem_mg* mg, const double* r, double* z, bool dir_ready) {
  SEM_ARG(ctx && mg && r && z, "NULL argument");
  SEM_ARG(r != z, "sem_mg_vcycle: r and z must not alias");
  sem_mg::Level& L0 = mg->lv[0];
  if (mg->f32) {
    const long n = (long)L0.mesh->nl;
    SEM_TRY(launch_convert_f64_f32(ctx->stream, n, r, L0.fb));
    SEM_TRY(vcycle<float>(ctx, mg, 0));
    return launch_convert_f32_f64(ctx->stream, n, L0.fx, z);
  }
  L0.b = const_cast<double*>(r);
  L0.x = z;
  const int s = vcycle<double>(ctx, mg, 0, dir_ready);
  L0.b = nullptr;
  L0.x = nullptr;
  return s;
}

}  // namespace

extern "C" {

int sem_mg_default_params(sem_mg_params* p) {
  SEM_ARG(p, "NULL argument");
  p->degree = 3;
  p->ratio = 20.0;
  p->degree_coarse = 8;
  p->npow = 20;
  p->safety = 1.1;
  p->max_levels = 32;
  p->precision = SEM_F64;
  return SEM_OK;
}

int sem_mg_create(sem_ctx* ctx, const sem_operator* op, const sem_mg_params* params,
                  sem_mg** out) {
  SEM_ARG(ctx && op && out, "NULL argument");
  SEM_TRY(check_op(op));
  sem_mg_params p;
  sem_mg_default_params(&p);
  if (params) p = *params;
  SEM_ARG(p.degree >= 1 && p.degree_coarse >= 1 && p.ratio > 1.0 && p.npow >= 1 &&
              p.safety >= 1.0 && p.max_levels >= 1,
          "sem_mg_create: bad parameters");
  SEM_ARG(p.precision == SEM_F64 || p.precision == SEM_F32,
          "sem_mg_create: precision must be SEM_F64 or SEM_F32");
  sem_mg* mg = new (std::nothrow) sem_mg();
  SEM_ARG(mg, "out of host memory");
  mg->prm = p;
  mg->device = ctx->device;
  mg->op = op;
  mg->f32 = p.precision == SEM_F32;
  const char* fz = std::getenv("SEM_MG_FUSE");
  mg->fuse = !(fz && std::atoi(fz) == 0);
  const char* fb = std::getenv("SEM_MG_BLOCK");
  mg->block = !(fb && std::atoi(fb) == 0);
  if (dalloc(&mg->part, kProducts * kParts + 8) != SEM_OK) {
    mg_free(mg);
    return SEM_ERR_HIP;
  }
  const int s = build(ctx, mg);
  if (s != SEM_OK) {
    mg_free(mg);
    return s;
  }
  *out = mg;
  return SEM_OK;
}

int sem_mg_destroy(sem_mg* mg) {
  mg_free(mg);
  return SEM_OK;
}

int sem_mg_num_levels(const sem_mg* mg, int* nlevels) {
  SEM_ARG(mg && nlevels, "NULL argument");
  *nlevels = (int)mg->lv.size();
  return SEM_OK;
}

int sem_mg_level_info(const sem_mg* mg, int level, int* p, int* Ex, int* Ey, double* lmax) {
  SEM_ARG(mg, "NULL argument");
  SEM_ARG(level >= 0 && level < (int)mg->lv.size(), "sem_mg_level_info: no level %d", level);
  const sem_mg::Level& L = mg->lv[level];
  if (p) *p = L.mesh->nr;
  if (Ex) *Ex = L.mesh->Ex;
  if (Ey) *Ey = L.mesh->Ey;
  if (lmax) *lmax = L.lmax;
  return SEM_OK;
}

int sem_mg_set_lmax(sem_mg* mg, int level, double lmax) {
  SEM_ARG(mg, "NULL argument");
  SEM_ARG(level >= 0 && level < (int)mg->lv.size(), "sem_mg_set_lmax: no level %d", level);
  SEM_ARG(lmax > 0.0 && std::isfinite(lmax), "sem_mg_set_lmax: lmax must be positive");
  mg->lv[level].lmax = lmax;
  return SEM_OK;
}

int sem_mg_vcycle(sem_ctx* ctx, sem_mg* mg, const double* r, double* z) {
  return vcycle_of(ctx, mg, r, z, false);
}

int sem_pcg_mg(sem_ctx* ctx, const sem_operator* op, sem_mg* mg, const double* b, double* x,
               double tol, int maxiter, sem_pcg_info* info) {
  SEM_ARG(ctx && op && mg && b && x, "NULL argument");
  SEM_ARG(op == mg->op, "sem_pcg_mg: mg was built for another operator");
  SEM_ARG(b != x, "sem_pcg_mg: b and x must not alias");
  SEM_ARG(maxiter >= 0 && tol >= 0.0, "sem_pcg_mg: bad limits");
  hipStream_t st = ctx->stream;
  const sem_mesh* m = op->mesh;
  const Layout g = m->layout();
  const long n = (long)m->nl;
  SEM_HIP(hipEventRecord(ctx->ev0, st));
  SEM_HIP(hipMemsetAsync(x, 0, sizeof(double) * n, st));
  SEM_HIP(hipMemcpyAsync(mg->pr, b, sizeof(double) * n, hipMemcpyDeviceToDevice, st));
  double res = 0.0;
  SEM_TRY(norm_host(ctx, mg, n, mg->pr, &res));
  SEM_TRY(ensure_pinned(ctx, 128 + sizeof(double) * pass_blocks(n)));
  double* norms = reinterpret_cast<double*>(static_cast<char*>(ctx->pinned) + 128);
  // the finest level's smoothing starts with the residual's update
  sem_mg::Level& L0 = mg->lv[0];
  const bool start = !mg->f32 && L0.fuse64 && mg->prm.degree > 1 && mg->lv.size() > 1;
  const double theta0 = ChebIter(L0.lmax, mg->prm.ratio).theta;
  int k = 0;
  bool conv = true;
  while (res > tol) {
    if (k == maxiter) {
      conv = false;
      break;
    }
    ++k;
    SEM_TRY(vcycle_of(ctx, mg, mg->pr, mg->pz, start && k > 1));
    // the inner products stay on the device, as parts: the loop waits once per
    // iteration, for the residual norm of its convergence test
    auto product = [&](int q) { return mg->part + q * kParts; };
    double* tz = product(1 + (k & 1));
    double* tprev = k > 1 ? product(1 + ((k - 1) & 1)) : nullptr;
    SEM_TRY(launch_wdot_part(st, g, mg->pr, mg->pz, tz, kParts));
    // FP32 cycle: the flexible (Polak-Ribiere) beta = <z_k, r_k - r_{k-1}>
    // / t_prev, which tolerates the cycle's rounding; FP64: pcg.jl:49
    const bool flex = mg->f32 && k > 1;
    if (flex) SEM_TRY(launch_wdot_part(st, g, mg->pq, mg->pz, product(4), kParts));
    hipLaunchKernelGGL(k_pdir, dim3(pass_blocks(n)), dim3(kParts), 0, st, mg->pz, mg->pp, tz,
                       tprev, flex ? product(4) : nullptr, n);
    SEM_HIP(hipGetLastError());
    SEM_TRY(apply(ctx, op, mg->pp, mg->pw));
    SEM_TRY(launch_wdot_part(st, g, mg->pp, mg->pw, product(3), kParts));
    hipLaunchKernelGGL(k_xr, dim3(pass_blocks(n)), dim3(kParts), 0, st, x, mg->pr, mg->pp, mg->pw,
                       tz, product(3), mg->f32 ? mg->pq : nullptr, norms, L0.dinv, start ? L0.d : nullptr,
                       theta0, n);
    SEM_HIP(hipGetLastError());
    SEM_HIP(hipStreamSynchronize(st));
    res = 0.0;
    for (int q = 0; q < pass_blocks(n); ++q)
      if (norms[q] > res || norms[q] != norms[q]) res = norms[q];
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
    set_error("sem_pcg_mg: residual is not finite after %d iterations", k);
    return SEM_ERR_NONFINITE;
  }
  return (conv && res <= tol) ? SEM_OK : SEM_WARN_MAXITER;
}

}  // extern "C"

// Dealiased advection, advect.jl:45-64, with J = Jr (x) Js the element
// interpolation to the dealiasing grid:
//   forward:   y = J' [ B_D ((J vx)(J Tx) + (J vy)(J Ty)) ]
//   transpose: the same linear map in T transposed factor by factor,
//              y = grad'( J'[(J vx) B_D (J w)], J'[(J vy) B_D (J w)] )
// with grad'(qx, qy) = Dr'(rx qx + ry qy) + (sx qx + sy qy) Ds.
//
// A workgroup of 128 threads takes as many consecutive elements as it has
// columns of the dealiasing grid for. A row thread (element, a) holds row a of
// the element's fields in registers: the gradient (its r-direction through one
// LDS transpose) and the s-direction interpolation of every field. A column
// thread (element, j) then holds column j of every interpolated field and walks
// the dealiasing nodes i: the r-direction interpolation of all fields, the
// pointwise product and the accumulation of its r-direction transpose use the
// same row i of Jr, so no value on the dealiasing grid is ever stored. A last row
// pass contracts over j. All coefficients come by scalar loads, of which D's and the
// rows' in flight do not all fit the scalar registers (forward: 91 spilled to vector lanes
// at P = 8, 502 at P = 16); LDS holds only the half-interpolated fields, read and
// written once.
//
// Meshes of few elements take the kernel below this one. What bounds this one: the
// latency of its phases, three to four waves a SIMD in flight (the bytes alone take 7 us,
// the multiply-adds 3 us of the 13 below). The loops
// over j and i are unrolled by three so that the coefficient rows' scalar loads run
// ahead: with one row at a time 12 nodes cost 12 waits. Per call, forward /
// transpose, us: 96x96 elements, 8 nodes, 12 dealiasing nodes 13.8 / 13.2 (one row
// at a time 19.7 / 17.4; one 256-thread workgroup per element with every operand in
// LDS and the sizes at run time, bound by two LDS reads a multiply-add, 34 / 34);
// 64x64, 12 and 18: 23.7 / 20.8. 64 or 256 threads a workgroup: no faster.
#include <algorithm>

#include "sem_device.h"

namespace sem {
namespace {

constexpr int kAdvThreads = 128;
typedef const double __attribute__((address_space(4)))* ConstD;   // scalar loads

struct AdvP {
  const double* T;    // w in the transpose
  const double* vx;
  const double* vy;
  const double* D;    // P x P, column-major (Dr = Ds: nr == ns)
  const double* rx;
  const double* ry;
  const double* sx;
  const double* sy;
  const double* BD;
  const double* Jr;   // pd rows of P
  const double* Js;
  double* y;
  int pd, Ex, E, ne;
};

template <int P, bool TR>
__global__ void __launch_bounds__(kAdvThreads) k_advect(const AdvP prm) {
  extern __shared__ double lds[];
  constexpr int NF = TR ? 3 : 4, NB = TR ? 2 : 1;   // fields up, fields back
  const int tid = threadIdx.x, pd = prm.pd, ne = prm.ne, Ex = prm.Ex;
  const int RS = (ne * P) | 1;   // row length: odd, column threads read down it
  const long L = (long)P * Ex, LD = (long)pd * Ex;
  const int g0 = blockIdx.x * ne;
  const int e = tid / P, a = tid - e * P;
  const bool row = tid < ne * P, act = row && g0 + e < prm.E;
  const int g = act ? g0 + e : g0;
  const long base = (g % Ex) * P + a + L * ((g / Ex) * P);
  ConstD D = (ConstD)(unsigned long long)prm.D;
  ConstD Jr = (ConstD)(unsigned long long)prm.Jr;
  ConstD Js = (ConstD)(unsigned long long)prm.Js;

  // out = D v or D' v of one vector
  auto mul = [&](const double (&v)[P], double (&o)[P]) {
#pragma unroll
    for (int b = 0; b < P; ++b) o[b] = v[0] * D[b];
#pragma unroll
    for (int k = 1; k < P; ++k)
#pragma unroll
      for (int b = 0; b < P; ++b) o[b] += v[k] * D[b + P * k];
  };
  auto mul_t = [&](const double (&v)[P], double (&o)[P]) {
#pragma unroll
    for (int b = 0; b < P; ++b) {
      double s = v[0] * D[P * b];
#pragma unroll
      for (int k = 1; k < P; ++k) s += v[k] * D[k + P * b];
      o[b] = s;
    }
  };
  // rows to columns and back: o = D u (or D' u) down the columns of the element
  // whose row a this thread holds; barriers before, between and after
  auto columns = [&](double (&u)[P], bool t) {
    if (row) {
#pragma unroll
      for (int b = 0; b < P; ++b) lds[b * RS + tid] = u[b];
    }
    __syncthreads();
    if (row) {
      double v[P], o[P];
      const int c = a * RS + e * P;
#pragma unroll
      for (int k = 0; k < P; ++k) v[k] = lds[c + k];
      if (t) mul_t(v, o);
      else mul(v, o);
#pragma unroll
      for (int k = 0; k < P; ++k) lds[c + k] = o[k];
    }
    __syncthreads();
    if (row) {
#pragma unroll
      for (int b = 0; b < P; ++b) u[b] = lds[b * RS + tid];
    }
    __syncthreads();
  };

  {
    double F[NF][P];
#pragma unroll
    for (int b = 0; b < P; ++b) F[0][b] = prm.T[base + L * b];
    if constexpr (!TR) {
      // the metric terms come with T, the velocities only once the gradient's
      // registers are free: they arrive while the products are formed
      double us[P], ur[P], M[4][P];
#pragma unroll
      for (int b = 0; b < P; ++b) {
        const long q = base + L * b;
        M[0][b] = prm.rx[q];
        M[1][b] = prm.ry[q];
        M[2][b] = prm.sx[q];
        M[3][b] = prm.sy[q];
      }
      mul(F[0], us);
#pragma unroll
      for (int b = 0; b < P; ++b) ur[b] = F[0][b];
      columns(ur, false);
#pragma unroll
      for (int b = 0; b < P; ++b) {
        F[0][b] = M[0][b] * ur[b] + M[2][b] * us[b];
        F[1][b] = M[1][b] * ur[b] + M[3][b] * us[b];
      }
    }
#pragma unroll
    for (int b = 0; b < P; ++b) {
      F[NF - 2][b] = prm.vx[base + L * b];
      F[NF - 1][b] = prm.vy[base + L * b];
    }
    // s-direction interpolation of the row
    if (row) {
#pragma unroll 3
      for (int j = 0; j < pd; ++j) {
        ConstD J = Js + j * P;
#pragma unroll
        for (int f = 0; f < NF; ++f) {
          double s = F[f][0] * J[0];
#pragma unroll
          for (int b = 1; b < P; ++b) s += F[f][b] * J[b];
          lds[(f * pd + j) * RS + tid] = s;
        }
      }
    }
  }
  __syncthreads();
  // column j of the dealiasing grid: interpolate, multiply, transpose back
  for (int c = tid; c < ne * pd; c += kAdvThreads) {
    const int e2 = c / pd, j = c - e2 * pd;
    const int gg = g0 + e2;
    if (gg >= prm.E) break;
    const double* bd = prm.BD + (gg % Ex) * pd + LD * ((gg / Ex) * pd + j);
    double A[NF][P], B[NB][P];
#pragma unroll
    for (int f = 0; f < NF; ++f)
#pragma unroll
      for (int k = 0; k < P; ++k) A[f][k] = lds[(f * pd + j) * RS + e2 * P + k];
#pragma unroll
    for (int f = 0; f < NB; ++f)
#pragma unroll
      for (int k = 0; k < P; ++k) B[f][k] = 0.0;
    double bn = bd[0];
#pragma unroll 3
    for (int i = 0; i < pd; ++i) {
      const double bi = bn;
      bn = bd[min(i + 1, pd - 1)];   // the next node's weight, in flight
      ConstD J = Jr + i * P;
      double X[NF];
#pragma unroll
      for (int f = 0; f < NF; ++f) X[f] = J[0] * A[f][0];
#pragma unroll
      for (int k = 1; k < P; ++k)
#pragma unroll
        for (int f = 0; f < NF; ++f) X[f] += J[k] * A[f][k];
      double q[NB];
      if constexpr (TR) {
        const double w = X[0] * bi;
        q[0] = X[1] * w;
        q[NB - 1] = X[2] * w;
      } else {
        q[0] = (X[2] * X[0] + X[3] * X[1]) * bi;
      }
#pragma unroll
      for (int k = 0; k < P; ++k)
#pragma unroll
        for (int f = 0; f < NB; ++f) B[f][k] += J[k] * q[f];
    }
    // (over the entries this thread read)
#pragma unroll
    for (int f = 0; f < NB; ++f)
#pragma unroll
      for (int k = 0; k < P; ++k) lds[(f * pd + j) * RS + e2 * P + k] = B[f][k];
  }
  __syncthreads();
  // the row again: contract over j
  double S[NB][P];
#pragma unroll
  for (int f = 0; f < NB; ++f)
#pragma unroll
    for (int b = 0; b < P; ++b) S[f][b] = 0.0;
  const int rt = row ? tid : 0;
#pragma unroll 3
  for (int j = 0; j < pd; ++j) {
    ConstD J = Js + j * P;
#pragma unroll
    for (int f = 0; f < NB; ++f) {
      const double v = lds[(f * pd + j) * RS + rt];
#pragma unroll
      for (int b = 0; b < P; ++b) S[f][b] += v * J[b];
    }
  }
  if constexpr (TR) {
    double p1[P], p2[P], o[P];
#pragma unroll
    for (int b = 0; b < P; ++b) {
      const long q = base + L * b;
      p1[b] = prm.rx[q] * S[0][b] + prm.ry[q] * S[NB - 1][b];
      p2[b] = prm.sx[q] * S[0][b] + prm.sy[q] * S[NB - 1][b];
    }
    __syncthreads();   // the sums over j were read
    columns(p1, true);
    mul_t(p2, o);
#pragma unroll
    for (int b = 0; b < P; ++b) S[0][b] = p1[b] + o[b];
  }
  if (act) {
#pragma unroll
    for (int b = 0; b < P; ++b) prm.y[base + L * b] = S[0][b];
  }
}

// The same for meshes of few elements: an element per workgroup of 256 threads, its
// fields and matrices in LDS, each phase a thread per output node (or three), all fields of
// a contraction together. Two LDS reads a multiply-add, but a chain of p or pd of them
// a phase instead of all of a row's or column's: while the chip has room for all
// elements at once that is what the call's time is. Forward / transpose, us, above and
// here: 8 nodes, 12 dealiasing nodes, 16x16 elements 8.5 / 8.0 and 5.6 / 5.3, 32x32 8.5 / 8.0
// and 6.5 / 6.3; 12 and 18, 16x16 14.3 / 12.8 and 8.5 / 8.0, 32x32 14.4 / 13.0 and 12.7 /
// 12.2; 16 and 24, 16x16 23.7 / 21.0 and 15.0 / 15.4.
constexpr int kElemThreads = 256;
static_assert(kMaxP * kMaxP <= kElemThreads, "one node per thread");
__host__ __device__ constexpr int elem_lds_doubles(int p, int pd) {
  return 8 * pd * p + 6 * p * p + 2 * pd * pd;
}
// Where it is taken, from sweeps over p = 2 to 16, pd from p to 24 and 4 to 2304 elements:
// its chains are clearly the shorter ones from p pd = 48 on (6 and 6 nodes, 16x16 elements,
// 5.1 / 5.1 above, 4.8 / 4.8 here; 7 and 7 6.2 / 5.9 and 5.1 / 5.0). The line in the elements,
// at which both take the same, falls with the rounds of nodes a phase takes (pd^2 / 256):
// 1250 to 1600, 1000 to 1250 and 500 to 1000 elements for one, two and three, where the last
// goes with the elements that 256 CUs (2048 threads and 160 KB of LDS each) have room for.
// The transpose's phases of 16 nodes are slower here: 16 and 16, 24x24 elements 16.6
// above, 19.6 here.
inline bool elem_better(int p, int pd, int E, int transpose) {
  const int room = 256 * std::min(8, 163840 / (int)(sizeof(double) * elem_lds_doubles(p, pd)));
  const int line = pd < 16 ? 1280 : pd < 23 ? 1024 : std::max(512, room / 2);
  return p * pd >= 48 && E <= std::min(p == 16 && transpose ? 512 : line, room);
}

template <bool TR>
__global__ void __launch_bounds__(kElemThreads) k_advect_elem(const AdvP prm, int p) {
  extern __shared__ double lds[];
  constexpr int NF = TR ? 3 : 4, NB = TR ? 2 : 1;   // fields up, fields back
  const int pd = prm.pd, pp = p * p, dp = pd * p, dd = pd * pd, tid = threadIdx.x;
  double* const sJr = lds;        // pd x p, column-major
  double* const sJs = sJr + dp;
  double* const sD = sJs + dp;    // p x p
  double* const sT = sD + pp;     // T
  double* const sF = sT + pp;     // Tx, Ty, vx, vy, or w, vx, vy
  double* const sA = sF + 4 * pp; // their r-direction interpolants, pd x p
  double* const sC = sA + 4 * dp; // the products, pd x pd
  double* const sE = sC + 2 * dd; // ... and back in r, p x pd
  const int ex = blockIdx.x % prm.Ex, ey = blockIdx.x / prm.Ex;
  const long L = (long)p * prm.Ex, LD = (long)pd * prm.Ex;
  const long d0 = (long)ex * pd + LD * ((long)ey * pd);
  // this thread's node (tid < pp) and dealiasing nodes
  const int a0 = tid % p, b0 = tid / p;
  const long gn = (long)ex * p + a0 + L * ((long)ey * p + b0);
  const bool own = tid < pp;
  double frx = 0, fry = 0, fsx = 0, fsy = 0;
  double bd[3] = {0, 0, 0};
  if (own) {
    frx = prm.rx[gn];
    fry = prm.ry[gn];
    fsx = prm.sx[gn];
    fsy = prm.sy[gn];
    (TR ? sF : sT)[tid] = prm.T[gn];
    sF[(NF - 2) * pp + tid] = prm.vx[gn];
    sF[(NF - 1) * pp + tid] = prm.vy[gn];
    sD[tid] = prm.D[tid];
  }
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    const int q = tid + i * kElemThreads;
    if (q < dd) bd[i] = prm.BD[d0 + q % pd + LD * (q / pd)];
  }
  for (int q = tid; q < dp; q += kElemThreads) {
    const int i = q / p, c = i + pd * (q - i * p);
    sJr[c] = prm.Jr[q];
    sJs[c] = prm.Js[q];
  }
  __syncthreads();
  if (!TR) {
    if (own) {
      double ur = 0, us = 0;
      for (int k = 0; k < p; ++k) ur += sD[a0 + p * k] * sT[k + p * b0];
      for (int k = 0; k < p; ++k) us += sT[a0 + p * k] * sD[b0 + p * k];
      sF[tid] = frx * ur + fsx * us;
      sF[pp + tid] = fry * ur + fsy * us;
    }
    __syncthreads();
  }
  for (int q = tid; q < dp; q += kElemThreads) {
    const int i = q % pd, b = q / pd;
    double s[NF] = {};
    for (int k = 0; k < p; ++k) {
      const double j = sJr[i + pd * k];
#pragma unroll
      for (int f = 0; f < NF; ++f) s[f] += j * sF[f * pp + k + p * b];
    }
#pragma unroll
    for (int f = 0; f < NF; ++f) sA[f * dp + q] = s[f];
  }
  __syncthreads();
#pragma unroll
  for (int n = 0; n < 3; ++n) {
    const int q = tid + n * kElemThreads;
    if (q < dd) {
      const int i = q % pd, j = q / pd;
      double X[NF] = {};
      for (int k = 0; k < p; ++k) {
        const double c = sJs[j + pd * k];
#pragma unroll
        for (int f = 0; f < NF; ++f) X[f] += sA[f * dp + i + pd * k] * c;
      }
      if (TR) {
        const double c = X[0] * bd[n];
        sC[q] = X[1] * c;
        sC[dd + q] = X[2] * c;
      } else {
        sC[q] = (X[NF - 2] * X[0] + X[NF - 1] * X[1]) * bd[n];
      }
    }
  }
  __syncthreads();
  for (int q = tid; q < dp; q += kElemThreads) {
    const int a = q % p, j = q / p;
    double e[NB] = {};
    for (int k = 0; k < pd; ++k) {
      const double c = sJr[k + pd * a];
#pragma unroll
      for (int f = 0; f < NB; ++f) e[f] += c * sC[f * dd + k + pd * j];
    }
#pragma unroll
    for (int f = 0; f < NB; ++f) sE[f * dp + q] = e[f];
  }
  __syncthreads();
  double s[NB] = {};
  if (own) {
    for (int k = 0; k < pd; ++k) {
      const double j = sJs[k + pd * b0];
#pragma unroll
      for (int f = 0; f < NB; ++f) s[f] += sE[f * dp + a0 + p * k] * j;
    }
    if (!TR) prm.y[gn] = s[0];
  }
  if (TR) {
    if (own) {
      sF[tid] = frx * s[0] + fry * s[NB - 1];
      sF[pp + tid] = fsx * s[0] + fsy * s[NB - 1];
    }
    __syncthreads();
    if (own) {
      double r = 0, t = 0;
      for (int k = 0; k < p; ++k) r += sD[k + p * a0] * sF[k + p * b0];
      for (int k = 0; k < p; ++k) t += sF[pp + a0 + p * k] * sD[k + p * b0];
      prm.y[gn] = r + t;
    }
  }
}

template <int P>
void go(hipStream_t st, AdvP q, int transpose) {
  // as many elements as the threads hold, within the 64 KiB a launch may ask for
  // (one element needs 4 x 24 rows of 17 at most)
  q.ne = kAdvThreads / std::max(P, q.pd);
  const int rows = std::max((transpose ? 3 : 4) * q.pd, P);
  auto bytes = [&] { return sizeof(double) * rows * ((q.ne * P) | 1); };
  while (q.ne > 1 && bytes() > 65536) --q.ne;
  const size_t lds = bytes();
  const dim3 grid((q.E + q.ne - 1) / q.ne), block(kAdvThreads);
  if (transpose) hipLaunchKernelGGL((k_advect<P, true>), grid, block, lds, st, q);
  else hipLaunchKernelGGL((k_advect<P, false>), grid, block, lds, st, q);
}

}  // namespace

int launch_advect(hipStream_t st, const sem_mesh* mV, const sem_mesh* mD, const double* J,
                  const double* T, const double* vx, const double* vy, double* y,
                  int transpose) {
  const int p = mV->nr, pd = mD->nr;
  double* const* f = mV->f;
  AdvP q{T, vx, vy, mV->Dr, f[SEM_RX], f[SEM_RY], f[SEM_SX], f[SEM_SY], mD->f[SEM_B], J,
         J + pd * p, y, pd, mV->Ex, mV->Ex * mV->Ey, 0};
  if (elem_better(p, pd, q.E, transpose)) {
    const size_t lds = sizeof(double) * elem_lds_doubles(p, pd);
    const dim3 grid(q.E), block(kElemThreads);
    if (transpose) hipLaunchKernelGGL(k_advect_elem<true>, grid, block, lds, st, q, p);
    else hipLaunchKernelGGL(k_advect_elem<false>, grid, block, lds, st, q, p);
    SEM_HIP(hipGetLastError());
    return SEM_OK;
  }
  switch (p) {
#define SEM_ADV_CASE(P) case P: go<P>(st, q, transpose); break;
    SEM_ADV_CASE(2) SEM_ADV_CASE(3) SEM_ADV_CASE(4) SEM_ADV_CASE(5) SEM_ADV_CASE(6)
    SEM_ADV_CASE(7) SEM_ADV_CASE(8) SEM_ADV_CASE(9) SEM_ADV_CASE(10) SEM_ADV_CASE(11)
    SEM_ADV_CASE(12) SEM_ADV_CASE(13) SEM_ADV_CASE(14) SEM_ADV_CASE(15) SEM_ADV_CASE(16)
#undef SEM_ADV_CASE
    default:
      set_error("advect: %d points per direction are not supported", p);
      return SEM_ERR_UNSUPPORTED;
  }
  SEM_HIP(hipGetLastError());
  return SEM_OK;
}

}  // namespace sem

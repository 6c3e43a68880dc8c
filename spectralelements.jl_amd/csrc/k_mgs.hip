// The bilinear levels of the multigrid cycle on their global nodes.
//
// With 2 x 2-node elements the assembled operator couples a node to its eight
// neighbours, and every vector of a level but the first has equal values at all
// copies of a node. So these levels work on one value per node with a nine-point
// stencil: A u (I) = sum_nb c_nb (u_nb - u_I) + m u_I, where c_nb are the assembled
// off-diagonal entries of the stiffness and m is the (diagonal) mass. The rows of
// the stiffness sum to zero, and in the difference form they do so exactly, as in
// the element form: in FP32 a stored diagonal would perturb smooth vectors by its
// rounding, which is of the size of the mass term itself on fine meshes. Entries
// are symmetric; kept are east, north, north-east and north-west.
//
// Two kernels:
// - k_sten: a tile of a level with a halo as wide as the applies of the launch, so
//   a whole pre-smoothing with its residual and restriction, or prolongation with
//   the residual and the post-smoothing, is one launch. One launch a pass (apply,
//   seams, start, transfers: 15 a level) costs 4.5 us each however small the
//   level; 62 us a level, now 10.
// - k_sten_cycle: the V-cycle over all levels from the first with at most
//   kBlkNodes nodes on, in one workgroup, each thread's nodes with their rows of the
//   operators in registers (FP64: 6 of 128 spilled), what the neighbours read of the
//   vectors in LDS: 107 us from 16 x 16 elements down with global memory between its
//   phases, now 23 from 32 x 32.
#include <algorithm>

#include "sem_device.h"
#include "sem_mgs.h"

namespace sem {
namespace {

// index i along a direction of n nodes; -1: none
__device__ __forceinline__ int nb(int i, int n, int per) {
  if (i >= 0 && i < n) return i;
  if (!per) return -1;
  i %= n;
  return i < 0 ? i + n : i;
}
__device__ __forceinline__ int uniform(int v) { return __builtin_amdgcn_readfirstlane(v); }
__device__ __forceinline__ StenLevel uniform(const StenLevel& v) {
  return StenLevel{uniform(v.nx),    uniform(v.ny),    uniform(v.Ex), uniform(v.Ey),
                   uniform(v.per_x), uniform(v.per_y), uniform(v.bc), uniform(v.loc)};
}
// the same for a node's neighbour: i from -1 to n
__device__ __forceinline__ int nb1(int i, int n, int per) {
  const int k = i < 0 ? i + n : i >= n ? i - n : i;
  return per || k == i ? k : -1;
}
// a local copy of global node I (P = 2): the left copy of element I, or the last row
__device__ __forceinline__ int lcopy(int I, int E) { return I < E ? 2 * I : 2 * E - 1; }

__device__ __forceinline__ bool masked(const StenLevel& V, int I, int J) {
  return ((V.bc & SEM_BC_XMIN) && I == 0) || ((V.bc & SEM_BC_XMAX) && I == V.nx - 1) ||
         ((V.bc & SEM_BC_YMIN) && J == 0) || ((V.bc & SEM_BC_YMAX) && J == V.ny - 1);
}

// The stencil of one node from the element factors at its copies. With X_b =
// u(1,b) - u(0,b), Y_a = u(a,1) - u(a,0) the element's energy is
// 1/4 sum_ab G11 X_b^2 + 2 G12 X_b Y_a + G22 Y_a^2; its mixed second
// derivatives are the entries below.
template <typename T>
__global__ void k_sten_build(StenLevel V, const double* __restrict__ G11,
                             const double* __restrict__ G12, const double* __restrict__ G22,
                             const double* __restrict__ B, const double* __restrict__ dinv,
                             double nu, double k, T* __restrict__ c) {
  const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
  const long ng = (long)V.nx * V.ny;
  if (t >= ng) return;
  const int I = (int)(t % V.nx), J = (int)(t / V.nx);
  const long L = 2L * V.Ex;
  // the elements right / left of and above / below the node (-1: none)
  const int er = I < V.Ex ? I : -1, el = I > 0 ? I - 1 : (V.per_x ? V.Ex - 1 : -1);
  const int eu = J < V.Ey ? J : -1, ed = J > 0 ? J - 1 : (V.per_y ? V.Ey - 1 : -1);
  auto at = [&](int ex, int ey, int a, int b) { return 2L * ex + a + L * (2L * ey + b); };
  double e = 0.0, n = 0.0, ne = 0.0, nw = 0.0, m = 0.0;
  if (er >= 0 && eu >= 0) {
    auto g = [&](const double* f, int a, int b) { return f[at(er, eu, a, b)]; };
    e += -0.25 * (g(G11, 0, 0) + g(G11, 1, 0)) + 0.25 * (g(G12, 1, 0) - g(G12, 0, 0));
    n += -0.25 * (g(G22, 0, 0) + g(G22, 0, 1)) + 0.25 * (g(G12, 0, 1) - g(G12, 0, 0));
    ne = -0.25 * (g(G12, 1, 0) + g(G12, 0, 1));
    if (B) m += g(B, 0, 0);
  }
  if (er >= 0 && ed >= 0) {
    auto g = [&](const double* f, int a, int b) { return f[at(er, ed, a, b)]; };
    e += -0.25 * (g(G11, 0, 1) + g(G11, 1, 1)) + 0.25 * (g(G12, 0, 1) - g(G12, 1, 1));
    if (B) m += g(B, 0, 1);
  }
  if (el >= 0 && eu >= 0) {
    auto g = [&](const double* f, int a, int b) { return f[at(el, eu, a, b)]; };
    n += -0.25 * (g(G22, 1, 0) + g(G22, 1, 1)) + 0.25 * (g(G12, 1, 0) - g(G12, 1, 1));
    nw = 0.25 * (g(G12, 0, 0) + g(G12, 1, 1));
    if (B) m += g(B, 1, 0);
  }
  if (el >= 0 && ed >= 0 && B) m += B[at(el, ed, 1, 1)];
  c[t] = T(nu * e);
  c[t + ng] = T(nu * n);
  c[t + 2 * ng] = T(nu * ne);
  c[t + 3 * ng] = T(nu * nw);
  c[t + 4 * ng] = T(k * m);
  c[t + 5 * ng] = T(dinv[lcopy(I, V.Ex) + L * lcopy(J, V.Ey)]);
}

// the nine entries of node (I, J), zero in masked rows; all zero without have (any
// valid I, J then)
template <typename T>
struct Row {
  T e, w, n, s, ne, sw, nw, se, m, dinv;
};
template <typename T, typename F>
__device__ __forceinline__ Row<T> load_row(const StenLevel& V, bool have, int I, int J, F f) {
  const int im = nb1(I - 1, V.nx, V.per_x), ip = nb1(I + 1, V.nx, V.per_x);
  const int jm = nb1(J - 1, V.ny, V.per_y);
  const int q = I + V.nx * J;
  Row<T> r;
  // loads without branches, all in flight together: a missing one reads the node's own
  auto get = [&](int arr, int i, int j) { return f(arr, i >= 0 && j >= 0 ? i + V.nx * j : q); };
  r.e = get(0, I, J);
  r.w = get(0, im, J);
  r.n = get(1, I, J);
  r.s = get(1, I, jm);
  r.ne = get(2, I, J);
  r.sw = get(2, im, jm);
  r.nw = get(3, I, J);
  r.se = get(3, ip, jm);
  r.m = get(4, I, J);
  r.dinv = f(5, q);
  const bool on = have && !masked(V, I, J);
  const bool w = on && im >= 0, s = on && jm >= 0;
  r.e = on ? r.e : T(0);
  r.w = w ? r.w : T(0);
  r.n = on ? r.n : T(0);
  r.s = s ? r.s : T(0);
  r.ne = on ? r.ne : T(0);
  r.sw = w && s ? r.sw : T(0);
  r.nw = on ? r.nw : T(0);
  r.se = s && ip >= 0 ? r.se : T(0);
  r.m = on ? r.m : T(0);
  r.dinv = have ? r.dinv : T(0);
  return r;
}
template <typename T>
__device__ __forceinline__ T fma_(T a, T b, T c) {
  if constexpr (sizeof(T) == 8) return __builtin_fma(a, b, c);
  else return __builtin_fmaf(a, b, c);
}
// A u at a node: u its value, the neighbours' values
template <typename T>
__device__ __forceinline__ T sten(const Row<T>& c, T u, T e, T w, T n, T s, T ne, T sw, T nw, T se) {
  T x = fma_(c.e, e - u, c.m * u);
  T y = c.w * (w - u);
  x = fma_(c.n, n - u, x);
  y = fma_(c.s, s - u, y);
  x = fma_(c.ne, ne - u, x);
  y = fma_(c.sw, sw - u, y);
  x = fma_(c.nw, nw - u, x);
  y = fma_(c.se, se - u, y);
  return x + y;
}

// bilinear interpolation to fine node (I, J) from the level below (its global
// nodes, or their first copies when the vector is element-local)
template <typename T, typename F>
__device__ __forceinline__ T interp(int I, int J, int nxc, int nyc, F xc) {
  const int i0 = I >> 1, j0 = J >> 1;
  int i1 = i0 + (I & 1), j1 = j0 + (J & 1);
  if (i1 >= nxc) i1 = 0;   // periodic
  if (j1 >= nyc) j1 = 0;
  const T a = T(0.5) * (xc(i0, j0) + xc(i1, j0)), b = T(0.5) * (xc(i0, j1) + xc(i1, j1));
  return T(0.5) * (a + b);
}
// full weighting of fine values r onto coarse node (I, J): the transpose
template <typename T, typename F>
__device__ __forceinline__ T restrict9(int I, int J, const StenLevel& V, F r) {
  T a[3][3];
#pragma unroll
  for (int dj = -1; dj <= 1; ++dj)
#pragma unroll
    for (int di = -1; di <= 1; ++di) {
      const bool in = (V.per_x || (2 * I + di >= 0 && 2 * I + di < V.nx)) &&
                      (V.per_y || (2 * J + dj >= 0 && 2 * J + dj < V.ny));
      const T rv = r(in ? di : 0, in ? dj : 0);
      a[dj + 1][di + 1] = in ? rv : T(0);
    }
  auto three = [](T x, T y, T z) { return y + T(0.5) * (x + z); };
  return three(three(a[0][0], a[0][1], a[0][2]), three(a[1][0], a[1][1], a[1][2]),
               three(a[2][0], a[2][1], a[2][2]));
}

// ---- one tile -------------------------------------------------------------
// 256 threads on a region of 32 x 32 nodes; thread (tx, ty) holds four nodes of
// column tx. H nodes on each side are the halo: an apply is right one node
// further in each time. Bound by latency: one exchange with memory, then an LDS
// pass and a barrier per apply. Regions of 32: the smallest whose halo of 4 (the
// default degree) still leaves over half of the work useful.
constexpr int kReg = 32, kTileThreads = 256, kNode = 4, kPitch = kReg + 2;

template <typename T>
__global__ void __launch_bounds__(kTileThreads) k_sten(const StenArgs<T> q) {
  __shared__ T u[2][kPitch * kPitch];
  __shared__ T cc[2][kStenHalo];   // the steps' coefficients: one wait for all
  const StenLevel V = q.V;
  const int tid = threadIdx.x, tx = tid % kReg, ty = (tid / kReg) * kNode;
  const int H = q.H, in = kReg - 2 * H;
  const int gi0 = blockIdx.x * in - H, gj0 = blockIdx.y * in - H;
  const long ng = (long)V.nx * V.ny, L = 2L * V.Ex;
  const int I = nb(gi0 + tx, V.nx, V.per_x);
  if (tid < kStenHalo) {
    cc[0][tid] = q.c1[tid];
    cc[1][tid] = q.c2[tid];
  }
  for (int t = tid; t < 2 * kPitch * kPitch; t += kTileThreads) (&u[0][0])[t] = T(0);

  Row<T> c[kNode];
  T r[kNode], d[kNode], x[kNode];
  long ig[kNode], il[kNode];   // global node; its first local copy
  bool own[kNode];
#pragma unroll
  for (int k = 0; k < kNode; ++k) {
    const int J = nb(gj0 + ty + k, V.ny, V.per_y);
    const bool ok = I >= 0 && J >= 0;
    ig[k] = ok ? I + (long)V.nx * J : 0;
    il[k] = ok ? lcopy(I, V.Ex) + L * lcopy(J, V.Ey) : 0;
    own[k] = tx >= H && tx < H + in && ty + k >= H && ty + k < H + in &&
             gi0 + tx < V.nx && gj0 + ty + k < V.ny;
    const int I1 = ok ? I : 0, J1 = ok ? J : 0;
    c[k] = load_row<T>(V, ok, I1, J1, [&](int arr, int g) { return q.c[g + ng * arr]; });
    const long ix = V.loc ? il[k] : ig[k];
    const T rv = q.rin[q.from == kFromZero ? ix : ig[k]];
    r[k] = ok ? rv : T(0);
    x[k] = d[k] = T(0);
    if (q.from != kFromZero) {
      const T xv = q.x[ix];
      x[k] = own[k] ? xv : T(0);
      const T dv = q.from == kFromState ? q.din[ig[k]]
                                        : interp<T>(I1, J1, q.nxc, q.nyc, [&](int i, int j) {
                                            return q.xc[i + (long)q.nxc * j];
                                          });
      d[k] = ok ? dv : T(0);
    }
  }
  __syncthreads();
  int p = 0;
  // w = A d at the thread's nodes
  auto apply = [&](T (&w)[kNode]) {
    T* b = u[p];
    p ^= 1;
    T* o = b + (ty + 1) * kPitch + tx + 1;
#pragma unroll
    for (int k = 0; k < kNode; ++k) o[k * kPitch] = d[k];
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kNode; ++k) {
      const T* a = o + k * kPitch;
      w[k] = sten(c[k], d[k], a[1], a[-1], a[kPitch], a[-kPitch], a[kPitch + 1], a[-kPitch - 1],
                  a[kPitch - 1], a[-kPitch + 1]);
    }
  };
  if (q.from == kFromCoarse) {   // r -= A e; x += e
    T w[kNode];
    apply(w);
#pragma unroll
    for (int k = 0; k < kNode; ++k) {
      r[k] = r[k] - w[k];
      x[k] = x[k] + d[k];
    }
  }
  if (q.from != kFromState) {
#pragma unroll
    for (int k = 0; k < kNode; ++k) {
      d[k] = c[k].dinv * r[k] / q.theta;
      x[k] = x[k] + d[k];
    }
  }
  for (int i = 0; i < q.nstep; ++i) {
    T w[kNode];
    apply(w);
#pragma unroll
    for (int k = 0; k < kNode; ++k) {
      r[k] = r[k] - w[k];
      d[k] = cheb_dir(cc[0][i], d[k], cc[1][i], c[k].dinv, r[k]);
      x[k] = x[k] + d[k];
    }
  }
  if (q.out == kOutRestrict) {
    T w[kNode];
    apply(w);
#pragma unroll
    for (int k = 0; k < kNode; ++k) r[k] = r[k] - w[k];
  }
#pragma unroll
  for (int k = 0; k < kNode; ++k) {
    if (!own[k]) continue;
    if (V.loc) {
      // every copy: the node's row and column, and the ones before (after a
      // periodic wrap: the last ones)
      const int J = gj0 + ty + k;
      const int a0 = lcopy(I, V.Ex), a1 = I > 0 ? 2 * I - 1 : (V.per_x ? 2 * V.Ex - 1 : 0);
      const int b0 = lcopy(J, V.Ey), b1 = J > 0 ? 2 * J - 1 : (V.per_y ? 2 * V.Ey - 1 : 0);
      q.x[a0 + L * b0] = x[k];
      q.x[a1 + L * b0] = x[k];
      q.x[a0 + L * b1] = x[k];
      q.x[a1 + L * b1] = x[k];
    } else {
      q.x[ig[k]] = x[k];
    }
    if (q.out != kOutX) q.rout[ig[k]] = r[k];
    if (q.out == kOutState) q.dout[ig[k]] = d[k];
  }
  if (q.out == kOutRestrict) {
    T* o = u[p] + (ty + 1) * kPitch + tx + 1;
#pragma unroll
    for (int k = 0; k < kNode; ++k) o[k * kPitch] = r[k];
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kNode; ++k) {
      const int J = gj0 + ty + k;
      if (!own[k] || (I & 1) || (J & 1)) continue;
      const int Ic = I >> 1, Jc = J >> 1;
      const T* a = o + k * kPitch;
      const T v = restrict9<T>(Ic, Jc, V, [&](int di, int dj) { return a[di + dj * kPitch]; });
      // the coarse boundary nodes are the fine ones
      q.bc[Ic + (long)q.nxc * Jc] = masked(V, I, J) ? T(0) : v;
    }
  }
}

// ---- all small levels in one workgroup --------------------------------------
// Every node of every level has its thread from the start: the levels' nodes lie one
// after the other, each level from a whole wave on, a thread has two of them, and what
// it needs of a node (row, neighbours, the nodes above and below it) stays in its
// registers for the whole cycle. So all that is loaded or computed once is so in
// parallel, and a visit of a level is its LDS passes and barriers only. A level of one
// wave's size is that wave's alone, without barriers. From 32 x 32 elements down 32 us
// with rows in LDS and set up per visit, 23 so.
constexpr int kCycThreads = 1024, kSlots = 2;
static_assert(kBlkWaves * 64 == kCycThreads * kSlots, "the threads' nodes");
// two offsets within a level in one register
__device__ __forceinline__ int pair(int lo, int hi) { return (lo & 0xffff) | (hi << 16); }
__device__ __forceinline__ int lo16(int v) { return (int)(short)v; }
__device__ __forceinline__ int hi16(int v) { return v >> 16; }

template <typename T>
__global__ void __launch_bounds__(kCycThreads) k_sten_cycle(const CycleArgs<T> args) {
  extern __shared__ unsigned char cyc_lds[];
  // The arguments lie in host memory: read line by line as the levels come to
  // them, each line would be a wait of a microsecond. One read of all of it.
  __shared__ CycleArgs<T> q;
  static_assert(sizeof(q) % 4 == 0 && sizeof(q) / 4 <= kCycThreads, "one word a thread");
  if (threadIdx.x < sizeof(q) / 4)
    reinterpret_cast<unsigned*>(&q)[threadIdx.x] =
        ((const unsigned*)(unsigned long long)__builtin_amdgcn_kernarg_segment_ptr())[threadIdx.x];
  // x and r of every node, two buffers of the direction
  T* const X0 = reinterpret_cast<T*>(cyc_lds);
  T* const R0 = X0 + args.nodes;
  T* const dbuf = R0 + args.nodes;
  const int tid = threadIdx.x, nlev = args.nlev;
  const int n0 = args.lv[0].V.nx * args.lv[0].V.ny;
  __syncthreads();

  Row<T> c[kSlots];
  T r[kSlots], d[kSlots], x[kSlots];
  int lev[kSlots], node[kSlots];   // the wave's level; the node within it (-1: none)
  // offsets in pairs: the node's neighbours, its fine node's, its coarse nodes'
  int di[kSlots], dj[kSlots], fi[kSlots], fj[kSlots], cd[kSlots];
  int fn[kSlots], cn[kSlots];   // the fine node (-1: masked), the first coarse node
#pragma unroll
  for (int s = 0; s < kSlots; ++s) {
    const int wave = uniform((tid >> 6) + s * (kCycThreads / 64));
    int l = 0;
    for (int k = 1; k < nlev; ++k)
      if (wave >= q.lv[k].wave) l = k;
    l = uniform(l);
    lev[s] = l;
    const CycleLevel<T>& Q = q.lv[l];
    const StenLevel V = uniform(Q.V);
    const int n = V.nx * V.ny, t = (wave - uniform(Q.wave)) * 64 + (tid & 63);
    const bool on = t < n;
    node[s] = on ? t : -1;
    const int t1 = on ? t : 0;
    const int J = V.nx == 1 ? t1 : (int)__umulhi(t1, Q.inv), I = t1 - J * V.nx;
    const T* const C = args.c + 6 * uniform(Q.off);
    c[s] = load_row<T>(V, on, I, J, [&](int arr, int g) { return C[g + n * arr]; });
    r[s] = d[s] = x[s] = T(0);
    if (l == 0) {
      const T bv = args.b[V.loc ? lcopy(I, V.Ex) + 2L * V.Ex * lcopy(J, V.Ey) : t1];
      r[s] = on ? bv : T(0);
    }
    // (a missing neighbour has a zero entry or weight: its value is the node's own)
    const int im = nb1(I - 1, V.nx, V.per_x), ip = nb1(I + 1, V.nx, V.per_x);
    const int jm = nb1(J - 1, V.ny, V.per_y), jp = nb1(J + 1, V.ny, V.per_y);
    di[s] = pair(im < 0 ? 0 : im - I, ip < 0 ? 0 : ip - I);
    dj[s] = pair(jm < 0 ? 0 : (jm - J) * V.nx, jp < 0 ? 0 : (jp - J) * V.nx);
    fn[s] = fi[s] = fj[s] = 0;
    if (l > 0) {   // the fine level's nodes around this one
      const StenLevel F = uniform(q.lv[l - 1].V);
      const int fI = 2 * I, fJ = 2 * J;
      const int a = nb1(fI - 1, F.nx, F.per_x), b = nb1(fI + 1, F.nx, F.per_x);
      const int e = nb1(fJ - 1, F.ny, F.per_y), f = nb1(fJ + 1, F.ny, F.per_y);
      fn[s] = uniform(q.lv[l - 1].off) + fI + F.nx * fJ;
      fi[s] = pair(a < 0 ? 0 : a - fI, b < 0 ? 0 : b - fI);
      fj[s] = pair(e < 0 ? 0 : (e - fJ) * F.nx, f < 0 ? 0 : (f - fJ) * F.nx);
      // masked rows start from zero
      if (masked(V, I, J)) fn[s] = -1;
    }
    cn[s] = cd[s] = 0;
    if (l < nlev - 1) {
      const StenLevel W = uniform(q.lv[l + 1].V);
      const int i0 = I >> 1, j0 = J >> 1;
      int i1 = i0 + (I & 1), j1 = j0 + (J & 1);
      if (i1 >= W.nx) i1 = 0;   // periodic
      if (j1 >= W.ny) j1 = 0;
      cn[s] = uniform(q.lv[l + 1].off) + i0 + W.nx * j0;
      cd[s] = pair(i1 - i0, (j1 - j0) * W.nx);
    }
  }

  for (int vis = 0; vis < 2 * nlev - 1; ++vis) {   // down, the last, up
    const bool up = vis >= nlev;
    const int l = up ? 2 * (nlev - 1) - vis : vis;
    const bool last = l == nlev - 1;
    const CycleLevel<T>& Q = q.lv[l];
    const int n = uniform(Q.V.nx) * uniform(Q.V.ny), off = uniform(Q.off), nstep = uniform(Q.nstep);
    const bool alone = n <= 64, in = lev[0] == l || lev[1] == l;
    if (!alone || in) {
      bool on[kSlots];
#pragma unroll
      for (int s = 0; s < kSlots; ++s) {
        on[s] = lev[s] == l && node[s] >= 0;
        if (!on[s]) continue;
        if (up) {
          const T* m = X0 + cn[s];
          const int ci = lo16(cd[s]), cj = hi16(cd[s]);
          const T a = T(0.5) * (m[0] + m[ci]), b = T(0.5) * (m[cj] + m[ci + cj]);
          d[s] = T(0.5) * (a + b);
        } else if (l > 0) {
          // full weighting of the fine residual, the transpose of the interpolation
          const bool z = fn[s] < 0;
          const T* m = R0 + (z ? 0 : fn[s]);
          const int fim = lo16(fi[s]), fip = hi16(fi[s]), fjm = lo16(fj[s]), fjp = hi16(fj[s]);
          const T wl = fim ? T(0.5) : T(0), wr = fip ? T(0.5) : T(0);
          const T wd = fjm ? T(0.5) : T(0), wu = fjp ? T(0.5) : T(0);
          auto three = [&](const T* p) { return p[0] + (wl * p[fim] + wr * p[fip]); };
          const T v = three(m) + (wd * three(m + fjm) + wu * three(m + fjp));
          r[s] = z ? T(0) : v;
        }
      }
      int p = 0;
      auto apply = [&](T (&w)[kSlots]) {
        T* b = dbuf + p * n0;
        p ^= 1;
#pragma unroll
        for (int s = 0; s < kSlots; ++s)
          if (on[s]) b[node[s]] = d[s];
        if (alone) {
          __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
          __builtin_amdgcn_wave_barrier();
          __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        } else {
          __syncthreads();
        }
#pragma unroll
        for (int s = 0; s < kSlots; ++s) {
          w[s] = T(0);
          if (!on[s]) continue;
          // (unpacked here each time: as loop invariants they would spill)
          int pi = di[s], pj = dj[s];
          asm volatile("" : "+v"(pi), "+v"(pj));
          const T* a = b + node[s];
          const int im = lo16(pi), ip = hi16(pi);
          const T* m = a + lo16(pj);
          const T* o = a + hi16(pj);
          w[s] = sten(c[s], d[s], a[ip], a[im], o[0], m[0], o[ip], m[im], o[im], m[ip]);
        }
      };
      // every update is the wave's own nodes' alone: the other slot keeps its values
      T w[kSlots];
      if (up) {
        apply(w);
#pragma unroll
        for (int s = 0; s < kSlots; ++s)
          if (on[s]) {
            r[s] = r[s] - w[s];
            x[s] = x[s] + d[s];
          }
      }
      const T theta = Q.theta;
#pragma unroll
      for (int s = 0; s < kSlots; ++s)
        if (on[s]) {
          d[s] = c[s].dinv * r[s] / theta;
          x[s] = up ? x[s] + d[s] : d[s];
        }
      T c1 = Q.c1[0], c2 = Q.c2[0];
      for (int i = 0; i < nstep; ++i) {
        const T a1 = c1, a2 = c2;
        c1 = Q.c1[(i + 1) % kBlkMaxDeg];   // the next step's, on their way
        c2 = Q.c2[(i + 1) % kBlkMaxDeg];
        apply(w);
#pragma unroll
        for (int s = 0; s < kSlots; ++s)
          if (on[s]) {
            r[s] = r[s] - w[s];
            d[s] = cheb_dir(a1, d[s], a2, c[s].dinv, r[s]);
            x[s] = x[s] + d[s];
          }
      }
      if (!up && !last) {
        apply(w);
#pragma unroll
        for (int s = 0; s < kSlots; ++s)
          if (on[s]) {
            r[s] = r[s] - w[s];
            R0[off + node[s]] = r[s];
          }
      }
      if (up || last) {
#pragma unroll
        for (int s = 0; s < kSlots; ++s)
          if (on[s]) X0[off + node[s]] = x[s];
      }
    }
    __syncthreads();
  }
  {
    const StenLevel V = uniform(q.lv[0].V);
    if (V.loc) {
      const int L = 2 * V.Ex, NC = 2 * V.Ey;
      for (int t = tid; t < L * NC; t += kCycThreads) {
        const int j = t / L, i = t - j * L;
        int I = (i + 1) >> 1, J = (j + 1) >> 1;
        if (I >= V.nx) I = 0;
        if (J >= V.ny) J = 0;
        args.x[t] = X0[I + V.nx * J];
      }
    } else {
      for (int t = tid; t < n0; t += kCycThreads) args.x[t] = X0[t];
    }
  }
}

}  // namespace

template <typename T>
int launch_sten_build(hipStream_t st, const StenLevel& V, const double* G11, const double* G12,
                      const double* G22, const double* B, const double* dinv, double nu, double k,
                      T* c) {
  const long ng = (long)V.nx * V.ny;
  hipLaunchKernelGGL((k_sten_build<T>), dim3((unsigned)((ng + 255) / 256)), dim3(256), 0, st, V,
                     G11, G12, G22, B, dinv, nu, k, c);
  SEM_HIP(hipGetLastError());
  return SEM_OK;
}

template <typename T>
int launch_sten(hipStream_t st, const StenArgs<T>& q) {
  const int applies = (q.from == kFromCoarse ? 1 : 0) + q.nstep + (q.out == kOutRestrict ? 2 : 0);
  if (q.nstep < 0 || q.nstep > kStenHalo || q.H < applies || q.H > kStenHalo) {
    set_error("multigrid: %d steps with a halo of %d", q.nstep, q.H);
    return SEM_ERR_ARG;
  }
  const int in = kReg - 2 * q.H;
  const dim3 grid((q.V.nx + in - 1) / in, (q.V.ny + in - 1) / in);
  hipLaunchKernelGGL((k_sten<T>), grid, dim3(kTileThreads), 0, st, q);
  SEM_HIP(hipGetLastError());
  return SEM_OK;
}

template <typename T>
int launch_sten_cycle(hipStream_t st, const CycleArgs<T>& q) {
  const int n0 = q.lv[0].V.nx * q.lv[0].V.ny;
  const size_t lds = sizeof(T) * 2 * ((size_t)q.nodes + n0);
  if (n0 > kBlkNodes || lds > (size_t)kBlkLds || q.waves > kBlkWaves) {
    set_error("multigrid: %d nodes for one workgroup", n0);
    return SEM_ERR_ARG;
  }
  hipLaunchKernelGGL((k_sten_cycle<T>), dim3(1), dim3(kCycThreads), lds, st, q);
  SEM_HIP(hipGetLastError());
  return SEM_OK;
}

#define SEM_MGS_INST(T)                                                                          \
  template int launch_sten_build<T>(hipStream_t, const StenLevel&, const double*, const double*, \
                                    const double*, const double*, const double*, double, double, \
                                    T*);                                                         \
  template int launch_sten<T>(hipStream_t, const StenArgs<T>&);                                  \
  template int launch_sten_cycle<T>(hipStream_t, const CycleArgs<T>&);
SEM_MGS_INST(double)
SEM_MGS_INST(float)
#undef SEM_MGS_INST

}  // namespace sem

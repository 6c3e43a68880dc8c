// The bilinear multigrid levels on their global nodes (k_mgs.hip): descriptors
// and launches.
#pragma once

#include "sem_common.h"

namespace sem {

// nodes of a level, its elements, Dirichlet bits; loc: x and the right-hand side
// are element-local vectors (the first such level, whose neighbours in the
// hierarchy are meshes of higher order), else one value per node
struct StenLevel {
  int nx, ny, Ex, Ey, per_x, per_y, bc, loc;
};

constexpr int kStenHalo = 8;       // applies of one tile launch, at most
constexpr int kBlkNodes = 34 * 34; // nodes of the first level of one workgroup's cycle
constexpr int kBlkLds = 56 * 1024;   // LDS of its vectors, beside the arguments' copy
constexpr int kBlkWaves = 32;          // its threads' nodes in waves, a level from a whole one on
constexpr int kBlkMaxLevels = 8;
constexpr int kBlkMaxDeg = 16;

enum { kFromZero, kFromCoarse, kFromState };
enum { kOutX, kOutState, kOutRestrict };

template <typename T>
struct StenArgs {
  StenLevel V;
  const T* c;                 // six arrays of nx ny: east, north, north-east, north-west, mass, dinv
  int from, out, H, nstep;
  const T *rin, *din, *xc;    // right-hand side or residual; direction; coarse x
  T *x, *rout, *dout, *bc;    // bc: the coarse right-hand side
  int nxc, nyc;               // the coarse level's nodes
  T theta;
  T c1[kStenHalo], c2[kStenHalo];
};

template <typename T>
struct CycleLevel {
  StenLevel V;
  int off, wave, nstep;       // nodes and waves of the levels before; smoothing steps
  unsigned inv;               // ceil(2^32 / nx): t / nx = mulhi(t, inv) for t < kBlkNodes, nx > 1
  T theta;
  T c1[kBlkMaxDeg], c2[kBlkMaxDeg];
};
template <typename T>
struct CycleArgs {
  int nlev, nodes, waves;     // nodes and waves of all levels
  const T* c;                 // the levels' coefficients, one after the other
  const T* b;
  T* x;
  CycleLevel<T> lv[kBlkMaxLevels];
};
static_assert(sizeof(CycleArgs<double>) <= 4096, "kernel arguments");

template <typename T>
int launch_sten_build(hipStream_t st, const StenLevel& V, const double* G11, const double* G12,
                      const double* G22, const double* B, const double* dinv, double nu, double k,
                      T* c);
template <typename T>
int launch_sten(hipStream_t st, const StenArgs<T>& q);
template <typename T>
int launch_sten_cycle(hipStream_t st, const CycleArgs<T>& q);

}  // namespace sem

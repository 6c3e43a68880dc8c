// Build-time generator: writes the GLL derivative matrices for P = 2..16 as
// exact hexadecimal literals, computed by the same host routine the library
// uses for Mesh.Dr / Mesh.Ds. Each table is a constexpr array so that, with a
// compile-time index, it folds to an immediate in the fused kernels. (As a switch it
// counted as its P^2 cases in every unrolled product: from P = 14 on the compiler
// kept the loops and walked the cases at run time, 236 us instead of 9 for an
// element operator at P = 15.)
#include <cstdio>

#include "sem_l0.h"

int main() {
  std::printf("// Generated by gen_dtables.cpp: GLL derivative matrices, column-major.\n");
  std::printf("#pragma once\nnamespace sem {\n");
  std::printf("template <int P> struct GllTable;\n");
  for (int P = 2; P <= 16; ++P) {
    std::vector<double> z(P), w(P), D(P * P);
    sem::gll(P, z.data(), w.data());
    sem::derivmat(P, z.data(), D.data());
    std::printf("template <> struct GllTable<%d> {\n  static constexpr double v[%d] = {\n", P, P * P);
    for (int i = 0; i < P * P; ++i) std::printf("      %a,\n", D[i]);
    std::printf("  };\n};\n");
  }
  std::printf("template <int P> __host__ __device__ constexpr double gll_d(int i) { return GllTable<P>::v[i]; }\n");
  std::printf("}  // namespace sem\n");
  return 0;
}

// wait_check.cpp -- DeviceSYMGS and DeviceMG (hpcg_amd/host) in the reference's
// row order report a sweep whose waits gave up: under a limit of 0 polls (tune
// "lex_polls") both return an error, under the default both return 0.
#include <cstdio>

#include "../../hpcg_amd/host/DeviceProblem.hpp"
#include "../../hpcg_amd/host/OptimizedKernels.hpp"
#include "../../hpcg_amd/host/driver/Driver.hpp"

int main() {
  Geometry *geom = new Geometry;
  GenerateGeometry(1, 0, 1, 0, 0, 0, 16, 16, 64, 1, 1, 1, geom);
  SparseMatrix A;
  InitializeSparseMatrix(A, geom);
  Vector b, x, xexact;
  GenerateProblem(A, &b, &x, &xexact);
  hpcg_amd::DeviceContext *c = hpcg_amd::EnsureDeviceProblem(A);
  if (!c) return 3;
  for (double polls : {0.0, 4194304.0}) {
    if (hpcgx_tune(c->problem, "lex_polls", polls)) return 3;
    const int s = hpcg_amd::DeviceSYMGS(A, b, x, HPCGX_ORDER_LEXICOGRAPHIC);
    const int m = hpcg_amd::DeviceMG(A, b, x, HPCGX_ORDER_LEXICOGRAPHIC);
    std::printf("polls %g: symgs %d mg %d\n", polls, s, m);
    if ((s != 0) != (polls == 0.0) || (m != 0) != (polls == 0.0)) return 1;
  }
  DeleteMatrix(A);
  return 0;
}

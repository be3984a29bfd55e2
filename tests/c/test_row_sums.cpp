// Host check of the nine-wave pass' sums over an element's quadrature rows (gather_rows in ptq2_rows.h)
// against long double.  Rows (1, qc) alone have the coefficients 0 and +-1 along y, so a slab's sum is exact and
// what is left is the sum over the slabs: that one is FP64.  With all rows it is as good as FP32 row
// sums allow.
#include <hip/hip_runtime.h>
// the device code under test, for the host
#undef __device__
#define __device__ __attribute__((device)) __attribute__((host))
#define __builtin_amdgcn_sched_barrier(mask) ((void)0)
#include "ptq2_rows.h"

#include <cmath>
#include <cstdio>
#include <random>
#include <vector>

using namespace ptq2;

static int check(bool all_rows, std::mt19937_64 &gen) {
  std::uniform_real_distribution<double> U(-1.0, 1.0);
  std::vector<float> ex((size_t)RWAVES * ROWVALS * BEL, 0.0f);
  int bad = 0;
  for (int lane = 0; lane < BEL; lane++)
    for (int row = 0; row < RWAVES; row++)
      for (int n = 0; n < ROWVALS; n++)
        ex[(size_t)(row * ROWVALS + n) * BEL + lane] = all_rows || row % 3 == 1 ? (float)U(gen) : 0.0f;
  for (int lane = 0; lane < BEL; lane++)
    for (int c = 0; c < 3; c++)
      for (int k = 0; k < 3; k++) {
        double bk[3], dk[3], Y[9];
        for (int qc = 0; qc < 3; qc++) {
          bk[qc] = qc == 1 ? (k == 1) : gB(qc, k);
          dk[qc] = 2.0 * gD(qc, k);
        }
        gather_rows(ex.data(), lane, c, bk, dk, Y);
        // nodal x values from the dual modal ones: (a - b, m - 2 a, a + b)
        const double tr[3][3] = {{0.0, -1.0, 1.0}, {1.0, 0.0, -2.0}, {0.0, 1.0, 1.0}};
        for (int j = 0; j < 3; j++)
          for (int i = 0; i < 3; i++) {
            long double ref = 0.0L, size = 0.0L;
            for (int m = 0; m < 3; m++)
              for (int row = 0; row < 9; row++) {
                const int qb = row % 3, qc = row / 3;
                const float *e = ex.data() + (size_t)(row * ROWVALS + 8 * c) * BEL + lane;
                const double vb = qb == 1 ? (j == 1) : gB(qb, j);
                const long double terms[3] = {m > 0 ? (long double)(bk[qc] * vb) * e[(size_t)(m - 1) * BEL] : 0.0L,
                                              (long double)(bk[qc] * 2.0 * gD(qb, j)) * e[(size_t)(2 + m) * BEL],
                                              (long double)(dk[qc] * vb) * e[(size_t)(5 + m) * BEL]};
                for (long double t : terms) {
                  ref += tr[i][m] * t;
                  size += std::fabs((double)(tr[i][m] * t));
                }
              }
            // exact rows: 6 rounded slab terms and 2 of the x transform; else 7 rounded row terms and coefficients
            const long double tol = (all_rows ? 16.0L * std::ldexp(1.0, -24) : 16.0L * std::ldexp(1.0, -53)) * size;
            if (std::fabs((double)(Y[i + 3 * j] - ref)) > (double)tol) bad++;
          }
      }
  if (bad) std::printf("%s rows: %d of %d values off\n", all_rows ? "all" : "middle", bad, BEL * 81);
  return bad;
}

int main() {
  std::mt19937_64 gen(7);
  if (check(false, gen) + check(true, gen)) return 1;
  std::printf("row sums ok\n");
  return 0;
}

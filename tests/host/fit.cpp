// The distance of the quaternion fit (fo_refine.h) against the smallest eigenvalue
// of the same 4x4 matrix in 113 bits.  Arguments: atoms, angle by which the
// structures are still turned against each other, noise.  Prints the largest
// relative error of 500 fits.
#include <random>

#include "fo_refine.h"

typedef __float128 Quad;

static Quad root(Quad x) {
  Quad r = sqrt((double)x);
  for (int i = 0; i < 4 && x > 0; ++i) r = (r + x / r) / 2;
  return r;
}

static Quad smallest(const double q[10]) {
  Quad A[4][4] = {{q[0], q[1], q[2], q[3]}, {q[1], q[4], q[5], q[6]},
                  {q[2], q[5], q[7], q[8]}, {q[3], q[6], q[8], q[9]}};
  for (int sweep = 0; sweep < 30; ++sweep)
    for (int p = 0; p < 4; ++p)
      for (int r = p + 1; r < 4; ++r) {
        if (A[p][r] == 0) continue;
        const Quad th = (A[r][r] - A[p][p]) / (2 * A[p][r]);
        const Quad t = (th >= 0 ? 1 : -1) / ((th < 0 ? -th : th) + root(th * th + 1));
        const Quad c = 1 / root(t * t + 1), s = t * c;
        for (int k = 0; k < 4; ++k) {
          const Quad a = A[k][p], b = A[k][r];
          A[k][p] = c * a - s * b;
          A[k][r] = s * a + c * b;
        }
        for (int k = 0; k < 4; ++k) {
          const Quad a = A[p][k], b = A[r][k];
          A[p][k] = c * a - s * b;
          A[r][k] = s * a + c * b;
        }
      }
  Quad e = A[0][0];
  for (int i = 1; i < 4; ++i) e = A[i][i] < e ? A[i][i] : e;
  return e;
}

int main(int argc, char** argv) {
  if (argc != 4) return 2;
  const int N = atoi(argv[1]);
  const double angle = atof(argv[2]), noise = atof(argv[3]), r = 1.6 * cbrt(N / 1000.0);
  std::mt19937_64 rng(N);
  std::normal_distribution<double> normal;
  double worst = 0;
  for (int rep = 0; rep < 500; ++rep) {
    const double a = angle * normal(rng), b = angle * normal(rng);
    double q[10] = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
    for (int i = 0; i < N; ++i) {
      const double x = r * normal(rng), y = r * normal(rng), z = r * normal(rng);
      const double u = cos(a) * x - sin(a) * y, v = sin(a) * x + cos(a) * y;
      fo::qmat_accum(q, x, y, z, cos(b) * u - sin(b) * z + noise * normal(rng),
                     v + noise * normal(rng), sin(b) * u + cos(b) * z + noise * normal(rng));
    }
    double dist, M[9];
    fo::kearsley_solve(q, &dist, M);
    const Quad exact = root(smallest(q));
    worst = fmax(worst, fabs((double)((dist - exact) / exact)));
  }
  printf("%.17g\n", worst);
}

// The 4x4 eigen-solve of the fit (fo_refine.h).  For each spectrum on the command
// line (four numbers, and how far the basis departs from the axes, 0: anywhere)
// and 300 random bases: the most sweeps, the largest error of an eigenvalue over
// the largest one, and of V^T V - 1.
#include <random>

#include "fo_refine.h"

int main(int argc, char** argv) {
  std::mt19937_64 rng(4);
  std::normal_distribution<double> normal;
  for (int a = 1; a + 4 < argc; a += 5) {
    const double off = atof(argv[a + 4]);
    double spec[4], worst = 0, orth = 0, top = 0;
    for (int i = 0; i < 4; ++i) top = fmax(top, fabs(spec[i] = atof(argv[a + i])));
    long sweeps = 0;
    for (int rep = 0; rep < 300; ++rep) {
      double B[4][4], A[4][4], V[4][4], w[4];
      for (int i = 0; i < 4; ++i) {  // an orthonormal basis
        for (int k = 0; k < 4; ++k) B[i][k] = off > 0 ? (i == k) + off * normal(rng) : normal(rng);
        for (int pass = 0; pass < 2; ++pass)
          for (int j = 0; j < i; ++j) {
            double d = 0;
            for (int k = 0; k < 4; ++k) d += B[i][k] * B[j][k];
            for (int k = 0; k < 4; ++k) B[i][k] -= d * B[j][k];
          }
        double n = 0;
        for (int k = 0; k < 4; ++k) n += B[i][k] * B[i][k];
        for (int k = 0; k < 4; ++k) B[i][k] /= sqrt(n);
      }
      for (int i = 0; i < 4; ++i)
        for (int j = 0; j <= i; ++j) {
          A[i][j] = 0;
          for (int k = 0; k < 4; ++k) A[i][j] += B[k][i] * spec[k] * B[k][j];
          A[j][i] = A[i][j];
        }
      emu::reciprocal_roots = 0;
      fo::jacobi4(A, V, w);
      // a sweep takes twelve reciprocal roots, fewer once entries are zero
      sweeps = std::max(sweeps, (emu::reciprocal_roots + 11) / 12);
      std::sort(w, w + 4);
      std::sort(spec, spec + 4);
      for (int i = 0; i < 4; ++i) worst = fmax(worst, fabs(w[i] - spec[i]) / top);
      for (int i = 0; i < 4; ++i)
        for (int j = 0; j < 4; ++j) {
          double d = i == j ? -1 : 0;
          for (int k = 0; k < 4; ++k) d += V[k][i] * V[k][j];
          orth = fmax(orth, fabs(d));
        }
    }
    printf("%ld %.3e %.3e\n", sweeps, worst, orth);
  }
}

// The assignment search (fo_refine.h) by workgroups of one to eight wavefronts.
// Arguments: threads, size, seed, 1 for the reversed wavefront order.  Prints
// the assignment or an error.
#include <random>

#include "fo_refine.h"

int main(int argc, char** argv) {
  if (argc != 5) return 2;
  const int threads = atoi(argv[1]), n = atoi(argv[2]);
  std::mt19937_64 rng(atoi(argv[3]));
  std::vector<double> c((size_t)n * n);
  for (double& v : c) v = (double)(rng() >> 11) * 0x1p-53;  // unrelated costs: many free rows
  std::vector<unsigned char> mem(fo::lap_lds_bytes(n) + 16);
  const fo::LapShared ls = fo::lap_carve(mem.data(), n);
  std::vector<int> rowsol(n, -1);
  double red[16];
  int redi[16];
  const std::string err = emu::run(threads, atoi(argv[4]) != 0, [&] {
    fo::lap_solve(
        n, [&](int i, int j) { return c[(size_t)i * n + j]; }, [](double k) { return k; },
        [](int, fo::ColMin&) { return false; }, ls, rowsol.data(), red, redi);
  });
  if (!err.empty()) {
    printf("error: %s\n", err.c_str());
    return 1;
  }
  for (int i = 0; i < n; ++i) printf("%d ", rowsol[i]);
  printf("\n");
  for (double v : c) printf("%.17g ", v);
  printf("\n");
}

// Internal (not exported) declarations shared by the kernel translation units
// and the host runtime of libfastoverlap_hip.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace fo {

// ---------------------------------------------------------------------------
// Spherical batch: one descriptor per pair (device copy is a plain array).
// ---------------------------------------------------------------------------
struct SphPair {
  int natoms;          // atoms in each structure of the pair
  int atom_off;        // first atom in the concatenated position arrays
  int L;               // Jmax of the pair
  int ngroups;         // permutation groups (species)
  int group_off;       // first group in the group arrays
  int ngath;           // atoms that belong to a group (sum of group sizes)
  int gath_off;        // first entry in the gathered-atom index list
  int pad0;
  long long coef_off;  // first complex entry of the pair's C^l (K(L) entries)
  long long rad_off;   // first double of the pair's radial block
  long long ylm_off;   // first complex entry of the pair's Y block Y[q(l,m)][g], m >= 0 (per structure)
  long long c32_off;   // first complex entry of the pair's FP32 C^l in the plane layout
  double scale;        // Gaussian width sigma (<= 0: automatic)
};

struct SphGroup {
  int size;            // atoms in the group
  int gath_off;        // offset of the group inside the pair's gathered list
  long long jk_off;    // prefix of size^2 over the pair's earlier groups
  long long rad_off;   // (L+1) * jk_off : offset inside the pair's radial block
};

// Doubles of a pair's block that hold the harmonic basis' projections of both
// structures, D[atom][degree <= L + 2 nmax][n] (basis 1; basis 0 keeps its
// projections in LDS).
__host__ __device__ inline long long harm_proj_doubles(int ngath, int L, int nmax, int basis) {
  return basis ? 2LL * ngath * (L + 2 * nmax + 1) * (nmax + 1) : 0;
}

// Whether the contraction's 32-bit byte offsets reach a pair's harmonics: an
// item reads the rows of one degree, or of up to four below 16 (at most 31),
// 16 bytes an atom, with a step's reads past the end.
__host__ __device__ inline bool contract_in_reach(int ngath, int L) {
  return 16LL * (L + 1 > 31 ? L + 1 : 31) * ngath <= (1LL << 32) - 4096;
}

// Kernels of the beta planes.
enum PlanePath { kPlaneDirect = 0, kPlaneFft = 1, kPlaneFold = 2 };

// Per (pair, orientation, plane) candidate record written by the plane
// kernels: the plane's values are split into kCandPerPlane parts (the
// spherical kernels: one per wavefront) and entry r lists the largest value
// of part r with a bound on the part's other values.  Entries are unordered;
// parts with no values hold -inf.
constexpr int kCandPerPlane = 4;
constexpr int kMaxCand = 64;     // FP64-re-evaluated candidates listed per grid
struct PlaneCand {
  float val[kCandPerPlane];   // largest value of each part
  int idx[kCandPerPlane];     // its flat grid index (ia*n+ib)*n+ig
  float rest[kCandPerPlane];  // upper bound on every other value of the part
};

// Per (pair, orientation) peak record written by the selection kernel.
struct SphPeak {
  int ind[3];          // integer argmax (alpha, beta, gamma)
  int ncand;           // FP64-re-evaluated candidates
  int noverflow;       // planes re-evaluated in full in FP64
  int pad;
  double value;        // FP64 grid value at the argmax
  double R0[3];        // interpolated Euler angles (fastoverlap/soft.py:127-130)
  double margin;       // FP64 value gap to the runner-up candidate (or +inf)
  double delta;        // FP32 error bound used to collect candidates
  double val32;        // largest FP32 grid value (plane kernels)
};

struct SphOpt {
  double R[3];         // optimised Euler angles
  double f;            // objective -Re sum conj(I) D(R)
  double gnorm;        // gradient max-norm at the last evaluated point
  int iters;
  int evals;           // objective evaluations, line search included
};

struct SphResult {
  double dist;
  double rmat[9];      // total rotation applied to (+/-)X2, row-major
  double R[3];         // Euler angles of the chosen orientation
  int inverted;
  int status;
};

// ---------------------------------------------------------------------------
// Periodic batch
// ---------------------------------------------------------------------------
struct PerPair {
  int natoms;
  int atom_off;
  int ngroups;
  int group_off;
  double box[3];
  double scale;        // sigma (> 0, resolved on the host)
  long long c_off;     // first complex entry of the pair's (2n+1)^3 product
};

struct PerGroup {
  int size;
  int atom_list_off;   // offset of the group in the atom index list
};

struct PerPeak {
  int ind[3];
  int ncand;
  int noverflow;
  int pad;
  double value;
  double disp[3];      // initial displacement (find_max * box / F)
  double margin;
  double delta;
};

struct PerResult {
  double dist;
  double disp[3];
  int iters;
  int status;
};

// ---- kernel launchers (implemented in the .hip files) ---------------------
// Threads of the finish (one workgroup a pair), whose assignment search is a chain
// of small reductions: one wavefront, without barriers, until the largest group
// reaches 192 atoms; then four, whose column scans are shorter; eight above 512 atoms
// while every pair has a CU, or few pairs (nlarge) have a group of 192.  Eight
// against four wavefronts: 64 pairs of 1000 atoms 652 / 924 us, of 544 269 / 295,
// unrelated 544-atom pairs 28.5 / 29.2 ms, 64 of 600 among 4000 small ones 312 /
// 343 us, one among 4095 305 / 336; but 128 among 4000 372 / 345, 320 pairs of 600
// atoms 632 / 571, 512 of 700 801 / 722, 128 of 600 with 896 of 400 672 / 611 (the
// workgroups of a CU wait for each other), and 512 unrelated atoms, which four
// wavefronts divide evenly, 28.3 / 27.6 ms.  Results do not depend on the number.
constexpr int kFinishLarge = 192;
__host__ __device__ inline int finish_threads(int npairs, int nlarge, int maxgroup) {
  if (maxgroup > 512 && (npairs <= 256 || nlarge <= 64)) return 512;
  return maxgroup >= kFinishLarge ? 256 : 64;
}

struct SphLaunch {
  int P;               // pairs
  int n;               // grid side 2B
  int Lmax;            // max L over the pairs
  int Lt;              // degree of the resident Wigner table
  int mingath;         // min gathered atoms over pairs
  int maxgath;         // max gathered atoms over pairs
  int maxatoms;        // max atoms over pairs
  int nlarge;          // pairs with a group of kFinishLarge atoms or more
  long long maxjk;     // max sum of group size^2 over pairs
  int norient;         // 1 or 2
  int mode;            // 0 = alignment (B = (-1)^l A), 1 = general (A,B given)
  int keep_grid;       // write the FP32 grid
  int center;          // subtract centroids
};

}  // namespace fo

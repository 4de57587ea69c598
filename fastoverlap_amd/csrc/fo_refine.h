// FP64 refinement building blocks run by one workgroup per problem:
//  * exact linear assignment (shortest augmenting path with potentials,
//    the method family of Jonker & Volgenant 1987 that the reference cites at
//    f90/alignutils.f90:482-580; the Python path solves the same LAP with
//    munkres, fastoverlap/utils.py:34-46);
//  * Kearsley (1989) quaternion superposition (fastoverlap/utils.py:169-275);
//  * Euler-angle rotation matrix (fastoverlap/utils.py:447-460).
#pragma once
#include <type_traits>

#include "fo_common.h"

namespace fo {

constexpr double kLapInf = 1e300;

// LDS layout of one LAP problem of size <= nmax (bytes = lap_lds_bytes(nmax)).
struct LapShared {
  double* u;
  double* v;
  double* minv;
  int* p;
  int* way;
  int* used;
  int* ra;  // column assigned to row i by the initial column reduction (n + 1: free)
};
FO_HD size_t lap_lds_bytes(int nmax) {
  return (size_t)(nmax + 1) * (3 * sizeof(double) + 4 * sizeof(int));
}
FO_DEV LapShared lap_carve(unsigned char* base, int nmax) {
  LapShared s;
  s.u = (double*)base;
  s.v = s.u + (nmax + 1);
  s.minv = s.v + (nmax + 1);
  s.p = (int*)(s.minv + (nmax + 1));
  s.way = s.p + (nmax + 1);
  s.used = s.way + (nmax + 1);
  s.ra = s.used + (nmax + 1);
  return s;
}

// Wavefront argmin of (value, index) pairs, ties to the smaller index:
// butterflies inside rows of 16 lanes by DPP (quad_perm [1,0,3,2],
// quad_perm [2,3,0,1], row_half_mirror, row_mirror), then the four row
// results through readlane.  Every lane must be active.
template <int CTRL>
FO_DEV void argmin_dpp_step(double& v, int& i) {
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_update_dpp(0, (int)(b & 0xffffffffLL), CTRL, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), CTRL, 0xf, 0xf, true);
  const double ov = __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
  const int oi = __builtin_amdgcn_update_dpp(0, i, CTRL, 0xf, 0xf, true);
  argmin_merge(v, i, ov, oi);
}
FO_DEV double readlane_d(double v, int lane) {
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_readlane((int)(b & 0xffffffffLL), lane);
  const int hi = __builtin_amdgcn_readlane((int)(b >> 32), lane);
  return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}
FO_DEV void wave_argmin_dpp(double& v, int& i) {
  argmin_dpp_step<0xB1>(v, i);
  argmin_dpp_step<0x4E>(v, i);
  argmin_dpp_step<0x141>(v, i);
  argmin_dpp_step<0x140>(v, i);
  double rv = readlane_d(v, 0);
  int ri = __builtin_amdgcn_readlane(i, 0);
#pragma unroll
  for (int r = 16; r < 64; r += 16) argmin_merge(rv, ri, readlane_d(v, r), __builtin_amdgcn_readlane(i, r));
  v = rv;
  i = ri;
}

// Cost of an assignment problem: cost(i, j) = fin(key(i, j)) with fin
// non-decreasing (squared distance and its square root, or the identity), so
// a column's minimum is searched on the keys and fin is taken of the few
// that improve it.  The result is the minimum of the costs at its smallest
// row, as if every cost had been formed.
struct ColMin {
  double key = INFINITY, key2 = INFINITY;  // smallest two keys
  double mn = kLapInf;
  int mi = 0;  // 1-based row, 0: none finite
  template <class Fin>
  FO_DEV void add(double k, int row, Fin fin) {
    key2 = fmin(key2, fmax(key, k));
    if (k < key) {
      key = k;
      const double c = fin(k);
      if (c < mn) {
        mn = c;
        mi = row;
      }
    }
  }
  // across the S lanes (a power of two) that scanned one column's rows
  FO_DEV void join(int S) {
    for (int o = 1; o < S; o <<= 1) {
      const double om = __shfl_xor(mn, o, 64), ok = __shfl_xor(key, o, 64),
                   o2 = __shfl_xor(key2, o, 64);
      const int oi = __shfl_xor(mi, o, 64);
      key2 = fmin(fmin(key2, o2), fmax(key, ok));
      key = fmin(key, ok);
      if (om < mn || (om == mn && oi && (!mi || oi < mi))) {
        mn = om;
        mi = oi;
      }
    }
  }
};

// Column j's nearest row as a wide kernel found it: cost and (1-based) row,
// and how much farther the second nearest row is.
struct NearRec {
  double mn, gap;
  int mi, pad;
};

// Minimum-cost assignment of an n x n cost matrix given by key(i, j) and fin
// (0-based, see ColMin).  rowsol[i] = column assigned to row i.  Ties in the
// column search are broken toward the smaller column index, so the result
// does not depend on the launch width.  near(j, m) may leave column j's
// minimum in m and return true, or return false to have all rows scanned.
// Costs are formed where they are used; the serial parts (the row of each
// column, the list of free rows) go over all threads or 64 rows a step: at
// 716 rows the walk over the rows alone took 36 us.
// Every thread of the block (at most eight wavefronts; red_v, red_i: 16
// entries of LDS) must call this; a one-wavefront block reduces without LDS or
// barrier.
// Returns false (rowsol = identity) if a non-finite cost stops the search.
template <class KeyF, class Fin, class Near>
FO_DEV bool lap_solve(int n, KeyF key, Fin fin, Near near, LapShared s, int* rowsol,
                      double* red_v, int* red_i) {
  const int t = threadIdx.x, bd = blockDim.x;
  auto cost = [&](int i, int j) { return fin(key(i, j)); };
  // column reduction (Jonker & Volgenant 1987): v[j] = min_i c(i, j), and
  // column j goes to its minimising row (ties: smallest row) unless an
  // earlier column took that row.  The duals (u = 0, v) are feasible and
  // tight on these pairs, so the search below only runs for the free rows.
  // S lanes share a column when the block has lanes to spare.
  int S = 1;
  while (2 * S <= 16 && 2 * S * n <= bd) S *= 2;
  const int part = t & (S - 1);
  for (int j = t / S; j < n; j += bd / S) {
    ColMin m;
    if (!near(j, m)) {
      m = ColMin{};
      int i = part;
      for (; i + 3 * S < n; i += 4 * S) {
        const double k0 = key(i, j), k1 = key(i + S, j), k2 = key(i + 2 * S, j),
                     k3 = key(i + 3 * S, j);
        if (fmin(fmin(k0, k1), fmin(k2, k3)) < m.key) {
          m.add(k0, i + 1, fin);
          m.add(k1, i + S + 1, fin);
          m.add(k2, i + 2 * S + 1, fin);
          m.add(k3, i + 3 * S + 1, fin);
        }
      }
      for (; i < n; i += S) m.add(key(i, j), i + 1, fin);
      m.join(S);
    }
    if (part == 0) {
      s.u[j + 1] = 0.0;
      s.v[j + 1] = m.mn < kLapInf ? m.mn : 0.0;  // non-finite column: left to the search
      s.p[j + 1] = 0;
      s.way[j + 1] = m.mi;  // candidate row, read once below
      s.ra[j + 1] = n + 1;  // row j + 1: free
    }
  }
  if (t == 0) {
    s.u[0] = s.v[0] = 0.0;
    s.p[0] = s.way[0] = 0;
  }
  __syncthreads();
  for (int j = 1 + t; j <= n; j += bd)
    if (s.way[j] > 0) atomicMin(&s.ra[s.way[j]], j);
  __syncthreads();
  for (int j = 1 + t; j <= n; j += bd)
    if (s.way[j] > 0 && s.ra[s.way[j]] == j) s.p[j] = s.way[j];
  __syncthreads();
  int half = 0;
  // the free rows in order, 64 at a time (every wavefront reads the same LDS
  // words, so the masks agree)
  for (int i64 = 0; i64 < n; i64 += 64) {
    const int ir = i64 + (t & 63) + 1;
    unsigned long long freem = __ballot(ir <= n && s.ra[ir] > n);
    while (freem) {
      const int i = i64 + __ffsll(freem);
      freem &= freem - 1;
      for (int j = t; j <= n; j += bd) {
        s.minv[j] = kLapInf;
        s.used[j] = 0;
      }
      if (t == 0) s.p[0] = i;
      __syncthreads();
      int j0 = 0;
      for (;;) {
        if (t == 0) s.used[j0] = 1;
        __syncthreads();
        const int i0 = s.p[j0];
        const double ui0 = s.u[i0];
        double best = kLapInf;
        int bj = 0x7fffffff;
        for (int j = 1 + t; j <= n; j += bd) {
          if (!s.used[j]) {
            double cur = cost(i0 - 1, j - 1) - ui0 - s.v[j];
            double mv = s.minv[j];
            if (cur < mv) {
              mv = cur;
              s.minv[j] = cur;
              s.way[j] = j0;
            }
            if (mv < best || (mv == best && j < bj)) {
              best = mv;
              bj = j;
            }
          }
        }
        wave_argmin_dpp(best, bj);
        if (bd > 64) {
          // the wavefronts' minima, in the half of the scratch that the
          // previous step did not use (its readers may still be at it)
          half ^= 8;
          if ((t & 63) == 0) {
            red_v[half + (t >> 6)] = best;
            red_i[half + (t >> 6)] = bj;
          }
          __syncthreads();
          best = red_v[half];
          bj = red_i[half];
          for (int w = 1; w < bd >> 6; ++w) argmin_merge(best, bj, red_v[half + w], red_i[half + w]);
        }
        if (bj == 0x7fffffff || !(best < kLapInf)) {
          // no finite reduced cost left: the costs are not finite numbers
          for (int k = t; k < n; k += bd) rowsol[k] = k;
          __syncthreads();
          return false;
        }
        // whether the column is free is read before the barrier: behind it the
        // first lane may already be at the augmentation, whose first store is
        // this entry, and a wavefront that read it late would stay in the loop
        const int row = s.p[bj];
        const double delta = best;
        for (int j = t; j <= n; j += bd) {
          if (s.used[j]) {
            s.u[s.p[j]] += delta;
            s.v[j] -= delta;
          } else {
            s.minv[j] -= delta;
          }
        }
        __syncthreads();
        j0 = bj;
        if (row == 0) break;
      }
      if (t == 0) {
        do {
          int j1 = s.way[j0];
          s.p[j0] = s.p[j1];
          j0 = j1;
        } while (j0);
      }
      __syncthreads();
    }
  }
  for (int j = 1 + t; j <= n; j += bd) rowsol[s.p[j] - 1] = j - 1;
  __syncthreads();
  return true;
}

// Eigenvalues w and eigenvectors (columns of V) of a symmetric 4x4 matrix by
// Jacobi sweeps.  The six rotations of a sweep go as three pairs of disjoint
// ones, whose angles are formed side by side: a rotation is a chain of a square
// root, a quotient and a reciprocal root, and the solve one lane's latency.
// The matrix is scaled by a power of two first, so that squares of its
// entries neither overflow nor vanish.  One rotation after another by
// quotients took 25000 cycles, more than the rest of a fit of 38 atoms.
// A rotation moves t a_pq from one diagonal entry to the other and sets the
// entry it is for to zero (Rutishauser 1966).  Forming these three by the
// products instead leaves a rounding of the largest entry in all of them, so
// that the smallest eigenvalue lost digits to the larger ones and equal ones (a
// cubic or icosahedral cluster) ran into the cap of 60 sweeps.  An entry within two
// roundings of the smaller of its diagonal entries, or 2^-60 of the largest, is
// left: between equal eigenvalues each sweep would turn it by 45 degrees, and
// their rows with it.  The finish of 2048 icosahedra of 13 atoms: 114 -> 21 us, of
// random clusters the same; rms error of the distance of 1000-atom pairs 1.29e-15
// -> 1.05e-15.
FO_DEV void jacobi4(double A[4][4], double V[4][4], double w[4]) {
  double big = 0.0;
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      V[i][j] = (i == j) ? 1.0 : 0.0;
      big = fmax(big, fabs(A[i][j]));
    }
  const int ex = big > 0.0 && big < INFINITY ? ilogb(big) : 0;
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) A[i][j] = ldexp(A[i][j], -ex);
  struct Angle {
    double t, c, s;
  };
  auto left = [](double app, double aqq, double apq) {
    return fabs(apq) <= __builtin_fma(0x1p-51, fmin(fabs(app), fabs(aqq)), 0x1p-60);
  };
  auto angle = [&](double app, double aqq, double apq) {
    // (no branch: the two angles are formed side by side)
    const double d = 0.5 * (aqq - app), r2 = d * d + apq * apq;
    const double den = fabs(d) + (r2 > 0.0 ? r2 * rsqrt(r2) : 0.0);
    Angle a;
    a.t = den > 0.0 && !left(app, aqq, apq) ? (d < 0.0 ? -apq : apq) / den : 0.0;
    a.c = rsqrt(a.t * a.t + 1.0);
    a.s = a.t * a.c;
    return a;
  };
  auto turn = [&](auto P, auto Q, const Angle& a) {
    constexpr int p = decltype(P)::value, q = decltype(Q)::value;
    const double move = a.t * A[p][q];
    A[p][p] -= move;
    A[q][q] += move;
    A[p][q] = A[q][p] = 0.0;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      if (k == p || k == q) continue;
      const double akp = A[k][p], akq = A[k][q];
      A[k][p] = A[p][k] = a.c * akp - a.s * akq;
      A[k][q] = A[q][k] = a.s * akp + a.c * akq;
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const double vkp = V[k][p], vkq = V[k][q];
      V[k][p] = a.c * vkp - a.s * vkq;
      V[k][q] = a.s * vkp + a.c * vkq;
    }
  };
  auto two = [&](auto P, auto Q, auto R, auto S) {
    const Angle a = angle(A[P.value][P.value], A[Q.value][Q.value], A[P.value][Q.value]);
    const Angle b = angle(A[R.value][R.value], A[S.value][S.value], A[R.value][S.value]);
    turn(P, Q, a);
    turn(R, S, b);
  };
  constexpr std::integral_constant<int, 0> i0{};
  constexpr std::integral_constant<int, 1> i1{};
  constexpr std::integral_constant<int, 2> i2{};
  constexpr std::integral_constant<int, 3> i3{};
  for (int sweep = 0; sweep < 60; ++sweep) {
    bool done = true;
#pragma unroll
    for (int p = 0; p < 4; ++p)
#pragma unroll
      for (int q = p + 1; q < 4; ++q) done &= left(A[p][p], A[q][q], A[p][q]);
    if (done) break;
    two(i0, i1, i2, i3);
    two(i0, i2, i1, i3);
    two(i0, i3, i1, i2);
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) w[i] = ldexp(A[i][i], ex);
}

// Quaternion -> rotation matrix (fastoverlap/utils.py:255-275), row-major.
FO_DEV void q2mx(const double qin[4], double R[9]) {
  double nq = sqrt(qin[0] * qin[0] + qin[1] * qin[1] + qin[2] * qin[2] + qin[3] * qin[3]);
  double Q[4] = {qin[0] / nq, qin[1] / nq, qin[2] / nq, qin[3] / nq};
  R[0] = 2.0 * (0.5 - Q[2] * Q[2] - Q[3] * Q[3]);
  R[4] = 2.0 * (0.5 - Q[1] * Q[1] - Q[3] * Q[3]);
  R[8] = 2.0 * (0.5 - Q[1] * Q[1] - Q[2] * Q[2]);
  R[1] = 2.0 * (Q[1] * Q[2] - Q[0] * Q[3]);
  R[3] = 2.0 * (Q[1] * Q[2] + Q[0] * Q[3]);
  R[2] = 2.0 * (Q[1] * Q[3] + Q[0] * Q[2]);
  R[6] = 2.0 * (Q[1] * Q[3] - Q[0] * Q[2]);
  R[5] = 2.0 * (Q[2] * Q[3] - Q[0] * Q[1]);
  R[7] = 2.0 * (Q[2] * Q[3] + Q[0] * Q[1]);
}

// Kearsley QMAT accumulated over one atom pair (x1 - com1, x2 - com2).
FO_DEV void qmat_accum(double q[10], double x1, double y1, double z1, double x2,
                       double y2, double z2) {
  double XM = x1 - x2, YM = y1 - y2, ZM = z1 - z2;
  double XP = x1 + x2, YP = y1 + y2, ZP = z1 + z2;
  q[0] += XM * XM + YM * YM + ZM * ZM;
  q[1] += -YP * ZM + YM * ZP;
  q[2] += -XM * ZP + XP * ZM;
  q[3] += -XP * YM + XM * YP;
  q[4] += YP * YP + ZP * ZP + XM * XM;
  q[5] += XM * YM - XP * YP;
  q[6] += XM * ZM - XP * ZP;
  q[7] += XP * XP + ZP * ZP + YM * YM;
  q[8] += YM * ZM - YP * ZP;
  q[9] += XP * XP + YP * YP + ZM * ZM;
}

// (hi, lo) += a b, lo holding what the sums and products round off
FO_DEV void add_product(double& hi, double& lo, double a, double b) {
#pragma clang fp contract(off)
  const double p = a * b, pe = __builtin_fma(a, b, -p), s = hi + p, t = s - hi;
  lo += ((hi - (s - t)) + (p - t)) + pe;
  hi = s;
}

// Solve the 4x4 problem: dist = sqrt(min eigenvalue) with the reference's
// clamp of small negative eigenvalues (fastoverlap/utils.py:236-248), and
// the rotation MR (row-major).
FO_DEV void kearsley_solve(const double q[10], double* dist, double MR[9]) {
  double A[4][4] = {{q[0], q[1], q[2], q[3]},
                    {q[1], q[4], q[5], q[6]},
                    {q[2], q[5], q[7], q[8]},
                    {q[3], q[6], q[8], q[9]}};
  double V[4][4], w[4];
  jacobi4(A, V, w);
  double e = w[0], qv[4] = {V[0][0], V[1][0], V[2][0], V[3][0]};
#pragma unroll
  for (int i = 1; i < 4; ++i)
    if (w[i] < e) {
      e = w[i];
#pragma unroll
      for (int k = 0; k < 4; ++k) qv[k] = V[k][i];
    }
  // one first-order correction of the pair against the matrix itself takes out what
  // the rotations rounded; near-equal eigenvalues leave the vector.  The
  // residual is summed in twice the precision: its terms are of the size of the
  // largest eigenvalue and the distance is the root of the smallest.
  double rv[4];
  const int at[4][4] = {{0, 1, 2, 3}, {1, 4, 5, 6}, {2, 5, 7, 8}, {3, 6, 8, 9}};
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    double hi = 0.0, lo = 0.0;
    add_product(hi, lo, -e, qv[i]);
#pragma unroll
    for (int j = 0; j < 4; ++j) add_product(hi, lo, q[at[i][j]], qv[j]);
    rv[i] = hi + lo;
  }
  const double wmax = fmax(fmax(w[0], w[1]), fmax(w[2], w[3])), e0 = e;
  e += qv[0] * rv[0] + qv[1] * rv[1] + qv[2] * rv[2] + qv[3] * rv[3];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const double gap = w[i] - e0;
    const double dot = V[0][i] * rv[0] + V[1][i] * rv[1] + V[2][i] * rv[2] + V[3][i] * rv[3];
    const double f = gap > 1e-6 * wmax ? dot / gap : 0.0;
#pragma unroll
    for (int k = 0; k < 4; ++k) qv[k] -= f * V[k][i];
  }
  if (e < 0.0) e = (fabs(e) < 1e-6) ? 0.0 : -e;
  *dist = sqrt(e);
  q2mx(qv, MR);
}

// EulerM(a, b, y) = My . Mb . Ma  (fastoverlap/utils.py:447-460), row-major.
FO_HD void euler_matrix(double a, double b, double y, double M[9]) {
  double sa, ca, sb, cb, sy, cy;
  sincos(a, &sa, &ca);
  sincos(b, &sb, &cb);
  sincos(y, &sy, &cy);
  // Mb . Ma
  double T[9] = {cb * ca, -cb * sa, -sb, sa, ca, 0.0, sb * ca, -sb * sa, cb};
  // My . T
  M[0] = cy * T[0] - sy * T[3];
  M[1] = cy * T[1] - sy * T[4];
  M[2] = cy * T[2] - sy * T[5];
  M[3] = sy * T[0] + cy * T[3];
  M[4] = sy * T[1] + cy * T[4];
  M[5] = sy * T[2] + cy * T[5];
  M[6] = T[6];
  M[7] = T[7];
  M[8] = T[8];
}

}  // namespace fo

// Periodic (bulk) overlap-alignment kernels for gfx950.
//
//   k_per_sf       structure factors C_s(k) = sum_j e^{-i k.r_j} for the
//                  (2n+1)^3 k-cube, separable per axis, and the weighted
//                  product sum_s C1_s conj(C2_s) e^{-|k|^2 s^2}   (FP64)
//   k_per_product  the same product from caller-supplied coefficients
//   k_per_plane    |forward 3D DFT| of the corner-padded product on an F^3
//                  grid, one x-plane per workgroup (pruned: only 2n+1 of F
//                  inputs per axis are non-zero), top candidates   (FP32)
//   k_per_select   FP64 re-evaluation of every candidate within the FP32
//                  error bound -> exact argmax, parabolic offsets, disp
//   k_per_refine   LAP + mean-shift iteration (FP64)
// (reference: fastoverlap/periodicAlignment.py:27-80, :384-460)
#include "fo_common.h"
#include "fo_internal.h"
#include "fo_refine.h"
#include <algorithm>

namespace fo {

// One k-vector's weighted overlap product: sum over the groups of C1 conj(C2)
// in this fused order, then the weight.  Every path to Cprod uses these two
// (the same coefficients give the same product to the last bit).
FO_DEV void overlap_add(double2& s, double2 c1, double2 c2) {
  s.x = __builtin_fma(c1.x, c2.x, __builtin_fma(c1.y, c2.y, s.x));
  s.y = __builtin_fma(c1.y, c2.x, __builtin_fma(-c1.x, c2.y, s.y));
}
FO_DEV double overlap_weight(const PerPair& d, int a, int b, int c) {
  const double kx = 2.0 * kPi * a / d.box[0];
  const double ky = 2.0 * kPi * b / d.box[1];
  const double kz = 2.0 * kPi * c / d.box[2];
  return exp(-(__builtin_fma(kx, kx, __builtin_fma(ky, ky, kz * kz))) * d.scale * d.scale);
}

// ---------------------------------------------------------------------------
// Structure factors on the matrix cores.  With cos / sin of a x, b y, c z
// (a, b, c >= 0, angles in units of the box) the sums over a group's atoms
//   S[X][Y][Z](a, b, c) = sum_j X_j(a) Y_j(b) Z_j(c),   X, Y, Z in {cos, sin},
// are NB^3 real numbers (NB = 2 nk + 1; sin(0) drops out) that give C(k) for
// every sign of a, b, c, and C(-k) = conj C(k) exactly: an eighth of the
// multiply-adds of the complex sum over the full cube.  Per a they are a
// real product over the atoms, rows (X, Y(b)) by columns Z(c).
//
// One workgroup per (a >= 0, pair), waves 0-3 on the first and 4-7 on the
// second structure.  Per tile of kSFTile atoms the phases of both structures
// go to LDS ([atom]: cos/sin a x, the NB values of y, the NB values of z),
// then v_mfma_f64_16x16x4f64 over four atoms a step: wave w owns row tile(s)
// w & 3 (+ 4) and all CT column tiles, the A operand X_j Y_j(b) is formed
// from two LDS reads.  The group's S of both structures then meet in LDS,
// where one thread forms C1, C2 of each (b, c) and adds their product.
//
// CT = ceil(NB / 16) column tiles; 2 NB rows are at most 4 tiles for CT <= 2
// and 8 above (two per wave).  Bound: the latency of the phase stage, which
// every a repeats (one sincospi per atom and axis, multiples by products) and
// its barriers; the products take 23 us of the 93 below at the matrix rate
// (34 of 48 rows and 17 of 32 columns used at nk = 8).  For CT <= 2 registers are
// held to 128, two workgroups a CU, so that one's phases run beside the other's
// products (114 -> 93 and 145 -> 125 us below, 19 spilled outside the product loop).  Against the complex
// VALU sum over the full cube: 256 atoms, nk = 8: 145 -> 23 us for one pair,
// 565 -> 93 us for 128; 24 pairs of 601..1024 atoms, nk = 14: 1428 -> 125 us;
// relative error against 64-bit-exact phases 1.6e-15 -> 0.8e-15 (256 atoms).
// ---------------------------------------------------------------------------
constexpr int kSFTile = 64;   // atoms per LDS tile
constexpr int kSFThreads = 512;

FO_HD int sf_stride(int NB) { return 2 * NB + 3; }  // doubles per atom (odd)

template <int CT>
__global__ void __launch_bounds__(kSFThreads, CT <= 2 ? 4 : 1) k_per_sf(
    const PerPair* __restrict__ pd, const PerGroup* __restrict__ grp,
    const int* __restrict__ atoms, const double* __restrict__ pos1,
    const double* __restrict__ pos2, int nk, double2* __restrict__ Cprod,
    double2* __restrict__ C1out, double2* __restrict__ C2out) {
  constexpr int RTW = CT <= 2 ? 1 : 2;                         // row tiles per wave
  constexpr int kMaxNB = 16 * CT - 1;                          // NB is odd
  constexpr int ITEMS = (kMaxNB * kMaxNB + kSFThreads - 1) / kSFThreads;
  extern __shared__ __align__(16) double sf_lds[];
  const int NB = 2 * nk + 1, SR = sf_stride(NB);
  const int a = blockIdx.x, p = blockIdx.y, t = threadIdx.x;
  const PerPair d = pd[p];
  const int wv = __builtin_amdgcn_readfirstlane(t >> 6), st = wv >> 2, wr = wv & 3;
  const int ln = t & 63, col = ln & 15, kq = ln >> 4;
  const int rows = a > 0 ? 2 * NB : NB;  // rows (X, beta): X * NB + beta; sin(0) = 0
  const int nrt = (rows + 15) >> 4;
  // this lane's A operand: LDS offsets of X and Y of row 16 rt + col (rows
  // beyond the last read the last row and are not stored)
  int ox[RTW], oy[RTW], oz[CT];
#pragma unroll
  for (int q = 0; q < RTW; ++q) {
    const int r = min(16 * (wr + 4 * q) + col, rows - 1);
    ox[q] = r >= NB ? 1 : 0;
    oy[q] = 2 + (r >= NB ? r - NB : r);
  }
#pragma unroll
  for (int c = 0; c < CT; ++c) oz[c] = 2 + NB + min(16 * c + col, NB - 1);
  double* const tile = sf_lds + st * kSFTile * SR;
  // phase stage: wave pj = (structure, axis), lane = atom of the tile
  static_assert(kSFTile == 64 && kSFThreads >= 6 * 64, "a wave per structure and axis");
  const int pj = wv, ps = pj >= 3 ? 1 : 0, pax = pj - 3 * ps, pa = ln;
  const double pbox = d.box[pj < 6 ? pax : 0];
  double2 prod[ITEMS];
#pragma unroll
  for (int q = 0; q < ITEMS; ++q) prod[q] = make_double2(0.0, 0.0);
  const long long plane = (long long)NB * NB, cube = plane * NB;
  for (int g = 0; g < d.ngroups; ++g) {
    const PerGroup G = grp[d.group_off + g];
    v4d acc[RTW][CT];
#pragma unroll
    for (int q = 0; q < RTW; ++q)
#pragma unroll
      for (int c = 0; c < CT; ++c) acc[q][c] = v4d{0.0, 0.0, 0.0, 0.0};
    // thread (s, axis, atom) of the phase stage; the next tile's coordinate is
    // loaded before the products of this one
    auto coord = [&](int j) {
      return pj < 2 * 3 && j < G.size
                 ? (ps ? pos2 : pos1)[3LL * (d.atom_off + atoms[G.atom_list_off + j]) + pax]
                 : 0.0;
    };
    double xnext = coord(pa);
    for (int j0 = 0; j0 < G.size; j0 += kSFTile) {
      const int jt = min(kSFTile, G.size - j0), jp = (jt + 3) & ~3;  // padded to MFMA steps
      __syncthreads();  // readers of the previous tile (or of S) are done
      if (pj < 2 * 3) {
        double* o = sf_lds + (ps * kSFTile + pa) * SR;
        const bool ok = pa < jt;  // padding atoms add nothing
        // x / box as its fraction of the nearest integer plus the quotient's
        // remainder: the base angle is as accurate as its last bit
        const double q = xnext / pbox, f = (q - rint(q)) + __builtin_fma(-q, pbox, xnext) / pbox;
        double sn, cs;
        sincospi(2.0 * (pax == 0 ? a : 1) * f, &sn, &cs);
        if (!ok) sn = cs = 0.0;
        if (pax == 0) {
          o[0] = cs;
          o[1] = sn;
        } else {
          o += pax == 1 ? 2 : 2 + NB;
          o[0] = ok ? 1.0 : 0.0;
          if (nk > 0) {
            o[1] = cs;
            o[2] = sn;
          }
          // e^{i m f} = e^{i h f} e^{i (m - h) f}, h = m / 2
          for (int m = 2; m <= nk; ++m) {
            const int h = m >> 1, k = m - h;
            const double hc = o[2 * h - 1], hs = o[2 * h], kc = o[2 * k - 1], ks = o[2 * k];
            o[2 * m - 1] = hc * kc - hs * ks;
            o[2 * m] = hc * ks + hs * kc;
          }
        }
        xnext = coord(j0 + kSFTile + pa);
      }
      __syncthreads();
      if (wr < nrt) {  // wave-uniform
#pragma unroll 2
        for (int s4 = 0; s4 < jp; s4 += 4) {
          const double* o = tile + (s4 + kq) * SR;
          double zv[CT], av[RTW];
#pragma unroll
          for (int c = 0; c < CT; ++c) zv[c] = o[oz[c]];
#pragma unroll
          for (int q = 0; q < RTW; ++q) av[q] = o[ox[q]] * o[oy[q]];
#pragma unroll
          for (int q = 0; q < RTW; ++q) {
            if (q > 0 && wr + 4 * q >= nrt) continue;  // wave-uniform
#pragma unroll
            for (int c = 0; c < CT; ++c) acc[q][c] = mfma64(av[q], zv[c], acc[q][c]);
          }
        }
      }
    }
    // S of both structures -> LDS [structure][row][gamma] (over the tiles)
    __syncthreads();
    double* const S = sf_lds + (long long)st * 2 * plane;
#pragma unroll
    for (int q = 0; q < RTW; ++q)
#pragma unroll
      for (int c = 0; c < CT; ++c)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int r = 16 * (wr + 4 * q) + 4 * i + kq, gm = 16 * c + col;
          if (r < rows && gm < NB) S[r * NB + gm] = acc[q][c][i];
        }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < ITEMS; ++q) {
      const int e = t + q * kSFThreads;
      if (e >= plane) continue;
      const int b = e / NB - nk, c = e % NB - nk;
      const int ab = abs(b), ac = abs(c);
      const double sb = b < 0 ? -1.0 : 1.0, sc = c < 0 ? -1.0 : 1.0;
      const int bc = ab ? 2 * ab - 1 : 0, cc = ac ? 2 * ac - 1 : 0;
      double2 C[2];
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        // row / column of the cosine; the sine follows it (none at 0)
        const double* Z = sf_lds + s * 2 * plane + bc * NB + cc;
        const int nb1 = ab ? NB : 0, nx = a > 0 ? (int)plane : 0;
        const double hb = ab ? sb : 0.0, hc = ac ? sc : 0.0, hx = a > 0 ? 1.0 : 0.0;
        const int z1 = ac ? 1 : 0;
        const double ccc = Z[0], ccs = Z[z1], csc = Z[nb1], css = Z[nb1 + z1];
        const double scc = Z[nx], scs = Z[nx + z1], ssc = Z[nx + nb1], sss = Z[nx + nb1 + z1];
        // (cx - i sx)(cy - i hb sy)(cz - i hc sz), the sine sums signed by b, c
        C[s].x = ccc - hx * hb * ssc - hb * hc * css - hx * hc * scs;
        C[s].y = -(hb * csc + hx * scc + hc * ccs - hx * hb * hc * sss);
      }
      overlap_add(prod[q], C[0], C[1]);
      if (C1out) {
        const long long o = (long long)(d.group_off + g) * cube;
        const long long kp = (nk + a) * plane + e, km = (nk - a) * plane + (plane - 1 - e);
        C1out[o + kp] = C[0];
        C2out[o + kp] = C[1];
        if (a > 0) {
          C1out[o + km] = cconj(C[0]);
          C2out[o + km] = cconj(C[1]);
        }
      }
    }
  }
#pragma unroll
  for (int q = 0; q < ITEMS; ++q) {
    const int e = t + q * kSFThreads;
    if (e >= plane) continue;
    const double2 v = cscale(prod[q], overlap_weight(d, a, e / NB - nk, e % NB - nk));
    double2* o = Cprod + d.c_off;
    o[(nk + a) * plane + e] = v;
    if (a > 0) o[(nk - a) * plane + (plane - 1 - e)] = cconj(v);
  }
}

// Weighted product from caller-supplied per-group coefficients
// (the Cs= path of fastoverlap/periodicAlignment.py:408-438).
__global__ void k_per_product(const PerPair* __restrict__ pd, int nk,
                              const double2* __restrict__ C1, const double2* __restrict__ C2,
                              double2* __restrict__ Cprod) {
  const int NB = 2 * nk + 1, p = blockIdx.y;
  const PerPair d = pd[p];
  const long long cube = (long long)NB * NB * NB;
  for (long long e = blockIdx.x * (long long)blockDim.x + threadIdx.x; e < cube;
       e += (long long)gridDim.x * blockDim.x) {
    const int a = (int)(e / (NB * NB)), b = (int)((e / NB) % NB), c = (int)(e % NB);
    double2 s = make_double2(0.0, 0.0);
    for (int g = 0; g < d.ngroups; ++g) {
      const long long o = (long long)(d.group_off + g) * cube + e;
      overlap_add(s, C1[o], C2[o]);
    }
    Cprod[d.c_off + e] = cscale(s, overlap_weight(d, a - nk, b - nk, c - nk));
  }
}

// The same product from per-structure coefficients shared by many pairs:
// pair p multiplies structure idx1[p] with structure idx2[p] (alignGroup's
// coefficient reuse, fastoverlap/periodicAlignment.py:466-473).  Cs holds
// nstruct x ngroups cubes; every pair has the same ngroups.
__global__ void k_per_product_indexed(const PerPair* __restrict__ pd, int nk,
                                      const double2* __restrict__ Cs, const int* __restrict__ idx1,
                                      const int* __restrict__ idx2, double2* __restrict__ Cprod) {
  const int NB = 2 * nk + 1, p = blockIdx.y;
  const PerPair d = pd[p];
  const long long cube = (long long)NB * NB * NB;
  const double2* A = Cs + (long long)idx1[p] * d.ngroups * cube;
  const double2* B = Cs + (long long)idx2[p] * d.ngroups * cube;
  for (long long e = blockIdx.x * (long long)blockDim.x + threadIdx.x; e < cube;
       e += (long long)gridDim.x * blockDim.x) {
    const int a = (int)(e / (NB * NB)), b = (int)((e / NB) % NB), c = (int)(e % NB);
    double2 s = make_double2(0.0, 0.0);
    for (int g = 0; g < d.ngroups; ++g)
      overlap_add(s, A[(long long)g * cube + e], B[(long long)g * cube + e]);
    Cprod[d.c_off + e] = cscale(s, overlap_weight(d, a - nk, b - nk, c - nk));
  }
}

// sum of |C| over the slice a = x of the product (workgroups x < NB), for the
// selection's error bound
FO_DEV void slice_abound(const double2* C, int x, int NB, double* out) {
  __shared__ double sa[4];
  if (x >= NB) return;
  const double2* S = C + (long long)x * NB * NB;
  double v = 0.0;
  for (int e = threadIdx.x; e < NB * NB; e += 256) v += sqrt(S[e].x * S[e].x + S[e].y * S[e].y);
  v = block_sum(v, sa);
  if (threadIdx.x == 0) out[x] = v;
}

// |f(x,y,z)|, f = sum_{a,b,c} C[a,b,c] e^{-2 pi i (a x + b y + c z)/F}, for
// one x-plane per workgroup (numpy fftn with C at the array corner,
// fastoverlap/periodicAlignment.py:439-440).  For products that need not be
// Hermitian (supplied coefficients) and where f itself is kept; k_per_plane_real
// serves the others.
__global__ void __launch_bounds__(256) k_per_plane(
    const PerPair* __restrict__ pd, int nk, int F, const double2* __restrict__ Cprod,
    const float2* __restrict__ twg, PlaneCand* __restrict__ cand, double* __restrict__ abound,
    float* __restrict__ grid, float2* __restrict__ cgrid) {
  extern __shared__ __align__(16) unsigned char smem[];
  const int NB = 2 * nk + 1;
  const int x = blockIdx.x, p = blockIdx.y, t = threadIdx.x, bd = blockDim.x;
  const PerPair d = pd[p];
  float2* tw = (float2*)smem;       // [F]
  float2* H = tw + F;               // [NB][NB]
  float2* G = H + NB * NB;          // [NB][F]
  float* rv = (float*)(G + NB * F);
  int* ri = (int*)(rv + 16);
  for (int k = t; k < F; k += bd) tw[k] = twg[k];
  __syncthreads();
  const double2* C = Cprod + d.c_off;
  for (int e = t; e < NB * NB; e += bd) {
    float2 acc = make_float2(0.f, 0.f);
    int ph = 0;
    for (int a = 0; a < NB; ++a) {
      const double2 cv = C[(long long)a * NB * NB + e];
      const float2 w = tw[ph];
      const float cx = (float)cv.x, cy = (float)cv.y;
      acc.x += cx * w.x - cy * w.y;
      acc.y += cx * w.y + cy * w.x;
      ph += x;
      if (ph >= F) ph -= F;
    }
    H[e] = acc;
  }
  __syncthreads();
  for (int e = t; e < NB * F; e += bd) {
    const int b = e / F, z = e % F;
    float2 acc = make_float2(0.f, 0.f);
    int ph = 0;
    for (int c = 0; c < NB; ++c) {
      const float2 h = H[b * NB + c];
      const float2 w = tw[ph];
      acc.x += h.x * w.x - h.y * w.y;
      acc.y += h.x * w.y + h.y * w.x;
      ph += z;
      if (ph >= F) ph -= F;
    }
    G[e] = acc;
  }
  __syncthreads();
  float bv = -INFINITY, dm = -INFINITY;
  int bi = 0x7fffffff;
  for (int e = t; e < F * F; e += bd) {
    const int y = e / F, z = e % F;
    float2 acc = make_float2(0.f, 0.f);
    int ph = 0;
    for (int b = 0; b < NB; ++b) {
      const float2 gv = G[b * F + z];
      const float2 w = tw[ph];
      acc.x += gv.x * w.x - gv.y * w.y;
      acc.y += gv.x * w.y + gv.y * w.x;
      ph += y;
      if (ph >= F) ph -= F;
    }
    const float val = sqrtf(acc.x * acc.x + acc.y * acc.y);
    const int flat = (x * F + y) * F + z;
    if (grid) grid[(long long)p * F * F * F + flat] = val;
    if (cgrid) cgrid[(long long)p * F * F * F + flat] = acc;
    if (val > bv) {
      dm = fmaxf(dm, bv);
      bv = val;
      bi = flat;
    } else {
      dm = fmaxf(dm, val);
    }
  }
  bool taken = false;
  PlaneCand out;
  float fifth = -INFINITY;
  for (int r = 0; r <= kCandPerPlane; ++r) {
    float v = taken ? -INFINITY : bv;
    int i = taken ? 0x7fffffff : bi;
    block_argmax(v, i, rv, ri);
    if (r < kCandPerPlane) {
      out.val[r] = v;
      out.idx[r] = i;
    } else {
      fifth = v;
    }
    if (!taken && i == bi && v == bv) taken = true;
  }
  int dummy = 0;
  block_argmax(dm, dummy, rv, ri);
  // one part: the block's top kCandPerPlane, the bound in rest[0]
  out.rest[0] = fmaxf(fifth, dm);
  for (int r = 1; r < kCandPerPlane; ++r) out.rest[r] = -INFINITY;
  if (t == 0) cand[(long long)p * F + x] = out;
  slice_abound(C, x, NB, abound + (long long)p * NB);
}

// The same planes for a Hermitian product (structure factors of real
// densities): up to a phase f is the real sum
//   g(x,y,z) = sum_{|a|,|b|,|c| <= nk} C[a,b,c] e^{-2 pi i (a x + b y + c z)/F}.
// Per plane x, with the real basis phi_0 = 1, phi_{2m-1} = cos m, phi_{2m} =
// sin m over b and over c (NB functions each):
//   1. H[b,c] = sum_a C w^{a x} for c >= 0 on the vector units, folded over
//      +-b into the real coefficients R[r over c][k over b] (LDS);
//   2. G[r][y] = sum_k R[r][k] phi_k(y)  and
//   3. g[y][z] = sum_r G[r][y] phi_r(z)  on v_mfma_f32_16x16x4f32: a
//      wavefront owns 16 columns y, and register i of lane group q, row 4 q + i
//      of a result tile of 2, is the A operand of 3 at the step i of the tile; it
//      holds the function r = 4 i + 3 - q of the tile, so that a step takes four
//      consecutive functions.
// All three sums run from the highest order down, +-a together in 1: the
// structure factors fall off with it, and a sum that starts at its small end
// rounds less.  rms error over the rms of the grid: 0.46e-7 for 256 atoms, nk = 8
// (upwards 1.6e-7, the complex transform 1.2e-7), 0.31e-7 for 1000, nk = 14 (1.5
// and 1.3e-7).
// phi: (NB + 1) rows of F in LDS, the last one zero (padding of r and k); the row
// stride is an odd multiple of 16, so the four rows of a step start in different
// banks.
// XP planes share the table; their products read C through the caches.
// Rounding, in units u = 2^-24 of sum |C| to first order: stage 1 rounds C, the
// twiddles, 2 NB additions a component and the fold, 2 NB + 3, times 2 for both
// components with |cos| + |sin| over b and c; 2 and 3 round phi, NB products and
// their sums, NB + 2 each, times sqrt 2 (sum |R| |phi| |phi| <= sqrt 2 sum |C|):
// 6.9 NB + 12 in all.  real_plane_delta, 9 NB + 64, is that with room for the
// second order and for matrix units that round products apart from sums.
// Against the complex transform on the vector units, which formed every F^2 NB
// term of a plane: 259 -> 72 us for 128 pairs of nk = 8, F = 64, 111 -> 33 us for
// 24 of nk = 14, F = 60, 20 -> 10 us for one pair.  Bound: stage 1 (two FP64
// products read, four conversions and eight FP32 operations a term) and the
// candidate test of every value.
constexpr int kPlaneXP = 4;
FO_HD double real_plane_delta(int NB) { return (9.0 * NB + 64.0) * 5.9604644775390625e-08; }
FO_HD int real_plane_fs(int F) { return ((F + 15) & ~15) | 16; }  // row stride of phi
FO_HD int real_plane_ks(int NB) { return ((NB + 3) & ~3) + 1; }  // row stride of R

template <int NT>
__global__ void __launch_bounds__(256) k_per_plane_real(
    const PerPair* __restrict__ pd, int nk, int F, int XP, const double2* __restrict__ Cprod,
    const float2* __restrict__ twg, PlaneCand* __restrict__ cand, double* __restrict__ abound,
    float* __restrict__ grid) {
  extern __shared__ __align__(16) unsigned char smem[];
  const int NB = 2 * nk + 1, FS = real_plane_fs(F), KS = real_plane_ks(NB);
  const int p = blockIdx.y, t = threadIdx.x, x0 = blockIdx.x * XP;
  const PerPair d = pd[p];
  float2* tw = (float2*)smem;         // [F], e^{-2 pi i j / F}
  float* phi = (float*)(tw + F);      // [NB + 1][FS]
  float* R = phi + (NB + 1) * FS;     // [XP][NB][KS]
  for (int k = t; k < F; k += 256) tw[k] = twg[k];
  __syncthreads();
  const double2* C = Cprod + d.c_off;
  const int nb = nk + 1, plane = NB * NB;
  for (int e = t; e < XP * nb * nb; e += 256) {
    const int xi = e / (nb * nb), r = e - xi * nb * nb, b = r / nb, c = r - b * nb;
    const int x = min(x0 + xi, F - 1);
    const double2* Cp = C + (nk + b) * NB + nk + c;
    const double2* Cm = C + (nk - b) * NB + nk + c;
    float2 hp = make_float2(0.f, 0.f), hm = hp;
    auto add = [&](float2& h, double2 z, float2 w) {
      const float zx = (float)z.x, zy = (float)z.y;
      h.x += zx * w.x - zy * w.y;
      h.y += zx * w.y + zy * w.x;
    };
    const long long mid = (long long)nk * plane;
    int ph = nk * x % F;
#pragma unroll 2
    for (int a = nk; a > 0; --a) {  // +-a together, the twiddle of -a is conjugate
      const long long o = (long long)a * plane;
      const float2 w = tw[ph], wc = make_float2(w.x, -w.y);
      const double2 up = Cp[mid + o], um = Cp[mid - o], vp = Cm[mid + o], vm = Cm[mid - o];
      add(hp, up, w);
      add(hp, um, wc);
      add(hm, vp, w);
      add(hm, vm, wc);
      ph -= x;
      if (ph < 0) ph += F;
    }
    add(hp, Cp[mid], make_float2(1.f, 0.f));
    add(hm, Cm[mid], make_float2(1.f, 0.f));
    const float sc = c ? 2.f : 1.f;  // the terms of -c
    float* re = R + ((long long)xi * NB + (c ? 2 * c - 1 : 0)) * KS;
    float* im = re + KS;  // c > 0 only
    if (b == 0) {
      re[0] = sc * hp.x;
      if (c) im[0] = sc * hp.y;
    } else {
      re[2 * b - 1] = sc * (hp.x + hm.x);
      re[2 * b] = sc * (hp.y - hm.y);
      if (c) {
        im[2 * b - 1] = sc * (hp.y + hm.y);
        im[2 * b] = -sc * (hp.x - hm.x);
      }
    }
  }
  for (int e = t; e < XP * NB * (KS - 1 - NB); e += 256) {
    const int row = e / (KS - 1 - NB);
    R[row * KS + NB + e - row * (KS - 1 - NB)] = 0.f;
  }
  for (int e = t; e < (NB + 1) * FS; e += 256) {
    const int k = e / FS, j = e - k * FS;
    float v = 0.f;
    if (k < NB && j < F) {
      const float2 w = tw[((k + 1) >> 1) * j % F];
      v = (k & 1) || k == 0 ? w.x : -w.y;
    }
    phi[e] = v;
  }
  __syncthreads();
  const int wv = __builtin_amdgcn_readfirstlane(t >> 6), ln = t & 63, col = ln & 15, q = ln >> 4;
  const int nyt = (F + 15) >> 4, ksteps = (NB + 3) >> 2;
  // function of row col of a result tile of stage 2
  const int fr = 4 * (col & 3) + 3 - (col >> 2);
  for (int xi = 0; xi < XP; ++xi) {
    const int x = x0 + xi;
    if (x >= F) break;  // uniform
    const float* Rx = R + (long long)xi * NB * KS;
    float bv = -INFINITY, dm = -INFINITY;
    int bi = 0x7fffffff;
    for (int yt = wv; yt < nyt; yt += 4) {
      v4f G[NT];
#pragma unroll
      for (int tt = 0; tt < NT; ++tt) G[tt] = v4f{0.f, 0.f, 0.f, 0.f};
      for (int s = ksteps - 1; s >= 0; --s) {
        const int k = 4 * s + 3 - q;
        const float b = phi[min(k, NB) * FS + 16 * yt + col];
#pragma unroll
        for (int tt = 0; tt < NT; ++tt) {
          const float a = Rx[min(16 * tt + fr, NB - 1) * KS + k];
          G[tt] = __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, G[tt], 0, 0, 0);
        }
      }
      for (int zt = 0; zt < nyt; ++zt) {
        const float* pz = phi + 16 * zt + col;
        v4f acc = v4f{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int tt = NT - 1; tt >= 0; --tt)
#pragma unroll
          for (int i = 3; i >= 0; --i) {
            if (16 * tt + 4 * i >= NB) continue;  // uniform
            const float b = pz[min(16 * tt + 4 * i + 3 - q, NB) * FS];
            acc = __builtin_amdgcn_mfma_f32_16x16x4f32(G[tt][i], b, acc, 0, 0, 0);
          }
        const int z = 16 * zt + col;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int y = 16 * yt + 4 * q + i;
          const float val = fabsf(acc[i]);
          if (y < F && z < F) {
            const int flat = (x * F + y) * F + z;
            if (grid) grid[(long long)p * F * F * F + flat] = val;
            if (val > bv) {
              dm = fmaxf(dm, bv);
              bv = val;
              bi = flat;
            } else {
              dm = fmaxf(dm, val);
            }
          }
        }
      }
    }
    float v[1] = {bv}, r[1] = {dm};
    int id[1] = {bi};
    wave_top2(v, id, r);
    if (ln == 0) {
      PlaneCand* o = cand + (long long)p * F + x;
      o->val[wv] = v[0];
      o->idx[wv] = id[0];
      o->rest[wv] = r[0];
    }
  }
  for (int xi = 0; xi < XP; ++xi) slice_abound(C, x0 + xi, NB, abound + (long long)p * NB);
}

struct PerGridCtx {
  int NB, F;
  const double2* C;
};

// FP64 |f| at up to kSelPoints grid points with at most three x and five
// (x, y) values among them, in one pass over the product: H[x][b, c] =
// sum_a C w^{a x} (XB of the x values a pass, coalesced over (b, c)), then
// G[x, y][c] = sum_b H w^{b y} and the points' sums over c, a wavefront each.
// tw: the F twiddles in LDS; H: [XB][NB^2], G: [kSelPairs][NB].  Every thread
// must call it (kSelThreads).
constexpr int kSelThreads = 512;
constexpr int kSelPoints = 7, kSelPairs = 5, kSelXs = 3;
struct SelPoints {
  int np, nxy, nx;
  int x[kSelXs];                       // distinct x
  int xy_x[kSelPairs], xy_y[kSelPairs];  // (index into x, y)
  int pt_xy[kSelPoints], pt_z[kSelPoints];
  double val[kSelPoints];
};
template <int XB>
FO_DEV void per_eval64(const PerGridCtx& c, SelPoints& s, const double2* tw, double2* H,
                       double2* G) {
  const int NB = c.NB, F = c.F, plane = NB * NB, t = threadIdx.x;
  for (int x0 = 0; x0 < s.nx; x0 += XB) {
    int xs[XB];
#pragma unroll
    for (int q = 0; q < XB; ++q) xs[q] = s.x[min(x0 + q, s.nx - 1)];
    for (int e = t; e < plane; e += kSelThreads) {
      double2 acc[XB];
      int ph[XB];
#pragma unroll
      for (int q = 0; q < XB; ++q) {
        acc[q] = make_double2(0.0, 0.0);
        ph[q] = 0;
      }
#pragma unroll 8
      for (int a = 0; a < NB; ++a) {
        const double2 v = c.C[(long long)a * plane + e];
#pragma unroll
        for (int q = 0; q < XB; ++q) {
          acc[q] = cadd(acc[q], cmul(v, tw[ph[q]]));
          ph[q] += xs[q];
          if (ph[q] >= F) ph[q] -= F;
        }
      }
#pragma unroll
      for (int q = 0; q < XB; ++q) H[q * plane + e] = acc[q];
    }
    __syncthreads();
    for (int e = t; e < s.nxy * NB; e += kSelThreads) {
      const int k = e / NB, cc = e - k * NB, q = s.xy_x[k] - x0, y = s.xy_y[k];
      if (q < 0 || q >= XB) continue;
      double2 acc = make_double2(0.0, 0.0);
      int ph = 0;
#pragma unroll 4
      for (int b = 0; b < NB; ++b) {
        acc = cadd(acc, cmul(H[q * plane + b * NB + cc], tw[ph]));
        ph += y;
        if (ph >= F) ph -= F;
      }
      G[e] = acc;
    }
    __syncthreads();
  }
  const int w = t >> 6, ln = t & 63;
  if (w < s.np) {
    // NB <= 63: one term a lane
    double2 v = make_double2(0.0, 0.0);
    if (ln < NB) v = cmul(G[s.pt_xy[w] * NB + ln], tw[(ln * s.pt_z[w]) % F]);
    const double vx = wave_sum(v.x), vy = wave_sum(v.y);
    if (ln == 0) s.val[w] = sqrt(vx * vx + vy * vy);
  }
  __syncthreads();
}
// LDS: twiddles, then H and G of the points or of a whole plane
FO_HD size_t sel_points_lds(int nk) {
  const size_t NB = 2 * (size_t)nk + 1, xb = nk <= 15 ? kSelXs : 1;
  return sizeof(double2) * (xb * NB * NB + kSelPairs * NB);
}
FO_HD size_t sel_plane_lds(int nk, int F) {
  const size_t NB = 2 * (size_t)nk + 1;
  return sizeof(double2) * (NB * NB + NB * F);
}
constexpr size_t kSelLds = 64 * 1024;  // two workgroups a CU
static inline size_t per_select_smem(int nk, int F) {
  const size_t pt = sel_points_lds(nk), pl = sel_plane_lds(nk, F);
  return sizeof(double2) * F + std::max(pt, pl <= kSelLds ? pl : 0);
}

// FP64 |f| over a whole plane x; returns its argmax (ties -> lower flat index).
// H: [NB^2], G: [NB][F], in LDS when they fit (sel_plane_lds), else global; tw:
// the twiddles in LDS, phases advance by integer steps.  Every thread must
// call it.
FO_DEV void per_plane64(const PerGridCtx& c, int x, double2* H, double2* G, const double2* tw,
                        double* red, int* redi, double& bestv, int& besti) {
  const int NB = c.NB, F = c.F, plane = NB * NB;
  for (int e = threadIdx.x; e < plane; e += kSelThreads) {
    double2 acc = make_double2(0.0, 0.0);
    int ph = 0;
#pragma unroll 8
    for (int a = 0; a < NB; ++a) {
      acc = cadd(acc, cmul(c.C[(long long)a * plane + e], tw[ph]));
      ph += x;
      if (ph >= F) ph -= F;
    }
    H[e] = acc;
  }
  __threadfence_block();
  __syncthreads();
  for (int e = threadIdx.x; e < NB * F; e += kSelThreads) {
    const int b = e / F, z = e - b * F;
    double2 acc = make_double2(0.0, 0.0);
    int ph = 0;
#pragma unroll 4
    for (int cc = 0; cc < NB; ++cc) {
      acc = cadd(acc, cmul(H[b * NB + cc], tw[ph]));
      ph += z;
      if (ph >= F) ph -= F;
    }
    G[e] = acc;
  }
  __threadfence_block();
  __syncthreads();
  double bv = -INFINITY;
  int bi = 0x7fffffff;
  for (int e = threadIdx.x; e < F * F; e += kSelThreads) {
    const int y = e / F, z = e - y * F;
    double2 acc = make_double2(0.0, 0.0);
    int ph = 0;
#pragma unroll 4
    for (int b = 0; b < NB; ++b) {
      acc = cadd(acc, cmul(G[b * F + z], tw[ph]));
      ph += y;
      if (ph >= F) ph -= F;
    }
    argmax_merge(bv, bi, sqrt(acc.x * acc.x + acc.y * acc.y), (x * F + y) * F + z);
  }
  block_argmax(bv, bi, red, redi);
  bestv = bv;
  besti = bi;
  __syncthreads();
}

// Error bound of the FP32 planes: |f| <= A = sum |C|; rounding of C, of the
// twiddles and of three DFT passes of NB terms each stays below delta =
// rel_delta A (per_plane_delta).  Candidates within 2 delta of the FP32
// maximum are re-evaluated in FP64.
// The product is read once for the argmax and its six neighbours when a single
// candidate is listed (the common case); as seven separate sums over the cube
// and one for A, each a chain of loads, this took 61 us for one pair of nk = 8
// and 255 us for 24 of nk = 14, now 14 and 30.  The real planes list one value a
// wavefront and have twice the bound of the complex ones, so one or two of 128
// pairs of nk = 8, fewer at nk = 14, have a whole plane to evaluate, which the others
// wait for: 33 and 61 us then.  Bound: load latency of one workgroup per pair.
template <int XB>
__global__ void __launch_bounds__(kSelThreads) k_per_select(
    const PerPair* __restrict__ pd, int nk, int F, const double2* __restrict__ Cprod,
    const double2* __restrict__ tw64, const PlaneCand* __restrict__ cand,
    const double* __restrict__ abound, double rel_delta, double2* __restrict__ scratch,
    long long scratch_stride, PerPeak* __restrict__ peaks) {
  extern __shared__ __align__(16) unsigned char smem[];
  __shared__ SelPoints sp;
  __shared__ double red[16];
  __shared__ int redi[16];
  __shared__ float rv[16];
  __shared__ int ri[16];
  __shared__ int s_cnt, s_ovf;
  __shared__ int s_cand[kMaxCand];
  __shared__ int s_ovfl[512];
  const int p = blockIdx.x, t = threadIdx.x;
  const PerPair d = pd[p];
  const int NB = 2 * nk + 1;
  PerGridCtx c;
  c.NB = NB;
  c.F = F;
  c.C = Cprod + d.c_off;
  double2* tw = (double2*)smem;
  double2* H = tw + F;
  double2* G = H + XB * NB * NB;
  for (int q = t; q < F; q += kSelThreads) tw[q] = tw64[q];
  const PlaneCand* pc = cand + (long long)p * F;
  float mv = -INFINITY;
  int mi = 0x7fffffff;
  for (int b = t; b < F; b += blockDim.x)
    for (int r = 0; r < kCandPerPlane; ++r) argmax_merge(mv, mi, pc[b].val[r], pc[b].idx[r]);
  block_argmax(mv, mi, rv, ri);
  const double A = block_sum(t < NB ? abound[(long long)p * NB + t] : 0.0, red);
  const double delta = rel_delta * A;
  const double thr = (double)mv - 2.0 * delta;
  if (t == 0) {
    s_cnt = 0;
    s_ovf = 0;
  }
  __syncthreads();
  for (int b = t; b < F; b += blockDim.x) {
    float rest = pc[b].rest[0];
    for (int r = 1; r < kCandPerPlane; ++r) rest = fmaxf(rest, pc[b].rest[r]);
    if ((double)rest >= thr) {
      int q = atomicAdd(&s_ovf, 1);
      s_ovfl[q] = b;
    } else {
      for (int r = 0; r < kCandPerPlane; ++r)
        if ((double)pc[b].val[r] >= thr) {
          int q = atomicAdd(&s_cnt, 1);
          if (q < kMaxCand) s_cand[q] = pc[b].idx[r];
        }
    }
  }
  __syncthreads();
  const int ncand = min(s_cnt, kMaxCand), novf = s_ovf;
  const bool cand_overflow = s_cnt > kMaxCand;
  if (t == 0) {
    for (int i = 1; i < ncand; ++i) {
      int v = s_cand[i], j = i - 1;
      while (j >= 0 && s_cand[j] > v) {
        s_cand[j + 1] = s_cand[j];
        --j;
      }
      s_cand[j + 1] = v;
    }
    for (int i = 1; i < novf; ++i) {
      int v = s_ovfl[i], j = i - 1;
      while (j >= 0 && s_ovfl[j] > v) {
        s_ovfl[j + 1] = s_ovfl[j];
        --j;
      }
      s_ovfl[j + 1] = v;
    }
  }
  __syncthreads();
  double best = -INFINITY, second = -INFINITY;
  int besti = 0x7fffffff;
  double2* Hg = sel_plane_lds(nk, F) <= kSelLds ? H : scratch + (long long)p * scratch_stride;
  double2* Gg = Hg + NB * NB;
  auto take = [&](double v, int i) {
    if (v > best || (v == best && i < besti)) {
      second = best;
      best = v;
      besti = i;
    } else if (v > second) {
      second = v;
    }
  };
  const bool merged = !cand_overflow && novf == 0 && ncand == 1;
  if (merged) {
    besti = s_cand[0];
  } else if (cand_overflow) {
    for (int x = 0; x < F; ++x) {
      double v;
      int i;
      per_plane64(c, x, Hg, Gg, tw, red, redi, v, i);
      take(v, i);
    }
  } else {
    for (int q = 0; q < ncand; ++q) {
      const int f = s_cand[q];
      if (t == 0) {
        sp.np = sp.nxy = sp.nx = 1;
        sp.x[0] = f / (F * F);
        sp.xy_x[0] = 0;
        sp.xy_y[0] = (f / F) % F;
        sp.pt_xy[0] = 0;
        sp.pt_z[0] = f % F;
      }
      __syncthreads();
      per_eval64<XB>(c, sp, tw, H, G);
      take(sp.val[0], f);
      __syncthreads();
    }
    for (int q = 0; q < novf; ++q) {
      double v;
      int i;
      per_plane64(c, s_ovfl[q], Hg, Gg, tw, red, redi, v, i);
      take(v, i);
    }
  }
  const int ind[3] = {besti / (F * F), (besti / F) % F, besti % F};
  // the argmax and its neighbours: points 0, then (+1, -1) per axis
  if (t == 0) {
    // (no listed point, as for a product that is not a number: ind is out of
    // range and is folded back)
    const int x0 = ind[0] % F, y0 = ind[1] % F, z0 = ind[2] % F;
    const int xp = (ind[0] + 1) % F, xm = (ind[0] + F - 1) % F;
    const int yp = (ind[1] + 1) % F, ym = (ind[1] + F - 1) % F;
    const int zp = (ind[2] + 1) % F, zm = (ind[2] + F - 1) % F;
    sp.np = kSelPoints;
    sp.nxy = kSelPairs;
    sp.nx = kSelXs;
    sp.x[0] = x0;
    sp.x[1] = xp;
    sp.x[2] = xm;
    const int ys[kSelPairs] = {y0, y0, y0, yp, ym};
    const int xy[kSelPoints] = {0, 1, 2, 3, 4, 0, 0};
    const int zs[kSelPoints] = {z0, z0, z0, z0, z0, zp, zm};
    for (int q = 0; q < kSelPairs; ++q) {
      sp.xy_x[q] = q < 3 ? q : 0;
      sp.xy_y[q] = ys[q];
    }
    for (int q = 0; q < kSelPoints; ++q) {
      sp.pt_xy[q] = xy[q];
      sp.pt_z[q] = zs[q];
    }
  }
  __syncthreads();
  per_eval64<XB>(c, sp, tw, H, G);
  if (merged) best = sp.val[0];
  double off[3];
  for (int ax = 0; ax < 3; ++ax) {
    const double y1 = sp.val[1 + 2 * ax], y3 = sp.val[2 + 2 * ax];
    off[ax] = (y3 - y1) / (2.0 * (2.0 * best - y1 - y3));
  }
  if (t == 0) {
    PerPeak pk;
    for (int ax = 0; ax < 3; ++ax) {
      pk.ind[ax] = ind[ax];
      pk.disp[ax] = (ind[ax] - off[ax]) * d.box[ax] / F;
    }
    pk.ncand = cand_overflow ? -1 : ncand;
    pk.noverflow = cand_overflow ? F : novf;
    pk.pad = 0;
    pk.value = best;
    pk.margin = best - second;
    pk.delta = delta;
    peaks[p] = pk;
  }
}

// ---------------------------------------------------------------------------
// Refinement (fastoverlap/periodicAlignment.py:27-80) with the intended LAP
// semantics: Euclidean minimum-image cost with rows = X1, X2[perm] ~ X1.
// ---------------------------------------------------------------------------
FO_DEV double pwrap(double v, double box) { return v - rint(v / box) * box; }
// squared minimum-image length (ib = 1 / box)
FO_DEV double pdist2(double dx, double dy, double dz, const double box[3], const double ib[3]) {
  dx -= rint(dx * ib[0]) * box[0];
  dy -= rint(dy * ib[1]) * box[1];
  dz -= rint(dz * ib[2]) * box[2];
  return dx * dx + dy * dy + dz * dz;
}

// The nearest row of every column (structure 2's atoms, displaced by the
// peak) over its group, for the refinement's first assignment.  64 entries of
// the pair's group lists per workgroup, four lanes a column; the rows of the
// workgroup's groups pass through LDS in tiles.  In the refinement's single
// workgroup this scan of all size^2 distances took most of its time (one
// wavefront a SIMD, every distance waiting on gathered loads).  Both kernels
// together against that: one pair of 256 atoms 226 -> 29 us, 24 pairs of
// 601..1024 atoms 1826 -> 82 us (a search over cells of the box inside the
// refinement took 661: its short, divergent loops wait on LDS).  Bound: the
// FP64 vector rate, 20 operations a distance.
constexpr int kNearCols = 64;
constexpr int kNearTile = 256;
__global__ void __launch_bounds__(256) k_per_nearest(
    const PerPair* __restrict__ pd, const PerGroup* __restrict__ grp,
    const int* __restrict__ atoms, const double* __restrict__ pos1,
    const double* __restrict__ pos2, const PerPeak* __restrict__ peaks,
    NearRec* __restrict__ near) {
  __shared__ double rows[kNearTile][3];
  __shared__ int s_range[2];
  const int p = blockIdx.y, t = threadIdx.x;
  const PerPair d = pd[p];
  if (d.ngroups < 1) return;
  const PerGroup* G = grp + d.group_off;
  const int base = G[0].atom_list_off;  // the pair's list entries are contiguous
  const int total = G[d.ngroups - 1].atom_list_off + G[d.ngroups - 1].size - base;
  const int e0 = blockIdx.x * kNearCols;
  if (e0 >= total) return;  // whole workgroup
  const int e = e0 + (t >> 2), part = t & 3;
  // the last group that starts at or before entry e (empty groups before it
  // start there too)
  int q = 0, hi = d.ngroups;
  const int ec = min(e, total - 1);
  while (hi - q > 1) {
    const int mid = (q + hi) >> 1;
    if (G[mid].atom_list_off - base <= ec)
      q = mid;
    else
      hi = mid;
  }
  const int r0 = G[q].atom_list_off - base, r1 = r0 + G[q].size;
  if (t == 0) s_range[0] = r0;
  if (t == 255) s_range[1] = r1;
  const double* x = pos1 + 3LL * d.atom_off;
  const int* ga = atoms + base;
  const double box[3] = {d.box[0], d.box[1], d.box[2]};
  const double ib[3] = {1.0 / box[0], 1.0 / box[1], 1.0 / box[2]};
  const double* Y = pos2 + 3LL * (d.atom_off + ga[ec]);
  const double b0 = Y[0] - peaks[p].disp[0], b1 = Y[1] - peaks[p].disp[1],
               b2 = Y[2] - peaks[p].disp[2];
  auto root = [](double k) { return sqrt(k); };
  ColMin m;
  __syncthreads();
  const int lo = s_range[0], end = s_range[1];
  for (int k0 = lo; k0 < end; k0 += kNearTile) {
    __syncthreads();  // readers of the previous tile are done
    for (int w = t; w < 3 * min(kNearTile, end - k0); w += 256)
      rows[w / 3][w % 3] = x[3 * ga[k0 + w / 3] + w % 3];
    __syncthreads();
    const int i1 = min(r1, k0 + kNearTile) - k0;
    int i = max(r0, k0) - k0;
    // rows of this lane: the group's row index modulo 4 is its part
    i += (part - (i + k0 - r0)) & 3;
    auto key = [&](int r) {
      return pdist2(rows[r][0] - b0, rows[r][1] - b1, rows[r][2] - b2, box, ib);
    };
    for (; i + 12 < i1; i += 16) {
      const double c0 = key(i), c1 = key(i + 4), c2 = key(i + 8), c3 = key(i + 12);
      if (fmin(fmin(c0, c1), fmin(c2, c3)) < m.key2) {
        m.add(c0, i + k0 - r0 + 1, root);
        m.add(c1, i + k0 - r0 + 5, root);
        m.add(c2, i + k0 - r0 + 9, root);
        m.add(c3, i + k0 - r0 + 13, root);
      }
    }
    for (; i < i1; i += 4) m.add(key(i), i + k0 - r0 + 1, root);
  }
  m.join(4);
  if (part == 0 && e < total) {
    NearRec r;
    r.mn = m.mn;
    r.gap = sqrt(m.key2) - sqrt(m.key);  // +inf for one row; NaN: never used
    r.mi = m.mi;
    r.pad = 0;
    near[base + e] = r;
  }
}

// LDS of the refinement beside the assignment arrays: the positions of the
// largest group's rows and displaced columns, when they fit
static inline size_t refine_lds_bytes(int nmax, bool staged) {
  const size_t lap = (lap_lds_bytes(nmax) + 15) & ~(size_t)15;
  return staged ? lap + 6 * sizeof(double) * (size_t)nmax : lap;
}
constexpr size_t kRefineLds = 160 * 1024;

__global__ void __launch_bounds__(256) k_per_refine(
    const PerPair* __restrict__ pd, const PerGroup* __restrict__ grp,
    const int* __restrict__ atoms, const double* __restrict__ pos1,
    const double* __restrict__ pos2, const PerPeak* __restrict__ peaks,
    const NearRec* __restrict__ near, int niter, int lap_nmax, int staged,
    int* __restrict__ perm, int* __restrict__ saveperm, int* __restrict__ rowsol,
    double* __restrict__ X1out, double* __restrict__ X2out, PerResult* __restrict__ res) {
  extern __shared__ __align__(16) unsigned char smem[];
  __shared__ double red[16];
  __shared__ int redi[16];
  __shared__ int s_same;
  const int p = blockIdx.x, t = threadIdx.x;
  const PerPair d = pd[p];
  const int N = d.natoms;
  const double* x = pos1 + 3LL * d.atom_off;
  const double* y = pos2 + 3LL * d.atom_off;
  int* pm = perm + d.atom_off;
  int* sp = saveperm + d.atom_off;
  int* rs = rowsol + d.atom_off;
  const double bx = d.box[0], by = d.box[1], bz = d.box[2];
  double disp[3] = {peaks[p].disp[0], peaks[p].disp[1], peaks[p].disp[2]};
  LapShared ls = lap_carve(smem, lap_nmax);

  const double box[3] = {bx, by, bz}, ib[3] = {1.0 / bx, 1.0 / by, 1.0 / bz};
  // group positions in LDS: rows x, columns y - disp
  double* g1 = (double*)(smem + ((lap_lds_bytes(lap_nmax) + 15) & ~(size_t)15));
  double* g2 = g1 + 3 * lap_nmax;
  // Column minima: the first assignment takes k_per_nearest's.  A later one
  // differs by a displacement e, which moves no minimum-image distance by
  // more than |e|: a column whose second nearest row was more than 2 |e|
  // farther keeps its nearest row, and only that distance is formed again;
  // the others scan their rows.
  const double start[3] = {disp[0], disp[1], disp[2]};
  bool first = true;

  auto hungarian = [&](int* out) {
    for (int a = t; a < N; a += blockDim.x) out[a] = a;
    __threadfence_block();
    __syncthreads();
    auto root = [](double k) { return sqrt(k); };
    const double e0 = disp[0] - start[0], e1 = disp[1] - start[1], e2 = disp[2] - start[2];
    const double safe = 2.0 * (1.0 + 1e-9) * sqrt(e0 * e0 + e1 * e1 + e2 * e2) +
                        1e-12 * (bx + by + bz);
    for (int g = 0; g < d.ngroups; ++g) {
      const PerGroup G = grp[d.group_off + g];
      const int n = G.size;
      const int* ga = atoms + G.atom_list_off;
      const NearRec* nr = near + G.atom_list_off;
      auto solve = [&](auto key) {
        lap_solve(n, key, root,
                  [&](int j, ColMin& m) {
                    const NearRec r = nr[j];
                    m.mi = r.mi;
                    m.mn = r.mn;
                    if (first) return true;
                    if (!(r.mi > 0 && r.gap > safe)) return false;
                    m.mn = root(key(r.mi - 1, j));
                    return true;
                  },
                  ls, rs, red, redi);
      };
      if (staged) {
        for (int e = t; e < 3 * n; e += blockDim.x) {
          const int i = e / 3, k = e - 3 * i;
          g1[e] = x[3 * ga[i] + k];
          g2[e] = y[3 * ga[i] + k] - (k == 0 ? disp[0] : (k == 1 ? disp[1] : disp[2]));
        }
        __syncthreads();
        solve([&](int i, int j) {
          const double *A = g1 + 3 * i, *B = g2 + 3 * j;
          return pdist2(A[0] - B[0], A[1] - B[1], A[2] - B[2], box, ib);
        });
      } else {
        const double d0 = disp[0], d1 = disp[1], d2 = disp[2];
        solve([&](int i, int j) {
          const double *A = x + 3 * ga[i], *B = y + 3 * ga[j];
          return pdist2(A[0] - (B[0] - d0), A[1] - (B[1] - d1), A[2] - (B[2] - d2), box, ib);
        });
      }
      for (int i = t; i < n; i += blockDim.x) out[ga[i]] = ga[rs[i]];
      __threadfence_block();
      __syncthreads();
    }
    first = false;
  };
  auto mean_shift = [&](const int* pr) {
    double s[3] = {0, 0, 0};
    for (int a = t; a < N; a += blockDim.x) {
      const double* B = y + 3 * pr[a];
      s[0] += pwrap(x[3 * a] - (B[0] - disp[0]), bx);
      s[1] += pwrap(x[3 * a + 1] - (B[1] - disp[1]), by);
      s[2] += pwrap(x[3 * a + 2] - (B[2] - disp[2]), bz);
    }
    block_sum_n<3>(s, red);
    for (int k = 0; k < 3; ++k) disp[k] -= s[k] / (double)N;
  };

  hungarian(sp);
  int it = 0;
  for (; it < niter; ++it) {
    mean_shift(sp);
    hungarian(pm);
    if (t == 0) s_same = 1;
    __syncthreads();
    for (int a = t; a < N; a += blockDim.x)
      if (pm[a] != sp[a]) s_same = 0;
    __syncthreads();
    const bool same = s_same;
    __syncthreads();
    if (same) break;
    for (int a = t; a < N; a += blockDim.x) sp[a] = pm[a];
    __threadfence_block();
    __syncthreads();
  }
  if (niter == 0) {
    for (int a = t; a < N; a += blockDim.x) pm[a] = sp[a];
    __threadfence_block();
    __syncthreads();
  }
  mean_shift(pm);
  double* o1 = X1out + 3LL * d.atom_off;
  double* o2 = X2out + 3LL * d.atom_off;
  double ss = 0.0;
  for (int a = t; a < N; a += blockDim.x) {
    const double* B = y + 3 * pm[a];
    const double u0 = pwrap(x[3 * a], bx), u1 = pwrap(x[3 * a + 1], by), u2 = pwrap(x[3 * a + 2], bz);
    const double v0 = pwrap(B[0] - disp[0], bx), v1 = pwrap(B[1] - disp[1], by),
                 v2 = pwrap(B[2] - disp[2], bz);
    o1[3 * a] = u0;
    o1[3 * a + 1] = u1;
    o1[3 * a + 2] = u2;
    o2[3 * a] = v0;
    o2[3 * a + 1] = v1;
    o2[3 * a + 2] = v2;
    const double e0 = pwrap(u0 - v0, bx), e1 = pwrap(u1 - v1, by), e2 = pwrap(u2 - v2, bz);
    ss += e0 * e0 + e1 * e1 + e2 * e2;
  }
  ss = block_sum(ss, red);
  if (t == 0) {
    PerResult r;
    r.dist = sqrt(ss);
    r.disp[0] = disp[0];
    r.disp[1] = disp[1];
    r.disp[2] = disp[2];
    r.iters = it;
    r.status = 0;
    res[p] = r;
  }
}

}  // namespace fo

namespace fo {

static inline int pcdiv(long long a, long long b) { return (int)((a + b - 1) / b); }

// the larger of the phase tiles and the group sums S of both structures
size_t per_sf_smem(int nk) {
  const size_t NB = 2 * (size_t)nk + 1;
  return sizeof(double) * std::max(2 * (size_t)kSFTile * sf_stride((int)NB), 4 * NB * NB);
}

void launch_per_sf(hipStream_t s, int P, int nk, const PerPair* pd, const PerGroup* grp,
                   const int* atoms, const double* pos1, const double* pos2, double2* Cprod,
                   double2* C1out, double2* C2out) {
  const dim3 g(nk + 1, P), b(kSFThreads);
  const size_t sm = per_sf_smem(nk);
  const int ct = (2 * nk + 1 + 15) / 16;
#define FO_SF(CT)                                                                             \
  hipLaunchKernelGGL(k_per_sf<CT>, g, b, sm, s, pd, grp, atoms, pos1, pos2, nk, Cprod, C1out, \
                     C2out)
  if (ct == 1)
    FO_SF(1);
  else if (ct == 2)
    FO_SF(2);
  else if (ct == 3)
    FO_SF(3);
  else
    FO_SF(4);
#undef FO_SF
}

void launch_per_product(hipStream_t s, int P, int nk, const PerPair* pd, const double2* C1,
                        const double2* C2, double2* Cprod) {
  const long long cube = (long long)(2 * nk + 1) * (2 * nk + 1) * (2 * nk + 1);
  hipLaunchKernelGGL(k_per_product, dim3(std::min(pcdiv(cube, 256), 256), P), dim3(256), 0, s, pd,
                     nk, C1, C2, Cprod);
}

size_t per_plane_smem(int nk, int F) {
  const int NB = 2 * nk + 1;
  return sizeof(float2) * ((size_t)F + (size_t)NB * NB + (size_t)NB * F) + 16 * sizeof(float) +
         16 * sizeof(int);
}

// real: the product is Hermitian and f itself is not kept
double per_plane_delta(int nk, int real) {
  const int NB = 2 * nk + 1;
  return real ? real_plane_delta(NB) : (4.0 * NB + 32.0) * 5.9604644775390625e-08;
}

static size_t real_plane_smem(int nk, int F, int XP) {
  const size_t NB = 2 * (size_t)nk + 1;
  return sizeof(float2) * F +
         sizeof(float) * ((NB + 1) * real_plane_fs(F) + XP * NB * real_plane_ks((int)NB));
}

void launch_per_plane(hipStream_t s, int P, int nk, int F, int real, const PerPair* pd,
                      const double2* Cprod, const float2* tw32, PlaneCand* cand, double* abound,
                      float* grid, float2* cgrid) {
  if (!real) {
    hipLaunchKernelGGL(k_per_plane, dim3(F, P), dim3(256), per_plane_smem(nk, F), s, pd, nk, F,
                       Cprod, tw32, cand, abound, grid, cgrid);
    return;
  }
  // four planes a workgroup when there are planes enough to fill the chip
  // that way (the basis table is made once for them), else one
  const int XP = (long long)P * F >= 1024 * kPlaneXP &&
                         real_plane_smem(nk, F, kPlaneXP) <= 64 * 1024
                     ? kPlaneXP
                     : 1;
  const dim3 g((F + XP - 1) / XP, P), b(256);
  const size_t sm = real_plane_smem(nk, F, XP);
  const int nt = (2 * nk + 1 + 15) / 16;
#define FO_PLANE(NT)                                                                          \
  hipLaunchKernelGGL(k_per_plane_real<NT>, g, b, sm, s, pd, nk, F, XP, Cprod, tw32, cand, abound, \
                     grid)
  if (nt == 1)
    FO_PLANE(1);
  else if (nt == 2)
    FO_PLANE(2);
  else if (nt == 3)
    FO_PLANE(3);
  else
    FO_PLANE(4);
#undef FO_PLANE
}

void launch_per_product_indexed(hipStream_t s, int P, int nk, const PerPair* pd,
                                const double2* Cs, const int* idx1, const int* idx2,
                                double2* Cprod) {
  const long long cube = (long long)(2 * nk + 1) * (2 * nk + 1) * (2 * nk + 1);
  hipLaunchKernelGGL(k_per_product_indexed, dim3(std::min(pcdiv(cube, 256), 256), P), dim3(256),
                     0, s, pd, nk, Cs, idx1, idx2, Cprod);
}

void launch_per_select(hipStream_t s, int P, int nk, int F, const PerPair* pd,
                       const double2* Cprod, const double2* tw64, const PlaneCand* cand,
                       const double* abound, double rel_delta, double2* scratch,
                       long long scratch_stride, PerPeak* peaks) {
  // three x values a pass while their sums over a fit LDS (NB <= 31: 46 KB)
  const size_t sm = per_select_smem(nk, F);
  if (nk <= 15)
    hipLaunchKernelGGL(k_per_select<3>, dim3(P), dim3(kSelThreads), sm, s, pd, nk, F, Cprod, tw64,
                       cand, abound, rel_delta, scratch, scratch_stride, peaks);
  else
    hipLaunchKernelGGL(k_per_select<1>, dim3(P), dim3(kSelThreads), sm, s, pd, nk, F, Cprod, tw64,
                       cand, abound, rel_delta, scratch, scratch_stride, peaks);
}

void launch_per_refine(hipStream_t s, int P, int lap_nmax, const PerPair* pd, const PerGroup* grp,
                       const int* atoms, const double* pos1, const double* pos2,
                       const PerPeak* peaks, int niter, int maxgath, NearRec* near, int* perm,
                       int* saveperm, int* rowsol, double* X1out, double* X2out, PerResult* res) {
  if (maxgath > 0)
    hipLaunchKernelGGL(k_per_nearest, dim3(pcdiv(maxgath, kNearCols), P), dim3(256), 0, s, pd, grp,
                       atoms, pos1, pos2, peaks, near);
  // (the reduction scratch is static, beside the dynamic part)
  const bool staged = refine_lds_bytes(lap_nmax, true) + 1024 <= kRefineLds;
  hipLaunchKernelGGL(k_per_refine, dim3(P), dim3(256), refine_lds_bytes(lap_nmax, staged), s, pd,
                     grp, atoms, pos1, pos2, peaks, near, niter, lap_nmax, staged ? 1 : 0, perm,
                     saveperm, rowsol, X1out, X2out, res);
}

}  // namespace fo

// ---------------------------------------------------------------------------
// Stand-alone LAP of two point sets (Hungarian methods of the drop-in
// classes: fastoverlap/sphericalAlignment.py:102-108 with squared distances,
// fastoverlap/periodicAlignment.py:94-107 with minimum-image distances).
// ---------------------------------------------------------------------------
namespace fo {

__global__ void __launch_bounds__(256) k_lap_align(int N, const double* __restrict__ X1,
                                                   const double* __restrict__ X2, int ngroups,
                                                   const int* __restrict__ gsize,
                                                   const int* __restrict__ goff,
                                                   const int* __restrict__ gatoms, int metric,
                                                   double bx, double by, double bz, int lap_nmax,
                                                   int* __restrict__ perm,
                                                   int* __restrict__ rowsol,
                                                   double* __restrict__ dist) {
  extern __shared__ __align__(16) unsigned char smem[];
  __shared__ double red[16];
  __shared__ int redi[16];
  const int t = threadIdx.x;
  LapShared ls = lap_carve(smem, lap_nmax);
  for (int a = t; a < N; a += blockDim.x) perm[a] = a;
  __threadfence_block();
  __syncthreads();
  for (int g = 0; g < ngroups; ++g) {
    const int* ga = gatoms + goff[g];
    const double box[3] = {bx, by, bz}, ib[3] = {1.0 / bx, 1.0 / by, 1.0 / bz};
    auto key = [&](int i, int j) {
      const double* A = X1 + 3 * ga[i];
      const double* B = X2 + 3 * ga[j];
      const double dx = A[0] - B[0], dy = A[1] - B[1], dz = A[2] - B[2];
      return metric == 1 ? pdist2(dx, dy, dz, box, ib) : dx * dx + dy * dy + dz * dz;
    };
    lap_solve(gsize[g], key, [&](double k) { return metric == 1 ? sqrt(k) : k; },
              [](int, ColMin&) { return false; }, ls, rowsol, red, redi);
    for (int i = t; i < gsize[g]; i += blockDim.x) perm[ga[i]] = ga[rowsol[i]];
    __threadfence_block();
    __syncthreads();
  }
  double ss = 0.0;
  for (int a = t; a < N; a += blockDim.x) {
    const double* A = X1 + 3 * a;
    const double* B = X2 + 3 * perm[a];
    double dx = A[0] - B[0], dy = A[1] - B[1], dz = A[2] - B[2];
    if (metric == 1) {
      dx = pwrap(dx, bx);
      dy = pwrap(dy, by);
      dz = pwrap(dz, bz);
    }
    ss += dx * dx + dy * dy + dz * dz;
  }
  ss = block_sum(ss, red);
  if (t == 0) *dist = sqrt(ss);
}

void launch_lap_align(hipStream_t s, int N, const double* X1, const double* X2, int ngroups,
                      const int* gsize, const int* goff, const int* gatoms, int metric,
                      const double* box, int lap_nmax, int* perm, int* rowsol, double* dist) {
  hipLaunchKernelGGL(k_lap_align, dim3(1), dim3(256), lap_lds_bytes(lap_nmax), s, N, X1, X2,
                     ngroups, gsize, goff, gatoms, metric, box ? box[0] : 1.0, box ? box[1] : 1.0,
                     box ? box[2] : 1.0, lap_nmax, perm, rowsol, dist);
}

}  // namespace fo

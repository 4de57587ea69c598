// Contraction of the spherical coefficients on the FP64 matrix cores:
//   C^l_{m1m2} = 4 pi^{5/2} s^3 sum_groups sum_{j,k in group}
//                Y1[l,m1,j] K_l[j,k] conj(Y2[l,m2,k])
// (fastoverlap/sphericalAlignment.py:273, :175), rows m1 >= 0 only: the rows
// m1 < 0 follow from C_{-m1,-m2} = (-1)^{m1+m2} conj(C_{m1m2}).
#include "fo_common.h"
#include "fo_internal.h"
#include <algorithm>
#include <type_traits>

namespace fo {

// ---------------------------------------------------------------------------
// One wavefront per (pair, degrees, block of rows), no LDS and no barrier.  In
// the real basis (Re Y_l^m, Im Y_l^m, m = 0..l) of both structures
//   P[c][rho] = sum_k Yb2[c][k] (sum_j K_l[j][k] Yb1[rho][j])
// are 2l+2 by 2l+2 real sums which give C for both signs of m2:
//   C_{m1, m2}  = (Prr + Pii) + i (Pir - Pri),
//   C_{m1,-m2}  = (-1)^{m2} [(Prr - Pii) + i (Pir + Pri)]
// (first letter the part of m1, second that of m2): half the products of the
// complex form, and 16-row tiles that fill at every eighth degree.
// For KT tiles of 16 atoms k at a time:
//   1. A[k][rho] over all j, four a step: operand A = K_l (lane: k = lane%16,
//      j = lane/16, straight from the radial slots), B = Yb1;
//   2. register i of A, row k = 4 i + lane/16, is the B operand of the step
//      that takes those atoms of the tile, operand A = Yb2: P += Yb2 A.
// Two tiles of a pair (Re, Im of the same m; even and odd atoms k) come with
// one 16-byte load a lane.  A step's operands are loaded two steps ahead (the
// barriers keep the compiler from mixing steps, which makes it wait for all of
// them).  Each lane holds the four parts of its (m1, m2), or shares them with
// lane ^ 8 in the mixed tile, and stores whole entries.
//
// Degrees >= 16 read K_l from its radial slot, one degree a wavefront.
// Degrees 0..15 start from the stored pair K_h, K_{h+1} at the top of their
// block of eight and descend K_{l-1} = K_{l+1} + (2l+1)/x K_l (i_l is the
// minimal solution, stable downwards), D degrees a wavefront.  x below
// kMinRadX = 2^-58 (an atom at the centre) counts as 2^-58, here and where the
// slots are filled: K_0 is the same to FP64 and K_l, l >= 1, moves by less than
// 2^-59 K_0.  With x = 2^-58 the degrees 8..15 are below x^8 / 17!! = 2^-489 of K_0,
// so it does not matter that K_15 and K_16 may vanish for two atoms whose distances
// differ by several widths; K_0..K_7 come from the slots 7 and 8, normal numbers
// until the Gaussian, and K_0 with it, is below 2^-530.
//
// Pairs with more than kSplitAtoms grouped atoms take four wavefronts per
// item, the k tiles dealt to them in equal shares and their P added through
// LDS in a fixed order.  Every output's reduction order depends on the pair
// alone.  Where the line lies: 4096 pairs of 13..147 atoms take 1.99 ms with
// one wavefront, 2.39 with four from 100 atoms on and 2.59 from 48 on (idle
// wavefronts hold registers), one pair of 160 atoms 75 us with one and 32 with
// four.
//
// All degrees share a launch: with one launch per class one pair of 100 atoms
// took 110 us instead of 44 (each class waits for its slowest item) and the 4096
// pairs 2.06 ms instead of 1.99, although the joint kernel spills 247 registers
// (262 with four wavefronts), outside its product loops.
//
// Bound: reading K and Y.  1000 atoms, degree 40: 26.0 GB past the L2 for 64 pairs
// (a slot once for every item of its degrees), 5 TB/s; of the 5.1 ms the products
// take 2.2 at the matrix rate (matrix units 55 % busy).  Items with all row tiles of
// a degree read a slot 40 times instead of 63 but leave one wavefront a SIMD: 6.3
// ms.  4096 pairs of 13..147 atoms, degrees 16..25: products 0.62 of 1.99 ms (34 %
// busy, with the padding), waits on loads (two wavefronts a SIMD) most of the rest.
// Against the two kernels it replaces (a workgroup per degree with A through LDS, the
// complex form, and for degrees <= 15 a fused one): 3.31 -> 1.99 ms and 9.62 -> 5.2
// ms; 16 pairs of 300..500 atoms 1006 -> 189 us, one pair of 500 at degree 30 988 ->
// 159 us.
// ---------------------------------------------------------------------------
constexpr int kSplitAtoms = 160;
constexpr double kMaxInvX = 1.0 / kMinRadX;

struct ContractArgs {
  const SphPair* pd;
  const SphGroup* grp;
  const double *rad1, *rad2;
  const double2 *Y1, *Y2;
  const double *R, *scale_eff;
  double2* I64;
  float2* I32;
  int n, P, items;
};

// Row tiles of a degree: T / 2 pairs, (re, im) of m = 16 pair + r, and for odd
// T one mixed tile, r < 8: re, r >= 8: im of m = 8 (T - 1) + r % 8.  A pair's
// operands are one 16-byte load a lane.  Offsets (bytes) of the T tiles from
// even tile t0 on at atom go + lane/16 of degree l's harmonics, one per pair and
// one for the mixed tile (m beyond l repeat the last).  Descriptors and offsets
// (unsigned) cover the degrees lb..l of one item, not the pair's whole block, which
// passes 2^31 bytes at 156000 grouped atoms of degree 40 (contract_in_reach).
FO_HD constexpr int row_units(int T) { return (T + 1) / 2; }
FO_DEV __amdgpu_buffer_rsrc_t degree_rsrc(const double2* Y, int lb, int l, int Ng) {
  const unsigned rows = qlm(l, l) + 1 - qlm(lb, 0);
  return buf_rsrc(Y + (long long)qlm(lb, 0) * Ng, (int)(rows * Ng * 16u));
}
template <int T>
FO_DEV void row_offsets(unsigned (&off)[row_units(T)], int lb, int l, int t0, int Ng) {
  const int col = threadIdx.x & 15, q = (threadIdx.x >> 4) & 3;
#pragma unroll
  for (int u = 0; u < row_units(T); ++u) {
    const bool mixed = 2 * u + 1 == T;
    const int m = 8 * (t0 + 2 * u) + (mixed ? col & 7 : col);
    off[u] = ((unsigned)(qlm(l, min(m, l)) - qlm(lb, 0)) * Ng + q) * 16u +
             (mixed ? (col >> 3) * 8 : 0);
  }
}
// the T operands of those tiles, shifted by `add` bytes
template <int T>
FO_DEV void row_load(double (&v)[T], __amdgpu_buffer_rsrc_t r,
                     const unsigned (&off)[row_units(T)], unsigned add) {
#pragma unroll
  for (int u = 0; u < T / 2; ++u) {
    const double2 x = load_d2(r, (int)(off[u] + add), 0);
    v[2 * u] = x.x;
    v[2 * u + 1] = x.y;
  }
  if constexpr (T & 1) v[T - 1] = load_d(r, (int)(off[T / 2] + add), 0);
}
// Tiles of atoms k: CNT / 2 pairs, tile 2 p + e holding the atoms 32 p + 2 r +
// e of the block, and for odd CNT one tile of 16 consecutive ones; again one
// load a pair (vk: byte offset of the block's first atom + 0, see kcol).
FO_DEV int kcol(int CNT, int kt, int r) {  // atom of row r of tile kt
  return kt < (CNT & ~1) ? 32 * (kt >> 1) + 2 * r + (kt & 1) : 16 * kt + r;
}
template <int CNT>
FO_DEV void col_load(double (&v)[CNT], __amdgpu_buffer_rsrc_t r, int off) {
  const int col = threadIdx.x & 15;
#pragma unroll
  for (int u = 0; u < CNT / 2; ++u) {
    const double2 x = load_d2(r, off + 16 * col + 256 * u, 0);
    v[2 * u] = x.x;
    v[2 * u + 1] = x.y;
  }
  if constexpr (CNT & 1) v[CNT - 1] = load_d(r, off + 8 * col + 128 * (CNT - 1), 0);
}

FO_DEV void store_c(const ContractArgs& a, const SphPair& d, int l, int m1, int m2, double x,
                    double y, double norm) {
  const double2 v = make_double2(norm * x, norm * y);
  a.I64[d.coef_off + kidx(l, m1, m2)] = v;
  a.I32[d.c32_off + (long long)qlm(l, m1) * a.n + plane_pos(plane_k(m2, a.n), a.n)] =
      make_float2((float)v.x, (float)v.y);
}
// The four sums of (m1, m2), first letter the part of m1 -> C of +m2 and / or
// -m2 (lanes beyond the degree store nothing).
FO_DEV void store_entry(const ContractArgs& a, const SphPair& d, int l, int m1, int m2, double rr,
                        double ii, double ir, double ri, bool plus, bool minus, double norm) {
  if (m1 > l || m2 > l) return;
  if (plus) store_c(a, d, l, m1, m2, rr + ii, ir - ri, norm);
  if (minus && m2 > 0) {
    const double s = (m2 & 1) ? -norm : norm;
    store_c(a, d, l, m1, -m2, rr - ii, ir + ri, s);
  }
}
// Register i (for a mixed column tile: i and i + 2, i < 2) of the tiles of one
// (column unit, row unit): v[2 e + f], e / f the column / row tile of a pair
// (0 for a mixed one); vi: the registers i + 2 of a mixed column tile.
FO_DEV void store_unit(const ContractArgs& a, const SphPair& d, int l, int mc, int mr, bool cmix,
                       bool rmix, int i, const double (&v)[4], const double (&vi)[2],
                       double norm) {
  const int col = threadIdx.x & 15, q = (threadIdx.x >> 4) & 3;
  const int m2 = mc + 4 * i + q;
  // values of this lane's m1 part(s): [row tile] re, im of m2
  const double r0 = v[0], i0 = cmix ? vi[0] : v[2];
  if (!rmix) {
    const double r1 = v[1], i1 = cmix ? vi[1] : v[3];
    store_entry(a, d, l, mr + col, m2, r0, i1, r1, i0, true, true, norm);
  } else {
    const double ro = __shfl_xor(r0, 8, 64), io = __shfl_xor(i0, 8, 64);
    const bool im1 = col >= 8;
    store_entry(a, d, l, mr + (col & 7), m2, im1 ? ro : r0, im1 ? i0 : io, im1 ? r0 : ro,
                im1 ? io : i0, !im1, im1, norm);
  }
}

// All tiles of one degree; WV > 1: the wavefronts' sums are added first (red:
// WV * 4 * 256 doubles of LDS).
template <int CT, int RT, int WV>
FO_DEV void store_degree(const ContractArgs& a, const SphPair& d, int l, int rt0,
                         const v4d (&P)[CT][RT], double norm, double* red) {
  const int ln = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
#pragma unroll
  for (int cu = 0; cu < row_units(CT); ++cu)
#pragma unroll
    for (int ru = 0; ru < row_units(RT); ++ru) {
      const bool cmix = 2 * cu + 1 == CT, rmix = 2 * ru + 1 == RT;
      const int mc = 16 * cu, mr = 8 * (rt0 + 2 * ru);
      const int nc = cmix ? 1 : 2, nr = rmix ? 1 : 2;
      if constexpr (WV == 1) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          if (cmix && i >= 2) continue;
          double v[4] = {0, 0, 0, 0}, vi[2] = {0, 0};
#pragma unroll
          for (int e = 0; e < 2; ++e)
#pragma unroll
            for (int f = 0; f < 2; ++f)
              if (e < nc && f < nr) {
                v[2 * e + f] = P[2 * cu + e][2 * ru + f][i];
                if (cmix) vi[f] = P[2 * cu][2 * ru + f][(i + 2) & 3];
              }
          store_unit(a, d, l, mc, mr, cmix, rmix, i, v, vi, norm);
        }
      } else {
        static_assert(WV == 4, "wavefront i stores register i");
        __syncthreads();  // readers of the previous unit are done
#pragma unroll
        for (int e = 0; e < 2; ++e)
#pragma unroll
          for (int f = 0; f < 2; ++f)
            if (e < nc && f < nr)
#pragma unroll
              for (int i = 0; i < 4; ++i)
                red[((wv * 4 + 2 * e + f) * 4 + i) * 64 + ln] = P[2 * cu + e][2 * ru + f][i];
        __syncthreads();
        if (!cmix || wv < 2) {  // uniform
          auto sum = [&](int tile, int i) {
            double x = red[(tile * 4 + i) * 64 + ln];
#pragma unroll
            for (int w = 1; w < WV; ++w) x += red[((w * 4 + tile) * 4 + i) * 64 + ln];
            return x;
          };
          double v[4] = {0, 0, 0, 0}, vi[2] = {0, 0};
#pragma unroll
          for (int e = 0; e < 2; ++e)
#pragma unroll
            for (int f = 0; f < 2; ++f)
              if (e < nc && f < nr) {
                v[2 * e + f] = sum(2 * e + f, wv);
                if (cmix) vi[f] = sum(f, wv + 2);
              }
          store_unit(a, d, l, mc, mr, cmix, rmix, wv, v, vi, norm);
        }
      }
    }
}

// P += Yb2 A of D degrees and CNT tiles from atom k0 of the group (go: its
// first atom) on (o2: row offsets of Yb2), U steps of four rows of A at a time
// with the next ones' operands loading meanwhile.
template <int D, int CT, int RT, int CNT>
FO_DEV void second_product(v4d (&P)[D][CT][RT], const v4d (&A)[D][CNT][RT],
                           __amdgpu_buffer_rsrc_t ry2, const unsigned (&o2)[D][row_units(CT)],
                           int k0, int go, int Ns) {
  constexpr int U = CT <= 2 ? 4 : (CT <= 4 ? 2 : 1), NU = 4 / U, NG = D * CNT * NU;
  const int q = (threadIdx.x >> 4) & 3;
  double y[2][U][CT];
  // atom of this lane's row 4 i + q of tile kt; its offset beyond o2 (which
  // already holds q atoms)
  auto atom = [&](int kt, int i) { return k0 + kcol(CNT, kt, 4 * i + q); };
  auto load = [&](int g, double(&v)[U][CT]) {
    const int kt = (g / NU) % CNT;
#pragma unroll
    for (int u = 0; u < U; ++u)
      row_load<CT>(v[u], ry2, o2[g / (NU * CNT)],
                   (unsigned)(go + atom(kt, U * (g % NU) + u) - q) * 16u);
  };
  load(0, y[0]);
#pragma unroll
  for (int g = 0; g < NG; ++g) {
    if (g + 1 < NG) load(g + 1, y[(g + 1) & 1]);
    __builtin_amdgcn_sched_barrier(0);  // the loads stay ahead of the products
    const int dd = g / (NU * CNT), kt = (g / NU) % CNT;
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int i = U * (g % NU) + u;
      const bool ok = atom(kt, i) < Ns;  // A holds other entries beyond
#pragma unroll
      for (int c = 0; c < CT; ++c) {
        const double v = ok ? y[g & 1][u][c] : 0.0;
#pragma unroll
        for (int r = 0; r < RT; ++r) P[dd][c][r] = mfma64(v, A[dd][kt][r][i], P[dd][c][r]);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
  }
}

// The k tiles [t0, t1) in blocks of at most KT, sizes as equal as can be:
// f(integral_constant<count>, first tile).
template <int KT, class F>
FO_DEV void tile_blocks(int t0, int t1, F&& f) {
  const int m = t1 - t0;
  if (m <= 0) return;
  const int nb = (m + KT - 1) / KT;
  for (int b = 0; b < nb; ++b) {
    const int a = t0 + m * b / nb, cnt = t0 + m * (b + 1) / nb - a;
    if (cnt == KT)
      f(std::integral_constant<int, KT>{}, a);
    else if (KT > 1 && cnt == KT - 1)
      f(std::integral_constant<int, (KT > 1 ? KT - 1 : 1)>{}, a);
    else if (KT > 2 && cnt == KT - 2)
      f(std::integral_constant<int, (KT > 2 ? KT - 2 : 1)>{}, a);
    else if (KT > 3 && cnt == KT - 3)
      f(std::integral_constant<int, (KT > 3 ? KT - 3 : 1)>{}, a);
  }
}

// Degree l >= 16, row tiles rt0 .. rt0 + RT - 1 of CT = ceil((2l+2)/16).
template <int RT, int CT, int KT, int WV>
FO_DEV void contract_high(const ContractArgs& a, const SphPair& d, int l, int rt0, double norm,
                          double* red) {
  static_assert(KT <= 4, "tile_blocks");
  const int q = (threadIdx.x >> 4) & 3;
  const int wv = WV > 1 ? __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) : 0;
  const int Ng = d.ngath;
  const __amdgpu_buffer_rsrc_t ry1 = degree_rsrc(a.Y1 + d.ylm_off, l, l, Ng);
  const __amdgpu_buffer_rsrc_t ry2 = degree_rsrc(a.Y2 + d.ylm_off, l, l, Ng);
  unsigned oy[row_units(RT)], o2[1][row_units(CT)];
  row_offsets<RT>(oy, l, l, rt0, Ng);
  row_offsets<CT>(o2[0], l, l, 0, Ng);
  v4d P[1][CT][RT];
#pragma unroll
  for (int c = 0; c < CT; ++c)
#pragma unroll
    for (int r = 0; r < RT; ++r) P[0][c][r] = v4d{0.0, 0.0, 0.0, 0.0};
  for (int g = 0; g < d.ngroups; ++g) {
    const SphGroup G = a.grp[d.group_off + g];
    const int Ns = G.size, go = G.gath_off, n4 = (Ns + 3) >> 2, nt = (Ns + 15) >> 4;
    // degree l in radial slot l - 13; reads past its end (j >= Ns) are zero
    const __amdgpu_buffer_rsrc_t rk =
        buf_rsrc(a.R + d.rad_off + G.rad_off + (long long)(l - 13) * Ns * Ns, Ns * Ns * 8);
    tile_blocks<KT>(nt * wv / WV, nt * (wv + 1) / WV, [&](auto CN, int tile) {
      constexpr int CNT = decltype(CN)::value;
      v4d A[1][CNT][RT];
#pragma unroll
      for (int kt = 0; kt < CNT; ++kt)
#pragma unroll
        for (int r = 0; r < RT; ++r) A[0][kt][r] = v4d{0.0, 0.0, 0.0, 0.0};
      const int vk = (q * Ns + 16 * tile) * 8;
      double ka[CNT], kb[CNT], ya[RT], yb[RT];
      auto load = [&](double(&k)[CNT], double(&y)[RT], int s) {
        col_load<CNT>(k, rk, vk + s * (32 * Ns));
        row_load<RT>(y, ry1, oy, go * 16u + s * 64u);
        __builtin_amdgcn_sched_barrier(0);  // step by step, so that waits count
      };
      auto mul = [&](const double(&k)[CNT], const double(&y)[RT]) {
#pragma unroll
        for (int kt = 0; kt < CNT; ++kt)
#pragma unroll
          for (int r = 0; r < RT; ++r) A[0][kt][r] = mfma64(k[kt], y[r], A[0][kt][r]);
      };
      load(ka, ya, 0);
      load(kb, yb, 1);
      for (int s = 0; s < n4; s += 2) {  // an odd last step multiplies zeros
        mul(ka, ya);
        load(ka, ya, s + 2);
        mul(kb, yb);
        load(kb, yb, s + 3);
      }
      second_product(P, A, ry2, o2, 16 * tile, go, Ns);
    });
  }
  store_degree<CT, RT, WV>(a, d, l, rt0, P[0], norm, red);
}

// Degrees h - PRE, h - PRE - 1, .. (D of them, those below 8 BLK are not
// stored) of block BLK (0: degrees 0..7, 1: 8..15), h the block's top degree.
template <int BLK, int PRE, int D, int KT, int WV>
FO_DEV void contract_low_tiles(const ContractArgs& a, const SphPair& d, int h, double sc,
                               const SphGroup& G, v4d (&P)[D][BLK + 1][BLK + 1]) {
  constexpr int RT = BLK + 1;  // 2l+2 <= 16 RT
  const int ln = threadIdx.x & 63, col = ln & 15, q = ln >> 4;
  const int wv = WV > 1 ? __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) : 0;
  const int Ng = d.ngath, Ns = G.size, go = G.gath_off, n4 = (Ns + 3) >> 2, nt = (Ns + 15) >> 4;
  const int lt = h - PRE, lb = max(lt - (D - 1), 0);  // the item's degrees
  const __amdgpu_buffer_rsrc_t ry1 = degree_rsrc(a.Y1 + d.ylm_off, lb, lt, Ng);
  const __amdgpu_buffer_rsrc_t ry2 = degree_rsrc(a.Y2 + d.ylm_off, lb, lt, Ng);
  const double c0 = 2.0 * h + 1.0;
  const long long ss = (long long)Ns * Ns;
  const double* K = a.R + d.rad_off + G.rad_off;
  const __amdgpu_buffer_rsrc_t rk0 = buf_rsrc(K + 2 * BLK * ss, (int)(ss * 8));
  const __amdgpu_buffer_rsrc_t rk1 = buf_rsrc(K + (2 * BLK + 1) * ss, (int)(ss * 8));
  const __amdgpu_buffer_rsrc_t rr1 = buf_rsrc(a.rad1 + d.gath_off + go, Ns * 8);
  unsigned oy[D][row_units(RT)];
#pragma unroll
  for (int dd = 0; dd < D; ++dd) row_offsets<RT>(oy[dd], lb, max(lt - dd, 0), 0, Ng);
  tile_blocks<KT>(nt * wv / WV, nt * (wv + 1) / WV, [&](auto CN, int tile) {
    constexpr int CNT = decltype(CN)::value;
    v4d A[D][CNT][RT];
#pragma unroll
    for (int dd = 0; dd < D; ++dd)
#pragma unroll
      for (int kt = 0; kt < CNT; ++kt)
#pragma unroll
        for (int r = 0; r < RT; ++r) A[dd][kt][r] = v4d{0.0, 0.0, 0.0, 0.0};
    // 1/x = (1/r1) (2 s^2 / r2), at most kMaxInvX (columns beyond the group
    // hold other rows' finite values, which the second product leaves out)
    double ir2[CNT];
#pragma unroll
    for (int kt = 0; kt < CNT; ++kt)
      ir2[kt] = 2.0 * sc * sc / a.rad2[d.gath_off + go + min(16 * tile + kcol(CNT, kt, col), Ns - 1)];
    const int vk = (q * Ns + 16 * tile) * 8;
    struct Step {
      double k0[CNT], k1[CNT], y[D][RT], r;
    } sa, sb;
    auto load = [&](Step& t, int s) {
      col_load<CNT>(t.k0, rk0, vk + s * (32 * Ns));
      col_load<CNT>(t.k1, rk1, vk + s * (32 * Ns));
      t.r = load_d(rr1, (4 * s + q) * 8, 0);
#pragma unroll
      for (int dd = 0; dd < D; ++dd) row_load<RT>(t.y[dd], ry1, oy[dd], go * 16u + s * 64u);
      __builtin_amdgcn_sched_barrier(0);  // step by step, so that waits count
    };
    auto mul = [&](Step& t) {
      const double irj = 1.0 / t.r;  // entries j >= Ns hold zeros
      double cx[CNT];
#pragma unroll
      for (int kt = 0; kt < CNT; ++kt) cx[kt] = fmin(irj * ir2[kt], kMaxInvX);
      auto down = [&](double cl) {
#pragma unroll
        for (int kt = 0; kt < CNT; ++kt) {
          const double nx = t.k1[kt] + cl * cx[kt] * t.k0[kt];
          t.k1[kt] = t.k0[kt];
          t.k0[kt] = nx;
        }
      };
#pragma unroll
      for (int u = 0; u < PRE; ++u) down(c0 - 2.0 * u);  // degrees of other wavefronts
#pragma unroll
      for (int dd = 0; dd < D; ++dd) {
#pragma unroll
        for (int kt = 0; kt < CNT; ++kt)
#pragma unroll
          for (int r = 0; r < RT; ++r) A[dd][kt][r] = mfma64(t.k0[kt], t.y[dd][r], A[dd][kt][r]);
        if (dd + 1 < D) down(c0 - 2.0 * (PRE + dd));
      }
    };
    load(sa, 0);
    load(sb, 1);
    for (int s = 0; s < n4; s += 2) {
      mul(sa);
      load(sa, s + 2);
      mul(sb);
      load(sb, s + 3);
    }
    second_product(P, A, ry2, oy, 16 * tile, go, Ns);  // the same rows
  });
}

template <int BLK, int PRE, int D, int KT, int WV>
FO_DEV void contract_low(const ContractArgs& a, const SphPair& d, double sc, double norm,
                         double* red) {
  const int h = min(8 * BLK + 7, d.L), top = h - PRE;
  if (top < 8 * BLK) return;  // uniform
  constexpr int RT = BLK + 1;
  static_assert(KT <= 4, "tile_blocks");
  v4d P[D][RT][RT];
#pragma unroll
  for (int dd = 0; dd < D; ++dd)
#pragma unroll
    for (int c = 0; c < RT; ++c)
#pragma unroll
      for (int r = 0; r < RT; ++r) P[dd][c][r] = v4d{0.0, 0.0, 0.0, 0.0};
  for (int g = 0; g < d.ngroups; ++g) {
    const SphGroup G = a.grp[d.group_off + g];
    contract_low_tiles<BLK, PRE, D, KT, WV>(a, d, h, sc, G, P);
  }
#pragma unroll
  for (int dd = 0; dd < D; ++dd)
    if (top - dd >= 8 * BLK)  // uniform
      store_degree<RT, RT, WV>(a, d, top - dd, 0, P[dd], norm, red);
}

// Items of a pair: degrees 0..7 in two items of four, 8..15 in four of two,
// then every degree >= 16 in blocks of row tiles, class T = ceil((2l+2)/16).
// Blocks and KT keep P, A and two steps of operands in 256 registers (two
// wavefronts a SIMD).
FO_HD constexpr int high_parts(int T) { return T == 3 ? 1 : (T == 4 ? 2 : (T <= 6 ? 3 : 4)); }
// One item: CLS 0 and 1 the low blocks, 3..7 the degrees of class T = CLS.
template <int CLS, int WV>
FO_DEV void contract_item(const ContractArgs& a, const SphPair& d, int it, double sc, double norm,
                          double* red) {
  if constexpr (CLS == 0) {
    if (it == 0) contract_low<0, 0, 4, 3, WV>(a, d, sc, norm, red);
    if (it == 1) contract_low<0, 4, 4, 3, WV>(a, d, sc, norm, red);
  } else if constexpr (CLS == 1) {
    if (it == 0) contract_low<1, 0, 2, 3, WV>(a, d, sc, norm, red);
    if (it == 1) contract_low<1, 2, 2, 3, WV>(a, d, sc, norm, red);
    if (it == 2) contract_low<1, 4, 2, 3, WV>(a, d, sc, norm, red);
    if (it == 3) contract_low<1, 6, 2, 3, WV>(a, d, sc, norm, red);
  } else {
    constexpr int np = high_parts(CLS);
    const int l = 8 * (CLS - 1) + it / np, part = it % np;
    if (l > d.L) return;
    if constexpr (CLS == 3) contract_high<3, 3, 3, WV>(a, d, l, 0, norm, red);
    if constexpr (CLS == 4) contract_high<2, 4, 4, WV>(a, d, l, 2 * part, norm, red);
    if constexpr (CLS == 5) {
      if (part < 2)
        contract_high<2, 5, 3, WV>(a, d, l, 2 * part, norm, red);
      else
        contract_high<1, 5, 4, WV>(a, d, l, 4, norm, red);
    }
    if constexpr (CLS == 6) contract_high<2, 6, 2, WV>(a, d, l, 2 * part, norm, red);
    if constexpr (CLS == 7) {
      if (part < 3)
        contract_high<2, 7, 1, WV>(a, d, l, 2 * part, norm, red);
      else
        contract_high<1, 7, 3, WV>(a, d, l, 6, norm, red);
    }
  }
}

// Items of a pair, the long ones first: classes T = 7 .. 3, then the low
// blocks.  Batches with a degree above 49 are refused (their beta planes do not
// fit LDS), so class 8 does not occur.
static inline int contract_items(int Lmax) {
  int n = 6;
  for (int l = 16; l <= Lmax; ++l) n += high_parts((l >> 3) + 1);
  return n;
}

template <int WV>
__global__ void __launch_bounds__(64 * WV, 2) k_sph_contract(const ContractArgs a) {
  __shared__ double red[WV > 1 ? WV * 4 * 256 : 1];
  int pp, it;
  if (!xcd_decode(a.P, a.items, pp, it)) return;
  const SphPair d = a.pd[pp];
  if ((d.ngath > kSplitAtoms) != (WV > 1)) return;  // the other launch's pair
  it = a.items - 1 - it;
  const double sc = a.scale_eff[pp];
  const double norm = 4.0 * pow(kPi, 2.5) * sc * sc * sc;
  if (it < 2) return contract_item<0, WV>(a, d, it, sc, norm, red);
  if (it < 6) return contract_item<1, WV>(a, d, it - 2, sc, norm, red);
  it -= 6;
  int T = 3;
  while (it >= 8 * high_parts(T)) it -= 8 * high_parts(T++);
  switch (T) {
    case 3: return contract_item<3, WV>(a, d, it, sc, norm, red);
    case 4: return contract_item<4, WV>(a, d, it, sc, norm, red);
    case 5: return contract_item<5, WV>(a, d, it, sc, norm, red);
    case 6: return contract_item<6, WV>(a, d, it, sc, norm, red);
    default: return contract_item<7, WV>(a, d, it, sc, norm, red);
  }
}

void launch_sph_contract(hipStream_t s, int P, int n, int Lmax, int mingath, int maxgath,
                         const SphPair* pd, const SphGroup* grp, const double* rad1,
                         const double* rad2, const double2* Y1, const double2* Y2,
                         const double* R, const double* scale_eff, double2* I64, float2* I32) {
  const ContractArgs a{pd, grp, rad1, rad2, Y1, Y2, R, scale_eff, I64, I32,
                       n,  P,   contract_items(Lmax)};
  const dim3 g(xcd_grid(P, a.items));
  if (mingath <= kSplitAtoms)
    hipLaunchKernelGGL(k_sph_contract<1>, g, dim3(64), 0, s, a);
  if (maxgath > kSplitAtoms)
    hipLaunchKernelGGL(k_sph_contract<4>, g, dim3(256), 0, s, a);
}

}  // namespace fo

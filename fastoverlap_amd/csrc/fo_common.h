// Shared device/host helpers for the fastoverlap MI355X (gfx950) kernels.
//
// Conventions (fixed by the reference's Python classes):
//  * C^l_{m1 m2} is stored "compact l-major": for l = 0..L, m1 = -l..l,
//    m2 = -l..l, at index kidx(l,m1,m2) = l(4l^2-1)/3 + (m1+l)(2l+1) + (m2+l).
//    The layout does not depend on L, so any prefix K(L) of a table built for
//    Lt >= L serves degree L.  (reference: the (l, m1, m2) enumeration order of
//    fastoverlap/sphericalAlignment.py:52-55 and fastoverlap/soft.py:57-59)
//  * SO(3) grid axes are (alpha, beta, gamma) = (axis 0, 1, 2) of an n^3 grid,
//    flat index (ia*n + ib)*n + ig (fastoverlap/soft.py:119-125).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#define FO_DEV __device__ __forceinline__
#define FO_HD __host__ __device__ __forceinline__

namespace fo {

constexpr double kPi = 3.141592653589793238462643383279502884;

FO_HD long long kcount(int L) {  // number of (l,m1,m2) with l <= L
  return (long long)(L + 1) * (2 * L + 1) * (2 * L + 3) / 3;
}
FO_HD long long kbase(int l) {  // first compact index of degree l
  return (long long)l * (2 * l - 1) * (2 * l + 1) / 3;
}
FO_HD long long kidx(int l, int m1, int m2) {
  return kbase(l) + (long long)(m1 + l) * (2 * l + 1) + (m2 + l);
}

// triangular index of (l, m), 0 <= m <= l
FO_HD int qlm(int l, int m) { return l * (l + 1) / 2 + m; }

// ---- stored radial slots ---------------------------------------------------
// The radial kernel stores, per (j, k) of a species group, the values of a
// few degrees ("slots", [slot][j][k]).  Degrees 0..15 are contracted in
// blocks of eight (0..7, 8..15), each from the two stored degrees at its top
// by the downward recurrence; degrees >= 16 one per slot.  Slot degrees, in
// increasing order:
//   L <= 7 :  L, L+1                    (block 0 = 0..L)
//   L <= 15:  7, 8, L, L+1              (block 1 = 8..L)
//   L >= 16:  7, 8, 15, 16, 17, ..., L  (degree l >= 16 in slot l - 13)
// Block b reads slots 2b (its top degree) and 2b + 1 (one above).  x =
// r1 r2 / 2 s^2 below kMinRadX counts as kMinRadX.
constexpr double kMinRadX = 0x1p-58;
FO_HD int rad_slots(int L) { return L <= 7 ? 2 : (L <= 15 ? 4 : L - 12); }
FO_HD int rad_slot_deg(int s, int L) {
  if (L <= 7) return L + s;
  if (s < 2) return 7 + s;
  return L <= 15 ? L + s - 2 : s + 13;
}

// ---- plane layout (FP32 operands of the iSOFT plane kernels) --------------
// Rows (l, m1) with 0 <= m1 <= l at row l(l+1)/2 + m1 (l-major, so the rows
// of degrees <= L are a prefix), n entries per row indexed by the gamma
// transform input k (m2 = k for k < n/2, k - n above) and zero where |m2| > l.
// Inside a row, entry k sits at plane_pos(k, n): lane-major for the grid
// sides of the two-pass transform (n = N1*N2, lane k1 owns k = k1 + N1*k2 and
// its N2 entries are contiguous); for other even n the entries m2 and -m2 side
// by side (2 m2 and 2 m2 + 1; m2 = 0 beside the unused k = n/2); in k order for
// odd n.
FO_HD int plane_n1(int n) {  // N1 of the two-pass transform, 0 if none
  switch (n) {
    case 16: return 4;
    case 32: case 64: return 8;
    case 128: case 256: return 16;
    default: return 0;
  }
}
FO_HD long long plane_rows(int L) { return (long long)(L + 1) * (L + 2) / 2; }
FO_HD int plane_k(int m2, int n) { return m2 < 0 ? m2 + n : m2; }
FO_HD int plane_pos(int k, int n) {
  const int n1 = plane_n1(n);
  if (n1) return (k % n1) * (n / n1) + k / n1;
  if (n & 1) return k;
  return k < n / 2 ? 2 * k : k == n / 2 ? 1 : 2 * (n - k) + 1;
}

// ---- complex helpers (double2 / float2 = re, im) -------------------------
FO_HD double2 cmul(double2 a, double2 b) {
  return make_double2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}
FO_HD float2 cmul(float2 a, float2 b) {
  return make_float2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}
FO_HD double2 cconj(double2 a) { return make_double2(a.x, -a.y); }
FO_HD float2 cconj(float2 a) { return make_float2(a.x, -a.y); }
FO_HD double2 cadd(double2 a, double2 b) { return make_double2(a.x + b.x, a.y + b.y); }
FO_HD float2 cadd(float2 a, float2 b) { return make_float2(a.x + b.x, a.y + b.y); }
FO_HD double2 cscale(double2 a, double s) { return make_double2(a.x * s, a.y * s); }
FO_HD float2 cscale(float2 a, float s) { return make_float2(a.x * s, a.y * s); }

// integer power by squaring (exponent >= 0); valid for negative bases
FO_HD double ipow(double x, int e) {
  double r = 1.0;
  while (e > 0) {
    if (e & 1) r *= x;
    x *= x;
    e >>= 1;
  }
  return r;
}

// ---- wave / block reductions (wave64) -------------------------------------
template <typename T>
FO_DEV T wave_sum(T v) {
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  return v;
}
template <typename T>
FO_DEV T wave_max(T v) {
  for (int off = 32; off > 0; off >>= 1) {
    T o = __shfl_xor(v, off, 64);
    v = o > v ? o : v;
  }
  return v;
}

// Deterministic block sum (fixed tree independent of launch size).
// `scratch` must hold blockDim.x/64 elements.  All threads receive the sum.
template <typename T>
FO_DEV T block_sum(T v, T* scratch) {
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  const int nw = (blockDim.x + 63) >> 6;
  v = wave_sum(v);
  __syncthreads();
  if (lane == 0) scratch[wid] = v;
  __syncthreads();
  T r = 0;
  for (int w = 0; w < nw; ++w) r += scratch[w];
  return r;
}

// Deterministic block sum of NV values at once (two barriers).  `scratch`
// must hold NV * blockDim.x/64 elements.  All threads receive the sums.
template <int NV, typename T>
FO_DEV void block_sum_n(T (&v)[NV], T* scratch) {
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  const int nw = (blockDim.x + 63) >> 6;
#pragma unroll
  for (int k = 0; k < NV; ++k) v[k] = wave_sum(v[k]);
  __syncthreads();
  if (lane == 0)
#pragma unroll
    for (int k = 0; k < NV; ++k) scratch[wid * NV + k] = v[k];
  __syncthreads();
#pragma unroll
  for (int k = 0; k < NV; ++k) {
    T r = 0;
    for (int w = 0; w < nw; ++w) r += scratch[w * NV + k];
    v[k] = r;
  }
}

// Block argmax on (value, index): larger value wins, ties -> smaller index.
FO_DEV void argmax_merge(float& v, int& i, float ov, int oi) {
  if (ov > v || (ov == v && oi < i)) {
    v = ov;
    i = oi;
  }
}
FO_DEV void argmax_merge(double& v, int& i, double ov, int oi) {
  if (ov > v || (ov == v && oi < i)) {
    v = ov;
    i = oi;
  }
}
template <typename T>
FO_DEV void wave_argmax(T& v, int& i) {
  for (int off = 32; off > 0; off >>= 1) {
    T ov = __shfl_xor(v, off, 64);
    int oi = __shfl_xor(i, off, 64);
    argmax_merge(v, i, ov, oi);
  }
}
// scratch: two arrays of blockDim.x/64 entries.  All threads get the result.
template <typename T>
FO_DEV void block_argmax(T& v, int& i, T* sv, int* si) {
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  const int nw = (blockDim.x + 63) >> 6;
  wave_argmax(v, i);
  __syncthreads();
  if (lane == 0) {
    sv[wid] = v;
    si[wid] = i;
  }
  __syncthreads();
  v = sv[0];
  i = si[0];
  for (int w = 1; w < nw; ++w) argmax_merge(v, i, sv[w], si[w]);
}

// Argmin with ties -> smaller index.
FO_DEV void argmin_merge(double& v, int& i, double ov, int oi) {
  if (ov < v || (ov == v && oi < i)) {
    v = ov;
    i = oi;
  }
}

// DPP row shifts (within rows of 16 lanes): row_shl:S gives lane i the value
// of lane i + S, row_shr:S that of lane i - S.
template <int CTRL>
FO_DEV float dpp_mov(float x) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), CTRL, 0xf, 0xf, true));
}

// Records (largest value v, its flat index i, largest of the other values
// s): larger value first, ties to the smaller index; the loser's largest
// value joins the others (so s counts a repeated maximum).
FO_DEV void top2_merge(float& v, int& i, float& s, float ov, int oi, float os) {
  const bool take = ov > v || (ov == v && oi < i);
  s = fmaxf(fmaxf(s, os), take ? v : ov);
  v = take ? ov : v;
  i = take ? oi : i;
}
// One butterfly of NO (v, i, s) records over a wavefront: inside each row of
// 16 lanes by DPP (quad_perm [1,0,3,2], quad_perm [2,3,0,1], row_half_mirror,
// row_mirror), the records interleaved, then the four row results through
// readlane.  Every lane must be active and gets the wavefront's records.
template <int CTRL, int NO>
FO_DEV void top2_dpp_step(float (&v)[NO], int (&i)[NO], float (&s)[NO]) {
  float ov[NO], os[NO];
  int oi[NO];
#pragma unroll
  for (int o = 0; o < NO; ++o) {
    ov[o] = dpp_mov<CTRL>(v[o]);
    oi[o] = __builtin_amdgcn_update_dpp(0, i[o], CTRL, 0xf, 0xf, true);
    os[o] = dpp_mov<CTRL>(s[o]);
  }
#pragma unroll
  for (int o = 0; o < NO; ++o) top2_merge(v[o], i[o], s[o], ov[o], oi[o], os[o]);
}
template <int NO>
FO_DEV void wave_top2(float (&v)[NO], int (&i)[NO], float (&s)[NO]) {
  top2_dpp_step<0xB1>(v, i, s);
  top2_dpp_step<0x4E>(v, i, s);
  top2_dpp_step<0x141>(v, i, s);
  top2_dpp_step<0x140>(v, i, s);
#pragma unroll
  for (int o = 0; o < NO; ++o) {
    float rv = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v[o]), 0));
    float rs = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(s[o]), 0));
    int ri = __builtin_amdgcn_readlane(i[o], 0);
#pragma unroll
    for (int r = 16; r < 64; r += 16)
      top2_merge(rv, ri, rs, __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v[o]), r)),
                 __builtin_amdgcn_readlane(i[o], r),
                 __int_as_float(__builtin_amdgcn_readlane(__float_as_int(s[o]), r)));
    v[o] = rv;
    i[o] = ri;
    s[o] = rs;
  }
}

// XCD-aware decode of a 1-D launch of 8 ceil(P/8) per workgroups over
// (pair, item): workgroup w serves pair (w % 8) + 8 (w / (8 per)) and item
// (w / 8) % per.  Workgroups are dealt to the 8 XCDs round-robin, so all
// items of a pair run on one XCD and share its L2.  False for the padding
// workgroups (pair >= P).
FO_DEV bool xcd_decode(int P, int per, int& p, int& item) {
  const int w = blockIdx.x;
  p = (w & 7) + 8 * (w / (8 * per));
  item = (w >> 3) % per;
  return p < P;
}
static inline unsigned xcd_grid(int P, int per) { return (unsigned)(8 * ((P + 7) / 8) * per); }

// Raw buffer access (gfx9 descriptor): a per-lane byte offset plus a
// wavefront-uniform one (scalar register); offsets at or beyond `bytes`
// read zero.
FO_DEV __amdgpu_buffer_rsrc_t buf_rsrc(const void* base, int bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), (short)0, bytes, 0x00020000);
}
FO_DEV float4 load_f4(__amdgpu_buffer_rsrc_t r, int voff, int soff) {
  typedef unsigned int u4 __attribute__((ext_vector_type(4)));
  const u4 w = __builtin_amdgcn_raw_buffer_load_b128(r, voff, soff, 0);
  return make_float4(__uint_as_float(w.x), __uint_as_float(w.y), __uint_as_float(w.z),
                     __uint_as_float(w.w));
}

FO_DEV double load_d(__amdgpu_buffer_rsrc_t r, int voff, int soff) {
  typedef unsigned int u2 __attribute__((ext_vector_type(2)));
  const u2 w = __builtin_amdgcn_raw_buffer_load_b64(r, voff, soff, 0);
  return __hiloint2double((int)w.y, (int)w.x);
}
FO_DEV double2 load_d2(__amdgpu_buffer_rsrc_t r, int voff, int soff) {
  typedef unsigned int u4 __attribute__((ext_vector_type(4)));
  const u4 w = __builtin_amdgcn_raw_buffer_load_b128(r, voff, soff, 0);
  return make_double2(__hiloint2double((int)w.y, (int)w.x), __hiloint2double((int)w.w, (int)w.z));
}

// FP64 matrix product step.  Lane layout: A operand lane -> (row lane%16, k
// lane/16), B operand lane -> (k lane/16, col lane%16), result register i of
// a lane -> (row 4 i + lane/16, col lane%16).
typedef float v4f __attribute__((ext_vector_type(4)));
typedef double v4d __attribute__((ext_vector_type(4)));
FO_DEV v4d mfma64(double a, double b, v4d c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

}  // namespace fo

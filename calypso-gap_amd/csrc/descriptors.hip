// wACSF descriptors on the GPU: one wavefront (one 64-thread workgroup) per
// centre atom, in FP64 or FP32.
//
// Forward (CAR2ACSF's xx, gappy/libgap/wacsf.f90:65-796): for every symmetry
// function line s the plain feature x[s] and the weighted one x[s + nsf]:
//   radial  (types 1, 3): sum_j exp(-a (r_ij - rs)^2) fc(r_ij)          (* w_j)
//   angular (types 2, 4): sum_{j<k} pref (1 + lam cos)^zeta
//                         exp(-eta (r_ij^2 + r_ik^2 + r_jk^2)) fc fc fc  (* w_j w_k)
// with fc(r) = (cos(pi r / rc) + 1) / 2, pi = 3.141592654, a term counted
// only when every distance is <= the line's cutoff, (a, rs) = (alpha, 0) for
// type 1 and (4, Rs) for type 3, lam = +1 (type 2) / -1 (type 4), and
// pref = 2^(1 - zeta) (= 1 at zeta = 1, the reference's only case).
//
// Backward (replaces the dense dxdy/strs of wacsf.f90 and the force and
// stress loops of gap_calc.f90:172-203): with g = dE/dx of the centre atom,
// every term depends on the positions only through the distances r_ij, r_ik,
// r_jk, so the kernel accumulates T = sum_s g_eff,s d(term_s)/d(distance)
// (g_eff = g_s + w g_{s+nsf}) and turns each T into force vectors along the
// distance and the virial T d d^T / r.  Nothing of size D x neighbours is
// stored.
//
// Work layout: the atom's neighbours live in LDS (positions relative to the
// centre, distance, weight, cutoff function per cutoff group).  Radial sums
// put one neighbour on each lane.  Angular sums read the atom's triplet list,
// built once per evaluation by k_build<true> (neighbour pairs j < k with all
// three distances within the largest angular cutoff, compacted with a
// ballot), 64 triplets per step, so every lane holds a live triplet and
// forward and backward share one enumeration.  The forward keeps NCH lines'
// partial sums in registers per lane and reduces them across the wavefront
// after each chunk of lines.  Lines are sorted by (cutoff group, eta, lambda,
// zeta), so exponentials, cutoff products and the powers (1 + lambda cos)^zeta
// are updated incrementally along a chunk (zeta = 2, 4, 16 by squaring).
#include <atomic>
#include <cmath>
#include <mutex>
#include <set>
#include <utility>

#include "gapx_internal.h"

namespace gapx {

namespace {

// FP64 elementary functions of the descriptor kernels, written for the
// arguments these kernels have (no infinities, no range reduction beyond what
// the formulas need), from minimax polynomials fitted with a Remez exchange.
// (67,647 atoms, D = 128: the FP64 forward 1262 -> 1134 us.)
// The library's exp costs about 30 vector instructions with its range checks,
// its sincos about 70 (and much code for large arguments), its square root and
// division about 17 and 11 with their scaling; these cost 18, 22, 11 and 5.
//
// The coefficients are kept in scalar registers (sconst): as plain literals
// each would be moved into a vector register again for its fused multiply-add,
// about ten more vector instructions per exponential.
__device__ __forceinline__ double sconst(double c) {
  asm("" : "+s"(c));
  return c;
}

// exp(y): y = n ln2 + r, |r| <= ln2 / 2, 1 + r + r^2 q(r) with q of degree 9
// (fit error 3.4e-18), scaled by 2^n.  Underflows to 0 and overflows to
// infinity through the scaling.  y must be within about 1e40: past 2^53 the
// remainder r grows with y's spacing, and its powers would overflow.  (The host
// keeps coefficients within 1e20, centres and a caller's distances within 1e9 A.)
__device__ __forceinline__ double exp64(double y) {
  const double n = __builtin_rint(y * sconst(1.4426950408889634));
  double r = fma(n, sconst(-6.93147180559945286e-01), y);
  r = fma(n, sconst(-2.31904681384629956e-17), r);
  double q = sconst(2.5117915126746086e-08);
  q = fma(q, r, sconst(2.76313397049011e-07));
  q = fma(q, r, sconst(2.755721613139287e-06));
  q = fma(q, r, sconst(2.480148978582598e-05));
  q = fma(q, r, sconst(0.00019841269917571867));
  q = fma(q, r, sconst(0.0013888888947156122));
  q = fma(q, r, sconst(0.008333333333307118));
  q = fma(q, r, sconst(0.04166666666651493));
  q = fma(q, r, sconst(0.166666666666667));
  q = fma(q, r, sconst(0.5000000000000013));
  q = fma(q, r, 1.0);
  q = fma(q, r, 1.0);
  return __builtin_amdgcn_ldexp(q, (int)n);
}

// The same with the constants held by the caller, for a loop that a single wave
// runs on its SIMD: formed per call they are 23 scalar moves, which that wave
// pays for in full.  (Elsewhere the moves hide behind other waves, and all of
// them ahead of the polynomial cost 1 % of an FP64 evaluation.)
struct ExpConst {
  double log2e, ln2_hi, ln2_lo, q[10];
  __device__ __forceinline__ ExpConst()
      : log2e(sconst(1.4426950408889634)), ln2_hi(sconst(-6.93147180559945286e-01)),
        ln2_lo(sconst(-2.31904681384629956e-17)),
        q{sconst(2.5117915126746086e-08), sconst(2.76313397049011e-07), sconst(2.755721613139287e-06),
          sconst(2.480148978582598e-05), sconst(0.00019841269917571867), sconst(0.0013888888947156122),
          sconst(0.008333333333307118), sconst(0.04166666666651493), sconst(0.166666666666667),
          sconst(0.5000000000000013)} {}
};
__device__ __forceinline__ double exp64(double y, const ExpConst &c) {
  const double n = __builtin_rint(y * c.log2e);
  double r = fma(n, c.ln2_hi, y);
  r = fma(n, c.ln2_lo, r);
  double q = c.q[0];
#pragma unroll
  for (int k = 1; k < 10; ++k) q = fma(q, r, c.q[k]);
  q = fma(q, r, 1.0);
  q = fma(q, r, 1.0);
  return __builtin_amdgcn_ldexp(q, (int)n);
}

// Cosine and sine of x = w r in [0, pi] (up to 1e-4 beyond), as -sin and cos
// of y = x - pi/2: odd and even polynomials in y (fit errors 2e-19, 6e-18).
__device__ __forceinline__ double quarter_shift(double w, double r) {
  return fma(w, r, sconst(-1.57079632679489656)) + sconst(-6.12323399573676604e-17);
}
__device__ __forceinline__ double sin_quarter(double y, double z) {
  double s = sconst(2.7184781158758493e-15);
  s = fma(s, z, sconst(-7.642711170741734e-13));
  s = fma(s, z, sconst(1.6058927767606374e-10));
  s = fma(s, z, sconst(-2.5052106605227996e-08));
  s = fma(s, z, sconst(2.7557319207770882e-06));
  s = fma(s, z, sconst(-0.00019841269841185862));
  s = fma(s, z, sconst(0.008333333333333113));
  s = fma(s, z, sconst(-0.16666666666666666));
  return fma(y * z, s, y);
}
__device__ __forceinline__ double cos_quarter(double z) {
  double c = sconst(4.616102920731384e-14);
  c = fma(c, z, sconst(-1.1463632624429262e-11));
  c = fma(c, z, sconst(2.0876592494655193e-09));
  c = fma(c, z, sconst(-2.7557317066796995e-07));
  c = fma(c, z, sconst(2.4801587285768175e-05));
  c = fma(c, z, sconst(-0.0013888888888829978));
  c = fma(c, z, sconst(0.04166666666666583));
  return fma(z * z, c, fma(-0.5, z, 1.0));
}

// 1 / x from the hardware estimate and two Newton steps.
__device__ __forceinline__ double rcp64(double x) {
  double v = __builtin_amdgcn_rcp(x);
  v = fma(v, fma(-x, v, 1.0), v);
  return fma(v, fma(-x, v, 1.0), v);
}

template <typename T>
struct Math;

// sqrt_rsq: e = sqrt(x) and i = 1 / e for x >= floor2().  cos1: 1 + cos(w r)
// for w r in [0, pi]; sincos1 also the sine, with w from turn().
template <>
struct Math<double> {
  static __device__ __forceinline__ double ex(double x) { return exp64(x); }
  static constexpr __device__ __forceinline__ double floor2() { return 1e-200; }
  static __device__ __forceinline__ double turn(double pirc) { return pirc; }
  static __device__ __forceinline__ void sqrt_rsq(double x, double &e, double &i) {
    const double y = __builtin_amdgcn_rsq(x);
    double g = x * y, h = 0.5 * y;
    double d = fma(-h, g, 0.5);
    g = fma(g, d, g);
    h = fma(h, d, h);
    e = fma(fma(-g, g, x), h, g);
    h = fma(h, fma(-h, e, 0.5), h);
    i = h + h;
  }
  static __device__ __forceinline__ double sq(double x) {
    double e, i;
    sqrt_rsq(fmax(x, floor2()), e, i);
    return e;
  }
  static __device__ __forceinline__ double cos1(double w, double r) {
    const double y = quarter_shift(w, r);
    return 1.0 - sin_quarter(y, y * y);
  }
  static __device__ __forceinline__ void sincos1(double w, double r, double &s, double &c1) {
    const double y = quarter_shift(w, r), z = y * y;
    s = cos_quarter(z);
    c1 = 1.0 - sin_quarter(y, z);
  }
  static __device__ __forceinline__ double pw(double b, double e) { return pow(b, e); }
};

template <>
struct Math<float> {
  static __device__ __forceinline__ float ex(float x) { return __expf(x); }
  static constexpr __device__ __forceinline__ float floor2() { return 1e-30f; }
  // v_sin_f32 and v_cos_f32 take revolutions
  static __device__ __forceinline__ float turn(float pirc) { return pirc * 0.159154943091895f; }
  static __device__ __forceinline__ void sqrt_rsq(float x, float &e, float &i) {
    i = __builtin_amdgcn_rsqf(x);
    e = x * i;
  }
  static __device__ __forceinline__ float sq(float x) { return __builtin_amdgcn_sqrtf(x); }
  static __device__ __forceinline__ float cos1(float w, float r) { return __cosf(w * r) + 1.f; }
  static __device__ __forceinline__ void sincos1(float w, float r, float &s, float &c1) {
    const float x = w * r;
    s = __builtin_amdgcn_sinf(x);
    c1 = __builtin_amdgcn_cosf(x) + 1.f;
  }
  static __device__ __forceinline__ float pw(float b, float e) { return powf(b, e); }
};

// Two values of T read as one LDS access (the backward's per-neighbour pairs).
template <typename T>
struct Pair;
template <>
struct Pair<float> {
  typedef float2 type;
};
template <>
struct Pair<double> {
  typedef double2 type;
};

template <typename T>
struct alignas(16) Quad {
  T v[4];
};

// A radial-table entry in the kernel's precision: the FP32 copy for FP32
// kernels (the same rounding as converting the FP64 entry, without a
// conversion per line and lane).
template <typename T>
__device__ __forceinline__ T rad_table(const double *t64, const float *t32, int s) {
  if constexpr (sizeof(T) == 4)
    return t32[s];
  else
    return t64[s];
}

// This wave's index in its workgroup, known uniform to the compiler: tables
// indexed by it are then read with scalar loads.
__device__ __forceinline__ int wave_index() { return __builtin_amdgcn_readfirstlane(threadIdx.x >> 6); }

template <typename T>
__device__ __forceinline__ T wave_sum(T v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}

// Powers (1 + lam cos)^zeta along lines sorted by (lam, zeta) within an eta
// group.  pw = base^z and pm = base^(z-1) for the current z; a new lambda or
// a smaller zeta restarts at z = 1; larger integer zetas are reached by
// squaring (z -> 2z) or one more factor (z -> z+1), decisions that are the
// same on every lane.
template <typename T>
struct PowState {
  T lam = T(0), base = T(0), pw = T(0), pm = T(1);
  int z = 0;
  __device__ __forceinline__ void at(T new_lam, int zi, T cth) {
    if (new_lam != lam || zi < z || z == 0) {
      lam = new_lam;
      base = T(1) + lam * cth;
      pw = base;
      pm = T(1);
      z = 1;
    }
    while (z < zi) {
      if (2 * z <= zi) {
        pm = pw * pm;
        pw = pw * pw;
        z *= 2;
      } else {
        pm = pw;
        pw = pw * base;
        z += 1;
      }
    }
  }
};

// P = pref base^zeta and dP/dcos = pref zeta lam base^(zeta-1) of line s.
template <typename T>
__device__ __forceinline__ void line_power(const SFDev &sf, int s, T cth, PowState<T> &ps, T &P, T &dP) {
  const int zi = sf.ang_zeta[s];
  const T lam = (T)sf.ang_lam[s];
  if (zi == 1) {
    ps.at(lam, 1, cth);
    P = ps.pw;
    dP = lam;
  } else if (zi > 1) {
    ps.at(lam, zi, cth);
    const T pref = (T)sf.ang_pref[s];
    P = pref * ps.pw;
    dP = pref * (T)zi * lam * ps.pm;
  } else {  // non-integer zeta
    const T base = T(1) + lam * cth, zr = (T)sf.ang_zeta_real[s], pref = (T)sf.ang_pref[s];
    const T b1 = (base > T(0)) ? Math<T>::pw(base, zr - T(1)) : T(0);
    P = pref * b1 * base;
    dP = pref * zr * lam * b1;
  }
}

// A feature's FP16 contraction operand: xt clamped to [-2^15, 2^15], so the
// hi part is finite and the lo part exact.  The host keeps every scaled
// sparse-point component within 2^14 on this path, so a clamped component
// still differs from each of them by more than 2^14: the kernel value is
// exp(-d2 / 2) with d2 > 2^28 whether the norm of the clamped or of the true
// row enters d2, i.e. 0 in FP32 and in FP64 alike.
__device__ __forceinline__ double fp16_operand(double xt) { return fmin(fmax(xt, -32768.0), 32768.0); }

__device__ __forceinline__ void split16(int mode, double xt, uint16_t &h, uint16_t &l) {
  if (mode == 1) {  // FP16 hi + lo of xt clamped to the FP16 range (see fp16_operand)
    const double xc = fp16_operand(xt);
    const _Float16 hi = (_Float16)xc, lo = (_Float16)(xc - (double)hi);
    h = __builtin_bit_cast(uint16_t, hi);
    l = __builtin_bit_cast(uint16_t, lo);
  } else {  // BF16 hi + lo
    const __bf16 hi = (__bf16)(float)xt, lo = (__bf16)(float)(xt - (double)(float)hi);
    h = __builtin_bit_cast(uint16_t, hi);
    l = __builtin_bit_cast(uint16_t, lo);
  }
}

// A row's outputs from its features in LDS, two features per thread (Dp is a
// multiple of 32, the rows are aligned): raw features, centred and scaled ones,
// the split operands; returns this thread's part of |xt|^2 in FP64.
template <typename T, int W>
__device__ __forceinline__ double write_features(const T *s_feat, size_t row, int Dp, int tid, const double *theta_inv,
                                                 const double *mu, int split_mode, const DescOut &out) {
  double xn = 0.0;
  for (int d = 2 * tid; d < Dp; d += 128 * W) {
    const T x0 = s_feat[d], x1 = s_feat[d + 1];
    const double2 ti = *(const double2 *)(theta_inv + d), m = *(const double2 *)(mu + d);
    const double t0 = (double)x0 * ti.x - m.x, t1 = (double)x1 * ti.y - m.y;
    xn += t0 * t0;
    xn += t1 * t1;
    if (out.x64) *(double2 *)(out.x64 + row + d) = make_double2((double)x0, (double)x1);
    if (out.x32) *(float2 *)(out.x32 + row + d) = make_float2((float)x0, (float)x1);
    if (out.xt64) *(double2 *)(out.xt64 + row + d) = make_double2(t0, t1);
    if (out.xt32) *(float2 *)(out.xt32 + row + d) = make_float2((float)t0, (float)t1);
    if (split_mode) {
      ushort2 h, l;
      split16(split_mode, t0, h.x, l.x);
      split16(split_mode, t1, h.y, l.y);
      *(ushort2 *)(out.xt_hi + row + d) = h;
      *(ushort2 *)(out.xt_lo + row + d) = l;
    }
  }
  return xn;
}

// Weight of a neighbour slot: the caller's (CAR2ACSF's neighbour table), or
// that of the neighbour's species.
__device__ __forceinline__ double slot_weight(const NeighborBufs &nb, const double *wz, const int *species,
                                              size_t slot) {
  return nb.nb_w ? nb.nb_w[slot] : wz[species[nb.nb_j[slot]]];
}

// Launch geometry of the descriptor kernels: LDS layout (neighbour slots,
// cutoff groups, padded features, radial lines) and the first atom of the
// launch (one workgroup per atom from atom0 on).
struct Lds {
  int KP, G, Dp;
  int atom0;
  int n_rad;
};

// Stage an atom's K neighbours in LDS: d = (dx, dy, dz, r), rw = (1 / r,
// weight) and per cutoff group g, at row g KP, the cutoff function fc(r), or
// with DERIV the pairs (fc, dfc/dr).  Threads tid, tid + nthr, ..
template <typename T, bool DERIV>
__device__ __forceinline__ void stage_neighbours(const NeighborBufs &nb, const double *wz, const int *species,
                                                 const SFDev &sf, int start, int K, int KP, T *s_d, T *s_rw, T *s_fc,
                                                 int tid, int nthr) {
  for (int a = tid; a < K; a += nthr) {
    const double2 *dd = (const double2 *)(nb.nb_d + 4 * (size_t)(start + a));
    const double2 xy = dd[0], zr = dd[1];
    const double r = zr.y;
    s_d[4 * a] = (T)xy.x;
    s_d[4 * a + 1] = (T)xy.y;
    s_d[4 * a + 2] = (T)zr.x;
    s_d[4 * a + 3] = (T)r;
    s_rw[2 * a] = (T)rcp64(r);
    s_rw[2 * a + 1] = (T)slot_weight(nb, wz, species, start + a);
    for (int g = 0; g < sf.n_groups; ++g) {
      const bool in = r <= sf.group_rc[g];
      const double w = sf.group_pirc[g];
      if constexpr (DERIV) {
        double sn, c1;
        Math<double>::sincos1(w, r, sn, c1);
        s_fc[2 * (g * KP + a)] = in ? (T)(0.5 * c1) : T(0);
        s_fc[2 * (g * KP + a) + 1] = in ? (T)(-0.5 * sn * w) : T(0);
      } else {
        s_fc[g * KP + a] = in ? (T)(0.5 * Math<double>::cos1(w, r)) : T(0);
      }
    }
  }
}

// An atom's triplet list; an entry q is the pair (q & mask, q >> shift).
struct TripletList {
  const void *list;
  int narrow;            // 16-bit entries
  uint32_t mask, shift;
  __device__ __forceinline__ TripletList(const TripletBufs &tb, int i)
      : list(tb.narrow ? (const void *)((const uint16_t *)tb.list + (size_t)i * tb.tcap)
                       : (const void *)((const uint32_t *)tb.list + (size_t)i * tb.tcap)),
        narrow(tb.narrow), mask(tb.narrow ? 0xffu : 0xffffu), shift(tb.narrow ? 8u : 16u) {}
};

// Triplet indices of wave steps t, t + stride, .. (4 steps) for one lane; the
// loads are issued together, one iteration ahead of their use, so a wave
// waits for global memory once per four steps at most.  Inactive entries
// point at neighbours 0 and 1 (valid whenever the list is not empty).
__device__ __forceinline__ void load_q4(const TripletList &tl, int nt, int t, int stride, uint32_t (&q)[4]) {
  if (tl.narrow) {
    const uint16_t *p = (const uint16_t *)tl.list;
#pragma unroll
    for (int u = 0; u < 4; ++u) q[u] = (t + u * stride < nt) ? p[t + u * stride] : (1u << 8);
  } else {
    const uint32_t *p = (const uint32_t *)tl.list;
#pragma unroll
    for (int u = 0; u < 4; ++u) q[u] = (t + u * stride < nt) ? p[t + u * stride] : (1u << 16);
  }
}

// Front of the queue, the rest moved up (static register indices: the step's
// body stays a single copy, so the kernel keeps its register budget).
__device__ __forceinline__ uint32_t pop_q4(uint32_t (&q)[4]) {
  const uint32_t v = q[0];
  q[0] = q[1];
  q[1] = q[2];
  q[2] = q[3];
  return v;
}

// ---------------------------------------------------------------------------
// triplet lists
// ---------------------------------------------------------------------------
// forward
// ---------------------------------------------------------------------------
template <typename T, int NCH>
__device__ __forceinline__ void ang_fwd_term(const TripletList &tl, uint32_t q, bool active, int c0,
                                             const SFDev &sf, const T *s_d,
                                             const T *s_rw, const T *s_fc, int KP, T (&acc)[NCH],
                                             T (&accw)[NCH]) {
  const int a = q & tl.mask, b = q >> tl.shift;
  const T ax = s_d[4 * a], ay = s_d[4 * a + 1], az = s_d[4 * a + 2], ra = s_d[4 * a + 3];
  const T bx = s_d[4 * b], by = s_d[4 * b + 1], bz = s_d[4 * b + 2], rb = s_d[4 * b + 3];
  const T ex = bx - ax, ey = by - ay, ez = bz - az;
  const T e2 = ex * ex + ey * ey + ez * ez;
  const T e = Math<T>::sq(e2);
  typedef typename Pair<T>::type P2;
  const P2 rwa = ((const P2 *)s_rw)[a], rwb = ((const P2 *)s_rw)[b];  // (1/r, w)
  const T cth = (ra * ra + rb * rb - e2) * (T(0.5) * rwa.x * rwb.x);
  const T S2 = ra * ra + rb * rb + e2;
  const T wab = rwa.y * rwb.y;
  const T on = active ? T(1) : T(0);
  int cur_g = -1;
  T F3 = 0, E = 0, cur_eta = T(-1);
  PowState<T> ps;
#pragma unroll
  for (int l = 0; l < NCH; ++l) {
    const int s = c0 + l;
    if (s < sf.n_ang) {
      const int g = sf.ang_group[s];
      if (g != cur_g) {
        cur_g = g;
        cur_eta = T(-1);  // E below carries this group's cutoff product
        const T rc = (T)sf.group_rc[g];
        const T fe = (e <= rc) ? T(0.5) * Math<T>::cos1((T)sf.group_pirc[g], e) : T(0);
        F3 = s_fc[g * KP + a] * s_fc[g * KP + b] * fe * on;
      }
      const T eta = (T)sf.ang_eta[s];
      if (eta != cur_eta) {
        cur_eta = eta;
        E = Math<T>::ex(-eta * S2) * F3;
      }
      T P, dP;
      line_power<T>(sf, s, cth, ps, P, dP);
      const T t = P * E;
      acc[l] += t;
      accw[l] += t * wab;
    }
  }
}

// W wavefronts per atom (workgroup of 64 W threads): neighbours, triplets
// and radial terms are split over the waves; each chunk's per-lane sums are
// reduced within a wave and then across the waves through LDS.
template <typename T, int NCH, int W>
__device__ __forceinline__ void chunk_reduce(T (&acc)[NCH], T (&accw)[NCH], int wv, int lane, int tid, int c0,
                                             int n, const int *__restrict__ feat, int nsf, T *s_part, T *s_feat) {
#pragma unroll
  for (int l = 0; l < NCH; ++l) {
    const T v = wave_sum(acc[l]);
    const T vw = wave_sum(accw[l]);
    if (lane == 0) {
      s_part[wv * 2 * NCH + l] = v;
      s_part[wv * 2 * NCH + NCH + l] = vw;
    }
  }
  __syncthreads();
  if (tid < 2 * NCH) {
    const int l = tid % NCH;
    if (c0 + l < n) {
      T sum = T(0);
#pragma unroll
      for (int w = 0; w < W; ++w) sum += s_part[w * 2 * NCH + tid];
      s_feat[feat[c0 + l] + (tid >= NCH ? nsf : 0)] = sum;
    }
  }
  __syncthreads();
}

// FG: the per-group cutoff tables live in the global buffer nb.fc_scratch
// (row of atom i) instead of LDS, for neighbour lists too long for the LDS
// layout (launched with one wavefront per atom).
template <typename T, int NCH, int W, bool FG>
__global__ __launch_bounds__(W > 4 ? 64 * W : 256) void k_desc_fwd(int N, const int *__restrict__ species,
                                                  const double *__restrict__ wz, NeighborBufs nb, TripletBufs tb,
                                                  SFDev sf, Lds L, const double *__restrict__ theta_inv,
                                                  const double *__restrict__ mu, int split_mode, DescOut out) {
  extern __shared__ __align__(16) unsigned char smem[];
  if ((int)blockIdx.x >= N) return;  // one workgroup per atom of [atom0, atom0 + N)
  const int i = L.atom0 + blockIdx.x;
  const int tid = threadIdx.x, wv = wave_index(), lane = tid & 63;
  const int KP = L.KP, Dp = L.Dp;
  double *s_xn = (double *)smem;  // [W], padded to 16 bytes
  T *s_d = (T *)(s_xn + ((W + 1) & ~1));
  T *s_rw = s_d + 4 * KP;         // [KP] pairs (1 / r, species weight)
  T *s_fc = FG ? (T *)nb.fc_scratch + (size_t)i * L.G * KP : s_rw + 2 * KP;
  T *s_feat = FG ? s_rw + 2 * KP : s_fc + L.G * KP;
  T *s_part = s_feat + Dp;  // [W * 2 * NCH]

  const int start = i * nb.kcap;
  const int K = nb.nb_count[i];
  if (K > KP) {  // the host sizes KP from the capacity; never index LDS past it
    if (tid == 0) atomicAdd(&nb.total[3], 1);
    return;
  }
  stage_neighbours<T, false>(nb, wz, species, sf, start, K, KP, s_d, s_rw, s_fc, tid, 64 * W);
  for (int d = tid; d < Dp; d += 64 * W) s_feat[d] = T(0);
  __syncthreads();

  // radial lines, NCH at a time
  for (int c0 = 0; c0 < sf.n_rad; c0 += NCH) {
    T acc[NCH], accw[NCH];
#pragma unroll
    for (int l = 0; l < NCH; ++l) acc[l] = accw[l] = T(0);
    for (int a = tid; a < K; a += 64 * W) {
      const T r = s_d[4 * a + 3], w = s_rw[2 * a + 1];
#pragma unroll
      for (int l = 0; l < NCH; ++l) {
        const int s = c0 + l;
        if (s < sf.n_rad) {
          const T dr = r - rad_table<T>(sf.rad_rs, sf.rad_rs32, s);
          const T t = Math<T>::ex(-rad_table<T>(sf.rad_a, sf.rad_a32, s) * dr * dr) * s_fc[sf.rad_group[s] * KP + a];
          acc[l] += t;
          accw[l] += t * w;
        }
      }
    }
    chunk_reduce<T, NCH, W>(acc, accw, wv, lane, tid, c0, sf.n_rad, sf.rad_feat, sf.nsf, s_part, s_feat);
  }

  // angular lines, NCH at a time, over the atom's triplet list
  const TripletList tl(tb, i);
  const int nt = tb.count[i];
  for (int c0 = 0; c0 < sf.n_ang; c0 += NCH) {
    T acc[NCH], accw[NCH];
#pragma unroll
    for (int l = 0; l < NCH; ++l) acc[l] = accw[l] = T(0);
    constexpr int ST = 64 * W;
    uint32_t qc[4], qn[4];
    load_q4(tl, nt, 64 * wv + lane, ST, qc);
    for (int t0 = 64 * wv; t0 < nt; t0 += 4 * ST) {
      load_q4(tl, nt, t0 + 4 * ST + lane, ST, qn);
#pragma unroll 1
      for (int u = 0; u < 4; ++u) {
        const uint32_t q = pop_q4(qc);
        ang_fwd_term<T, NCH>(tl, q, t0 + u * ST + lane < nt, c0, sf, s_d, s_rw, s_fc, KP, acc, accw);
      }
#pragma unroll
      for (int u = 0; u < 4; ++u) qc[u] = qn[u];
    }
    chunk_reduce<T, NCH, W>(acc, accw, wv, lane, tid, c0, sf.n_ang, sf.ang_feat, sf.nsf, s_part, s_feat);
  }

  double xn = write_features<T, W>(s_feat, (size_t)i * Dp, Dp, tid, theta_inv, mu, split_mode, out);
  xn = wave_sum(xn);
  if (lane == 0) s_xn[wv] = xn;
  __syncthreads();
  if (tid == 0) {
    double v = 0.0;
#pragma unroll
    for (int w = 0; w < W; ++w) v += s_xn[w];
    out.xn[i] = v;
  }
}

// ---------------------------------------------------------------------------
// grid form of the angular table: eta x (lambda = +1, -1) x zeta, zeta in
// {1, 2, 4, 8, 16}, one cutoff group (SFDev::grid).  Powers come from one
// squaring chain per lambda, (lambda, zeta) products are unrolled, and only
// the eta loop is a (uniform) runtime loop.
// ---------------------------------------------------------------------------
// With pref_k = 2^(1 - zeta_k) (the only prefactor the tables hold), the
// angular factor is pref_k b^zeta_k = 2 u^zeta_k for u = b / 2 = (1 + lam cos)
// / 2, lam = +1 (p) and -1 (m).  This returns the halves P_k = u^zeta_k and
// dP_k/dcos = lam zeta_k u^(zeta_k - 1) / 2; the callers put the factor 2 on
// their per-triplet products once.  zeta_k = 2^zlog[k] with zlog ascending:
// one squaring chain, advanced by uniform trip counts (registers only; an
// indexed table of powers would go to scratch memory).
// Z16: the zeta list is {1, 2, 4, 16} (zlog {0, 1, 2, 4}, the usual grid),
// known at compile time, so the chain is straight-line code with the same
// multiplications in the same order.
// RAWQ: dPp and dPm are the bare u^(zeta_k - 1) (the callers carry the factors
// lam zeta_k / 2 elsewhere).
template <typename T, int NZ, bool DERIV, bool Z16, bool RAWQ = false>
__device__ __forceinline__ void grid_powers(T cth, const SFDev &sf, T (&Pp)[NZ], T (&Pm)[NZ], T (&dPp)[NZ],
                                            T (&dPm)[NZ]) {
  static_assert(!Z16 || NZ == 4, "the {1, 2, 4, 16} list has four zetas");
  const T hc = T(0.5) * cth;
  T p = T(0.5) + hc, m = T(0.5) - hc;  // u^(2^t)
  T qp = T(1), qm = T(1);              // u^(2^t - 1)
  int t = 0;
#pragma unroll
  for (int k = 0; k < NZ; ++k) {
    const int j = Z16 ? (k < 3 ? k : 4) : sf.zlog[k];
    if constexpr (Z16) {
#pragma unroll
      for (int u = 0; u < 4; ++u)  // at most 4 squarings per zeta; t and j are constants here
        if (t < j) {
          if (DERIV) {
            qp *= p;
            qm *= m;
          }
          p *= p;
          m *= m;
          ++t;
        }
    } else {
      for (; t < j; ++t) {
        if (DERIV) {
          qp *= p;
          qm *= m;
        }
        p *= p;
        m *= m;
      }
    }
    Pp[k] = p;
    Pm[k] = m;
    if (DERIV) {
      const T hz = RAWQ ? T(1) : T(0.5) * (T)sf.zeta_k[k];  // zeta_k / 2, exact
      dPp[k] = RAWQ ? qp : hz * qp;
      dPm[k] = RAWQ ? qm : -hz * qm;
    }
  }
}

// exp(-eta x) as the grid kernels evaluate it: in FP32 the hardware 2^x with
// the coefficient -eta log2(e) formed once per eta (one multiplication per
// term instead of two); in FP64 exp64.
template <typename T>
__device__ __forceinline__ T eta_coef(T eta);
template <>
__device__ __forceinline__ float eta_coef<float>(float eta) { return -eta * 1.44269504088896341f; }
template <>
__device__ __forceinline__ double eta_coef<double>(double eta) { return -eta; }
// 2 A / |coefficient|: the factor that turns coefficient times dr into -2 A dr.
template <typename T>
constexpr __device__ __forceinline__ T slope_factor() {
  return sizeof(T) == 4 ? T(1.38629436111989062) : T(2);
}
__device__ __forceinline__ float exp_coef(float c, float x) { return __builtin_amdgcn_exp2f(c * x); }
__device__ __forceinline__ double exp_coef(double c, double x) { return exp64(c * x); }

// Sum NV per-lane values over the workgroup: s_out[j] = total of v[j].  Within
// a wavefront a butterfly reduce-scatter: at offset m (32, 16, .., 1) every
// lane keeps the half of its live values selected by its own bit m and adds
// the partner's copy of that half, so lane l ends with the total of value l
// (NV padded to 32 or 64; for 32 the butterfly runs within each half-wave and
// the halves' totals are added last).  NV - 1 exchanges instead of NV full
// wave reductions; the offsets 32 and 16 use gfx950's lane swaps (below).
// The waves' totals are then added in wave order (deterministic).
// One butterfly level per instantiation, so every register index is a
// compile-time constant (a loop over M left rolled by the compiler would
// index the array at run time).
// gfx950's lane swaps between the halves of a wave (permlane32) or between
// the 16-lane rows of each half (permlane16), applied to a pair (a, b): a
// becomes {a, b} of the lower halves (rows 0 and 2) and b becomes {a, b} of
// the upper ones (rows 1 and 3), as the lanes see them.  Then a + b gives every
// lower lane its own a plus its partner's a, and every upper lane its own b
// plus its partner's b: one butterfly step without a shuffle and two selects.
template <int M>
__device__ __forceinline__ void swap_halves(unsigned &a, unsigned &b) {
  static_assert(M == 32 || M == 16, "lane swaps exist for offsets 32 and 16");
  if constexpr (M == 32) {
    const auto r = __builtin_amdgcn_permlane32_swap(a, b, false, false);
    a = r[0];
    b = r[1];
  } else {
    const auto r = __builtin_amdgcn_permlane16_swap(a, b, false, false);
    a = r[0];
    b = r[1];
  }
}

template <int M>
__device__ __forceinline__ float swap_sum(float a, float b) {
  unsigned u = __float_as_uint(a), v = __float_as_uint(b);
  swap_halves<M>(u, v);
  return __uint_as_float(u) + __uint_as_float(v);
}

template <int M>
__device__ __forceinline__ double swap_sum(double a, double b) {
  unsigned long long u = __double_as_longlong(a), v = __double_as_longlong(b);
  unsigned ul = (unsigned)u, uh = (unsigned)(u >> 32), vl = (unsigned)v, vh = (unsigned)(v >> 32);
  swap_halves<M>(ul, vl);
  swap_halves<M>(uh, vh);
  return __longlong_as_double((long long)(((unsigned long long)uh << 32) | ul)) +
         __longlong_as_double((long long)(((unsigned long long)vh << 32) | vl));
}

// The value of the lane at l ^ M for M = 8, 4, 2, 1 (within a row of 16 lanes)
// by cross-lane moves of the vector units instead of a trip through LDS: a row
// rotation by 8, quad permutations for 1 and 2, and for 4 the reversal of each
// half row (l ^ 7) after that of each quad (l ^ 3).
template <int CTRL>
__device__ __forceinline__ unsigned dpp32(unsigned v) {
  return __builtin_amdgcn_update_dpp(0, v, CTRL, 0xf, 0xf, true);
}
template <int M>
__device__ __forceinline__ unsigned lane_xor(unsigned v) {
  static_assert(M == 8 || M == 4 || M == 2 || M == 1, "within a row");
  if constexpr (M == 8) return dpp32<0x128>(v);                // row_ror:8
  if constexpr (M == 4) return dpp32<0x141>(dpp32<0x1B>(v));   // quad_perm:[3,2,1,0], row_half_mirror
  if constexpr (M == 2) return dpp32<0x4E>(v);                 // quad_perm:[2,3,0,1]
  return dpp32<0xB1>(v);                                       // quad_perm:[1,0,3,2]
}
template <int M>
__device__ __forceinline__ float lane_xor(float v) {
  return __uint_as_float(lane_xor<M>(__float_as_uint(v)));
}
template <int M>
__device__ __forceinline__ double lane_xor(double v) {
  const unsigned long long u = __double_as_longlong(v);
  const unsigned lo = lane_xor<M>((unsigned)u), hi = lane_xor<M>((unsigned)(u >> 32));
  return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

template <typename T, int M, int NVP>
__device__ __forceinline__ void butterfly(T (&x)[NVP], int lane) {
  if constexpr (M == 32 || M == 16) {
#pragma unroll
    for (int j = 0; j < M; ++j) x[j] = swap_sum<M>(x[j], x[j + M]);
    butterfly<T, M / 2, NVP>(x, lane);
  } else if constexpr (M >= 1) {
    const bool upper = (lane & M) != 0;
#pragma unroll
    for (int j = 0; j < M; ++j) {
      const T send = upper ? x[j] : x[j + M];
      const T keep = upper ? x[j + M] : x[j];
      x[j] = keep + lane_xor<M>(send);
    }
    butterfly<T, M / 2, NVP>(x, lane);
  }
}

// Within the wave: lane l returns the total of v[l % NVP], NVP the next power
// of two (8 to 64) from NV; with fewer than 64 values the butterfly (offsets
// NVP / 2 .. 1) stays within NVP lanes and the groups' totals are added last.
template <typename T, int NV>
__device__ __forceinline__ T wave_totals(T (&v)[NV], int lane) {
  static_assert(NV <= 64, "at most 64 values");
  constexpr int NVP = NV <= 8 ? 8 : NV <= 16 ? 16 : NV <= 32 ? 32 : 64;
  T x[NVP];
#pragma unroll
  for (int j = 0; j < NVP; ++j) x[j] = (j < NV) ? v[j] : T(0);
  butterfly<T, NVP / 2, NVP>(x, lane);
#pragma unroll
  for (int o = NVP; o < 64; o <<= 1) x[0] += __shfl_xor(x[0], o, 64);
  return x[0];
}

template <typename T, int NV, int W>
__device__ __forceinline__ void group_sum(T (&v)[NV], int wv, int lane, int tid, T *s_part, T *s_out) {
  const T x = wave_totals<T, NV>(v, lane);
  if (W == 1) {
    if (lane < NV) s_out[lane] = x;
    __syncthreads();
    return;
  }
  if (lane < NV) s_part[wv * NV + lane] = x;
  __syncthreads();
  for (int j = tid; j < NV; j += 64 * W) {
    T sum = T(0);
#pragma unroll
    for (int w = 0; w < W; ++w) sum += s_part[w * NV + j];
    s_out[j] = sum;
  }
  __syncthreads();
}

template <typename T, int NZ>
struct GridShape {
  static constexpr int CAP = 32;  // (plain, weighted) pairs per pass
  static constexpr int NE = (CAP / (2 * NZ)) > 0 ? CAP / (2 * NZ) : 1;  // etas per pass
  static constexpr int NV = NE * 2 * NZ * 2;
};

// Bound by VALU issue: per triplet the distances, one cutoff product and an exp
// per eta; per atom the radial lines and the reductions.  With the triplets left
// out 500 of the FP32 kernel's 830 us remained at 65,000 atoms of 80 neighbours,
// so the per-atom part counts as much as the triplets: reductions by cross-lane
// moves (lane_xor) instead of LDS exchanges, a radial chunk of one cutoff group
// without tests, two features a thread in the epilogue.  Together, per batch of
// 67,647 atoms: FP64 1120 -> 974 us, FP32 413 -> 375; 65,000 atoms, FP32, without
// forces to follow: 830 -> 750.  Every sum keeps its order, and FP32 features
// their bits: the surrogate rounds them to BF16.
template <typename T, int NZ, int W, bool Z16, bool FG>
__global__ __launch_bounds__(W > 4 ? 64 * W : 256) void k_desc_fwd_grid(int N, const int *__restrict__ species,
                                                       const double *__restrict__ wz, NeighborBufs nb,
                                                       TripletBufs tb, SFDev sf, Lds L,
                                                       const double *__restrict__ theta_inv,
                                                       const double *__restrict__ mu, int split_mode, DescOut out) {
  constexpr int NE = GridShape<T, NZ>::NE, NV = GridShape<T, NZ>::NV;
  constexpr int RCH = W <= 2 ? 16 : 32 / W;  // radial lines per chunk
  extern __shared__ __align__(16) unsigned char smem[];
  if ((int)blockIdx.x >= N) return;  // one workgroup per atom of [atom0, atom0 + N)
  const int i = L.atom0 + blockIdx.x;
  const int tid = threadIdx.x, wv = wave_index(), lane = tid & 63;
  const int KP = L.KP, Dp = L.Dp;
  double *s_xn = (double *)smem;  // [W], padded to 16 bytes
  T *s_d = (T *)(s_xn + ((W + 1) & ~1));
  T *s_rw = s_d + 4 * KP;       // [KP] pairs (1 / r, species weight)
  T *s_fc = FG ? (T *)nb.fc_scratch + (size_t)i * L.G * KP : s_rw + 2 * KP;
  T *s_feat = FG ? s_rw + 2 * KP : s_fc + L.G * KP;
  T *s_part = s_feat + Dp;      // [W * NV]
  T *s_sum = s_part + W * NV;   // [NV]

  const int start = i * nb.kcap;
  const int K = nb.nb_count[i];
  if (K > KP) {
    if (tid == 0) atomicAdd(&nb.total[3], 1);
    return;
  }
  stage_neighbours<T, false>(nb, wz, species, sf, start, K, KP, s_d, s_rw, s_fc, tid, 64 * W);
  for (int d = tid; d < Dp; d += 64 * W) s_feat[d] = T(0);
  __syncthreads();

  // radial lines, RCH at a time, each chunk by one wave over all neighbours:
  // plain sums in acc[0, RCH), weighted ones in acc[RCH, 2 RCH), reduced
  // within the wave (with W waves the chunks of a usual table run beside each
  // other, and none needs an exchange between waves)
  for (int c0 = wv * RCH; c0 < sf.n_rad; c0 += W * RCH) {
    T acc[2 * RCH];
#pragma unroll
    for (int l = 0; l < 2 * RCH; ++l) acc[l] = T(0);
    if (c0 + RCH <= sf.n_rad && sf.rad_g >= 0) {
      // a whole chunk of one cutoff group: no test per line, the tables read
      // in wide scalar loads and the cutoff once per neighbour
      for (int a = lane; a < K; a += 64) {
        const T r = s_d[4 * a + 3], w = s_rw[2 * a + 1], fc = s_fc[sf.rad_g * KP + a];
#pragma unroll
        for (int l = 0; l < RCH; ++l) {
          const T dr = r - rad_table<T>(sf.rad_rs, sf.rad_rs32, c0 + l);
          const T t = Math<T>::ex(-rad_table<T>(sf.rad_a, sf.rad_a32, c0 + l) * dr * dr) * fc;
          acc[l] += t;
          acc[RCH + l] += t * w;
        }
      }
    } else {
      for (int a = lane; a < K; a += 64) {
        const T r = s_d[4 * a + 3], w = s_rw[2 * a + 1];
#pragma unroll
        for (int l = 0; l < RCH; ++l) {
          const int s = c0 + l;
          if (s < sf.n_rad) {
            const T dr = r - rad_table<T>(sf.rad_rs, sf.rad_rs32, s);
            const T t = Math<T>::ex(-rad_table<T>(sf.rad_a, sf.rad_a32, s) * dr * dr) * s_fc[sf.rad_group[s] * KP + a];
            acc[l] += t;
            acc[RCH + l] += t * w;
          }
        }
      }
    }
    const T v = wave_totals<T, 2 * RCH>(acc, lane);
    const int l = lane % RCH;
    if (lane < 2 * RCH && c0 + l < sf.n_rad) s_feat[sf.rad_feat[c0 + l] + (lane >= RCH ? sf.nsf : 0)] = v;
  }

  // angular lines in grid form, NE etas per pass
  const TripletList tl(tb, i);
  const int nt = tb.count[i];
  const int g = sf.g_ang;
  const T rc = (T)sf.group_rc[g];
  const T pirc = (T)sf.group_pirc[g];
  for (int h0 = 0; h0 < sf.n_eta; h0 += NE) {
    T acc[NV];
#pragma unroll
    for (int j = 0; j < NV; ++j) acc[j] = T(0);
    T ceta_h[NE];  // this pass's exp coefficients (uniform), formed once
#pragma unroll
    for (int hh = 0; hh < NE; ++hh)
      ceta_h[hh] = eta_coef<T>((h0 + hh < sf.n_eta) ? (T)sf.ang_eta[(h0 + hh) * 2 * NZ] : T(0));
    constexpr int ST = 64 * W;
    uint32_t qc[4], qn[4];
    load_q4(tl, nt, 64 * wv + lane, ST, qc);
    for (int t00 = 64 * wv; t00 < nt; t00 += 4 * ST) {
      load_q4(tl, nt, t00 + 4 * ST + lane, ST, qn);
#pragma unroll 1
      for (int u = 0; u < 4; ++u) {
        const bool act = t00 + u * ST + lane < nt;
        const uint32_t q = pop_q4(qc);
        const int a = q & tl.mask, b = q >> tl.shift;
        const T ax = s_d[4 * a], ay = s_d[4 * a + 1], az = s_d[4 * a + 2], ra = s_d[4 * a + 3];
        const T bx = s_d[4 * b], by = s_d[4 * b + 1], bz = s_d[4 * b + 2], rb = s_d[4 * b + 3];
        const T ex = bx - ax, ey = by - ay, ez = bz - az;
        const T e2 = ex * ex + ey * ey + ez * ez;
        const T e = Math<T>::sq(e2);
        typedef typename Pair<T>::type P2;
        const P2 rwa = ((const P2 *)s_rw)[a], rwb = ((const P2 *)s_rw)[b];  // (1/r, w)
        const T cth = (ra * ra + rb * rb - e2) * (T(0.5) * rwa.x * rwb.x);
        const T S2 = ra * ra + rb * rb + e2;
        const T wab = rwa.y * rwb.y;
        // 2 fc(r_jk): the factor 2 of the halved powers (grid_powers) rides here
        const T fe2 = (e <= rc) ? Math<T>::cos1(pirc, e) : T(0);
        const T F3 = act ? s_fc[g * KP + a] * s_fc[g * KP + b] * fe2 : T(0);
        T Pp[NZ], Pm[NZ], dPp[NZ], dPm[NZ];
        grid_powers<T, NZ, false, Z16>(cth, sf, Pp, Pm, dPp, dPm);
#pragma unroll
        for (int hh = 0; hh < NE; ++hh) {
          const int h = h0 + hh;
          if (h < sf.n_eta) {
            // plain and weighted sums as four FMAs per zeta (E w_ab formed once)
            const T E = exp_coef(ceta_h[hh], S2) * F3, Ew = E * wab;
#pragma unroll
            for (int k = 0; k < NZ; ++k) {
              acc[(hh * 2 + 0) * NZ + k] += E * Pp[k];
              acc[(hh * 2 + 1) * NZ + k] += E * Pm[k];
              acc[NV / 2 + (hh * 2 + 0) * NZ + k] += Ew * Pp[k];
              acc[NV / 2 + (hh * 2 + 1) * NZ + k] += Ew * Pm[k];
            }
          }
        }
      }
#pragma unroll
      for (int u = 0; u < 4; ++u) qc[u] = qn[u];
    }
    group_sum<T, NV, W>(acc, wv, lane, tid, s_part, s_sum);
    for (int j = tid; j < NV; j += 64 * W) {
      const int jl = j % (NV / 2);            // (hh, li, k)
      const int h = h0 + jl / (2 * NZ);
      if (h < sf.n_eta) s_feat[sf.ang_feat[h0 * 2 * NZ + jl] + (j >= NV / 2 ? sf.nsf : 0)] = s_sum[j];
    }
    __syncthreads();
  }

  double xn = write_features<T, W>(s_feat, (size_t)i * Dp, Dp, tid, theta_inv, mu, split_mode, out);
  xn = wave_sum(xn);
  if (lane == 0) s_xn[wv] = xn;
  __syncthreads();
  if (tid == 0) {
    double v = 0.0;
#pragma unroll
    for (int w = 0; w < W; ++w) v += s_xn[w];
    out.xn[i] = v;
  }
}

// Values per eta record of the grid-form backward (see k_desc_bwd): 4 NZ g
// values, eta and its exp coefficient, rounded up to whole 16-byte groups.
template <int NZ>
struct EtaRec {
  static constexpr int RS = NZ > 0 ? (4 * NZ + 2 + 3) & ~3 : 0;
};

// The grid-form backward's per-eta sums over the 2 NZ lines,
//   sb_h = sum_z (gA_hz + w gW_hz) P_z,   sa_h the same with dP_z / dcos,
// need all 4 NZ values of g per eta for every triplet.  Read from LDS as
// records (one address for the whole wave), those reads were 20 (FP32) to 36
// (FP64) of the 34 to 50 LDS instructions per 64 triplets, and with the LDS
// busy 72-79 % of the time they bounded the kernel; so g stays in registers
// spread over the lanes, in the forms below.

// FP32 on the matrix cores: v_mfma_f32_4x4x1_16b_f32 multiplies, in each of
// 16 groups of four lanes, a column of four A values by a row of four B values.
// With B = P_z of each lane's own triplet and A = g of four etas for line z
// (held by the lanes 4 z .. 4 z + 3 of one register and broadcast to every group:
// cbsz 4, abid z), lane l's four results are its own triplet's four partial
// sums: no data moves between lanes, each is an FP32 fused multiply-add as
// on the vector units, and 96 of the 220 vector instructions per 64 triplets
// move to the otherwise idle matrix cores.
typedef float v4f __attribute__((ext_vector_type(4)));

// Registers of one set of four etas: lane 4 z + i holds line z of eta i, plain
// (a) and weighted (w), for P (p) and, with the factor lam zeta / 2, for the
// bare derivative powers (q).
struct EtaSet {
  float ap, wp, aq, wq;
};

template <int NZ>
__device__ __forceinline__ EtaSet load_eta_set(const SFDev &sf, const float *s_g, int set, int lane) {
  const int h = 4 * set + (lane & 3), z = lane >> 2;
  EtaSet e{0.f, 0.f, 0.f, 0.f};
  if (h < sf.n_eta && z < 2 * NZ) {
    const int s = h * 2 * NZ + z, f = sf.ang_feat[s];
    const float hz = (z < NZ ? 0.5f : -0.5f) * (float)sf.ang_zeta[s];
    e.ap = s_g[f];
    e.wp = s_g[f + sf.nsf];
    e.aq = hz * e.ap;
    e.wq = hz * e.wp;
  }
  return e;
}

template <int Z, int NZ>
__device__ __forceinline__ void eta_products(const EtaSet &e, const float (&Pp)[NZ], const float (&Pm)[NZ],
                                             const float (&Qp)[NZ], const float (&Qm)[NZ], v4f &ba, v4f &bw, v4f &aa,
                                             v4f &aw) {
  if constexpr (Z < 2 * NZ) {
    constexpr int k = Z % NZ;
    const float P = Z < NZ ? Pp[k] : Pm[k], Q = Z < NZ ? Qp[k] : Qm[k];
    ba = __builtin_amdgcn_mfma_f32_4x4x1f32(e.ap, P, ba, 4, Z, 0);
    bw = __builtin_amdgcn_mfma_f32_4x4x1f32(e.wp, P, bw, 4, Z, 0);
    aa = __builtin_amdgcn_mfma_f32_4x4x1f32(e.aq, Q, aa, 4, Z, 0);
    aw = __builtin_amdgcn_mfma_f32_4x4x1f32(e.wq, Q, aw, 4, Z, 0);
    eta_products<Z + 1, NZ>(e, Pp, Pm, Qp, Qm, ba, bw, aa, aw);
  }
}

// FP64 through the cross-lane operand of the vector units: a row of 16 lanes
// holds an eta's line values, line z in lane z, and v_fmac_f64 takes one of
// them, broadcast over the row (row_newbcast), as its multiplicand.  A block
// does lines Z .. Z + NB - 1; its first instruction waits out the two states
// between a vector write of a register and its cross-lane read.
#define GAPX_ROW_LINE(z, p, q)                                    \
  "v_fmac_f64_dpp %0, %4, " p " row_newbcast:" z " row_mask:0xf bank_mask:0xf\n" \
  "v_fmac_f64_dpp %1, %5, " p " row_newbcast:" z " row_mask:0xf bank_mask:0xf\n" \
  "v_fmac_f64_dpp %2, %4, " q " row_newbcast:" z " row_mask:0xf bank_mask:0xf\n" \
  "v_fmac_f64_dpp %3, %5, " q " row_newbcast:" z " row_mask:0xf bank_mask:0xf\n"
template <int Z, int NZ>
__device__ __forceinline__ void row_products(double ga, double gw, const double (&Pp)[NZ], const double (&Pm)[NZ],
                                             const double (&dPp)[NZ], const double (&dPm)[NZ], double &ba, double &bw,
                                             double &aa, double &aw) {
  static_assert(2 * NZ <= 16, "a row has 16 lanes");
  auto P = [&](int z) { return z < NZ ? Pp[z] : Pm[z - NZ]; };
  auto Q = [&](int z) { return z < NZ ? dPp[z] : dPm[z - NZ]; };
  if constexpr (Z + 4 <= 2 * NZ) {
    asm("s_nop 1\n" GAPX_ROW_LINE("%c14", "%6", "%10") GAPX_ROW_LINE("%c15", "%7", "%11")
            GAPX_ROW_LINE("%c16", "%8", "%12") GAPX_ROW_LINE("%c17", "%9", "%13")
        : "+&v"(ba), "+&v"(bw), "+&v"(aa), "+&v"(aw)
        : "v"(ga), "v"(gw), "v"(P(Z)), "v"(P(Z + 1)), "v"(P(Z + 2)), "v"(P(Z + 3)), "v"(Q(Z)), "v"(Q(Z + 1)),
          "v"(Q(Z + 2)), "v"(Q(Z + 3)), "i"(Z), "i"(Z + 1), "i"(Z + 2), "i"(Z + 3));
    row_products<Z + 4, NZ>(ga, gw, Pp, Pm, dPp, dPm, ba, bw, aa, aw);
  } else if constexpr (Z + 2 <= 2 * NZ) {
    asm("s_nop 1\n" GAPX_ROW_LINE("%c10", "%6", "%8") GAPX_ROW_LINE("%c11", "%7", "%9")
        : "+&v"(ba), "+&v"(bw), "+&v"(aa), "+&v"(aw)
        : "v"(ga), "v"(gw), "v"(P(Z)), "v"(P(Z + 1)), "v"(Q(Z)), "v"(Q(Z + 1)), "i"(Z), "i"(Z + 1));
    row_products<Z + 2, NZ>(ga, gw, Pp, Pm, dPp, dPm, ba, bw, aa, aw);
  }
}
#undef GAPX_ROW_LINE

// g of the grid-form backward in registers, for tables of at most 4 ES etas
// (ES > 0: FP32 up to two sets, FP64 one); ES = 0: from the LDS records.
template <typename T, int ES>
struct EtaRegs;
template <int ES>
struct EtaRegs<float, ES> {
  EtaSet set[ES > 0 ? ES : 1];
};
template <int ES>
struct EtaRegs<double, ES> {
  double ga[4], gw[4];  // row lane z: line z of eta h
};

template <typename T, int NZ, bool Z16, int ES>
__device__ __forceinline__ void ang_bwd_grid(const TripletList &tl, uint32_t q, bool active,
                                             const SFDev &sf, const T *s_d, const T *s_rw,
                                             const T *s_fd, const T *s_er, const EtaRegs<T, ES> &er,
                                             const T (&ceta)[4 * ES + 1], const T (&eta)[4 * ES + 1], int KP, T rc,
                                             T pirc, double *s_T, double *s_F) {
  // idle lanes work on neighbours 0 and 1 (the products need every lane) and
  // add nothing at the end
  const int a = q & tl.mask, b = q >> tl.shift;
  const T ax = s_d[4 * a], ay = s_d[4 * a + 1], az = s_d[4 * a + 2], ra = s_d[4 * a + 3];
  const T bx = s_d[4 * b], by = s_d[4 * b + 1], bz = s_d[4 * b + 2], rb = s_d[4 * b + 3];
  typedef typename Pair<T>::type P2;
  const P2 rwa = ((const P2 *)s_rw)[a], rwb = ((const P2 *)s_rw)[b];  // (1/r, w)
  const T ria = rwa.x, rib = rwb.x;
  const T ex = bx - ax, ey = by - ay, ez = bz - az;
  // the floor keeps 1 / e finite for coincident neighbours (their vector is 0)
  const T e2 = fma(ex, ex, fma(ey, ey, fma(ez, ez, Math<T>::floor2())));
  T e, ie;
  Math<T>::sqrt_rsq(e2, e, ie);
  const T inv2ab = T(0.5) * ria * rib;
  const T cth = (ra * ra + rb * rb - e2) * inv2ab;
  const T S2 = ra * ra + rb * rb + e2;
  const T dca = rib - cth * ria, dcb = ria - cth * rib, dce = -e * (T(2) * inv2ab);
  const T wab = rwa.y * rwb.y;
  const int g = sf.g_ang;
  const P2 fda = ((const P2 *)s_fd)[g * KP + a], fdb = ((const P2 *)s_fd)[g * KP + b];  // (fc, dfc)
  const T fa = fda.x, dfa = fda.y, fb = fdb.x, dfb = fdb.y;
  const bool in = e <= rc;
  T sine, cos1;
  Math<T>::sincos1(Math<T>::turn(pirc), e, sine, cos1);
  // 2 fc(r_jk) and its derivative: every term below carries exactly one of
  // them, which puts the factor 2 of the halved powers (grid_powers) on all
  const T fe = in ? cos1 : T(0);
  const T dfe = in ? -sine * pirc : T(0);
  T Pp[NZ], Pm[NZ], dPp[NZ], dPm[NZ];
  constexpr bool kMfma = ES > 0 && sizeof(T) == 4;
  grid_powers<T, NZ, true, Z16, kMfma>(cth, sf, Pp, Pm, dPp, dPm);
  T SA = 0, SB = 0, SC = 0;
  // one eta's sums over the lines times its exponential
  auto add_eta = [&](T sa, T sb, T E, T et) {
    const T t = sb * E;
    SA += sa * E;
    SB += t;
    SC += et * t;
  };
  if constexpr (kMfma) {
#pragma unroll
    for (int u = 0; u < ES; ++u) {
      v4f ba{0.f, 0.f, 0.f, 0.f}, bw = ba, aa = ba, aw = ba;
      eta_products<0, NZ>(er.set[u], Pp, Pm, dPp, dPm, ba, bw, aa, aw);
#pragma unroll
      for (int i = 0; i < 4; ++i)
        add_eta(aa[i] + wab * aw[i], ba[i] + wab * bw[i], exp_coef(ceta[4 * u + i], S2), eta[4 * u + i]);
    }
  } else if constexpr (ES > 0) {
#pragma unroll
    for (int h = 0; h < 4; ++h) {
      if (h < sf.n_eta) {
        T ba = 0, bw = 0, aa = 0, aw = 0;
        row_products<0, NZ>(er.ga[h], er.gw[h], Pp, Pm, dPp, dPm, ba, bw, aa, aw);
        add_eta(aa + wab * aw, ba + wab * bw, exp_coef(ceta[h], S2), eta[h]);
      }
    }
  } else {
    // from the LDS records: the lines' g contracted with the powers (sb) and
    // with their cos-derivatives (sa), each sum started from its first term.
    // Long lists leave one wave per SIMD here (LDS), so what one wave waits for
    // counts: a record is read whole before its use, two etas per trip, the
    // exponential's constants once per triplet, and in reads of 16 bytes, which
    // the compiler makes only of a type with that alignment (nine etas, one wave
    // per atom, 4-byte alignment -> 16: 12,000 atoms of 181 neighbours FP32 1621 ->
    // 1388 us, FP64 3742 -> 3253, of 63 neighbours 232 -> 194 and 437 -> 377).
    typename std::conditional<sizeof(T) == 8, ExpConst, int>::type ec{};
#pragma unroll 2
    for (int h = 0; h < sf.n_eta; ++h) {
      const Quad<T> *rec = (const Quad<T> *)(s_er + h * EtaRec<NZ>::RS);
      T v[EtaRec<NZ>::RS];
#pragma unroll
      for (int j = 0; j < EtaRec<NZ>::RS / 4; ++j) {
        const Quad<T> q = rec[j];
#pragma unroll
        for (int i = 0; i < 4; ++i) v[4 * j + i] = q.v[i];
      }
      T E;
      if constexpr (sizeof(T) == 8)
        E = exp64(v[4 * NZ + 1] * S2, ec);
      else
        E = exp_coef(v[4 * NZ + 1], S2);
      T sa = 0, sb = 0;
#pragma unroll
      for (int k = 0; k < NZ; ++k) {
        const T gp = v[k] + wab * v[2 * NZ + k], gm = v[NZ + k] + wab * v[3 * NZ + k];
        sa = k == 0 ? gp * dPp[0] : fma(gp, dPp[k], sa);
        sb = k == 0 ? gp * Pp[0] : fma(gp, Pp[k], sb);
        sa = fma(gm, dPm[k], sa);
        sb = fma(gm, Pm[k], sb);
      }
      add_eta(sa, sb, E, v[4 * NZ]);
    }
  }
  const T F = fa * fb * fe, FA = F * SA, FC = T(-2) * F * SC;
  const T Ta = FA * dca + ra * FC + SB * (dfa * (fb * fe));
  const T Tb = FA * dcb + rb * FC + SB * (dfb * (fa * fe));
  const T Te = FA * dce + e * FC + SB * (fa * fb * dfe);
  const T sc = Te * ie;  // at e = 0 the vector is 0
  const T ux = sc * ex, uy = sc * ey, uz = sc * ez;
  if (active) {
    atomicAdd(&s_T[a], (double)Ta);
    atomicAdd(&s_T[b], (double)Tb);
    atomicAdd(&s_F[3 * b], (double)ux);
    atomicAdd(&s_F[3 * b + 1], (double)uy);
    atomicAdd(&s_F[3 * b + 2], (double)uz);
    atomicAdd(&s_F[3 * a], (double)-ux);
    atomicAdd(&s_F[3 * a + 1], (double)-uy);
    atomicAdd(&s_F[3 * a + 2], (double)-uz);
  }
}

// ---------------------------------------------------------------------------
// backward
// ---------------------------------------------------------------------------
template <typename T>
__device__ __forceinline__ void ang_bwd_term(const TripletList &tl, uint32_t q, bool active,
                                             const SFDev &sf, const T *s_d,
                                             const T *s_rw, const T *s_fd, const T *s_gA, const T *s_gW, int KP,
                                             double *s_T, double *s_F) {
  if (!active) return;
  const int a = q & tl.mask, b = q >> tl.shift;
  const T ax = s_d[4 * a], ay = s_d[4 * a + 1], az = s_d[4 * a + 2], ra = s_d[4 * a + 3];
  const T bx = s_d[4 * b], by = s_d[4 * b + 1], bz = s_d[4 * b + 2], rb = s_d[4 * b + 3];
  const T ex = bx - ax, ey = by - ay, ez = bz - az;
  const T e2 = fma(ex, ex, fma(ey, ey, fma(ez, ez, Math<T>::floor2())));
  T e, ie;
  Math<T>::sqrt_rsq(e2, e, ie);
  typedef typename Pair<T>::type P2;
  const P2 rwa = ((const P2 *)s_rw)[a], rwb = ((const P2 *)s_rw)[b];  // (1/r, w)
  const T ria = rwa.x, rib = rwb.x;
  const T inv2ab = T(0.5) * ria * rib;
  const T cth = (ra * ra + rb * rb - e2) * inv2ab;
  const T S2 = ra * ra + rb * rb + e2;
  const T dca = rib - cth * ria, dcb = ria - cth * rib, dce = -e * (T(2) * inv2ab);
  const T wab = rwa.y * rwb.y;
  T Ta = 0, Tb = 0, Te = 0;
  T SA = 0, SB = 0, SC = 0;
  T fa = 0, dfa = 0, fb = 0, dfb = 0, fe = 0, dfe = 0;
  int cur_g = -1;
  T E = 0, cur_eta = T(-1);
  PowState<T> ps;
  auto flush = [&]() {
    const T F = fa * fb * fe;
    Ta += F * SA * dca - T(2) * ra * F * SC + SB * dfa * fb * fe;
    Tb += F * SA * dcb - T(2) * rb * F * SC + SB * fa * dfb * fe;
    Te += F * SA * dce - T(2) * e * F * SC + SB * fa * fb * dfe;
  };
  for (int s = 0; s < sf.n_ang; ++s) {
    const int g = sf.ang_group[s];
    if (g != cur_g) {
      if (cur_g >= 0) flush();
      cur_g = g;
      SA = SB = SC = T(0);
      const T rc = (T)sf.group_rc[g];
      fa = s_fd[2 * (g * KP + a)];
      dfa = s_fd[2 * (g * KP + a) + 1];
      fb = s_fd[2 * (g * KP + b)];
      dfb = s_fd[2 * (g * KP + b) + 1];
      const bool in = e <= rc;
      const T pirc = (T)sf.group_pirc[g];
      T sine, cos1;
      Math<T>::sincos1(Math<T>::turn(pirc), e, sine, cos1);
      fe = in ? T(0.5) * cos1 : T(0);
      dfe = in ? T(-0.5) * sine * pirc : T(0);
    }
    const T eta = (T)sf.ang_eta[s];
    if (eta != cur_eta) {
      cur_eta = eta;
      E = Math<T>::ex(-eta * S2);
    }
    const T gE = (s_gA[s] + wab * s_gW[s]) * E;
    T P, dP;
    line_power<T>(sf, s, cth, ps, P, dP);
    const T B = gE * P;
    SA += gE * dP;
    SB += B;
    SC += eta * B;
  }
  if (cur_g >= 0) flush();
  atomicAdd(&s_T[a], (double)Ta);
  atomicAdd(&s_T[b], (double)Tb);
  const T s = Te * ie;
  const T ux = s * ex, uy = s * ey, uz = s * ez;
  atomicAdd(&s_F[3 * b], (double)ux);
  atomicAdd(&s_F[3 * b + 1], (double)uy);
  atomicAdd(&s_F[3 * b + 2], (double)uz);
  atomicAdd(&s_F[3 * a], (double)-ux);
  atomicAdd(&s_F[3 * a + 1], (double)-uy);
  atomicAdd(&s_F[3 * a + 2], (double)-uz);
}

// Doubles of the accumulators' region: T and F of W waves, or g if larger.
template <typename T, int W>
__host__ __device__ constexpr int bwd_acc_doubles(const Lds &L) {
  return 4 * W * L.KP * 8 >= L.Dp * (int)sizeof(T) ? 4 * W * L.KP : L.Dp * (int)sizeof(T) / 8;
}

// FORM: 0 the generic form; for grid tables of NZ zetas NZ, NZ + 10 or NZ + 20
// with ES = 1, 2 or 0: at most 4 ES etas, whose g stays in registers
// (ang_bwd_grid), or any number, read from LDS records (bwd_sets).
constexpr int bwd_form(int nz, int es) { return nz == 0 ? 0 : nz + (es == 1 ? 0 : es == 2 ? 10 : 20); }
constexpr int form_sets(int form) { return form == 0 || form >= 20 ? 0 : form >= 10 ? 2 : 1; }
//
// LDS bounds the workgroups in flight (96 bytes per neighbour in FP64, 64 in
// FP32, beside it), so g shares its place with the accumulators, which start
// once it has gone into registers and records.
//
// Measured, one wave per atom: 67,647 atoms of 45 to 95 neighbours (D = 128,
// four etas) FP64 1710 -> 1280 us, mixed 781 -> 673 us; 4096 atoms FP64 152 ->
// 118 us, mixed 78 -> 64 us; 32,768 atoms of 91 neighbours (D = 256, eight
// etas) mixed 944 -> 794 us.  Of the mixed 694 us before the shared place the
// triplets took about 455 (their instructions issue for about 400 of them), the
// radial lines 85, the neighbours' tables 72, the contraction's finish 61.
//
// The bound of two waves per SIMD (256 registers) keeps the matrix results in
// ordinary vector registers; without it they would be copied from the
// accumulation registers, 16 more instructions per triplet.
template <typename T, int W, int FORM, bool Z16, bool FG>
__global__ __launch_bounds__(W > 4 ? 64 * W : 256, 2) void k_desc_bwd(int N, const int *__restrict__ species,
                                                  const double *__restrict__ wz, NeighborBufs nb, TripletBufs tb,
                                                  SFDev sf, Lds L, GradSrc gs, double *__restrict__ slot_f,
                                                  double *__restrict__ atom_vir) {
  constexpr int GNZ = FORM % 10, ES = form_sets(FORM);
  extern __shared__ __align__(16) unsigned char smem[];
  if ((int)blockIdx.x >= N) return;  // one workgroup per atom of [atom0, atom0 + N)
  const int i = L.atom0 + blockIdx.x;
  const int tid = threadIdx.x, wv = wave_index(), lane = tid & 63;
  const int KP = L.KP, Dp = L.Dp, G = L.G;
  // per-wave accumulators in FP64 for both precisions (LDS FP64 atomics are
  // also the faster ones here), summed in wave order at the end: deterministic
  double *s_vir = (double *)smem;  // [W * 6]
  double *s_T = s_vir + 6 * W;     // [W][KP]
  double *s_F = s_T + W * KP;      // [W][3 KP]
  T *s_g = (T *)s_T;               // [Dp] g, until the accumulators start
  T *s_d = (T *)(s_T + bwd_acc_doubles<T, W>(L));
  T *s_rw = s_d + 4 * KP;    // [KP] pairs (1 / r, species weight)
  // [G][KP] pairs (fc, dfc/dr) per cutoff group, in LDS or (FG) in the
  // atom's row of the global buffer
  T *s_fd = FG ? (T *)nb.fc_scratch + (size_t)i * 2 * G * KP : s_rw + 2 * KP;
  // radial lines: records (g plain, g weighted, exp coefficient, rs)
  T *s_rr = FG ? s_rw + 2 * KP : s_fd + 2 * G * KP;
  // generic form: per angular line, g of the plain and of the weighted feature
  T *s_gA = s_rr + 4 * sf.n_rad;
  T *s_gW = s_gA + sf.n_ang;
  // grid form without registers (ES = 0): one record per eta, [g plain (2 NZ) |
  // g weighted (2 NZ) | eta | exp coefficient | pad], so that a pass reads its
  // eta's values from one base address; 16-byte aligned records (every region
  // above has a multiple of 4 values).  An eta's record has at most 8 NZ values
  // for its 2 NZ lines, so the radial and the angular regions together hold
  // at most 4 (n_rad + n_ang) <= 2 Dp values.
  constexpr int RS = EtaRec<GNZ>::RS;
  static_assert(GNZ == 0 || RS == 4 * (GNZ + 1), "the record length in bwd_tables");
  static_assert(RS <= 8 * GNZ, "radial and eta records within 2 Dp values");
  T *s_er = s_gA;

  const int start = i * nb.kcap;
  const int K = nb.nb_count[i];
  if (K > KP) {
    if (tid == 0) atomicAdd(&nb.total[3], 1);
    return;
  }
  stage_neighbours<T, true>(nb, wz, species, sf, start, K, KP, s_d, s_rw, s_fd, tid, 64 * W);
  if (GNZ > 0 && ES == 0)
    for (int h = tid; h < sf.n_eta; h += 64 * W) {
      s_er[h * RS + 4 * GNZ] = (T)sf.ang_eta[h * 2 * GNZ];
      s_er[h * RS + 4 * GNZ + 1] = eta_coef<T>((T)sf.ang_eta[h * 2 * GNZ]);
    }
  const size_t row = (size_t)i * Dp;
  if (gs.splits > 0) {
    // the contraction's finish for this atom (same order as k_gpr_finish)
    const double E = split_sum(gs.splits, [&](int sp) { return gs.Epart[(size_t)sp * gs.Np + i]; });
    if (tid == 0) gs.eatom[i] = E;
    // two features per thread: Dp is a multiple of 32, rows are 16-byte aligned
    for (int d = 2 * tid; d < Dp; d += 128 * W) {
      double G0, G1;
      const size_t at = (size_t)i * Dp + d, step = (size_t)gs.Np * Dp;
      if (gs.Gpart) {
        auto part = [&](int sp) { return *(const double2 *)(gs.Gpart + sp * step + at); };
        split_sum2(gs.splits, part, G0, G1);
      } else {
        auto part = [&](int sp) { return *(const float2 *)(gs.Gpart32 + sp * step + at); };
        split_sum2(gs.splits, part, G0, G1);
      }
      double x0, x1;
      if (gs.xt64) {
        const double2 x = *(const double2 *)(gs.xt64 + at);
        x0 = x.x, x1 = x.y;
      } else {
        const float2 x = *(const float2 *)(gs.xt32 + at);
        x0 = (double)x.x, x1 = (double)x.y;
      }
      const double2 ti = *(const double2 *)(gs.theta_inv + d);
      const double g0 = -(x0 * E - G0) * ti.x, g1 = -(x1 * E - G1) * ti.y;
      // Scalar stores, which the compiler joins: a vector type's store may alias
      // any table, and the line loops would then read the int tables with vector
      // loads and wait for them (two cutoffs, 16 angular lines, 4096 atoms of 221
      // neighbours: the backward 5104 -> 4574 us in FP64, 2079 -> 1871 mixed).
      if (gs.g64_out) {
        gs.g64_out[at] = g0;
        gs.g64_out[at + 1] = g1;
        s_g[d] = (T)g0;
        s_g[d + 1] = (T)g1;
      } else {
        const float f0 = (float)g0, f1 = (float)g1;
        gs.g32_out[at] = f0;
        gs.g32_out[at + 1] = f1;
        s_g[d] = (T)f0;
        s_g[d + 1] = (T)f1;
      }
    }
  } else {
    for (int d = tid; d < Dp; d += 64 * W) s_g[d] = gs.g64 ? (T)gs.g64[row + d] : (T)gs.g32[row + d];
  }
  __syncthreads();
  for (int s = tid; s < sf.n_rad; s += 64 * W) {
    const int f = sf.rad_feat[s];
    s_rr[4 * s] = s_g[f];
    s_rr[4 * s + 1] = s_g[f + sf.nsf];
    s_rr[4 * s + 2] = eta_coef<T>(rad_table<T>(sf.rad_a, sf.rad_a32, s));
    s_rr[4 * s + 3] = rad_table<T>(sf.rad_rs, sf.rad_rs32, s);
  }
  for (int s = tid; s < (ES > 0 ? 0 : sf.n_ang); s += 64 * W) {
    const int f = sf.ang_feat[s];
    if constexpr (GNZ > 0) {
      const int h = s / (2 * GNZ), k = s - h * 2 * GNZ;
      s_er[h * RS + k] = s_g[f];
      s_er[h * RS + 2 * GNZ + k] = s_g[f + sf.nsf];
    } else {
      s_gA[s] = s_g[f];
      s_gW[s] = s_g[f + sf.nsf];
    }
  }
  // registers of the grid form: g over the lanes, the etas and their
  // exponential coefficients (uniform; 0 past the last eta)
  EtaRegs<T, ES> er;
  T ceta[4 * ES + 1], eta[4 * ES + 1];
  if constexpr (ES > 0) {
#pragma unroll
    for (int h = 0; h < 4 * ES; ++h) {
      eta[h] = h < sf.n_eta ? (T)sf.ang_eta[h * 2 * GNZ] : T(0);
      ceta[h] = eta_coef<T>(eta[h]);
    }
    if constexpr (sizeof(T) == 4) {
#pragma unroll
      for (int u = 0; u < ES; ++u) er.set[u] = load_eta_set<GNZ>(sf, s_g, u, lane);
    } else {
#pragma unroll
      for (int h = 0; h < 4; ++h) {
        const int z = lane & 15;
        const bool live = h < sf.n_eta && z < 2 * GNZ;
        const int f = live ? sf.ang_feat[h * 2 * GNZ + z] : 0;
        er.ga[h] = live ? s_g[f] : 0.0;
        er.gw[h] = live ? s_g[f + sf.nsf] : 0.0;
      }
    }
  }
  __syncthreads();  // g is consumed: its place becomes the accumulators
  // this wave's vector accumulators (its s_T row is written by the radial part)
  for (int k = lane; k < 3 * K; k += 64) s_F[3 * wv * KP + k] = 0.0;

  // radial: the lines split over the waves, 64 neighbours at a time; the last
  // R < 64 of a longer list (half of the atoms of a usual cell have one) take
  // 2^lg lanes per neighbour, each with a share of the lines
  typedef typename Pair<T>::type P2;
  for (int a0 = 0; a0 < K; a0 += 64) {
    const int R = K - a0;
    const int lg = R > 32 ? 0 : R > 16 ? 1 : R > 8 ? 2 : R > 4 ? 3 : 4;
    const int part = lane & ((1 << lg) - 1), a = min(a0 + (lane >> lg), K - 1);
    const T r = s_d[4 * a + 3], w = s_rw[2 * a + 1];
    T acc = 0;
    int g = sf.rad_g;  // the cutoff group of every radial line, or -1
    P2 f = ((const P2 *)s_fd)[max(g, 0) * KP + a];  // (fc, dfc)
    for (int s = (wv << lg) + part; s < sf.n_rad; s += W << lg) {
      const Quad<T> q = ((const Quad<T> *)s_rr)[s];  // g, g weighted, c, rs
      if (sf.rad_g < 0 && sf.rad_group[s] != g) {
        g = sf.rad_group[s];
        f = ((const P2 *)s_fd)[g * KP + a];
      }
      // d/dr [exp(-A (r - rs)^2) fc], with c = -A log2(e) in FP32
      const T dr = r - q.v[3], x = q.v[2] * dr;
      acc += (q.v[0] + w * q.v[1]) * (exp_coef(x, dr) * (x * (slope_factor<T>() * f.x) + f.y));
    }
    for (int o = 1; o < 1 << lg; o <<= 1) acc += __shfl_xor(acc, o, 64);
    if (part == 0 && a0 + (lane >> lg) < K) s_T[wv * KP + a] = (double)acc;
  }
  __syncthreads();

  if (sf.n_ang > 0) {
    const TripletList tl(tb, i);
    const int nt = tb.count[i];
    const T rcA = (T)sf.group_rc[sf.g_ang], pirc = (T)sf.group_pirc[sf.g_ang];
    constexpr int ST = 64 * W;
    uint32_t qc[4], qn[4];
    load_q4(tl, nt, 64 * wv + lane, ST, qc);
    for (int t0 = 64 * wv; t0 < nt; t0 += 4 * ST) {
      load_q4(tl, nt, t0 + 4 * ST + lane, ST, qn);
#pragma unroll 1
      for (int u = 0; u < 4; ++u) {
        if (t0 + u * ST >= nt) break;
        const bool act = t0 + u * ST + lane < nt;
        const uint32_t q = pop_q4(qc);
        if constexpr (GNZ > 0)
          ang_bwd_grid<T, GNZ, Z16, ES>(tl, q, act, sf, s_d, s_rw, s_fd, s_er, er, ceta, eta, KP, rcA, pirc,
                                        s_T + wv * KP, s_F + 3 * wv * KP);
        else
          ang_bwd_term<T>(tl, q, act, sf, s_d, s_rw, s_fd, s_gA, s_gW, KP, s_T + wv * KP, s_F + 3 * wv * KP);
      }
#pragma unroll
      for (int u = 0; u < 4; ++u) qc[u] = qn[u];
    }
  }
  __syncthreads();

  // per-slot force contributions dE_i/dR(slot atom) and the virial: the
  // radial part T d d^T / r plus F_slot d^T for the r_jk forces (each triplet's
  // u (r_k - r_j)^T is u r_k^T - u r_j^T, so summing F_slot d^T over the slots
  // gives the triplet sum with one product per slot instead of per triplet)
  double vir[6] = {0, 0, 0, 0, 0, 0};
  for (int a = tid; a < K; a += 64 * W) {
    const T r = s_d[4 * a + 3];
    double Ts = 0.0, Fx = 0.0, Fy = 0.0, Fz = 0.0;
#pragma unroll
    for (int w = 0; w < W; ++w) {
      Ts += s_T[w * KP + a];
      Fx += s_F[3 * (w * KP + a)];
      Fy += s_F[3 * (w * KP + a) + 1];
      Fz += s_F[3 * (w * KP + a) + 2];
    }
    const double sc = Ts / (double)r;
    const double dx = s_d[4 * a], dy = s_d[4 * a + 1], dz = s_d[4 * a + 2];
    if constexpr (sizeof(T) == 4) {
      // the FP32 kernels (mixed runs) store the slot forces in FP32: half the
      // bytes written here and read by the force gather
      float *o = (float *)slot_f + 3 * (size_t)(start + a);
      o[0] = (float)(sc * dx + Fx);
      o[1] = (float)(sc * dy + Fy);
      o[2] = (float)(sc * dz + Fz);
    } else {
      double *o = slot_f + 3 * (size_t)(start + a);
      o[0] = sc * dx + Fx;
      o[1] = sc * dy + Fy;
      o[2] = sc * dz + Fz;
    }
    vir[0] += sc * dx * dx + Fx * dx;
    vir[1] += sc * dy * dy + Fy * dy;
    vir[2] += sc * dz * dz + Fz * dz;
    vir[3] += sc * dx * dy + Fx * dy;
    vir[4] += sc * dy * dz + Fy * dz;
    vir[5] += sc * dx * dz + Fx * dz;
  }
  const double vt = wave_totals<double, 6>(vir, lane);
  if (lane < 6) s_vir[6 * wv + lane] = vt;
  __syncthreads();
  if (tid < 6) {
    double v = 0.0;
#pragma unroll
    for (int w = 0; w < W; ++w) v += s_vir[6 * w + tid];
    atom_vir[6 * (size_t)i + tid] = v;
  }
}

// LDS bytes of each kernel's layout; FG: the cutoff tables in global memory.
template <typename T, int NCH, int W, bool FG>
size_t fwd_lds(const Lds &L) {
  return ((W + 1) & ~1) * sizeof(double) +
         (size_t)(6 * L.KP + (FG ? 0 : L.G * L.KP) + L.Dp + W * 2 * NCH) * sizeof(T);
}

// tables: values of the backward's line tables (bwd_tables).
template <typename T, int W, bool FG>
size_t bwd_lds(const Lds &L, int tables) {
  return (6 * W + (size_t)bwd_acc_doubles<T, W>(L)) * sizeof(double) +
         (size_t)(6 * L.KP + (FG ? 0 : 2 * L.G * L.KP) + tables) * sizeof(T);
}

// The layout that sets the longest accepted list: every other one is smaller.
template <typename T>
size_t list_limit_lds(const Lds &L) {
  return (6 + 4 * (size_t)L.KP) * sizeof(double) + (size_t)(6 * L.KP + 3 * L.Dp) * sizeof(T);
}

template <typename T, int NZ, int W, bool FG>
size_t fwd_grid_lds(const Lds &L) {
  constexpr int NV = GridShape<T, NZ>::NV;
  return ((W + 1) & ~1) * sizeof(double) +
         (size_t)(6 * L.KP + (FG ? 0 : L.G * L.KP) + L.Dp + W * NV + NV) * sizeof(T);
}

// Layouts with several wavefronts per atom stay within 64 KB, so that several
// workgroups share a CU.  A one-wave layout may take the device's whole
// per-workgroup LDS (160 KB on gfx950) for long neighbour lists; past that the
// cutoff tables move to global memory (FG).
constexpr size_t kLdsBudget = 64 * 1024;

// Per-workgroup LDS limit of the current device, queried once per device.
size_t lds_limit() {
  static std::atomic<long long> cache[64] = {};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return kLdsBudget;
  long long v = cache[dev].load(std::memory_order_relaxed);
  if (v == 0) {
    int b = 0;
    if (hipDeviceGetAttribute(&b, hipDeviceAttributeMaxSharedMemoryPerBlock, dev) != hipSuccess ||
        b < (int)kLdsBudget)
      b = (int)kLdsBudget;
    v = b;
    cache[dev].store(v, std::memory_order_relaxed);
  }
  return (size_t)v;
}

// A kernel launched with more than 64 KB of dynamic LDS is first allowed the
// device's limit (once per kernel and device, outside any stream capture:
// the eager run that precedes a capture makes the same launches).
hipError_t allow_lds(const void *kernel, size_t bytes) {
  if (bytes <= kLdsBudget) return hipSuccess;
  static std::mutex mu;
  static std::set<std::pair<int, const void *>> done;
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  std::lock_guard<std::mutex> lk(mu);
  if (done.count({dev, kernel})) return hipSuccess;
  e = hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_limit());
  if (e == hipSuccess) done.insert({dev, kernel});
  return e;
}

// Launch shape of a descriptor kernel: the most wavefronts per atom (up to
// `waves`, at most `wmax`) whose layout fits 64 KB, else one wavefront within
// the device's limit, else one wavefront with the cutoff tables in global
// memory.  bytes(W, fg) is the layout's LDS size.  False if nothing fits
// (the host caps the list length so that the last form always does).
template <typename F>
bool pick_shape(int waves, int wmax, F bytes, int &W, bool &fg) {
  fg = false;
  for (int w = 8; w >= 2; w /= 2)
    if (w <= wmax && waves >= w && bytes(w, false) <= kLdsBudget) {
      W = w;
      return true;
    }
  W = 1;
  if (bytes(1, false) <= lds_limit()) return true;
  fg = true;
  return bytes(1, true) <= lds_limit();
}

template <typename T, int NCH, int W, bool FG>
hipError_t fwd_launch(hipStream_t s, int N, const int *species, const double *wz, const NeighborBufs &nb,
                      const TripletBufs &tb, const SFDev &sf, Lds L, const double *theta_inv, const double *mu,
                      int split_mode, DescOut out) {
  const size_t lds = fwd_lds<T, NCH, W, FG>(L);
  const hipError_t e = allow_lds((const void *)k_desc_fwd<T, NCH, W, FG>, lds);
  if (e != hipSuccess) return e;
  k_desc_fwd<T, NCH, W, FG><<<N, 64 * W, lds, s>>>(N, species, wz, nb, tb, sf, L, theta_inv, mu, split_mode, out);
  return hipGetLastError();
}

template <typename T, int NCH>
hipError_t fwd_waves(int waves, hipStream_t s, int N, const int *species, const double *wz, const NeighborBufs &nb,
                     const TripletBufs &tb, const SFDev &sf, Lds L, const double *theta_inv, const double *mu,
                     int split_mode, DescOut out) {
  int W;
  bool fg;
  auto bytes = [&](int w, bool g) {
    if (w == 8) return fwd_lds<T, NCH, 8, false>(L);
    if (w == 4) return fwd_lds<T, NCH, 4, false>(L);
    if (w == 2) return fwd_lds<T, NCH, 2, false>(L);
    return g ? fwd_lds<T, NCH, 1, true>(L) : fwd_lds<T, NCH, 1, false>(L);
  };
  if (!pick_shape(waves, 8, bytes, W, fg) || (fg && !nb.fc_scratch)) return hipErrorInvalidValue;
  if (fg) return fwd_launch<T, NCH, 1, true>(s, N, species, wz, nb, tb, sf, L, theta_inv, mu, split_mode, out);
  if (W == 1) return fwd_launch<T, NCH, 1, false>(s, N, species, wz, nb, tb, sf, L, theta_inv, mu, split_mode, out);
  if (W == 2) return fwd_launch<T, NCH, 2, false>(s, N, species, wz, nb, tb, sf, L, theta_inv, mu, split_mode, out);
  if (W == 8) return fwd_launch<T, NCH, 8, false>(s, N, species, wz, nb, tb, sf, L, theta_inv, mu, split_mode, out);
  return fwd_launch<T, NCH, 4, false>(s, N, species, wz, nb, tb, sf, L, theta_inv, mu, split_mode, out);
}

// zeta list {1, 2, 4, 16}: the grid kernels' specialisation with a compile-time chain
bool zeta_1_2_4_16(const SFDev &sf) {
  return sf.nz == 4 && sf.zlog[0] == 0 && sf.zlog[1] == 1 && sf.zlog[2] == 2 && sf.zlog[3] == 4;
}

// Sets of four etas whose g the backward of this table keeps in registers; 0:
// from LDS records.  In FP32 three quarters or half of a set's matrix products
// are zeros for one and two etas, and where long lists leave one wave per SIMD
// nothing hides their time.  Registers and records there, us, one wave per atom:
// one eta of four zetas 12,000 atoms of 63 neighbours 121 112, of 181 864 689;
// of three 113 109, 778 696; of one 102 104, 626 620; two etas of four zetas 121
// 121, 865 773 and 4096 atoms of 436 2396 2081; of five 130 133, 912 868 (but
// 30,000 of 63 292 306), of three 114 117, 769 761, of two 111 114, 706 729, of
// one 104 109, 632 659.
template <typename T>
int bwd_sets(const SFDev &sf) {
  if (!sf.grid) return 0;
  if (sizeof(T) == 8) return sf.n_eta <= 4 ? 1 : 0;
  if (sf.n_eta == 1 || (sf.n_eta == 2 && sf.nz == 4)) return 0;
  return sf.n_eta <= 4 ? 1 : sf.n_eta <= 8 ? 2 : 0;
}

// Values of its line tables in LDS: radial records, then eta records or the
// generic form's g (at most 2 Dp, see k_desc_bwd).
template <typename T>
int bwd_tables(const SFDev &sf) {
  return 4 * sf.n_rad + (!sf.grid ? 2 * sf.n_ang : bwd_sets<T>(sf) > 0 ? 0 : sf.n_eta * 4 * (sf.nz + 1));
}

template <typename T, int W, int GNZ, bool Z16, bool FG, int ES>
hipError_t bwd_launch_as(hipStream_t s, int N, const int *species, const double *wz, const NeighborBufs &nb,
                      const TripletBufs &tb, const SFDev &sf, Lds L, const GradSrc &gs, double *slot_f,
                      double *atom_vir) {
  const size_t lds = bwd_lds<T, W, FG>(L, bwd_tables<T>(sf));
  const hipError_t e = allow_lds((const void *)k_desc_bwd<T, W, bwd_form(GNZ, ES), Z16, FG>, lds);
  if (e != hipSuccess) return e;
  k_desc_bwd<T, W, bwd_form(GNZ, ES), Z16, FG><<<N, 64 * W, lds, s>>>(N, species, wz, nb, tb, sf, L, gs, slot_f, atom_vir);
  return hipGetLastError();
}

template <typename T, int W, int GNZ, bool Z16, bool FG>
hipError_t bwd_launch(hipStream_t s, int N, const int *species, const double *wz, const NeighborBufs &nb,
                      const TripletBufs &tb, const SFDev &sf, Lds L, const GradSrc &gs, double *slot_f,
                      double *atom_vir) {
  if constexpr (GNZ > 0) {
    const int sets = bwd_sets<T>(sf);
    if (sets == 1) return bwd_launch_as<T, W, GNZ, Z16, FG, 1>(s, N, species, wz, nb, tb, sf, L, gs, slot_f, atom_vir);
    if constexpr (sizeof(T) == 4)
      if (sets == 2) return bwd_launch_as<T, W, GNZ, Z16, FG, 2>(s, N, species, wz, nb, tb, sf, L, gs, slot_f, atom_vir);
  }
  return bwd_launch_as<T, W, GNZ, Z16, FG, 0>(s, N, species, wz, nb, tb, sf, L, gs, slot_f, atom_vir);
}

template <typename T, int W, bool FG>
hipError_t bwd_grid(hipStream_t s, int N, const int *species, const double *wz, const NeighborBufs &nb,
                    const TripletBufs &tb, const SFDev &sf, Lds L, const GradSrc &gs, double *slot_f,
                    double *atom_vir) {
  if (!sf.grid) return bwd_launch<T, W, 0, false, FG>(s, N, species, wz, nb, tb, sf, L, gs, slot_f, atom_vir);
  switch (sf.nz) {
    case 1: return bwd_launch<T, W, 1, false, FG>(s, N, species, wz, nb, tb, sf, L, gs, slot_f, atom_vir);
    case 2: return bwd_launch<T, W, 2, false, FG>(s, N, species, wz, nb, tb, sf, L, gs, slot_f, atom_vir);
    case 3: return bwd_launch<T, W, 3, false, FG>(s, N, species, wz, nb, tb, sf, L, gs, slot_f, atom_vir);
    case 4:
      if (zeta_1_2_4_16(sf))
        return bwd_launch<T, W, 4, true, FG>(s, N, species, wz, nb, tb, sf, L, gs, slot_f, atom_vir);
      return bwd_launch<T, W, 4, false, FG>(s, N, species, wz, nb, tb, sf, L, gs, slot_f, atom_vir);
    default: return bwd_launch<T, W, 5, false, FG>(s, N, species, wz, nb, tb, sf, L, gs, slot_f, atom_vir);
  }
}

template <typename T, int NZ, int W, bool Z16, bool FG>
hipError_t fwd_grid_launch(hipStream_t s, int N, const int *species, const double *wz, const NeighborBufs &nb,
                           const TripletBufs &tb, const SFDev &sf, Lds L, const double *theta_inv, const double *mu,
                           int split_mode, DescOut out) {
  const size_t lds = fwd_grid_lds<T, NZ, W, FG>(L);
  const hipError_t e = allow_lds((const void *)k_desc_fwd_grid<T, NZ, W, Z16, FG>, lds);
  if (e != hipSuccess) return e;
  k_desc_fwd_grid<T, NZ, W, Z16, FG><<<N, 64 * W, lds, s>>>(N, species, wz, nb, tb, sf, L, theta_inv, mu,
                                                            split_mode, out);
  return hipGetLastError();
}

template <typename T, int NZ, bool Z>
hipError_t fwd_grid_nz(int waves, hipStream_t s, int N, const int *species, const double *wz, const NeighborBufs &nb,
                       const TripletBufs &tb, const SFDev &sf, Lds L, const double *theta_inv, const double *mu,
                       int split_mode, DescOut out) {
  int W;
  bool fg;
  auto bytes = [&](int w, bool g) {
    if (w == 8) return fwd_grid_lds<T, NZ, 8, false>(L);
    if (w == 4) return (size_t)-1;  // one, two or eight waves
    if (w == 2) return fwd_grid_lds<T, NZ, 2, false>(L);
    return g ? fwd_grid_lds<T, NZ, 1, true>(L) : fwd_grid_lds<T, NZ, 1, false>(L);
  };
  if (!pick_shape(waves, 8, bytes, W, fg) || (fg && !nb.fc_scratch)) return hipErrorInvalidValue;
  if (fg) return fwd_grid_launch<T, NZ, 1, Z, true>(s, N, species, wz, nb, tb, sf, L, theta_inv, mu, split_mode, out);
  if (W == 8)
    return fwd_grid_launch<T, NZ, 8, Z, false>(s, N, species, wz, nb, tb, sf, L, theta_inv, mu, split_mode, out);
  if (W == 2)
    return fwd_grid_launch<T, NZ, 2, Z, false>(s, N, species, wz, nb, tb, sf, L, theta_inv, mu, split_mode, out);
  return fwd_grid_launch<T, NZ, 1, Z, false>(s, N, species, wz, nb, tb, sf, L, theta_inv, mu, split_mode, out);
}

template <typename T>
hipError_t fwd_grid(int waves, hipStream_t s, int N, const int *species, const double *wz, const NeighborBufs &nb,
                    const TripletBufs &tb, const SFDev &sf, Lds L, const double *theta_inv, const double *mu,
                    int split_mode, DescOut out) {
  switch (sf.nz) {
    case 1: return fwd_grid_nz<T, 1, false>(waves, s, N, species, wz, nb, tb, sf, L, theta_inv, mu, split_mode, out);
    case 2: return fwd_grid_nz<T, 2, false>(waves, s, N, species, wz, nb, tb, sf, L, theta_inv, mu, split_mode, out);
    case 3: return fwd_grid_nz<T, 3, false>(waves, s, N, species, wz, nb, tb, sf, L, theta_inv, mu, split_mode, out);
    case 4:
      if (zeta_1_2_4_16(sf))
        return fwd_grid_nz<T, 4, true>(waves, s, N, species, wz, nb, tb, sf, L, theta_inv, mu, split_mode, out);
      return fwd_grid_nz<T, 4, false>(waves, s, N, species, wz, nb, tb, sf, L, theta_inv, mu, split_mode, out);
    default: return fwd_grid_nz<T, 5, false>(waves, s, N, species, wz, nb, tb, sf, L, theta_inv, mu, split_mode, out);
  }
}

// Whether some descriptor kernel of this table needs its cutoff tables in
// global memory at KP slots (its one-wave LDS layout exceeds the device's limit).
template <typename T>
bool needs_global_tables(const SFDev &sf, const Lds &L) {
  const size_t lim = lds_limit();
  if (bwd_lds<T, 1, false>(L, bwd_tables<T>(sf)) > lim) return true;
  if (!sf.grid) return fwd_lds<T, 16, 1, false>(L) > lim;
  return fwd_grid_lds<T, 5, 1, false>(L) > lim;  // the widest grid layout
}

// Whether every descriptor kernel of this table has a layout for KP slots.
template <typename T>
bool fits(const SFDev &sf, const Lds &L) {
  const size_t lim = lds_limit();
  if (list_limit_lds<T>(L) > lim) return false;
  if (!sf.grid) return fwd_lds<T, 16, 1, true>(L) <= lim;
  return fwd_grid_lds<T, 5, 1, true>(L) <= lim;
}

template <typename T>
hipError_t bwd_fit(int waves, hipStream_t s, int N, const int *species, const double *wz, const NeighborBufs &nb,
                   const TripletBufs &tb, const SFDev &sf, Lds L, const GradSrc &gs, double *slot_f,
                   double *atom_vir) {
  int W;
  bool fg;
  auto bytes = [&](int w, bool g) {
    const int tables = bwd_tables<T>(sf);
    if (w == 8) return bwd_lds<T, 8, false>(L, tables);
    if (w == 4) return bwd_lds<T, 4, false>(L, tables);
    if (w == 2) return bwd_lds<T, 2, false>(L, tables);
    return g ? bwd_lds<T, 1, true>(L, tables) : bwd_lds<T, 1, false>(L, tables);
  };
  if (!pick_shape(waves, 8, bytes, W, fg) || (fg && !nb.fc_scratch)) return hipErrorInvalidValue;
  if (fg) return bwd_grid<T, 1, true>(s, N, species, wz, nb, tb, sf, L, gs, slot_f, atom_vir);
  if (W == 8) return bwd_grid<T, 8, false>(s, N, species, wz, nb, tb, sf, L, gs, slot_f, atom_vir);
  if (W == 4) return bwd_grid<T, 4, false>(s, N, species, wz, nb, tb, sf, L, gs, slot_f, atom_vir);
  if (W == 2) return bwd_grid<T, 2, false>(s, N, species, wz, nb, tb, sf, L, gs, slot_f, atom_vir);
  return bwd_grid<T, 1, false>(s, N, species, wz, nb, tb, sf, L, gs, slot_f, atom_vir);
}

}  // namespace

// Largest per-atom neighbour count the descriptor kernels take (every
// kernel of the table then has a layout within the device's LDS limit, with
// the cutoff tables in global memory where needed), capped at kMaxNeighbors.
int max_neighbors_for_lds(bool fp64, const SFDev &sf, int Dp) {
  const int G = sf.n_groups > 0 ? sf.n_groups : 1;
  int kp = kMaxNeighbors;
  for (; kp > 8; kp -= 8) {
    const Lds L{kp, G, Dp, 0, sf.n_rad};
    if (fp64 ? fits<double>(sf, L) : fits<float>(sf, L)) break;
  }
  return kp;
}

// A long list is worth several waves per atom whenever one each leaves a CU with
// fewer waves than hide their latencies: about 8 in FP64, 16 in FP32.  How many
// it has follows from the LDS (places) and from how N atoms fill the rounds.
// One, two and four waves, us (places): FP64, 181 neighbours of seven cutoffs
// (5) 4096 atoms 3860 2259 2311, 8000 7037 4460 4573; of one (10) 1500 463 456
// 385, 3000 852 697 743, 4096 830 962 956, 8000 1681 1750 1868.  FP32, seven (11)
// 4096 1433 1015 859; one (21) 1500 377 239 211, 3000 415 404 355, 4096 430 489
// 440, 8000 820 829 833.  Lists of 95 stay with the waves their number asks for
// (one cutoff, 3000 atoms: FP64 279 257 328, FP32 136 143 150).
int default_waves_fwd(bool fp64, const SFDev &sf, int Dp, int KP, int N) {
  const int waves = waves_within(N, fwd_wave_cap(fp64), 1);
  if (sf.grid || KP < 192 || N <= 0) return waves;
  const Lds L{KP, sf.n_groups > 0 ? sf.n_groups : 1, Dp, 0, sf.n_rad};
  const size_t bytes = fp64 ? fwd_lds<double, 16, 1, false>(L) : fwd_lds<float, 16, 1, false>(L);
  const double places = (double)std::max<size_t>(1, lds_limit() / bytes), atoms = N / 256.0;
  const double in_flight = atoms / std::ceil(atoms / places);
  return in_flight < (fp64 ? 7.5 : 15.0) ? std::max(waves, 4) : waves;
}

size_t desc_table_scratch_bytes(bool fp64, const SFDev &sf, int Dp, int KP, int N) {
  const int G = sf.n_groups > 0 ? sf.n_groups : 1;
  const Lds L{KP, G, Dp, 0, sf.n_rad};
  if (!(fp64 ? needs_global_tables<double>(sf, L) : needs_global_tables<float>(sf, L))) return 0;
  return (size_t)N * 2 * G * KP * (fp64 ? sizeof(double) : sizeof(float));
}

hipError_t launch_descriptors_fwd(hipStream_t s, bool fp64, int N, const int *species, const double *wz,
                                  const NeighborBufs &nb, const TripletBufs &tb, const SFDev &sf,
                                  const double *theta_inv, const double *mu, int split_mode, DescOut out, int chunk,
                                  int waves, int KP, int atom0) {
  Lds L{KP, sf.n_groups > 0 ? sf.n_groups : 1, out.Dp, atom0, sf.n_rad};
  if (N <= 0) return hipSuccess;
  if (sf.grid) {
    if (fp64) return fwd_grid<double>(waves, s, N, species, wz, nb, tb, sf, L, theta_inv, mu, split_mode, out);
    return fwd_grid<float>(waves, s, N, species, wz, nb, tb, sf, L, theta_inv, mu, split_mode, out);
  }
  if (fp64) {
    if (chunk <= 8) return fwd_waves<double, 8>(waves, s, N, species, wz, nb, tb, sf, L, theta_inv, mu, split_mode, out);
    return fwd_waves<double, 16>(waves, s, N, species, wz, nb, tb, sf, L, theta_inv, mu, split_mode, out);
  }
  if (chunk <= 8) return fwd_waves<float, 8>(waves, s, N, species, wz, nb, tb, sf, L, theta_inv, mu, split_mode, out);
  return fwd_waves<float, 16>(waves, s, N, species, wz, nb, tb, sf, L, theta_inv, mu, split_mode, out);
}

hipError_t launch_descriptors_bwd(hipStream_t s, bool fp64, int N, const int *species, const double *wz,
                                  const NeighborBufs &nb, const TripletBufs &tb, const SFDev &sf, int Dp,
                                  const GradSrc &gs, double *slot_f, double *atom_vir, int waves, int KP,
                                  int atom0) {
  Lds L{KP, sf.n_groups > 0 ? sf.n_groups : 1, Dp, atom0, sf.n_rad};
  if (N <= 0) return hipSuccess;
  // the LDS layout's 16-byte reads of g need KP (slots per atom) a multiple of 4
  if (KP % 4 != 0) return hipErrorInvalidValue;
  if (fp64) return bwd_fit<double>(waves, s, N, species, wz, nb, tb, sf, L, gs, slot_f, atom_vir);
  return bwd_fit<float>(waves, s, N, species, wz, nb, tb, sf, L, gs, slot_f, atom_vir);
}

}  // namespace gapx

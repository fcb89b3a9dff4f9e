// hg_physics.hpp -- device arithmetic of HORMONE's hydro step for gfx950.
//
// Every function keeps the reference's Fortran evaluation order (left to
// right, x**2 == x*x) so that, compiled without FMA contraction
// (-ffp-contract=off) and with IEEE division and square root, the FP64 path
// rounds exactly like the reference.  MIN/MAX/SIGN follow the reference's
// compiled semantics: max(a,b) = a>b ? a : b, min(a,b) = a<b ? a : b, n-ary
// forms fold left, sign(a,b) = copysign(|a|,b).
//
// Functions are templated on the arithmetic type R so the same code serves
// the FP64 path (R = double) and the reconstruction/Riemann part of the
// FP32-mixed path (R = float).
#pragma once

#include <hip/hip_runtime.h>

namespace hg {

template <class R> __device__ __forceinline__ R mx2(R a, R b) { return a > b ? a : b; }
template <class R> __device__ __forceinline__ R mn2(R a, R b) { return a < b ? a : b; }
template <class R> __device__ __forceinline__ R mx3(R a, R b, R c) { return mx2(mx2(a, b), c); }
template <class R> __device__ __forceinline__ R mn3(R a, R b, R c) { return mn2(mn2(a, b), c); }
__device__ __forceinline__ double sgn(double a, double b) { return copysign(fabs(a), b); }
__device__ __forceinline__ float sgn(float a, float b) { return copysignf(fabsf(a), b); }
// FP64: IEEE (correctly rounded) square root and division, as the reference.
// FP32 (mixed-precision path only): the hardware v_sqrt_f32 / v_rcp_f32
// approximations (about 1 ulp), which is what makes that path cheaper.
__device__ __forceinline__ double rsqrt_(double a) { return sqrt(a); }
__device__ __forceinline__ float rsqrt_(float a) { return __builtin_amdgcn_sqrtf(a); }
__device__ __forceinline__ double fdiv(double a, double b) { return a / b; }
__device__ __forceinline__ float fdiv(float a, float b) { return a * __builtin_amdgcn_rcpf(b); }
__device__ __forceinline__ double abs_(double a) { return fabs(a); }
__device__ __forceinline__ float abs_(float a) { return fabsf(a); }

// ---- division by a shared denominator ---------------------------------------
// FP64 (SH = true): q = a / b by the same instruction sequence as the
// compiler's IEEE division -- v_div_scale of b and of a, v_rcp_f64 of the
// scaled b refined by two Newton steps, v_div_fmas, v_div_fixup -- with the
// reciprocal of b computed once and shared by every numerator.
// v_div_scale leaves b unscaled except for operands of extreme exponent (b
// denormal or beyond 2^1022, a tiny, or a/b near the overflow or denormal
// range); then the shared reciprocal is not the one a / b would use, and
// qdiv recomputes that lane's quotient with a plain division.  Where the
// scaled b is NaN (a or b zero or NaN) v_div_fixup returns the special
// result (0, inf or NaN) without reading the reciprocal.  Every quotient is
// therefore bit-identical to a / b.
struct Den64 {
  double b, r;
};
template <class R> struct DenX {  // plain division (FP64 IEEE, FP32 approximate)
  R b;
};
template <bool SH, class R> __device__ __forceinline__ auto mkden(R b) {
  if constexpr (SH) {
    double r = __builtin_amdgcn_rcp(b);
    double e = fma(-b, r, 1.0);
    r = fma(r, e, r);
    e = fma(-b, r, 1.0);
    r = fma(r, e, r);
    return Den64{b, r};
  } else {
    return DenX<R>{b};
  }
}
__device__ __forceinline__ double qdiv(const Den64 &D, double a) {
  bool flag, vcc;
  const double sb = __builtin_amdgcn_div_scale(a, D.b, false, &flag);  // scaled b
  const double n = __builtin_amdgcn_div_scale(a, D.b, true, &vcc);    // scaled a
  const double m = n * D.r;
  const double t = fma(-D.b, m, n);
  double q = __builtin_amdgcn_div_fixup(__builtin_amdgcn_div_fmas(t, D.r, m, vcc), D.b, a);
  if (__builtin_islessgreater(sb, D.b)) {
    // rare: keep this a branch (the compiler would otherwise speculate the
    // full division on every lane and select)
    double x = a;
    asm volatile("" : "+v"(x));
    q = x / D.b;
  }
  return q;
}
template <class R> __device__ __forceinline__ R qdiv(const DenX<R> &D, R a) {
  return fdiv(a, D.b);
}

// A point no instruction is moved across: between the parts of a long straight
// block it bounds the values in flight (the tests of the fast form would be
// put off to its end, the plain form's divisions all interleaved: 30 to 70
// spilled registers).
__device__ __forceinline__ void fence() { __builtin_amdgcn_sched_barrier(0); }

enum { LIM_FLAT = 0, LIM_MINMOD = 1, LIM_MC = 2 };

// fluxlimiter.f90:40-56 (generalised minmod); dx = idx(i:i+1)
// Dab: the denominator dxa + dxb (a grid function, shared by every variable
// of the cell).
template <class R, class DN>
__device__ __forceinline__ R minmod_d(R u0, R u1, R u2, R dxa, R dxb, const DN &Dab) {
  R x = R(1.4) * (u2 - u1) * dxb;
  R y = R(1.4) * (u1 - u0) * dxa;
  R z = qdiv(Dab, (u2 - u0) * dxa * dxb);
  R s = sgn(R(1), x);
  return s * mx2(R(0), mn3(abs_(x), s * y, s * z));
}
template <class R>
__device__ __forceinline__ R minmod(R u0, R u1, R u2, R dxa, R dxb) {
  return minmod_d(u0, u1, u2, dxa, dxb, mkden<false>(dxa + dxb));
}

// fluxlimiter.f90:58-75 (modified MC).  cf, cb and the centre spacings are
// pure grid functions; they are evaluated here from the same coordinate
// operands as in the reference so they round identically.
//
// modified_mc_d takes the per-cell grid factors: dxp = xp - x0,
// cf = (xp - x0)/(xi0 - x0), cb = (x0 - xm)/(x0 - xim) and the shared
// denominators Dm = x0 - xm and Dp = xp - x0.
template <class R, class DN>
__device__ __forceinline__ R modified_mc_d(R u0, R u1, R u2, R dxp, R cf, R cb, const DN &Dm,
                                           const DN &Dp) {
  R top = qdiv(Dm, (u1 - u0) * dxp);
  R bot = u2 - u1;
  R sig = sgn(R(1), bot);
  return qdiv(Dp, sig * mx2(R(0), mn3(sig * R(0.5) * (bot + top), sig * cf * bot, sig * cb * top)));
}
template <class R>
__device__ __forceinline__ R modified_mc(R u0, R u1, R u2, R xm, R x0, R xp,
                                         R xim, R xi0) {
  R cf = fdiv(xp - x0, xi0 - x0);
  R cb = fdiv(x0 - xm, x0 - xim);
  return modified_mc_d(u0, u1, u2, xp - x0, cf, cb, mkden<false>(x0 - xm), mkden<false>(xp - x0));
}

// gamma - 1 where it is used: one value for a whole sweep was kept in a register
// pair across the solver, and spilled
__device__ __forceinline__ double gam_1(double gam) {
  asm volatile("" : "+s"(gam));
  return gam - 1.0;
}

// get_eint, eos.f90:846-865
template <class R>
__device__ __forceinline__ R get_eint(bool mag, R etot, R d, R v1, R v2, R v3, R b1,
                                      R b2, R b3) {
  R vsq = v1 * v1 + v2 * v2 + v3 * v3;
  R eint = etot - R(0.5) * d * vsq;
  if (mag) eint = eint - R(0.5) * (b1 * b1 + b2 * b2 + b3 * b3);
  return eint;
}

// get_cf, eos.f90:351-365
// get_cf_d takes the density as a shared denominator.
template <class R, class DN>
__device__ __forceinline__ R get_cf_d(const DN &Dd, R cs, R b1, R b2, R b3) {
  R asq = cs * cs;
  R bb1 = qdiv(Dd, b1 * b1);
  R bb2 = qdiv(Dd, b2 * b2);
  R bb3 = qdiv(Dd, b3 * b3);
  R bbsq = bb1 + bb2 + bb3;
  return rsqrt_(R(0.5) * (asq + bbsq + rsqrt_((asq + bbsq) * (asq + bbsq) - R(4) * asq * bb1)));
}
template <class R>
__device__ __forceinline__ R get_cf(R d, R cs, R b1, R b2, R b3) {
  return get_cf_d(mkden<false>(d), cs, b1, b2, b3);
}

// hlldflux + fstar, hlldflux.f90:19-179, without the radiation component
// (erl = err = 0 on this path; its flux only feeds irad).  f[0..8] are
// tmpflux(1..9).
template <class R>
__device__ __forceinline__ void hlld(R f[9], R cfl, R cfr, R v1l, R v1r, R v2l, R v2r,
                                     R v3l, R v3r, R dl, R dr, R el, R er, R ptl,
                                     R ptr, R b1l, R b1r, R b2l, R b2r, R b3l, R b3r,
                                     R phil, R phir, R ch) {
  const R h = R(0.5);
  R b1 = h * ((b1l + b1r) - fdiv(phir - phil, ch));
  R phi = h * ((phil + phir) - (b1r - b1l) * ch);

  R sl = mn3(v1r - cfr, v1l - cfl, R(0));
  R sr = mx3(v1r + cfr, v1l + cfl, R(0));

  R slv = sl - v1l, srv = sr - v1r;
  const auto Dden = mkden<false>(srv * dr - slv * dl);
  R sm = qdiv(Dden, srv * dr * v1r - slv * dl * v1l - ptr + ptl);
  fence();
  R pta = qdiv(Dden, srv * dr * ptl - slv * dl * ptr + dl * dr * srv * slv * (v1r - v1l));
  fence();

  R slm = sl - sm, srm = sr - sm;
  const auto Dslm = mkden<false>(slm), Dsrm = mkden<false>(srm);
  R dla = qdiv(Dslm, dl * slv);
  fence();
  R dra = qdiv(Dsrm, dr * srv);
  fence();

  R sqla = rsqrt_(dla), sqra = rsqrt_(dra);
  fence();
  R sla = sm - fdiv(abs_(b1), sqla);
  fence();
  R sra = sm + fdiv(abs_(b1), sqra);
  fence();

  R b1b1 = b1 * b1;
  const auto Dl = mkden<false>(dl * slv * slm - b1b1);
  const auto Dr = mkden<false>(dr * srv * srm - b1b1);
  R v2la = v2l - qdiv(Dl, b1 * b2l * (sm - v1l));
  fence();
  R v2ra = v2r - qdiv(Dr, b1 * b2r * (sm - v1r));
  fence();
  R v3la = v3l - qdiv(Dl, b1 * b3l * (sm - v1l));
  fence();
  R v3ra = v3r - qdiv(Dr, b1 * b3r * (sm - v1r));
  fence();

  R numl = dl * slv * slv - b1b1;
  R numr = dr * srv * srv - b1b1;
  R b2la = qdiv(Dl, b2l * numl);
  fence();
  R b2ra = qdiv(Dr, b2r * numr);
  fence();
  R b3la = qdiv(Dl, b3l * numl);
  fence();
  R b3ra = qdiv(Dr, b3r * numr);
  fence();

  R ela = qdiv(Dslm, slv * el - ptl * v1l + pta * sm +
                         b1 * ((v1l * b1 + v2l * b2l + v3l * b3l) -
                               (sm * b1 + v2la * b2la + v3la * b3la)));
  fence();
  R era = qdiv(Dsrm, srv * er - ptr * v1r + pta * sm +
                         b1 * ((v1r * b1 + v2r * b2r + v3r * b3r) -
                               (sm * b1 + v2ra * b2ra + v3ra * b3ra)));
  fence();

  R sb1 = sgn(R(1), b1);
  const auto Dsqs = mkden<false>(sqla + sqra);
  R v2aa = qdiv(Dsqs, sqla * v2la + sqra * v2ra + (b2ra - b2la) * sb1);
  fence();
  R v3aa = qdiv(Dsqs, sqla * v3la + sqra * v3ra + (b3ra - b3la) * sb1);
  fence();
  R sqp = rsqrt_(dla * dra);
  fence();
  R b2aa = qdiv(Dsqs, sqla * b2ra + sqra * b2la + sqp * (v2ra - v2la) * sb1);
  fence();
  R b3aa = qdiv(Dsqs, sqla * b3ra + sqra * b3la + sqp * (v3ra - v3la) * sb1);
  fence();

  R vbaa = v2aa * b2aa + v3aa * b3aa;
  R eraa = era + sb1 * sqra * ((v2ra * b2ra + v3ra * b3ra) - vbaa);
  R elaa = ela - sb1 * sqla * ((v2la * b2la + v3la * b3la) - vbaa);
  fence();

  R signsm = sgn(h, sm);
  R sortsla = h + sgn(h, sla);
  R sortsra = h + sgn(h, -sra);
  R sortslr = h - sgn(h, sla * sra);

  R d_ = (h + signsm) * dla + (h - signsm) * dra;
  R v2_ = sortsla * v2la + sortslr * v2aa + sortsra * v2ra;
  R v3_ = sortsla * v3la + sortslr * v3aa + sortsra * v3ra;
  fence();
  R b2_ = sortsla * b2la + sortslr * b2aa + sortsra * b2ra;
  R b3_ = sortsla * b3la + sortslr * b3aa + sortsra * b3ra;
  fence();
  R e_ = sortsla * ela + (h - sgn(h, sla * sm)) * elaa + (h + sgn(h, -sm * sra)) * eraa +
         (h - sgn(h, sra)) * era;

  // fstar, hlldflux.f90:156-179 with (d,v1,v2,v3,b1,b2,b3,e,p) =
  // (d_, sm, v2_, v3_, b1, b2_, b3_, e_, pta)
  f[0] = d_ * sm;
  f[1] = d_ * sm * sm + pta - b1 * b1;
  f[2] = d_ * sm * v2_ - b1 * b2_;
  f[3] = d_ * sm * v3_ - b1 * b3_;
  f[4] = (e_ + pta) * sm - b1 * (sm * b1 + v2_ * b2_ + v3_ * b3_);
  f[5] = phi;
  f[6] = b2_ * sm - b1 * v2_;
  f[7] = b3_ * sm - b1 * v3_;
  f[8] = ch * ch * b1;
}
// ---- checked fast arithmetic (the FP64 sweeps) --------------------------------
// The compiler's FP64 division and square root spend about half of their
// instructions on scaling operands of extreme exponent (v_div_scale,
// v_ldexp) and on special results.  The sweep runs them without: fdiv is the
// same Newton sequence on unscaled operands (4 instructions and a reciprocal
// shared by every division by that denominator), fsqrt the same coupled
// iteration.  Where nothing would have been scaled they give the same bits.
// Whether that held is recorded, not branched on: every divisor, dividend
// and radicand goes into a Chk, and a wavefront in which one was out of range
// computes its cells again with plain divisions and square roots
// (cell_slopes, face_flux).  One test per face instead of a branch per
// division leaves the compiler one straight block to schedule.  The y and z
// sweeps are bound by VALU issue (78% busy with the quarter-rate reciprocals
// counted as one), so this is their time: 1,530 -> 1,125 VALU instructions per
// wavefront (256^3 MHD polytrope), 2,075 -> 1,760 us per stage for both (shear
// layer); hydro (160^3, three directions in one launch) 594 -> 437 us.
//
// Chk: pos() takes a value that has to be positive with an exponent in
// [-256, 255], neg() a negative one, leaf() one of either sign that is zero (its
// frexp exponent is 0 then) or has an exponent of at least -600, num() (known-answer
// records) one with an exponent in [-256, 255], differ() a pair whose order
// decides.
//
// What is tested, and why it is enough.  A quotient or root without scaling is
// exact unless its dividend or radicand is below 2^-968 (an inexact residual),
// the divisor extreme, or the quotient overflows or is denormal.
// * Every cell (odd_cell): d, e and e_int in range, which leaves no NaN or
//   infinity in the velocities and fields they hold the energy of, |m| <= 2^257
//   and |b| <= 2^129; m and b leaves.  Face densities and energies, the squared
//   sound speeds, and every divisor and radicand of the solver: in range.  So
//   no divisor is extreme and no quotient overflows.
// * Leaves make the face states exact.  Differences of neighbours are 0 or at
//   least 2^-652; with the grid factors' ranges (Axis::fast) the limiters'
//   dividends are then at least 2^-870 and their quotients 2^-970, so the
//   slopes, the face momenta and fields (0 or above 2^-690) and their
//   velocities are exact, and so is sm: -ptr + ptl leaves a dividend of 0 or of
//   pt's last place (2^-567) or more.  psi has no slopes; dphi is a leaf.
// * What is left are tiny dividends made of products.  Their quotients are
//   below 2^-712 and wrong by an ulp at most.  Such a value is lost in a sum
//   with any value in range: the energies and pressures, the wave speeds (a
//   fast speed is in range), pta.  In a side's transverse star states it is
//   tested for: the velocity or the dividend taken off it is a leaf (less()),
//   and the fields' factor is 0 or has 2^-257 or more, so that their dividends
//   are 0 or above 2^-947.  The inner states are made of these, with dividends
//   of 0 or above 2^-900: exact as well, unless a star density is 2^279 times
//   below its side's (a quotient could be denormal).
// * Zeros may have the other sign: of a momentum or field of a ghost (a wall
//   makes -0 of +0), and of slopes (vmin and vmax do not order zeros).  That
//   reaches the fluxes as the sign of a zero only.  The selections are by sm
//   and the Alfven speeds; sm's zero is +0 (x - ptr + ptl), and where b1 is a
//   zero both Alfven speeds have sm's sign.  And an update shows no flux
//   divergence's zero: with the source's +0 the sum is +0.  Only gravity's
//   source may be -0, and only a momentum of -0 shows that (minus_zero).
// A wavefront that runs both forms takes 1.7 (MHD) to 2 (hydro) times as long:
// 56^3, three directions in one launch, every wavefront: 40 -> 70 us, 22 -> 44.
// With every -0 refused, that was each wavefront at a wall of gas at rest, or of
// zero normal field, or with inflow; with 2^-256 as the limit of what was tested,
// up to 70% of an MHD blast wave's (96^3, 16 steps after the start: 846 us per
// step, now 505), whose velocities fall off through that ahead of the front.
// The tests are asm volatile so that each is made where its value is computed:
// written as expressions they were gathered at the end of the block, with
// every tested value kept in registers until then (162 VGPRs against 126; 102
// with the fluxes forced before the branch, see line_faces).
struct Chk {
  unsigned n = 0, p = 0;
  bool near = false;
  __device__ __forceinline__ void num(double x) {
    unsigned t;
    asm volatile(
        "v_frexp_exp_i32_f64 %1, %2\n\tv_add_u32 %1, 0x100, %1\n\tv_or_b32 %0, %0, %1"
        : "+v"(n), "=&v"(t)
        : "v"(x));
  }
  template <int LOW = 600>
  __device__ __forceinline__ void leaf(double x) {
    unsigned t;
    asm volatile(
        "v_frexp_exp_i32_f64 %1, %2\n\tv_add_u32 %1, %3, %1\n\tv_or_b32 %0, %0, %1"
        : "+v"(p), "=&v"(t)
        : "v"(x), "i"(LOW));
  }
  // x = z - a/d: leaf() of the larger of x and a
  __device__ __forceinline__ void less(double x, double a) {
    double y;
    unsigned t;
    asm volatile(
        "v_max_f64 %2, |%3|, |%4|\n\tv_frexp_exp_i32_f64 %1, %2\n\t"
        "v_add_u32 %1, 0x258, %1\n\tv_or_b32 %0, %0, %1"
        : "+v"(p), "=&v"(t), "=&v"(y)
        : "v"(x), "v"(a));
  }
  __device__ __forceinline__ void pos(double x) { high<0xd0100000u>(__double2hiint(x)); }
  __device__ __forceinline__ void neg(double x) { high<0x50100000u>(__double2hiint(x)); }
  // d = x - y, y >= 0: false (0 - 0 apart) within 2^-48 of y
  __device__ __forceinline__ void differ(double d, double y) { near |= fabs(d) < 0x1p-48 * y; }
  __device__ __forceinline__ bool bad() const {
    return (n & ~511u) || (p & 0xe0000000u) || near;
  }

 private:
  template <unsigned MINUS>  // -(high word of the smallest value in range)
  __device__ __forceinline__ void high(int hi) {
    unsigned t;
    asm volatile("v_add_u32 %1, %3, %2\n\tv_or_b32 %0, %0, %1"
                 : "+v"(p), "=&v"(t)
                 : "v"(hi), "i"(MINUS));
  }
};

__device__ __forceinline__ Den64 fden(double b) { return mkden<true>(b); }
__device__ __forceinline__ double fdiv_(const Den64 &D, double a) {
  const double m = a * D.r;
  return __builtin_amdgcn_div_fixup(fma(fma(-D.b, m, a), D.r, m), D.b, a);
}
__device__ __forceinline__ double fsqrt(double x) {
  const double y = __builtin_amdgcn_rsq(x);
  double g = x * y, h = 0.5 * y;
  const double r = fma(-h, g, 0.5);
  g = fma(g, r, g);
  h = fma(h, r, h);
  g = fma(fma(-g, g, x), h, g);
  return fma(fma(-g, g, x), h, g);
}
// min and max of two numbers, one instruction (the reference's a < b ? a : b
// takes three; they differ for NaN, which the sweep's cells are tested for,
// and in the sign of a zero, see Chk).  fmin() would add two
// instructions that quiet signalling NaNs.
__device__ __forceinline__ double vmin(double a, double b) {
  double r;
  asm("v_min_f64 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
  return r;
}
__device__ __forceinline__ double vmax(double a, double b) {
  double r;
  asm("v_max_f64 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
  return r;
}
__device__ __forceinline__ double vmax0(double a) {
  double r;
  asm("v_max_f64 %0, %1, 0" : "=v"(r) : "v"(a));
  return r;
}
// the sign bit of x, and y with its sign flipped by such a bit: y * sgn(1, x)
// without the multiplication
__device__ __forceinline__ unsigned sbit(double x) {
  return (unsigned)__double2hiint(x) & 0x80000000u;
}
__device__ __forceinline__ double flip(double y, unsigned s) {
  return __hiloint2double((int)((unsigned)__double2hiint(y) ^ s), __double2loint(y));
}
// 0.5 + sgn(0.5, x) and 0.5 - sgn(0.5, x) as bit operations on x's high word:
// 1 or 0 by the sign bit
__device__ __forceinline__ double wpos(int hi) {
  return __hiloint2double(~(hi >> 31) & 0x3ff00000, 0);
}
__device__ __forceinline__ double wneg(int hi) {
  return __hiloint2double((hi >> 31) & 0x3ff00000, 0);
}

// Grid factors of one cell's slopes (k_geo): dxp = xp - x0, bm = x0 - xm,
// the two limiter ratios, the half widths and, for minmod, the inverse
// spacings; Dp, Dm, Dab are the denominators with their reciprocals.
struct Geo {
  Den64 Dp, Dm, Dab;
  double cf, cb, hl, hr, ida, idb;
};

// Limited slope of one variable, modified_mc / minmod with the operations
// that only move a sign taken out: sig*0.5*(bot+top) = flip(0.5*(bot+top)),
// sig*cf*bot = cf*|bot|, sig*cb*top = flip(cb*top) (rounding is symmetric).
template <int LIM>
__device__ __forceinline__ double fslope(double u0, double u1, double u2, const Geo &G) {
  if constexpr (LIM == LIM_MINMOD) {
    const double x = 1.4 * (u2 - u1) * G.idb;
    const double y = 1.4 * (u1 - u0) * G.ida;
    const unsigned s = sbit(x);
    const double z = fdiv_(G.Dab, (u2 - u0) * G.ida * G.idb);
    return flip(vmax0(vmin(vmin(fabs(x), flip(y, s)), flip(z, s))), s);
  } else {
    const double top = fdiv_(G.Dm, (u1 - u0) * G.Dp.b);
    const double bot = u2 - u1;
    const unsigned s = sbit(bot);
    const double m = vmin(vmin(flip(0.5 * (bot + top), s), G.cf * fabs(bot)), flip(G.cb * top, s));
    return fdiv_(G.Dp, flip(vmax0(m), s));
  }
}

// Both face states of a cell, after the e_int guard: FL at its left face, FR
// at its right one, of d e m1 m2 m3 (b1 b2 b3), with the density's
// reciprocal for the velocities (DL, DR).  qv, ql, qr as cell_slopes.  The
// guard's own face values are the Riemann states unless it resets the slopes
// to zero (then they are the cell's value), so nothing is evaluated twice.
//
// vmin and vmax may give a slope's zero the other sign (Chk: zeros).
template <bool MAG, int LIM>
__device__ __forceinline__ void cell_faces(const double qv[9], const double ql[9],
                                           const double qr[9], const Geo &G, double FL[8],
                                           double FR[8], Den64 &DL, Den64 &DR, Chk &k) {
  constexpr int NS = MAG ? 8 : 5;
  if constexpr (LIM == LIM_FLAT) {
#pragma unroll
    for (int s = 0; s < 8; ++s) FL[s] = FR[s] = s < NS ? qv[s] : 0.0;
    DL = DR = fden(qv[0]);
    return;
  }
#pragma unroll
  for (int s = 0; s < 8; ++s) {
    if (s >= NS) {
      FL[s] = FR[s] = 0.0;
      continue;
    }
    const double S = fslope<LIM>(ql[s], qv[s], qr[s], G);
    FL[s] = qv[s] - G.hl * S;
    FR[s] = qv[s] + G.hr * S;
    if (s % 4 == 3) fence();
  }
  fence();
  k.pos(FL[0]);
  k.pos(FR[0]);
  k.pos(FL[1]);
  k.pos(FR[1]);
  DL = fden(FL[0]);
  DR = fden(FR[0]);
  const double kl = 0.5 * (FL[2] * FL[2] + FL[3] * FL[3] + FL[4] * FL[4]);
  const double kr = 0.5 * (FR[2] * FR[2] + FR[3] * FR[3] + FR[4] * FR[4]);
  double eintl = FL[1] - fdiv_(DL, kl);
  double eintr = FR[1] - fdiv_(DR, kr);
  if (MAG) {
    eintl = eintl - 0.5 * (FL[5] * FL[5] + FL[6] * FL[6] + FL[7] * FL[7]);
    eintr = eintr - 0.5 * (FR[5] * FR[5] + FR[6] * FR[6] + FR[7] * FR[7]);
  }
  const double el_ = ql[8], em_ = qv[8], er_ = qr[8];
  if (eintl >= vmax(el_, em_) || eintl <= vmin(el_, em_) || eintr >= vmax(em_, er_) ||
      eintr <= vmin(em_, er_)) {
#pragma unroll
    for (int s = 0; s < NS; ++s) FL[s] = FR[s] = qv[s];
    DL = DR = fden(qv[0]);
  }
}

// The lowest exponent of three values, zeros (exponent 0) and those above 1 apart.
__device__ __forceinline__ int lowest(double x, double y, double z) {
  const int a = __builtin_amdgcn_frexp_exp(x), b = __builtin_amdgcn_frexp_exp(y),
            c = __builtin_amdgcn_frexp_exp(z);
  return min(min(a, b), c);
}

// A cell the fast form is not for: d, e or e_int out of range, or a momentum (the
// lowest exponent mlow) or field that is no leaf.
template <bool MAG>
__device__ __forceinline__ bool odd_cell(const double qv[9], int mlow) {
  Chk k;
  k.pos(qv[0]);
  k.pos(qv[1]);
  k.pos(qv[8]);
  return k.bad() || min(mlow, MAG ? lowest(qv[5], qv[6], qv[7]) : 0) < -600;
}

// get_cf, the checked fast form
__device__ __forceinline__ double fast_cf(const Den64 &Dd, double cs, double b1, double b2,
                                          double b3, Chk &k) {
  const double asq = cs * cs;
  const double bb1 = fdiv_(Dd, b1 * b1);
  const double bb2 = fdiv_(Dd, b2 * b2);
  const double bb3 = fdiv_(Dd, b3 * b3);
  const double s = asq + (bb1 + bb2 + bb3);
  const double r = s * s - 4.0 * asq * bb1;
  k.pos(r);
  return fsqrt(0.5 * (s + fsqrt(r)));
}

// hlldflux + fstar as hlld(), in the checked fast form.  Dch: ch with its
// reciprocal.  Hydro (MAG false): with B = 0 and psi = 0 the transverse
// states, the Alfven states and every term with b1 are the identity or a
// zero, and both Alfven speeds are sm, so only the contact's selection is
// left; what changes is the sign of a zero flux (Chk: zeros), and with exact
// face states every value selected is exact.
template <bool MAG>
__device__ __forceinline__ void hlld_fast(double f[9], double cfl, double cfr, double v1l,
                                          double v1r, double v2l, double v2r, double v3l,
                                          double v3r, double dl, double dr, double el, double er,
                                          double ptl, double ptr, double b1l, double b1r,
                                          double b2l, double b2r, double b3l, double b3r,
                                          double phil, double phir, const Den64 &Dch, Chk &k) {
  double b1 = 0.0, phi = 0.0;
  const double ch = Dch.b;
  if constexpr (MAG) {  // first: psi and the sides' normal fields are done with then
    const double dphi = phir - phil;
    k.leaf(dphi);
    b1 = 0.5 * ((b1l + b1r) - fdiv_(Dch, dphi));
    phi = 0.5 * ((phil + phir) - (b1r - b1l) * ch);
    fence();
  }
  const double sl = vmin(vmin(v1r - cfr, v1l - cfl), 0.0);
  const double sr = vmax(vmax(v1r + cfr, v1l + cfl), 0.0);
  const double slv = sl - v1l, srv = sr - v1r;
  const double den = srv * dr - slv * dl;
  k.pos(den);
  const Den64 Dden = fden(den);
  const double smn = srv * dr * v1r - slv * dl * v1l - ptr + ptl;
  const double pan = srv * dr * ptl - slv * dl * ptr + dl * dr * srv * slv * (v1r - v1l);
  const double sm = fdiv_(Dden, smn), pta = fdiv_(Dden, pan);
  const double slm = sl - sm, srm = sr - sm;
  k.neg(slm);
  k.pos(srm);
  const Den64 Dslm = fden(slm), Dsrm = fden(srm);
  const double dla = fdiv_(Dslm, dl * slv), dra = fdiv_(Dsrm, dr * srv);
  k.pos(dla);
  k.pos(dra);
  fence();
  const int hsm = __double2hiint(sm);
  if constexpr (!MAG) {
    const double ela = fdiv_(Dslm, slv * el - ptl * v1l + pta * sm);
    const double era = fdiv_(Dsrm, srv * er - ptr * v1r + pta * sm);
    const double wl = wpos(hsm), wr = wneg(hsm);
    const double d_ = wl * dla + wr * dra;
    const double v2_ = wl * v2l + wr * v2r, v3_ = wl * v3l + wr * v3r;
    f[0] = d_ * sm;
    f[1] = d_ * sm * sm + pta;
    f[2] = d_ * sm * v2_;
    f[3] = d_ * sm * v3_;
    f[4] = ((wl * ela + wr * era) + pta) * sm;
    f[5] = f[6] = f[7] = f[8] = 0.0;
    return;
  }
  const double sqla = fsqrt(dla), sqra = fsqrt(dra);
  // the Alfven speeds sm -+ |b1|/sqrt(rho) only select by their sign: that of
  // sm*sqrt(rho) -+ |b1|, unless the two nearly cancel
  const double ab1 = fabs(b1);
  const double sla = fma(sm, sqla, -ab1), sra = fma(sm, sqra, ab1);
  k.differ(sla, ab1);
  k.differ(sra, ab1);
  fence();

  const double b1b1 = b1 * b1;
  // one side after the other: a side's face values are done with then
  const double dnl = dl * slv * slm - b1b1;
  k.pos(dnl);
  const Den64 Dl = fden(dnl);
  const double a2l = b1 * b2l * (sm - v1l), a3l = b1 * b3l * (sm - v1l);
  const double v2la = v2l - fdiv_(Dl, a2l), v3la = v3l - fdiv_(Dl, a3l);
  k.less(v2la, a2l);
  k.less(v3la, a3l);
  const double numl = dl * slv * slv - b1b1;
  k.leaf<256>(numl);
  const double b2la = fdiv_(Dl, b2l * numl);
  const double b3la = fdiv_(Dl, b3l * numl);
  const double ela = fdiv_(Dslm, slv * el - ptl * v1l + pta * sm +
                                     b1 * ((v1l * b1 + v2l * b2l + v3l * b3l) -
                                           (sm * b1 + v2la * b2la + v3la * b3la)));
  fence();
  const double dnr = dr * srv * srm - b1b1;
  k.pos(dnr);
  const Den64 Dr = fden(dnr);
  const double a2r = b1 * b2r * (sm - v1r), a3r = b1 * b3r * (sm - v1r);
  const double v2ra = v2r - fdiv_(Dr, a2r), v3ra = v3r - fdiv_(Dr, a3r);
  k.less(v2ra, a2r);
  k.less(v3ra, a3r);
  const double numr = dr * srv * srv - b1b1;
  k.leaf<256>(numr);
  const double b2ra = fdiv_(Dr, b2r * numr);
  const double b3ra = fdiv_(Dr, b3r * numr);
  const double era = fdiv_(Dsrm, srv * er - ptr * v1r + pta * sm +
                                     b1 * ((v1r * b1 + v2r * b2r + v3r * b3r) -
                                           (sm * b1 + v2ra * b2ra + v3ra * b3ra)));
  fence();
  const unsigned s1 = sbit(b1);
  const Den64 Dsqs = fden(sqla + sqra);
  const double v2aa = fdiv_(Dsqs, sqla * v2la + sqra * v2ra + flip(b2ra - b2la, s1));
  const double v3aa = fdiv_(Dsqs, sqla * v3la + sqra * v3ra + flip(b3ra - b3la, s1));
  const double sqp = fsqrt(dla * dra);
  const double b2aa = fdiv_(Dsqs, sqla * b2ra + sqra * b2la + flip(sqp * (v2ra - v2la), s1));
  const double b3aa = fdiv_(Dsqs, sqla * b3ra + sqra * b3la + flip(sqp * (v3ra - v3la), s1));

  fence();
  const double vbaa = v2aa * b2aa + v3aa * b3aa;
  const double eraa = era + flip(sqra * ((v2ra * b2ra + v3ra * b3ra) - vbaa), s1);
  const double elaa = ela - flip(sqla * ((v2la * b2la + v3la * b3la) - vbaa), s1);

  const int hla = __double2hiint(sla), hra = __double2hiint(sra);
  const double wl = wpos(hla), wr = wneg(hra), wa = wneg(hla ^ hra);
  const double d_ = wpos(hsm) * dla + wneg(hsm) * dra;
  const double v2_ = wl * v2la + wa * v2aa + wr * v2ra;
  const double v3_ = wl * v3la + wa * v3aa + wr * v3ra;
  const double b2_ = wl * b2la + wa * b2aa + wr * b2ra;
  const double b3_ = wl * b3la + wa * b3aa + wr * b3ra;
  const double e_ = wl * ela + wneg(hla ^ hsm) * elaa + wneg(hsm ^ hra) * eraa + wr * era;
  f[0] = d_ * sm;
  f[1] = d_ * sm * sm + pta - b1b1;
  f[2] = d_ * sm * v2_ - b1 * b2_;
  f[3] = d_ * sm * v3_ - b1 * b3_;
  f[4] = (e_ + pta) * sm - b1 * (sm * b1 + v2_ * b2_ + v3_ * b3_);
  f[5] = phi;
  f[6] = b2_ * sm - b1 * v2_;
  f[7] = b3_ * sm - b1 * v3_;
  f[8] = ch * ch * b1;
}

// Face states to flux, as face_flux: L the left cell's FR, R_ the right
// cell's FL, Dl and Dr their densities' reciprocals.  A face density or
// internal energy that is not positive fails its test (pos), so the
// reference's stop on it is left to the plain form.
template <int DIR, bool MAG>
__device__ __forceinline__ void face_fast(const double L[8], const double R_[8], double phil,
                                          double phir, const Den64 &Dl, const Den64 &Dr,
                                          double gam, const Den64 &Dch, double t[9], Chk &k) {
  constexpr int a_ = DIR, b_ = (DIR + 1) % 3, c_ = (DIR + 2) % 3;
  struct Side {
    double v1, v2, v3, b1, b2, b3, pt, cf;
  };
  auto side = [&](const double F[8], const Den64 &Df) {
    Side o;
    o.v1 = fdiv_(Df, F[2 + a_]);
    o.v2 = fdiv_(Df, F[2 + b_]);
    o.v3 = fdiv_(Df, F[2 + c_]);
    o.b1 = MAG ? F[5 + a_] : 0.0;
    o.b2 = MAG ? F[5 + b_] : 0.0;
    o.b3 = MAG ? F[5 + c_] : 0.0;
    o.pt = gam_1(gam) * get_eint(MAG, F[1], F[0], o.v1, o.v2, o.v3, o.b1, o.b2, o.b3);
    const double as = fdiv_(Df, gam * o.pt);
    k.pos(as);
    o.cf = fsqrt(as);
    if (MAG) {
      o.pt = o.pt + 0.5 * (o.b1 * o.b1 + o.b2 * o.b2 + o.b3 * o.b3);
      o.cf = fast_cf(Df, o.cf, o.b1, o.b2, o.b3, k);
    }
    fence();  // one side after the other, for the registers
    return o;
  };
  const Side l = side(L, Dl), r = side(R_, Dr);
  // without B get_cf is sqrt(0.5*(cs^2 + sqrt(cs^4))) = cs exactly: the
  // square root of a rounded square is the number itself
  hlld_fast<MAG>(t, l.cf, r.cf, l.v1, r.v1, l.v2, r.v2, l.v3, r.v3, L[0], R_[0], L[1], R_[1],
                 l.pt, r.pt, l.b1, r.b1, l.b2, r.b2, l.b3, r.b3, phil, phir, Dch, k);
}

// ---- FP32-mixed HLLD in perturbation form ----------------------------------
// The Riemann solver of hlld() above (hlldflux.f90:19-179, same star states,
// same state selection), rearranged so that FP32 only ever carries
// differences.  Every star state is written as the left face state plus a
// correction, and the returned flux is the FP64 flux function of the left
// state (fstar with the GLM normal field b1 and the left total pressure)
// plus an FP32 correction.  In exact arithmetic this equals hlld(); in
// rounding, the FP32 error scales with the jump across the face instead of
// with the flux itself, so smooth and near-static flows (a hydrostatic star,
// a weak shear layer) stay close to the FP64 result while the wave speeds,
// divisions and square roots run at FP32 cost.
//
// l, r: FP64 face primitives d, v1 (normal), v2, v3, b2, b3, e (total
// energy), pt (total pressure).  b1: GLM normal field (FP64).  cfl, cfr:
// fast speeds.  Writes f[0..4], f[6], f[7]; the GLM components f[5], f[8]
// are the caller's.
__device__ __forceinline__ void hlld_delta(double f[9], const double l[8], const double r[8],
                                           double b1, float cfl, float cfr) {
  const float h = 0.5f;
  const float dl = (float)l[0], dr = (float)r[0];
  const float v1l = (float)l[1], v1r = (float)r[1];
  const float v2l = (float)l[2], v2r = (float)r[2], v3l = (float)l[3], v3r = (float)r[3];
  const float b2l = (float)l[4], b2r = (float)r[4], b3l = (float)l[5], b3r = (float)r[5];
  const float b1f = (float)b1;
  // jumps across the face, differenced in FP64
  const float Dd = (float)(r[0] - l[0]), Dv1 = (float)(r[1] - l[1]);
  const float Dv2 = (float)(r[2] - l[2]), Dv3 = (float)(r[3] - l[3]);
  const float Db2 = (float)(r[4] - l[4]), Db3 = (float)(r[5] - l[5]);
  const float De = (float)(r[6] - l[6]), Dpt = (float)(r[7] - l[7]);
  const float ehl = (float)(l[6] + l[7]), ehr = (float)(r[6] + r[7]);

  const float sl = mn3(v1r - cfr, v1l - cfl, 0.0f);
  const float sr = mx3(v1r + cfr, v1l + cfl, 0.0f);
  const float slv = sl - v1l, srv = sr - v1r;
  const float den = srv * dr - slv * dl;
  const float dv = fdiv(srv * dr * Dv1 - Dpt, den);  // sm - v1l
  const float dvr = dv - Dv1;                         // sm - v1r
  const float sm = v1l + dv;
  const float slm = slv - dv, srm = srv - dvr;        // sl - sm, sr - sm
  const float dp = dl * slv * dv;                     // pta - ptl
  const float dpr = dr * srv * dvr;                   // pta - ptr
  const float ddla = fdiv(dl * dv, slm);              // dla - dl
  const float ddra = fdiv(dr * dvr, srm);             // dra - dr
  const float dla = dl + ddla, dra = dr + ddra;
  const float sqla = rsqrt_(dla), sqra = rsqrt_(dra);
  const float ab1 = abs_(b1f);
  const float sla = sm - fdiv(ab1, sqla), sra = sm + fdiv(ab1, sqra);

  const float b1b1 = b1f * b1f;
  const float idenl = fdiv(1.0f, dl * slv * slm - b1b1);
  const float idenr = fdiv(1.0f, dr * srv * srm - b1b1);
  // single-star transverse states relative to their own side
  const float dv2l = -b1f * b2l * dv * idenl, dv3l = -b1f * b3l * dv * idenl;
  const float dv2r = -b1f * b2r * dvr * idenr, dv3r = -b1f * b3r * dvr * idenr;
  const float gl = dl * slv * dv * idenl, gr = dr * srv * dvr * idenr;
  const float db2l = b2l * gl, db3l = b3l * gl, db2r = b2r * gr, db3r = b3r * gr;
  const float b2la = b2l + db2l, b3la = b3l + db3l, b2ra = b2r + db2r, b3ra = b3r + db3r;
  // (v.B) of the side state minus that of its star state
  const float xl = -b1f * dv - (v2l * db2l + dv2l * b2la) - (v3l * db3l + dv3l * b3la);
  const float xr = -b1f * dvr - (v2r * db2r + dv2r * b2ra) - (v3r * db3r + dv3r * b3ra);
  const float dela = fdiv(ehl * dv + dp * sm + b1f * xl, slm);   // ela - el
  const float dera = fdiv(ehr * dvr + dpr * sm + b1f * xr, srm);  // era - er

  // double-star (Alfven) states, relative to the left face state
  const float sb1 = sgn(1.0f, b1f);
  const float isqs = fdiv(1.0f, sqla + sqra);
  const float sqp = rsqrt_(dla * dra);
  const float dv2ra = Dv2 + dv2r, dv3ra = Dv3 + dv3r;  // v2ra - v2l
  const float db2ra = Db2 + db2r, db3ra = Db3 + db3r;  // b2ra - b2l
  const float dv2aa = (sqla * dv2l + sqra * dv2ra + (db2ra - db2l) * sb1) * isqs;
  const float dv3aa = (sqla * dv3l + sqra * dv3ra + (db3ra - db3l) * sb1) * isqs;
  const float db2aa = (sqla * db2ra + sqra * db2l + sqp * (dv2ra - dv2l) * sb1) * isqs;
  const float db3aa = (sqla * db3ra + sqra * db3l + sqp * (dv3ra - dv3l) * sb1) * isqs;
  const float b2aa = b2l + db2aa, b3aa = b3l + db3aa;
  // (v2 b2 + v3 b3) of a state minus that of the Alfven state
  const float pla = v2l * (db2l - db2aa) + dv2l * b2la - dv2aa * b2aa +
                    v3l * (db3l - db3aa) + dv3l * b3la - dv3aa * b3aa;
  const float pra = v2l * (db2ra - db2aa) + dv2ra * b2ra - dv2aa * b2aa +
                    v3l * (db3ra - db3aa) + dv3ra * b3ra - dv3aa * b3aa;
  const float delaa = dela - sb1 * sqla * pla;              // elaa - el
  const float deraa = (De + dera) + sb1 * sqra * pra;       // eraa - el

  // state selection (hlldflux.f90:140-154), as corrections to the left state
  const float signsm = sgn(h, sm);
  const float wla = h + sgn(h, sla), wra = h + sgn(h, -sra), waa = h - sgn(h, sla * sra);
  const float dd_ = (h + signsm) * ddla + (h - signsm) * (Dd + ddra);
  const float dv2_ = wla * dv2l + waa * dv2aa + wra * dv2ra;
  const float dv3_ = wla * dv3l + waa * dv3aa + wra * dv3ra;
  const float db2_ = wla * db2l + waa * db2aa + wra * db2ra;
  const float db3_ = wla * db3l + waa * db3aa + wra * db3ra;
  const float de_ = wla * dela + (h - sgn(h, sla * sm)) * delaa +
                    (h + sgn(h, -sm * sra)) * deraa + (h - sgn(h, sra)) * (De + dera);
  const float v2_ = v2l + dv2_, v3_ = v3l + dv3_, b2_ = b2l + db2_, b3_ = b3l + db3_;

  // fstar(selected) - fstar(left), hlldflux.f90:156-179
  const float dlv1l = (float)(l[0] * l[1]);
  const float df0 = dd_ * sm + dl * dv;
  const float df1 = df0 * sm + dlv1l * dv + dp;
  const float df2 = df0 * v2_ + dlv1l * dv2_ - b1f * db2_;
  const float df3 = df0 * v3_ + dlv1l * dv3_ - b1f * db3_;
  const float dvb = b1f * dv + (dv2_ * b2_ + v2l * db2_) + (dv3_ * b3_ + v3l * db3_);
  const float df4 = (de_ + dp) * sm + ehl * dv - b1f * dvb;
  const float df6 = db2_ * sm + b2l * dv - b1f * dv2_;
  const float df7 = db3_ * sm + b3l * dv - b1f * dv3_;

  // FP64 flux function of the left state
  const double u = l[1], du = l[0] * l[1];
  f[0] = du + (double)df0;
  f[1] = du * u + l[7] - b1 * b1 + (double)df1;
  f[2] = du * l[2] - b1 * l[4] + (double)df2;
  f[3] = du * l[3] - b1 * l[5] + (double)df3;
  f[4] = (l[6] + l[7]) * u - b1 * (u * b1 + l[2] * l[4] + l[3] * l[5]) + (double)df4;
  f[6] = l[4] * u - b1 * l[2] + (double)df6;
  f[7] = l[5] * u - b1 * l[3] + (double)df7;
}

}  // namespace hg

// dyn_math.h — pair arithmetic shared by the gfx950 kernels and the host-side
// fixed-point replay.
//
// Every function here uses only operations whose results IEEE-754 fixes
// exactly (add, sub, mul, fma, rint, ldexp, integer bit moves, exact
// conversions), so a host build of this header produces bit-identical
// per-pair forces and therefore bit-identical fixed-point sums.  Nothing here
// calls a vendor transcendental: rsqrt is a bit-level seed plus three Newton
// steps, exp is Cody–Waite reduction plus a degree-6 polynomial, and erfc is
// exp(-x²)·erfcx(x) with a degree-16 Chebyshev-derived polynomial for erfcx on
// [0, 4] (coefficients fitted here with numpy against scipy.special.erfcx; the
// fit's max relative error evaluated in f32 is 1.4e-7).
//
// Physics follows the reference:
//   LJ 12-6:           src/forces.rs:10-21, src/cuda/cuda.cu:40-63
//   erfc Coulomb:      src/cuda/cuda.cu:147-180 (F = qq (erfc(βr)/r² + 2β/√π e^{-β²r²}/r) r̂,
//                      E = qq erfc(βr)/r, zero at r ≥ cutoff)
//   soft-core LJ:      src/cuda/cuda.cu:73-144, src/non_bonded.rs:883-941
//   staged schedule:   src/alchemical.rs:82-100
//   min image (GPU):   src/cuda/util.cu:53-59 (rint, round half to even)
//   min image (CPU):   src/barostat.rs:162-170 (division then round half away)
//
// Compile with contraction off (-ffp-contract=off on both hipcc and g++):
// every fused multiply-add below is written out as dyn_fmaf().
#pragma once

#include <stdint.h>

#if defined(__HIPCC__)
#include <hip/hip_runtime.h>
#define DYN_HD __host__ __device__ inline
#else
#include <math.h>
#include <string.h>
#define DYN_HD static inline
struct float2 {
  float x, y;
};
struct float4 {
  float x, y, z, w;
};
struct double2 {
  double x, y;
};
#endif

#if defined(__clang__)
#pragma clang fp contract(off)
#endif

// ---------------------------------------------------------------------------
// Constants shared with the reference (values and meaning).
// ---------------------------------------------------------------------------
// src/non_bonded.rs:55-56 (1-4 scale factors, Amber convention).
#define DYN_SCALE_LJ_14 0.5f
#define DYN_SCALE_COUL_14 (1.0f / 1.2f)
// src/non_bonded.rs:63 (sqrt of 332.0522 kcal·Å/(mol·e²)).
#define DYN_CHARGE_UNIT_SCALER 18.2223f
// src/cuda/util.cu:18
#define DYN_INV_SQRT_PI 0.5641895835477563f
// src/alchemical.rs:55-65
#define DYN_SOFT_CORE_ALPHA 0.5f
#define DYN_SOFT_CORE_SIGMA_MIN 3.0f

// Fixed-point force scale: 2^32 units per kcal/(mol·Å).  Range ±2^31
// kcal/(mol·Å) in an int64 accumulator, resolution 2.3e-10.
#define DYN_FX_SCALE 4294967296.0
#define DYN_FX_INV_SCALE (1.0 / 4294967296.0)
// A single contribution is clamped to ±2^18 before conversion so the
// magic-number conversion below stays exact (needs |f·2^32| < 2^51).
#define DYN_FX_CLAMP 262144.0f
// Fixed-point charge-grid scale for SPME spreading: 2^32 units per charge
// unit (charges are in sqrt(kcal·Å/mol)).
#define DYN_GRID_FX_SCALE 4294967296.0

// ---------------------------------------------------------------------------
// Primitive operations
// ---------------------------------------------------------------------------
DYN_HD float dyn_fmaf(float a, float b, float c) {
#if defined(__HIP_DEVICE_COMPILE__)
  return __builtin_fmaf(a, b, c);
#else
  return fmaf(a, b, c);
#endif
}

DYN_HD double dyn_fma(double a, double b, double c) {
#if defined(__HIP_DEVICE_COMPILE__)
  return __builtin_fma(a, b, c);
#else
  return fma(a, b, c);
#endif
}

DYN_HD float dyn_floorf(float x) {
#if defined(__HIP_DEVICE_COMPILE__)
  return __builtin_floorf(x);
#else
  return floorf(x);
#endif
}

DYN_HD float dyn_rintf(float x) {
#if defined(__HIP_DEVICE_COMPILE__)
  return __builtin_rintf(x);
#else
  return rintf(x);
#endif
}

// Round half away from zero (Rust f32::round).
DYN_HD float dyn_roundf(float x) {
#if defined(__HIP_DEVICE_COMPILE__)
  return __builtin_roundf(x);
#else
  return roundf(x);
#endif
}

DYN_HD float dyn_ldexpf(float x, int e) {
#if defined(__HIP_DEVICE_COMPILE__)
  return __builtin_ldexpf(x, e);
#else
  return ldexpf(x, e);
#endif
}

DYN_HD uint32_t dyn_f2u(float f) {
#if defined(__HIP_DEVICE_COMPILE__)
  return __float_as_uint(f);
#else
  uint32_t u;
  memcpy(&u, &f, 4);
  return u;
#endif
}

DYN_HD float dyn_u2f(uint32_t u) {
#if defined(__HIP_DEVICE_COMPILE__)
  return __uint_as_float(u);
#else
  float f;
  memcpy(&f, &u, 4);
  return f;
#endif
}

DYN_HD int64_t dyn_d2bits(double d) {
#if defined(__HIP_DEVICE_COMPILE__)
  return (int64_t)__double_as_longlong(d);
#else
  int64_t u;
  memcpy(&u, &d, 8);
  return u;
#endif
}

DYN_HD float dyn_minf(float a, float b) { return a < b ? a : b; }
DYN_HD float dyn_maxf(float a, float b) { return a > b ? a : b; }

// 1/sqrt(x) for normal positive x: bit-level seed, three Newton steps.
// Max relative error 1.2e-7 over [1e-12, 1e12] (checked in tests).
DYN_HD float dyn_rsqrtf(float x) {
  float y = dyn_u2f(0x5f375a86u - (dyn_f2u(x) >> 1));
  const float hx = 0.5f * x;
  y = y * dyn_fmaf(-hx, y * y, 1.5f);
  y = y * dyn_fmaf(-hx, y * y, 1.5f);
  y = y * dyn_fmaf(-hx, y * y, 1.5f);
  return y;
}

// exp(y) for y in [-80, 0] (callers clamp).  Cody–Waite: y = n ln2 + r,
// |r| <= ln2/2, exp(r) by a degree-6 polynomial (max rel error 7.4e-8),
// scale by 2^n with an exact ldexp.
DYN_HD float dyn_exp_neg(float y) {
  y = dyn_maxf(y, -80.0f);
  const float n = dyn_rintf(y * 1.44269502f);
  float r = dyn_fmaf(n, -0.693145752f, y);  // ln2 high part (exact product)
  r = dyn_fmaf(n, -1.42860677e-06f, r);     // ln2 low part
  float p = 0x1.6d940cp-10f;
  p = dyn_fmaf(p, r, 0x1.125b1cp-7f);
  p = dyn_fmaf(p, r, 0x1.55547ep-5f);
  p = dyn_fmaf(p, r, 0x1.555430p-3f);
  p = dyn_fmaf(p, r, 0x1.000000p-1f);
  p = dyn_fmaf(p, r, 1.0f);
  p = dyn_fmaf(p, r, 1.0f);
  return dyn_ldexpf(p, (int)n);
}

// erfcx(x) = exp(x²) erfc(x) on [0, 4]; x is clamped into that range (the
// pair kernels only evaluate x = β r with r < cutoff).
DYN_HD float dyn_erfcx(float x) {
  x = dyn_minf(dyn_maxf(x, 0.0f), 4.0f);
  const float t = dyn_fmaf(x, 0.5f, -1.0f);
  float p = 0x1.1d0172p-12f;
  p = dyn_fmaf(p, t, -0x1.1b8896p-11f);
  p = dyn_fmaf(p, t, 0x1.226feep-21f);
  p = dyn_fmaf(p, t, -0x1.72ec3cp-15f);
  p = dyn_fmaf(p, t, 0x1.dce904p-10f);
  p = dyn_fmaf(p, t, -0x1.b0d348p-9f);
  p = dyn_fmaf(p, t, 0x1.26a02ep-8f);
  p = dyn_fmaf(p, t, -0x1.0564bap-7f);
  p = dyn_fmaf(p, t, 0x1.d63ce0p-7f);
  p = dyn_fmaf(p, t, -0x1.854ac8p-6f);
  p = dyn_fmaf(p, t, 0x1.367e3cp-5f);
  p = dyn_fmaf(p, t, -0x1.e0054ap-5f);
  p = dyn_fmaf(p, t, 0x1.64920cp-4f);
  p = dyn_fmaf(p, t, -0x1.fa9e76p-4f);
  p = dyn_fmaf(p, t, 0x1.5672b2p-3f);
  p = dyn_fmaf(p, t, -0x1.b57032p-3f);
  p = dyn_fmaf(p, t, 0x1.058672p-2f);
  return p;
}

// erfc(x) for x >= 0 from the two pieces above.
DYN_HD float dyn_erfcf(float x) {
  return dyn_exp_neg(-(x * x)) * dyn_erfcx(x);
}

// ---------------------------------------------------------------------------
// Fixed-point conversion.  round-to-nearest-even of f·2^32 as int64, computed
// with one f64 fma against 1.5·2^52 so the integer lands in the low mantissa
// bits (exact for |f·2^32| < 2^51; contributions are clamped to ±2^18).
// ---------------------------------------------------------------------------
DYN_HD int64_t dyn_fx(float f) {
  f = dyn_minf(dyn_maxf(f, -DYN_FX_CLAMP), DYN_FX_CLAMP);
  const double d = dyn_fma((double)f, DYN_FX_SCALE, 6755399441055744.0);
  return dyn_d2bits(d) - (int64_t)0x4338000000000000LL;
}

DYN_HD int64_t dyn_fx_d(double f, double scale) {
  const double d = dyn_fma(f, scale, 6755399441055744.0);
  return dyn_d2bits(d) - (int64_t)0x4338000000000000LL;
}

// dyn_fx for a double value (FP64 pair option): same clamp, same units.
DYN_HD int64_t dyn_fx64(double f) {
  f = f < -(double)DYN_FX_CLAMP ? -(double)DYN_FX_CLAMP : (f > (double)DYN_FX_CLAMP ? (double)DYN_FX_CLAMP : f);
  return dyn_fx_d(f, DYN_FX_SCALE);
}

// ---------------------------------------------------------------------------
// Minimum image.
// ---------------------------------------------------------------------------
// Kernel convention: dv - rint(dv·inv_ext)·ext with one rounding (fma).
DYN_HD float dyn_min_image_rint(float dv, float ext, float inv_ext) {
  return dyn_fmaf(-dyn_rintf(dv * inv_ext), ext, dv);
}

// The reference's CPU convention, reproduced bit for bit: true division,
// round half away from zero, then a separate multiply and subtract
// (src/barostat.rs:162-170).  Used by the neighbor-list build so its pair
// set matches the reference's brute-force build exactly.
DYN_HD float dyn_min_image_ref(float dv, float ext) {
  const float k = dyn_roundf(dv / ext);
  const float m = k * ext;
  return dv - m;
}

// |d|² as the reference's Vec3::magnitude_squared: (x² + y²) + z².
DYN_HD float dyn_norm2_ref(float x, float y, float z) {
  const float a = x * x;
  const float b = y * y;
  const float c = z * z;
  return (a + b) + c;
}

// ---------------------------------------------------------------------------
// Pair interactions.  All return the scalar s with F_on_i = s · d, d = r_i - r_j,
// so the virial contribution d·F is s·r².
// ---------------------------------------------------------------------------
// LJ with combined c6 = 4εσ⁶, c12 = 4εσ¹².
DYN_HD void dyn_lj(float rinv2, float c6, float c12, float* s, float* e) {
  const float rinv6 = rinv2 * rinv2 * rinv2;
  const float t12 = c12 * rinv6;
  *e = (t12 - c6) * rinv6;
  *s = dyn_fmaf(12.0f, t12, -6.0f * c6) * rinv6 * rinv2;
}

// erfc-screened Coulomb.  r2 = r², rinv = 1/r, qq = q_i q_j (Amber-scaled
// charges), beta = Ewald splitting parameter, beta2 = β², two_b_sqrtpi =
// 2β/√π.
DYN_HD void dyn_coul_erfc(float r2, float rinv, float qq, float beta,
                          float beta2, float two_b_sqrtpi, float* s, float* e) {
  const float r = r2 * rinv;
  const float ex = dyn_exp_neg(-(r2 * beta2));
  const float g = dyn_erfcx(r * beta);
  const float qe = qq * ex;
  const float gr = g * rinv;
  *e = qe * gr;
  *s = qe * (rinv * rinv) * (gr + two_b_sqrtpi);
}

// 1/x for normal positive x: bit-level seed (max rel. error 0.0506), one
// third-order and one Newton step.  Max relative error 1.3e-7 over the
// normal range of the pair distances (checked in tests).
DYN_HD float dyn_rcpf(float x) {
  float y = dyn_u2f(0x7ef31000u - dyn_f2u(x));
  float e = dyn_fmaf(-x, y, 1.0f);
  y = dyn_fmaf(y, dyn_fmaf(e, e, e), y);
  e = dyn_fmaf(-x, y, 1.0f);
  return dyn_fmaf(y, e, y);
}

// Tabulated erfc Coulomb of the pair kernel.  With x = βr and y = x² = β²r²
// the force scalar is s = qq·β³·Ψ(y), Ψ(y) = φ(x)/x³, φ(x) = erfc(x) +
// (2/√π) x e^{−x²}, and the energy E = qq·β·Λ(y), Λ(y) = erfc(x)/x.  Ψ and Λ
// are tabulated over y itself, so a pair inside the table needs no square
// root, reciprocal or exponential: 16 octaves of y from 2⁻¹¹, 64 intervals
// each, found from the exponent's low four bits and the mantissa's top six
// (any bit pattern finds an entry, so a lane outside the cutoff reads inside
// the table too).  Each entry is the cubic Hermite piece of its interval
// (values and derivatives from the closed forms, in double) in t = y − the
// interval's lower end, which is exact.  The interpolation error is below
// 1e-8 relative for y ≤ 1, 7e-7 at y = 16 (where Ψ and Λ are e⁻¹⁶ of the
// bare Coulomb terms).  Evaluation uses only IEEE-exact operations (mul,
// sub, fma, bit masks), so the host replay, given the same table, reproduces
// it bit for bit.
//
// Pairs closer than the table's first octave (r below 0.07 Å at β =
// 0.3123/Å) take φ(x) and erfc(x) over x = βr on [0, 4]: DYN_COUL_X_N cubic
// Hermite pieces each (error ≤ h⁴/384·max|f⁗| ≈ 1e-10, h = 1/128).
//
// A small β would leave most pairs below the first octave (at 0.005/Å all
// within 4.4 Å).  The tables are then over y = b²r² with b = 2ᵏβ, and hold
// 2⁻³ᵏΨ(y/4ᵏ) and 2⁻ᵏΛ(y/4ᵏ): s = qq·b³·(entry), E = qq·b·(entry) as before.
// k = dyn_coul_tab_shift(β, cutoff) is 0 from β·cutoff = 0.5 on and the least
// that brings b·cutoff there below, so the first octave ends at 0.044 cutoffs at
// most.
//
// Layout: two halves of DYN_COUL_TAB_N entries, the forces' (φ by x, then Ψ
// by y) and the energies' (erfc by x, then Λ by y).
#define DYN_COUL_X_N 512
#define DYN_COUL_TAB_XMAX 4.0f
#define DYN_COUL_TAB_SCALE 128.0f  // intervals per unit of x
#define DYN_COUL_Y_N 1024
#define DYN_COUL_Y_MIN 0x1p-11f
#define DYN_COUL_TAB_N (DYN_COUL_X_N + DYN_COUL_Y_N)

// The cubic of one half (entry_off 0 or 1) at u = x · DYN_COUL_TAB_SCALE.
DYN_HD float dyn_tab_cubic_u(const float4* tab, int entry_off, float u) {
  const float fl = dyn_floorf(u);
  int i = (int)fl;
  i = i < 0 ? 0 : (i > DYN_COUL_X_N - 1 ? DYN_COUL_X_N - 1 : i);
  const float t = u - fl;
  const float4 c = tab[entry_off * DYN_COUL_TAB_N + i];
  return dyn_fmaf(dyn_fmaf(dyn_fmaf(c.w, t, c.z), t, c.y), t, c.x);
}

DYN_HD float dyn_tab_cubic(const float4* tab, int entry_off, float x) {
  return dyn_tab_cubic_u(tab, entry_off, x * DYN_COUL_TAB_SCALE);
}

// An entry times a factor (b³ of the forces, b of the energies).
DYN_HD float4 dyn_tab_scale(float4 c, float f) {
  c.x *= f;
  c.y *= f;
  c.z *= f;
  c.w *= f;
  return c;
}

// f times the piece of ytab (DYN_COUL_Y_N entries, Ψ or Λ) at y ≥
// DYN_COUL_Y_MIN; SCALED: the entries hold that factor already (the pair
// kernel's copies in LDS).
template <bool SCALED>
DYN_HD float dyn_tab_y(const float4* ytab, float y, float f) {
  const uint32_t lo = dyn_f2u(y) & 0xFFFE0000u;  // the interval's lower end
  const float t = y - dyn_u2f(lo);
  // the entry's byte offset (bits 17 to 26 as an index, times 16)
#if defined(__HIP_DEVICE_COMPILE__)
  // one instruction (lo's low 17 bits are clear; the compiler would shift y
  // and mask the result instead)
  uint32_t at;
  asm("v_bfe_u32 %0, %1, 13, 14" : "=v"(at) : "v"(lo));
#else
  const uint32_t at = (lo >> 13) & (16u * (DYN_COUL_Y_N - 1));
#endif
  float4 c = *(const float4*)((const char*)ytab + at);
  if (!SCALED) c = dyn_tab_scale(c, f);
  return dyn_fmaf(dyn_fmaf(dyn_fmaf(c.w, t, c.z), t, c.y), t, c.x);
}

// r² below which a pair's y = r²b² may lie below the y tables (with room for
// the product's rounding); never below the r² of coincident sites.
DYN_HD float dyn_coul_r2_lo(float b2) {
  return dyn_maxf(1e-16f, 1.0001f * DYN_COUL_Y_MIN / b2);
}

// The k of the y tables (see above; a host function), β > 0.
static inline int dyn_coul_tab_shift(float beta, float cutoff) {
  int k = 0;
  while (ldexp((double)beta, k) * (double)cutoff < 0.5) ++k;
  return k;
}

// The x tables' form, for pairs below the y tables.
DYN_HD void dyn_coul_erfc_close(float r2, float qq, float beta, const float4* tab, float* s,
                                float* e) {
  const float rinv = dyn_rsqrtf(r2);
  const float u = (r2 * rinv) * (beta * DYN_COUL_TAB_SCALE);
  *s = qq * ((rinv * rinv) * rinv) * dyn_tab_cubic_u(tab, 0, u);
  *e = qq * rinv * dyn_tab_cubic_u(tab, 1, u);
}

// The tabulated pair at any r² (both forms; b = 2ᵏβ).
DYN_HD void dyn_coul_erfc_tab(float r2, float qq, float beta, float b, const float4* tab, float* s,
                              float* e) {
  const float b2 = b * b;
  if (!(r2 > dyn_coul_r2_lo(b2))) {
    dyn_coul_erfc_close(r2, qq, beta, tab, s, e);
    return;
  }
  const float y = r2 * b2;
  *s = qq * dyn_tab_y<false>(tab + DYN_COUL_X_N, y, b2 * b);
  *e = qq * dyn_tab_y<false>(tab + DYN_COUL_TAB_N + DYN_COUL_X_N, y, b);
}

// The table (2·DYN_COUL_TAB_N float4 as 8·DYN_COUL_TAB_N floats) of shift k,
// built on the host in double from the closed forms (a host function).
static inline void dyn_coul_tab_build(float* out, int shift) {
  const double k2 = 1.1283791670955126;  // 2/√π
  // the Hermite piece over an interval of width h, in t = argument − lower
  // end times sc
  auto piece = [](float* c, double f0, double f1, double d0, double d1, double h, double sc) {
    d0 *= h;
    d1 *= h;
    c[0] = (float)f0;
    c[1] = (float)(d0 * sc);
    c[2] = (float)((3.0 * (f1 - f0) - 2.0 * d0 - d1) * sc * sc);
    c[3] = (float)((2.0 * (f0 - f1) + d0 + d1) * sc * sc * sc);
  };
  // one erfc and one exponential a node: the two ends of neighbouring
  // intervals are one node
  struct Node { double f, df, e, de; };
  auto node_x = [&](double x) {
    const double er = erfc(x), ex = exp(-x * x);
    return Node{er + k2 * x * ex, -2.0 * k2 * x * x * ex, er, -k2 * ex};
  };
  const double down3 = ldexp(1.0, -3 * shift);
  auto node_y = [&](double y) {
    const double w = sqrt(y), x = ldexp(w, -shift), er = erfc(x), ex = exp(-x * x);
    const double psi = (er + k2 * x * ex) / (y * w);
    return Node{psi, (-k2 * ex * down3 - 1.5 * psi) / y, er / w, -0.5 * psi};
  };
  auto put = [&](int at, const Node& a, const Node& b, double h, double sc) {
    piece(out + 4 * at, a.f, b.f, a.df, b.df, h, sc);
    piece(out + 4 * (DYN_COUL_TAB_N + at), a.e, b.e, a.de, b.de, h, sc);
  };
  const double h = 1.0 / (double)DYN_COUL_TAB_SCALE;
  Node a = node_x(0.0);
  for (int i = 0; i < DYN_COUL_X_N; ++i) {
    const Node b = node_x((i + 1) * h);
    put(i, a, b, h, 1.0);
    a = b;
  }
  a = node_y((double)DYN_COUL_Y_MIN);
  for (int k = 0; k < DYN_COUL_Y_N; ++k) {
    // octave 0 starts at DYN_COUL_Y_MIN = 2⁻¹¹ (biased exponent 116)
    const double lo = ldexp(1.0, k / 64 - 11), hy = lo / 64.0;
    const Node b = node_y(lo + (k % 64 + 1) * hy);
    put(DYN_COUL_X_N + ((((k / 64 + 116) & 15) << 6) | (k % 64)), a, b, hy, 1.0 / hy);
    a = b;
  }
}

// erf-screened Coulomb qq·erf(βr)/r, i.e. the part of a pair's Coulomb
// interaction carried by the reciprocal sum.  Used for exclusion
// corrections.  For small βr the direct series avoids cancellation.
DYN_HD void dyn_coul_erf(float r2, float rinv, float qq, float beta,
                         float beta2, float two_b_sqrtpi, float* s, float* e) {
  const float r = r2 * rinv;
  const float x = r * beta;
  const float ex = dyn_exp_neg(-(r2 * beta2));
  float erf_x;
  if (x < 0.5f) {
    // erf(x) = 2/√π Σ (-1)^n x^(2n+1)/(n!(2n+1)), 7 terms: rel err < 1e-9 for x < 0.5.
    const float x2 = x * x;
    float p = -1.0f / 75600.0f;
    p = dyn_fmaf(p, x2, 1.0f / 9360.0f);
    p = dyn_fmaf(p, x2, -1.0f / 1320.0f);
    p = dyn_fmaf(p, x2, 1.0f / 216.0f);
    p = dyn_fmaf(p, x2, -1.0f / 42.0f);
    p = dyn_fmaf(p, x2, 1.0f / 10.0f);
    p = dyn_fmaf(p, x2, -1.0f / 3.0f);
    p = dyn_fmaf(p, x2, 1.0f);
    erf_x = 1.1283791670955126f * x * p;
  } else {
    erf_x = 1.0f - ex * dyn_erfcx(x);
  }
  const float er = erf_x * rinv;
  *e = qq * er;
  // d/dr [erf(βr)/r] = -erf/r² + (2β/√π) e^{-β²r²}/r ; s = -(dE/dr)/r
  *s = qq * (rinv * rinv) * (er - two_b_sqrtpi * ex);
}

// Staged decoupling schedule (src/alchemical.rs:82-100).
struct DynSchedule {
  float coulomb_scale;
  float coulomb_dscale_dlambda;
  float lj_lambda;
  float lj_dlambda_dlambda;
};

DYN_HD DynSchedule dyn_schedule(float lambda) {
  lambda = dyn_minf(1.0f, dyn_maxf(0.0f, lambda));
  DynSchedule s;
  if (lambda < 0.5f) {
    s.coulomb_scale = 1.0f - 2.0f * lambda;
    s.coulomb_dscale_dlambda = -2.0f;
    s.lj_lambda = 0.0f;
    s.lj_dlambda_dlambda = 0.0f;
  } else {
    s.coulomb_scale = 0.0f;
    s.coulomb_dscale_dlambda = 0.0f;
    s.lj_lambda = 2.0f * lambda - 1.0f;
    s.lj_dlambda_dlambda = 2.0f;
  }
  return s;
}

// Beutler soft-core LJ decoupling with p = 1 (src/cuda/cuda.cu:73-144):
// V = (1-λ) V_LJ(r_sc), r_sc⁶ = r⁶ + α σ_sc⁶ λ, σ_sc = max(σ, σ_min).
// Written with sigma/eps (not c6/c12) because σ_sc depends on σ.
// Returns s (F = s·d), energy and dV/dλ.  r_sc⁻² = (r_sc⁶)^(-1/3) comes from
// a Newton iteration for the inverse cube root (bit-level seed), and
// r_sc⁻¹ = r_sc⁻² · rsqrt(r_sc⁻²); no division or pow is needed.
DYN_HD float dyn_inv_cbrt(float a) {
  // y ≈ a^(-1/3); Newton on f(y) = y^-3 - a: y ← y (4 - a y³)/3.
  float y = dyn_u2f(0x54aaaaaau - dyn_f2u(a) / 3u);
  for (int k = 0; k < 5; ++k) {
    const float y3 = y * y * y;
    y = y * dyn_fmaf(-a, y3, 4.0f) * (1.0f / 3.0f);
  }
  return y;
}

DYN_HD void dyn_lj_soft_core(float r2, float sigma, float eps, float lambda,
                             float* s, float* e, float* dhdl) {
  *s = 0.0f;
  *e = 0.0f;
  *dhdl = 0.0f;
  if (eps == 0.0f || r2 < 0.0f) return;
  lambda = dyn_minf(1.0f, dyn_maxf(0.0f, lambda));
  const float scale = 1.0f - lambda;
  const float ss = dyn_maxf(sigma, DYN_SOFT_CORE_SIGMA_MIN);
  const float ss2 = ss * ss;
  const float ss6 = ss2 * ss2 * ss2;
  const float r6 = r2 * r2 * r2;
  const float rsc6 = r6 + DYN_SOFT_CORE_ALPHA * ss6 * lambda;
  if (!(rsc6 > 0.0f)) return;
  const float inv_rsc2 = dyn_inv_cbrt(rsc6);
  const float inv_rsc = inv_rsc2 * dyn_rsqrtf(inv_rsc2);
  const float sg2 = sigma * sigma;
  const float sr2 = sg2 * inv_rsc2;
  const float sr6 = sr2 * sr2 * sr2;
  const float sr12 = sr6 * sr6;
  const float hard_fmag = 24.0f * eps * dyn_fmaf(2.0f, sr12, -sr6) * inv_rsc;  // |F_LJ(r_sc)|
  const float hard_e = 4.0f * eps * (sr12 - sr6);
  // F(r) = scale · F_LJ(r_sc) · (r/r_sc)^5 r̂, so s = F/r = scale·F_LJ·r⁴/r_sc⁵
  const float inv_rsc5 = inv_rsc2 * inv_rsc2 * inv_rsc;
  *s = hard_fmag * scale * (r2 * r2) * inv_rsc5;
  *e = hard_e * scale;
  // dr_sc/dλ = α σ_sc⁶ / (6 r_sc⁵)
  const float drsc = DYN_SOFT_CORE_ALPHA * ss6 * inv_rsc5 * (1.0f / 6.0f);
  *dhdl = -hard_e - scale * hard_fmag * drsc;
}

// ---------------------------------------------------------------------------
// Cardinal B-spline weights for SPME (Essmann et al. 1995, eq. 4.1 recursion).
// u is the fractional grid coordinate within its cell (w in [0,1)); the
// weights are for grid points k0-(order-1) .. k0 where k0 = floor(position).
// th[j] is the weight for offset j (grid index k0 - order + 1 + j), dth its
// derivative with respect to the fractional coordinate.
// ---------------------------------------------------------------------------
// R = float for the f32 paths (bit-identical on device and host), double for
// the FP64 SPME option.
template <int ORDER, class R = float>
DYN_HD void dyn_bspline(R w, R* th, R* dth) {
  // order 2
  R m[ORDER];
  m[0] = R(1) - w;
  m[1] = w;
  for (int k = 2; k < ORDER - 1; ++k) {
    // raise from order k to k+1
    const R div = R(1) / (R)k;
    m[k] = div * w * m[k - 1];
    for (int j = 1; j < k; ++j) {
      m[k - j] = div * ((w + (R)j) * m[k - j - 1] + ((R)(k - j + 1) - w) * m[k - j]);
    }
    m[0] = div * (R(1) - w) * m[0];
  }
  // derivative of the order-ORDER spline from the order-(ORDER-1) values
  dth[0] = -m[0];
  for (int j = 1; j < ORDER - 1; ++j) dth[j] = m[j - 1] - m[j];
  dth[ORDER - 1] = m[ORDER - 2];
  // final raise to ORDER
  {
    const int k = ORDER - 1;
    const R div = R(1) / (R)k;
    m[k] = div * w * m[k - 1];
    for (int j = 1; j < k; ++j) {
      m[k - j] = div * ((w + (R)j) * m[k - j - 1] + ((R)(k - j + 1) - w) * m[k - j]);
    }
    m[0] = div * (R(1) - w) * m[0];
  }
  for (int j = 0; j < ORDER; ++j) th[j] = m[j];
}

// engine.h — device-side types of the native nonbonded engine, shared by the
// kernels and the host fixed-point replay.
#pragma once

#include "dyn_math.h"

// Site classes.  Clusters hold sites of one class only, so a cluster pair
// knows from its two classes which interactions exist: solute–solute LJ +
// Coulomb, solute–O LJ, solute–charged Coulomb, O–O LJ, charged–charged
// Coulomb; O–charged pairs have neither and are never listed.
#define DYN_CLS_SOLUTE 0
#define DYN_CLS_WATER_O 1
#define DYN_CLS_WATER_Q 2

#define DYN_CL_SIZE 8  // sites per cluster; a wave holds 8 i slots × 8 j slots
#define DYN_CHUNK 16   // default j groups (of 8 j slots) per work item of the pair kernel

// A row of the pair list (one i cluster) holds j slots: every slot of a
// nearby cluster that lies within the list radius of at least one i slot it
// interacts with.  The slots are grouped by class, each class segment padded
// to a multiple of 8 with the null slot, and a list entry stores
// slot | class << DYN_JCLS_SHIFT.  A group is 8 consecutive entries.
#define DYN_JCLS_SHIFT 30
#define DYN_JSLOT_MASK ((1u << DYN_JCLS_SHIFT) - 1u)

// Exclusion group of a cluster slot: the water molecule (≥ 0) for water
// sites, −2 − site for solute atoms (unique), −1 for padding.  Two slots
// interact only if their groups differ and neither is padding; solute–solute
// cluster pairs additionally carry an explicit 64-bit mask for the 1-2, 1-3
// and 1-4 exclusions.
#define DYN_GID_PAD (-1)

DYN_HD bool dyn_slot_pair_valid(int gi, int gj) {
  return gi != gj && gi != DYN_GID_PAD && gj != DYN_GID_PAD;
}

// Interaction kinds of a cluster pair (from the two classes).
#define DYN_KIND_SS 0  // LJ (type table) + Coulomb
#define DYN_KIND_SO 1  // LJ (type table)
#define DYN_KIND_SQ 2  // Coulomb
#define DYN_KIND_OO 3  // LJ (O–O constants)
#define DYN_KIND_QQ 4  // Coulomb
#define DYN_KIND_NONE 5

DYN_HD int dyn_kind(int ci, int cj) {
  if (ci > cj) {
    const int t = ci;
    ci = cj;
    cj = t;
  }
  if (ci == DYN_CLS_SOLUTE) return cj == DYN_CLS_SOLUTE ? DYN_KIND_SS : (cj == DYN_CLS_WATER_O ? DYN_KIND_SO : DYN_KIND_SQ);
  if (ci == DYN_CLS_WATER_O) return cj == DYN_CLS_WATER_O ? DYN_KIND_OO : DYN_KIND_NONE;
  return DYN_KIND_QQ;
}

// Type word of a slot: the LJ type in the low bits, DYN_TYPE_ALCH when the
// site belongs to the decoupled (alchemical) molecule.
#define DYN_TYPE_ALCH 0x10000
#define DYN_TYPE_MASK 0xffff

struct DynPairParams {
  float ext[3], inv_ext[3];
  float rc2;        // Coulomb (and list) cutoff squared
  float lj_rc2;     // LJ cutoff squared
  float beta, beta2, two_b_sqrtpi;
  float c6_oo, c12_oo;
  int n_types;      // LJ type tables are (n_types × n_types) float2
  int alch_on;      // a decoupled molecule exists
  DynSchedule sch;  // staged decoupling schedule at the current λ
  float tab_b, tab_b2;     // the b of its y tables, b²
  const float4* coul_tab;  // the erfc Coulomb table (dyn_coul_tab_build)
};

// The two Coulomb tables a lane reads (dyn_math.h): Ψ and Λ over y = b²r².
// The pair kernel reads copies in LDS, multiplied by b³ and b (etab is not
// read by a forces-only evaluation).
struct DynCoulTabs {
  const float4 *ftab, *etab;
};
DYN_HD DynCoulTabs dyn_coul_tabs(const float4* coul_tab) {
  return DynCoulTabs{coul_tab + DYN_COUL_X_N, coul_tab + DYN_COUL_TAB_N + DYN_COUL_X_N};
}

// The pair (i, j) of the given kind at squared distance r2: the scalar s
// (F_i = s·d) and energies, zero for an inactive lane.  `active` already
// includes the list mask; the cutoff test happens here.  r2_lo =
// dyn_coul_r2_lo(b²).  No square root or reciprocal of r² is taken for
// Coulomb pairs (tabulated over b²r²); LJ takes 1/r² directly.  SCALED: tabs
// holds the tables multiplied by b³ and b.  Returns whether the pair interacts but lies below
// the Coulomb tables: then s and the energies are not set, and
// dyn_tile_close gives them.
template <int KIND, bool SCALED>
DYN_HD bool dyn_tile_eval(float r2, float qi, float qj, float c6, float c12, bool active, float r2_lo,
                          const DynPairParams& P, const DynCoulTabs& tabs, float* s_out, float* e_lj,
                          float* e_c, int* hit) {
  constexpr bool kLj = KIND == DYN_KIND_SS || KIND == DYN_KIND_SO || KIND == DYN_KIND_OO;
  constexpr bool kCoul = KIND == DYN_KIND_SS || KIND == DYN_KIND_SQ || KIND == DYN_KIND_QQ;
  // (no short-circuits: every lane takes the same path)
  const bool near_ = active & (r2 < P.rc2);
  const bool in = near_ & (r2 > (kCoul ? r2_lo : 1e-16f));
  const bool lj_in = in & (r2 <= P.lj_rc2);
  float s = 0.f, elj = 0.f, ec = 0.f;
  if (kLj) dyn_lj(dyn_rcpf(r2), c6, c12, &s, &elj);
  if (kCoul) {
    const float y = r2 * P.tab_b2;
    const float qq = qi * qj;
    const float sc = qq * dyn_tab_y<SCALED>(tabs.ftab, y, P.tab_b2 * P.tab_b);
    ec = qq * dyn_tab_y<SCALED>(tabs.etab, y, P.tab_b);
    s = kLj ? (r2 <= P.lj_rc2 ? sc + s : sc) : sc;
    *s_out = in ? s : 0.f;
    *e_lj = kLj && lj_in ? elj : 0.f;
    *e_c = in ? ec : 0.f;
  } else {
    *s_out = lj_in ? s : 0.f;
    *e_lj = lj_in ? elj : 0.f;
    *e_c = 0.f;
  }
  *hit = in ? 1 : 0;
  return kCoul && (near_ & !in);
}

// A pair dyn_tile_eval returned true for (sites that coincide do not
// interact).
template <int KIND>
DYN_HD void dyn_tile_close(float r2, float qi, float qj, float c6, float c12, const DynPairParams& P,
                           float* s_out, float* e_lj, float* e_c, int* hit) {
  *s_out = *e_lj = *e_c = 0.f;
  *hit = r2 > 1e-16f ? 1 : 0;
  if (!*hit) return;
  dyn_coul_erfc_close(r2, qi * qj, P.beta, P.coul_tab, s_out, e_c);
  if (KIND == DYN_KIND_SS && r2 <= P.lj_rc2) {
    float sl;
    dyn_lj(dyn_rcpf(r2), c6, c12, &sl, e_lj);
    *s_out = *s_out + sl;
  }
}

// (c6, c12) of a pair of the given kind.
template <int KIND>
DYN_HD float2 dyn_tile_c(int ti, int tj, const DynPairParams& P, const float2* lj_table) {
  float2 c;
  c.x = P.c6_oo;
  c.y = P.c12_oo;
  if (KIND == DYN_KIND_SS || KIND == DYN_KIND_SO)
    c = lj_table[(ti & DYN_TYPE_MASK) * P.n_types + (tj & DYN_TYPE_MASK)];
  return c;
}

// One lane of an 8×8 tile from the two sites: displacement d (minimum
// image), scalar s, energies, squared distance (0 for an inactive lane).
template <int KIND>
DYN_HD void dyn_tile_pair(const float pi[4], int ti, const float pj[4], int tj, bool active,
                          const DynPairParams& P, const float2* lj_table, float d[3],
                          float* s_out, float* e_lj, float* e_c, float* r2_out, int* hit) {
  for (int a = 0; a < 3; ++a) d[a] = dyn_min_image_rint(pi[a] - pj[a], P.ext[a], P.inv_ext[a]);
  const float r2 = dyn_fmaf(d[2], d[2], dyn_fmaf(d[1], d[1], d[0] * d[0]));
  const float2 c = dyn_tile_c<KIND>(ti, tj, P, lj_table);
  if (dyn_tile_eval<KIND, false>(r2, pi[3], pj[3], c.x, c.y, active, dyn_coul_r2_lo(P.tab_b2), P,
                                 dyn_coul_tabs(P.coul_tab), s_out, e_lj, e_c, hit))
    dyn_tile_close<KIND>(r2, pi[3], pj[3], c.x, c.y, P, s_out, e_lj, e_c, hit);
  *r2_out = *hit ? r2 : 0.f;
}

// FP64 variant for the precision sweep: the same interactions from the same
// f32 inputs (positions, charges, combined σ and ε), every operation in
// double with the math library's erfc, exp and sqrt; c6/c12 from a double
// table.  Not bit-replayed on the host: it is
// checked against the FP64 oracle instead.
template <int KIND>
DYN_HD void dyn_tile_pair_f64(const float pi[4], int ti, const float pj[4], int tj, bool active,
                              const DynPairParams& P, const double2* lj64, double d[3],
                              double* s_out, double* e_lj, double* e_c, double* r2_out, int* hit) {
  double r2 = 0.0;
  for (int a = 0; a < 3; ++a) {
    const double L = (double)P.ext[a];
    double v = (double)pi[a] - (double)pj[a];
    v -= L * rint(v / L);
    d[a] = v;
    r2 += v * v;
  }
  const bool in = active && r2 < (double)P.rc2 && r2 > 1e-16;
  const double r2s = in ? r2 : 1.0;
  const double rinv = 1.0 / sqrt(r2s);
  double s = 0.0, elj = 0.0, ec = 0.0;
  if (KIND == DYN_KIND_SS || KIND == DYN_KIND_SO || KIND == DYN_KIND_OO) {
    // the O–O pair too comes from the table (its f32 constants are rounded)
    const double2 c = lj64[(ti & DYN_TYPE_MASK) * P.n_types + (tj & DYN_TYPE_MASK)];
    const double c6 = c.x, c12 = c.y;
    const double rinv2 = rinv * rinv, rinv6 = rinv2 * rinv2 * rinv2;
    const bool lj_in = in && r2 <= (double)P.lj_rc2;
    s = lj_in ? (12.0 * c12 * rinv6 - 6.0 * c6) * rinv6 * rinv2 : 0.0;
    elj = lj_in ? (c12 * rinv6 - c6) * rinv6 : 0.0;
  }
  if (KIND == DYN_KIND_SS || KIND == DYN_KIND_SQ || KIND == DYN_KIND_QQ) {
    const double qq = (double)pi[3] * (double)pj[3];
    const double beta = (double)P.beta, r = r2s * rinv;
    const double g = erfc(beta * r) * rinv;
    const double sc = qq * (g + 1.1283791670955126 * beta * exp(-beta * beta * r2s)) * rinv * rinv;
    s += in ? sc : 0.0;
    ec = in ? qq * g : 0.0;
  }
  *s_out = s;
  *e_lj = elj;
  *e_c = ec;
  *r2_out = in ? r2 : 0.0;
  *hit = in ? 1 : 0;
}

// Alchemical pair (src/cuda/cuda.cu:367-566) within the cutoff: two sites on
// different sides of the decoupled molecule (exactly one carries
// DYN_TYPE_ALCH) take Beutler soft-core LJ at the schedule's LJ λ and Coulomb
// scaled by the schedule's factor, and return dH/dλ.  lj_se holds the
// combined (σ, ε) of each type pair.
template <int KIND>
DYN_HD void dyn_tile_alch(float r2, float qi, float qj, int ti, int tj, const DynPairParams& P,
                          const float2* lj_se, float* s_out, float* e_lj, float* e_c, float* dh) {
  const float rinv = dyn_rsqrtf(r2);
  float s = 0.f, elj = 0.f, ec = 0.f, dhh = 0.f;
  if (KIND == DYN_KIND_SS || KIND == DYN_KIND_SO) {
    if (r2 <= P.lj_rc2) {
      const float2 se = lj_se[(ti & DYN_TYPE_MASK) * P.n_types + (tj & DYN_TYPE_MASK)];
      float ssc, esc, dd;
      dyn_lj_soft_core(r2, se.x, se.y, P.sch.lj_lambda, &ssc, &esc, &dd);
      s = ssc;
      elj = esc;
      dhh = dd * P.sch.lj_dlambda_dlambda;
    }
  }
  if (KIND == DYN_KIND_SS || KIND == DYN_KIND_SQ) {
    float sc, ee;
    dyn_coul_erfc(r2, rinv, qi * qj, P.beta, P.beta2, P.two_b_sqrtpi, &sc, &ee);
    s = s + sc * P.sch.coulomb_scale;
    ec = ee * P.sch.coulomb_scale;
    dhh = dhh + ee * P.sch.coulomb_dscale_dlambda;
  }
  *s_out = s;
  *e_lj = elj;
  *e_c = ec;
  *dh = dhh;
}

// dyn_tile_pair with alchemical pairs (every other lane returns
// dyn_tile_pair's result bit for bit).
template <int KIND>
DYN_HD void dyn_tile_pair_alch(const float pi[4], int ti, const float pj[4], int tj, bool active,
                               const DynPairParams& P, const float2* lj_table,
                               const float2* lj_se, float d[3], float* s_out, float* e_lj,
                               float* e_c, float* r2_out, int* hit, float* dh) {
  dyn_tile_pair<KIND>(pi, ti, pj, tj, active, P, lj_table, d, s_out, e_lj, e_c, r2_out, hit);
  *dh = 0.f;
  if (((ti ^ tj) & DYN_TYPE_ALCH) != 0 && *hit)
    dyn_tile_alch<KIND>(*r2_out, pi[3], pj[3], ti, tj, P, lj_se, s_out, e_lj, e_c, dh);
}

// corr.h — the exclusion and 1-4 corrections of an evaluation, a device
// function that launches share.
//
// Reference semantics: src/non_bonded.rs:763-790.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <functional>

#include "common.h"
#include "dyn_math.h"
#include "engine.h"
#include "wave.h"

namespace dyn {

// Correction pairs: kind 1 = 1-4 pair (scaled real-space LJ + Coulomb, plus
// the reciprocal correction of the mode), kind 0 = excluded pair (standard
// mode: remove qq·erf(βr)/r from the reciprocal sum).
struct CorrArgs {
  DynPairParams P;
  const float4* wpos;      // per site (x, y, z, q)
  const int32_t* ltype;    // per site type word (DYN_TYPE_ALCH marks the decoupled molecule)
  const float2* lj_table;
  const float2* lj_se;     // (σ, ε) per type pair, for soft-core
  const uint32_t* ci;
  const uint32_t* cj;
  const uint8_t* kind;
  uint32_t n;
  int mode;
  int recip_on;            // reciprocal corrections only accompany the SPME sum
  uint32_t nblk;           // workgroups (one partial each)
  int64_t* mol_e;          // n_mol² molecule-pair energies, or null
  const int32_t* mol_of;
  uint32_t n_mol;
  int64_t* fx;             // site forces, component-major
  uint32_t n_sites;
  double* partials;        // kCorrVals per block: e_lj14, e_c14, e_corr, vir_sr, vir_recip, dH/dλ
};

constexpr int kCorrBlock = 256;
constexpr int kCorrVals = 7;  // per-block sums of the correction kernel
__device__ __forceinline__ void corr_terms(const CorrArgs& A, uint32_t block) {
  __shared__ double red[kCorrVals * (kCorrBlock / kWaveLanes)];
  if (block >= A.nblk) return;  // partials exist for the system's own blocks
  // e_lj14, e_c14, e_corr, vir_sr, vir_recip, dH/dλ, 1-4 pairs within the cutoff
  double acc[kCorrVals] = {0, 0, 0, 0, 0, 0, 0};
  // molecule-pair matrix: a running entry per thread (1-4 pairs lie within
  // one molecule), flushed when the entry changes and once at the end
  int mkey = -1;
  double me = 0.0;
  for (uint32_t k = block * kCorrBlock + threadIdx.x; k < A.n; k += A.nblk * kCorrBlock) {
    if (A.kind[k] == 0 && !A.recip_on) continue;
    const uint32_t i = A.ci[k], j = A.cj[k];
    const float4 a = A.wpos[i], b = A.wpos[j];
    float d0 = dyn_min_image_rint(a.x - b.x, A.P.ext[0], A.P.inv_ext[0]);
    float d1 = dyn_min_image_rint(a.y - b.y, A.P.ext[1], A.P.inv_ext[1]);
    float d2 = dyn_min_image_rint(a.z - b.z, A.P.ext[2], A.P.inv_ext[2]);
    const float r2 = dyn_fmaf(d2, d2, dyn_fmaf(d1, d1, d0 * d0));
    if (!(r2 > 1e-12f)) continue;
    const float rinv = dyn_rsqrtf(r2);
    const float qq = a.w * b.w;
    float s_sr = 0.f, s_rc = 0.f;
    double e_pair = 0.0;  // the 1-4 pair's energy (molecule-pair matrix)
    if (A.kind[k] == 1) {
      if (r2 < A.P.rc2) acc[6] += 1.0;
      // a 1-4 pair across the decoupled molecule's boundary is also an
      // alchemical pair (src/non_bonded.rs:581-599)
      const bool cross = A.P.alch_on && ((A.ltype[i] ^ A.ltype[j]) & DYN_TYPE_ALCH) != 0;
      const int tab = (A.ltype[i] & DYN_TYPE_MASK) * A.P.n_types + (A.ltype[j] & DYN_TYPE_MASK);
      if (r2 <= A.P.lj_rc2) {
        float sl, el;
        if (cross) {
          const float2 se = A.lj_se[tab];
          float dd;
          dyn_lj_soft_core(r2, se.x, se.y, A.P.sch.lj_lambda, &sl, &el, &dd);
          acc[5] += (double)(DYN_SCALE_LJ_14 * (dd * A.P.sch.lj_dlambda_dlambda));
        } else {
          const float2 c = A.lj_table[tab];
          dyn_lj(rinv * rinv, c.x, c.y, &sl, &el);
        }
        s_sr += DYN_SCALE_LJ_14 * sl;
        acc[0] += (double)(DYN_SCALE_LJ_14 * el);
        e_pair += (double)(DYN_SCALE_LJ_14 * el);
      }
      if (r2 < A.P.rc2) {
        float sc, ec;
        dyn_coul_erfc(r2, rinv, qq, A.P.beta, A.P.beta2, A.P.two_b_sqrtpi, &sc, &ec);
        sc = 0.833333333f * sc;
        ec = 0.833333333f * ec;
        if (cross) {
          acc[5] += (double)(ec * A.P.sch.coulomb_dscale_dlambda);
          sc = sc * A.P.sch.coulomb_scale;
          ec = ec * A.P.sch.coulomb_scale;
        }
        s_sr += sc;
        acc[1] += (double)ec;
        e_pair += (double)ec;
      }
      if (!A.recip_on) {
        // no reciprocal sum, nothing to correct
      } else if (A.mode == DYN_MODE_REFERENCE) {
        // vacuum correction (1/1.2 − 1)·qq/r² along r̂, force only
        s_rc = (DYN_SCALE_COUL_14 - 1.0f) * qq * (rinv * rinv * rinv);
      } else {
        float se, ee;
        dyn_coul_erf(r2, rinv, qq, A.P.beta, A.P.beta2, A.P.two_b_sqrtpi, &se, &ee);
        s_rc = -(1.0f - DYN_SCALE_COUL_14) * se;
        acc[2] += (double)(-(1.0f - DYN_SCALE_COUL_14) * ee);
      }
    } else {
      float se, ee;
      dyn_coul_erf(r2, rinv, qq, A.P.beta, A.P.beta2, A.P.two_b_sqrtpi, &se, &ee);
      s_rc = -se;
      acc[2] += (double)(-ee);
    }
    acc[3] += (double)(s_sr * r2);
    acc[4] += (double)(s_rc * r2);
    if (A.mol_e && e_pair != 0.0) {
      const int mi = A.mol_of[i], mj = A.mol_of[j];
      if (mi != mj) {  // both orders (src/non_bonded.rs:350-361)
        const uint64_t v = (uint64_t)dyn_fx64(e_pair);
        atomicAdd(reinterpret_cast<unsigned long long*>(A.mol_e + mi * (int)A.n_mol + mj), v);
        atomicAdd(reinterpret_cast<unsigned long long*>(A.mol_e + mj * (int)A.n_mol + mi), v);
      } else {
        const int key = mi * (int)A.n_mol + mi;
        if (key != mkey) {
          if (mkey >= 0)
            atomicAdd(reinterpret_cast<unsigned long long*>(A.mol_e + mkey),
                      (unsigned long long)dyn_fx64(me));
          mkey = key;
          me = 0.0;
        }
        me += e_pair;
      }
    }
    const float s = s_sr + s_rc;
    const int64_t q0 = dyn_fx(s * d0), q1 = dyn_fx(s * d1), q2 = dyn_fx(s * d2);
    atomicAdd(reinterpret_cast<unsigned long long*>(A.fx + i), (unsigned long long)q0);
    atomicAdd(reinterpret_cast<unsigned long long*>(A.fx + A.n_sites + i), (unsigned long long)q1);
    atomicAdd(reinterpret_cast<unsigned long long*>(A.fx + 2 * (size_t)A.n_sites + i), (unsigned long long)q2);
    atomicAdd(reinterpret_cast<unsigned long long*>(A.fx + j), (unsigned long long)(-q0));
    atomicAdd(reinterpret_cast<unsigned long long*>(A.fx + A.n_sites + j), (unsigned long long)(-q1));
    atomicAdd(reinterpret_cast<unsigned long long*>(A.fx + 2 * (size_t)A.n_sites + j), (unsigned long long)(-q2));
  }
  if (A.mol_e) wave_add_fx(A.mol_e, mkey, me);
  if (!A.partials) return;  // forces only
  // wave sums by shuffles, then the block's waves in a fixed order
  for (int v = 0; v < kCorrVals; ++v)
    for (int m = kWaveLanes / 2; m >= 1; m >>= 1) acc[v] += __shfl_xor(acc[v], m, kWaveLanes);
  if ((threadIdx.x & (kWaveLanes - 1)) == 0)
    for (int v = 0; v < kCorrVals; ++v) red[v * (kCorrBlock / kWaveLanes) + threadIdx.x / kWaveLanes] = acc[v];
  __syncthreads();
  if (threadIdx.x < kCorrVals) {
    double t = 0.0;
    for (int w = 0; w < kCorrBlock / kWaveLanes; ++w) t += red[threadIdx.x * (kCorrBlock / kWaveLanes) + w];
    A.partials[kCorrVals * block + threadIdx.x] = t;
  }
}

// An evaluation's corrections.
struct CorrWork {
  unsigned blocks = 0;  // workgroups of the system that needs most
  std::function<CorrArgs(uint32_t)> args;
};

}  // namespace dyn

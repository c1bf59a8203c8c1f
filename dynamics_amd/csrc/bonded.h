// bonded.h — float vectors and the bonded terms of an MD step, a device
// function that the step's launches share.
//
// Reference semantics: src/bonded_forces.rs:11-200.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <functional>

#include "dyn_math.h"

namespace dyn {

struct V3 {
  float x, y, z;
};
__device__ __forceinline__ V3 v3(float x, float y, float z) { return {x, y, z}; }
__device__ __forceinline__ V3 operator+(V3 a, V3 b) { return {a.x + b.x, a.y + b.y, a.z + b.z}; }
__device__ __forceinline__ V3 operator-(V3 a, V3 b) { return {a.x - b.x, a.y - b.y, a.z - b.z}; }
__device__ __forceinline__ V3 operator*(V3 a, float s) { return {a.x * s, a.y * s, a.z * s}; }
__device__ __forceinline__ float dot(V3 a, V3 b) { return a.x * b.x + a.y * b.y + a.z * b.z; }
__device__ __forceinline__ V3 cross(V3 a, V3 b) {
  return {a.y * b.z - a.z * b.y, a.z * b.x - a.x * b.z, a.x * b.y - a.y * b.x};
}
__device__ __forceinline__ V3 ld(const float4& p) { return {p.x, p.y, p.z}; }

struct Box {
  float L[3];
};
// Reciprocal, square root and reciprocal square root by the hardware
// instructions (about 1 ulp): the integrator's constraint, rigid-body and
// bonded arithmetic needs no correctly rounded division.
__device__ __forceinline__ float hw_rcp(float x) { return __builtin_amdgcn_rcpf(x); }
__device__ __forceinline__ float hw_sqrt(float x) { return __builtin_amdgcn_sqrtf(x); }
__device__ __forceinline__ float hw_rsqrt(float x) { return __builtin_amdgcn_rsqf(x); }

// src/barostat.rs:141-170: dv − round(dv/ext)·ext.
// A displacement within half a box (most are) is its own image; the three
// correctly rounded divisions are passed over unless a lane needs them.
__device__ __forceinline__ V3 min_image(V3 d, const Box& b) {
  if (!(fabsf(d.x) < 0.49f * b.L[0] && fabsf(d.y) < 0.49f * b.L[1] && fabsf(d.z) < 0.49f * b.L[2]))
    d = {dyn_min_image_ref(d.x, b.L[0]), dyn_min_image_ref(d.y, b.L[1]), dyn_min_image_ref(d.z, b.L[2])};
  return d;
}

constexpr int kBondedBlock = 256;

struct BondedArgs {
  const float4* x;
  Box B;
  uint32_t n_dyn;
  uint32_t n_bond, n_angle, n_dihe;
  const uint32_t* bond;   // 2 per term
  const float2* bond_p;   // k, r0
  const uint32_t* angle;  // 3 per term (vertex in the middle)
  const float2* angle_p;  // k, θ0
  const uint32_t* dihe;   // 4 per term
  const float4* dihe_p;   // k, periodicity (an integer 0..6), cos(phase), sin(phase)
  int64_t* f;             // fixed point, component-major over solute atoms
  double* partials;       // 4 per block: bond, angle, dihedral energy, virial
  uint32_t nblk;          // workgroups of the system (one partial each)
};

__device__ __forceinline__ void add_f(int64_t* f, uint32_t nd, uint32_t i, V3 v) {
  atomicAdd(reinterpret_cast<unsigned long long*>(f + i), (unsigned long long)dyn_fx(v.x));
  atomicAdd(reinterpret_cast<unsigned long long*>(f + nd + i), (unsigned long long)dyn_fx(v.y));
  atomicAdd(reinterpret_cast<unsigned long long*>(f + 2 * (size_t)nd + i), (unsigned long long)dyn_fx(v.z));
}

// Harmonic bonds and angles (U = k(r − r0)², k(θ − θ0)²) and periodic
// dihedrals (U = k(1 + cos(nφ − γ)), φ the IUPAC torsion angle); one
// thread per term, fixed-point force sums.  The virial Σ r_a·F_a of each
// term is taken relative to one of its atoms (src/bonded.rs:41-46, :79-83,
// :124-130; the same sign convention for every term).  A workgroup of
// kBondedBlock threads per block of terms.
__device__ __forceinline__ void bonded_terms(const BondedArgs& A, uint32_t block) {
  __shared__ double red[4][kBondedBlock / 64];
  if (block >= A.nblk) return;  // partials exist for the system's own blocks
  const uint32_t t = block * kBondedBlock + threadIdx.x;
  double e[4] = {0.0, 0.0, 0.0, 0.0};
  const uint32_t nd = A.n_dyn;
  if (t < A.n_bond) {
    const uint32_t i = A.bond[2 * t], j = A.bond[2 * t + 1];
    const V3 d = min_image(ld(A.x[j]) - ld(A.x[i]), A.B);
    const float r = hw_sqrt(dot(d, d));
    const float2 p = A.bond_p[t];
    const float dr = r - p.y;
    const V3 fi = d * (2.0f * p.x * dr * hw_rcp(fmaxf(r, 1e-8f)));
    add_f(A.f, nd, i, fi);
    add_f(A.f, nd, j, fi * -1.0f);
    e[0] = (double)(p.x * dr * dr);
    e[3] = -(double)dot(d, fi);  // (r_i − r_j)·F_i
  } else if (t - A.n_bond < A.n_angle) {
    const uint32_t q = t - A.n_bond;
    const uint32_t i = A.angle[3 * q], j = A.angle[3 * q + 1], k = A.angle[3 * q + 2];
    const V3 b0 = min_image(ld(A.x[i]) - ld(A.x[j]), A.B);
    const V3 b2 = min_image(ld(A.x[k]) - ld(A.x[j]), A.B);
    const float l0s = dot(b0, b0), l2s = dot(b2, b2);
    if (l0s >= 1e-8f && l2s >= 1e-8f) {
      const float il0 = hw_rsqrt(l0s), il2 = hw_rsqrt(l2s);
      const V3 u0 = b0 * il0, u2 = b2 * il2;
      const float ct = fminf(1.0f, fmaxf(-1.0f, dot(u0, u2)));
      const float th = acosf(ct);
      const float ist = hw_rcp(fmaxf(hw_sqrt(1.0f - ct * ct), 1e-8f));
      const float2 p = A.angle_p[q];
      const float dth = th - p.y;
      const float dedt = 2.0f * p.x * dth;
      const V3 g0 = (u0 * ct - u2) * (il0 * ist);
      const V3 g2 = (u2 * ct - u0) * (il2 * ist);
      const V3 f0 = g0 * -dedt, f2 = g2 * -dedt;
      add_f(A.f, nd, i, f0);
      add_f(A.f, nd, k, f2);
      add_f(A.f, nd, j, (f0 + f2) * -1.0f);
      e[1] = (double)(p.x * dth * dth);
      e[3] = (double)dot(b0, f0) + (double)dot(b2, f2);
    }
  } else if (t - A.n_bond - A.n_angle < A.n_dihe) {
    const uint32_t q = t - A.n_bond - A.n_angle;
    const uint32_t i = A.dihe[4 * q], j = A.dihe[4 * q + 1], k = A.dihe[4 * q + 2],
                   l = A.dihe[4 * q + 3];
    const V3 b1 = min_image(ld(A.x[j]) - ld(A.x[i]), A.B);
    const V3 b2 = min_image(ld(A.x[k]) - ld(A.x[j]), A.B);
    const V3 b3 = min_image(ld(A.x[l]) - ld(A.x[k]), A.B);
    const V3 n1 = cross(b1, b2), n2 = cross(b2, b3);
    const float n1s = dot(n1, n1), n2s = dot(n2, n2), b2s = dot(b2, b2);
    const float b2l = hw_sqrt(b2s);
    if (n1s >= 1e-6f && n2s >= 1e-6f && b2l >= 1e-6f) {
      // cos φ, sin φ of the IUPAC torsion φ = atan2(|b2| b1·n2, n1·n2); then
      // cos nφ, sin nφ by the angle-addition recurrence and the phase by one
      // more rotation: cos(nφ − γ), sin(nφ − γ) without trigonometric calls
      const float4 p = A.dihe_p[q];
      const float y = b2l * dot(b1, n2), x = dot(n1, n2);
      const float rinv = hw_rsqrt(x * x + y * y);
      const float c1 = x * rinv, s1 = y * rinv;
      float cn = 1.0f, sn = 0.0f;
      const int nper = (int)p.y;
      for (int k = 0; k < nper; ++k) {
        const float c2 = cn * c1 - sn * s1;
        sn = sn * c1 + cn * s1;
        cn = c2;
      }
      const float cos_arg = cn * p.z + sn * p.w;   // cos(nφ − γ)
      const float sin_arg = sn * p.z - cn * p.w;   // sin(nφ − γ)
      const float dedphi = -p.x * p.y * sin_arg;
      // ∂φ/∂x_i = −|b2|/|n1|² n1, ∂φ/∂x_l = |b2|/|n2|² n2; the inner atoms
      // take the lever-arm split of the two
      const V3 gi = n1 * (-b2l * hw_rcp(n1s)), gl = n2 * (b2l * hw_rcp(n2s));
      const float ib2s = hw_rcp(b2s);
      const float ta = dot(b1, b2) * ib2s, tb = dot(b3, b2) * ib2s;
      const V3 gj = gl * tb - gi * (1.0f + ta);
      const V3 gk = gi * ta - gl * (1.0f + tb);
      add_f(A.f, nd, i, gi * -dedphi);
      add_f(A.f, nd, j, gj * -dedphi);
      add_f(A.f, nd, k, gk * -dedphi);
      add_f(A.f, nd, l, gl * -dedphi);
      e[2] = (double)(p.x * (1.0f + cos_arg));
      // relative to atom j: r_i − r_j = −b1, r_k − r_j = b2, r_l − r_j = b2 + b3
      e[3] = -(double)dot(b1, gi * -dedphi) + (double)dot(b2, gk * -dedphi) +
             (double)dot(b2 + b3, gl * -dedphi);
    }
  }
  if (!A.partials) return;  // forces only
  // wave sums by shuffles, then the block's waves in a fixed order
  for (int c = 0; c < 4; ++c)
    for (int m = 32; m >= 1; m >>= 1) e[c] += __shfl_xor(e[c], m, 64);
  if ((threadIdx.x & 63) == 0)
    for (int c = 0; c < 4; ++c) red[c][threadIdx.x / 64] = e[c];
  __syncthreads();
  if (threadIdx.x < 4) {
    double t = 0.0;
    for (int w = 0; w < kBondedBlock / 64; ++w) t += red[threadIdx.x][w];
    A.partials[4 * block + threadIdx.x] = t;
  }
}

// Bonded terms an MD step hands to its engines' evaluation.
struct SideWork {
  unsigned blocks = 0;  // workgroups of the system that needs most
  std::function<BondedArgs(uint32_t)> args;
  std::function<uint64_t*(uint32_t)> step;  // a count to advance by one before them, or none
};

}  // namespace dyn

// pme.hip — SPME reciprocal space on gfx950: fixed-point B-spline charge
// spreading, real mixed-radix (8/4/2/9/3/5) Stockham FFTs staged through LDS, the
// influence-function convolution fused into the x-axis pass with FP64 energy
// and virial reductions, and the force gather.  Replaces the `ewald` crate's
// PmeRecip (used at src/non_bonded.rs:681-795, :850-875).
#include <hip/hip_runtime.h>

#include <type_traits>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <memory>
#include <vector>

#include "bonded.h"
#include "common.h"
#include "corr.h"
#include "wave.h"
#include "dyn_math.h"
#include "pme.h"

#pragma clang fp contract(off)

namespace dyn {

bool is_235_smooth(uint32_t n) {
  if (n == 0) return false;
  for (uint32_t p : {2u, 3u, 5u})
    while (n % p == 0) n /= p;
  return n == 1;
}

// Radices of an FFT of length N, the first in the lowest four bits (0: no
// more): few stages — 8 while what is left of the twos is not 2 or 4, then 4s,
// 2; 9, 3; 5.
static uint64_t fft_plan(uint32_t N) {
  uint64_t plan = 0;
  int at = 0;
  uint32_t n = N;
  auto take = [&](uint32_t r) {
    plan |= (uint64_t)r << at;
    at += 4;
    n /= r;
  };
  while (n % 8 == 0 && (n % 16 != 0 || n % 32 == 0)) take(8);
  while (n % 4 == 0) take(4);
  while (n % 2 == 0) take(2);
  while (n % 9 == 0) take(9);
  while (n % 3 == 0) take(3);
  while (n % 5 == 0) take(5);
  if (n != 1) throw Error(DYN_ERR_ARG, fmt("grid size %u has a prime factor above 5", N));
  return plan;
}

}  // namespace dyn

using namespace dyn;

namespace {

constexpr int kFftBlock = 256;
constexpr int kFftCap = 4096;      // complex elements of a pass's LDS buffer, at most
constexpr int kFftLines = 16;      // lines per workgroup where the grid has enough of them
constexpr size_t kPlaneLds = 64u << 10;  // LDS of a plane launch and its workgroups, at most
constexpr unsigned kPlaneGroups = 256;

// Complex arithmetic on float2 (the default SPME) or double2 (the FP64
// option).
template <class C>
struct CxT;
template <>
struct CxT<float2> {
  using R = float;
  __device__ static float2 mk(float x, float y) { return make_float2(x, y); }
  static constexpr float c3 = -0.5f, s3 = 0.866025403784438647f;
  static constexpr float c51 = 0.309016994374947424f, c52 = -0.809016994374947424f;
  static constexpr float s51 = 0.951056516295153572f, s52 = 0.587785252292473129f;
  static constexpr float h = 0.707106781186547524f;  // √½; cos and sin of 40°, 80°, 160°:
  static constexpr float c91 = 0.766044443118978035f, s91 = 0.642787609686539327f;
  static constexpr float c92 = 0.173648177666930349f, s92 = 0.984807753012208059f;
  static constexpr float c94 = -0.939692620785908384f, s94 = 0.342020143325668733f;
};
template <>
struct CxT<double2> {
  using R = double;
  __device__ static double2 mk(double x, double y) { return make_double2(x, y); }
  static constexpr double c3 = -0.5, s3 = 0.866025403784438647;
  static constexpr double c51 = 0.309016994374947424, c52 = -0.809016994374947424;
  static constexpr double s51 = 0.951056516295153572, s52 = 0.587785252292473129;
  static constexpr double h = 0.707106781186547524;
  static constexpr double c91 = 0.766044443118978035, s91 = 0.642787609686539327;
  static constexpr double c92 = 0.173648177666930349, s92 = 0.984807753012208059;
  static constexpr double c94 = -0.939692620785908384, s94 = 0.342020143325668733;
};

template <class C>
__device__ __forceinline__ C cadd(C a, C b) { return CxT<C>::mk(a.x + b.x, a.y + b.y); }
template <class C>
__device__ __forceinline__ C csub(C a, C b) { return CxT<C>::mk(a.x - b.x, a.y - b.y); }
__device__ __forceinline__ float rfma(float a, float b, float c) { return __builtin_fmaf(a, b, c); }
__device__ __forceinline__ double rfma(double a, double b, double c) { return __builtin_fma(a, b, c); }
// a + b·s
template <class C>
__device__ __forceinline__ C cfma(C b, typename CxT<C>::R s, C a) {
  return CxT<C>::mk(rfma(b.x, s, a.x), rfma(b.y, s, a.y));
}
template <class C>
__device__ __forceinline__ C cscale(C a, typename CxT<C>::R s) { return CxT<C>::mk(a.x * s, a.y * s); }
// multiply by SIGN·i
template <int SIGN, class C>
__device__ __forceinline__ C cmul_si(C a) {
  return SIGN < 0 ? CxT<C>::mk(a.y, -a.x) : CxT<C>::mk(-a.y, a.x);
}
// v · w where w = tw (SIGN = −1) or conj(tw) (SIGN = +1)
template <int SIGN, class C>
__device__ __forceinline__ C ctw(C v, C t) {
  const typename CxT<C>::R ti = SIGN < 0 ? t.y : -t.y;
  return CxT<C>::mk(rfma(v.x, t.x, -(v.y * ti)), rfma(v.x, ti, v.y * t.x));
}

template <int SIGN, class C>
__device__ __forceinline__ void dft2(C* v) {
  const C a = v[0], b = v[1];
  v[0] = cadd(a, b);
  v[1] = csub(a, b);
}
template <int SIGN, class C>
__device__ __forceinline__ void dft4(C* v) {
  const C s02 = cadd(v[0], v[2]), d02 = csub(v[0], v[2]);
  const C s13 = cadd(v[1], v[3]), d13 = cmul_si<SIGN>(csub(v[1], v[3]));
  v[0] = cadd(s02, s13);
  v[2] = csub(s02, s13);
  v[1] = cadd(d02, d13);
  v[3] = csub(d02, d13);
}
template <int SIGN, class C>
__device__ __forceinline__ void dft3(C* v) {
  const C t = cadd(v[1], v[2]);
  const C d = cmul_si<SIGN>(csub(v[1], v[2]));
  const C a = cfma(t, CxT<C>::c3, v[0]);
  v[0] = cadd(v[0], t);
  v[1] = cfma(d, CxT<C>::s3, a);
  v[2] = cfma(d, -CxT<C>::s3, a);
}
template <int SIGN, class C>
__device__ __forceinline__ void dft5(C* v) {
  const auto c1 = CxT<C>::c51, c2 = CxT<C>::c52, s1 = CxT<C>::s51, s2 = CxT<C>::s52;
  const C t1 = cadd(v[1], v[4]), t2 = cadd(v[2], v[3]);
  const C d1 = csub(v[1], v[4]), d2 = csub(v[2], v[3]);
  const C a1 = cfma(t1, c1, cfma(t2, c2, v[0]));
  const C a2 = cfma(t1, c2, cfma(t2, c1, v[0]));
  const C b1 = cmul_si<SIGN>(cfma(d1, s1, cscale(d2, s2)));
  const C b2 = cmul_si<SIGN>(cfma(d1, s2, cscale(d2, -s1)));
  v[0] = cadd(v[0], cadd(t1, t2));
  v[1] = cadd(a1, b1);
  v[4] = csub(a1, b1);
  v[2] = cadd(a2, b2);
  v[3] = csub(a2, b2);
}

template <int SIGN, class C>
__device__ __forceinline__ void dft8(C* v) {
  const auto h = CxT<C>::h;
  C e[4] = {v[0], v[2], v[4], v[6]}, o[4] = {v[1], v[3], v[5], v[7]};
  dft4<SIGN>(e);
  dft4<SIGN>(o);
  const C i1 = cmul_si<SIGN>(o[1]), i3 = cmul_si<SIGN>(o[3]);
  o[1] = cadd(o[1], i1);  // times √½: · e^{SIGN·iπ/4}
  o[2] = cmul_si<SIGN>(o[2]);
  o[3] = csub(i3, o[3]);  // times √½: · e^{SIGN·3iπ/4}
  v[0] = cadd(e[0], o[0]);
  v[4] = csub(e[0], o[0]);
  v[1] = cfma(o[1], h, e[1]);
  v[5] = cfma(o[1], -h, e[1]);
  v[2] = cadd(e[2], o[2]);
  v[6] = csub(e[2], o[2]);
  v[3] = cfma(o[3], h, e[3]);
  v[7] = cfma(o[3], -h, e[3]);
}
template <int SIGN, class C>
__device__ __forceinline__ void dft9(C* v) {
  using R = typename CxT<C>::R;
  const R sg = SIGN < 0 ? R(-1) : R(1);
  C c[3][3];
#pragma unroll
  for (int q = 0; q < 3; ++q) {
    c[q][0] = v[q];
    c[q][1] = v[q + 3];
    c[q][2] = v[q + 6];
    dft3<SIGN>(c[q]);
  }
  auto mul = [&](C z, R wc, R ws) { return CxT<C>::mk(rfma(z.x, wc, -(z.y * (sg * ws))), rfma(z.x, sg * ws, z.y * wc)); };
  c[1][1] = mul(c[1][1], CxT<C>::c91, CxT<C>::s91);
  c[1][2] = mul(c[1][2], CxT<C>::c92, CxT<C>::s92);
  c[2][1] = mul(c[2][1], CxT<C>::c92, CxT<C>::s92);
  c[2][2] = mul(c[2][2], CxT<C>::c94, CxT<C>::s94);
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    C o[3] = {c[0][k], c[1][k], c[2][k]};
    dft3<SIGN>(o);
    v[k] = o[0];
    v[k + 3] = o[1];
    v[k + 6] = o[2];
  }
}

// The reciprocal fast_div takes (within an ulp: no correctly rounded
// division, whose latency a small pass would show).
__device__ __forceinline__ float fast_rcp(int d) { return __builtin_amdgcn_rcpf((float)d); }

// x / d for 0 ≤ x < 2²² by a float reciprocal and one correction step.
__device__ __forceinline__ int fast_div(int x, int d, float rd) {
  int q = (int)((float)x * rd);
  const int rem = x - q * d;
  if (rem < 0) --q;
  else if (rem >= d) ++q;
  return q;
}

// One radix-R Stockham stage of nl lines of length N in LDS, element n of
// line l at a[n·S + l]: consecutive threads take consecutive lines, so a
// wave's LDS accesses are contiguous, and the index arithmetic is paid once
// per R points.  Ns: length of the sub-transforms so far, M = N/Ns.  The
// twiddle index r·k·(M/R) stays below N.
template <int SIGN, int R, class C>
__device__ __forceinline__ void fft_stage(const C* __restrict__ a, C* __restrict__ b, int nl, int S,
                                          int N, int Ns, int M, const C* __restrict__ tw) {
  const int NR = N / R, tws = M / R;
  const float rnl = fast_rcp(nl), rNs = fast_rcp(Ns);
  const int total = nl * NR;
  for (int i = threadIdx.x; i < total; i += blockDim.x) {
    const int j = fast_div(i, nl, rnl);
    const int l = i - j * nl;
    const C* src = a + j * S + l;
    C v[R];
#pragma unroll
    for (int r = 0; r < R; ++r) v[r] = src[r * NR * S];
    int d = j * R;
    if (Ns > 1) {
      const int q = fast_div(j, Ns, rNs), k = j - q * Ns;
      d = q * Ns * R + k;
#pragma unroll
      for (int r = 1; r < R; ++r) v[r] = ctw<SIGN>(v[r], tw[r * k * tws]);
    }
    if constexpr (R == 8) dft8<SIGN>(v);
    else if constexpr (R == 4) dft4<SIGN>(v);
    else if constexpr (R == 2) dft2<SIGN>(v);
    else if constexpr (R == 9) dft9<SIGN>(v);
    else if constexpr (R == 3) dft3<SIGN>(v);
    else dft5<SIGN>(v);
    C* dst = b + d * S + l;
#pragma unroll
    for (int r = 0; r < R; ++r) dst[r * Ns * S] = v[r];
  }
  __syncthreads();
}

// Stockham autosort FFT of nl lines held in LDS (fft_stage's layout), plan
// as fft_plan packs it.  Returns the buffer holding the (natural-order)
// result.  A line sees the same stages and arithmetic in every kernel and
// grouping.
template <int SIGN, class C>
__device__ __forceinline__ C* lds_fft(C* a, C* b, int nl, int S, int N, uint64_t plan,
                                      const C* __restrict__ tw) {
  int Ns = 1, M = N;
  for (; plan != 0; plan >>= 4) {
    const int R = (int)(plan & 15u);
    if (R == 8) fft_stage<SIGN, 8>(a, b, nl, S, N, Ns, M, tw), M /= 8;
    else if (R == 4) fft_stage<SIGN, 4>(a, b, nl, S, N, Ns, M, tw), M /= 4;
    else if (R == 2) fft_stage<SIGN, 2>(a, b, nl, S, N, Ns, M, tw), M /= 2;
    else if (R == 9) fft_stage<SIGN, 9>(a, b, nl, S, N, Ns, M, tw), M /= 9;
    else if (R == 3) fft_stage<SIGN, 3>(a, b, nl, S, N, Ns, M, tw), M /= 3;
    else fft_stage<SIGN, 5>(a, b, nl, S, N, Ns, M, tw), M /= 5;
    C* t = a;
    a = b;
    b = t;
    Ns *= R;
  }
  return a;
}

// The transforms.  The charge grid and the potential are real, so the
// spectrum holds only kz = 0 … Kz/2 (nh values a line), which halves the y
// and x passes: two z lines (y = 2p and 2p + 1 of an x plane, a pair) are the
// real and imaginary parts of one complex transform, taken apart after it
// and put together before the inverse one.  Spectrum element (x, y, kz) lies
// at (x·Ky + y)·nh + kz.
//
// Bound: memory and LDS traffic, and launch latency on small grids.  A
// workgroup of a y or x pass takes about 16 consecutive kz (128 bytes) of
// every element of its lines: whole cache lines, which with 4 consecutive
// values were fetched by four workgroups on different XCDs.  Radix 8 and 9
// stages halve the LDS exchanges of radix 4 and 3.  128³ alone: z pass 12 µs, y 14,
// x with the convolution 17 (complex radix-4 passes of 4 lines: 12 to 28, and 37).
struct FftGeom {
  int K[3];
  int nh;  // kz values of the spectrum: K[2]/2 + 1
  int np;  // z-line pairs per x plane
  int L;   // lines (pairs, kz columns) per workgroup
  uint64_t plan[3];
};
static_assert(sizeof(FftGeom) == 48, "FftGeom has no padding");

// Sizes known to be the same in every lane (an argument pack in memory would
// keep them, and all index arithmetic on them, in vector registers).
__device__ __forceinline__ int uni(int v) { return __builtin_amdgcn_readfirstlane(v); }
__device__ __forceinline__ FftGeom uni(const FftGeom& g) {
  FftGeom u;
  for (int a = 0; a < 3; ++a) u.K[a] = uni(g.K[a]);
  u.nh = uni(g.nh);
  u.np = uni(g.np);
  u.L = uni(g.L);
  for (int a = 0; a < 3; ++a)
    u.plan[a] = (uint64_t)(uint32_t)uni((int)(g.plan[a] >> 32)) << 32 | (uint32_t)uni((int)g.plan[a]);
  return u;
}

// A pair's line spectra from the transform X of its combination: A = (X(k) +
// conj X(−k))/2, B = (X(k) − conj X(−k))/2i.
template <class C>
__device__ __forceinline__ void pair_split(C x, C y, C& A, C& B) {
  using R = typename CxT<C>::R;
  A = CxT<C>::mk(R(0.5) * (x.x + y.x), R(0.5) * (x.y - y.y));
  B = CxT<C>::mk(R(0.5) * (x.y + y.y), R(0.5) * (y.x - x.x));
}

// Puts A(k) + iB(k) of a pair into column l of the LDS lines, at k and, from
// the conjugates, at N − k (the values at k = 0 and N/2 are real).
template <class C>
__device__ __forceinline__ void pair_join(C* __restrict__ a, int S, int l, int k, int N, C A, C B) {
  if (k == 0 || 2 * k == N) {
    a[k * S + l] = CxT<C>::mk(A.x, B.x);
    return;
  }
  a[k * S + l] = CxT<C>::mk(A.x - B.y, A.y + B.x);
  a[(N - k) * S + l] = CxT<C>::mk(A.x + B.y, B.x - A.y);
}

// put(e, load(e)) for the workgroup's e in [0, n), a thread's next kAhead
// loads in flight together (one after another they cost a memory latency
// each: most of a pass on the smaller grids).
constexpr int kAhead = 8;
template <class Load, class Put>
__device__ __forceinline__ void for_loaded(int n, Load&& load, Put&& put) {
  for (int e0 = threadIdx.x; e0 < n; e0 += kAhead * blockDim.x) {
    decltype(load(0)) v[kAhead];
#pragma unroll
    for (int u = 0; u < kAhead; ++u) {
      const int e = e0 + u * blockDim.x;
      if (e < n) v[u] = load(e);
    }
#pragma unroll
    for (int u = 0; u < kAhead; ++u) {
      const int e = e0 + u * blockDim.x;
      if (e < n) put(e, v[u]);
    }
  }
}

template <class C>
__device__ __forceinline__ void load_tw(C* __restrict__ dst, const C* __restrict__ src, int n) {
  for (int k = threadIdx.x; k < n; k += blockDim.x) dst[k] = src[k];
}

// Fixed-point charges of nl z-line pairs from pair q0 on into LDS lines.
template <class C>
__device__ __forceinline__ void load_pairs(C* __restrict__ a, int S, const int64_t* __restrict__ grid_fx,
                                           const FftGeom& g, int q0, int nl) {
  using R = typename CxT<C>::R;
  const int N = g.K[2];
  const float rN = fast_rcp(N), rnp = fast_rcp(g.np);
  for_loaded(2 * nl * N, [&](int e) -> int64_t {
    const int l2 = fast_div(e, N, rN), n = e - l2 * N;
    const int q = q0 + (l2 >> 1), x = fast_div(q, g.np, rnp), y = 2 * (q - x * g.np) + (l2 & 1);
    return y < g.K[1] ? grid_fx[((size_t)x * g.K[1] + y) * N + n] : 0;
  }, [&](int e, int64_t v) {
    const int l2 = fast_div(e, N, rN), n = e - l2 * N;
    reinterpret_cast<R*>(a)[2 * (n * S + (l2 >> 1)) + (l2 & 1)] = (R)((double)v * (1.0 / DYN_GRID_FX_SCALE));
  });
}
template <class C>
__device__ __forceinline__ void store_pairs(const C* __restrict__ a, int S,
                                            typename CxT<C>::R* __restrict__ phi, const FftGeom& g,
                                            int q0, int nl) {
  using R = typename CxT<C>::R;
  const int N = g.K[2];
  const float rN = fast_rcp(N), rnp = fast_rcp(g.np);
  for (int e = threadIdx.x; e < 2 * nl * N; e += blockDim.x) {
    const int l2 = fast_div(e, N, rN), n = e - l2 * N, l = l2 >> 1;
    const int q = q0 + l, x = fast_div(q, g.np, rnp), y = 2 * (q - x * g.np) + (l2 & 1);
    if (y < g.K[1])
      phi[((size_t)x * g.K[1] + y) * N + n] = reinterpret_cast<const R*>(a)[2 * (n * S + l) + (l2 & 1)];
  }
}

// LDS row stride of nl z-line pairs (odd: the loads along z write down a
// column of LDS).
__host__ __device__ inline int pair_stride(int nl) { return nl | 1; }

// z pass of g.L pairs per workgroup: charges to spectrum (FWD) or spectrum
// to potential.
template <bool FWD, class C>
__device__ __forceinline__ void
k_fft_z(C* __restrict__ spec, const int64_t* __restrict__ grid_fx, typename CxT<C>::R* __restrict__ phi,
        FftGeom geom, const C* __restrict__ tw) {
  const FftGeom g = uni(geom);
  extern __shared__ __align__(16) unsigned char smem_raw[];
  const int q0 = blockIdx.x * g.L, pairs = g.K[0] * g.np;
  if (q0 >= pairs) return;  // beyond this system's lines
  const int N = g.K[2], nl = min(g.L, pairs - q0), S = pair_stride(g.L);
  C* A = reinterpret_cast<C*>(smem_raw);
  C* B = A + N * S;
  C* s_tw = B + N * S;
  load_tw(s_tw, tw, N);
  const float rnh = fast_rcp(g.nh), rnp = fast_rcp(g.np);
  if (FWD) {
    load_pairs(A, S, grid_fx, g, q0, nl);
    __syncthreads();
    const C* X = lds_fft<-1>(A, B, nl, S, N, g.plan[2], s_tw);
    for (int e = threadIdx.x; e < nl * g.nh; e += blockDim.x) {
      const int l = fast_div(e, g.nh, rnh), k = e - l * g.nh;
      const int q = q0 + l, x = fast_div(q, g.np, rnp), y = 2 * (q - x * g.np);
      C a, b;
      pair_split(X[k * S + l], X[(k ? N - k : 0) * S + l], a, b);
      C* out = spec + ((size_t)x * g.K[1] + y) * g.nh + k;
      out[0] = a;
      if (y + 1 < g.K[1]) out[g.nh] = b;
    }
  } else {
    struct Two { C a, b; };
    for_loaded(nl * g.nh, [&](int e) {
      const int l = fast_div(e, g.nh, rnh), k = e - l * g.nh;
      const int q = q0 + l, x = fast_div(q, g.np, rnp), y = 2 * (q - x * g.np);
      const C* in = spec + ((size_t)x * g.K[1] + y) * g.nh + k;
      return Two{in[0], y + 1 < g.K[1] ? in[g.nh] : CxT<C>::mk(0, 0)};
    }, [&](int e, const Two& v) {
      const int l = fast_div(e, g.nh, rnh);
      pair_join(A, S, l, e - l * g.nh, N, v.a, v.b);
    });
    __syncthreads();
    const C* X = lds_fft<+1>(A, B, nl, S, N, g.plan[2], s_tw);
    store_pairs(X, S, phi, g, q0, nl);
  }
}

// y pass of g.L consecutive kz of an x plane per workgroup, in place.
template <int SIGN, class C>
__device__ __forceinline__ void
k_fft_y(C* __restrict__ spec, FftGeom geom, const C* __restrict__ tw) {
  const FftGeom g = uni(geom);
  extern __shared__ __align__(16) unsigned char smem_raw[];
  if (g.K[0] == 0) return;  // takes no part: no tiles to divide by either
  const int tiles = (g.nh + g.L - 1) / g.L;
  const int x = blockIdx.x / tiles, k0 = (blockIdx.x - x * tiles) * g.L;
  if (x >= g.K[0]) return;  // beyond this system's lines
  const int N = g.K[1], nl = min(g.L, g.nh - k0);
  C* A = reinterpret_cast<C*>(smem_raw);
  C* B = A + N * g.L;
  C* s_tw = B + N * g.L;
  load_tw(s_tw, tw, N);
  C* base = spec + (size_t)x * N * g.nh + k0;
  const float rnl = fast_rcp(nl);
  for_loaded(N * nl, [&](int e) {
    const int n = fast_div(e, nl, rnl), l = e - n * nl;
    return base[(size_t)n * g.nh + l];
  }, [&](int e, C v) { A[e] = v; });
  __syncthreads();
  const C* X = lds_fft<SIGN>(A, B, nl, nl, N, g.plan[1], s_tw);
  for (int e = threadIdx.x; e < N * nl; e += blockDim.x) {
    const int n = fast_div(e, nl, rnl), l = e - n * nl;
    base[(size_t)n * g.nh + l] = X[e];
  }
}

// The z and y passes of one direction in one launch, a workgroup per x
// plane in LDS: the same arithmetic as the separate passes, a launch and a
// round trip of the spectrum less (pme_run says where).
constexpr int kPlaneBlock = 512;  // (1024: 3% faster alone, but 28,000-site MD steps, which run it beside
                                  // the pair kernel, 7% slower)
template <bool FWD>
__device__ __forceinline__ void
k_fft_plane(float2* __restrict__ spec, const int64_t* __restrict__ grid_fx, float* __restrict__ phi,
            FftGeom geom, const float2* __restrict__ twy,
            const float2* __restrict__ twz) {
  const FftGeom g = uni(geom);
  extern __shared__ __align__(16) unsigned char smem_raw[];
  const int x = blockIdx.x;
  if (x >= g.K[0]) return;  // beyond this system's planes
  const int NY = g.K[1], NZ = g.K[2], nh = g.nh, S = pair_stride(g.np);
  const int cap = max(NZ * S, NY * nh);
  float2* A = reinterpret_cast<float2*>(smem_raw);
  float2* B = A + cap;
  float2* s_twy = B + cap;
  float2* s_twz = s_twy + NY;
  load_tw(s_twy, twy, NY);
  load_tw(s_twz, twz, NZ);
  const float rnh = fast_rcp(nh);
  float2* plane = spec + (size_t)x * NY * nh;
  if (FWD) {
    load_pairs(A, S, grid_fx, g, x * g.np, g.np);
    __syncthreads();
    float2* X = lds_fft<-1>(A, B, g.np, S, NZ, g.plan[2], s_twz);
    float2* Y = X == A ? B : A;
    for (int e = threadIdx.x; e < g.np * nh; e += blockDim.x) {
      const int l = fast_div(e, nh, rnh), k = e - l * nh;
      float2 a, b;
      pair_split(X[k * S + l], X[(k ? NZ - k : 0) * S + l], a, b);
      Y[2 * l * nh + k] = a;
      if (2 * l + 1 < NY) Y[(2 * l + 1) * nh + k] = b;
    }
    __syncthreads();
    const float2* Z = lds_fft<-1>(Y, X, nh, nh, NY, g.plan[1], s_twy);
    for (int e = threadIdx.x; e < NY * nh; e += blockDim.x) plane[e] = Z[e];
  } else {
    for_loaded(NY * nh, [&](int e) { return plane[e]; }, [&](int e, float2 v) { A[e] = v; });
    __syncthreads();
    float2* Y = lds_fft<+1>(A, B, nh, nh, NY, g.plan[1], s_twy);
    float2* X = Y == A ? B : A;
    for (int e = threadIdx.x; e < g.np * nh; e += blockDim.x) {
      const int l = fast_div(e, nh, rnh), k = e - l * nh;
      pair_join(X, S, l, k, NZ, Y[2 * l * nh + k],
                2 * l + 1 < NY ? Y[(2 * l + 1) * nh + k] : make_float2(0.f, 0.f));
    }
    __syncthreads();
    const float2* Z = lds_fft<+1>(X, Y, g.np, S, NZ, g.plan[2], s_twz);
    store_pairs(Z, S, phi, g, x * g.np, g.np);
  }
}

// Energy and virial in units of 2⁻³², then what each leaves in units of 2⁻⁶⁴.
constexpr int kConvSums = 4;
// The wave's four sums, sum v in the lanes of row v (16 lanes): a swap of
// half-waves leaves one value in each half, a swap of rows one in each row, four
// rotations add a row.  (24 shuffles otherwise.)
__device__ __forceinline__ uint64_t wave_sums(const uint64_t (&v)[kConvSums]) {
  auto two = [](uint64_t a) { return make_uint2((uint32_t)a, (uint32_t)(a >> 32)); };
  auto one = [](uint32_t lo, uint32_t hi) { return (uint64_t)hi << 32 | lo; };
  auto half = [&](uint64_t a, uint64_t b) {
    const uint2 x = two(a), y = two(b);
    const auto lo = __builtin_amdgcn_permlane32_swap(x.x, y.x, false, false);
    const auto hi = __builtin_amdgcn_permlane32_swap(x.y, y.y, false, false);
    return one(lo[0], hi[0]) + one(lo[1], hi[1]);
  };
  const uint2 x = two(half(v[0], v[2])), y = two(half(v[1], v[3]));
  const auto lo = __builtin_amdgcn_permlane16_swap(x.x, y.x, false, false);
  const auto hi = __builtin_amdgcn_permlane16_swap(x.y, y.y, false, false);
  uint64_t s = one(lo[0], hi[0]) + one(lo[1], hi[1]);
  auto turn = [&](auto ctrl) {
    const uint2 t = two(s);
    s += one((uint32_t)__builtin_amdgcn_mov_dpp((int)t.x, decltype(ctrl)::value, 0xf, 0xf, true),
             (uint32_t)__builtin_amdgcn_mov_dpp((int)t.y, decltype(ctrl)::value, 0xf, 0xf, true));
  };
  turn(std::integral_constant<int, 0x128>{});  // row_ror:8, 4, 2, 1
  turn(std::integral_constant<int, 0x124>{});
  turn(std::integral_constant<int, 0x122>{});
  turn(std::integral_constant<int, 0x121>{});
  return s;
}
// Adds x and what its rounding to 2⁻³² leaves to the two sums, in the same
// units but each kFxBias too large (taken off once per workgroup; sums wrap).
// x is clamped as every fixed-point value is.
constexpr uint64_t kFxBias = 0x4338000000000000LL;  // bits of 1.5·2⁵²
__device__ __forceinline__ void add_fx128(double x, uint64_t& hi, uint64_t& lo) {
  x = fmin(fmax(x, -(double)DYN_FX_CLAMP), (double)DYN_FX_CLAMP);
  const double d = __builtin_fma(x, DYN_FX_SCALE, 0x1.8p52);
  const double rest = __builtin_fma(x, DYN_FX_SCALE, 0x1.8p52 - d);
  hi += (uint64_t)__double_as_longlong(d);
  lo += (uint64_t)__double_as_longlong(__builtin_fma(rest, DYN_FX_SCALE, 0x1.8p52));
}
struct ConvArgs {
  float invL[3];
  double pi2_over_b2;  // π²/β²
};

// x pass fused with the convolution, g.L consecutive (y, kz) columns per
// workgroup: forward FFT along x, multiply by G(m) (accumulating ½G|F[Q]|² and
// its virial weight), inverse FFT along x.  A kz inside the half spectrum
// stands for −kz too.  Each point's energy is computed in f64 and summed in
// fixed point, so the sums do not depend on the grouping of the lines; two
// words (2⁻³² and what that rounds away, 2⁻⁶⁴), since most of a fine grid's points
// are smaller than 2⁻³³ (with one word two charges of 0.1 on 64³ lost 1.8e-5 of
// their energy; with two and the sums over a wave by wave_sums 7.8 µs on 64³ and
// 17.4 on 128³, with one word and shuffles 8.1 and 17.6).
template <class C>
__device__ __forceinline__ void
k_fft_conv_x(C* __restrict__ spec, FftGeom geom, const C* __restrict__ tw,
             const typename CxT<C>::R* __restrict__ G, ConvArgs V, int64_t* __restrict__ partials) {
  const FftGeom g = uni(geom);
  extern __shared__ __align__(16) unsigned char smem_raw[];
  __shared__ uint64_t red[kConvSums][kFftBlock / 64];
  const int N = g.K[0], cols = g.K[1] * g.nh, c0 = blockIdx.x * g.L;
  if (c0 >= cols) return;  // beyond this system's lines
  const int nl = min(g.L, cols - c0);
  C* A = reinterpret_cast<C*>(smem_raw);
  C* B = A + N * g.L;
  C* s_tw = B + N * g.L;
  load_tw(s_tw, tw, N);
  const float rnl = fast_rcp(nl), rnh = fast_rcp(g.nh);
  for_loaded(N * nl, [&](int e) {
    const int n = fast_div(e, nl, rnl), l = e - n * nl;
    return spec[(size_t)n * cols + c0 + l];
  }, [&](int e, C v) { A[e] = v; });
  __syncthreads();
  C* X = lds_fft<-1>(A, B, nl, nl, N, g.plan[0], s_tw);
  uint64_t sum[kConvSums] = {0, 0, 0, 0};
  for_loaded(N * nl, [&](int e) {
    const int n = fast_div(e, nl, rnl);
    return G[(size_t)n * cols + c0 + e - n * nl];
  }, [&](int e, typename CxT<C>::R gv) {
    const int n = fast_div(e, nl, rnl), c = c0 + e - n * nl;
    C v = X[e];
    const int my = fast_div(c, g.nh, rnh), mz = c - my * g.nh;
    const double fx = (n <= N / 2 ? n : n - N) * (double)V.invL[0];
    const double fy = (my <= g.K[1] / 2 ? my : my - g.K[1]) * (double)V.invL[1];
    const double fz = mz * (double)V.invL[2];
    const double msq = fx * fx + fy * fy + fz * fz;
    const double wz = mz == 0 || 2 * mz == g.K[2] ? 0.5 : 1.0;
    const double en = wz * (double)gv * ((double)v.x * (double)v.x + (double)v.y * (double)v.y);
    add_fx128(en, sum[0], sum[2]);
    add_fx128(en * (1.0 - 2.0 * V.pi2_over_b2 * msq), sum[1], sum[3]);
    v.x *= gv;
    v.y *= gv;
    X[e] = v;
  });
  const uint64_t w = wave_sums(sum);
  if ((threadIdx.x & 15) == 0) red[(threadIdx.x >> 4) & 3][threadIdx.x / 64] = w;
  __syncthreads();
  if (threadIdx.x < kConvSums) {
    uint64_t s = 0;
    for (int k = 0; k < kFftBlock / 64; ++k) s += red[threadIdx.x][k];
    partials[kConvSums * blockIdx.x + threadIdx.x] = (int64_t)(s - (uint64_t)(N * nl) * kFxBias);
  }
  const C* Z = lds_fft<+1>(X, X == A ? B : A, nl, nl, N, g.plan[0], s_tw);
  for (int e = threadIdx.x; e < N * nl; e += blockDim.x) {
    const int n = fast_div(e, nl, rnl), l = e - n * nl;
    spec[(size_t)n * cols + c0 + l] = Z[e];
  }
}

struct SplineArgs {
  int K[3];
  float sc[3];    // K/L
  double scd[3];  // K/L in double (FP64 option)
};

constexpr int kBrickBlock = 256;
constexpr int kRowY = kBrick + 1, kRowX = kBrick * kRowY + 1;  // LDS strides of a brick (bank spread)

// Per charge: its home brick (the brick of its base grid point) and a rank
// in it; the charge goes to slot rank of the brick's fixed-capacity list
// (cap slots per brick).  A full brick sets *status |= status_bit (the caller
// enlarges the lists and evaluates again).  The rank order depends on atomic
// timing; the brick sums are integers, so the spread grid does not.
__device__ __forceinline__ void k_pme_bin(const float4* __restrict__ xyzq, uint32_t n, BinArgs B) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  pme_bin_charge(B, i < n ? xyzq[i] : make_float4(0.f, 0.f, 0.f, 0.f), i < n);
}

// k_pme_bin from pinned host memory, leaving the charges on the device too.
__device__ __forceinline__ void k_pme_take(const float4* __restrict__ h, uint32_t n,
                                           float4* __restrict__ xyzq, BinArgs B) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  const float4 p = i < n ? h[i] : make_float4(0.f, 0.f, 0.f, 0.f);
  if (i < n) xyzq[i] = p;
  pme_bin_charge(B, p, i < n);
}

// Forces (n floats), energy, virial and the list status to pinned host memory.
__device__ __forceinline__ void k_pme_out(const float* __restrict__ f, uint32_t n,
                                          const double* __restrict__ res,
                                          const unsigned int* __restrict__ status,
                                          float* __restrict__ h_f, double* __restrict__ h_rep) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) h_f[i] = f[i];
  if (i < 2u) h_rep[i] = res[i];
  if (i == 2u) h_rep[2] = (double)*status;
}

// Home bricks along one axis whose charges can reach the points [lo, hi]
// (lo a brick start): a charge with base point k0 covers k0 − ORDER + 1 … k0
// (mod K), so k0 runs over lo … hi + ORDER − 1 (mod K): the bricks of
// lo … e1 (e1 < K), then, past the wrap, those of 0 … e2 that come before
// lo's brick.  At most 3 bricks (ORDER ≤ 5, 8-point bricks).
struct HomeRange {
  int b0, n1, n;  // first brick, bricks before the wrap, bricks in all
  __device__ int brick(int j) const { return j < n1 ? b0 + j : j - n1; }
};
template <int ORDER>
__device__ __forceinline__ HomeRange home_bricks(int lo, int hi, int K) {
  const int len = min(hi - lo + ORDER, K);
  const int last = lo + len - 1;
  HomeRange r;
  r.b0 = lo / kBrick;
  r.n1 = min(last, K - 1) / kBrick - r.b0 + 1;
  const int e2 = last - K;  // last point past the wrap (< 0: none)
  r.n = r.n1 + (e2 >= 0 && r.b0 > 0 ? min(e2 / kBrick, r.b0 - 1) + 1 : 0);
  return r;
}

// Grid point j of the ORDER points that end at base point k0 (mod K): one
// conditional addition (an integer remainder, 84 a charge, was most of the
// spread's and the gather's instructions).
template <int ORDER>
__device__ __forceinline__ int stencil_point(int k0, int j, int K) {
  const int g = k0 - ORDER + 1 + j;
  return g < 0 ? g + K : g;
}

// One workgroup per brick: every charge of the reaching home bricks adds its
// stencil points inside the brick to an LDS brick (int64 LDS adds of the
// same fixed-point values the replay sums), which is then stored once.  The
// home bricks' charge lists are walked as one flattened index space.
//
// Bound: the latency of the dependent loads (counts, then charges) on small
// grids, instruction issue on large ones.  So a lane per home brick reads the
// counts, the lists hold the charges themselves and no integer remainder is
// taken per point: 24,000 charges, order 5, on 80³ 28.9 -> 12.4 µs; order 4
// keeps its time (21,000 on 64³ 12.4 µs, 192,000 on 128³ 39).  Tried and slower: a thread
// per charge and x point (order 5 18.6 µs), or per charge, x and y with the
// weights in LDS (17.1); two 32-bit LDS adds for each 64-bit one (13.7, 43 at
// 128³).
//
// The corrections (C, n_corr workgroups after the n_brick of the bricks) and
// the bonded terms (B, the workgroups after them) of the evaluation ride in the
// same launch: all three are chains of memory latencies.  28,000 sites: 12.4 µs
// alone, 16.2 with the bonded terms, which made the launch before this one
// 5.1 µs longer.
template <int ORDER, class R>
__device__ __forceinline__ void
k_pme_spread(SplineArgs S, uint32_t nbx, uint32_t nby, uint32_t nbz, const uint32_t* __restrict__ count,
             const float4* __restrict__ items, uint32_t cap, int64_t* __restrict__ grid,
             const CorrArgs& C, const BondedArgs& B, uint32_t n_brick, uint32_t n_corr) {
  static_assert(kBrickBlock == kBondedBlock && kBrickBlock == kCorrBlock, "one block size");
  if (blockIdx.x >= n_brick) {
    const uint32_t k = blockIdx.x - n_brick;
    if (k < n_corr) corr_terms(C, k);
    else bonded_terms(B, k - n_corr);
    return;
  }
  __shared__ unsigned long long acc[kBrick * kRowX];
  __shared__ uint32_t s_c0[32], s_end[32];
  const uint32_t b = blockIdx.x;
  if (b >= nbx * nby * nbz) return;  // beyond this system's bricks
  const int bz = (int)(b % nbz), by = (int)((b / nbz) % nby), bx = (int)(b / (nbz * nby));
  const int lo[3] = {bx * kBrick, by * kBrick, bz * kBrick};
  const int hi[3] = {min(lo[0] + kBrick, S.K[0]) - 1, min(lo[1] + kBrick, S.K[1]) - 1,
                     min(lo[2] + kBrick, S.K[2]) - 1};
  if (threadIdx.x < 32) {
    // at most 27 home bricks; the rest of the 32 entries are empty
    const HomeRange hx = home_bricks<ORDER>(lo[0], hi[0], S.K[0]);
    const HomeRange hy = home_bricks<ORDER>(lo[1], hi[1], S.K[1]);
    const HomeRange hz = home_bricks<ORDER>(lo[2], hi[2], S.K[2]);
    const int q = threadIdx.x, ix = q / 9, iy = q / 3 - 3 * ix, iz = q - 3 * (q / 3);
    uint32_t h = 0, c = 0;
    if (ix < hx.n && iy < hy.n && iz < hz.n) {
      h = ((uint32_t)hx.brick(ix) * nby + (uint32_t)hy.brick(iy)) * nbz + (uint32_t)hz.brick(iz);
      c = min(count[h], cap);
    }
    uint32_t end = c;
    for (int off = 1; off < 32; off <<= 1) {
      const uint32_t u = __shfl_up(end, off, 32);
      if (q >= off) end += u;
    }
    s_end[q] = end;
    s_c0[q] = h * cap + c - end;  // (mod 2³²: entry t of the whole lies at s_c0 + t)
  }
  for (int k = threadIdx.x; k < kBrick * kRowX; k += kBrickBlock) acc[k] = 0ull;
  __syncthreads();
  const uint32_t total = s_end[31];
  for (uint32_t t = threadIdx.x; t < total; t += kBrickBlock) {
    uint32_t q = 0;  // the first list that ends beyond t
#pragma unroll
    for (uint32_t step = 16; step >= 1; step >>= 1)
      if (s_end[q + step - 1] <= t) q += step;
    const float4 p = items[(size_t)(uint32_t)(s_c0[q] + t)];
    if (p.w == 0.0f) continue;
    int k0[3];
    R th[3][ORDER], dth[ORDER];
    const R xs[3] = {(R)p.x, (R)p.y, (R)p.z};
    for (int a = 0; a < 3; ++a) {
      R w;
      frac_coord<R>(xs[a], std::is_same<R, float>::value ? (R)S.sc[a] : (R)S.scd[a], S.K[a], k0[a], w);
      dyn_bspline<ORDER, R>(w, th[a], dth);
    }
    for (int jx = 0; jx < ORDER; ++jx) {
      const int gx = stencil_point<ORDER>(k0[0], jx, S.K[0]);
      if (gx < lo[0] || gx > hi[0]) continue;
      const R qx = (R)p.w * th[0][jx];
      unsigned long long* const row = acc + (gx - lo[0]) * kRowX;
      for (int jy = 0; jy < ORDER; ++jy) {
        const int gy = stencil_point<ORDER>(k0[1], jy, S.K[1]);
        if (gy < lo[1] || gy > hi[1]) continue;
        const R qxy = qx * th[1][jy];
        for (int jz = 0; jz < ORDER; ++jz) {
          const int gz = stencil_point<ORDER>(k0[2], jz, S.K[2]);
          if (gz < lo[2] || gz > hi[2]) continue;
          const R v = qxy * th[2][jz];
          atomicAdd(row + (gy - lo[1]) * kRowY + (gz - lo[2]),
                    (unsigned long long)dyn_fx_d((double)v, DYN_GRID_FX_SCALE));
        }
      }
    }
  }
  __syncthreads();
  for (int k = threadIdx.x; k < kBrick * kBrick * kBrick; k += kBrickBlock) {
    const int x = lo[0] + k / (kBrick * kBrick), y = lo[1] + (k / kBrick) % kBrick,
              z = lo[2] + k % kBrick;
    if (x <= hi[0] && y <= hi[1] && z <= hi[2])
      grid[((size_t)x * S.K[1] + y) * S.K[2] + z] = (int64_t)acc[(x - lo[0]) * kRowX + (y - lo[1]) * kRowY + (z - lo[2])];
  }
}

template <class R>
__device__ __forceinline__ int64_t fx_of(R f) {
  if constexpr (std::is_same<R, float>::value) return dyn_fx(f);
  else return dyn_fx64(f);
}

// Order 4: four lanes per charge (a quad), lane g its x point g; the quad's
// sums are added by DPP and lane c stores component c.  Bound: the
// latency of a charge's dependent loads (charge, its grid points, its force
// row), so that small systems gain from more and shorter chains: 1,500
// charges 7.0 -> 4.7 µs, 21,000 8.9 -> 7.2, 32 systems of 100,000 together
// 20.9 -> 14.4.  Order 5 takes a thread per charge: five x points leave a quad
// uneven (24,000 charges: 13.1 µs, one thread each 10.0).
constexpr int gather_lanes(int order) { return order == 4 ? 4 : 1; }
constexpr int kGatherBlock = 256;
template <class R>
__device__ __forceinline__ R quad_sum(R v);
template <>
__device__ __forceinline__ float quad_sum(float v) {
  v += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0xB1, 0xf, 0xf, true));
  return v + __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x4E, 0xf, 0xf, true));
}
template <>
__device__ __forceinline__ double quad_sum(double v) {
  v += __shfl_xor(v, 1, 64);
  return v + __shfl_xor(v, 2, 64);
}
template <int ORDER, class R>
__device__ __forceinline__ void k_pme_gather(const float4* __restrict__ xyzq, uint32_t n, SplineArgs S,
                             const R* __restrict__ phi, const uint32_t* __restrict__ site,
                             int64_t* __restrict__ fx, int comp_major, uint32_t nsites,
                             float* __restrict__ fout, float fscale,
                             const int64_t* __restrict__ partials, int nbp,
                             double* __restrict__ res, uint32_t* __restrict__ brick_count,
                             uint32_t nbk) {
  // partials: the convolution's per-workgroup energy and virial sums in
  // fixed point (nbp workgroups, kConvSums words each)
  constexpr bool F32 = std::is_same<R, float>::value;
  // the spread has read the brick counts: clear them for the next binning
  if (brick_count)
    for (uint32_t k = blockIdx.x * blockDim.x + threadIdx.x; k < nbk; k += gridDim.x * blockDim.x)
      brick_count[k] = 0u;
  if (res && blockIdx.x == 0) {
    // the first workgroup also sums the convolution's energy and virial
    // partials
    __shared__ uint64_t red[kConvSums][kGatherBlock / 64];
    uint64_t sum[kConvSums] = {0, 0, 0, 0};
    for (int b = threadIdx.x; b < nbp; b += kGatherBlock)
      for (int v = 0; v < kConvSums; ++v) sum[v] += (uint64_t)partials[kConvSums * b + v];
    const uint64_t w = wave_sums(sum);
    if ((threadIdx.x & 15) == 0) red[(threadIdx.x >> 4) & 3][threadIdx.x / 64] = w;
    __syncthreads();
    if (threadIdx.x < 2) {
      uint64_t hi = 0, lo = 0;
      for (int k = 0; k < kGatherBlock / 64; ++k) {
        hi += red[threadIdx.x][k];
        lo += red[threadIdx.x + 2][k];
      }
      res[threadIdx.x] = ((double)(int64_t)hi + (double)(int64_t)lo * DYN_FX_INV_SCALE) * DYN_FX_INV_SCALE;
    }
  }
  constexpr int kLanes = gather_lanes(ORDER);
  const uint32_t i = (blockIdx.x * kGatherBlock + threadIdx.x) / kLanes;
  const int g = kLanes == 1 ? 0 : (int)(threadIdx.x & 3u);
  if (i >= n) return;  // (whole quads)
  const float4 p = xyzq[i];
  const uint32_t s = site ? site[i] : 0u;
  R f[3] = {R(0), R(0), R(0)};
  if (p.w != 0.0f) {
    int k0[3];
    R th[3][ORDER], dth[3][ORDER];
    const R xs[3] = {(R)p.x, (R)p.y, (R)p.z};
    R sc[3];
    for (int a = 0; a < 3; ++a) {
      sc[a] = F32 ? (R)S.sc[a] : (R)S.scd[a];
      R w;
      frac_coord<R>(xs[a], sc[a], S.K[a], k0[a], w);
      dyn_bspline<ORDER, R>(w, th[a], dth[a]);
    }
    R sx = R(0), sy = R(0), sz = R(0);
#pragma unroll
    for (int j0 = 0; j0 < ORDER; j0 += kLanes) {
      const int jx = j0 + g;
      R tx = th[0][j0], dx = dth[0][j0];
#pragma unroll
      for (int j = 1; j < kLanes; ++j) {
        tx = g == j ? th[0][j0 + j] : tx;
        dx = g == j ? dth[0][j0 + j] : dx;
      }
      const int gx = stencil_point<ORDER>(k0[0], jx, S.K[0]);
      for (int jy = 0; jy < ORDER; ++jy) {
        const int gy = stencil_point<ORDER>(k0[1], jy, S.K[1]);
        const R* row = phi + ((size_t)gx * S.K[1] + gy) * S.K[2];
        const R txy = tx * th[1][jy];
        const R dxy = dx * th[1][jy];
        const R tdy = tx * dth[1][jy];
        for (int jz = 0; jz < ORDER; ++jz) {
          const int gz = stencil_point<ORDER>(k0[2], jz, S.K[2]);
          const R ph = row[gz];
          if constexpr (F32) {
            sx = dyn_fmaf(ph, dxy * th[2][jz], sx);
            sy = dyn_fmaf(ph, tdy * th[2][jz], sy);
            sz = dyn_fmaf(ph, txy * dth[2][jz], sz);
          } else {
            sx = fma(ph, dxy * th[2][jz], sx);
            sy = fma(ph, tdy * th[2][jz], sy);
            sz = fma(ph, txy * dth[2][jz], sz);
          }
        }
      }
    }
    if (kLanes == 4) {
      sx = quad_sum(sx);
      sy = quad_sum(sy);
      sz = quad_sum(sz);
    }
    f[0] = -(R)p.w * sc[0] * sx * (R)fscale;
    f[1] = -(R)p.w * sc[1] * sy * (R)fscale;
    f[2] = -(R)p.w * sc[2] * sz * (R)fscale;
  }
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    if (kLanes == 4 && g != c) continue;
    if (!site) {
      fout[3 * (size_t)i + c] = (float)f[c];
    } else if (comp_major & 2) {
      // every site has one charge: no other thread of this pass touches it
      // (a second pass over the same sites is a later launch)
      fx[(size_t)c * nsites + s] += fx_of(f[c]);
    } else {
      atomicAdd(reinterpret_cast<unsigned long long*>(fx + (comp_major ? (size_t)c * nsites + s : 3 * (size_t)s + c)),
                (unsigned long long)fx_of(f[c]));
    }
  }
}

// Geometry of the pass along an axis over nsys systems: kFftLines lines per
// workgroup (128 bytes of consecutive kz), fewer where the lines are long or
// the launch would have fewer than 256 workgroups; kz tiles of a y pass of
// about equal width.
FftGeom pass_geom(const PmeCore& c, int axis, uint32_t nsys, size_t elem) {
  const uint32_t* K = c.K;
  FftGeom g;
  for (int a = 0; a < 3; ++a) g.K[a] = (int)K[a];
  g.nh = (int)K[2] / 2 + 1;
  g.np = ((int)K[1] + 1) / 2;
  const int N = g.K[axis];
  const int64_t lines = axis == 2 ? (int64_t)g.K[0] * g.np : (int64_t)(axis == 1 ? g.K[0] : g.K[1]) * g.nh;
  const int fit = std::max(1, (int)(kFftCap * sizeof(float2) / elem) / N);
  int L = std::min(kFftLines, fit);
  while (L > 4 && lines * std::max<uint32_t>(nsys, 1) / L < 256) L /= 2;
  if (axis == 1) {
    const int tiles = std::max(1, (g.nh + L / 4) / L);
    L = std::min((g.nh + tiles - 1) / tiles, fit);
  }
  g.L = L;
  for (int a = 0; a < 3; ++a) g.plan[a] = c.plan[a];
  return g;
}
unsigned pass_groups(const FftGeom& g, int axis) {
  if (axis == 1) return (unsigned)(g.K[0] * ((g.nh + g.L - 1) / g.L));
  const int lines = axis == 2 ? g.K[0] * g.np : g.K[1] * g.nh;
  return (unsigned)((lines + g.L - 1) / g.L);
}
size_t pass_lds(const FftGeom& g, int axis, size_t elem) {
  const size_t N = (size_t)g.K[axis], S = (size_t)(axis == 2 ? pair_stride(g.L) : g.L);
  return (2 * N * S + N) * elem;
}
size_t plane_lds(const FftGeom& g) {
  const size_t cap = std::max((size_t)g.K[2] * pair_stride(g.np), (size_t)g.K[1] * g.nh);
  return (2 * cap + g.K[1] + g.K[2]) * sizeof(float2);
}

}  // namespace

namespace dyn {

void PmeCore::init(int dev, hipStream_t s, Profiler* p, const uint32_t k[3], const float l[3],
                   float b, int ord, bool fp64) {
  f64 = fp64;
  device = dev;
  stream = s;
  prof = p;
  for (int a = 0; a < 3; ++a) {
    DYN_REQUIRE(k[a] >= (uint32_t)ord && k[a] <= 1024, "grid size %u out of range [%d, 1024]",
                k[a], ord);
    DYN_REQUIRE(is_235_smooth(k[a]), "grid size %u must factor into 2, 3 and 5", k[a]);
    K[a] = k[a];
    plan[a] = fft_plan(k[a]);
  }
  DYN_REQUIRE(ord == 4 || ord == 5, "B-spline order must be 4 or 5 (got %d)", ord);
  DYN_REQUIRE(b > 0.f && std::isfinite(b), "beta must be > 0");
  order = ord;
  beta = b;
  ngrid = (size_t)K[0] * K[1] * K[2];
  nspec = (size_t)K[0] * K[1] * (K[2] / 2 + 1);
  grid_fx.reserve(ngrid);
  for (int a = 0; a < 3; ++a) nbk[a] = (K[a] + kBrick - 1) / kBrick;
  const size_t nb = (size_t)nbk[0] * nbk[1] * nbk[2];
  brick_count.reserve(nb + 1);
  cap_brick = 0;
  status.reserve(1);
  // the binning pass counts into zeroed counts; the gather clears them again
  DYN_HIP(hipMemsetAsync(brick_count.p, 0, sizeof(uint32_t) * (nb + 1), stream));
  DYN_HIP(hipMemsetAsync(status.p, 0, sizeof(unsigned int), stream));
  if (f64) {
    cgrid64.reserve(nspec + (ngrid + 1) / 2);
    G64.reserve(nspec);
  } else {
    cgrid.reserve(nspec + (ngrid + 1) / 2);
    G.reserve(nspec);
  }
  for (int a = 0; a < 3; ++a) {
    std::vector<float2> t(K[a]);
    std::vector<double2> t64(K[a]);
    for (uint32_t m = 0; m < K[a]; ++m) {
      const double ang = -2.0 * M_PI * (double)m / (double)K[a];
      t[m] = make_float2((float)std::cos(ang), (float)std::sin(ang));
      t64[m] = make_double2(std::cos(ang), std::sin(ang));
    }
    if (f64) {
      tw64[a].reserve(K[a]);
      DYN_HIP(hipMemcpyAsync(tw64[a].p, t64.data(), sizeof(double2) * K[a], hipMemcpyHostToDevice,
                             stream));
    } else {
      tw[a].reserve(K[a]);
      DYN_HIP(hipMemcpyAsync(tw[a].p, t.data(), sizeof(float2) * K[a], hipMemcpyHostToDevice,
                             stream));
    }
    DYN_HIP(hipStreamSynchronize(stream));
  }
  // energy and virial partials of every x-pass workgroup (at most one per line)
  partials.reserve(kConvSums * (size_t)K[1] * (K[2] / 2 + 1));
  res_dev.reserve(2);
  set_moduli();
  set_box(l);
}

// Influence function at every point of the half spectrum (set_box), in double:
// G(m) = exp(−π²|m|²/β²)/(π V |m|²) · Π_a |b_a(m_a)|², m_a = m'_a/L_a with
// m'_a the signed index; G(0) = 0.  bsq: 1/|b_a|² per axis, axes concatenated.
template <class R>
__global__ void __launch_bounds__(256)
k_pme_influence(R* __restrict__ G, const double* __restrict__ bsq, uint32_t K0, uint32_t K1,
                uint32_t K2, double il0, double il1, double il2, double inv_piv, double pi2_b2) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  const uint32_t nh = K2 / 2 + 1;
  if (i >= (size_t)K0 * K1 * nh) return;
  const uint32_t mz = (uint32_t)(i % nh);
  const size_t r = i / nh;
  const uint32_t my = (uint32_t)(r % K1), mx = (uint32_t)(r / K1);
  const double fx = (mx <= K0 / 2 ? (double)mx : (double)mx - K0) * il0;
  const double fy = (my <= K1 / 2 ? (double)my : (double)my - K1) * il1;
  const double fz = (double)mz * il2;
  const double msq = fx * fx + fy * fy + fz * fz;
  double val = 0.0;
  if (msq > 0)
    val = exp(-pi2_b2 * msq) * inv_piv / msq * bsq[mx] * bsq[K0 + my] * bsq[K0 + K1 + mz];
  G[i] = (R)val;
}

// |b(m)|⁻² per axis (Essmann eq. 4.4) from the order-n cardinal B-spline at
// the integers; a vanishing modulus (odd order at m = K/2) takes the mean of
// its neighbours.
void PmeCore::set_moduli() {
  std::vector<double> Mn(order + 1, 0.0);
  if (order == 4) {
    Mn[1] = 1.0 / 6;
    Mn[2] = 4.0 / 6;
    Mn[3] = 1.0 / 6;
  } else {
    Mn[1] = 1.0 / 24;
    Mn[2] = 11.0 / 24;
    Mn[3] = 11.0 / 24;
    Mn[4] = 1.0 / 24;
  }
  std::vector<double> all;
  for (int a = 0; a < 3; ++a) {
    const int Ka = (int)K[a];
    std::vector<double> mod(Ka);
    for (int m = 0; m < Ka; ++m) {
      double re = 0, im = 0;
      for (int k = 0; k <= order - 2; ++k) {
        const double ang = 2.0 * M_PI * (double)m * k / Ka;
        re += Mn[k + 1] * std::cos(ang);
        im += Mn[k + 1] * std::sin(ang);
      }
      mod[m] = re * re + im * im;
    }
    for (int m = 0; m < Ka; ++m)
      if (mod[m] < 1e-7) mod[m] = 0.5 * (mod[(m - 1 + Ka) % Ka] + mod[(m + 1) % Ka]);
    for (int m = 0; m < Ka; ++m) all.push_back(1.0 / mod[m]);
  }
  bsq.reserve(all.size());
  DYN_HIP(hipMemcpyAsync(bsq.p, all.data(), sizeof(double) * all.size(), hipMemcpyHostToDevice,
                         stream));
  DYN_HIP(hipStreamSynchronize(stream));
}

// A new box: the influence function is recomputed on the device (the grid
// and its FFT plan stay; the reference rebuilds its PmeRecip instead,
// src/non_bonded.rs:850-875).
void PmeCore::set_box(const float l[3]) {
  for (int a = 0; a < 3; ++a) {
    DYN_REQUIRE(l[a] > 0.f && std::isfinite(l[a]), "box length must be > 0");
    L[a] = l[a];
  }
  const double V = (double)L[0] * L[1] * L[2];
  const double b2 = (double)beta * beta;
  const unsigned grid = (unsigned)((nspec + 255) / 256);
  const double il0 = 1.0 / (double)L[0], il1 = 1.0 / (double)L[1], il2 = 1.0 / (double)L[2];
  if (f64)
    hipLaunchKernelGGL((k_pme_influence<double>), dim3(grid), dim3(256), 0, stream, G64.p, bsq.p,
                       K[0], K[1], K[2], il0, il1, il2, 1.0 / (M_PI * V), M_PI * M_PI / b2);
  else
    hipLaunchKernelGGL((k_pme_influence<float>), dim3(grid), dim3(256), 0, stream, G.p, bsq.p,
                       K[0], K[1], K[2], il0, il1, il2, 1.0 / (M_PI * V), M_PI * M_PI / b2);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) throw Error(DYN_ERR_HIP, fmt("launch of k_pme_influence: %s", hipGetErrorString(e)));
}

// Brick lists for n charges: three times the mean per brick plus 64, in
// multiples of 32 (grown further when a brick overflows).
void PmeCore::ensure_cap(uint32_t n) {
  const size_t nb = (size_t)nbk[0] * nbk[1] * nbk[2];
  const double mean = (double)n * (double)(kBrick * kBrick * kBrick) / (double)ngrid;
  const uint32_t want = ((uint32_t)(3.0 * mean) + 64 + 31) & ~31u;
  if (want > cap_brick) cap_brick = want;
  brick_items.reserve(nb * cap_brick);
}

BinArgs PmeCore::bin_args(unsigned int* st, unsigned int bit) const {
  BinArgs B;
  std::memset(&B, 0, sizeof B);
  for (int a = 0; a < 3; ++a) {
    B.K[a] = (int)K[a];
    B.sc[a] = (float)((double)K[a] / (double)L[a]);
    B.nb[a] = nbk[a];
  }
  B.count = brick_count.p;
  B.items = brick_items.p;
  B.cap = cap_brick;
  B.status = st ? st : status.p;
  B.status_bit = st ? bit : 1u;
  return B;
}
void PmeCore::grow() {
  cap_brick = std::max<uint32_t>(64, 2 * cap_brick);
  brick_items.reserve((size_t)nbk[0] * nbk[1] * nbk[2] * cap_brick);
}

// One SPME evaluation per system of the pass, each stage one launch for all
// of them (per precision and B-spline order present).  A system with a null
// core takes part in no stage (its packs describe empty work: no charges, no
// bricks, no lines, no result); neither does it in the launches of the other
// precision or order.
void pme_run(const BatchRun& R, Profiler& prof, const PmeRun* runs, int tag, const CorrWork* corr,
             const SideWork* side) {
  const uint32_t ns = R.n;
  std::vector<SplineArgs> S(ns);
  std::vector<FftGeom> gz(ns), gy(ns), gx(ns);
  unsigned g_n = 1, g_b = 1, bz = 1, by = 1, bx = 1;
  size_t shz = 0, shy = 0, shx = 0;
  bool any = false, ord[2][2] = {{false, false}, {false, false}}, prec[2] = {false, false};
  for (uint32_t i = 0; i < ns; ++i) {
    const PmeRun& r = runs[i];
    std::memset(&S[i], 0, sizeof S[i]);
    std::memset(&gz[i], 0, sizeof gz[i]);
    gy[i] = gx[i] = gz[i];
    if (!r.core) continue;
    const PmeCore& c = *r.core;
    any = true;
    ord[c.f64][c.order == 5] = true;
    prec[c.f64] = true;
    for (int a = 0; a < 3; ++a) {
      S[i].K[a] = (int)c.K[a];
      S[i].sc[a] = (float)((double)c.K[a] / (double)c.L[a]);
      S[i].scd[a] = (double)c.K[a] / (double)c.L[a];
    }
    r.core->ensure_cap(r.n);
    const size_t el = c.f64 ? sizeof(double2) : sizeof(float2);
    gz[i] = pass_geom(c, 2, ns, el);
    gy[i] = pass_geom(c, 1, ns, el);
    gx[i] = pass_geom(c, 0, ns, el);
    g_n = std::max(g_n, grid_all(r.n, 256));
    g_b = std::max(g_b, c.nbk[0] * c.nbk[1] * c.nbk[2]);
    bz = std::max(bz, pass_groups(gz[i], 2));
    by = std::max(by, pass_groups(gy[i], 1));
    bx = std::max(bx, pass_groups(gx[i], 0));
    shz = std::max(shz, pass_lds(gz[i], 2, el));
    shy = std::max(shy, pass_lds(gy[i], 1, el));
    shx = std::max(shx, pass_lds(gx[i], 0, el));
  }
  if (!any) return;
  auto on = [&](uint32_t i) { return runs[i].core != nullptr; };
  auto nq = [&](uint32_t i) { return on(i) ? runs[i].n : 0u; };
  auto nb = [&](uint32_t i, int a) { return on(i) ? runs[i].core->nbk[a] : 0u; };
  auto cp = [&](uint32_t i) { return runs[i].core; };
  // this system in the launch of precision F64 (and order ORDER when given)
  auto mine = [&](uint32_t i, bool f64, int order) {
    return on(i) && cp(i)->f64 == f64 && (order == 0 || cp(i)->order == order);
  };
  // every grid point belongs to exactly one brick and is stored by it, so
  // the grid needs no clearing
  {
    Profiler::Scope ps(prof, "pme_spread");
    bool bin_any = false;
    for (uint32_t i = 0; i < ns; ++i) bin_any = bin_any || (on(i) && !runs[i].binned);
    if (bin_any)
      launch<k_pme_bin>(R, "k_pme_bin", tag, g_n, 256, 0, [&](uint32_t i) {
        const bool o = on(i) && !runs[i].binned;
        BinArgs B;
        std::memset(&B, 0, sizeof B);
        if (o) B = cp(i)->bin_args(runs[i].status, runs[i].status_bit);
        return args<k_pme_bin>(runs[i].xyzq, o ? nq(i) : 0u, B);
      });
    // (the first of the pass's spread launches takes the corrections and the
    // bonded terms)
    unsigned n_corr = corr ? corr->blocks : 0u, n_bond = side ? side->blocks : 0u;
    auto spread = [&](auto F, const char* name, bool f64, int order) {
      const unsigned nc = n_corr, nt = n_bond;
      n_corr = n_bond = 0u;
      const unsigned g = g_b + nc + nt;
      launch<decltype(F)::value, kBrickBlock>(R, name, tag, g, kBrickBlock, 0, [&](uint32_t i) {
        const bool m = mine(i, f64, order);
        CorrArgs Cr;
        std::memset(&Cr, 0, sizeof Cr);
        if (nc) Cr = corr->args(i);
        BondedArgs B;
        std::memset(&B, 0, sizeof B);
        if (nt) B = side->args(i);
        return args<decltype(F)::value>(S[i], m ? nb(i, 0) : 0u, m ? nb(i, 1) : 0u,
                                        m ? nb(i, 2) : 0u,
                                        m ? (const uint32_t*)cp(i)->brick_count.p : nullptr,
                                        m ? (const float4*)cp(i)->brick_items.p : nullptr,
                                        m ? cp(i)->cap_brick : 0u,
                                        m ? cp(i)->grid_fx.p : nullptr, Cr, B, g_b, nc);
      });
    };
#define DYN_SPREAD(O, T, F64)                                                                    \
  if (ord[F64][O == 5])                                                                          \
    spread(std::integral_constant<decltype(&k_pme_spread<O, T>), &k_pme_spread<O, T>>{},         \
           "k_pme_spread<" #O ", " #T ">", F64, O);
    DYN_SPREAD(4, float, 0)
    DYN_SPREAD(5, float, 0)
    DYN_SPREAD(4, double, 1)
    DYN_SPREAD(5, double, 1)
#undef DYN_SPREAD
  }
#define DYN_IC(F) std::integral_constant<decltype(&F), &F>{}
  struct TF {
    using type = float2;
  };
  struct TD {
    using type = double2;
  };
  // an FFT pass over the systems of one precision: C = float2 or double2
  auto spec_of = [&](uint32_t i, auto Ctag) -> typename decltype(Ctag)::type* {
    if constexpr (std::is_same<typename decltype(Ctag)::type, double2>::value) return cp(i)->cgrid64.p;
    else return cp(i)->cgrid.p;
  };
  auto phi_of = [&](uint32_t i, auto Ctag) {
    using Rt = typename CxT<typename decltype(Ctag)::type>::R;
    return reinterpret_cast<Rt*>(spec_of(i, Ctag) + cp(i)->nspec);
  };
  auto tw_of = [&](uint32_t i, int axis, auto Ctag) -> const typename decltype(Ctag)::type* {
    if constexpr (std::is_same<typename decltype(Ctag)::type, double2>::value) return cp(i)->tw64[axis].p;
    else return cp(i)->tw[axis].p;
  };
  auto none = [](FftGeom g) {  // no lines in any pass
    g.K[0] = g.K[1] = 0;
    g.L = std::max(g.L, 1);
    return g;
  };
  auto fft_z = [&](auto F, auto Ctag, const char* name) {
    using C = typename decltype(Ctag)::type;
    using Rt = typename CxT<C>::R;
    launch<decltype(F)::value, kFftBlock>(R, name, tag, bz, kFftBlock, shz, [&](uint32_t i) {
      const bool m = mine(i, std::is_same<C, double2>::value, 0);
      return args<decltype(F)::value>(m ? spec_of(i, Ctag) : (C*)nullptr,
                                      m ? (const int64_t*)cp(i)->grid_fx.p : nullptr,
                                      m ? phi_of(i, Ctag) : (Rt*)nullptr, m ? gz[i] : none(gz[i]),
                                      m ? tw_of(i, 2, Ctag) : (const C*)nullptr);
    });
  };
  auto fft_y = [&](auto F, auto Ctag, const char* name) {
    using C = typename decltype(Ctag)::type;
    launch<decltype(F)::value, kFftBlock>(R, name, tag, by, kFftBlock, shy, [&](uint32_t i) {
      const bool m = mine(i, std::is_same<C, double2>::value, 0);
      return args<decltype(F)::value>(m ? spec_of(i, Ctag) : (C*)nullptr, m ? gy[i] : none(gy[i]),
                                      m ? tw_of(i, 1, Ctag) : (const C*)nullptr);
    });
  };
  auto conv = [&](auto F, auto Ctag, const char* name) {
    using C = typename decltype(Ctag)::type;
    constexpr bool F64 = std::is_same<C, double2>::value;
    launch<decltype(F)::value, kFftBlock>(R, name, tag, bx, kFftBlock, shx, [&](uint32_t i) {
      const bool m = mine(i, F64, 0);
      ConvArgs Cv;
      std::memset(&Cv, 0, sizeof Cv);
      const typename CxT<C>::R* G = nullptr;
      if (m) {
        for (int a = 0; a < 3; ++a) Cv.invL[a] = 1.0f / cp(i)->L[a];
        Cv.pi2_over_b2 = M_PI * M_PI / ((double)cp(i)->beta * cp(i)->beta);
        if constexpr (F64) G = cp(i)->G64.p;
        else G = cp(i)->G.p;
      }
      return args<decltype(F)::value>(m ? spec_of(i, Ctag) : (C*)nullptr, m ? gx[i] : none(gx[i]),
                                      m ? tw_of(i, 0, Ctag) : (const C*)nullptr, G, Cv,
                                      m ? cp(i)->partials.p : nullptr);
    });
  };
  // the z and y passes of each direction as one plane launch, where the
  // planes are few (a launch saved: 64³ 10 µs against 13 and a launch gap,
  // 80³ 14.3 against 15.3) and their LDS leaves room for other kernels' workgroups;
  // many or large planes are as fast or faster as two passes (16 grids of
  // 45³: 18.6 against 16.6; 128³: 26 against 28 alone, 102 against 52 beside the pair
  // kernel)
  bool planes = prec[0];
  size_t shp = 0;
  unsigned bp = 1, groups = 0;
  for (uint32_t i = 0; i < ns; ++i) {
    if (!mine(i, false, 0)) continue;
    const size_t s = plane_lds(gz[i]);
    groups += cp(i)->K[0];
    planes = planes && s <= kPlaneLds && groups <= kPlaneGroups;
    shp = std::max(shp, s);
    bp = std::max(bp, cp(i)->K[0]);
  }
  auto plane = [&](auto F, const char* name) {
    launch<decltype(F)::value, kPlaneBlock>(R, name, tag, bp, kPlaneBlock, shp, [&](uint32_t i) {
      const bool m = mine(i, false, 0);
      return args<decltype(F)::value>(m ? spec_of(i, TF{}) : (float2*)nullptr,
                                      m ? (const int64_t*)cp(i)->grid_fx.p : nullptr,
                                      m ? phi_of(i, TF{}) : (float*)nullptr, m ? gz[i] : none(gz[i]),
                                      m ? tw_of(i, 1, TF{}) : (const float2*)nullptr,
                                      m ? tw_of(i, 2, TF{}) : (const float2*)nullptr);
    });
  };
  if (prec[0]) {
    if (planes) {
      Profiler::Scope ps(prof, "pme_fft_zy_fwd");
      plane(DYN_IC((k_fft_plane<true>)), "k_fft_plane fwd");
    } else {
      { Profiler::Scope ps(prof, "pme_fft_z_fwd");
        fft_z(DYN_IC((k_fft_z<true, float2>)), TF{}, "k_fft_z fwd"); }
      { Profiler::Scope ps(prof, "pme_fft_y_fwd");
        fft_y(DYN_IC((k_fft_y<-1, float2>)), TF{}, "k_fft_y fwd"); }
    }
    { Profiler::Scope ps(prof, "pme_fft_x_conv");
      conv(DYN_IC((k_fft_conv_x<float2>)), TF{}, "k_fft_conv_x"); }
    if (planes) {
      Profiler::Scope ps(prof, "pme_fft_yz_inv");
      plane(DYN_IC((k_fft_plane<false>)), "k_fft_plane inv");
    } else {
      { Profiler::Scope ps(prof, "pme_fft_y_inv");
        fft_y(DYN_IC((k_fft_y<1, float2>)), TF{}, "k_fft_y inv"); }
      { Profiler::Scope ps(prof, "pme_fft_z_inv");
        fft_z(DYN_IC((k_fft_z<false, float2>)), TF{}, "k_fft_z inv"); }
    }
  }
  if (prec[1]) {
    { Profiler::Scope ps(prof, "pme_fft_z_fwd");
      fft_z(DYN_IC((k_fft_z<true, double2>)), TD{}, "k_fft_z fwd f64"); }
    { Profiler::Scope ps(prof, "pme_fft_y_fwd");
      fft_y(DYN_IC((k_fft_y<-1, double2>)), TD{}, "k_fft_y fwd f64"); }
    { Profiler::Scope ps(prof, "pme_fft_x_conv");
      conv(DYN_IC((k_fft_conv_x<double2>)), TD{}, "k_fft_conv_x f64"); }
    { Profiler::Scope ps(prof, "pme_fft_y_inv");
      fft_y(DYN_IC((k_fft_y<1, double2>)), TD{}, "k_fft_y inv f64"); }
    { Profiler::Scope ps(prof, "pme_fft_z_inv");
      fft_z(DYN_IC((k_fft_z<false, double2>)), TD{}, "k_fft_z inv f64"); }
  }
  {
    Profiler::Scope ps(prof, "pme_gather");
    auto gather = [&](auto F, auto Ctag, int order) {
      const unsigned gg = g_n * (256 / kGatherBlock) * (unsigned)gather_lanes(order);
      using C = typename decltype(Ctag)::type;
      constexpr bool F64 = std::is_same<C, double2>::value;
      launch<decltype(F)::value, kGatherBlock>(R, "k_pme_gather",
                                               tag * 4 + (F64 ? 2 : 0) + (order == 5), gg,
                                               kGatherBlock, 0, [&](uint32_t i) {
        const bool m = mine(i, F64, order);
        const typename CxT<C>::R* phi = nullptr;
        if (m) phi = phi_of(i, Ctag);
        return args<decltype(F)::value>(runs[i].xyzq, m ? nq(i) : 0u, S[i], phi, runs[i].site,
                                        runs[i].fx, runs[i].comp_major, runs[i].nsites,
                                        runs[i].f_out, runs[i].fscale,
                                        m ? (const int64_t*)cp(i)->partials.p : nullptr,
                                        m ? (int)pass_groups(gx[i], 0) : 0,
                                        m ? runs[i].res : nullptr,
                                        m ? cp(i)->brick_count.p : nullptr,
                                        m ? nb(i, 0) * nb(i, 1) * nb(i, 2) : 0u);
      });
    };
    if (ord[0][0]) gather(DYN_IC((k_pme_gather<4, float>)), TF{}, 4);
    if (ord[0][1]) gather(DYN_IC((k_pme_gather<5, float>)), TF{}, 5);
    if (ord[1][0]) gather(DYN_IC((k_pme_gather<4, double>)), TD{}, 4);
    if (ord[1][1]) gather(DYN_IC((k_pme_gather<5, double>)), TD{}, 5);
  }
#undef DYN_IC
}

}  // namespace dyn

// ---------------------------------------------------------------------------
// Standalone PmeRecip replacement
// ---------------------------------------------------------------------------
struct dyn_pme {
  std::string err;
  int device = 0;
  hipStream_t stream = nullptr;
  Profiler prof;
  PmeCore core;
  DevBuf<float4> xyzq;
  DevBuf<float> fout;
  PinnedBuf<float4> h_xyzq;
  bool computed = false;
  ~dyn_pme() {
    if (stream) (void)hipStreamDestroy(stream);
  }
};

extern "C" int dyn_pme_create(dyn_pme** out, int device, uint32_t nx, uint32_t ny, uint32_t nz,
                              float lx, float ly, float lz, float alpha, uint32_t order) {
  try {
    DYN_REQUIRE(out != nullptr, "out is null");
    *out = nullptr;
    int ndev = 0;
    DYN_HIP(hipGetDeviceCount(&ndev));
    DYN_REQUIRE(device >= 0 && device < ndev, "device %d not present (%d devices)", device, ndev);
    std::unique_ptr<dyn_pme> p(new dyn_pme());
    p->device = device;
    DeviceGuard g(device);
    DYN_HIP(hipStreamCreateWithFlags(&p->stream, hipStreamNonBlocking));
    p->prof.stream = p->stream;
    const uint32_t K[3] = {nx, ny, nz};
    const float L[3] = {lx, ly, lz};
    p->core.init(device, p->stream, &p->prof, K, L, alpha, (int)order, false);
    *out = p.release();
    return DYN_OK;
  } catch (const Error& e) {
    set_global_error(e.what());
    return e.code;
  } catch (const std::exception& e) {
    set_global_error(e.what());
    return DYN_ERR_HIP;
  }
}

extern "C" void dyn_pme_destroy(dyn_pme* pme) {
  if (!pme) return;
  try {
    DeviceGuard g(pme->device);
    delete pme;
  } catch (...) {
  }
}

extern "C" const char* dyn_pme_last_error(const dyn_pme* pme) {
  return pme ? pme->err.c_str() : dyn_global_last_error();
}

extern "C" int dyn_pme_forces_and_virial(dyn_pme* pme, uint32_t n, const float* pos,
                                         const float* q, float* f_out, double* energy,
                                         double* virial) {
  if (!pme) {
    set_global_error("null handle");
    return DYN_ERR_ARG;
  }
  DYN_API_BODY(pme, {
    DeviceGuard g(pme->device);
    DYN_REQUIRE(n == 0 || (pos && q), "null positions or charges");
    const size_t nn = std::max<uint32_t>(n, 1);
    pme->xyzq.reserve(nn);
    pme->fout.reserve(3 * nn);
    pme->h_xyzq.reserve(nn + 2);
    // four running sums of q²: one would be a chain of additions
    double qs[4] = {0.0, 0.0, 0.0, 0.0};
    int bad = 0;
    for (uint32_t i = 0; i < n; ++i) {
      const float x = pos[3 * (size_t)i], y = pos[3 * (size_t)i + 1], z = pos[3 * (size_t)i + 2], c = q[i];
      // (a product with zero is zero unless a factor is not finite)
      bad |= (x * 0.0f + y * 0.0f) + (z * 0.0f + c * 0.0f) != 0.0f;
      pme->h_xyzq.p[i] = make_float4(x, y, z, c);
      qs[i & 3] += (double)c * (double)c;
    }
    if (bad)
      for (uint32_t i = 0; i < n; ++i)
        DYN_REQUIRE(std::isfinite(pos[3 * (size_t)i]) && std::isfinite(pos[3 * (size_t)i + 1]) &&
                        std::isfinite(pos[3 * (size_t)i + 2]) && std::isfinite(q[i]),
                    "non-finite input at charge %u", i);
    const double q2 = (qs[0] + qs[1]) + (qs[2] + qs[3]);
    // the charges from pinned host memory, the results into it (over the
    // charges, read by then; energy, virial and status after them): no copies,
    // one wait
    PmeCore& core = pme->core;
    PmeRun r;
    r.core = &core;
    r.n = n;
    r.xyzq = pme->xyzq.p;
    r.f_out = pme->fout.p;
    r.fscale = 1.0f;
    r.res = core.res_dev.p;
    r.binned = true;
    BatchRun R;
    R.stream = pme->stream;
    R.cache = &core.cache;
    R.n = 1;
    float* const h_f = reinterpret_cast<float*>(pme->h_xyzq.p);
    double* const rep = reinterpret_cast<double*>(pme->h_xyzq.p + nn);
    const float4* src = pme->h_xyzq.p;
    // a brick list that overflowed: enlarge and evaluate again
    for (int attempt = 0;; ++attempt) {
      core.ensure_cap(n);
      if (src)
        launch<k_pme_take>(R, "k_pme_take", 0, grid_all(nn, 256), 256, 0, [&](uint32_t) {
          return args<k_pme_take>(src, n, pme->xyzq.p, core.bin_args(nullptr, 0));
        });
      else
        r.binned = false;  // from the device's copy
      pme_run(R, pme->prof, &r, 0);
      launch<k_pme_out>(R, "k_pme_out", 0, grid_all(3 * nn, 256), 256, 0, [&](uint32_t) {
        return args<k_pme_out>((const float*)pme->fout.p, 3u * n, (const double*)core.res_dev.p,
                               (const unsigned int*)core.status.p, h_f, rep);
      });
      DYN_HIP(hipStreamSynchronize(pme->stream));
      if (rep[2] == 0.0) break;
      src = nullptr;
      DYN_HIP(hipMemsetAsync(core.status.p, 0, sizeof(unsigned int), pme->stream));
      if (attempt >= 4) throw Error(DYN_ERR_CAPACITY, "SPME brick lists keep overflowing");
      core.grow();
    }
    const double res[2] = {rep[0], rep[1]};
    if (n && f_out) memcpy(f_out, h_f, sizeof(float) * 3 * (size_t)n);
    const double e_self = (double)pme->core.beta / std::sqrt(M_PI) * q2;
    if (energy) *energy = res[0] - e_self;
    if (virial) *virial = res[1];
    pme->computed = true;
  });
}

extern "C" int dyn_pme_get_fixed_grid(dyn_pme* pme, int64_t* out, uint64_t n_values) {
  if (!pme) {
    set_global_error("null handle");
    return DYN_ERR_ARG;
  }
  DYN_API_BODY(pme, {
    DeviceGuard g(pme->device);
    if (!pme->computed) throw Error(DYN_ERR_STATE, "no compute yet");
    DYN_REQUIRE(out && n_values >= pme->core.ngrid, "need %zu values", pme->core.ngrid);
    DYN_HIP(hipMemcpyAsync(out, pme->core.grid_fx.p, sizeof(int64_t) * pme->core.ngrid,
                           hipMemcpyDeviceToHost, pme->stream));
    DYN_HIP(hipStreamSynchronize(pme->stream));
  });
}

extern "C" int dyn_pme_grid_n(float lx, float ly, float lz, float spacing, uint32_t out[3]) {
  try {
    DYN_REQUIRE(out, "out is null");
    DYN_REQUIRE(spacing > 0.f && std::isfinite(spacing), "spacing must be > 0");
    const float l[3] = {lx, ly, lz};
    for (int a = 0; a < 3; ++a) {
      DYN_REQUIRE(l[a] > 0.f && std::isfinite(l[a]), "box length must be > 0");
      uint32_t n = (uint32_t)std::ceil((double)l[a] / (double)spacing);
      if (n < 5) n = 5;
      while (!is_235_smooth(n)) ++n;
      out[a] = n;
    }
    return DYN_OK;
  } catch (const Error& e) {
    set_global_error(e.what());
    return e.code;
  }
}

// Device helpers of the SPH step shared by the pass kernels (sph_pass.hip)
// and the other step kernels (sph_kernels.hip): SPH kernel functions, EOS,
// accumulators, scene sources, the neighbour-membership walk and reductions.
#pragma once

#include <type_traits>

#include "blockscan.hpp"
#include "sph.hpp"

#define GCLSPH_INLINE __attribute__((always_inline))  // of a lambda

namespace gclsph {

// ---------------------------------------------------------------- math helpers
__device__ __forceinline__ double powi_d(double x, int p) {
#pragma clang fp contract(off)
  // binary powering, same operation sequence as the oracle's powi
  double r = 1.0, b = x;
  bool first = true;
  while (p > 0) {
    if (p & 1) {
      r = first ? b : r * b;
      first = false;
    }
    p >>= 1;
    if (p) b = b * b;
  }
  return r;
}

// powfancy7th (src/gpukernels_sph.jl:499-515) for γ == 7; x^(1/γ) otherwise.
__device__ __forceinline__ double pf7(double x, int gamma, double ginv) {
#pragma clang fp contract(off)
  if (gamma == 7) {
    unsigned long long bits = (unsigned long long)__double_as_longlong(fabs(x));
    unsigned long long tb = 0x36cd000000000000ull + bits / 7ull;
    double t = copysign(__longlong_as_double((long long)tb), x);
#pragma unroll 1
    for (int it = 0; it < 2; ++it) {
      double t2 = t * t;
      double t3 = t2 * t;
      double t4 = t2 * t2;
      double xot4 = x / t4;
      t = t - t * (t3 - xot4) / (4.0 * t3 + 3.0 * xot4);
    }
    return t;
  }
  return pow(x, ginv);
}

// WendlandC2 (SPHKernels.jl): W = ((1+4u)(1-u)^4) σ H⁻ᴰ, dW = -20u(1-u)^3 σ H⁻⁽ᴰ⁺¹⁾.
__device__ __forceinline__ double W_d(double u, double wnorm) {
#pragma clang fp contract(off)
  if (u < 1.0) {
    double um1 = 1.0 - u;
    um1 = um1 * um1;
    um1 = um1 * um1;
    return ((1.0 + 4.0 * u) * um1) * wnorm;
  }
  return 0.0;
}
__device__ __forceinline__ double dW_d(double u, double dwnorm) {
#pragma clang fp contract(off)
  if (u < 1.0) {
    double um1 = 1.0 - u;
    double um13 = um1 * um1 * um1;
    return -20.0 * u * um13 * dwnorm;
  }
  return 0.0;
}
// The FP32 pair arithmetic names its fused multiply-adds: every kernel that
// evaluates a pair (and every copy of a pair body in an unrolled loop) then
// rounds alike, which contraction by the compiler does not promise.
__device__ __forceinline__ float W_f(float r, float Hinv, float wnorm) {
#pragma clang fp contract(off)
  const float u = r * Hinv;
  if (u < 1.0f) {
    float um1 = __builtin_fmaf(-r, Hinv, 1.0f);
    um1 = um1 * um1;
    um1 = um1 * um1;
    return (__builtin_fmaf(4.0f, u, 1.0f) * um1) * wnorm;
  }
  return 0.0f;
}

// FP64 pair arithmetic.  A pair of the Float64 path once cost ten IEEE
// divisions (11 instructions each), a square root (~18) and powfancy7th: ~330
// VALU instructions, and the passes were bound by them.  Here the divisions
// share one reciprocal, 1/ρ comes with the partner's record, ∇W needs no
// 1/r (dW/dr / r is a polynomial of r) and the hydrostatic term is its series.

// 1/x, and sqrt(x) with sqrt(0) = 0: the hardware seed and Newton steps, to
// about an ulp for normal x away from the ends of the FP64 range.
__device__ __forceinline__ double rcp_d(double x) {
#pragma clang fp contract(off)
  double r = __builtin_amdgcn_rcp(x);
  r = __builtin_fma(__builtin_fma(-x, r, 1.0), r, r);
  return __builtin_fma(__builtin_fma(-x, r, 1.0), r, r);
}
__device__ __forceinline__ double sqrt_d(double x) {
#pragma clang fp contract(off)
  const double y = __builtin_amdgcn_rsq(x);
  double s = x * y, h = 0.5 * y;
  const double e = __builtin_fma(-h, s, 0.5);
  s = __builtin_fma(s, e, s);
  h = __builtin_fma(h, e, h);
  s = __builtin_fma(__builtin_fma(-s, s, x), h, s);
  return x == 0.0 ? 0.0 : s;
}
// (dW/dr)/r at distance r, i.e. ∇W = dx · dWr: -20 (1-u)^3 dwnorm / H (u/r =
// 1/H).  FP64: NaN for coincident particles, as the reference's dW/r.
__device__ __forceinline__ double dWr(double r2, double r, const SphConst& C) {
#pragma clang fp contract(off)
  const double um1 = __builtin_fma(-r, C.Hinv, 1.0);
  const double w = um1 > 0.0 ? C.dwr * (um1 * um1 * um1) : 0.0;
  return r2 != 0.0 ? w : __builtin_nan("");
}
__device__ __forceinline__ float dWr(float, float r, const SphConst& C) {
#pragma clang fp contract(off)
  const float um1 = __builtin_fmaf(-r, C.f_Hinv, 1.0f);
  return um1 > 0.0f ? C.f_dwr * (um1 * um1 * um1) : 0.0f;
}
// ρ0·(powfancy7th(1+z) - 1) of the δ-SPH term.  powfancy7th stops two Halley
// steps after a guess from the bit pattern, 3.87e-13 below the root near 1 (an
// offset linear in z on either side of 0); that times ρ0 and the stiffness of
// the term shows in ∂ρ/∂t, so results agree with the reference's only if it is
// kept.  γ = 7 (G7), |z| < 2^-8 (z is ~1e-3 at most between partners of the
// scenes here): the binomial series of the root plus that offset, within
// 4e-16 of powfancy7th's real-number value (its own rounding is 2e-16) and
// without its four divisions.  Other γ take pow, in kernels of their own: its
// registers cost the γ = 7 kernels a wave per SIMD.
template <bool G7>
__device__ __forceinline__ double hydro_drho_d(double z, const SphConst& C) {
#pragma clang fp contract(off)
  if constexpr (G7) {
    if (fabs(z) < 0x1p-8) {
      double t = __builtin_fma(z, 81549.0 / 5764801.0, -1989.0 / 117649.0);
      t = __builtin_fma(z, t, 351.0 / 16807.0);
      t = __builtin_fma(z, t, -65.0 / 2401.0);
      t = __builtin_fma(z, t, 13.0 / 343.0);
      t = __builtin_fma(z, t, -3.0 / 49.0);
      t = __builtin_fma(z, t, 1.0 / 7.0 - 5.43e-12);
      return C.rho0 * __builtin_fma(z, t, __builtin_fma(fabs(z), -5.84e-12, -3.8692e-13));
    }
    return C.rho0 * pf7(1 + z, 7, C.ginv) - C.rho0;
  } else {
    if (C.gamma == 7) return hydro_drho_d<true>(z, C);  // beside other γ in a batch
    return C.rho0 * pf7(1 + z, C.gamma, C.ginv) - C.rho0;
  }
}
// 1/ρb, 1/(ρa + ρb) and 1/(r² + η²) of a pair: FP64 from one reciprocal, 1/ρb
// from the record where it is stored; FP32 from the hardware reciprocals of
// ρb(ρa + ρb) (densities near ρ0, so the product stays far from the FP32 range
// limits) and r² + η².
template <typename R>
struct Inv3 {
  R rhob, sum, den;
};
__device__ __forceinline__ Inv3<double> inv_stored(double irhob, double sum, double den) {
#pragma clang fp contract(off)
  const double r = rcp_d(sum * den);
  return {irhob, r * den, r * sum};
}
__device__ __forceinline__ Inv3<double> inv_all(double rhob, double sum, double den) {
#pragma clang fp contract(off)
  const double bs = rhob * sum, r = rcp_d(bs * den), rd = r * den;
  return {rd * sum, rd * rhob, r * bs};
}
template <int D>
__device__ __forceinline__ Inv3<double> pair_inv(const PartnerN64<D>& q, double, double sum, double den) {
  return inv_stored(q.irho, sum, den);
}
template <int D>
__device__ __forceinline__ Inv3<double> pair_inv(const PartnerH64<D>& q, double, double sum, double den) {
  return inv_stored(q.irh, sum, den);
}
__device__ __forceinline__ Inv3<double> pair_inv(const PartnerH64<3>& q, double, double sum, double den) {
  return inv_all(q.rh, sum, den);
}
template <typename Q>
__device__ __forceinline__ Inv3<float> pair_inv(const Q&, float rhob, float sum, float den) {
#pragma clang fp contract(off)
  const float r = __builtin_amdgcn_rcpf(rhob * sum);
  return {sum * r, rhob * r, __builtin_amdgcn_rcpf(den)};
}
template <int D>
__device__ __forceinline__ void set_irho(PartnerN64<D>& q) {
  q.irho = 1.0 / q.rho;
}
template <int D>
__device__ __forceinline__ void set_irho(PartnerH64<D>& q) {
  q.irh = 1.0 / q.rh;
}
__device__ __forceinline__ void set_irho(PartnerH64<3>&) {}
// sin(πs), |s| <= 1/2: its Taylor series (the first term dropped is below 2^-59)
__device__ __forceinline__ double sinpi_d(double s) {
#pragma clang fp contract(off)
  constexpr double p = 3.14159265358979323846, p2 = p * p;
  constexpr double c3 = p * p2 / 6, c5 = c3 * p2 / 20, c7 = c5 * p2 / 42, c9 = c7 * p2 / 72, c11 = c9 * p2 / 110,
                   c13 = c11 * p2 / 156, c15 = c13 * p2 / 210, c17 = c15 * p2 / 272, c19 = c17 * p2 / 342,
                   c21 = c19 * p2 / 420;
  const double w = s * s;
  double t = __builtin_fma(w, c21, -c19);
  t = __builtin_fma(w, t, c17);
  t = __builtin_fma(w, t, -c15);
  t = __builtin_fma(w, t, c13);
  t = __builtin_fma(w, t, -c11);
  t = __builtin_fma(w, t, c9);
  t = __builtin_fma(w, t, -c7);
  t = __builtin_fma(w, t, c5);
  t = __builtin_fma(w, t, -c3);
  return s * __builtin_fma(w, t, p);
}
// ∂v∂tpF! coefficient s·cos(1.5π r/2h)/(r + 0.1h) for r < 2h:
// cos(πy) = -sin(π(y - 1/2)), y in [0, 1.5), folded into [-1/2, 1/2]
__device__ __forceinline__ double surf_d(double r, const SphConst& C) {
#pragma clang fp contract(off)
  const double y = r * C.st_pi;
  return -C.s * sinpi_d(y > 1.0 ? 1.5 - y : y - 0.5) * rcp_d(r + C.st_01h);
}

// Tait EOS (src/gpukernels_sph.jl:691-697): 0 if ptype <= 1 and ρ < ρ0.
__device__ __forceinline__ double eos_d(double rho, int32_t pt, const SphConst& C) {
#pragma clang fp contract(off)
  if (pt <= 1 && rho < C.rho0) return 0.0;
  return C.P0 * (powi_d(rho / C.rho0, C.gamma) - 1);
}
// ptype(a)·ptype(b) > 0 of the reference (an Int64 product) for int32 types:
// both positive or both negative, without the 64-bit multiply.
__device__ __forceinline__ bool same_kind(int32_t pa, int32_t pb) { return (pa > 0 && pb > 0) || (pa < 0 && pb < 0); }

// FP32-split EOS on δρ: P0((1+e)^7 - 1) = P0 e (7 + 21e + 35e² + 35e³ + 21e⁴ + 7e⁵ + e⁶).
__device__ __forceinline__ float eos_f(float drho, int32_t pt, const SphConst& C) {
#pragma clang fp contract(off)
  if (pt <= 1 && drho < 0.0f) return 0.0f;
  const float e = drho * C.f_inv_rho0;
  float poly = __builtin_fmaf(e, 7.0f + e, 21.0f);
  poly = __builtin_fmaf(e, poly, 35.0f);
  poly = __builtin_fmaf(e, poly, 35.0f);
  poly = __builtin_fmaf(e, poly, 21.0f);
  poly = __builtin_fmaf(e, poly, 7.0f);
  return C.f_P0 * (e * poly);
}
// dr - ρ0((1+z)^(1/7) - 1) without cancellation (the δ-SPH term's density
// difference less its hydrostatic part): binomial series, exact function for
// |z| > 1e-2.
__device__ __forceinline__ float minus_hydro(float dr, float z, const SphConst& C) {
#pragma clang fp contract(off)
  float t;
  if (fabsf(z) < 1e-2f) {
    t = __builtin_fmaf(z, -65.0f / 2401.0f, 13.0f / 343.0f);
    t = __builtin_fmaf(z, t, -3.0f / 49.0f);
    t = z * __builtin_fmaf(z, t, 1.0f / 7.0f);
  } else {
    t = expm1f(log1pf(z) * (1.0f / 7.0f));
  }
  return __builtin_fmaf(-C.f_rho0, t, dr);
}

// FP32-split ∂v∂tpF! coefficient s·cos(1.5π r/2h)/(r + 0.1h), for r < 2h: the
// hardware cosine (argument in turns, here in [0, 0.75)) and reciprocal.
__device__ __forceinline__ float surf_f(float r, const SphConst& C) {
#pragma clang fp contract(off)
  return C.f_s * __builtin_amdgcn_cosf(r * C.f_st_turn) * __builtin_amdgcn_rcpf(r + C.f_st_01h);
}

// Value of lane K of the quad (four consecutive lanes, all active).
template <int K>
__device__ __forceinline__ uint32_t quad_lane(uint32_t v) {
  return uint32_t(__builtin_amdgcn_mov_dpp(int(v), K * 0x55, 0xf, 0xf, true));
}
template <int K>
__device__ __forceinline__ float quad_lane(float v) {
  return __uint_as_float(quad_lane<K>(__float_as_uint(v)));
}
template <int K>
__device__ __forceinline__ double quad_lane(double v) {
  return __hiloint2double(int(quad_lane<K>(uint32_t(__double2hiint(v)))), int(quad_lane<K>(uint32_t(__double2loint(v)))));
}

// The terms one partner adds to a particle's N sums, and the sums: FP64 in
// both precisions (an FP32 term costs a conversion and an addition).
template <int N, typename R>
struct Terms {
  R v[N] = {};
};
template <int N, typename R>
struct Sums {
  double s[N] = {};
  __device__ __forceinline__ void add(const Terms<N, R>& t) {
#pragma unroll
    for (int i = 0; i < N; ++i) s[i] += double(t.v[i]);
  }
  // the terms of the quad's four lanes, in lane order
  __device__ __forceinline__ void add_quad(const Terms<N, R>& t) {
#pragma unroll
    for (int i = 0; i < N; ++i) {
      s[i] += double(quad_lane<0>(t.v[i]));
      s[i] += double(quad_lane<1>(t.v[i]));
      s[i] += double(quad_lane<2>(t.v[i]));
      s[i] += double(quad_lane<3>(t.v[i]));
    }
  }
  __device__ __forceinline__ R get(int i) const { return R(s[i]); }
};

template <int D>
__device__ __forceinline__ double dotd(const double* a, const double* b) {
#pragma clang fp contract(off)
  double s = a[0] * b[0] + a[1] * b[1];
  if (D == 3) s = s + a[2] * b[2];
  return s;
}
// dotd with fused multiply-adds, where no comparison reads it
__device__ __forceinline__ double fma_(double a, double b, double c) { return __builtin_fma(a, b, c); }
__device__ __forceinline__ float fma_(float a, float b, float c) { return __builtin_fmaf(a, b, c); }
template <int D>
__device__ __forceinline__ double dotm(const double* a, const double* b) {
#pragma clang fp contract(off)
  double s = fma_(a[1], b[1], a[0] * b[0]);
  if (D == 3) s = fma_(a[2], b[2], s);
  return s;
}
template <int D>
__device__ __forceinline__ float dotf(const float* a, const float* b) {
#pragma clang fp contract(off)
  float s = fma_(a[0], b[0], a[1] * b[1]);
  if (D == 3) s = fma_(a[2], b[2], s);
  return s;
}

// Buffers of the current state within a step, after the rebuild stage: a
// rebuild writes the other ones, and the flag is cleared when the step ends.
__device__ __forceinline__ int cur_parity(const StepCtl* c) { return c->parity ^ c->rebuild; }
__device__ __forceinline__ int cur_pparity(const StepCtl* c) { return c->pparity ^ c->rebuild; }

// Positions of the pair-list membership test: the current positions when this
// step rebuilt (or when no later step can skip a rebuild), else the stored
// rebuild positions.
template <int D, typename R>
__device__ __forceinline__ void membership_ptrs(const SphBufs<R>& B, const StepFlags& F, int p, int rebuilt,
                                                const double** XM) {
  bool cur = rebuilt || !F.need_xrb;
#pragma unroll
  for (int k = 0; k < 3; ++k) XM[k] = cur ? B.X[p][k < D ? k : 1] : B.XRB[k < D ? k : 1];
}

// Logical number of this block with an XCD-aware order: workgroups are dealt
// to the 8 XCDs round robin (block b runs on XCD b % 8), and renumbering so
// that each XCD walks one contiguous range of logical blocks (cell-sorted
// particles) keeps the neighbourhoods shared by consecutive blocks, and by the
// stencil rows above and below, inside one XCD's L2.
__device__ __forceinline__ unsigned xcd_block() {
  const unsigned G = gridDim.x, b = blockIdx.x;
  const unsigned q = G / 8, r = G % 8, xcd = b % 8, i = b / 8;
  return xcd < r ? xcd * (q + 1) + i : r * (q + 1) + (xcd - r) * q + i;
}

// Where a kernel finds its problem.  One problem: the descriptor is a kernel
// argument (constant memory the compiler may reload at will, which keeps
// register pressure as low as plain arguments).  Several problems: an array of
// descriptors in device memory and maps from blocks to (problem, block of the
// problem) or (problem, cell tile).
template <typename R>
struct OneScene {
  SceneDev<R> d;
};
template <typename R>
struct ManyScenes {
  const SceneDev<R>* __restrict__ S;
  const int2* __restrict__ pmap;
  const int2* __restrict__ cmap;
  const int2* __restrict__ pmap512;  // (problem, 512-particle block of the problem)
  const int2* __restrict__ qmap;     // (problem, 64-particle block of the problem): a quad of lanes per particle
};
// Blocks of BS threads (128, 256 or 512) over one problem's particles: m.y is
// the block's index in units of BS particles, so particle a = m.y·BS + tid;
// Quad: blocks of 256 threads over 64 particles, m.y in units of 64.
template <int BS = kBlock, bool Quad = false, typename R>
__device__ __forceinline__ const SceneDev<R>& particle_scene(const OneScene<R>& s, int2& m) {
  m = make_int2(0, int(xcd_block()));
  return s.d;
}
// Descriptor i of a batch, read through the constant address space: the
// descriptors are not written while a kernel runs, so their loads are
// invariant (scalar loads the compiler may repeat at will, as for a kernel
// argument), and the buffer pointers read from them are used as global-memory
// pointers instead of falling back to flat addressing.
template <typename R>
__device__ __forceinline__ const SceneDev<R>& batch_scene(const ManyScenes<R>& s, int i) {
  using CS = const __attribute__((address_space(4))) SceneDev<R>;
  CS* c = (CS*)(s.S);
  return *(const SceneDev<R>*)(c + i);
}
template <int BS = kBlock, bool Quad = false, typename R>
__device__ __forceinline__ const SceneDev<R>& particle_scene(const ManyScenes<R>& s, int2& m) {
  static_assert(BS == 128 || BS == 256 || BS == 512, "block sizes of the particle maps");
  static_assert(!Quad || BS == 256, "quads come in blocks of 256 threads");
  const unsigned L = xcd_block();
  if constexpr (Quad) {
    m = s.qmap[L];
  } else if constexpr (BS == 256) {
    m = s.pmap[L];
  } else if constexpr (BS == 128) {  // halves of the 256-particle blocks
    const int2 e = s.pmap[L >> 1];
    m = make_int2(e.x, e.y * 2 + int(L & 1u));
  } else {
    m = s.pmap512[L];
  }
  return batch_scene(s, m.x);
}
template <typename R>
__device__ __forceinline__ const SceneDev<R>& tile_scene(const OneScene<R>& s, int2& m) {
  m = make_int2(0, int(blockIdx.x));
  return s.d;
}
template <typename R>
__device__ __forceinline__ const SceneDev<R>& tile_scene(const ManyScenes<R>& s, int2& m) {
  m = s.cmap[blockIdx.x];
  return batch_scene(s, m.x);
}
template <typename R>
__device__ __forceinline__ const SceneDev<R>& scene_at(const OneScene<R>& s, unsigned) {
  return s.d;
}
template <typename R>
__device__ __forceinline__ const SceneDev<R>& scene_at(const ManyScenes<R>& s, unsigned i) {
  return batch_scene(s, int(i));
}

// Per-step switches of a problem, from its per-call switches and control block.
template <typename R>
__device__ __forceinline__ StepFlags step_flags(const SceneDev<R>& sd) {
  StepFlags F = sd.F;
  const StepCtl* c = sd.B.ctl;
  const int it = c->iter;
  F.synced_prev = c->synced;
  F.cspm_fire = F.cspmn > 0 && it % F.cspmn == 0;
  F.corr_on = F.dpc_on || F.xsph_on || F.cspm_fire;
  F.want_out = it == c->nsteps;
  return F;
}

// Binds the problem of this block: B, C, G, F and the particle index a.
#define GCLSPH_SCENE_OF(ss, BS, Quad)                         \
  int2 m;                                                     \
  const SceneDev<R>& sd = particle_scene<BS, Quad, R>(ss, m); \
  const SphBufs<R>& B = sd.B;                                 \
  const SphConst& C = sd.C;                                   \
  const CellGeom& G = sd.G;                                   \
  const StepFlags F = step_flags(sd);                         \
  (void)C;                                                    \
  (void)G;                                                    \
  (void)F
#define GCLSPH_SCENE(ss)              \
  GCLSPH_SCENE_OF(ss, kBlock, false); \
  const int64_t a = int64_t(m.y) * kBlock + threadIdx.x
// In the pair kernels: a particle per thread, or (Quad) per four threads, the
// first of which writes its results.
#define GCLSPH_SCENE_PAIR(ss, BS, Quad)                                                                   \
  GCLSPH_SCENE_OF(ss, BS, Quad);                                                                          \
  const int64_t a = (Quad) ? int64_t(m.y) * 64 + (threadIdx.x >> 2) : int64_t(m.y) * (BS) + threadIdx.x;  \
  const bool writer = !(Quad) || (threadIdx.x & 3) == 0

// Member bits of one window [lo, hi) (hi - lo <= 32) of a stencil row: bit j is
// set when candidate lo + j is a partner of particle a, i.e. b != a and
// r^2 < dist^2 with the reference's expression (no FMA).  Candidates are read
// four at a time so their loads are in flight together; reads run up to 3 past
// hi, which the position arrays' padding keeps in bounds, and those bits are
// dropped.
template <int D>
__device__ __forceinline__ uint32_t window_bits(const double* x0, const double* x1, const double* x2, double xa0,
                                                double xa1, double xa2, int64_t a, int32_t lo, int32_t hi,
                                                double dist2) {
#pragma clang fp contract(off)
  const double* p0 = x0 + lo;
  const double* p1 = x1 + lo;
  const double* p2 = x2 + lo;
  const int32_t len = hi - lo;
  uint32_t mk = 0;
  for (int32_t j = 0; j < len; j += 4) {
    double c0[4], c1[4], c2[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      c0[u] = p0[j + u];
      c1[u] = p1[j + u];
      if (D == 3) c2[u] = p2[j + u];
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const double d0 = xa0 - c0[u];
      const double d1 = xa1 - c1[u];
      double r2 = d0 * d0 + d1 * d1;
      if (D == 3) {
        const double d2 = xa2 - c2[u];
        r2 = r2 + d2 * d2;
      }
      mk |= uint32_t(r2 < dist2) << (j + u);
    }
  }
  if (len < 32) mk &= (1u << len) - 1u;
  const int64_t self = a - lo;
  if (self >= 0 && self < len) mk &= ~(1u << self);
  return mk;
}

// window_bits for the stencil scan inside the pair loops (a particle whose
// windows overflowed the membership store): one candidate at a time, so the
// scan adds few registers to the loop around it (the four-wide form above
// sets the register count, and so the occupancy, of every pair kernel).  Same
// expression, same bits.
template <int D>
__device__ __forceinline__ uint32_t window_bits_lean(const double* x0, const double* x1, const double* x2,
                                                     double xa0, double xa1, double xa2, int64_t a, int32_t lo,
                                                     int32_t hi, double dist2) {
#pragma clang fp contract(off)
  uint32_t mk = 0;
#pragma clang loop unroll(disable)
  for (int32_t b = lo; b < hi; ++b) {
    const double d0 = xa0 - x0[b];
    const double d1 = xa1 - x1[b];
    double r2 = d0 * d0 + d1 * d1;
    if (D == 3) {
      const double d2 = xa2 - x2[b];
      r2 = r2 + d2 * d2;
    }
    mk |= uint32_t(r2 < dist2 && b != a) << (b - lo);
  }
  return mk;
}

// Sorted range [b, e) of stencil row k (dy = k%3 - 1, dz = k/3 - 1) of cell c;
// empty when the row lies outside the grid.
template <int D>
__device__ __forceinline__ void row_range(const CellGeom& g, const int32_t* __restrict__ start, int32_t c, int k,
                                          int32_t& b, int32_t& e) {
  const int64_t gx = g.grid[0], gy = g.grid[1];
  int64_t ix, iy, iz;
  cell_xyz<D>(g, c, ix, iy, iz);
  const int64_t xl = ix > 0 ? ix - 1 : 0, xh = ix + 1 < gx ? ix + 1 : gx - 1;
  const int64_t y = iy + (k % 3) - 1;
  const int64_t z = D == 3 ? iz + (k / 3) - 1 : 0;
  const bool in = y >= 0 && y < gy && (D == 2 || (z >= 0 && z < g.grid[2]));
  const int64_t row = gx * (y + gy * z);
  b = in ? start[row + xl] : 0;
  e = in ? start[row + xh + 1] : 0;
}

// Element of a per-particle array at a 32-bit byte offset: the load then uses
// the scalar base + 32-bit vector offset addressing form (no 64-bit address
// arithmetic per partner).  Arrays stay below 4 GiB (the problem size limit
// checked at construction).
template <typename T>
__device__ __forceinline__ T ldo(const T* base, uint32_t byte_off) {
  return *reinterpret_cast<const T*>(reinterpret_cast<const char*>(base) + byte_off);
}

// Record b of a partner-record array (n particles) as 16-byte loads: word i at
// word i·n + b where RecordWords<T> says the array keeps words apart (2D),
// else at word b·(sizeof(T)/16) + i.  Offsets are 64-bit (the arrays are larger
// than the 8-byte elements the 32-bit offsets above are sized for); b, a
// partner index in [0, n), is taken unsigned (no sign extension per load).
template <typename T>
__device__ __forceinline__ T ld_rec(const void* base, uint32_t b, int64_t n) {
  static_assert(sizeof(T) % 16 == 0, "records are whole 16-byte words");
  constexpr int kW = int(sizeof(T) / 16);
  constexpr bool apart = RecordWords<T>::value;
  const uint4* p = reinterpret_cast<const uint4*>(base) + (apart ? uint64_t(b) : uint64_t(b) * kW);
  uint4 w[kW];
#pragma unroll
  for (int i = 0; i < kW; ++i) w[i] = p[apart ? i * n : i];
  T r;
  __builtin_memcpy(&r, w, sizeof(T));
  return r;
}

// The words of record b that hold its position (the other fields read as zero).
template <typename T>
__device__ __forceinline__ T ld_pos(const void* base, uint32_t b, int64_t n) {
  constexpr int kW = int(sizeof(T) / 16), kHead = int((T::kPosBytes + 15) / 16);
  constexpr bool apart = RecordWords<T>::value;
  const uint4* p = reinterpret_cast<const uint4*>(base) + (apart ? uint64_t(b) : uint64_t(b) * kW);
  uint4 w[kW] = {};
#pragma unroll
  for (int i = 0; i < kHead; ++i) w[i] = p[apart ? i * n : i];
  T r;
  __builtin_memcpy(&r, w, sizeof(T));
  return r;
}

template <typename T>
__device__ __forceinline__ void st_rec(void* base, int64_t a, const T& r, int64_t n) {
  constexpr int kW = int(sizeof(T) / 16);
  constexpr bool apart = RecordWords<T>::value;
  uint4 w[kW];
  __builtin_memcpy(w, &r, sizeof(T));
  uint4* p = reinterpret_cast<uint4*>(base) + (apart ? a : a * kW);
#pragma unroll
  for (int i = 0; i < kW; ++i) p[apart ? i * n : i] = w[i];
}

// ---- 2D partner records staged in LDS
// The pair passes with one lane per particle read a partner's record ~36 times
// for each particle, at 64 places per load, and were bound by the CU's L1 (FP64:
// an access each cycle; FP32-split: 0.93, with the VALU at 0.9).  A block's
// particles are consecutive cells, so their partners lie in three ranges of
// sorted indices (~3.4 BS records), which the block copies to LDS once, by
// coalesced loads.  Two of a record's 16-byte words are staged: all of an
// FP32-split one, half of an FP64 one; the other FP64 words stay with the L1.
// Three words staged left LDS for three waves per SIMD instead of four (1.02 M
// particles FP64: 52 KiB a block).  FP32-split passes are then bound by VALU
// issue (1.0 per CU and cycle).  4.05 M particles FP32-split: passes 414 + 481
// -> 380 + 433 us; 1.02 M FP64: 189 + 259 -> 180 + 230 us.
constexpr int kStagedWords = 2;
// Records staged at most.  The rows above and below a block's cells hold up to
// 4/3 of its particles where the cell size is 3.6 lattice spacings, and each row
// the cells beside its ends.  Short of this many (3 BS + 160) a half of the
// blocks of a lattice fell back to global memory.
template <int BS>
constexpr int kStageCap = 15 * BS / 4 + 128;

// Where the records of the block's stencil rows are staged: record b of row r at
// b + d[r].  The row of a window is taken to be the last one that begins at or
// before it: where ranges overlap, that one reaches at least as far.
struct RowMap {
  int32_t s1, s2;
  int32_t d0, d1, d2;
  __device__ __forceinline__ int32_t at(int32_t b) const {
    const int32_t v0 = d0, v1 = d1, v2 = d2;  // values: a choice between members would keep them in memory
    int32_t d = b >= s1 ? v1 : v0;
    d = b >= s2 ? v2 : d;
    return d;
  }
};

// Stages the first Words words of the records of the three stencil rows around
// the block's particles [a0, a0 + BS): row r is one range of sorted indices,
// from the cell before the first particle's to the one after the last's (more
// than the particles need where the block goes over a row end; in a narrow grid
// the ranges overlap).  False when they don't fit or some particle has no stored
// membership (nc < 0): the block then reads global memory.  Called by the whole
// block.
template <int BS, int Words, typename R>
__device__ __forceinline__ bool stage_rows(uint4 (*lds)[kStageCap<BS>], const void* base, const SphBufs<R>& B,
                                           const CellGeom& G, int64_t a0, int nc, RowMap& map) {
  const int64_t last = (a0 + BS < B.n ? a0 + BS : B.n) - 1, gx = G.grid[0], nce = G.ncells();
  const int64_t c0 = B.skey[a0], c1 = B.skey[last];
  int32_t s[3], e[3];
#pragma unroll
  for (int r = 0; r < 3; ++r) {
    const int64_t lo = c0 + gx * (r - 1) - 1, hi = c1 + gx * (r - 1) + 2;
    s[r] = __builtin_amdgcn_readfirstlane(B.start[lo < 0 ? 0 : (lo > nce ? nce : lo)]);
    e[r] = __builtin_amdgcn_readfirstlane(B.start[hi < 0 ? 0 : (hi > nce ? nce : hi)]);
  }
  const int32_t n0 = e[0] - s[0], n1 = n0 + (e[1] - s[1]), n2 = n1 + (e[2] - s[2]);
  if (!__syncthreads_and(n2 <= kStageCap<BS> && nc >= 0)) return false;
  map = {s[1], s[2], -s[0], n0 - s[1], n1 - s[2]};
  const uint4* p = reinterpret_cast<const uint4*>(base);
  for (int32_t i = threadIdx.x; i < n2; i += BS) {
    const int32_t b = i - (i < n0 ? map.d0 : i < n1 ? map.d1 : map.d2);
#pragma unroll
    for (int w = 0; w < Words; ++w) lds[w][i] = p[w * B.n + b];
  }
  __syncthreads();
  return true;
}

// Record b, staged at place i; its words beyond Words come from global memory.
template <typename T, int Words, int Cap>
__device__ __forceinline__ T ld_staged(const uint4 (*lds)[Cap], int32_t i, const void* base, uint32_t b,
                                       int64_t n) {
  constexpr int kW = int(sizeof(T) / 16);
  uint4 w[kW];
#pragma unroll
  for (int k = 0; k < Words; ++k) w[k] = lds[k][i];
  if constexpr (Words < kW) {
    const uint4* p = reinterpret_cast<const uint4*>(base) + b;
#pragma unroll
    for (int k = Words; k < kW; ++k) w[k] = p[k * n];
  }
  T r;
  __builtin_memcpy(&r, w, sizeof(T));
  return r;
}

// ---- 3D cell frames and per-cell membership windows
// 3D membership entries hold one window of at most kWin3 candidates inside
// one stencil cell: the member bits in the low kWin3 bits of the low word and
// above them the cell's offset o from the particle's own cell, coded
// (ox+1) + 3(oy+1) + 9(oz+1); the high word is the window base.  The
// FP32-split 3D pair kernels turn that code into the per-window separation
// constants of their cell frames (partner records in 3D hold positions as
// offsets from their cell's frame origin).
constexpr uint32_t kWinMask3 = (1u << kWin3) - 1u;
__device__ __forceinline__ uint32_t win_code3(int ox, int oy, int oz) {
  return uint32_t(ox + 1) + 3u * uint32_t(oy + 1) + 9u * uint32_t(oz + 1);
}

// Origin of the cell frame along axis d of grid coordinate i (0-based).
// Every writer and reader of a 3D record evaluates this same expression.
__device__ __forceinline__ double frame_origin(const SphConst& C, const CellGeom& G, int d, int64_t i) {
#pragma clang fp contract(off)
  return G.off64[d] + double(i) * C.fcs[d];
}

// Frame origins of sorted cell c.
__device__ __forceinline__ void cell_frame3(const SphConst& C, const CellGeom& G, int32_t c, double fr[3]) {
  int64_t ix, iy, iz;
  cell_xyz<3>(G, c, ix, iy, iz);
  fr[0] = frame_origin(C, G, 0, ix);
  fr[1] = frame_origin(C, G, 1, iy);
  fr[2] = frame_origin(C, G, 2, iz);
}

// Separation constants of a particle at xa in sorted cell c: km[d] = xa_d -
// frame_d(c_d - 1), rounded once, and the frame cell sizes cf (FP32-exact).
// For a partner b in the stencil cell at offset o, xa - xb = K - xo_b with
// K = km - (o + 1)·cf, one FMA whose product is exact.
struct FrameK3 {
  float km[3];
  float cf[3];
};
__device__ __forceinline__ FrameK3 frame_k3(const SphConst& C, const CellGeom& G, int32_t c, const double* xa) {
  int64_t i[3];
  cell_xyz<3>(G, c, i[0], i[1], i[2]);
  FrameK3 t;
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    t.km[d] = float(xa[d] - frame_origin(C, G, d, i[d] - 1));
    t.cf[d] = C.f_fcs[d];
  }
  return t;
}
// Window constants of one partner (3D FP32-split); an empty type elsewhere.
struct Win3 {
  float k[3];
};
struct NoWin {};

// Position fields of the FP32-split partner records: FP64 in 2D; in 3D the
// FP32 offset from the frame origins fr of the particle's sorted cell.
template <int D>
__device__ __forceinline__ void put_x(PartnerN<D>& r, int d, double x, const double*) {
  r.x[d] = x;
}
__device__ __forceinline__ void put_x(PartnerN<3>& r, int d, double x, const double* fr) {
  r.xo[d] = float(x - fr[d]);
}
template <int D>
__device__ __forceinline__ void put_x(PartnerN64<D>& r, int d, double x, const double*) {
  r.x[d] = x;
}
template <int D>
__device__ __forceinline__ void put_x(PartnerH<D>& r, int d, double x, const double*) {
  r.xh[d] = x;
}
__device__ __forceinline__ void put_x(PartnerH<3>& r, int d, double x, const double* fr) {
  r.xo[d] = float(x - fr[d]);
}
// FP32 separation x_a - x_b along d from partner b's record: the FP64
// difference rounded once (2D), or the window constant of b's cell minus b's
// frame offset (3D).
template <int D>
__device__ __forceinline__ float sep_x(const double* xa, const PartnerN<D>& q, int d) {
  return float(xa[d] - q.x[d]);
}
__device__ __forceinline__ float sep_x(const double*, const PartnerN<3>& q, int d, const Win3& w) {
  return w.k[d] - q.xo[d];
}
template <int D>
__device__ __forceinline__ float sep_x(const double* xa, const PartnerH<D>& q, int d) {
  return float(xa[d] - q.xh[d]);
}
__device__ __forceinline__ float sep_x(const double*, const PartnerH<3>& q, int d, const Win3& w) {
  return w.k[d] - q.xo[d];
}
// A partner's type as the pair kernels read it, and its pressure.  2D
// records keep the pressure in the type's place and the type's class in the
// two lowest mantissa bits of the FP64 y, read back as the representative
// type -1, 0, 1 or 2 (the same answer to every test a pair term makes: > 0,
// > 1, < 0, <= 1).  Those bits move y by at most 3 ulp of FP64, far below the
// FP32 rounding of a separation; the membership store reads the position
// arrays, not the records.
__device__ __forceinline__ double with_class(double y, int32_t pt) {
  const uint32_t c = pt < 0 ? 0u : (pt == 0 ? 1u : (pt == 1 ? 2u : 3u));
  const uint64_t u = uint64_t(__double_as_longlong(y));
  return __longlong_as_double((long long)((u & ~uint64_t(3)) | c));
}
__device__ __forceinline__ int32_t class_pt(double y) { return int32_t(uint32_t(__double_as_longlong(y)) & 3u) - 1; }
template <int D>
__device__ __forceinline__ int32_t rec_pt(const PartnerN<D>& r) {
  return class_pt(r.x[1]);
}
__device__ __forceinline__ int32_t rec_pt(const PartnerN<3>& r) { return r.pt; }
template <int D>
__device__ __forceinline__ int32_t rec_pt(const PartnerH<D>& r) {
  return class_pt(r.xh[1]);
}
__device__ __forceinline__ int32_t rec_pt(const PartnerH<3>& r) { return r.pt; }
template <int D>
__device__ __forceinline__ float rec_P(const PartnerN<D>& r, const SphConst&) {
  return r.P;
}
__device__ __forceinline__ float rec_P(const PartnerN<3>& r, const SphConst& C) { return eos_f(r.rho, r.pt, C); }
template <int D>
__device__ __forceinline__ float rec_P(const PartnerH<D>& r, const SphConst&) {
  return r.P;
}
__device__ __forceinline__ float rec_P(const PartnerH<3>& r, const SphConst& C) { return eos_f(r.rh, r.pt, C); }
// Type and pressure into a record whose position is already in place.
template <int D>
__device__ __forceinline__ void set_pt(PartnerN<D>& r, int32_t pt, float P) {
  r.x[1] = with_class(r.x[1], pt);
  r.P = P;
}
__device__ __forceinline__ void set_pt(PartnerN<3>& r, int32_t pt, float) { r.pt = pt; }
template <int D>
__device__ __forceinline__ void set_pt(PartnerH<D>& r, int32_t pt, float P) {
  r.xh[1] = with_class(r.xh[1], pt);
  r.P = P;
}
__device__ __forceinline__ void set_pt(PartnerH<3>& r, int32_t pt, float) { r.pt = pt; }

// Frame origins of particle a (3D; nothing to compute in 2D).
template <int D, typename R>
__device__ __forceinline__ void particle_frame(const SphBufs<R>& B, const SphConst& C, const CellGeom& G, int64_t a,
                                               double fr[3]) {
  if constexpr (D == 3) cell_frame3(C, G, B.skey[a], fr);
  else fr[0] = fr[1] = fr[2] = 0.0;
}
// Separation constants of particle a at position xa (3D FP32-split).
template <int D, typename R>
__device__ __forceinline__ FrameK3 particle_k(const SphBufs<R>& B, const SphConst& C, const CellGeom& G, int64_t a,
                                              const double* xa) {
  if constexpr (D == 3) return frame_k3(C, G, B.skey[a], xa);
  else return FrameK3{};
}

// Neighbour-list partners b of particle a in a fixed order (stencil rows in
// order, ascending sorted index inside a row; in 3D each row visited cell by
// cell, which is the same order), a window of candidates with its member bits at
// a time: from the membership store (Stored), or, for a particle that needs more
// entries than the store holds (nc < 0), computed from the membership positions
// (Scanned).  Each lane runs its own sequence, so all lanes of a wave execute the
// (long) pair body together.  The two are separate loops: one that could do both
// carried the scan's state through every trip (XSPH in 3D FP32-split: 86
// registers instead of 67), and its store path waited for the entry that it had
// just asked for.  A call of 31,962 particles in 3D FP64 with all corrections:
// 3.27 -> 3.09 ms.
// Fr (3D only): also the current window's separation constants, from the
// particle's FrameK3.
template <bool Fr>
struct Window {
  uint32_t c = 0;  // members not yet taken; bit t: candidate cb + t
  int32_t cb = 0;
  FrameK3 kt;   // Fr: the particle's separation constants
  float wk[3];  // Fr: constants of the current window

  // Another partner is waiting in the window.
  __device__ __forceinline__ bool has() const { return c != 0; }

  // The window's next partner.
  __device__ __forceinline__ int32_t take() {
    const int32_t b = cb + __builtin_ctz(c);
    c &= c - 1;
    return b;
  }
  // As take(), with the separation constants of the window.
  __device__ __forceinline__ int32_t take(Win3& w) {
    constants(w);
    return take();
  }
  __device__ __forceinline__ int32_t take(NoWin&) { return take(); }

  // The quad's four lanes hold the same state: lane i takes the i-th of the
  // window's next four partners, or `none` (on = false) past its last.
  template <typename W>
  __device__ __forceinline__ int32_t take_quad(bool& on, const int32_t none, W& w) {
    const uint32_t i = threadIdx.x & 3u;
    uint32_t m = c;
    m = i > 0 ? m & (m - 1) : m;
    m = i > 1 ? m & (m - 1) : m;
    m = i > 2 ? m & (m - 1) : m;
    on = m != 0;
    const int32_t b = on ? cb + __builtin_ctz(m) : none;
    if constexpr (Fr) constants(w);
    c = quad_lane<3>(m & (m - 1));
    return b;
  }

  __device__ __forceinline__ void constants(Win3& w) const {
    w.k[0] = wk[0];
    w.k[1] = wk[1];
    w.k[2] = wk[2];
  }
  __device__ __forceinline__ void set_window(uint32_t code) {
    if constexpr (Fr) {
      // base-3 digits of code < 27: q / 3 = (q · 11) >> 5 for q < 27
      const uint32_t q3 = (code * 11u) >> 5, q9 = (q3 * 11u) >> 5;
      const uint32_t o1[3] = {code - 3u * q3, q3 - 3u * q9, q9};
#pragma unroll
      for (int d = 0; d < 3; ++d) wk[d] = fmaf(float(o1[d]), -kt.cf[d], kt.km[d]);
    }
  }
};

// The halves of a stored entry, in registers of their own: shared with the
// entry's, they would leave the load of the next one no place but a second pair,
// copied (and so waited for) at once.
__device__ __forceinline__ void split_entry(uint64_t e, uint32_t& bits, uint32_t& base) {
  asm("v_mov_b32 %0, %1" : "=&v"(bits) : "v"(uint32_t(e)));
  asm("v_mov_b32 %0, %1" : "=&v"(base) : "v"(uint32_t(e >> 32)));
}

// The nc stored entries, read one ahead: the entry asked for when a window
// begins is first needed when it is empty.  The load has no condition (the store
// has a row more than entries may fill, and what the last load reads is not
// used), so its result needs no second register and no wait at the load.
template <int D, typename R, bool Fr = false>
struct Stored : Window<Fr> {
  static_assert(!Fr || cell_windows<D, R>(), "cell frames come with cell windows");
  const int64_t n;
  const uint64_t* pe;
  uint64_t nxt;
  int left;  // entries not yet begun

  __device__ __forceinline__ Stored(const SphBufs<R>& B, int64_t a, int nc, const FrameK3* kt_ = nullptr)
      : n(B.n), pe(B.NE + a), nxt(*pe), left(nc) {
    if constexpr (Fr) this->kt = *kt_;
  }
  // An empty window gives way to the next one (entries have member bits).
  __device__ __forceinline__ void refill() {
    if (this->c == 0 && left > 0) {
      uint32_t bits, base;
      split_entry(nxt, bits, base);
      if constexpr (cell_windows<D, R>()) {
        this->set_window(bits >> kWin3);
        bits &= kWinMask3;
      }
      this->c = bits;
      this->cb = int32_t(base);
      --left;
      pe += n;
      nxt = *pe;
    }
  }
};

template <int D, typename R, bool Fr = false>
struct Scanned : Window<Fr> {
  const SphBufs<R>& B;
  const CellGeom& G;
  const double* const xm0;  // membership positions, held by value
  const double* const xm1;
  const double* const xm2;
  const double dist2;
  const int64_t a;
  int k = -1;
  int32_t w0 = 0, re = 0;
  int j = 3;  // 3D: cell of row k, 0..2 for ox = -1..1

  __device__ __forceinline__ Scanned(const SphBufs<R>& B_, int64_t a_, const CellGeom& G_, const double* const* XM_,
                                     double dist2_, const FrameK3* kt_ = nullptr)
      : B(B_), G(G_), xm0(XM_[0]), xm1(XM_[1]), xm2(XM_[2]), dist2(dist2_), a(a_) {
    if constexpr (Fr) this->kt = *kt_;
  }
  __device__ __forceinline__ void refill() {
    if constexpr (cell_windows<D, R>()) {
      // stencil cell by cell, windows of kWin3 candidates inside a cell
      while (this->c == 0) {
        if (w0 >= re) {
          if (++j > 2) {
            j = 0;
            if (++k >= Rows<3>::N) break;
          }
          int64_t cx, cy, cz;
          cell_xyz<3>(G, B.skey[a], cx, cy, cz);
          const int64_t x = cx + j - 1, y = cy + (k % 3) - 1, z = cz + (k / 3) - 1;
          const bool in = x >= 0 && x < G.grid[0] && y >= 0 && y < G.grid[1] && z >= 0 && z < G.grid[2];
          const int64_t cell = x + G.grid[0] * (y + G.grid[1] * z);
          w0 = in ? B.start[cell] : 0;
          re = in ? B.start[cell + 1] : 0;
          this->set_window(win_code3(j - 1, (k % 3) - 1, (k / 3) - 1));
          continue;
        }
        const int32_t hi = re < w0 + kWin3 ? re : w0 + kWin3;
        this->c = window_bits_lean<3>(xm0, xm1, xm2, xm0[a], xm1[a], xm2[a], a, w0, hi, dist2);
        this->cb = w0;
        w0 = hi;
      }
    } else {
      while (this->c == 0) {
        if (w0 >= re) {
          if (++k >= Rows<D>::N) break;
          row_range<D>(G, B.start, B.skey[a], k, w0, re);
          continue;
        }
        const int32_t hi = re < w0 + 32 ? re : w0 + 32;
        this->c = window_bits_lean<D>(xm0, xm1, xm2, xm0[a], xm1[a], D == 3 ? xm2[a] : 0.0, a, w0, hi, dist2);
        this->cb = w0;
        w0 = hi;
      }
    }
  }
};

// The partner loops below leave together: a lane without partners left sits
// out the remaining trips (masked off), and the loop ends when no lane of the
// wave has one.  A loop whose lanes leave one by one makes the compiler carry
// every loop value in a second set of registers with copies on each trip.
template <int D, typename R, typename F>
__device__ __forceinline__ void for_each_partner(const SphBufs<R>& B, int64_t a, int nc, const CellGeom& G,
                                                 const double* const* XM, double dist2, F&& body) {
  const auto loop = [&](auto&& it) GCLSPH_INLINE {
    for (;;) {
      it.refill();
      const bool m = it.has();
      if (!__any(m)) break;
      if (m) body(it.take());
    }
  };
  loop(Stored<D, R>(B, a, nc));
  if (nc < 0) loop(Scanned<D, R>(B, a, G, XM, dist2));
}

// As for_each_partner, with the partner data split off: fetch(b) loads what
// the body needs of partner b, body(partner, terms[, window]) evaluates what
// the pair adds to the sums.  Pipe: the fetch of the next partner is issued
// before the body of the current one runs, so the loads overlap the pair
// arithmetic (at the cost of the registers holding both partners' data).
// Frames (3D FP32-split readers of partner records): kt holds the particle's
// separation constants and the body receives the partner's window constants.
//
// Quad: the four lanes of a particle evaluate four partners of a window at
// once and every lane adds their terms in partner order, so the sums are those
// of one lane, bit for bit, whatever a launch chooses.  A particle's partners
// are a serial loop (~36 trips in 2D, ~160 in 3D), and a small problem leaves
// most of the 1024 SIMDs without a wave: there a quad finishes in about a
// third of the trips.  With the chip full the extra selection and additions
// (~50 instructions per trip beside a body of ~100) only cost.
template <bool Pipe, bool Quad, int D, int N, typename R, bool Frames = false, typename Fetch, typename F>
__device__ __forceinline__ Sums<N, R> sum_partners(const SphBufs<R>& B, int64_t a, int nc, const CellGeom& G,
                                                   const double* const* XM, double dist2, Fetch&& fetch, F&& body,
                                                   const FrameK3* kt = nullptr) {
  constexpr bool Fr = Frames && D == 3 && std::is_same<R, float>::value;
  using W = typename std::conditional<Fr, Win3, NoWin>::type;
  Sums<N, R> sum;
  auto run = [&](const bool on, const auto& f, const W& w) GCLSPH_INLINE {
    if constexpr (Quad) {
      Terms<N, R> t;
      if (on) {
        if constexpr (Fr) body(f, t, w);
        else body(f, t);
      }
      sum.add_quad(t);
    } else if (on) {
      Terms<N, R> t;
      if constexpr (Fr) body(f, t, w);
      else body(f, t);
      sum.add(t);
    }
  };
  auto one_by_one = [&](auto&& it) GCLSPH_INLINE {
    for (;;) {
      it.refill();
      if (!__any(it.has())) break;
      W w{};
      if constexpr (Quad) {
        bool on;
        const int32_t b = it.take_quad(on, int32_t(a), w);
        run(on, fetch(b), w);
      } else if (it.has()) {
        run(true, fetch(it.take(w)), w);
      }
    }
  };
  if constexpr (!Pipe) {
    one_by_one(Stored<D, R, Fr>(B, a, nc, kt));
  } else {
    // two partners in flight, alternating between two sets of registers; a lane
    // without a next partner fetches a valid address again and skips the body
    Stored<D, R, Fr> it(B, a, nc, kt);
    // this lane's next partner; `none` (a valid index) and on = false without one
    auto take = [&](bool& on, const int32_t none, W& w) GCLSPH_INLINE {
      if constexpr (Quad) {
        return it.take_quad(on, none, w);
      } else {
        on = it.has();
        return on ? it.take(w) : none;
      }
    };
    it.refill();
    if (__any(it.has())) {
      W w0{}, w1{};
      bool m0, m1;
      int32_t b0 = take(m0, int32_t(a), w0);
      auto f0 = fetch(b0);
      for (;;) {
        it.refill();
        bool more = __any(it.has());
        const int32_t b1 = take(m1, b0, w1);
        auto f1 = fetch(b1);
        run(m0, f0, w0);
        if (!more) break;
        it.refill();
        more = __any(it.has());
        b0 = take(m0, b1, w0);
        f0 = fetch(b0);
        run(m1, f1, w1);
        if (!more) break;
      }
    }
  }
  if (nc < 0) one_by_one(Scanned<D, R, Fr>(B, a, G, XM, dist2, kt));
  return sum;
}

// The same over records staged in LDS (2D, one lane a particle, stored windows
// only): fetch(b, i) reads record b, staged at place i.
template <int N, typename R, typename Fetch, typename F>
__device__ __forceinline__ Sums<N, R> sum_staged(const SphBufs<R>& B, int64_t a, int nc, const RowMap& map,
                                                 Fetch&& fetch, F&& body) {
  Sums<N, R> sum;
  const uint64_t* pe = B.NE + a;
  uint64_t nxt = *pe;
  int left = nc;
  uint32_t c = 0;
  int32_t cb = 0, at = 0;
  for (;;) {
    if (c == 0 && left > 0) {
      uint32_t base;
      split_entry(nxt, c, base);
      cb = int32_t(base);
      at = cb + map.at(cb);
      --left;
      pe += B.n;
      nxt = *pe;
    }
    if (!__any(c != 0)) return sum;
    if (c != 0) {
      const int32_t k = __builtin_ctz(c);
      const auto f = fetch(cb + k, at + k);
      c &= c - 1;
      Terms<N, R> t;
      body(f, t);
      sum.add(t);
    }
  }
}

// ---------------------------------------------------------------- the pair
// Squared distance as the cut-offs compare it: FP64 unfused, as the reference
// has it.
template <int D>
__device__ __forceinline__ double dist2_of(const double* dx) {
  return dotd<D>(dx, dx);
}
template <int D>
__device__ __forceinline__ float dist2_of(const float* dx) {
  return dotf<D>(dx, dx);
}
__device__ __forceinline__ double root_of(double x) { return sqrt_d(x); }
__device__ __forceinline__ float root_of(float x) { return __builtin_amdgcn_sqrtf(x); }
// What a pair takes from its particle alone.
template <typename R>
struct Own {
  R rho;   // ρ_a
  R drho;  // what the records hold: ρ_a, or δρ_a in FP32-split
  R P;
  R mPi;   // -m0/ρ_a, of the pressure term
  int32_t pt;
};
template <typename R>
__device__ __forceinline__ Own<R> own_of(R drho, R P, int32_t pt, const SphConst& C) {
#pragma clang fp contract(off)
  Own<R> o;
  o.drho = drho;
  o.P = P;
  o.pt = pt;
  if constexpr (std::is_same<R, double>::value) {
    o.rho = drho;
    o.mPi = -C.m0 * (1.0 / drho);
  } else {
    o.rho = C.f_rho0 + drho;
    o.mPi = -C.f_m0 * __builtin_amdgcn_rcpf(o.rho);
  }
  return o;
}

// What the pair (a, b) adds to a's acceleration (t.v[0..D-1]) and ∂ρ/∂t
// (t.v[D]): ∂ρ∂tDDT! (src/gpukernels_sph.jl:579-625), ∂v∂t! (:755-772), ∂v∂t_av!
// (:869-897), ∂v∂t_visc! (:967-980), ∂v∂tpF! (:1387-1397) and the wall force k
// (0: 2dx, 1: bound_l).  dx, dv: separation and relative velocity of the state
// the rates are taken at; dg, rg2, rg: the separation (and its length) ∇W and
// the wall force are taken at (xⁿ; Same: dx is it).  ∇W = dg·dwr, so the terms
// along ∇W share one coefficient of dg.  The terms every pair has are evaluated
// and selected, without branches.  q: the partner's record; rb, ptb, Pb its
// density as held, type and pressure.
template <int D, bool G7, bool Same, typename Q>
__device__ __forceinline__ void pair_terms(const SphConst& C, const StepFlags& F, const Own<double>& o, const Q& q,
                                           double rb, int32_t ptb, double Pb, const double* dx, const double* dv,
                                           const double* dg, double rg2, double rg, int k, Terms<D + 1, double>& t) {
#pragma clang fp contract(off)
  const double dwr = dWr(rg2, rg, C);
  const double r2 = Same ? rg2 : dist2_of<D>(dx);
  const double dxdg = Same ? r2 : dotm<D>(dx, dg);
  const double dvdx = dotm<D>(dv, dx);
  const double dvdg = Same ? dvdx : dotm<D>(dv, dg);
  const Inv3<double> iv = pair_inv(q, rb, o.rho + rb, r2 + C.eta2);
  const bool both = o.pt > 0 && ptb > 0;
  {  // ∂ρ/∂t: m0 dwr (dv·dg - 2hδc0 (ρb - ρa - hydrostatic) (dx·dg) / (ρb (r² + η²))), diffusion for ptype > 1 only
    const double e = C.DDTkh * ((rb - o.rho) - hydro_drho_d<G7>(C.DDTgz * dx[1], C)) * iv.den * dxdg;
    // selected, not scaled by 0: a partner's NaN or infinite density stops here
    const double w = o.pt > 1 ? fma_(-e, iv.rhob, dvdg) : dvdg;
    t.v[D] = both ? C.m0 * dwr * w : 0.0;
  }
  double f = (o.P + Pb) * iv.rhob * o.mPi;             // pressure
  const double av = C.av * fmin(dvdx, 0.0) * iv.den;  // artificial viscosity, approaching pairs
  f = both ? fma_(av, iv.sum, f) : f;
  f = same_kind(o.pt, ptb) ? f * dwr : 0.0;
  double ax[3] = {0.0, 0.0, 0.0};
  if (both) {
    if (F.nu_on) {
      const double term = C.nu4 * (dxdg * dwr) * (iv.sum * iv.den);
#pragma unroll
      for (int d = 0; d < D; ++d) ax[d] = term * dv[d];
    }
    if (F.s_on && r2 < C.st_t2) {
      const double g = surf_d(Same ? rg : sqrt_d(r2), C) * (1.0 / C.m0);
#pragma unroll
      for (int d = 0; d < D; ++d) ax[d] = fma_(g, dx[d], ax[d]);
    }
  }
  if ((o.pt > 0) != (ptb > 0) && rg2 < C.fb_t2[k]) {  // fbmolforce! (:1891-1901)
    const double q1 = C.fb_r0[k] / (rg + C.fb_eta2[k]);
    const double Fc = C.fb_d[k] * (powi_d(q1, 12) - powi_d(q1, 4)) / (rg2 + C.fb_eta2[k]);
#pragma unroll
    for (int d = 0; d < D; ++d) ax[d] = fma_(dg[d], Fc, ax[d]);
  }
#pragma unroll
  for (int d = 0; d < D; ++d) t.v[d] = fma_(f, dg[d], ax[d]);
}

// FP32-split: the same terms in FP32.
template <int D, bool G7, bool Same, typename Q>
__device__ __forceinline__ void pair_terms(const SphConst& C, const StepFlags& F, const Own<float>& o, const Q& q,
                                           float drb, int32_t ptb, float Pb, const float* dx, const float* dv,
                                           const float* dg, float rg2, float rg, int k, Terms<D + 1, float>& t) {
#pragma clang fp contract(off)
  const float dwr = dWr(rg2, rg, C);
  const float r2 = Same ? rg2 : dotf<D>(dx, dx);
  const float dvdx = dotf<D>(dv, dx);
  const float rhob = C.f_rho0 + drb;
  const Inv3<float> iv = pair_inv(q, rhob, o.rho + rhob, r2 + C.f_eta2);
  const bool both = o.pt > 0 && ptb > 0;
  const float dxg = (Same ? r2 : dotf<D>(dx, dg)) * dwr;  // dx·∇W
  {
    const float s = C.f_m0 * dwr * (Same ? dvdx : dotf<D>(dv, dg));
    const float vd = C.f_DDTkh * minus_hydro(drb - o.drho, C.f_DDTgz * dx[1], C) * iv.den;
    const float sd = fma_(-(vd * dxg * C.f_m0), iv.rhob, s);
    t.v[D] = both ? (o.pt > 1 ? sd : s) : 0.0f;
  }
  const float Pt = (o.P + Pb) * iv.rhob * o.mPi;
  float f = same_kind(o.pt, ptb) ? Pt : 0.0f;
  {
    const float dmu = C.f_h * fminf(dvdx, 0.0f) * iv.den;  // AV acts on approaching pairs only
    const float dPi = (-C.f_alpha * C.f_c0 * dmu) * (2.0f * iv.sum);
    f -= both ? dPi * C.f_m0 : 0.0f;
  }
  f *= dwr;
  float ax[3] = {0.0f, 0.0f, 0.0f};
  if (both) {
    if (F.nu_on) {
      const float term = 4.0f * C.f_nu * C.f_m0 * dxg * (iv.sum * iv.den);
#pragma unroll
      for (int d = 0; d < D; ++d) ax[d] = term * dv[d];
    }
    if (F.s_on) {
      const float r = Same ? rg : __builtin_amdgcn_sqrtf(r2);
      if (r < C.f_st_2h) {
        const float g = surf_f(r, C);
        if constexpr (Same) {
          f = fma_(g, C.f_inv_m0, f);
        } else {
#pragma unroll
          for (int d = 0; d < D; ++d) ax[d] = fma_(g * dx[d], C.f_inv_m0, ax[d]);
        }
      }
    }
  }
#pragma unroll
  for (int d = 0; d < D; ++d) ax[d] = fma_(f, dg[d], ax[d]);
  if ((o.pt > 0) != (ptb > 0) && rg < C.f_fb_r0[k]) {
    // wall force: FP32 while q = r0/(r + η²) < 32 (q^12 < 1.2e18, far inside
    // the FP32 range), FP64 for the (rare) closer pairs
    const float q1 = C.f_fb_r0[k] * __builtin_amdgcn_rcpf(rg + C.f_fb_eta2[k]);
    if (q1 < 32.0f) {
      const float q2 = q1 * q1, q4 = q2 * q2, q8 = q4 * q4;
      const float Fc = C.f_fb_d[k] * fma_(q4, q8, -q4) * __builtin_amdgcn_rcpf(rg2 + C.f_fb_eta2[k]);
#pragma unroll
      for (int d = 0; d < D; ++d) ax[d] = fma_(dg[d], Fc, ax[d]);
    } else {
      const double p1 = C.fb_r0[k] / (double(rg) + C.fb_eta2[k]);
      const double p2 = p1 * p1, p4 = p2 * p2, p8 = p4 * p4;
      const double Fc = C.fb_d[k] * (p4 * p8 - p4) / (double(rg2) + C.fb_eta2[k]);
#pragma unroll
      for (int d = 0; d < D; ++d) ax[d] += float(double(dg[d]) * Fc);
    }
  }
#pragma unroll
  for (int d = 0; d < D; ++d) t.v[d] = ax[d];
}

__device__ __forceinline__ double nanmax(double a, double b) { return (a > b || a != a) ? a : b; }

constexpr int kRedSlots = 64;

// Block maximum (NaN wins) folded into one of kRedSlots slots by an atomic max
// on its bit pattern (non-negative doubles order like their bits, NaN above
// +Inf); spreading blocks over many slots avoids one hot address.  Every
// thread of the block must call it.
template <int BS = kBlock>
__device__ __forceinline__ void block_max(double v, bool active, double* slots, int blk) {
  __shared__ double wm[BS / 64];
  double m = wave_max(active ? v : 0.0);
  if ((threadIdx.x & 63) == 0) wm[threadIdx.x >> 6] = m;
  __syncthreads();
  if (threadIdx.x == 0) {
    double r = wm[0];
#pragma unroll
    for (int w = 1; w < BS / 64; ++w) r = nanmax(r, wm[w]);
    atomic_max_nonneg(reinterpret_cast<unsigned long long*>(slots) + (blk % kRedSlots), r);
  }
  __syncthreads();
}

// Calls f with the scene source of L: the descriptor by value for one problem,
// the device descriptor array and maps for several.
template <typename R, typename Fn>
inline void with_scenes(const LaunchSet& L, Fn&& f) {
  if (L.one) f(OneScene<R>{*static_cast<const SceneDev<R>*>(L.one)});
  else f(ManyScenes<R>{static_cast<const SceneDev<R>*>(L.scenes), L.pmap, L.cmap, L.pmap512, L.qmap});
}

}  // namespace gclsph

// Particle-centric SPH step kernels.
//
// Every pair kernel of the reference (src/gpukernels_sph.jl) runs one thread per
// *pair* and scatters both halves with FP64 atomics.  Here one thread owns one
// particle `a` of the cell-sorted state and gathers over the 3^D cells around
// it; the pairs it visits are exactly the reference's neighbour list (same
// cells, r^2 < dist^2 at the positions of the last rebuild).  For the pair
// (a, b) it evaluates the reference's per-pair expression for a's side — with
// Δx = x_a - x_b, which is the reference's Δx or its exact negation — so the
// per-pair values match the reference's and only the summation order differs.
// Sums are per-thread and deterministic; there are no floating-point atomics.
//
// Pass 1 (tⁿ) fuses sphW!/sph∇W!, ∂ρ∂tDDT!, pressure!, ∂v∂t!, ∂v∂t_av!,
// ∂v∂t_visc!, ∂v∂t_addgrav!, fbmolforce!, ∂v∂tpF! and the three half-step
// updates (src/sphproblem.jl:244-274).  Pass 2 (t^{n+1/2}) fuses the second
// evaluation with symplectic_update! and the Δt / rebuild reductions
// (src/sphproblem.jl:277-335).
//
// R = double: the Float64 path.  Squared distances, the branch decisions (r < r0
// as a test of r², clamps) and the updates are evaluated in the reference's
// operation order with FMA contraction off, so they see the same values as the
// reference would.  The pair terms are the reference's to a few ulp: their ten
// divisions, square roots and powfancy7th are the arithmetic of sph_device.hpp
// (~85 VALU instructions per pair, ~330 as written, when VALU issue bound the
// passes).  1.02 M particles in 2D: a step 0.77 -> 0.50 ms; 191 k in 3D: 1.45x
// per call.
// R = float: the FP32-split path (density stored as ρ-ρ0, FP32 pair terms
// summed in FP64, Float64 positions and Δt).
#include <atomic>

#include "sph_device.hpp"

namespace gclsph {

// Pass kernels come in variants that differ only in code generation and
// launch shape (so their results are bit-identical: one thread computes one
// particle whatever the block): Pipe fetches the next partner's data before the
// current pair body (two register sets), W asks the compiler for at least W
// waves per SIMD (fewer registers; W = 3 for exactly three, which in 3D
// FP32-split keeps pass 2's partner records in L1: 848 us for 883,376
// particles, 930 with four), BS is the block size.  The step driver
// picks one per pass by timing them on live steps.
//
// ---- pass 1 ---------------------------------------------------------------
template <int D, typename R, typename SS, bool Pipe, int W, int BS, bool G7, bool Quad>
__global__ __launch_bounds__(BS) __attribute__((amdgpu_waves_per_eu(W, W == 3 ? 3 : 8))) void k_pass1(SS ss) {
#pragma clang fp contract(off)
  GCLSPH_SCENE_PAIR(ss, BS, Quad);
  const StepCtl* ctl = B.ctl;
  const int p = cur_parity(ctl), pp = cur_pparity(ctl), rebuilt = ctl->rebuild;
  const double dt = ctl->dt;
  constexpr bool kStage = D == 2 && !Quad;  // a quad's block has 64 particles: as much to stage for a quarter of the use
  bool staged = false;
  RowMap map{};
  int nc = 0;
  using Nb = typename Records<D, R>::N;
  __shared__ uint4 lds[kStage ? kStagedWords : 1][kStage ? kStageCap<BS> : 1];
  if constexpr (kStage) {
    const int64_t a0 = int64_t(m.y) * BS;
    if (a0 >= B.n) return;  // whole block
    nc = a < B.n ? B.NC[a] : 0;
    staged = stage_rows<BS, kStagedWords>(lds, B.PRN, B, G, a0, nc, map);
    if (a >= B.n) return;
  } else {
    if (a >= B.n) return;
    nc = B.NC[a];
  }
  const double* X[3] = {B.X[p][0], B.X[p][1], B.X[p][D == 3 ? 2 : 1]};
  const R* V[3] = {B.V[p][0], B.V[p][1], B.V[p][D == 3 ? 2 : 1]};
  const R* RHO = B.RHO[p];
  const int32_t* PT = B.PT[pp];
  const double* XM[3];
  membership_ptrs<D>(B, F, p, rebuilt, XM);

  double xa[3];
  R va[3];
#pragma unroll
  for (int k = 0; k < D; ++k) {
    xa[k] = X[k][a];
    va[k] = V[k][a];
  }
  const R sa = RHO[a];
  const int32_t pta = PT[a];
  constexpr int kDrho = D;  // sums: D accelerations, ∂ρ/∂t

  auto fetch = [&](const int32_t b, const auto... at) GCLSPH_INLINE {
    if constexpr (sizeof...(at) > 0) return ld_staged<Nb, kStagedWords>(lds, at..., B.PRN, b, B.n);
    else return ld_rec<Nb>(B.PRN, b, B.n);
  };
  if constexpr (std::is_same<R, double>::value) {
    const Own<R> own = own_of<R>(sa, B.PN[a], pta, C);
    auto pair = [&](const Nb& q, auto& t) GCLSPH_INLINE {
      double dx[3], dv[3];
#pragma unroll
      for (int d = 0; d < D; ++d) {
        dx[d] = xa[d] - q.x[d];
        dv[d] = va[d] - q.v[d];
      }
      const double r2 = dist2_of<D>(dx);
      pair_terms<D, G7, true>(C, F, own, q, q.rho, q.pt, q.P, dx, dv, dx, r2, root_of(r2), 0, t);
    };
    Sums<D + 1, R> sum;
    if constexpr (kStage) {
      if (staged) sum = sum_staged<D + 1, R>(B, a, nc, map, fetch, pair);
      else sum = sum_partners<Pipe, Quad, D, D + 1, R>(B, a, nc, G, XM, C.dist2, fetch, pair);
    } else {
      sum = sum_partners<Pipe, Quad, D, D + 1, R>(B, a, nc, G, XM, C.dist2, fetch, pair);
    }
    // ∂v∂t_addgrav!, then the half-step updates (:270-274)
    double av[3];
#pragma unroll
    for (int d = 0; d < D; ++d) av[d] = sum.get(d);
    if (!writer) return;
    av[1] = av[1] - C.g;
    double rh0, vh0[3], xh0[3];
    if (F.synced_prev) {
      rh0 = sa;
#pragma unroll
      for (int d = 0; d < D; ++d) {
        vh0[d] = va[d];
        xh0[d] = xa[d];
      }
    } else {
      const bool mv = rebuilt;  // the reorder moved the old half-step state to XH/VH/RH
      rh0 = mv ? B.RH[a] : B.RH2[a];
#pragma unroll
      for (int d = 0; d < D; ++d) {
        vh0[d] = mv ? B.VH[d][a] : B.VH2[d][a];
        xh0[d] = mv ? B.XH[d][a] : B.XH2[d][a];
      }
    }
    const double hdt = dt * 0.5;
    double rv = rh0 + sum.get(kDrho) * hdt;
    if (rv < C.rho0 && pta < 0) rv = C.rho0;
    const double Ph = eos_d(rv, pta, C);
    B.RH[a] = rv;
    B.PH[a] = Ph;
    PartnerH64<D> rec{};
#pragma unroll
    for (int d = 0; d < D; ++d) {
      double vv = vh0[d];
      if (pta > 1) vv += av[d] * hdt;
      const double xh = xh0[d] + vv * hdt;
      B.VH[d][a] = vv;
      B.XH[d][a] = xh;
      rec.xn[d] = xa[d];
      rec.xh[d] = xh;
      rec.vh[d] = vv;
    }
    rec.rh = rv;
    rec.P = Ph;
    rec.pt = pta;
    set_irho(rec);
    st_rec(B.PRH, a, rec, B.n);
  } else {
    // ---------------- FP32-split
    const Own<R> own = own_of<R>(sa, B.PN[a], pta, C);
    const FrameK3 kt = particle_k<D, R>(B, C, G, a, xa);
    auto pair = [&](const Nb& q, auto& t, const auto&... win) GCLSPH_INLINE {
      float dx[3], dv[3];
#pragma unroll
      for (int d = 0; d < D; ++d) {
        dx[d] = sep_x(xa, q, d, win...);
        dv[d] = va[d] - q.v[d];
      }
      const float r2 = dist2_of<D>(dx);
      pair_terms<D, G7, true>(C, F, own, q, q.rho, rec_pt(q), rec_P(q, C), dx, dv, dx, r2, root_of(r2), 0, t);
    };
    Sums<D + 1, R> sum;
    if constexpr (kStage) {
      if (staged) sum = sum_staged<D + 1, R>(B, a, nc, map, fetch, pair);
      else sum = sum_partners<Pipe, Quad, D, D + 1, R, true>(B, a, nc, G, XM, C.dist2, fetch, pair, &kt);
    } else {
      sum = sum_partners<Pipe, Quad, D, D + 1, R, true>(B, a, nc, G, XM, C.dist2, fetch, pair, &kt);
    }
    float av[3];
#pragma unroll
    for (int d = 0; d < D; ++d) av[d] = sum.get(d);
    if (!writer) return;
    av[1] = av[1] - C.f_g;
    float rh0, vh0[3];
    double xh0[3];
    if (F.synced_prev) {
      rh0 = sa;
#pragma unroll
      for (int d = 0; d < D; ++d) {
        vh0[d] = va[d];
        xh0[d] = xa[d];
      }
    } else {
      const bool mv = rebuilt;
      rh0 = mv ? B.RH[a] : B.RH2[a];
#pragma unroll
      for (int d = 0; d < D; ++d) {
        vh0[d] = mv ? B.VH[d][a] : B.VH2[d][a];
        xh0[d] = mv ? B.XH[d][a] : B.XH2[d][a];
      }
    }
    const float hdt = float(dt * 0.5);
    float rv = fma_(sum.get(kDrho), hdt, rh0);
    if (rv < 0.0f && pta < 0) rv = 0.0f;
    B.RH[a] = rv;
    const float Ph = eos_f(rv, pta, C);
    B.PH[a] = Ph;
    PartnerHX<D> rec{};
    double fr[3];
    particle_frame<D, R>(B, C, G, a, fr);
#pragma unroll
    for (int d = 0; d < D; ++d) {
      float vv = vh0[d];
      if (pta > 1) vv = fma_(av[d], hdt, vv);
      const double xh = fma_(double(vv), dt * 0.5, xh0[d]);
      B.VH[d][a] = vv;
      B.XH[d][a] = xh;
      put_x(rec.h, d, xh, fr);
      rec.h.vh[d] = vv;
      rec.dn[d] = float(xh - xa[d]);
    }
    rec.h.rh = rv;
    set_pt(rec.h, pta, Ph);
    if (F.synced_prev) st_rec(B.PRH, a, rec.h, B.n);  // pass 2 derives xⁿ
    else st_rec(B.PRH, a, rec, B.n);
  }
}

// ---- pass 2 + symplectic update ------------------------------------------
template <int D, typename R, typename SS, bool Pipe, int W, int BS, bool G7, bool Quad>
__global__ __launch_bounds__(BS) __attribute__((amdgpu_waves_per_eu(W, W == 3 ? 3 : 8))) void k_pass2(SS ss) {
#pragma clang fp contract(off)
  GCLSPH_SCENE_PAIR(ss, BS, Quad);
  StepCtl* ctl = B.ctl;
  const int p = cur_parity(ctl), q = p ^ 1, pp = cur_pparity(ctl), rebuilt = ctl->rebuild;
  const double dt = ctl->dt;
  const bool active = a < B.n;
  double red_cdx = 0.0, red_acc = 0.0, red_visc = 0.0;
  constexpr bool kStage = D == 2 && !Quad;
  bool staged = false;
  RowMap map{};
  const int nc = active ? B.NC[a] : 0;
  __shared__ uint4 lds[kStage ? kStagedWords : 1][kStage ? kStageCap<BS> : 1];
  if constexpr (kStage) {
    const int64_t a0 = int64_t(m.y) * BS;
    if (a0 < B.n) staged = stage_rows<BS, kStagedWords>(lds, B.PRH, B, G, a0, nc, map);
  }
  if (active) {
    const double* X[3] = {B.X[p][0], B.X[p][1], B.X[p][D == 3 ? 2 : 1]};
    const double* XH[3] = {B.XH[0], B.XH[1], B.XH[D == 3 ? 2 : 1]};
    const R* VH[3] = {B.VH[0], B.VH[1], B.VH[D == 3 ? 2 : 1]};
    const R* RH = B.RH;
    const int32_t* PT = B.PT[pp];
    const double* XM[3];
    membership_ptrs<D>(B, F, p, rebuilt, XM);
    double xa[3], xha[3];
    R vha[3];
#pragma unroll
    for (int k = 0; k < D; ++k) {
      xa[k] = X[k][a];
      xha[k] = XH[k][a];
      vha[k] = VH[k][a];
    }
    const R sha = RH[a];
    const int32_t pta = PT[a];
    constexpr int kDrho = D;  // sums: D accelerations, ∂ρ/∂t
    R av[3];
    R Pha, drho_v;
    if constexpr (std::is_same<R, double>::value) {
      const double rhoa = sha;
      Pha = B.PH[a];
      const Own<R> own = own_of<R>(sha, Pha, pta, C);
      using Nb = PartnerH64<D>;
      auto fetch = [&](const int32_t b, const auto... at) GCLSPH_INLINE {
        if constexpr (sizeof...(at) > 0) return ld_staged<Nb, kStagedWords>(lds, at..., B.PRH, b, B.n);
        else return ld_rec<Nb>(B.PRH, b, B.n);
      };
      auto pair = [&](const Nb& q, auto& t) GCLSPH_INLINE {
        double dxn[3], dx[3], dv[3];
#pragma unroll
        for (int d = 0; d < D; ++d) {
          dxn[d] = xa[d] - q.xn[d];
          dx[d] = xha[d] - q.xh[d];
          dv[d] = vha[d] - q.vh[d];
        }
        // ∇W from pass 1 (positions xⁿ, src/sphproblem.jl:246,281); the wall
        // force at xⁿ with (bound_D, bound_l) (:295)
        const double r2n = dist2_of<D>(dxn);
        pair_terms<D, G7, false>(C, F, own, q, q.rh, q.pt, q.P, dx, dv, dxn, r2n, root_of(r2n), 1, t);
      };
      Sums<D + 1, R> sum;
      if constexpr (kStage) {
        if (staged) sum = sum_staged<D + 1, R>(B, a, nc, map, fetch, pair);
        else sum = sum_partners<Pipe, Quad, D, D + 1, R>(B, a, nc, G, XM, C.dist2, fetch, pair);
      } else {
        sum = sum_partners<Pipe, Quad, D, D + 1, R>(B, a, nc, G, XM, C.dist2, fetch, pair);
      }
#pragma unroll
      for (int d = 0; d < D; ++d) av[d] = sum.get(d);
      av[1] = av[1] - C.g;
      drho_v = sum.get(kDrho);
      if (writer) {
        // symplectic_update! (src/gpukernels_sph.jl:1204-1245)
        const double epsi = -(drho_v / rhoa) * dt;
        double rv = B.RHO[p][a] * (2 - epsi) / (2 + epsi);
        if (rv < C.rho0 && pta <= 1) rv = C.rho0;
        const double Pn = eos_d(rv, pta, C);
        B.RHO[q][a] = rv;
        B.PN[a] = Pn;
        if (F.corr_on) B.RH2[a] = rv;
        const double ml = pta > 1 ? 1.0 : 0.0;
        double xn[3], vn[3];
        PartnerN64<D> rec{};
#pragma unroll
        for (int d = 0; d < D; ++d) {
          double vv = B.V[p][d][a];
          double nv = vv + av[d] * dt * ml;
          double dd = (vv + nv) * 0.5 * dt;
          double cd = dd;
          if (F.need_cdx) {
            cd = (rebuilt ? 0.0 : B.CDX[d][a]) + dd;
            B.CDX[d][a] = cd;
          }
          red_cdx = fmax(red_cdx, fabs(cd)) + (cd != cd ? cd : 0.0);
          double xv = xa[d] + dd;
          xn[d] = xv;
          vn[d] = nv;
          B.V[q][d][a] = nv;
          B.X[q][d][a] = xv;
          rec.x[d] = xv;
          rec.v[d] = nv;
          if (F.corr_on) {
            B.VH2[d][a] = nv;
            B.XH2[d][a] = xv;
          }
        }
        rec.rho = rv;
        rec.P = Pn;
        rec.pt = pta;
        set_irho(rec);
        st_rec(B.PRN, a, rec, B.n);  // partner record of the next step's pass 1
        if (F.ts) {
          red_acc = sqrt(dotd<D>(av, av));
          if (F.visc_in_pass2) red_visc = fabs(C.h * dotd<D>(vn, xn) / (dotd<D>(xn, xn) + C.dt_eta2));
        }
      }
    } else {
      const float rhoa = C.f_rho0 + sha;
      Pha = B.PH[a];
      const Own<R> own = own_of<R>(sha, Pha, pta, C);
      // tⁿ separation from the half-step state when x½ = xⁿ + v½·Δt/2, else
      // from the displacement x½ - xⁿ that pass 1 appended to the records
      // xⁿa - xⁿb = (x½a - x½b) - (da - db) with d = x½ - xⁿ, the displacement
      // part in FP32 (its size is of order |v|·Δt): derived, d = v½·Δt/2
      // (PartnerH records); else d from the records (PartnerHX).  The choice
      // holds for the whole step, so the loop is compiled once for each.
      const float fhdt = float(dt * 0.5);
      float dna[3];
#pragma unroll
      for (int d = 0; d < D; ++d) dna[d] = float(xha[d] - xa[d]);
      const FrameK3 kt = particle_k<D, R>(B, C, G, a, xha);
      auto gather = [&](auto derive_c) GCLSPH_INLINE {
      constexpr bool derive = decltype(derive_c)::value;
      using Nb = std::conditional_t<derive, PartnerH<D>, PartnerHX<D>>;
      auto fetch = [&](const int32_t b, const auto... at) GCLSPH_INLINE {
        if constexpr (sizeof...(at) > 0) return ld_staged<Nb, kStagedWords>(lds, at..., B.PRH, b, B.n);
        else return ld_rec<Nb>(B.PRH, b, B.n);
      };
      auto pair = [&](const Nb& r, auto& t, const auto&... win) GCLSPH_INLINE {
        const PartnerH<D>* qp;
        if constexpr (derive) qp = &r;
        else qp = &r.h;
        const PartnerH<D>& q = *qp;
        float dxn[3], dx[3], dv[3];
#pragma unroll
        for (int d = 0; d < D; ++d) {
          dx[d] = sep_x(xha, q, d, win...);
          dv[d] = vha[d] - q.vh[d];
          if constexpr (derive) dxn[d] = fma_(-dv[d], fhdt, dx[d]);
          else dxn[d] = dx[d] - (dna[d] - r.dn[d]);
        }
        const float r2n = dist2_of<D>(dxn);
        pair_terms<D, G7, false>(C, F, own, q, q.rh, rec_pt(q), rec_P(q, C), dx, dv, dxn, r2n, root_of(r2n), 1, t);
      };
      if constexpr (kStage) {
        if (staged) return sum_staged<D + 1, R>(B, a, nc, map, fetch, pair);
      }
      return sum_partners<Pipe, Quad, D, D + 1, R, true>(B, a, nc, G, XM, C.dist2, fetch, pair, &kt);
      };
      const auto sum = F.synced_prev ? gather(std::true_type{}) : gather(std::false_type{});
#pragma unroll
      for (int d = 0; d < D; ++d) av[d] = sum.get(d);
      av[1] = av[1] - C.f_g;
      drho_v = sum.get(kDrho);
      if (writer) {
        // symplectic update on δρ: ρ(2-ε)/(2+ε) - ρ0 = (2δρ - ε(2ρ0 + δρ)) / (2 + ε)
        const float fdt = float(dt);
        const float erate = -(drho_v / rhoa), epsi = erate * fdt;
        const float dr_n = B.RHO[p][a];
          float rv = fma_(2.0f, dr_n, -(epsi * fma_(2.0f, C.f_rho0, dr_n))) / fma_(erate, fdt, 2.0f);
        if (rv < 0.0f && pta <= 1) rv = 0.0f;
        B.RHO[q][a] = rv;
        const float Pn = eos_f(rv, pta, C);
        B.PN[a] = Pn;
        if (F.corr_on) B.RH2[a] = rv;
        const float ml = pta > 1 ? 1.0f : 0.0f;
        double xn[3], vn[3];
        PartnerN<D> rec{};
        double fr[3];
        particle_frame<D, R>(B, C, G, a, fr);
#pragma unroll
        for (int d = 0; d < D; ++d) {
          float vv = B.V[p][d][a];
          float nv = fma_(av[d] * fdt, ml, vv);
          const double vm = (double(vv) + double(nv)) * 0.5;
          double cd = vm * dt;
          if (F.need_cdx) {
            cd = fma_(vm, dt, rebuilt ? 0.0 : B.CDX[d][a]);
            B.CDX[d][a] = cd;
          }
          red_cdx = fmax(red_cdx, fabs(cd)) + (cd != cd ? cd : 0.0);
          const double xv = fma_(vm, dt, xa[d]);
          xn[d] = xv;
          vn[d] = nv;
          B.V[q][d][a] = nv;
          B.X[q][d][a] = xv;
          put_x(rec, d, xv, fr);
          rec.v[d] = nv;
          if (F.corr_on) {
            B.VH2[d][a] = nv;
            B.XH2[d][a] = xv;
          }
        }
        rec.rho = rv;
        set_pt(rec, pta, Pn);
        st_rec(B.PRN, a, rec, B.n);  // partner record of the next step's pass 1
        if (F.ts) {
          float a2 = dotf<D>(av, av);
          red_acc = sqrt(double(a2));
          if (F.visc_in_pass2) red_visc = fabs(C.h * dotd<D>(vn, xn) / (dotd<D>(xn, xn) + C.dt_eta2));
        }
      }
    }
    if (F.want_out && writer) {
#pragma unroll
      for (int d = 0; d < D; ++d) B.ACC[d][a] = av[d];
      B.DRHO[a] = drho_v;
      B.PBUF[a] = Pha;
    }
  }
  block_max<BS>(red_cdx, active, B.RED, m.y);
  if (F.ts) {
    block_max<BS>(red_acc, active, B.RED + kRedSlots, m.y);
    if (F.visc_in_pass2) block_max<BS>(red_visc, active, B.RED + 2 * kRedSlots, m.y);
  }
}

// ------------------------------------------------------------ host launchers
namespace {
// Blocks of BS threads covering every problem of L: the 256-particle blocks of
// the particle map, twice as many 128-thread blocks, or the 512-particle map.
template <int BS>
unsigned pass_grid(const LaunchSet& L) {
  return BS == 256 ? L.pblocks : BS == 128 ? 2 * L.pblocks : L.pblocks512;
}
template <int D, typename R, bool Pipe, int W, int BS, bool G7 = true, bool Quad = false>
void pass1_as(const LaunchSet& L, hipStream_t s, size_t lds) {
  with_scenes<R>(L, [&](auto ss) {
    k_pass1<D, R, decltype(ss), Pipe, W, BS, G7, Quad><<<Quad ? L.qblocks : pass_grid<BS>(L), BS, lds, s>>>(ss);
  });
}
template <int D, typename R, bool Pipe, int W, int BS, bool G7 = true, bool Quad = false>
void pass2_as(const LaunchSet& L, hipStream_t s, size_t lds) {
  with_scenes<R>(L, [&](auto ss) {
    k_pass2<D, R, decltype(ss), Pipe, W, BS, G7, Quad><<<Quad ? L.qblocks : pass_grid<BS>(L), BS, lds, s>>>(ss);
  });
}
// Unused dynamic LDS per block of BS threads that leaves room for at most
// kPassCapWaves waves per SIMD (B = 4·kPassCapWaves·64/BS blocks per CU: B
// blocks fit the CU's LDS, B + 1 do not); 0 when the cap would need more LDS
// than a block may have.  Queried once per device.
size_t cap_lds(int bs) {
  static std::atomic<int64_t> per_cu[64], per_block[64];  // 0: not queried yet
  int dev = 0;
  GCL_HIP(hipGetDevice(&dev));
  if (dev < 0 || dev >= 64) return 0;
  if (per_cu[dev].load() == 0) {
    int cu = 0, blk = 0;
    GCL_HIP(hipDeviceGetAttribute(&cu, hipDeviceAttributeMaxSharedMemoryPerMultiprocessor, dev));
    GCL_HIP(hipDeviceGetAttribute(&blk, hipDeviceAttributeMaxSharedMemoryPerBlock, dev));
    per_block[dev].store(blk);
    per_cu[dev].store(cu);
  }
  const size_t cu = size_t(per_cu[dev].load()), blk = size_t(per_block[dev].load());
  const size_t blocks = size_t(4 * kPassCapWaves * 64 / bs);
  const size_t lds = cu / (blocks + 1) + 1024;  // the static LDS of a 3D pass block is below 1 KiB (2D has no cap)
  return blocks * lds <= cu && lds <= blk ? lds : 0;
}
// Code generation cg, 3D: 0 pipelined; 1 not pipelined; 2 pipelined, three waves
// per SIMD; 3 (FP32-split) not pipelined, >= 5 waves/SIMD, which makes FP64
// spill: there it is 1.  2D, where the records are staged, has one: four waves
// per SIMD, as the staged records allow (FP64 pass 2 by itself would take the
// registers of three: 246 us, 230 so, 1.02 M particles).  Prefetch concerns its
// blocks whose rows don't fit alone: FP32-split has it (614,072 particles, smoothing
// length 2.2 and 3 times the usual: a step 899 -> 843, 1841 -> 1789 us), FP64 has
// no registers for it.
template <int D, typename R, int BS>
void pass1_cg(const LaunchSet& L, hipStream_t s, int cg, size_t lds) {
  if constexpr (D == 2) {
    pass1_as<D, R, std::is_same<R, float>::value, 4, BS>(L, s, 0);
  } else {
    constexpr bool f32 = std::is_same<R, float>::value;
    switch (cg) {
      case 0: pass1_as<D, R, true, 1, BS>(L, s, lds); break;
      case 2: pass1_as<D, R, true, 3, BS>(L, s, lds); break;
      case 3: pass1_as<D, R, false, f32 ? 5 : 1, BS>(L, s, lds); break;
      default: pass1_as<D, R, false, 1, BS>(L, s, lds); break;
    }
  }
}
template <int D, typename R, int BS>
void pass2_cg(const LaunchSet& L, hipStream_t s, int cg, size_t lds) {
  if constexpr (D == 2) {
    pass2_as<D, R, std::is_same<R, float>::value, 4, BS>(L, s, 0);
  } else {
    constexpr bool f32 = std::is_same<R, float>::value;
    switch (cg) {
      case 0: pass2_as<D, R, true, 1, BS>(L, s, lds); break;
      case 2: pass2_as<D, R, true, 3, BS>(L, s, lds); break;
      case 3: pass2_as<D, R, false, f32 ? 5 : 1, BS>(L, s, lds); break;
      default: pass2_as<D, R, false, 1, BS>(L, s, lds); break;
    }
  }
}
}  // namespace

// variant = cg + kPassCodegen·bs + kPassCodegen·kPassBlockSizes·oc (bs 0: 256,
// 1: 128, 2: 512 threads per block; oc 1: occupancy cap)
template <int D, typename R>
void launch_pass1(const LaunchSet& L, hipStream_t s, int variant) {
  if constexpr (std::is_same<R, double>::value) {
    if (!L.gamma7) {  // another γ: one kernel, whatever the variant, and its quads
      if (variant == kPassQuad) pass1_as<D, R, false, 1, 256, false, true>(L, s, 0);
      else pass1_as<D, R, false, 1, 256, false>(L, s, 0);
      return;
    }
  }
  if (variant == kPassQuad) {
    pass1_as<D, R, true, 1, 256, true, true>(L, s, 0);
    return;
  }
  const int cg = variant % kPassCodegen, bs = pass_block_size(variant);
  const size_t lds = pass_cap(variant) ? cap_lds(bs) : 0;
  switch (bs) {
    case 128: pass1_cg<D, R, 128>(L, s, cg, lds); break;
    case 512: pass1_cg<D, R, 512>(L, s, cg, lds); break;
    default: pass1_cg<D, R, 256>(L, s, cg, lds); break;
  }
}
template <int D, typename R>
void launch_pass2(const LaunchSet& L, hipStream_t s, int variant) {
  if constexpr (std::is_same<R, double>::value) {
    if (!L.gamma7) {  // another γ: one kernel, whatever the variant, and its quads
      if (variant == kPassQuad) pass2_as<D, R, false, 1, 256, false, true>(L, s, 0);
      else pass2_as<D, R, false, 1, 256, false>(L, s, 0);
      return;
    }
  }
  if (variant == kPassQuad) {
    pass2_as<D, R, true, 1, 256, true, true>(L, s, 0);
    return;
  }
  const int cg = variant % kPassCodegen, bs = pass_block_size(variant);
  const size_t lds = pass_cap(variant) ? cap_lds(bs) : 0;
  switch (bs) {
    case 128: pass2_cg<D, R, 128>(L, s, cg, lds); break;
    case 512: pass2_cg<D, R, 512>(L, s, cg, lds); break;
    default: pass2_cg<D, R, 256>(L, s, cg, lds); break;
  }
}

#define GCLSPH_INSTANTIATE_PASS(D, R)                                     \
  template void launch_pass1<D, R>(const LaunchSet&, hipStream_t, int);  \
  template void launch_pass2<D, R>(const LaunchSet&, hipStream_t, int);

GCLSPH_INSTANTIATE_PASS(2, double)
GCLSPH_INSTANTIATE_PASS(3, double)
GCLSPH_INSTANTIATE_PASS(2, float)
GCLSPH_INSTANTIATE_PASS(3, float)

}  // namespace gclsph

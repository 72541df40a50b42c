// SPH step kernels other than the two pair passes (sph_pass.hip): the rebuild
// (counting sort, reorder, membership store), the corrections after the update
// (DPC, XSPH, CSPM), the Δt / time / rebuild-flag commit, the diagnostics,
// and the host launchers.  Conventions as in sph_pass.hip: one thread per
// particle of the cell-sorted state, gathers over the stored neighbour-list
// membership, FP64 in the reference's operation order without FMA contraction
// (R = double) or FP32 pair terms with FP64 sums (R = float, FP32-split).
#include "sph_device.hpp"

namespace gclsph {

// acc·16 + the four bits (r_u < dist2), candidate 0 the highest: four FP64
// compares into SGPR lane masks, then four add-with-carry steps acc+acc+bit.
// Each mask is read three instructions after it is written (gfx950 needs two
// wait states between a VALU write of an SGPR and its use as a carry-in).
__device__ __forceinline__ uint32_t push_lt4(uint32_t acc, double r0, double r1, double r2, double r3,
                                             double dist2) {
  uint64_t c0, c1, c2, c3, co;
  asm("v_cmp_gt_f64_e64 %1, %6, %7\n\t"
      "v_cmp_gt_f64_e64 %2, %6, %8\n\t"
      "v_cmp_gt_f64_e64 %3, %6, %9\n\t"
      "v_cmp_gt_f64_e64 %4, %6, %10\n\t"
      "v_addc_co_u32_e64 %0, %5, %0, %0, %1\n\t"
      "v_addc_co_u32_e64 %0, %5, %0, %0, %2\n\t"
      "v_addc_co_u32_e64 %0, %5, %0, %0, %3\n\t"
      "v_addc_co_u32_e64 %0, %5, %0, %0, %4"
      : "+v"(acc), "=&s"(c0), "=&s"(c1), "=&s"(c2), "=&s"(c3), "=&s"(co)
      : "s"(dist2), "v"(r0), "v"(r1), "v"(r2), "v"(r3));
  return acc;
}

// Window mask from the pushed bits: len candidates pushed in groups of four
// (candidate t at bit nc-1-t, nc = len rounded up to 4) become bit t, the
// candidates past len and the particle itself cleared.
__device__ __forceinline__ uint32_t window_mask(uint32_t acc, int32_t len, int64_t a, int32_t lo) {
  const int32_t nc = (len + 3) & ~3;
  uint32_t mk = __builtin_bitreverse32(acc << (32 - nc));
  if (len < 32) mk &= (1u << len) - 1u;
  const int32_t self = int32_t(a) - lo;
  if (self >= 0 && self < len) mk &= ~(1u << self);
  return mk;
}

// window_bits over candidate positions staged in LDS (2D: (x, y) pairs): lp
// points at candidate lo.  Same arithmetic, so the same bits.
__device__ __forceinline__ uint32_t window_bits_lds(const double2* lp, double xa0, double xa1, int64_t a,
                                                    int32_t lo, int32_t hi, double dist2) {
#pragma clang fp contract(off)
  const int32_t len = hi - lo;
  uint32_t acc = 0;
  for (int32_t j = 0; j < len; j += 4) {
    double2 c[4];
    double r[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) c[u] = lp[j + u];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const double d0 = xa0 - c[u].x;
      const double d1 = xa1 - c[u].y;
      r[u] = d0 * d0 + d1 * d1;
    }
    acc = push_lt4(acc, r[0], r[1], r[2], r[3], dist2);
  }
  return window_mask(acc, len, a, lo);
}

// 3D: the same over positions staged as (x, y) pairs and z.
__device__ __forceinline__ uint32_t window_bits_lds3(const double2* lp, const double* lz, double xa0, double xa1,
                                                     double xa2, int64_t a, int32_t lo, int32_t hi, double dist2) {
#pragma clang fp contract(off)
  const int32_t len = hi - lo;
  uint32_t acc = 0;
  for (int32_t j = 0; j < len; j += 4) {
    double2 c[4];
    double c2[4];
    double r[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      c[u] = lp[j + u];
      c2[u] = lz[j + u];
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const double d0 = xa0 - c[u].x;
      const double d1 = xa1 - c[u].y;
      const double d2 = xa2 - c2[u];
      double r2 = d0 * d0 + d1 * d1;
      r[u] = r2 + d2 * d2;
    }
    acc = push_lt4(acc, r[0], r[1], r[2], r[3], dist2);
  }
  return window_mask(acc, len, a, lo);
}

// The candidates of a stencil row that can pass the membership test, where
// the rank orders every cell by x (so a row, three consecutive cells of one
// y and z, is in x order): [lo, hi) (at most 256) narrowed by bisection over the
// staged x (lp[b].x of candidate b) to the first b with xa - x_b < dist and, from
// there, the first b with xa - x_b <= -dist; the two searches go in step, their
// loads in flight together.  Every candidate outside has |fl(xa - x_b)| >=
// dist, the same FP64 difference the test squares, so its r^2 rounds to at
// least fl(dist^2) = dist2 and the test fails.  A NaN coordinate (never a
// member: its r^2 is NaN) compares false both ways; the bisection still only
// drops candidates whose real x lies beyond an x it found outside the range,
// since the real x are in order.
__device__ __forceinline__ void x_range(const double2* lp, double xa, double dist, int32_t& lo, int32_t& hi) {
  if (lo >= hi) return;
  int32_t l = lo, u = lo;
#pragma unroll
  for (int32_t step = 128; step > 0; step >>= 1) {
    const int32_t pl = l + step, pu = u + step;
    const double dl = xa - lp[(pl < hi ? pl : hi) - 1].x, du = xa - lp[(pu < hi ? pu : hi) - 1].x;
    l = pl <= hi && dl >= dist ? pl : l;
    u = pu <= hi && !(du <= -dist) ? pu : u;
  }
  // 255 of 256 reached
  if (l < hi && xa - lp[l].x >= dist) ++l;
  if (u < hi && !(xa - lp[u].x <= -dist)) ++u;
  lo = l;
  hi = u;
}

// Least real distance along one axis from coordinate x in cell i (0-based) to
// any point binned into cell i + o, o in {-1, 0, 1}, less a margin for the
// rounding of the binning; edge cells, which also hold what lies outside the
// grid, reach outward only.  0 for NaN.
__device__ __forceinline__ double axis_gap(double x, double off, double cs, int64_t i, int o) {
  if (o == 0) return 0.0;
  const double u = x - off, edge = double(o > 0 ? i + 1 : i) * cs;
  const double gap = o > 0 ? edge - u : u - edge;
  return fmax(gap - 1e-13 * (fabs(u) + fabs(edge) + cs), 0.0);
}

// The stored windows of a particle: each starts at a member and holds the
// members among the next 32 candidates (row) or the next kWin3 of its cell
// (cells), from the member bits of up to 64 candidates of a row at a time.
struct Windows {
  uint64_t* out;
  int64_t n;
  int cap;
  int cnt = 0;
  __device__ __forceinline__ void put(int32_t base, uint32_t bits) {
    if (cnt < cap) out[int64_t(cnt) * n] = (uint64_t(uint32_t(base)) << 32) | bits;
    ++cnt;
  }
  // bit t: candidate b + t
  __device__ __forceinline__ void row(int32_t b, uint64_t bits) {
    while (bits != 0) {
      const int t0 = __builtin_ctzll(bits);
      b += t0;
      bits >>= t0;
      put(b, uint32_t(bits));
      b += 32;
      bits >>= 32;
    }
  }
  // the same of the row's three cells, cell ox = j - 1 being [sb[j], sb[j + 1])
  __device__ __forceinline__ void cells(int32_t b, uint64_t bits, const int32_t* sb, int oy, int oz) {
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      const int32_t e = sb[j + 1] - b;  // candidates left in the cell
      if (e <= 0) continue;
      uint64_t in = bits;
      int32_t c = b;
      if (e < 64) {
        in &= (uint64_t(1) << e) - 1u;
        bits >>= e;
        b += e;
      } else {
        bits = 0;
      }
      while (in != 0) {
        const int t0 = __builtin_ctzll(in);
        c += t0;
        in >>= t0;
        put(c, (win_code3(j - 1, oy, oz) << kWin3) | (uint32_t(in) & kWinMask3));
        c += kWin3;
        in >>= kWin3;
      }
    }
  }
};
// test(lo, hi): member bits of up to 32 candidates; of up to 64 here.
template <typename Test>
__device__ __forceinline__ uint64_t bits64(int32_t lo, int32_t hi, const Test& test) {
  const int32_t mid = hi < lo + 32 ? hi : lo + 32;
  uint64_t bits = test(lo, mid);
  if (mid < hi) bits |= uint64_t(test(mid, hi)) << 32;
  return bits;
}

// Candidates staged in LDS per wave: 2D 400 positions (the union of a wave's
// three stencil rows holds ~300 on a uniform lattice), 26 KiB per block, six
// blocks per CU; 3D one row at a time, 256 positions (~180), 25 KiB.
constexpr int kNmaskWave = 400;
constexpr int kNmaskRow = 256;

// ------------------------------------------------------------------ kernels
// Commits the rebuild of a problem (one thread per problem): the reordered
// buffers become the current ones.
template <typename R>
__device__ __forceinline__ void commit_rebuild(const SceneDev<R>& sd, StepCtl* ctl) {
  if (!ctl->rebuild) return;
  ctl->parity ^= 1;
  ctl->pparity ^= 1;
  ctl->updaten += 1;
  const long long mp = *sd.maxcell;
  if (mp > ctl->mppcell) ctl->mppcell = (long long)ceil(double(mp) * 1.05 + 1);  // src/celllist.jl:105-106
  ctl->rebuild = 0;
}

template <typename R, typename SS>
__global__ void k_commit_rebuild(SS ss) {
  const SceneDev<R>& sd = scene_at<R>(ss, blockIdx.x);
  if (threadIdx.x == 0) commit_rebuild(sd, sd.B.ctl);
}

// New sorted position s takes the state of old position perm[s] (its
// position is already there: the rank kernel moves the positions, and moving
// the other fields there too measured slower: its stores are scattered where
// the loads here are); returns the particle's position (xs) for a membership
// test that follows.
template <int D, typename R>
__device__ __forceinline__ void reorder_one(const SphBufs<R>& B, const SphConst& C, const CellGeom& G,
                                            const StepFlags& F, const StepCtl* ctl, int64_t s, double* xs) {
  const int p = ctl->parity, q = p ^ 1, pp = ctl->pparity, pq = pp ^ 1;
  const int32_t src = B.perm[s];
  R vs[3];
#pragma unroll
  for (int k = 0; k < D; ++k) {
    const double xv = B.X[q][k][s];
    const R vv = B.V[p][k][src];
    xs[k] = xv;
    vs[k] = vv;
    B.V[q][k][s] = vv;
    if (F.write_xrb) B.XRB[k][s] = xv;
    if (!F.synced_prev) {  // previous half-step state moves with its particle
      B.XH[k][s] = B.XH2[k][src];
      B.VH[k][s] = B.VH2[k][src];
    }
  }
  const R rv = B.RHO[p][src];
  const int32_t pt = B.PT[pp][src];
  B.RHO[q][s] = rv;
  typename Records<D, R>::N rec{};
  double fr[3];
  particle_frame<D, R>(B, C, G, s, fr);  // s's cell in the new order
#pragma unroll
  for (int k = 0; k < D; ++k) {
    put_x(rec, k, xs[k], fr);
    rec.v[k] = vs[k];
  }
  rec.rho = rv;
  if constexpr (std::is_same<R, double>::value) {
    const double P = eos_d(rv, pt, C);
    B.PN[s] = P;
    rec.P = P;
    rec.pt = pt;
    set_irho(rec);
  } else {
    const float P = eos_f(rv, pt, C);
    B.PN[s] = P;
    set_pt(rec, pt, P);
  }
  st_rec(B.PRN, s, rec, B.n);
  if (!F.synced_prev) B.RH[s] = B.RH2[src];
  B.PT[pq][s] = pt;
  B.ID[pq][s] = B.ID[pp][src];
}

// Neighbour-list membership of the last rebuild, stored per particle as
// (mask, base) entries: one window of candidates [base, base + len) with its
// member bits in the low word.  Windows of up to 32 candidates of one
// stencil row, or in 3D FP32-split of up to kWin3 candidates inside one
// stencil cell with the cell's offset coded above the member bits
// (win_code3), which is what the cell frames of its partner records need.
// Each window starts at a member (the first one not covered by the window
// before it), so with the rows in x order a particle's partners fill few
// windows; stored in stencil order.  Entry e of particle a is NE[e * n + a]; NC[a]
// is the entry count, or -1 when the particle needs more than necap entries
// (its partners are then found by scanning the stencil).
//
// It runs in the kernel that reorders the state, from the rebuild positions in
// the new order, which the rank kernel wrote (the other fields move in this
// kernel, which needs no other block's writes).  xa: a's rebuild position.
// Wave-level only (no block barrier).
//
// 3D: a wave takes its 9 stencil rows one after the other: it stages the
// candidates of a row of all its particles in its LDS slice, the next row's
// loads in flight, and every lane tests its own row there: the candidates whose
// x lies within the half width that the row's distance in y and z leaves of
// the sphere (~330 of the ~1050 candidates of a particle).  A row beyond the
// slice is tested whole from global memory: same expression, same bits.  Bound
// by the LDS reads of the tests (24 B each, lanes at different places).
// 883,376 particles: 0.50 ms staged by the block, a plane at a time behind two
// barriers, narrowed to |x_a - x_b| < dist only, and in a launch of its own (its
// reorder 36 us more); with the reorder 0.45 ms here.  31,962: 95 + 7 -> 84 us.
template <typename R>
__device__ __forceinline__ void nmask3_new(const SphBufs<R>& B, const SphConst& C, const CellGeom& G,
                                           const StepCtl* ctl, int64_t a, int64_t a0, const double* xa,
                                           double2 (*lds_xy)[kNmaskRow + 4], double (*lds_z)[kNmaskRow + 4]) {
  const bool active = a < B.n;
  const double dist2 = C.dist2;
  const int q = ctl->parity ^ 1;  // the new order (committed after this kernel)
  const double* XN[3] = {B.X[q][0], B.X[q][1], B.X[q][2]};
  Windows win{B.NE + a, B.n, B.necap};
  const int w = __builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6));
  const int lane = int(threadIdx.x & 63);
  const int64_t aw = a0 + 64 * w;
  if (aw >= B.n) return;  // whole wave
  double2* lxy = lds_xy[w];
  double* lz = lds_z[w];
  const int64_t gx = G.grid[0], gy = G.grid[1], gz = G.grid[2], nce = G.ncells();
  // the wave's candidates of row r: one contiguous range [ub, ue)
  const int64_t c0 = B.skey[aw], c1 = B.skey[aw + 63 < B.n ? aw + 63 : B.n - 1];
  auto row_offset = [&](int r) { return gx * (r % 3 - 1) + gx * gy * (r / 3 - 1); };
  auto bound_of = [&](int64_t c) { return B.start[c < 0 ? 0 : (c > nce ? nce : c)]; };
  constexpr int kSlots = kNmaskRow / 64;
  double v[kSlots][3];
  int32_t ub, ue;
  auto prefetch = [&](int r) {
    ub = bound_of(c0 + row_offset(r) - 1);
    ue = bound_of(c1 + row_offset(r) + 2);
    if (ue - ub > kNmaskRow) return;
#pragma unroll
    for (int t = 0; t < kSlots; ++t) {
      const int32_t b = ub + lane + 64 * t;
      if (b < ue) {
#pragma unroll
        for (int k = 0; k < 3; ++k) v[t][k] = XN[k][b];
      }
    }
  };
  int64_t ix = 0, iy = 0, iz = 0;
  cell_xyz<3>(G, B.skey[active ? a : aw], ix, iy, iz);
  double cs[3];
#pragma unroll
  for (int k = 0; k < 3; ++k) cs[k] = 1.0 / G.hinv64[k];
  prefetch(0);
#pragma unroll 1
  for (int r = 0; r < 9; ++r) {
    const int oy = r % 3 - 1, oz = r / 3 - 1;
    const int32_t wb = ub;
    const bool staged = ue - ub <= kNmaskRow;  // uniform over the wave
    if (staged) {
#pragma unroll
      for (int t = 0; t < kSlots; ++t) {
        if (ub + lane + 64 * t < ue) {
          lxy[lane + 64 * t] = make_double2(v[t][0], v[t][1]);
          lz[lane + 64 * t] = v[t][2];
        }
      }
    }
    // the cell boundaries of the particle's row: cell ox = j - 1 is
    // [sb[j], sb[j + 1]) when it lies in the grid
    const int64_t y = iy + oy, z = iz + oz;
    const bool in = active && y >= 0 && y < gy && z >= 0 && z < gz;
    int32_t sb[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) sb[t] = in ? bound_of(gx * (y + gy * z) + ix - 1 + t) : 0;
    if (r < 8) prefetch(r + 1);
    // the wave's LDS operations complete in issue order; the fence keeps the
    // compiler from moving the reads below ahead of these writes
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
    const double gap_y = axis_gap(xa[1], G.off64[1], cs[1], iy, oy), gap_z = axis_gap(xa[2], G.off64[2], cs[2], iz, oz);
    const double h2 = dist2 * (1.0 + 1e-12) - (gap_y * gap_y + gap_z * gap_z);
    if (in && !(h2 < 0.0)) {
      int32_t rb = ix >= 1 ? sb[0] : sb[1];
      int32_t re = ix + 1 < gx ? sb[3] : sb[2];
      const double2* lp = lxy - wb;  // candidate b at lp[b]
      const double* lq = lz - wb;
      if (staged) x_range(lp, xa[0], fmin(C.dist, sqrt(h2) * (1.0 + 1e-12)), rb, re);
      auto test = [&](int32_t lo, int32_t hi) {
        return staged ? window_bits_lds3(lp + lo, lq + lo, xa[0], xa[1], xa[2], a, lo, hi, dist2)
                      : window_bits<3>(XN[0], XN[1], XN[2], xa[0], xa[1], xa[2], a, lo, hi, dist2);
      };
      for (int32_t w0 = rb; w0 < re; w0 += 64) {
        const uint64_t bits = bits64(w0, re < w0 + 64 ? re : w0 + 64, test);
        // FP32-split: windows of one cell (the cell frames of the records need it)
        if constexpr (cell_windows<3, R>()) win.cells(w0, bits, sb, oy, oz);
        else win.row(w0, bits);
      }
    }
    __builtin_amdgcn_wave_barrier();  // the next row overwrites the staged positions
  }
  if (active) B.NC[a] = win.cnt <= win.cap ? win.cnt : -1;
}

// 2D: the wave stages the union of its three rows at once.
template <typename R>
__device__ __forceinline__ void nmask2_new(const SphBufs<R>& B, const SphConst& C, const CellGeom& G,
                                           const StepCtl* ctl, int64_t a, int64_t a0, const double* xa,
                                           double2 (*lds)[kNmaskWave + 4]) {
  const bool active = a < B.n;
  const double dist2 = C.dist2;
  const int q = ctl->parity ^ 1;  // the new order (committed after this kernel)
  const double* XN[2] = {B.X[q][0], B.X[q][1]};
  Windows win{B.NE + a, B.n, B.necap};
  const int w = __builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6));
  const int lane = int(threadIdx.x & 63);
  const int64_t aw = a0 + 64 * w;
  if (aw >= B.n) return;  // whole wave
  RowUnion u;
  row_union(u, B.start, B.skey, G, B.n, aw);
  const int32_t total = u.uo[3];
  if (total <= kNmaskWave) {  // uniform over the wave
    double2* wl = lds[w];
    const int32_t d0 = u.ub[0] - u.uo[0], d1 = u.ub[1] - u.uo[1], d2 = u.ub[2] - u.uo[2];
    // four slots per lane per trip, their loads in flight together; a slot
    // past the union repeats the last valid one's loads and is not written
    for (int32_t i0 = lane; i0 < total; i0 += 4 * 64) {
      double2 v[4];
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const int32_t i = i0 + 64 * t < total ? i0 + 64 * t : total - 1;
        const int32_t b = i + (i >= u.uo[2] ? d2 : (i >= u.uo[1] ? d1 : d0));
        v[t] = make_double2(XN[0][b], XN[1][b]);
      }
#pragma unroll
      for (int t = 0; t < 4; ++t)
        if (i0 + 64 * t < total) wl[i0 + 64 * t] = v[t];
    }
    // the wave's LDS operations complete in issue order; the fence keeps the
    // compiler from moving the reads below ahead of these writes
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
    if (active) {
      const Rows<2> rows = stencil_rows<2>(G, B.start, B.skey[a]);
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        const double2* lrow = wl + (u.uo[k] - u.ub[k]);  // candidate b at lrow[b]
        // (a row of ~35 candidates: bounding it to |x_a - x_b| < dist by
        // bisection, as in 3D, costs more than the tests it saves)
        auto test = [&](int32_t lo, int32_t hi) {
          return window_bits_lds(lrow + lo, xa[0], xa[1], a, lo, hi, dist2);
        };
        for (int32_t w0 = rows.b[k]; w0 < rows.e[k]; w0 += 64)
          win.row(w0, bits64(w0, rows.e[k] < w0 + 64 ? rows.e[k] : w0 + 64, test));
      }
    }
  } else if (active) {
    const Rows<2> rows = stencil_rows<2>(G, B.start, B.skey[a]);
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      auto test = [&](int32_t lo, int32_t hi) {
        return window_bits<2>(XN[0], XN[1], XN[1], xa[0], xa[1], 0.0, a, lo, hi, dist2);
      };
      for (int32_t w0 = rows.b[k]; w0 < rows.e[k]; w0 += 64)
        win.row(w0, bits64(w0, rows.e[k] < w0 + 64 ? rows.e[k] : w0 + 64, test));
    }
  }
  if (active) B.NC[a] = win.cnt <= win.cap ? win.cnt : -1;
}

// Rebuild tail in one kernel: the reorder of the state and the membership
// store of the same particles, which are independent of each other (one
// launch instead of two).
template <typename R, typename SS>
__global__ __launch_bounds__(256) void k_reorder_nmask2(SS ss) {
  GCLSPH_SCENE(ss);
  const StepCtl* ctl = B.ctl;
  if (ctl->rebuild == 0) return;
  const int64_t a0 = int64_t(m.y) * kBlock;
  if (a0 >= B.n) return;  // whole block
  __shared__ double2 lds[kBlock / 64][kNmaskWave + 4];  // +4: window reads run up to 3 past a row's end
  double xa[3] = {0.0, 0.0, 0.0};
  if (a < B.n) reorder_one<2, R>(B, C, G, F, ctl, a, xa);
  nmask2_new<R>(B, C, G, ctl, a, a0, xa, lds);
}

template <typename R, typename SS>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4))) void k_reorder_nmask3(SS ss) {
  GCLSPH_SCENE(ss);
  const StepCtl* ctl = B.ctl;
  if (ctl->rebuild == 0) return;
  const int64_t a0 = int64_t(m.y) * kBlock;
  if (a0 >= B.n) return;  // whole block
  __shared__ double2 lds_xy[kBlock / 64][kNmaskRow + 4];  // +4: window reads run up to 3 past a row's end
  __shared__ double lds_z[kBlock / 64][kNmaskRow + 4];
  double xa[3] = {0.0, 0.0, 0.0};
  if (a < B.n) reorder_one<3, R>(B, C, G, F, ctl, a, xa);
  nmask3_new<R>(B, C, G, ctl, a, a0, xa, lds_xy, lds_z);
}

// ---- corrections after the update (src/sphproblem.jl:303-322) --------------
// dpcreg! (src/gpukernels_sph.jl:1500-1553): ∑Δv_dpc into DV; P = EOS(ρ^{n+1}).
template <int D, typename R, bool Quad, typename SS>
__global__ __launch_bounds__(256) void k_dpc_sum(SS ss) {
#pragma clang fp contract(off)
  GCLSPH_SCENE_PAIR(ss, kBlock, Quad);
  if (!F.dpc_on) return;
  const StepCtl* ctl = B.ctl;
  const int p = cur_parity(ctl), q = p ^ 1, pp = cur_pparity(ctl), rebuilt = ctl->rebuild;
  const double dt = ctl->dt;
  if (a >= B.n) return;
  const double* X[3] = {B.X[q][0], B.X[q][1], B.X[q][D == 3 ? 2 : 1]};
  const R* V[3] = {B.V[q][0], B.V[q][1], B.V[q][D == 3 ? 2 : 1]};
  const R* RHO = B.RHO[q];
  const int32_t* PT = B.PT[pp];
  const double* XM[3];
  membership_ptrs<D>(B, F, p, rebuilt, XM);
  const int32_t pta = PT[a];
  const int nc = B.NC[a];
  double xa[3];
  R va[3];
#pragma unroll
  for (int d = 0; d < D; ++d) {
    xa[d] = X[d][a];
    va[d] = V[d][a];
  }
  // Partners from the records, which hold the updated state (pass 2).  A partner
  // at l0 or beyond adds nothing (its W and so χ are 0), and l0 is a fraction
  // of H: only positions are fetched ahead, the rest of a record for the few
  // partners nearer than l0.  The kernel is bound by the L1's tag rate, a
  // lookup per lane and 16-byte word: 0.53 -> 0.46 ms for 883,376 particles
  // (3D FP32-split, half the words).
  using Nb = typename Records<D, R>::N;
  struct Head {
    Nb r;
    int32_t b;
  };
  auto fetch = [&](const int32_t b) { return Head{ld_pos<Nb>(B.PRN, b, B.n), b}; };
  const R Pa = B.PN[a];
  if (F.want_out && writer) B.PBUF[a] = Pa;
  if (pta <= 0) {  // every DPC pair needs ptype > 0 on both sides
#pragma unroll
    for (int d = 0; d < D; ++d)
      if (writer) B.DV[d][a] = R(0);
    return;
  }
  if constexpr (std::is_same<R, double>::value) {
    const double rhoa = RHO[a];
    const auto sum = sum_partners<true, Quad, D, D, R>(B, a, nc, G, XM, C.dist2, fetch, [&](const Head& h, auto& t) {
      double dx[3], dv[3];
#pragma unroll
      for (int d = 0; d < D; ++d) dx[d] = xa[d] - h.r.x[d];
      const double r2 = dotd<D>(dx, dx);
      const double r = sqrt_d(r2);
      const double u = r * C.dpc_l0inv;
      if (u >= 1.0) return;
      const Nb n = ld_rec<Nb>(B.PRN, h.b, B.n);
      if (n.pt <= 0) return;
#pragma unroll
      for (int d = 0; d < D; ++d) dv[d] = va[d] - n.v[d];
      const double rhob = n.rho;
      const double w = W_d(u, C.dpc_wnorm);
      const double chi = sqrt(w * C.dpc_whinv);
      const double kk = u < C.dpc_lim ? 1.0 : chi;
      double lo = C.dpc_lambda * fabs(Pa + n.P), cap = C.dpc_lambda * C.dpc_pmax;
      double pt = lo < cap ? lo : cap;
      pt = pt > C.dpc_pmin ? pt : C.dpc_pmin;
      const double Pb_dpc = chi * pt;
      const double vr = dotd<D>(dv, dx);
      if (vr < 0) {
        double vrdr = vr / (r2 + C.dpc_eta2);
#pragma unroll
        for (int d = 0; d < D; ++d) t.v[d] = kk * (-vrdr * dx[d]);
      } else {
        double tvar = 2 * dt * Pb_dpc / ((rhoa + rhob) * (r2 + C.dpc_eta2));
#pragma unroll
        for (int d = 0; d < D; ++d) t.v[d] = tvar * dx[d];
      }
    });
#pragma unroll
    for (int d = 0; d < D; ++d)
      if (writer) B.DV[d][a] = sum.get(d);
  } else {
    const float rhoa = C.f_rho0 + RHO[a];
    const float fdt = float(dt);
    const FrameK3 kt = particle_k<D, R>(B, C, G, a, xa);
    const auto sum = sum_partners<true, Quad, D, D, R, true>(B, a, nc, G, XM, C.dist2, fetch, [&](const Head& h, auto& t,
                                                                                          const auto&... win) {
      float dx[3], dv[3];
#pragma unroll
      for (int d = 0; d < D; ++d) dx[d] = sep_x(xa, h.r, d, win...);
      const float r2 = dotf<D>(dx, dx);
      const float r = __builtin_amdgcn_sqrtf(r2), u = r * C.f_dpc_l0inv;
      if (u >= 1.0f) return;
      const Nb n = ld_rec<Nb>(B.PRN, h.b, B.n);
      if (rec_pt(n) <= 0) return;
#pragma unroll
      for (int d = 0; d < D; ++d) dv[d] = va[d] - n.v[d];
      const float rhob = C.f_rho0 + n.rho;
      const float w = W_f(r, C.f_dpc_l0inv, C.f_dpc_wnorm);
      const float chi = __builtin_amdgcn_sqrtf(w * C.f_dpc_whinv);
      const float kk = u < C.f_dpc_lim ? 1.0f : chi;
      const float lo = C.f_dpc_lambda * fabsf(Pa + rec_P(n, C)), cap = C.f_dpc_lambda * C.f_dpc_pmax;
      float pt = lo < cap ? lo : cap;
      pt = pt > C.f_dpc_pmin ? pt : C.f_dpc_pmin;
      const float Pb_dpc = chi * pt;
      const float vr = dotf<D>(dv, dx);
      const float den = __builtin_amdgcn_rcpf(r2 + C.f_dpc_eta2);
      if (vr < 0.0f) {
        const float vrdr = vr * den;
#pragma unroll
        for (int d = 0; d < D; ++d) t.v[d] = kk * (-vrdr * dx[d]);
      } else {
        const float tvar = 2.0f * fdt * Pb_dpc * __builtin_amdgcn_rcpf(rhoa + rhob) * den;
#pragma unroll
        for (int d = 0; d < D; ++d) t.v[d] = tvar * dx[d];
      }
    }, &kt);
#pragma unroll
    for (int d = 0; d < D; ++d)
      if (writer) B.DV[d][a] = sum.get(d);
  }
}

// update_dpcreg! (src/gpukernels_sph.jl:1617-1632)
template <int D, typename R, typename SS>
__global__ void k_dpc_apply(SS ss) {
#pragma clang fp contract(off)
  GCLSPH_SCENE(ss);
  if (!F.dpc_on) return;
  const StepCtl* ctl = B.ctl;
  const int q = cur_parity(ctl) ^ 1, pp = cur_pparity(ctl);
  const double dt = ctl->dt;
  if (a >= B.n || B.PT[pp][a] <= 1) return;
  bool any = false;
#pragma unroll
  for (int d = 0; d < D; ++d) any |= B.DV[d][a] != R(0);
  if (!any) return;  // no partner nearer than l0
  double fr[3];
  particle_frame<D, R>(B, C, G, a, fr);
  using N = typename Records<D, R>::N;
  N rec = ld_rec<N>(B.PRN, a, B.n);
  const int32_t pt = B.PT[pp][a];
#pragma unroll
  for (int d = 0; d < D; ++d) {
    R dv = B.DV[d][a];
    const R nv = B.V[q][d][a] + dv;
    const double nx = B.X[q][d][a] + double(dv) * dt;
    B.V[q][d][a] = nv;
    B.X[q][d][a] = nx;
    rec.v[d] = nv;
    put_x(rec, d, nx, fr);
  }
  if constexpr (!std::is_same<R, double>::value) set_pt(rec, pt, B.PN[a]);  // the 2D type class sits in y
  st_rec(B.PRN, a, rec, B.n);
}

// Partner records of the XSPH pass in the Records::N layout: xⁿ (the
// positions XSPH weighs with), v and ρ after the update and the DPC, ptype.
// They go over the half-step records, which pass 2 was the last to read.
template <int D, typename R, typename SS>
__global__ void k_xsph_rec(SS ss) {
  GCLSPH_SCENE(ss);
  if (!F.xsph_on) return;
  const StepCtl* ctl = B.ctl;
  const int p = cur_parity(ctl), q = p ^ 1, pp = cur_pparity(ctl);
  if (a >= B.n) return;
  typename Records<D, R>::N rec{};
  double fr[3];
  particle_frame<D, R>(B, C, G, a, fr);
#pragma unroll
  for (int d = 0; d < D; ++d) {
    put_x(rec, d, B.X[p][d][a], fr);
    rec.v[d] = B.V[q][d][a];
  }
  rec.rho = B.RHO[q][a];
  if constexpr (std::is_same<R, double>::value) rec.pt = B.PT[pp][a];
  else set_pt(rec, B.PT[pp][a], B.PN[a]);
  st_rec(B.PRH, a, rec, B.n);
}

// xsphcorr! + update_xsphcorr! (src/gpukernels_sph.jl:1757-1838): W at xⁿ.
// At most four waves per SIMD: with the seven that its registers allow, their
// partners' records displace each other in the CU's L1 (883,376 particles in 3D
// FP32-split: 565 us at seven, 530 at five, 496 at four).
template <int D, typename R, bool Quad, typename SS>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 4))) void k_xsph(SS ss) {
#pragma clang fp contract(off)
  GCLSPH_SCENE_PAIR(ss, kBlock, Quad);
  if (!F.xsph_on) return;
  const StepCtl* ctl = B.ctl;
  const int p = cur_parity(ctl), q = p ^ 1, pp = cur_pparity(ctl), rebuilt = ctl->rebuild;
  const double dt = ctl->dt;
  if (a >= B.n) return;
  const int32_t* PT = B.PT[pp];
  const int32_t pta = PT[a];
  if (pta <= 1) return;
  const double* XN[3] = {B.X[p][0], B.X[p][1], B.X[p][D == 3 ? 2 : 1]};
  const R* V[3] = {B.V[q][0], B.V[q][1], B.V[q][D == 3 ? 2 : 1]};
  const R* RHO = B.RHO[q];
  const double* XM[3];
  membership_ptrs<D>(B, F, p, rebuilt, XM);
  const int nc = B.NC[a];
  double xa[3];
  R va[3];
#pragma unroll
  for (int d = 0; d < D; ++d) {
    xa[d] = XN[d][a];
    va[d] = V[d][a];
  }
  // xⁿ, v, ρ and ptype of a partner from the records of k_xsph_rec
  using Nb = typename Records<D, R>::N;
  auto fetch = [&](const int32_t b) { return ld_rec<Nb>(B.PRH, b, B.n); };
  double out[3];
  if constexpr (std::is_same<R, double>::value) {
    const double rhoa = RHO[a];
    const auto sum = sum_partners<true, Quad, D, D, R>(B, a, nc, G, XM, C.dist2, fetch, [&](const Nb& n, auto& t) {
      if (n.pt <= 1) return;
      double dx[3];
#pragma unroll
      for (int d = 0; d < D; ++d) dx[d] = xa[d] - n.x[d];
      const double r = sqrt(dotd<D>(dx, dx));
      const double w = W_d(r * C.Hinv, C.wnorm);
      const double xs = C.xsph_c * w / (rhoa + n.rho);
#pragma unroll
      for (int d = 0; d < D; ++d) t.v[d] = (n.v[d] - va[d]) * xs;
    });
#pragma unroll
    for (int d = 0; d < D; ++d) out[d] = sum.get(d);
  } else {
    const float rhoa = C.f_rho0 + RHO[a];
    const FrameK3 kt = particle_k<D, R>(B, C, G, a, xa);
    const auto sum = sum_partners<true, Quad, D, D, R, true>(B, a, nc, G, XM, C.dist2, fetch, [&](const Nb& n, auto& t,
                                                                                          const auto&... win) {
      if (rec_pt(n) <= 1) return;
      float dx[3];
#pragma unroll
      for (int d = 0; d < D; ++d) dx[d] = sep_x(xa, n, d, win...);
      const float r = __builtin_amdgcn_sqrtf(dotf<D>(dx, dx));
      const float w = W_f(r, C.f_Hinv, C.f_wnorm);
      const float xs = C.f_xsph_c * w * __builtin_amdgcn_rcpf(rhoa + (C.f_rho0 + n.rho));
#pragma unroll
      for (int d = 0; d < D; ++d) t.v[d] = (n.v[d] - va[d]) * xs;
    }, &kt);
#pragma unroll
    for (int d = 0; d < D; ++d) out[d] = double(sum.get(d));
  }
  if (!writer) return;
  double fr[3];
  particle_frame<D, R>(B, C, G, a, fr);
  using N = typename Records<D, R>::N;
  N rec = ld_rec<N>(B.PRN, a, B.n);
#pragma unroll
  for (int d = 0; d < D; ++d) {
    const double nx = B.X[q][d][a] + out[d] * dt;
    B.X[q][d][a] = nx;
    put_x(rec, d, nx, fr);
  }
  if constexpr (!std::is_same<R, double>::value) set_pt(rec, pta, B.PN[a]);  // the 2D type class sits in y
  st_rec(B.PRN, a, rec, B.n);
}

// cspmcorr! (src/gpukernels_sph.jl:1693-1719): ρ = Σ m0 W / Σ m0 W / ρ_b, W at xⁿ.
template <int D, typename R, bool Quad, typename SS>
__global__ __launch_bounds__(256) void k_cspm_sum(SS ss) {
#pragma clang fp contract(off)
  GCLSPH_SCENE_PAIR(ss, kBlock, Quad);
  if (!F.cspm_fire) return;
  const StepCtl* ctl = B.ctl;
  const int p = cur_parity(ctl), q = p ^ 1, pp = cur_pparity(ctl), rebuilt = ctl->rebuild;
  if (a >= B.n) return;
  const int32_t* PT = B.PT[pp];
  const int32_t pta = PT[a];
  const double* XN[3] = {B.X[p][0], B.X[p][1], B.X[p][D == 3 ? 2 : 1]};
  const R* RHO = B.RHO[q];
  const double* XM[3];
  membership_ptrs<D>(B, F, p, rebuilt, XM);
  double s1 = 0.0, s2 = 0.0;
  if (pta > 0) {
    const int nc = B.NC[a];
    double xa[3];
#pragma unroll
    for (int d = 0; d < D; ++d) xa[d] = XN[d][a];
    struct Nb {
      double x[3];
      R rho;
      int32_t pt;
    };
    auto fetch = [&](const int32_t b) {
      const uint32_t o8 = uint32_t(b) * 8u, oR = uint32_t(b) * uint32_t(sizeof(R)), o4 = uint32_t(b) * 4u;
      Nb n;
#pragma unroll
      for (int d = 0; d < D; ++d) n.x[d] = ldo(XN[d], o8);
      n.rho = ldo(RHO, oR);
      n.pt = ldo(PT, o4);
      return n;
    };
    if constexpr (std::is_same<R, double>::value) {
      const auto sum = sum_partners<true, Quad, D, 2, R>(B, a, nc, G, XM, C.dist2, fetch, [&](const Nb& n, auto& t) {
        if (n.pt <= 0) return;
        double dx[3];
#pragma unroll
        for (int d = 0; d < D; ++d) dx[d] = xa[d] - n.x[d];
        const double w = W_d(sqrt(dotd<D>(dx, dx)) * C.Hinv, C.wnorm);
        t.v[0] = C.m0 * w;
        t.v[1] = w * C.m0 / n.rho;
      });
      s1 = sum.s[0];
      s2 = sum.s[1];
    } else {
      // on δρ: with e = δρ_b/ρ0, ρ' - ρ0 = ρ0 Σ m0W e/(1+e) / Σ m0W/(1+e), which
      // is s1/s2 - ρ0 without the cancellation against ρ0
      const auto sum = sum_partners<true, Quad, D, 2, R>(B, a, nc, G, XM, C.dist2, fetch, [&](const Nb& n, auto& t) {
        if (n.pt <= 0) return;
        float dx[3];
#pragma unroll
        for (int d = 0; d < D; ++d) dx[d] = float(xa[d] - n.x[d]);
        const float w = W_f(__builtin_amdgcn_sqrtf(dotf<D>(dx, dx)), C.f_Hinv, C.f_wnorm);
        const float inv_rho0 = 1.0f / C.f_rho0, e = n.rho * inv_rho0;
        const float mw = C.f_m0 * w * __builtin_amdgcn_rcpf(fma_(n.rho, inv_rho0, 1.0f));
        t.v[0] = mw * e;
        t.v[1] = mw;
      });
      s1 = sum.s[0] * C.rho0;
      s2 = sum.s[1];
    }
  }
  if (writer) B.TMP[a] = s1 / s2;  // ρ (FP64 path) or ρ - ρ0 (FP32-split); NaN without partners
}

template <int D, typename R, typename SS>
__global__ void k_cspm_apply(SS ss) {
  GCLSPH_SCENE(ss);
  if (!F.cspm_fire) return;
  const StepCtl* ctl = B.ctl;
  const int q = cur_parity(ctl) ^ 1, pp = cur_pparity(ctl);
  if (a >= B.n) return;
  double nr = B.TMP[a];
  if (nr != nr) return;
  const int32_t pt = B.PT[pp][a];
  if constexpr (std::is_same<R, double>::value) {
    B.RHO[q][a] = nr;
    const double P = eos_d(nr, pt, C);
    B.PN[a] = P;
    using N = typename Records<D, R>::N;
    N rec = ld_rec<N>(B.PRN, a, B.n);
    rec.rho = nr;
    rec.P = P;
    set_irho(rec);
    st_rec(B.PRN, a, rec, B.n);
  } else {
    const float d = float(nr);
    B.RHO[q][a] = d;
    const float P = eos_f(d, pt, C);
    B.PN[a] = P;
    using N = typename Records<D, R>::N;
    N rec = ld_rec<N>(B.PRN, a, B.n);
    rec.rho = d;
    set_pt(rec, pt, P);
    st_rec(B.PRN, a, rec, B.n);
  }
}

// PN = EOS(current density) for every particle (after construction).
template <typename R, typename SS>
__global__ void k_init_pn(SS ss) {
  GCLSPH_SCENE(ss);
  const StepCtl* ctl = B.ctl;
  const int p = ctl->parity, pp = ctl->pparity;
  if (a >= B.n) return;
  const R rv = B.RHO[p][a];
  const int32_t pt = B.PT[pp][a];
  if constexpr (std::is_same<R, double>::value) B.PN[a] = eos_d(rv, pt, C);
  else B.PN[a] = eos_f(rv, pt, C);
}

// Δt viscous rate over the corrected state (src/gpukernels_sph.jl:1325-1334).
template <int D, typename R, typename SS>
__global__ void k_dt_visc(SS ss) {
  GCLSPH_SCENE(ss);
  if (!(F.ts && !F.visc_in_pass2)) return;  // the whole block belongs to one problem
  StepCtl* ctl = B.ctl;
  const int q = cur_parity(ctl) ^ 1;
  const bool active = a < B.n;
  double v = 0.0;
  if (active) {
    double vn[3], xn[3];
#pragma unroll
    for (int d = 0; d < D; ++d) {
      vn[d] = double(B.V[q][d][a]);
      xn[d] = B.X[q][d][a];
    }
    v = fabs(C.h * dotd<D>(vn, xn) / (dotd<D>(xn, xn) + C.dt_eta2));
  }
  block_max(v, active, B.RED + 2 * kRedSlots, m.y);
}

__device__ __forceinline__ double jl_min(double a, double b) { return (a != a || b != b) ? a + b : (a < b ? a : b); }
__device__ __forceinline__ double jl_max(double a, double b) { return (a != a || b != b) ? a + b : (a > b ? a : b); }

// End of step: commits the new state, rebuild flag, time and Δt
// (src/sphproblem.jl:325-335, src/gpukernels_sph.jl:1293-1323).
template <typename R, typename SS>
__global__ void k_finalize(SS ss) {
  // one wave per problem: lane l reads slot l of each reduction and clears it
  // for the next step
  const SceneDev<R>& sd = scene_at<R>(ss, blockIdx.x);
  const StepFlags F = step_flags(sd);
  const SphConst& C = sd.C;
  StepCtl* ctl = sd.B.ctl;
  double* red = sd.B.RED;
  const int ts = F.ts, corr_on = F.corr_on;
  const int l = threadIdx.x;
  double tot[3];
  for (int k = 0; k < 3; ++k) {
    const double v = red[k * kRedSlots + l];
    red[k * kRedSlots + l] = 0.0;
    tot[k] = wave_max(v);
  }
  if (l != 0) return;
  commit_rebuild(sd, ctl);
  double cdx = tot[0];
  if (cdx > 0.9 * C.nui) ctl->rebuild = 1;
  ctl->maxcdx_out = jl_max(ctl->maxcdx_out, cdx);
  ctl->etime += ctl->dt;
  if (ts) {
    double amax = tot[1];
    double vmax = tot[2];
    double dt1 = sqrt(C.h / (3 * amax));
    double dt2 = C.h / (C.c0 + vmax);
    double dt = C.CFL * jl_min(dt1, dt2);
    dt = jl_min(jl_max(dt, C.tl0), C.tl1);
    ctl->dt = dt;
  }
  ctl->parity ^= 1;
  ctl->synced = corr_on ? 0 : 1;
  ctl->iter += 1;
}

// sph∑W! + sph∑∇W! over the current positions (src/gpukernels_sph.jl:139-156, :332-359).
template <int D, typename R, typename SS>
__global__ __launch_bounds__(256) void k_diag(SS ss, int xm_mode, int use_masks) {
#pragma clang fp contract(off)
  GCLSPH_SCENE(ss);
  const StepCtl* ctl = B.ctl;
  const int p = ctl->parity, pp = ctl->pparity;
  if (a >= B.n) return;
  const double* X[3] = {B.X[p][0], B.X[p][1], B.X[p][D == 3 ? 2 : 1]};
  // membership positions: 0 = stored rebuild positions, 1 = the step's start
  // positions (other buffer), 2 = the current positions
  const int mp = xm_mode == 1 ? (p ^ 1) : p;
  const double* XM[3];
#pragma unroll
  for (int k = 0; k < 3; ++k) XM[k] = xm_mode == 0 ? B.XRB[k < D ? k : 1] : B.X[mp][k < D ? k : 1];
  const int32_t* PT = B.PT[pp];
  const bool pa = PT[a] > 0;
  double sw = 0.0, sg[3] = {0.0, 0.0, 0.0};
  const int nc = use_masks ? B.NC[a] : -1;
  for_each_partner<D>(B, a, nc, G, XM, C.dist2, [&](const int32_t b) {
      if (pa != (PT[b] > 0)) return;
      double dx[3];
#pragma unroll
      for (int d = 0; d < D; ++d) dx[d] = X[d][a] - X[d][b];
      const double r = sqrt(dotd<D>(dx, dx));
      const double u = r * C.Hinv;
      sw += W_d(u, C.wnorm);
      const double dwk_r = dW_d(u, C.dwnorm) / r;
#pragma unroll
      for (int d = 0; d < D; ++d) sg[d] += dx[d] * dwk_r;
  });
  B.SUMW[a] = sw;
#pragma unroll
  for (int d = 0; d < D; ++d) B.SUMGW[d][a] = sg[d];
}

// ------------------------------------------------- rebuild: counting sort
// The problem's cell-sorted order is rebuilt by a counting sort over its cells
// (src/gpukernels_cls.jl:29-101 bins particles with atomics into a dense table):
// histogram with per-particle arrival slots, exclusive scan into cell starts,
// scatter, and a per-cell rank by input index (the previous sorted position),
// which makes the order deterministic.  Every kernel returns at once for a
// problem whose control block does not ask for a rebuild.

// Cell of every particle (current positions) and its arrival slot.
template <int D, typename R, typename SS>
__global__ void kb_cellmap(SS ss) {
  GCLSPH_SCENE(ss);
  const StepCtl* ctl = B.ctl;
  if (ctl->rebuild == 0) return;
  clear_scan_words(sd.scan_tmp, sd.ncells, a, (B.n + kBlock - 1) / kBlock * kBlock);
  if (a == 0) *sd.maxcell = 0;
  if (a >= B.n) return;
  const int p = ctl->parity;
  int32_t c[3] = {1, 1, 1};
#pragma unroll
  for (int k = 0; k < D; ++k) c[k] = cell_coord<double>(B.X[p][k][a], G, k, 0);
  const int64_t lin = int64_t(c[0] - 1) + G.grid[0] * (int64_t(c[1] - 1) + G.grid[1] * int64_t(c[2] - 1));
  const int32_t key = int32_t(lin);
  sd.key[a] = key;
  sd.slot[a] = wave_aggregated_slot(sd.cnt, key);
}

// Cell starts from the histogram, which is zero again afterwards;
// start[ncells] = n.
template <int Rows, typename R, typename SS>
__global__ __launch_bounds__(kScanThreads) void kb_cell_starts(SS ss) {
  int2 m;
  const SceneDev<R>& sd = tile_scene<R>(ss, m);
  if (sd.B.ctl->rebuild == 0) return;
  scan_tile<Rows, true>(sd.cnt, sd.start, sd.ncells, sd.scan_tmp, sd.maxcell);
}

// Sort key of an x coordinate: its bit pattern made unsigned-monotone (order
// of the key = order of the value for every non-NaN x; -0 before +0).
__device__ __forceinline__ uint64_t x_order_key(double x) {
  const uint64_t u = uint64_t(__double_as_longlong(x));
  return (u >> 63) ? ~u : (u | (uint64_t(1) << 63));
}

template <int D, typename R, typename SS>
__global__ void kb_scatter(SS ss) {
  GCLSPH_SCENE(ss);
  if (B.ctl->rebuild == 0 || a >= B.n) return;
  sd.tmp[sd.start[sd.key[a]] + sd.slot[a]] = int32_t(a);
}

// Rank inside the cell by (x, input index): the final order is (cell, x,
// input), so the candidates of a stencil row (three consecutive cells of one
// y, and z) are in x order (the cell of a coordinate is a non-decreasing
// function of it): a particle's partners in a row are then near each other,
// so they fill fewer stored windows, and in 3D the membership store bounds
// each particle's candidates in a row to |x_a - x_b| < dist by bisection.
// The order is the same for every run (ties in x by input index).  The
// particle's position (loaded first: its x is the key) moves to its new place
// here, so the membership store after it reads the candidates of a stencil
// row as contiguous ranges of the new position arrays instead of through the
// permutation.
template <int D, typename R, typename SS>
__global__ __launch_bounds__(256) void kb_rank(SS ss) {
  GCLSPH_SCENE(ss);
  if (B.ctl->rebuild == 0) return;
  const int64_t a0 = int64_t(m.y) * kBlock;
  if (a0 >= B.n) return;  // whole block
  // the (x key, input) of the block's slots, which hold the whole cell of
  // most of its particles, are shared through LDS; a cell across the block's
  // edge reads its members' x from global memory
  __shared__ uint64_t lk[kBlock];
  __shared__ int32_t li[kBlock];
  const int p = B.ctl->parity;
  const bool active = a < B.n;
  int32_t i = 0;
  double x[3] = {0.0, 0.0, 0.0};
  if (active) {
    i = sd.tmp[a];
#pragma unroll
    for (int k = 0; k < D; ++k) x[k] = B.X[p][k][i];
  }
  const uint64_t ki = x_order_key(x[0]);
  lk[threadIdx.x] = ki;
  li[threadIdx.x] = i;
  __syncthreads();
  if (!active) return;
  const int32_t c = sd.key[i];
  const int32_t b = sd.start[c], e = sd.start[c + 1];
  const int32_t s0 = int32_t(a0), s1 = int32_t(a0 + kBlock < B.n ? a0 + kBlock : B.n);
  // four compares per trip (indices clamped into the cell, which holds at
  // least this particle; the clamped ones are not counted)
  int32_t r = 0;
  if (b >= s0 && e <= s1) {
    for (int32_t k = b; k < e; k += 4) {
      int32_t v[4];
      uint64_t kv[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int32_t j = (k + u < e ? k + u : e - 1) - s0;
        v[u] = li[j];
        kv[u] = lk[j];
      }
#pragma unroll
      for (int u = 0; u < 4; ++u) r += (k + u < e) & ((kv[u] < ki) | ((kv[u] == ki) & (v[u] < i)));
    }
  } else {
    const double* X0 = B.X[p][0];
    for (int32_t k = b; k < e; k += 4) {
      int32_t v[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) v[u] = sd.tmp[k + u < e ? k + u : e - 1];
      uint64_t kv[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) kv[u] = x_order_key(X0[v[u]]);
#pragma unroll
      for (int u = 0; u < 4; ++u) r += (k + u < e) & ((kv[u] < ki) | ((kv[u] == ki) & (v[u] < i)));
    }
  }
  sd.perm[b + r] = i;
  sd.skey[b + r] = c;
#pragma unroll
  for (int k = 0; k < D; ++k) B.X[p ^ 1][k][b + r] = x[k];
}

// ------------------------------------------------------------ host launchers
template <int D, typename R>
void launch_rebuild(const LaunchSet& L, hipStream_t s) {
  with_scenes<R>(L, [&](auto ss) {
    using SS = decltype(ss);
    kb_cellmap<D, R, SS><<<L.pblocks, kBlock, 0, s>>>(ss);
    with_scan_rows(L.scan_rows, [&](auto rows) {
      kb_cell_starts<rows(), R, SS><<<L.ctiles, kScanThreads, 0, s>>>(ss);
    });
    kb_scatter<D, R, SS><<<L.pblocks, kBlock, 0, s>>>(ss);
    kb_rank<D, R, SS><<<L.pblocks, kBlock, 0, s>>>(ss);
    if constexpr (D == 2) k_reorder_nmask2<R, SS><<<L.pblocks, kBlock, 0, s>>>(ss);
    else k_reorder_nmask3<R, SS><<<L.pblocks, kBlock, 0, s>>>(ss);
  });
}
template <int D, typename R>
void launch_commit_rebuild(const LaunchSet& L, hipStream_t s) {
  with_scenes<R>(L, [&](auto ss) { k_commit_rebuild<R, decltype(ss)><<<L.count, 64, 0, s>>>(ss); });
}
template <int D, typename R>
void launch_init_pn(const LaunchSet& L, hipStream_t s) {
  with_scenes<R>(L, [&](auto ss) { k_init_pn<R, decltype(ss)><<<L.pblocks, kBlock, 0, s>>>(ss); });
}
template <int D, typename R>
void launch_dpc(const LaunchSet& L, hipStream_t s) {
  with_scenes<R>(L, [&](auto ss) {
    if (L.quad) k_dpc_sum<D, R, true, decltype(ss)><<<L.qblocks, kBlock, 0, s>>>(ss);
    else k_dpc_sum<D, R, false, decltype(ss)><<<L.pblocks, kBlock, 0, s>>>(ss);
    k_dpc_apply<D, R, decltype(ss)><<<L.pblocks, kBlock, 0, s>>>(ss);
  });
}
template <int D, typename R>
void launch_xsph(const LaunchSet& L, hipStream_t s) {
  with_scenes<R>(L, [&](auto ss) {
    k_xsph_rec<D, R, decltype(ss)><<<L.pblocks, kBlock, 0, s>>>(ss);
    if (L.quad) k_xsph<D, R, true, decltype(ss)><<<L.qblocks, kBlock, 0, s>>>(ss);
    else k_xsph<D, R, false, decltype(ss)><<<L.pblocks, kBlock, 0, s>>>(ss);
  });
}
template <int D, typename R>
void launch_cspm(const LaunchSet& L, hipStream_t s) {
  with_scenes<R>(L, [&](auto ss) {
    if (L.quad) k_cspm_sum<D, R, true, decltype(ss)><<<L.qblocks, kBlock, 0, s>>>(ss);
    else k_cspm_sum<D, R, false, decltype(ss)><<<L.pblocks, kBlock, 0, s>>>(ss);
    k_cspm_apply<D, R, decltype(ss)><<<L.pblocks, kBlock, 0, s>>>(ss);
  });
}
template <int D, typename R>
void launch_dt_visc(const LaunchSet& L, hipStream_t s) {
  with_scenes<R>(L, [&](auto ss) { k_dt_visc<D, R, decltype(ss)><<<L.pblocks, kBlock, 0, s>>>(ss); });
}
template <int D, typename R>
void launch_finalize(const LaunchSet& L, hipStream_t s) {
  with_scenes<R>(L, [&](auto ss) { k_finalize<R, decltype(ss)><<<L.count, kRedSlots, 0, s>>>(ss); });
}
template <int D, typename R>
void launch_diag(const LaunchSet& L, int xm_mode, int use_masks, hipStream_t s) {
  with_scenes<R>(L, [&](auto ss) {
    k_diag<D, R, decltype(ss)><<<L.pblocks, kBlock, 0, s>>>(ss, xm_mode, use_masks);
  });
}

#define GCLSPH_INSTANTIATE(D, R)                                                         \
  template void launch_rebuild<D, R>(const LaunchSet&, hipStream_t);                     \
  template void launch_commit_rebuild<D, R>(const LaunchSet&, hipStream_t);              \
  template void launch_init_pn<D, R>(const LaunchSet&, hipStream_t);                     \
  template void launch_dpc<D, R>(const LaunchSet&, hipStream_t);                         \
  template void launch_xsph<D, R>(const LaunchSet&, hipStream_t);                        \
  template void launch_cspm<D, R>(const LaunchSet&, hipStream_t);                        \
  template void launch_dt_visc<D, R>(const LaunchSet&, hipStream_t);                     \
  template void launch_finalize<D, R>(const LaunchSet&, hipStream_t);                    \
  template void launch_diag<D, R>(const LaunchSet&, int, int, hipStream_t);

GCLSPH_INSTANTIATE(2, double)
GCLSPH_INSTANTIATE(3, double)
GCLSPH_INSTANTIATE(2, float)
GCLSPH_INSTANTIATE(3, float)

}  // namespace gclsph

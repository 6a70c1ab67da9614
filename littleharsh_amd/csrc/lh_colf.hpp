// lh_colf.hpp -- the column stage of an RK3 substep in one kernel: RHS0 and the rhs of
// solveU/solveV, the velocity solves of LUsolU/LUsolV (tridLU_3D_IB.f90:106-116, 179-189), the
// constant-flow-rate correction of the (0,0) column (flowrate_corr, littleharsh.f90:453-485),
// solveP with LUsolP (littleharsh.f90:557-612, tridLU_3D_IB.f90:362-396) and v_corr
// (littleharsh.f90:826-929).
//
// A block owns CB adjacent spectral columns and the whole height of the channel: thread
// (l, q) = (tid % CB, tid / CB) holds R consecutive levels of column l, chunk q, in registers.
// Each first-order recurrence of the Thomas algorithm (x_s = A_s + B_s x_{s-1}) is run inside
// every chunk from zero, the chunk ends are combined through LDS in chunk order, and each
// thread adds B_first .. B_s times its true incoming value.  So a column's rows are loaded
// once and stored once: 10 fields in (u, v, w, p, Nu_old and Nu_new of three components; the
// pressure rows are read a second time from the L2) and 4 out, where one thread per column has
// to park its eliminated rows in HBM and read them back, and walks the planes one memory
// latency at a time.
#pragma once
#include <type_traits>
#include "lh_col.hpp"

namespace lh {

// parts of the column stage (the stage hooks run them one at a time)
constexpr int kColVel = 1, kColPres = 2, kColAll = kColVel | kColPres;

// LDS table, one row per plane s: the operator rows and LU factors of the two shared velocity
// matrices, and the metrics.  14 doubles: the rows of the chunks of a wave, R planes apart,
// start on distinct banks.
struct ColTab {
  double wu[3], lu[3];   // dyu2i(1..3, s); lower, 1/pivot, scaled upper of the u-grid LU
  double wv[3], lv[3];   // the same on the v grid
  double hu, hv;         // dthdyu(s), dthdyv(s)
};
// rows of the table: every plane, and the last chunk's rows past them (copies of the last)
__host__ __device__ constexpr int colf_rows(int nyu, int nc, int R) { return nyu > nc * R + 1 ? nyu : nc * R + 1; }

// LDS of a block: the table, then per chunk and column three complex chunk values, then per
// chunk and column one factor, then the two velocity factors per chunk
inline size_t colf_lds_bytes(int nyu, int nc, int R, int cb) {
  return ((size_t)colf_rows(nyu, nc, R) * sizeof(ColTab) + 15) / 16 * 16 +
         (size_t)nc * cb * (3 * sizeof(double2) + sizeof(double)) + (size_t)nc * 2 * sizeof(double);
}

// Rows of a field from a base in scalar registers and a 32-bit byte offset per lane (a field of
// the largest channel k_col takes holds 0.7 GB)
struct ColF {
  typedef double D2 __attribute__((ext_vector_type(2)));
  char __attribute__((address_space(1)))* b;
  __device__ __forceinline__ explicit ColF(const void* p) {
    const unsigned long long v = reinterpret_cast<unsigned long long>(p);
    const unsigned lo = __builtin_amdgcn_readfirstlane((unsigned)v);
    const unsigned hi = __builtin_amdgcn_readfirstlane((unsigned)(v >> 32));
    b = reinterpret_cast<char __attribute__((address_space(1)))*>(((unsigned long long)hi << 32) | lo);
  }
  __device__ __forceinline__ double2 ld(unsigned o) const {
    const D2 v = *reinterpret_cast<const D2 __attribute__((address_space(1)))*>(b + o);
    return d2(v.x, v.y);
  }
  // row o of this field, or of the field `other` bytes away where sel is set
  __device__ __forceinline__ double2 ld_sel(unsigned o, bool sel, long long other) const {
    const D2 v = *reinterpret_cast<const D2 __attribute__((address_space(1)))*>(b + ((long long)o + (sel ? other : 0ll)));
    return d2(v.x, v.y);
  }
  __device__ __forceinline__ long long to(const ColF& f) const { return f.b - b; }
  __device__ __forceinline__ double ld1(unsigned o) const {
    return *reinterpret_cast<const double __attribute__((address_space(1)))*>(b + o);
  }
  __device__ __forceinline__ void st(unsigned o, double2 a) const {
    D2 v;
    v.x = a.x;
    v.y = a.y;
    *reinterpret_cast<D2 __attribute__((address_space(1)))*>(b + o) = v;
  }
  // (a store of values that nothing reads before they have left the caches)
  __device__ __forceinline__ void st_nt(unsigned o, double2 a) const {
    D2 v;
    v.x = a.x;
    v.y = a.y;
    __builtin_nontemporal_store(v, reinterpret_cast<D2 __attribute__((address_space(1)))*>(b + o));
  }
};

// PRE: every row a thread reads is loaded ahead of the first barrier (small R: the chain of
// memory latencies sets the time); otherwise the rows of one component at a time, BR together.
template <int R, int CB, int BR, bool PRE, int MODE>
__device__ __forceinline__ void colf_block(const RHS& a, const COL& ca, const Dims& dm, const double* yvp, int c0,
                                           char* smem) {
  constexpr int NF = PRE ? 3 : 1, NR = PRE ? R : BR;
  const int tid = threadIdx.x, l = tid % CB, q = tid / CB, ncb = blockDim.x / CB;
  const int np = dm.nyp, ncol = dm.ncol, nyu = dm.nyu, nyv = dm.nyv;
  const int nc = (np + R - 1) / R;                    // chunks of this channel (<= ncb)
  const bool live = q < nc && c0 + l < ncol;
  const int nlv = min(R, np - q * R);                 // levels of this thread (<= 0: idle)
  const int at = q * CB + l;
  constexpr bool vel = (MODE & kColVel) != 0, pres = (MODE & kColPres) != 0;
  const bool use_old = a.C2 != 0.0;                   // C2 = -cRK is 0 in substep 1
  const double2 zero = d2(0.0, 0.0);
  const unsigned pl = (unsigned)ncol * 16u;           // bytes of a plane
  const int c = min(c0 + l, ncol - 1);
  // first level (plane of u and w, face of v) and the column's byte offset.  COLF_FRESH makes
  // the compiler form a phase's addresses from them anew: kept from phase to phase they would
  // take more registers than the rows do.
  int s0 = 1 + q * R;
  unsigned cb = (unsigned)c * 16u;
#define COLF_FRESH() asm volatile("" : "+v"(s0), "+v"(cb))
  auto off = [&](int s) { return (unsigned)s * pl + cb; };
  const ColF u1(ca.u1), u2(ca.u2), u3(ca.u3), pr(ca.p), dg3(ca.dg3);
  double2 x[3][R];                                    // u, w, v of this thread's levels
  double2 pp[NR + 1], um[NF], u0[NF], up[NF][NR], vo[NF][NR], vn[NF][NR];
  double a3[R], a3p = 0.0;
  // canopy planes among this thread's levels, bit r
  unsigned canu = 0, canv = 0;
  if (vel && live) {
#pragma unroll
    for (int r = 0; r < R; ++r) {
      canu |= gp(a.ib_u)[min(s0 + r, nyu - 1)] ? 1u << r : 0u;
      canv |= gp(a.ib_v)[min(s0 + r, nyv - 1)] ? 1u << r : 0u;
    }
  }
  // rows r0 .. r0 + NR - 1 of component f (0 u, 1 w, 2 v); a canopy plane's rhs comes from the
  // immersed-boundary stage: it takes the place of Nu_new, and of Nu_old, which is not needed
  auto load = [&](auto fc, auto nc_, auto rc) {
    constexpr int f = decltype(fc)::value, n = decltype(nc_)::value, r0 = decltype(rc)::value;
    const ColF uu(f == 0 ? a.u1 : (f == 1 ? a.u3 : a.u2)), no(f == 0 ? a.no1 : (f == 1 ? a.no3 : a.no2)),
        nn(f == 0 ? a.nn1 : (f == 1 ? a.nn3 : a.nn2)), rr(f == 0 ? a.r1 : (f == 1 ? a.r3 : a.r2));
    // in substep 1 Nu_old has the factor zero: Nu_new's row is read in its place (a cache hit)
    const ColF old = use_old ? no : nn;
    const int top = f < 2 ? nyu - 1 : nyv - 1;        // the boundary row above
    if constexpr (!PRE) {
#pragma unroll
      for (int e = 0; e < NR + (f == 2 ? 1 : 0); ++e)
        if (r0 + e <= R) pp[e] = pr.ld(off(min(s0 - 1 + r0 + e, np - 1)));
    }
    if constexpr (r0 == 0) {
      um[n] = uu.ld(off(s0 - 1));
      u0[n] = uu.ld(off(min(s0, top)));
    }
#pragma unroll
    for (int e = 0; e < NR; ++e)
      if (r0 + e < R) up[n][e] = uu.ld(off(min(s0 + r0 + e + 1, top)));
#pragma unroll
    for (int e = 0; e < NR; ++e)
      if (r0 + e < R) {
        const unsigned o = off(min(s0 + r0 + e, top));
        const bool can = ((f < 2 ? canu : canv) >> (r0 + e)) & 1u;
        vn[n][e] = nn.ld_sel(o, can, nn.to(rr));
        vo[n][e] = old.ld_sel(o, can, old.to(rr));
      }
  };
  using I0 = std::integral_constant<int, 0>;
  using I1 = std::integral_constant<int, 1>;
  using I2 = std::integral_constant<int, 2>;
  if (live) {
    if (vel) {
      if constexpr (PRE) {
#pragma unroll
        for (int r = 0; r <= R; ++r) pp[r] = pr.ld(off(min(s0 - 1 + r, np - 1)));
        load(I0{}, I0{}, I0{});
        load(I1{}, I1{}, I0{});
        load(I2{}, I2{}, I0{});
      }
    }
    if constexpr (PRE) {
      if (q > 0) a3p = dg3.ld1(off(s0 - 2) / 2u);
#pragma unroll
      for (int r = 0; r < R; ++r) a3[r] = dg3.ld1(off(min(s0 - 1 + r, np - 1)) / 2u);
    }
  }
  ColTab* const tab = reinterpret_cast<ColTab*>(smem);
  const int nrow = colf_rows(nyu, nc, R);
  double2* const sE = reinterpret_cast<double2*>(smem + (nrow * sizeof(ColTab) + 15) / 16 * 16);   // [3][ncb][CB]
  double* const sP = reinterpret_cast<double*>(sE + 3 * ncb * CB);                                // [ncb][CB]
  double* const sG = sP + ncb * CB;                                                                // [ncb][2]
  for (int s = tid; s < nrow; s += blockDim.x) {
    ColTab t;
    const int su = min(s, nyu - 1), sv = min(s, nyv - 1);
#pragma unroll
    for (int m = 0; m < 3; ++m) {
      t.wu[m] = gp(a.dyu2i)[3 * su + m];
      t.lu[m] = gp(ca.ayu)[3 * su + m];
      t.wv[m] = gp(a.dyv2i)[3 * sv + m];
      t.lv[m] = gp(ca.ayv)[3 * sv + m];
    }
    t.hu = gp(ca.dthdyu)[su];
    t.hv = gp(ca.dthdyv)[sv];
    tab[s] = t;
  }
  auto E = [&](int f, int k) -> double2& { return sE[(f * ncb + k) * CB + l]; };
  const double dt = gp(a.scal)[S_DT];
  __syncthreads();
  if constexpr (vel) {
    // ---- rhs and the elimination of each chunk from zero
    if (live) {
      double gu = 1.0, gv = 1.0;                      // product of the chunk's forward factors
      const RhsCol k = rhs_col(a, dm, c, 0);
      auto rows = [&](auto fc, auto nc_, auto rc) {
        constexpr int f = decltype(fc)::value, n = decltype(nc_)::value, r0 = decltype(rc)::value;
        double2 prev = zero;
        if constexpr (r0 > 0) prev = x[f][r0 - 1];
#pragma unroll
        for (int e = 0; e < NR; ++e) {
          const int r = r0 + e;
          if (r < R) {
            const ColTab& t = tab[s0 + r];
            const double* const w = f < 2 ? t.wu : t.wv;
            const double* const lu = f < 2 ? t.lu : t.lv;
            const double2 Lu = dadd(dadd(drm(w[0], um[n]), drm(k.k2 + w[1], u0[n])), drm(w[2], up[n][e]));
            double2 du = dadd(drm(a.C1, Lu), drm(a.C2, vo[n][e]));
            if (f < 2) {
              du = dadd(du, dim(-a.dR * (f == 0 ? k.kx : k.kz), pp[e]));
              if (f == 0) du.x += k.mp;
            } else {
              du = dadd(du, drm(-a.dR * dm.ddthetavi * t.hv, dsub(pp[e + 1], pp[e])));
            }
            du = dsub(du, drm(a.g, vn[n][e]));
            double2 rhs = drm(k.axzi, dadd(u0[n], drm(k.dt, du)));
            const bool can = ((f < 2 ? canu : canv) >> r) & 1u;
            rhs.x = can ? vn[n][e].x : rhs.x;
            rhs.y = can ? vn[n][e].y : rhs.y;
            um[n] = u0[n];
            u0[n] = up[n][e];
            prev = drm(lu[1], dsub(rhs, drm(lu[0], prev)));
            // (rows past the top are not used: the back substitution starts below them)
            if (f == 0) gu *= -lu[1] * lu[0];
            if (f == 2) gv *= -lu[1] * lu[0];
            x[f][r] = prev;
          }
        }
      };
      auto batch = [&](auto fc, auto rc) {
        constexpr int f = decltype(fc)::value, r0 = decltype(rc)::value;
        if constexpr (r0 < R) {
          if constexpr (PRE) {
            rows(fc, fc, rc);
          } else {
            COLF_FRESH();
            load(fc, I0{}, rc);
            rows(fc, I0{}, rc);
            __builtin_amdgcn_sched_barrier(0);
          }
        }
      };
      auto comp = [&](auto fc) {
        constexpr int f = decltype(fc)::value;
        static_assert(3 * NR >= R, "three batches of rows");
        batch(fc, I0{});
        batch(fc, std::integral_constant<int, NR>{});
        batch(fc, std::integral_constant<int, 2 * NR>{});
        E(f, q) = x[f][R - 1];
      };
      comp(I0{});
      comp(I1{});
      comp(I2{});
      if (l == 0) { sG[2 * q] = gu; sG[2 * q + 1] = gv; }
    }
    __syncthreads();
    double2 in[3] = {zero, zero, zero};
    if (live) {
      // (unrolled: the chunk values of several steps are read together)
#pragma unroll 8
      for (int k = 0; k < q; ++k) {
        const double g0 = sG[2 * k], g1 = sG[2 * k + 1];
        in[0] = dadd(E(0, k), drm(g0, in[0]));
        in[1] = dadd(E(1, k), drm(g0, in[1]));
        in[2] = dadd(E(2, k), drm(g1, in[2]));
      }
    }
    __syncthreads();
    if (live) {
      // true eliminated rows, then the back substitution of the chunk: from the boundary row
      // above in the last chunk, from zero in the others
      COLF_FRESH();
      double2 top[2] = {zero, zero};                  // the last eliminated row of u, w
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const ColTab& t = tab[s0 + r];
        const double m = -t.lu[1] * t.lu[0];
        in[0] = drm(m, in[0]);
        in[1] = drm(m, in[1]);
        in[2] = drm(-t.lv[1] * t.lv[0], in[2]);
#pragma unroll
        for (int f = 0; f < 3; ++f) x[f][r] = dadd(x[f][r], in[f]);
        if (r < nlv) {
          top[0] = x[0][r];
          top[1] = x[1][r];
        }
        if (!PRE && r % BR == BR - 1) __builtin_amdgcn_sched_barrier(0);
      }
      // last row of the u grid: rhs = 0; the wall row of the v grid is zero
      const bool last = q == nc - 1;
      double2 b[3];
      {
        const double* const lt = tab[nyu - 1].lu;
#pragma unroll
        for (int f = 0; f < 2; ++f) b[f] = last ? drm(lt[1], dsub(zero, drm(lt[0], top[f]))) : zero;
        b[2] = zero;
      }
      if (!pres && last) {
        u1.st(off(nyu - 1), b[0]);
        u3.st(off(nyu - 1), b[1]);
      }
      double hu = 1.0, hv = 1.0;
      COLF_FRESH();
#pragma unroll
      for (int r = R - 1; r >= 0; --r) {
        const ColTab& t = tab[s0 + r];
        const bool oku = r < nlv, okv = s0 + r < nyv - 1;
#pragma unroll
        for (int f = 0; f < 3; ++f) {
          const double2 v = dsub(x[f][r], drm(f < 2 ? t.lu[2] : t.lv[2], b[f]));
          const bool ok = f < 2 ? oku : okv;
          b[f].x = ok ? v.x : b[f].x;
          b[f].y = ok ? v.y : b[f].y;
          x[f][r] = b[f];                             // past the top: the boundary value
        }
        hu = oku ? -t.lu[2] * hu : hu;
        hv = okv ? -t.lv[2] * hv : hv;
        if (!PRE && r % BR == 0) __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int f = 0; f < 3; ++f) E(f, q) = b[f];
      if (l == 0) { sG[2 * q] = hu; sG[2 * q + 1] = hv; }
    }
    __syncthreads();
    if (live) {
      in[0] = in[1] = in[2] = zero;
#pragma unroll 8
      for (int k = nc - 1; k > q; --k) {
        const double g0 = sG[2 * k], g1 = sG[2 * k + 1];
        in[0] = dadd(E(0, k), drm(g0, in[0]));
        in[1] = dadd(E(1, k), drm(g0, in[1]));
        in[2] = dadd(E(2, k), drm(g1, in[2]));
      }
      COLF_FRESH();
      // zero incoming values in the last chunk, the only one with rows past the top
#pragma unroll
      for (int r = R - 1; r >= 0; --r) {
        const ColTab& t = tab[s0 + r];
        in[0] = drm(-t.lu[2], in[0]);
        in[1] = drm(-t.lu[2], in[1]);
        in[2] = drm(-t.lv[2], in[2]);
        const bool okv = s0 + r < nyv - 1;            // the wall face stays zero
        x[0][r] = dadd(x[0][r], in[0]);
        x[1][r] = dadd(x[1][r], in[1]);
        x[2][r] = okv ? dadd(x[2][r], in[2]) : zero;
        if (!PRE && r % BR == 0) __builtin_amdgcn_sched_barrier(0);
      }
    }
    __syncthreads();
  }
  if constexpr (!pres) {
    if (live) {
#pragma unroll
      for (int r = 0; r < R; ++r)
        if (r < nlv) {
          const unsigned o = off(s0 + r);
          u1.st(o, x[0][r]);
          u3.st(o, x[1][r]);
          u2.st(o, x[2][r]);
        }
      if (q == 0) {
        u1.st(off(0), dsub(zero, drm(tab[0].lu[2], x[0][0])));
        u3.st(off(0), dsub(zero, drm(tab[0].lu[2], x[1][0])));
        u2.st(off(0), zero);
      }
    }
    return;
  } else {
  double2 vlow = zero;                                // v at the face below this thread's levels
  if (!vel && live) {
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const unsigned o = off(min(s0 + r, np));
      x[0][r] = u1.ld(o);
      x[1][r] = u3.ld(o);
      x[2][r] = u2.ld(o);
    }
    vlow = u2.ld(off(s0 - 1));
  }
  if (vel) {
    if (live) E(2, q) = x[2][R - 1];
    __syncthreads();
    if (live && q > 0) vlow = E(2, q - 1);
  }
  // constant flow rate: the block of column 0 sums the flow rate in chunk order and adds
  // g times the response u11 of the mean flow to a unit pressure gradient (from k_prep)
  if (ca.ctu && c0 == 0) {                            // uniform over the block
    const CTU& ct = ca.ct;
    const gptr<const double> yv = gp(yvp);
    double s = 0.0;
    if (live && l == 0) {
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const int j = s0 + r - dm.d;                  // Fortran plane index
        if (j >= 1 && j <= dm.ny - 1 && r < nlv) s += (yv[j + dm.d] - yv[j - 1 + dm.d]) * x[0][r].x;
        __builtin_amdgcn_sched_barrier(0);
      }
      sP[at] = s;
    }
    __syncthreads();
    if (live && l == 0) {
      double qx0 = 0.0;
      for (int k = 0; k < nc; ++k) qx0 += sP[k * CB];
      const gptr<const double> u11 = gp(ct.work);     // u11(0..ny), then qx1
      const gptr<double> scal = gp(ca.scal);
      const double g = (scal[S_QXT] - qx0) / u11[dm.ny + 1];
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const int j = s0 + r - dm.d;
        if (j >= 0 && j <= dm.ny && r < nlv) x[0][r].x += g * u11[j];
        __builtin_amdgcn_sched_barrier(0);
      }
      if (q == 0) {
        scal[S_MPGX] = scal[S_MPGX] + g;
        scal[S_DGX] = g;
      }
    }
    __syncthreads();                                  // sP is written again below
  }
  // ---- solveP: divergence, psi = div / (dt (a + b)), elimination of LUsolP in chunks
  const int i = c % dm.mx, k = c / dm.mx;
  const double kx = gp(ca.k1x)[i], kz = gp(ca.k1z)[k];
  const double dv = dm.ddthetavi;
  double2 y[R];
  {
    const double k2x = gp(ca.k2x)[i], k2z = gp(ca.k2z)[k];
    const double dtirk = (1.0 / dt) / ca.ab;
    const double dypin = gp(ca.yu)[2 + dm.d] - gp(ca.yu)[1 + dm.d];
    double m[R];                                       // -lower / pivot of a row
    double g = 1.0;
    if (live) {
      COLF_FRESH();
      if (!PRE && q > 0) a3p = dg3.ld1(off(s0 - 2) / 2u);
      double2 prev = zero;
#pragma unroll
      for (int r0 = 0; r0 < R; r0 += BR) {
        double a3b[BR];
#pragma unroll
        for (int e = 0; e < BR; ++e)
          if (r0 + e < R) a3b[e] = PRE ? a3[r0 + e] : dg3.ld1(off(min(s0 - 1 + r0 + e, np - 1)) / 2u);
#pragma unroll
        for (int e = 0; e < BR; ++e) {
          const int r = r0 + e;
          if (r < R) {
            // (rows past the top give values that nothing reads)
            const int s = s0 + r;
            // the row's lower entry and inverse pivot from the operator and the upper below it
            // (the operations k_buildP formed a3 with)
            const PoisRow w =
                poisson_row_v(s - 1, c == 0, k2x, k2z, np, dv, tab[s].hu, tab[s - 1].hv, tab[s].hv, dypin);
            const double piv = 1.0 / (w.dg - w.lo * a3p);
            a3p = a3b[e];
            const double2 dvg =
                dadd(dadd(dim(kx, x[0][r]), dim(kz, x[1][r])), drm(dv * tab[s].hu, dsub(x[2][r], vlow)));
            vlow = x[2][r];
            double2 ps = drm(dtirk, dvg);
            if (c == 0 && s == 1) ps = zero;
            prev = drm(piv, dsub(ps, drm(w.lo, prev)));
            m[r] = -piv * w.lo;
            g *= m[r];
            y[r] = prev;
            if (!PRE) __builtin_amdgcn_sched_barrier(0);
          }
        }
        if (!PRE) __builtin_amdgcn_sched_barrier(0);
      }
      E(0, q) = prev;
      sP[at] = g;
    }
    __syncthreads();
    double2 in = zero;
    if (live)
#pragma unroll 8
      for (int e = 0; e < q; ++e) in = dadd(E(0, e), drm(sP[e * CB + l], in));
    __syncthreads();
    if (live) {
#pragma unroll
      for (int r = 0; r < R; ++r) {
        in = drm(m[r], in);
        y[r] = dadd(y[r], in);
      }
    }
  }
  if (live) {
    COLF_FRESH();
    double2 b = zero;
    double h = 1.0;
    if (!PRE) {
#pragma unroll
      for (int r = 0; r < R; ++r) a3[r] = dg3.ld1(off(min(s0 - 1 + r, np - 1)) / 2u);
    }
#pragma unroll
    for (int r = R - 1; r >= 0; --r) {
      const double2 v = dsub(y[r], drm(a3[r], b));
      const bool ok = r < nlv;
      b.x = ok ? v.x : b.x;
      b.y = ok ? v.y : b.y;
      y[r] = b;
      h = ok ? -a3[r] * h : h;
    }
    E(1, q) = b;
    sP[at] = h;
  }
  __syncthreads();
  if (!live) return;                                   // no barrier follows
  double2 in = zero;
#pragma unroll 8
  for (int e = nc - 1; e > q; --e) in = dadd(E(1, e), drm(sP[e * CB + l], in));
  // ---- p += psi and v_corr, walking down: `in` is psi of the level above (zero in the last
  // chunk)
  const double dtrk = dt * ca.ab;
  const double kxr = dtrk * kx, kzr = dtrk * kz, dtrk_u2 = dtrk * dv;
  double2 above = in;
  COLF_FRESH();
#pragma unroll
  for (int r0 = R - 1; r0 >= 0; r0 -= BR) {
    double2 pv[BR];
#pragma unroll
    for (int e = 0; e < BR; ++e)
      if (r0 - e >= 0) pv[e] = pr.ld(off(min(s0 - 1 + r0 - e, np - 1)));
#pragma unroll
    for (int e = 0; e < BR; ++e) {
      const int r = r0 - e;
      if (r >= 0) {
        const int s = s0 + r;
        in = drm(-a3[r], in);
        const double2 ps = dadd(y[r], in);
        if (r < nlv) {
          const unsigned o = off(s);
          pr.st(o - pl, dadd(pv[e], ps));
          x[0][r] = dsub(x[0][r], dim(kxr, ps));
          x[1][r] = dsub(x[1][r], dim(kzr, ps));
          u1.st(o, x[0][r]);
          u3.st(o, x[1][r]);
          u2.st(o, s == np ? zero : dsub(x[2][r], drm(dtrk_u2 * tab[s].hv, dsub(above, ps))));
          above = ps;
          if (s == np) {
            u1.st(o + pl, drm(-ca.gw1, x[0][r]));
            u3.st(o + pl, drm(-ca.gw1, x[1][r]));
          }
        }
      }
    }
    if (!PRE) __builtin_amdgcn_sched_barrier(0);
  }
  if (q == 0) {
    u1.st(off(0), drm(-ca.gw0, x[0][0]));
    u3.st(off(0), drm(-ca.gw0, x[1][0]));
    u2.st(off(0), zero);
  }
  }
#undef COLF_FRESH
}

}  // namespace lh

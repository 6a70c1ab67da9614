// lh_zw.hpp -- the z assembly with one wavefront per column line (gfx950, FP64), for planes of 576 x 576
// and of 384 x 384 collocation points.
//
// The z transform is linear and ikx constant along a z line, so the six products of a level are
// transformed as they are and combined afterwards (UU .. VW their transforms, kept modes only):
//   Nu1(l) = ikx UU(l) + ikz UW(l) + m_u (UV(l) - UV(l-1))
//   Nu3(l) = ikx UW(l) + ikz WW(l) + m_u (VW(l) - VW(l-1))
//   Nu2(l) = ikx UV(l) + ikz VW(l) + m_v (VV(l+1) - VV(l))
// which reads every product row once (one block per field would read nine rows for six) and
// takes the same six transforms per level.  UV(l) completes Nu1(l) and at once begins Nu1(l+1),
// so that three sums of 6 values per lane (4 at 384 points) are all a wave carries from product to
// product.
//
// The x pass writes the products in tiles: the N / 2 row pairs (z, z + N / 2) of 8 kx columns of one
// product and level are one contiguous run of N / 2 x 16 values, row pair p holding P[k] and P[N
// - k] of its columns (P the spectrum of the packed rows).  A block of eight waves owns one
// column group and a chunk of levels and takes one tile after the other: the next tile streams
// from HBM straight into one half of the LDS (global_load_lds, no registers) while the waves
// transform the tile in the other half, wave w column w, without a barrier among them, with the lanes
// and radices of the x pass (lh_xw.hpp, lh_xs.hpp) and the column's own places in the tile as its
// transpose line.  One barrier per tile, and a second where a finished sum leaves.
//
// LDS image of a tile: chunks of four row pairs (64 values, one wave-wide load) 65 values apart,
// value e = 8 part + column of pair p at place (e + 2 (p % 4)) % 16 of its 16, which spreads the
// z-strided reads of a column over the banks.
//
// Bound by memory: 384 x 289 x 384 reads 3.2 GB of products and writes 1.0 GB of Nu, 0.86 ms at the
// 4.9 TB/s of a large copy, and measures 0.97 ms.  The block-level assembly (k_zasm, one block per
// field) read 4.6 GB there and took 1.66 ms.  On the way: column-strided stores of 16 bytes 1.34 ms,
// the blocks of a chunk on one XCD 1.16, product loads that leave no lines in the L2 1.08, runs of
// eight columns through the LDS 0.97.  The transforms alone take 0.62 ms.  256 x 97 x 256: 0.16 ms
// (k_zasm 0.29), floor 0.13.
#pragma once
#include "lh_colf.hpp"
#include "lh_nl.hpp"
#include "lh_xs.hpp"

namespace lh {
namespace zw {

constexpr int COLS = 8;                       // columns per tile
constexpr int CHB = 65 * 16;                  // bytes between chunks of the LDS image
// values between the tiles of adjacent column groups: one row pair more than the plane has
__host__ __device__ constexpr int tile(int pz) { return (pz / 2 + 1) * 16; }
__host__ __device__ constexpr int groups(int mx) { return (mx + COLS - 1) / COLS; }
// values of the product buffer: [product][level][column group][row pair][part][column]
inline size_t zp_values(int nlev, int mx, int pz) { return (size_t)6 * nlev * groups(mx) * tile(pz); }

// the forward transform of N = R1 x 64 points in the places of a column (see k_zw): R1 values of a lane
// behind its last transpose, SL slots ahead of the first
template <int N_> struct Shape {
  static constexpr int N = N_, NP = N / 2, CH = NP / 4;       // points, row pairs, chunks
  static constexpr int R1 = N / 64, SL = R1 > 8 ? R1 : 8;
  static constexpr int BUFB = CH * CHB;                       // bytes of a tile image
  static constexpr int NK = 2 * N / 3, KJ = NK / 64;          // kept modes, per lane
  static constexpr int TWN = N + 64;                          // table: w_N^{+n t} at 64 n + t, w_64^{+j} at N + j
  static constexpr size_t LDS = 2 * (size_t)BUFB + TWN * sizeof(double2) + NK * sizeof(double);
  static_assert(CH % 8 == 0 && 8 * CH >= NK, "eight waves load a tile; a finished sum fits a column's places");
};

}  // namespace zw

struct ZW {
  const double2* zp;                         // product tiles
  const double2* tw;                         // w_N^{-j}, j < N
  double2 *nu1, *nu2, *nu3;                  // Nu_new of this substep
  const double *dthdyu, *dthdyv, *k1x, *k1z;
  int lc;                                    // levels per block
  const PREP* prep;                          // as in ZASM
  double* cfl;
};

template <int N>
__global__ void __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2))) k_zw(ZW a, Dims dm) {
  using C = double2;
  using S = zw::Shape<N>;
  constexpr int R1 = S::R1, KJ = S::KJ;
  extern __shared__ char smem_raw[];
  const int tid = threadIdx.x, t = tid & 63;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  int bid = blockIdx.x;
  if (a.prep) {
    if (bid < kPrepBlocks) {
      if (tid < 64) prep_block(*a.prep, a.cfl, bid, tid);
      return;
    }
    bid -= kPrepBlocks;
  }
  const int nlev = dm.nyu - 2, mx = dm.mx, ncol = dm.ncol;
  const int ng = zw::groups(mx);
  // The groups of a chunk of levels run on one XCD (blocks go round the XCDs in launch order): runs of
  // eight columns are not whole cache lines, as mx is odd, and a line that two XCDs write leaves each
  // L2 in parts.
  {
    const int nb = gridDim.x - (a.prep ? kPrepBlocks : 0);
    const int x = bid & 7, per = nb >> 3, rest = nb & 7;
    bid = x * per + min(x, rest) + (bid >> 3);
  }
  const int g = bid % ng, l0 = (bid / ng) * a.lc, l1 = min(l0 + a.lc, nlev);
  if (l0 >= l1) return;
  C* const tw = reinterpret_cast<C*>(smem_raw + 2 * S::BUFB);
  double* const kzt = reinterpret_cast<double*>(tw + S::TWN);
  for (int e = tid; e < S::TWN; e += 512) {
    const C w = a.tw[e < N ? (e >> 6) * (e & 63) % N : R1 * (e - N)];
    tw[e] = mk<C>(w.x, -w.y);
  }
  for (int e = tid; e < S::NK; e += 512) kzt[e] = a.k1z[e];

  // ---- this lane's part of a tile load: place i of a chunk holds value e of pair i / 16
  const int pl = t >> 4, ev = ((t & 15) - 2 * pl) & 15;
  const unsigned src = (unsigned)(pl * 16 + ev) * 16u + (unsigned)wv * 1024u;
  const bool ld_ok = g * zw::COLS + (ev & 7) < mx;      // columns past the plane are not loaded
  // CH / 8 wave-wide loads of 16 bytes per lane into the LDS at m0 + 16 lane.  As asm, because the
  // compiler makes every later LDS read wait for them (it cannot tell the two tile images apart);
  // the loop waits for them itself, ahead of the barrier that hands the tile over.  Nor does it put wait
  // states into asm: the load reads M0 one state after its write at the earliest, and the scalar
  // registers of its base five after a vector instruction's (v_readlane's).  s_mov and s_nop are five.
  const unsigned lds0 = (unsigned)(unsigned long long)(__attribute__((address_space(3))) char*)smem_raw +
                        (unsigned)wv * zw::CHB;
  auto issue = [&](int q, int l, int buf) {
    const ColF tile(a.zp + (((size_t)q * nlev + l) * ng + g) * zw::tile(N));     // (base in scalar registers)
    if (ld_ok) {
#pragma unroll
      for (int j = 0; j < S::CH / 8; ++j)
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 3\n\tglobal_load_lds_dwordx4 %1, %2 nt"
                     :
                     : "s"(__builtin_amdgcn_readfirstlane(lds0 + (unsigned)buf * S::BUFB + (unsigned)j * (8 * zw::CHB))),
                       "v"(src), "s"(tile.b + j * 8192)
                     : "memory", "m0");
    }
  };

  // ---- this wave's column
  const int col = g * zw::COLS + wv;
  const bool k0 = col == 0;
  const double sc = 0.5 / ((double)dm.px * (double)N);      // 1/px, 1/pz and the halving of the row separation
  const double kx = sc * a.k1x[min(col, mx - 1)];
  const int n1 = min(t >> 3, R1 - 1), t1 = t & 7;              // (lanes past R1 x 8 repeat the last ones)
  auto place = [&](int p, int part) {                          // byte address of this column's value of pair p
    return (p >> 2) * zw::CHB + (p & 3) * 256 + ((part * 8 + wv + 2 * (p & 3)) & 15) * 16;
  };
  // rows z = n1 + R1 (t1 + 8 s), s < 4, pair with s + 4; a ninth n1 = 8 goes across the lanes: slot 8
  // holds z = 8 + 9 bitrev6(t)
  constexpr int PS = 8 * R1 / 4;                               // chunks from one s to the next
  const int p0 = n1 + R1 * t1, z8 = 8 + 9 * (int)(__brev((unsigned)t) >> 26);
  const int p8 = z8 >= S::NP ? z8 - S::NP : z8;
  const int ra = place(p0, 0), rb = k0 ? ra : place(p0, 1);
  const int ra8 = R1 == 9 ? place(p8, 0) : 0, rb8 = R1 == 9 && !k0 ? place(p8, 1) : ra8;
  // transpose line of the wave: value j (0..7) of line c (0..63) at chunk c, pair j / 2 of it, part j % 2
  auto slot = [&](int j) { return (j >> 1) * 256 + (((j & 1) * 8 + wv + 2 * (j >> 1)) & 15) * 16; };
  const int wr = (8 * n1 + t1) * zw::CHB;                      // this lane's line
  const int rd1 = 8 * n1 * zw::CHB + slot(t1);                 // value t1 of lines 8 n1 + m
  const int rd2 = t1 * zw::CHB + slot(t >> 3);                 // value t / 8 of lines 8 m + t1
  // a finished sum: value j of lane t at line t, or, where the image has fewer than 64 chunks, at line
  // t % 32 from value 4 (t / 32) on
  constexpr bool HALF = S::CH < 64;
  auto pline = [](int r) { return (HALF ? r & 31 : r) * zw::CHB; };
  auto pval = [](int r, int j) { return HALF ? j + 4 * (r >> 5) : j; };

  // A finished sum leaves through the column's places in the tile image it was formed from (lane t's
  // values as line t, in the layout of the transpose), so that the block's waves store whole runs of
  // eight columns: this lane stores column t % 8 of the rows kz = 8 w + t / 8 + 64 j.
  const int srow = 8 * wv + (t >> 3), sc8 = t & 7;
  const int sr = pline(srow);
  const bool st_ok = g * zw::COLS + sc8 < mx;
  const unsigned no = (unsigned)(srow * mx + min(g * zw::COLS + sc8, mx - 1)) * 16u;
  auto sslot = [&](int j) { return (j >> 1) * 256 + (((j & 1) * 8 + sc8 + 2 * (j >> 1)) & 15) * 16; };
  auto parked = [&](C (&w)[KJ], int b) {
#pragma unroll
    for (int j = 0; j < KJ; ++j) w[j] = *reinterpret_cast<const C*>(smem_raw + b * S::BUFB + sr + sslot(pval(srow, j)));
  };
  auto store = [&](double2* nu, int s, const C (&w)[KJ]) {
    if (st_ok) {
#pragma unroll
      for (int j = 0; j < KJ; ++j) {
        const ColF f(nu + (size_t)s * ncol + (size_t)(64 * j) * mx);
        f.st(no, w[j]);
      }
    }
  };
  C N1[KJ], N2[KJ], N3[KJ];
#pragma unroll
  for (int j = 0; j < KJ; ++j) N1[j] = N2[j] = N3[j] = mk<C>(0, 0);
  // tiles in the order uu, uw, ww, uv, vw of level l, vv of level l + 1; products before level l0 only
  // begin the sums of the first one
  int q = l0 > 0 ? 3 : 5, l = l0 - 1, buf = 0;
  auto lev = [&](int qq, int ll) { return qq == 5 ? ll + 1 : ll; };
  issue(q == 3 ? 4 : 3, lev(q, l), 0);
  double2* done = nullptr;                                      // field parked in the image of the tile before
  int dl = 0;                                                   // and its plane
  bool stored = false;
  __syncthreads();                                              // the tables
  for (;;) {
    q = __builtin_amdgcn_readfirstlane(q);
    l = __builtin_amdgcn_readfirstlane(l);
    int qn = q == 5 ? 0 : q + 1, ln = q == 5 ? l + 1 : l;
    bool more = ln < l1 && !(qn == 5 && ln + 1 >= nlev);
    // the tile's loads are older than the stores of the tile before
    static_assert(KJ == 6 || KJ == 4, "stores of a sum");
    if (stored && KJ == 6) asm volatile("s_waitcnt vmcnt(6) lgkmcnt(0)" ::: "memory");
    else if (stored) asm volatile("s_waitcnt vmcnt(4) lgkmcnt(0)" ::: "memory");
    else asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    C w[KJ];
    stored = done != nullptr;
    if (stored) {
      parked(w, buf ^ 1);
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
    }
    // buffer order of the products in zp: 0 uu, 1 uw, 2 ww, 3 vv, 4 uv, 5 vw
    if (more) issue(qn < 3 ? qn : (qn == 5 ? 3 : qn + 1), lev(qn, ln), buf ^ 1);
    asm volatile("" ::: "memory");
    if (stored) store(done, dl, w);
    done = nullptr;
    char* const tb = smem_raw + buf * S::BUFB;
    auto at = [&](int o) -> C& { return *reinterpret_cast<C*>(tb + o); };
    C v[S::SL];
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const C P = at(ra + s * PS * zw::CHB), Q = at(rb + s * PS * zw::CHB);
      v[s] = mk<C>(P.x + Q.x, k0 ? 0.0 : P.y - Q.y);
      v[s + 4] = mk<C>(P.y + Q.y, k0 ? 0.0 : Q.x - P.x);
    }
    if constexpr (R1 == 9) {
      const C P = at(ra8), Q = at(rb8);
      const bool hi = (t & 1) != 0;                             // z8 >= NP
      v[8] = hi ? mk<C>(P.y + Q.y, k0 ? 0.0 : Q.x - P.x) : mk<C>(P.x + Q.x, k0 ? 0.0 : P.y - Q.y);
      v[8] = xw::dit64_fwd(v[8], t, tw + (N - xw::TW64));
    }
    // forward transform (xw::fwd576, xs::Whole384 on this line's places)
    {
      C c8[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) c8[e] = v[e];
      xw::dft8_t<false>(c8);
#pragma unroll
      for (int e = 1; e < 8; ++e) c8[xw::brev3(e)] = xw::cmc(c8[xw::brev3(e)], tw[N + t1 * e]);
      xw::mem_fence_compiler();
#pragma unroll
      for (int e = 0; e < 8; ++e) at(wr + slot(e)) = c8[xw::brev3(e)];
      xw::mem_fence_compiler();
#pragma unroll
      for (int m = 0; m < 8; ++m) c8[m] = at(rd1 + m * zw::CHB);
      xw::mem_fence_compiler();
      xw::dft8_t<false>(c8);
#pragma unroll
      for (int e = 0; e < 8; ++e) at(wr + slot(e)) = c8[xw::brev3(e)];
      xw::mem_fence_compiler();
    }
    {
      C y[R1];
#pragma unroll
      for (int m = 0; m < (R1 < 8 ? R1 : 8); ++m) y[m] = at(rd2 + m * 8 * zw::CHB);
      xw::mem_fence_compiler();
      if constexpr (R1 == 9) y[8] = v[8];
#pragma unroll
      for (int m = 1; m < R1; ++m) y[m] = xw::cmc(y[m], tw[m * 64 + t]);
      if constexpr (R1 == 9) {
        xw::dft9_t<false>(y);
#pragma unroll
        for (int r = 0; r < R1; ++r) v[r] = y[xw::perm9(r)];
      } else {
        xs::Dft<R1, false>::run(y);
#pragma unroll
        for (int r = 0; r < R1; ++r) v[r] = y[r];
      }
    }
    // kept modes k = t + 64 j: the first and the last KJ / 2 slots of the line
    C X[KJ];
#pragma unroll
    for (int j = 0; j < KJ; ++j) X[j] = v[j < KJ / 2 ? j : j + R1 - KJ];
    auto add_kx = [&](C (&n)[KJ]) {
#pragma unroll
      for (int j = 0; j < KJ; ++j) n[j] = mk<C>(n[j].x - kx * X[j].y, n[j].y + kx * X[j].x);
    };
    auto add_kz = [&](C (&n)[KJ]) {
#pragma unroll
      for (int j = 0; j < KJ; ++j) {
        const double kz = sc * kzt[t + 64 * j];
        n[j] = mk<C>(n[j].x - kz * X[j].y, n[j].y + kz * X[j].x);
      }
    };
    // the upper operand of a y difference completes sum n, plane s of field nu; the next level's
    // sum begins with its lower operand
    auto finish = [&](C (&n)[KJ], double2* nu, double m, double mnext) {
#pragma unroll
      for (int j = 0; j < KJ; ++j) n[j] = mk<C>(n[j].x + m * X[j].x, n[j].y + m * X[j].y);
      if (l >= l0) {
        xw::mem_fence_compiler();
#pragma unroll
        for (int j = 0; j < KJ; ++j) at(pline(t) + slot(pval(t, j))) = n[j];
        xw::mem_fence_compiler();
        done = nu;
        dl = l + 1;
      }
#pragma unroll
      for (int j = 0; j < KJ; ++j) n[j] = mk<C>(-mnext * X[j].x, -mnext * X[j].y);
    };
    // (through the constant address space: scalar loads, which do not wait for the tile in flight)
    using KP = const __attribute__((address_space(4))) double*;
    const double ms = sc * dm.ddthetavi;
    if (q == 0) {
      add_kx(N1);
    } else if (q == 1) {
      add_kz(N1);
      add_kx(N3);
    } else if (q == 2) {
      add_kz(N3);
    } else if (q == 3) {
      finish(N1, a.nu1, ms * ((KP)a.dthdyu)[l + 1], ms * ((KP)a.dthdyu)[l + 2]);
      add_kx(N2);
    } else if (q == 4) {
      finish(N3, a.nu3, ms * ((KP)a.dthdyu)[l + 1], ms * ((KP)a.dthdyu)[l + 2]);
      add_kz(N2);
    } else {
      finish(N2, a.nu2, ms * ((KP)a.dthdyv)[l + 1], ms * ((KP)a.dthdyv)[l + 2]);
    }
    if (!more) break;
    q = qn;
    l = ln;
    buf ^= 1;
  }
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  C w[KJ];
  parked(w, buf);
  store(done, dl, w);
}

}  // namespace lh

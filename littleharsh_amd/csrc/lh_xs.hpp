// lh_xs.hpp -- the nonlinear x pass in FP64 at 48, 72, 96, 144 and 384 points (gfx950): every line
// stays with the lanes of one wavefront, as in lh_xw.hpp at 576.
//
// A line of N = R1 T points has T lanes of R1 points each, so that a wave takes 64 / T row pairs
// at once:
//
//   x[n1 + R1 n2] = sum_t wT^{n2 t} ( wN^{n1 t} sum_r X[t + T r] w_{R1}^{n1 r} )
//
// lane t loads X[t + T r], r < R1, straight from the Z rows and does the inner sum and the twiddle
// in its registers; one transpose through the wave's LDS line hands lane n1 < R1 the T values of its
// outer sum, after which it holds x[n1 + R1 n2] in slot n2.  The forward transform takes the same
// steps backwards and ends with X[t + T r] in lane t.  One transpose per transform, no barrier:
//   48 = 6 x 8 (8 lines per wave), 72 = 8 x 9 (7), 96 = 8 x 12 (5), 144 = 12 x 12 (5).
// At 384 = 6 x 64 the line has the whole wave and the outer sums of 64 run as 8 x 8 with a second
// transpose, eight lanes per n1.
//
// Lanes without a part of their own (n1 >= R1; those past the last whole line; lines past the last
// row pair) repeat the work of another one: they read and write what it does, and only their global
// stores are left out.
//
// Bound by latency and by the FP64 rate of the few waves there are: a wave is a chain of nine
// transforms per level, 0.7 (48 points) to 1.1 us (144) each with one or two waves per SIMD.  Measured
// per launch, this pass and before it the one of a block per row pair (k_xraw2, five waves to a line
// group, a barrier after each stage): 32 x 41 x 32 9.9 us (20.6), 64 x 97 x 64 23.6 us (39),
// 96 x 145 x 96 48 us (67), 256 x 97 x 256 200 us (365; 0.68 GB, 138 us at the 4.9 TB/s of a copy).
// At 48 and 384 points the registers hold a level's three loads at once (14.1 against 15.0 us at
// 32 x 41 x 32 unsplit, 200 against 205 us at 256 x 97 x 256); the others fetch field by field.
// Three waves per SIMD at 384 (168 registers) are slower, 218 us.
#pragma once
#include "lh_colf.hpp"
#include "lh_xw.hpp"

namespace lh {
namespace xs {

// Every multiplication here is written out as a product or as a fused multiply-add, and the compiler
// may fuse nothing by itself: it would round one and the same transform differently in the loop, ahead
// of it and in the split kernel, and the results must not depend on the launch.
__device__ __forceinline__ double2 prod(double2 f, double2 g) {
#pragma clang fp contract(off)
  return mk<double2>(f.x * g.x, f.y * g.y);
}
__device__ __forceinline__ double2 mean(double2 f, double2 g) {
#pragma clang fp contract(off)
  return mk<double2>(0.5 * (f.x + g.x), 0.5 * (f.y + g.y));
}
// a w, or a conj(w)
template <bool CONJ> __device__ __forceinline__ double2 turn(double2 a, double2 w) {
#pragma clang fp contract(off)
  return CONJ ? mk<double2>(fma(a.x, w.x, a.y * w.y), fma(a.y, w.x, -(a.x * w.y)))
              : mk<double2>(fma(a.x, w.x, -(a.y * w.y)), fma(a.y, w.x, a.x * w.y));
}
// In-register DFT of size R, natural order: 4, 3 and 2 points, and composites as in DFT
template <int R, bool INV> struct Dft {
  static __device__ __forceinline__ void run(double2* v) {
    constexpr int A = split<R>::A, B = split<R>::B;
    double2 y[R];
#pragma unroll
    for (int n2 = 0; n2 < B; ++n2) {
      double2 t[A];
#pragma unroll
      for (int n1 = 0; n1 < A; ++n1) t[n1] = v[n2 + B * n1];
      Dft<A, INV>::run(t);
#pragma unroll
      for (int k1 = 0; k1 < A; ++k1) {
        const int m = (n2 * k1) % R;
        double2 z = t[k1];
        if (4 * m == R) z = rot<INV>(z);
        else if (2 * m == R) z = mk<double2>(-z.x, -z.y);
        else if (4 * m == 3 * R) z = rot<!INV>(z);
        else if (m != 0) z = turn<INV>(z, mk<double2>(wre<R>(m), wim<R>(m)));
        y[n2 * A + k1] = z;
      }
    }
#pragma unroll
    for (int k1 = 0; k1 < A; ++k1) {
      double2 t[B];
#pragma unroll
      for (int n2 = 0; n2 < B; ++n2) t[n2] = y[n2 * A + k1];
      Dft<B, INV>::run(t);
#pragma unroll
      for (int k2 = 0; k2 < B; ++k2) v[k1 + A * k2] = t[k2];
    }
  }
};
template <bool INV> struct Dft<2, INV> : DFT<2, INV, double2> {};
template <bool INV> struct Dft<4, INV> : DFT<4, INV, double2> {};
template <bool INV> struct Dft<3, INV> {
  static __device__ __forceinline__ void run(double2* v) {
    const double s = INV ? 0.86602540378443864676 : -0.86602540378443864676;
    const double2 t = cadd(v[1], v[2]), d = csub(v[1], v[2]);
    const double2 c = mk<double2>(fma(-0.5, t.x, v[0].x), fma(-0.5, t.y, v[0].y));
    v[0] = cadd(v[0], t);
    v[1] = mk<double2>(fma(-s, d.y, c.x), fma(s, d.x, c.y));
    v[2] = mk<double2>(fma(s, d.y, c.x), fma(-s, d.x, c.y));
  }
};
__device__ __forceinline__ double2 cfl_uv(double2 u, double2 v, double dxi, double dyi) {
#pragma clang fp contract(off)
  return mk<double2>(fma(fabs(v.x), dyi, fabs(u.x) * dxi), fma(fabs(v.y), dyi, fabs(u.y) * dxi));
}
__device__ __forceinline__ double cfl_max(double cmax, double2 uv, double2 w, double dzi) {
  return nanmax(cmax, nanmax(fma(fabs(w.x), dzi, uv.x), fma(fabs(w.y), dzi, uv.y)));
}

// N = R1 x T, T lanes per line; LP: values between the rows of a transpose (odd, so that lanes a row
// apart hit different banks), LS: values between the lines of a wave (= T mod 8: a write continues
// from one line to the next without a bank twice)
template <int N_, int R1_, int T_, int LS_, int WPB_, int CAP_> struct Two {
  static constexpr int N = N_, R1 = R1_, T = T_, MX = N / 3 + 1;
  static constexpr int SL = T;                       // slots of a field per lane
  static constexpr int LPW = 64 / T;                 // lines per wave
  static constexpr int LP = T | 1, LS = LS_, LINE = LPW * LS;
  static constexpr int TWN = N;                      // table: w_N^{+n1 t} at n1 T + t
  static constexpr int WPB = WPB_;                   // waves per block
  static constexpr int CAP = CAP_;                   // waves per CU (LDS, registers)
  static constexpr bool EARLY = T <= 8;              // registers for a level's three loads at once
  static_assert(N == R1 * T && R1 <= T && LS >= R1 * LP, "line shape");
  static __device__ __forceinline__ int tw_power(int e) { return (e / T) * (e % T); }
  static __device__ __forceinline__ void inv(double2 (&v)[SL], int t, double2* buf, const double2* tw) {
    Dft<R1, true>::run(v);
#pragma unroll
    for (int n = 1; n < R1; ++n) v[n] = turn<false>(v[n], tw[n * T + t]);
    xw::mem_fence_compiler();
#pragma unroll
    for (int n = 0; n < R1; ++n) buf[n * LP + t] = v[n];
    xw::mem_fence_compiler();
    const double2* const row = buf + min(t, R1 - 1) * LP;
#pragma unroll
    for (int s = 0; s < T; ++s) v[s] = row[s];
    xw::mem_fence_compiler();
    Dft<T, true>::run(v);
  }
  static __device__ __forceinline__ void fwd(double2 (&v)[SL], int t, double2* buf, const double2* tw) {
    Dft<T, false>::run(v);
    double2* const row = buf + min(t, R1 - 1) * LP;
    xw::mem_fence_compiler();
#pragma unroll
    for (int s = 0; s < T; ++s) row[s] = v[s];
    xw::mem_fence_compiler();
#pragma unroll
    for (int n = 0; n < R1; ++n) v[n] = buf[n * LP + t];
    xw::mem_fence_compiler();
#pragma unroll
    for (int n = 1; n < R1; ++n) v[n] = turn<true>(v[n], tw[n * T + t]);
    Dft<R1, false>::run(v);
  }
};

// 384 = 6 x 64, a line per wave
struct Whole384 {
  static constexpr int N = 384, R1 = 6, T = 64, MX = N / 3 + 1;
  static constexpr int SL = 8, LPW = 1, LS = 6 * 72, LINE = LS;
  static constexpr int TWN = N + 64;                 // and w_64^{+j} at N + j
  static constexpr int WPB = 4, CAP = 8;
  static constexpr bool EARLY = true;
  static __device__ __forceinline__ int tw_power(int e) { return e < N ? (e / T) * (e % T) : 6 * (e - N); }
  static __device__ __forceinline__ void inv(double2 (&v)[SL], int t, double2* buf, const double2* tw) {
    using C = double2;
    const int t1 = t & 7, g = min(t >> 3, R1 - 1);
    Dft<R1, true>::run(v);
#pragma unroll
    for (int n = 1; n < R1; ++n) v[n] = turn<false>(v[n], tw[n * T + t]);
    xw::mem_fence_compiler();
#pragma unroll
    for (int n = 0; n < R1; ++n) buf[n * T + t] = v[n];
    xw::mem_fence_compiler();
    C b[8];
#pragma unroll
    for (int t2 = 0; t2 < 8; ++t2) b[t2] = buf[g * T + t1 + 8 * t2];
    xw::mem_fence_compiler();
    Dft<8, true>::run(b);
#pragma unroll
    for (int m2 = 1; m2 < 8; ++m2) b[m2] = turn<false>(b[m2], tw[N + m2 * t1]);
#pragma unroll
    for (int m2 = 0; m2 < 8; ++m2) buf[g * 72 + m2 * 9 + t1] = b[m2];
    xw::mem_fence_compiler();
#pragma unroll
    for (int q = 0; q < 8; ++q) b[q] = buf[g * 72 + t1 * 9 + q];
    xw::mem_fence_compiler();
    Dft<8, true>::run(b);
#pragma unroll
    for (int m1 = 0; m1 < 8; ++m1) v[m1] = b[m1];
  }
  static __device__ __forceinline__ void fwd(double2 (&v)[SL], int t, double2* buf, const double2* tw) {
    using C = double2;
    const int t1 = t & 7, g = min(t >> 3, R1 - 1);
    Dft<8, false>::run(v);
#pragma unroll
    for (int q = 1; q < 8; ++q) v[q] = turn<true>(v[q], tw[N + t1 * q]);
    xw::mem_fence_compiler();
#pragma unroll
    for (int q = 0; q < 8; ++q) buf[g * 72 + t1 * 9 + q] = v[q];
    xw::mem_fence_compiler();
    C b[8];
#pragma unroll
    for (int m2 = 0; m2 < 8; ++m2) b[m2] = buf[g * 72 + m2 * 9 + t1];
    xw::mem_fence_compiler();
    Dft<8, false>::run(b);
#pragma unroll
    for (int t2 = 0; t2 < 8; ++t2) buf[g * T + t1 + 8 * t2] = b[t2];
    xw::mem_fence_compiler();
#pragma unroll
    for (int n = 0; n < R1; ++n) v[n] = buf[n * T + t];
    xw::mem_fence_compiler();
#pragma unroll
    for (int n = 1; n < R1; ++n) v[n] = turn<true>(v[n], tw[n * T + t]);
    Dft<R1, false>::run(v);
  }
};

template <int N> struct Family;
template <> struct Family<48> : Two<48, 6, 8, 56, 4, 8> {};
template <> struct Family<72> : Two<72, 8, 9, 73, 4, 8> {};
template <> struct Family<96> : Two<96, 8, 12, 108, 2, 6> {};
template <> struct Family<144> : Two<144, 12, 12, 156, 2, 6> {};
template <> struct Family<384> : Whole384 {};

// rows (z0, z0 + 1) of a Z plane -> X[t + T r] of their packed line in slot r (zero past the kept
// modes); get(row, mode) reads a row
template <typename F, class Get> __device__ __forceinline__ void pack(double2 (&v)[F::SL], int t, Get get) {
  double2 a[F::R1], b[F::R1];
#pragma unroll
  for (int r = 0; r < F::R1; ++r) {
    const int first = F::T * r, last = first + F::T - 1;
    if (first >= F::MX && last <= F::N - F::MX) continue;       // (decided when compiling)
    const int k = t + first;
    const int i = k < F::MX ? k : (k > F::N - F::MX ? F::N - k : 0);
    a[r] = get(0, i);
    b[r] = get(1, i);
  }
#pragma unroll
  for (int r = 0; r < F::R1; ++r) {
    const int first = F::T * r, last = first + F::T - 1;
    v[r] = mk<double2>(0, 0);
    if (first >= F::MX && last <= F::N - F::MX) continue;
    const int k = t + first;
    if (last < F::MX) {
      v[r] = mk<double2>(a[r].x - b[r].y, a[r].y + b[r].x);
      if (r == 0 && t == 0) v[r] = mk<double2>(a[r].x, b[r].x);   // mode 0 drops its imaginary parts
    } else if (first > F::N - F::MX) {
      v[r] = mk<double2>(a[r].x + b[r].y, b[r].x - a[r].y);
    } else if (k < F::MX) {
      v[r] = mk<double2>(a[r].x - b[r].y, a[r].y + b[r].x);
    } else if (k > F::N - F::MX) {
      v[r] = mk<double2>(a[r].x + b[r].y, b[r].x - a[r].y);
    }
  }
}

// forward spectrum P -> the pair's row at byte offset o: P[k] at k, P[N - k] at MX + k
template <typename F> __device__ __forceinline__ void store(const double2 (&v)[F::SL], const ColF& d, unsigned o, int t) {
#pragma unroll
  for (int r = 0; r < F::R1; ++r) {
    const int k = t + F::T * r;
    if (k < F::MX) d.st(o + (unsigned)k * 16u, v[r]);
    else if (k > F::N - F::MX) d.st(o + (unsigned)(F::MX + F::N - k) * 16u, v[r]);
  }
}

// the same as one row pair of the product tiles of lh_zw.hpp (as xw::store_tile), group values apart
template <typename F>
__device__ __forceinline__ void store_tile(const double2 (&v)[F::SL], const ColF& d, int group, int t) {
#pragma unroll
  for (int r = 0; r < F::R1; ++r) {
    const int k = t + F::T * r, m = F::N - k;
    if (k < F::MX) d.st_nt((unsigned)((k >> 3) * group + (k & 7)) * 16u, v[r]);
    else if (m < F::MX) d.st_nt((unsigned)((m >> 3) * group + 8 + (m & 7)) * 16u, v[r]);
  }
}

constexpr int kSplitWaves = 3;
template <typename F> constexpr size_t split_lds_bytes() {
  return sizeof(double2) * ((size_t)F::TWN + (size_t)kSplitWaves * F::LINE);
}
template <typename F> constexpr size_t lds_bytes() {
  return sizeof(double2) * ((size_t)F::TWN + (size_t)F::WPB * (F::LINE + 64 * F::SL)) + sizeof(double) * F::WPB * 64;
}

}  // namespace xs

// One wave per (F::LPW row pairs, chunk of lc levels); the walk over the levels, the fields carried
// and the park line are those of k_xw576.
// TILE (one line per wave): rows z and z + pz / 2 pair up and the products go out in tiles
template <int N, bool CFL, bool TILE>
__global__ void __launch_bounds__(64 * xs::Family<N>::WPB) __attribute__((amdgpu_waves_per_eu(2)))
    k_xs(XW a, Dims dm) {
  using F = xs::Family<N>;
  static_assert(!TILE || F::LPW == 1, "tiles: the row pair is the wave's");
  using C = double2;
  constexpr int SL = F::SL;
  extern __shared__ char smem_raw[];
  C* const tw = reinterpret_cast<C*>(smem_raw);
  for (int e = threadIdx.x; e < F::TWN; e += blockDim.x) {
    const C w = static_cast<const C*>(a.tw)[F::tw_power(e) % N];       // w_N^{-j}
    tw[e] = mk<C>(w.x, -w.y);
  }
  __syncthreads();
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int ln = min(lane / F::T, F::LPW - 1), t = lane % F::T;
  C* const wbase = tw + F::TWN + wv * (F::LINE + 64 * SL);
  C* const buf = wbase + ln * F::LS;
  C* const pk = wbase + F::LINE + lane;          // park line: slot s at pk[64 s]
  const int nlev = dm.nyu - 2, npair = dm.pz / 2, nwc = (npair + F::LPW - 1) / F::LPW;
  const int item = blockIdx.x * F::WPB + wv;
  const int l0 = (item / nwc) * a.lc, l1 = min(l0 + a.lc, nlev);
  if (l0 >= l1) return;
  const int pr = (item % nwc) * F::LPW + ln;
  const bool st_ok = pr < npair && lane < F::LPW * F::T;
  const unsigned o = (unsigned)min(pr, npair - 1) * (unsigned)((TILE ? 1 : 2) * F::MX * sizeof(C));
  const int second = TILE ? npair * F::MX : F::MX;              // from a pair's first row to its second
  const size_t slot = (size_t)dm.pz * F::MX;
  const C* zu = static_cast<const C*>(a.zu);
  const C* zw = static_cast<const C*>(a.zw);
  const C* zv = static_cast<const C*>(a.zv);
  const C* zp = static_cast<const C*>(a.zp);
  double* const cm = reinterpret_cast<double*>(tw + F::TWN + F::WPB * (F::LINE + 64 * SL)) + threadIdx.x;
  if constexpr (CFL) *cm = 0.0;
  C cu[SL], cw[SL], p[SL];
  auto park = [&](const C (&x)[SL]) {
    xw::mem_fence_compiler();
#pragma unroll
    for (int s = 0; s < SL; ++s) pk[64 * s] = x[s];
    xw::mem_fence_compiler();
  };
  auto fetch = [&](C (&x)[SL], const C* z, int s) {
    const ColF A(z + (size_t)s * slot);
    xs::pack<F>(x, t, [&](int row, int i) { return A.ld(o + (unsigned)(row * second + i) * 16u); });
  };
  auto out = [&](int q, int l, C (&x)[SL]) {
    F::fwd(x, t, buf, tw);
    if constexpr (TILE) {
      const int group = (npair + 1) * 16;
      xs::store_tile<F>(x, ColF(zp + ((size_t)q * nlev + l) * ((F::MX + 7) / 8) * group + pr * 16), group, t);
    } else {
      if (st_ok) xs::store<F>(x, ColF(zp + ((size_t)q * nlev + l) * slot), o, t);
    }
  };
  fetch(cu, zu, l0 + 1);
  if constexpr (!F::EARLY) F::inv(cu, t, buf, tw);
  fetch(cw, zw, l0 + 1);
  if constexpr (!F::EARLY) F::inv(cw, t, buf, tw);
  fetch(p, zv, l0);
  if constexpr (F::EARLY) {
    F::inv(cu, t, buf, tw);
    F::inv(cw, t, buf, tw);
  }
  F::inv(p, t, buf, tw);
  park(p);                                        // V(j-1)
  for (int l = l0; l < l1; ++l) {
    // V(j), the face above: vv and the CFL maximum at the centre, from V(j-1) parked
    C vj[SL];
    C nu[SL], nw[SL];
    fetch(vj, zv, l + 1);
    if constexpr (F::EARLY) {
      fetch(nu, zu, l + 2);
      fetch(nw, zw, l + 2);
    }
    F::inv(vj, t, buf, tw);
#pragma unroll
    for (int s = 0; s < SL; ++s) {
      const C vb = pk[64 * s];
      p[s] = xs::mean(vb, vj[s]);
    }
    xw::mem_fence_compiler();
    park(cw);                                     // W(j) waits while V(j) stays resident
    if constexpr (CFL) {
      const double dyi = a.dthdyu[l + 1];
      double cmax = *cm;
#pragma unroll
      for (int s = 0; s < SL; ++s) {
        const C w = pk[64 * s];
        cmax = xs::cfl_max(cmax, xs::cfl_uv(cu[s], p[s], dm.dxi, dyi), w, dm.dzi);
      }
      *cm = cmax;
    }
#pragma unroll
    for (int s = 0; s < SL; ++s) p[s] = xs::prod(p[s], p[s]);
    out(3, l, p);
#pragma unroll
    for (int s = 0; s < SL; ++s) p[s] = xs::prod(cu[s], cu[s]);
    out(0, l, p);
#pragma unroll
    for (int s = 0; s < SL; ++s) {
      const C w = pk[64 * s];
      p[s] = xs::prod(cu[s], w);
    }
    out(1, l, p);
#pragma unroll
    for (int s = 0; s < SL; ++s) {
      const C w = pk[64 * s];
      p[s] = xs::prod(w, w);
    }
    out(2, l, p);
    // U(j+1): uv at the face, then carried
    if constexpr (!F::EARLY) fetch(nu, zu, l + 2);
#pragma unroll
    for (int s = 0; s < F::R1; ++s) p[s] = nu[s];
    F::inv(p, t, buf, tw);
#pragma unroll
    for (int s = 0; s < SL; ++s) {
      cu[s] = xs::prod(xs::mean(cu[s], p[s]), vj[s]);
    }
    out(4, l, cu);
#pragma unroll
    for (int s = 0; s < SL; ++s) cu[s] = p[s];
    // W(j+1): vw at the face, then carried; W(j) comes back from the park line, which then takes
    // V(j) for the next level
    if constexpr (!F::EARLY) fetch(nw, zw, l + 2);
#pragma unroll
    for (int s = 0; s < F::R1; ++s) p[s] = nw[s];
    F::inv(p, t, buf, tw);
    xw::mem_fence_compiler();
#pragma unroll
    for (int s = 0; s < SL; ++s) {
      const C w = pk[64 * s];
      pk[64 * s] = vj[s];
      vj[s] = xs::prod(xs::mean(w, p[s]), vj[s]);
    }
    xw::mem_fence_compiler();
    out(5, l, vj);
#pragma unroll
    for (int s = 0; s < SL; ++s) cw[s] = p[s];
  }
  if constexpr (CFL) {
    double cmax = *cm;
    for (int off = 32; off > 0; off >>= 1) cmax = nanmax(cmax, __shfl_down(cmax, off, 64));
    if (lane == 0) atomic_max_pos(a.scal + S_CFLMAX, cmax);
  }
}

// The same for one level per work item, its products shared out over three waves that hold their
// fields in registers: (uu, uw, ww), (uv and the CFL maximum), (vv, vw).  The longest chain is six
// transforms instead of twelve, for fifteen (with the CFL maximum seventeen) in all instead of twelve.
template <int N, bool CFL>
__global__ void __launch_bounds__(64 * xs::kSplitWaves) __attribute__((amdgpu_waves_per_eu(2)))
    k_xs_split(XW a, Dims dm) {
  using F = xs::Family<N>;
  using C = double2;
  constexpr int SL = F::SL;
  extern __shared__ char smem_raw[];
  C* const tw = reinterpret_cast<C*>(smem_raw);
  for (int e = threadIdx.x; e < F::TWN; e += blockDim.x) {
    const C w = static_cast<const C*>(a.tw)[F::tw_power(e) % N];       // w_N^{-j}
    tw[e] = mk<C>(w.x, -w.y);
  }
  __syncthreads();
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int ln = min(lane / F::T, F::LPW - 1), t = lane % F::T;
  C* const buf = tw + F::TWN + wv * F::LINE + ln * F::LS;
  const int nlev = dm.nyu - 2, npair = dm.pz / 2, nwc = (npair + F::LPW - 1) / F::LPW;
  const int item = blockIdx.x * xs::kSplitWaves + wv;
  const int role = item % 3, l = item / 3 / nwc;
  if (l >= nlev) return;
  const int pr = (item / 3 % nwc) * F::LPW + ln;
  const bool st_ok = pr < npair && lane < F::LPW * F::T;
  const unsigned o = (unsigned)min(pr, npair - 1) * (unsigned)(2 * F::MX * sizeof(C));
  const size_t slot = (size_t)dm.pz * F::MX;
  const C* zu = static_cast<const C*>(a.zu);
  const C* zw = static_cast<const C*>(a.zw);
  const C* zv = static_cast<const C*>(a.zv);
  const C* zp = static_cast<const C*>(a.zp);
  auto field = [&](C (&x)[SL], const C* z, int s) {
    const ColF A(z + (size_t)s * slot);
    xs::pack<F>(x, t, [&](int row, int i) { return A.ld(o + (unsigned)(row * F::MX + i) * 16u); });
    F::inv(x, t, buf, tw);
  };
  auto out = [&](int q, C (&x)[SL]) {
    F::fwd(x, t, buf, tw);
    if (st_ok) xs::store<F>(x, ColF(zp + ((size_t)q * nlev + l) * slot), o, t);
  };
  auto mul = [&](C (&x)[SL], const C (&f)[SL], const C (&g)[SL]) {
#pragma unroll
    for (int s = 0; s < SL; ++s) x[s] = xs::prod(f[s], g[s]);
  };
  auto mean = [&](C (&x)[SL], const C (&f)[SL]) {
#pragma unroll
    for (int s = 0; s < SL; ++s) x[s] = xs::mean(f[s], x[s]);
  };
  C f[SL], g[SL], p[SL];
  if (role == 0) {
    field(f, zu, l + 1);
    field(g, zw, l + 1);
    mul(p, f, g);
    out(1, p);
    mul(f, f, f);
    out(0, f);
    mul(g, g, g);
    out(2, g);
  } else if (role == 1) {
    field(f, zu, l + 1);
    field(g, zv, l + 1);
    if constexpr (CFL) {
      field(p, zv, l);
      mean(p, g);                                 // v at the centre
      const double dyi = a.dthdyu[l + 1];
#pragma unroll
      for (int s = 0; s < SL; ++s)
        p[s] = xs::cfl_uv(f[s], p[s], dm.dxi, dyi);
      C w[SL];
      field(w, zw, l + 1);
      double cmax = 0.0;
#pragma unroll
      for (int s = 0; s < SL; ++s)
        cmax = xs::cfl_max(cmax, p[s], w[s], dm.dzi);
      for (int off = 32; off > 0; off >>= 1) cmax = nanmax(cmax, __shfl_down(cmax, off, 64));
      if (lane == 0) atomic_max_pos(a.scal + S_CFLMAX, cmax);
    }
    field(p, zu, l + 2);
    mean(p, f);
    mul(p, p, g);
    out(4, p);
  } else {
    field(g, zv, l + 1);
    field(p, zv, l);
    mean(p, g);
    mul(p, p, p);
    out(3, p);
    field(f, zw, l + 1);
    field(p, zw, l + 2);
    mean(p, f);
    mul(p, p, g);
    out(5, p);
  }
}

}  // namespace lh

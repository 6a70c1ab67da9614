// lh_ibp.hpp -- the canopy forcing of one plane in one block (gfx950, FP64, transform lengths up to
// 144): inverse z, inverse x, the canopy mask, forward x and forward z (tridLU_3D_IB.f90:224-245,
// 306-325) with the plane in LDS from its rhs modes to the forced ones.
//
// The plane lies in LDS as [z][kx], mx odd, so that lanes a row apart hit different banks.  A wave
// takes 64 / T columns, later 64 / T row pairs, with the lanes and radices of lh_xs.hpp; the
// transposes run in the places of the line itself (along x, where a packed line is longer than its
// rows' modes, real and imaginary parts one after the other), and no wave waits for another but
// between the four directions.
//
// A tip plane's forcing is -beta Lu_y on its canopy points and the rhs elsewhere.  As the transforms
// are linear it is rhs - F(m F^-1(rhs + beta Lu_y)), m the canopy mask: one trip for both fields.
// What the trip of the rhs itself would have done to it has to be done by hand: the column of mode
// kx = 0 keeps the part that belongs to a real row.
//
// Bound by latency: some sixty blocks, each a chain of two loads, four rounds of transforms and a
// store.  Per substep, this launch and before it the three of the stage (z, x and z over all planes):
// 32 x 41 x 32 9.0 us (24.5), 64 x 97 x 64 16.6 us (33.7), 96 x 145 x 96 25.7 us (38).  With up to 16
// waves; eight measure 9.1, 17.1 and 27.6.  Both fields of a tip one after the other take 15, 29 and
// 52 us, in two blocks with a fence between them 23, 67 and 117 (the fence writes an L2 back).
#pragma once
#include "lh_xs.hpp"

namespace lh {

// one block: everything it has to know in one record, so that it waits for memory twice (record, data)
struct IbpJob {
  double2* fld;                          // modes of the plane's rhs, forced in place
  const double2* lu;                     // Lu_y of a tip plane, or null
  const unsigned char* mask;             // [pz][px]
  const double* scal;
  const double2 *twx, *twz;              // w_N^{-j}
  double bre;                            // bRK(kRK)/Re
};

namespace ibp {

template <int PX, int PZ> struct Shape {
  using X = xs::Family<PX>;
  using Z = xs::Family<PZ>;
  static constexpr int LD = X::MX, NZ = 2 * PZ / 3;
  static constexpr int GX = (PZ / 2 + X::LPW - 1) / X::LPW, GZ = (LD + Z::LPW - 1) / Z::LPW;
  static constexpr int WANT = GX > GZ ? GX : GZ;
  static constexpr int WAVES = WANT < 4 ? 4 : (WANT > 16 ? 16 : WANT);
  static constexpr size_t LDS = sizeof(double2) * ((size_t)PZ * LD + X::TWN + Z::TWN) + (size_t)PZ * PX;
};

// place of value (n, t) of a column's transpose, in rows: row n holds its T values turned by n
// where T is even (the lanes that read rows n = 0, 1, .. then hit different banks)
template <typename F> __device__ __forceinline__ int place(int n, int t) {
  if (F::T % 2) return n * F::T + t;
  return n * F::T + (t + n < F::T ? t + n : t + n - F::T);
}

// inverse transform along a column (elements LD apart): X[t + T r] in slot r in, x[n1 + R1 s] in slot s
// of lane n1 out
template <typename F, int LD>
__device__ __forceinline__ void inv_column(double2 (&v)[F::SL], int t, int n1, double2* col, const double2* tw) {
  xs::Dft<F::R1, true>::run(v);
#pragma unroll
  for (int n = 1; n < F::R1; ++n) v[n] = xs::turn<false>(v[n], tw[n * F::T + t]);
  xw::mem_fence_compiler();
#pragma unroll
  for (int n = 0; n < F::R1; ++n) col[place<F>(n, t) * LD] = v[n];
  xw::mem_fence_compiler();
#pragma unroll
  for (int s = 0; s < F::T; ++s) v[s] = col[place<F>(n1, s) * LD];
  xw::mem_fence_compiler();
  xs::Dft<F::T, true>::run(v);
}
template <typename F, int LD>
__device__ __forceinline__ void fwd_column(double2 (&v)[F::SL], int t, int n1, double2* col, const double2* tw) {
  xs::Dft<F::T, false>::run(v);
  xw::mem_fence_compiler();
#pragma unroll
  for (int s = 0; s < F::T; ++s) col[place<F>(n1, s) * LD] = v[s];
  xw::mem_fence_compiler();
#pragma unroll
  for (int n = 0; n < F::R1; ++n) v[n] = col[place<F>(n, t) * LD];
  xw::mem_fence_compiler();
#pragma unroll
  for (int n = 1; n < F::R1; ++n) v[n] = xs::turn<true>(v[n], tw[n * F::T + t]);
  xs::Dft<F::R1, false>::run(v);
}
// one part (real or imaginary) of a transpose in a row pair's places, out[] = in[] seen from the
// other side: lane t gives rows n = 0 .. R1-1 at t and takes row n1, or the reverse
template <typename F, bool INV, class Put, class Take>
__device__ __forceinline__ void turn_part(int t, int n1, double* buf, Put put, Take take) {
  xw::mem_fence_compiler();
  if constexpr (INV) {
#pragma unroll
    for (int n = 0; n < F::R1; ++n) buf[n * F::LP + t] = put(n);
    xw::mem_fence_compiler();
#pragma unroll
    for (int s = 0; s < F::T; ++s) take(s, buf[n1 * F::LP + s]);
  } else {
#pragma unroll
    for (int s = 0; s < F::T; ++s) buf[n1 * F::LP + s] = put(s);
    xw::mem_fence_compiler();
#pragma unroll
    for (int n = 0; n < F::R1; ++n) take(n, buf[n * F::LP + t]);
  }
  xw::mem_fence_compiler();
}
template <typename F, bool INV>
__device__ __forceinline__ void turn_pair(double2 (&v)[F::SL], int t, int n1, double* buf) {
  static_assert(F::R1 * F::LP <= 4 * F::MX, "a part of a line fits the places of its two rows");
  turn_part<F, INV>(t, n1, buf, [&](int i) { return v[i].x; }, [&](int i, double a) { v[i].x = a; });
  turn_part<F, INV>(t, n1, buf, [&](int i) { return v[i].y; }, [&](int i, double a) { v[i].y = a; });
}

}  // namespace ibp

template <int PX, int PZ>
__global__ void __launch_bounds__((64 * ibp::Shape<PX, PZ>::WAVES))
    __attribute__((amdgpu_waves_per_eu(((ibp::Shape<PX, PZ>::WAVES + 3) / 4))))
    k_ib_plane(const IbpJob* __restrict__ jt) {
  using S = ibp::Shape<PX, PZ>;
  using X = typename S::X;
  using Z = typename S::Z;
  using C = double2;
  constexpr int LD = S::LD, NT = 64 * S::WAVES, MX = LD;
  extern __shared__ char smem_raw[];
  C* const pl = reinterpret_cast<C*>(smem_raw);
  C* const twx = pl + PZ * LD;
  C* const twz = twx + X::TWN;
  unsigned char* const mask = reinterpret_cast<unsigned char*>(twz + Z::TWN);
  const IbpJob J = jt[blockIdx.x];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  // mode kz <-> row: the negative ones at the end of the padded line
  auto row_of = [](int kz) { return kz < S::NZ / 2 ? kz : kz + (PZ - S::NZ); };
  constexpr int NE = S::NZ * MX, M = (NE + NT - 1) / NT;      // elements of the plane, per thread
  const double beta = J.bre * gp(J.scal)[S_DT];
  const bool tip = J.lu != nullptr;
  {
    C a[M];
#pragma unroll
    for (int q = 0; q < M; ++q) a[q] = gld((const C*)J.fld, min(tid + q * NT, NE - 1));
    if (tip) {
#pragma unroll
      for (int q = 0; q < M; ++q) {
        const C l = gld(J.lu, min(tid + q * NT, NE - 1));
        a[q] = mk<C>(fma(beta, l.x, a[q].x), fma(beta, l.y, a[q].y));
      }
    }
#pragma unroll
    for (int q = 0; q < M; ++q) {
      const int e = min(tid + q * NT, NE - 1);
      pl[row_of(e / MX) * LD + e % MX] = a[q];
    }
  }
  for (int e = tid; e < X::TWN; e += NT) {
    const C w = gld(J.twx, X::tw_power(e) % PX);
    twx[e] = mk<C>(w.x, -w.y);
  }
  for (int e = tid; e < Z::TWN; e += NT) {
    const C w = gld(J.twz, Z::tw_power(e) % PZ);
    twz[e] = mk<C>(w.x, -w.y);
  }
  {
    const gptr<const unsigned> src = gp(reinterpret_cast<const unsigned*>(J.mask));
    for (int e = tid; e < PZ * PX / 4; e += NT) reinterpret_cast<unsigned*>(mask)[e] = src[e];
  }
  const int lnx = min(lane / X::T, X::LPW - 1), tx = lane % X::T, nx1 = min(tx, X::R1 - 1);
  const int lnz = min(lane / Z::T, Z::LPW - 1), tz = lane % Z::T, nz1 = min(tz, Z::R1 - 1);
  __syncthreads();
  for (int g = wv; g < S::GZ; g += S::WAVES) {
    C* const col = pl + min(g * Z::LPW + lnz, MX - 1);
    C v[Z::SL];
#pragma unroll
    for (int r = 0; r < Z::R1; ++r) {
      const int k = tz + Z::T * r;
      const bool kept = k < S::NZ / 2 || k >= PZ - S::NZ / 2;
      const C a = col[(kept ? k : 0) * LD];
      v[r] = kept ? a : mk<C>(0, 0);
    }
    ibp::inv_column<Z, LD>(v, tz, nz1, col, twz);
#pragma unroll
    for (int s = 0; s < Z::T; ++s) col[(nz1 + Z::R1 * s) * LD] = v[s];
  }
  __syncthreads();
  for (int g = wv; g < S::GX; g += S::WAVES) {
    const int z0 = 2 * min(g * X::LPW + lnx, PZ / 2 - 1);
    C* const row = pl + z0 * LD;
    C v[X::SL];
    xs::pack<X>(v, tx, [&](int r, int i) { return row[r * LD + i]; });
    xs::Dft<X::R1, true>::run(v);
#pragma unroll
    for (int n = 1; n < X::R1; ++n) v[n] = xs::turn<false>(v[n], twx[n * X::T + tx]);
    ibp::turn_pair<X, true>(v, tx, nx1, reinterpret_cast<double*>(row));
    xs::Dft<X::T, true>::run(v);
    // rows z0 (real parts) and z0 + 1 (imaginary parts): 0 on the canopy points, or, for a tip, off them
    const unsigned char* const m0 = mask + z0 * PX;
#pragma unroll
    for (int s = 0; s < X::T; ++s) {
      const int x = nx1 + X::R1 * s;
      v[s] = mk<C>((m0[x] != 0) == tip ? v[s].x : 0.0, (m0[PX + x] != 0) == tip ? v[s].y : 0.0);
    }
    xs::Dft<X::T, false>::run(v);
    ibp::turn_pair<X, false>(v, tx, nx1, reinterpret_cast<double*>(row));
#pragma unroll
    for (int n = 1; n < X::R1; ++n) v[n] = xs::turn<true>(v[n], twx[n * X::T + tx]);
    xs::Dft<X::R1, false>::run(v);
    // the pair's spectrum P: P[k] in row z0, P[PX - k] in row z0 + 1
#pragma unroll
    for (int r = 0; r < X::R1; ++r) {
      const int k = tx + X::T * r;
      if (k < MX) row[k] = v[r];
      else if (k > PX - MX) row[LD + PX - k] = v[r];
    }
  }
  __syncthreads();
  const double sc = 0.5 / ((double)PX * (double)PZ);       // 1/px, 1/pz and the halving of the row separation
  for (int g = wv; g < S::GZ; g += S::WAVES) {
    const int i = min(g * Z::LPW + lnz, MX - 1);
    C* const col = pl + i;
    const bool k0 = i == 0, hi = (nz1 & 1) != 0;           // (R1 is even: a lane's rows are all even or all odd)
    C v[Z::SL];
#pragma unroll
    for (int s = 0; s < Z::T; ++s) {
      const int zb = nz1 + Z::R1 * s - (hi ? 1 : 0);
      const C P = col[zb * LD], Q = k0 ? P : col[(zb + 1) * LD];
      v[s] = hi ? mk<C>(sc * (P.y + Q.y), k0 ? 0.0 : sc * (Q.x - P.x))
                : mk<C>(sc * (P.x + Q.x), k0 ? 0.0 : sc * (P.y - Q.y));
    }
    ibp::fwd_column<Z, LD>(v, tz, nz1, col, twz);
#pragma unroll
    for (int r = 0; r < Z::R1; ++r) col[(tz + Z::T * r) * LD] = v[r];
  }
  __syncthreads();
  C a[M];
#pragma unroll
  for (int q = 0; q < M; ++q) {
    const int e = min(tid + q * NT, NE - 1);
    a[q] = pl[row_of(e / MX) * LD + e % MX];
  }
  if (tip) {
#pragma unroll
    for (int q = 0; q < M; ++q) {
      const int e = min(tid + q * NT, NE - 1), kz = e / MX;
      C r = gld((const C*)J.fld, e);
      if (e % MX == 0) {                         // the real row's part: half of mode kz and of -kz conjugate
        const C o = kz == S::NZ / 2 ? mk<C>(0, 0) : gld((const C*)J.fld, (kz ? S::NZ - kz : 0) * MX);
        r = mk<C>(0.5 * (r.x + o.x), 0.5 * (r.y - o.y));
      }
      a[q] = csub(r, a[q]);
    }
    __syncthreads();                             // (every element has been read)
  }
#pragma unroll
  for (int q = 0; q < M; ++q)
    if (tid + q * NT < NE) gst(J.fld, tid + q * NT, a[q]);
}

}  // namespace lh

// kernels_spectral.hpp -- the transforms of coftxy and cofitxy, and of the field
// downloads, on the transform that takes its input from and hands its output
// to the caller's registers (fft_io).
//
// Rows and columns in a kernel each, with a half spectrum in memory between
// them: launch-bound below about 256^2, bound by memory from 1024^2 (each
// kernel reads and writes the field once).  Against the kernels that stage
// their rows or columns in LDS first, forward and backward together: 256^2
// 16.5 -> 14.4 us, 384^2 19.8 -> 17.2, 512^2 21.8 -> 17.1, 1024^2 37.5 -> 31.2,
// 2048^2 70.9 -> 64.6.  Grids of 64 x 64, 128 x 32 and 64 x 32 take one
// workgroup and one kernel a direction: 64^2 forward 5.7 -> 4.4 us, backward 5.6
// -> 4.0 (128 x 64, with twice the entries: 5.9 -> 5.7, not taken).
// The same passes and formulas as those kernels, so the same bits.
#pragma once
#include "kernels_fused.hpp"

namespace fsibe {

// Rows, RPB of them per workgroup (each within one wave where NT <= 64).
template <int H, int NT, int RPB>
__device__ __forceinline__ void rows_fwd_body(const double *__restrict__ f, double2 *__restrict__ out,
                                              const double2 *__restrict__ twx, int ny, int bid) {
  extern __shared__ double2 lds[];
  constexpr bool WAVE = NT * RPB <= 64;
  static_assert(RPB == 1 || WAVE, "several rows per workgroup: each within one wave");
  using Out = FftOut<H, NT>;
  const int rr = threadIdx.x / NT, t = threadIdx.x - rr * NT, y = bid * RPB + rr;
  double2 *xb = lds + rr * padlen(H);
  const bool act = y < ny;
  const double2 *src = reinterpret_cast<const double2 *>(f) + (size_t)y * H;
  FftTw<H, NT> T;
  T.load(twx, 2, t);
  double2 z[Out::N];
  fft_io<H, NT, false, 1, WAVE, false>(
      xb, T, t, act, [&](int, int, int e) { return src[e]; },
      [&](int i, int r, int, double2 x) { z[i * Out::R + r] = x; });
  grp_sync<WAVE>();
#pragma unroll
  for (int i = 0; i < Out::ITEMS; ++i) {
    if (Out::M % NT != 0 && t + i * NT >= Out::M) continue;
#pragma unroll
    for (int r = 0; r < Out::R; ++r) xb[pidx(t + i * NT + r * Out::M)] = z[i * Out::R + r];
  }
  grp_sync<WAVE>();
  if (!act) return;
#pragma unroll
  for (int i = 0; i < (H + NT - 1) / NT; ++i) {
    const int k = t + i * NT;
    if (H % NT != 0 && k >= H) continue;
    out[(size_t)y * H + k] = r2c_one(xb[pidx(k)], xb[pidx(k == 0 ? 0 : H - k)], twx[k]);
  }
}
template <int H, int NT, int RPB>
__device__ __forceinline__ void rows_inv_body(const double2 *__restrict__ in, double *__restrict__ f,
                                              const double2 *__restrict__ twx, int ny, int bid) {
  extern __shared__ double2 lds[];
  constexpr bool WAVE = NT * RPB <= 64;
  const int rr = threadIdx.x / NT, t = threadIdx.x - rr * NT, y = bid * RPB + rr;
  const bool act = y < ny;
  const double2 *src = in + (size_t)y * H;
  double2 *dst = reinterpret_cast<double2 *>(f) + (size_t)y * H;
  FftTw<H, NT> T;
  T.load(twx, 2, t);
  fft_io<H, NT, true, 1, WAVE, false>(
      lds + rr * padlen(H), T, t, act,
      [&](int, int, int e) { return c2r_elem(src[e], src[e == 0 ? 0 : H - e], e, cconj(twx[e])); },
      [&](int, int, int e, double2 x) { dst[e] = x; });
}
// half spectra -> column transform -> x norm -> packed layout (cof_fftw33.f90:165-189)
template <int L, int TX, int NT>
__device__ __forceinline__ void cols_fwd_body(const double2 *__restrict__ in, double *__restrict__ fk,
                                              const double2 *__restrict__ twy, int H, double norm, int bid, int nblk) {
  extern __shared__ double2 lds[];
  constexpr int NTHR = TX * NT, hy = L / 2;
  constexpr bool WAVE = NTHR <= 64;
  using Out = FftOut<L, NT>;
  const int tid = threadIdx.x, cc = tid % TX, t = tid / TX, nx = 2 * H;
  const int kx = xcd_remap(bid, nblk) * TX + cc;
  double2 *xb = lds + cc;
  FftTw<L, NT> T;
  T.load(twy, 1, t);
  double2 z[Out::N];
  fft_io<L, NT, false, TX, WAVE, false>(
      xb, T, t, true, [&](int, int, int e) { return in[(size_t)e * H + kx]; },
      [&](int i, int r, int, double2 x) { z[i * Out::R + r] = x; });
  grp_sync<WAVE>();
#pragma unroll
  for (int i = 0; i < Out::ITEMS; ++i) {
    if (Out::M % NT != 0 && t + i * NT >= Out::M) continue;
#pragma unroll
    for (int r = 0; r < Out::R; ++r) xb[pidx(t + i * NT + r * Out::M) * TX] = z[i * Out::R + r];
  }
  grp_sync<WAVE>();
#pragma unroll
  for (int i = 0; i < (hy + NT - 1) / NT; ++i) {
    const int ky = t + i * NT;
    if (hy % NT != 0 && ky >= hy) continue;
    double2 r0, r1;
    const double2 p = xb[pidx(ky) * TX];
    if (ky == 0) {
      r0 = make_double2(p.x * norm, p.y * norm);
      r1 = make_double2(0.0, 0.0);
    } else {
      const double2 m = xb[pidx(L - ky) * TX];
      r0 = make_double2(0.5 * (p.x + m.x) * norm, 0.5 * (p.y + m.y) * norm);
      r1 = make_double2(0.5 * (p.y - m.y) * norm, 0.5 * (-p.x + m.x) * norm);
    }
    reinterpret_cast<double2 *>(fk + (size_t)(2 * ky) * nx)[kx] = r0;
    reinterpret_cast<double2 *>(fk + (size_t)(2 * ky + 1) * nx)[kx] = r1;
  }
}
// packed layout -> half spectra (cof_fftw33.f90:211-231) -> inverse column transform
template <int L, int TX, int NT>
__device__ __forceinline__ void cols_inv_body(const double *__restrict__ fk, double2 *__restrict__ out,
                                              const double2 *__restrict__ twy, int H, int bid, int nblk) {
  extern __shared__ double2 lds[];
  constexpr int NTHR = TX * NT, hy = L / 2;
  constexpr bool WAVE = NTHR <= 64;
  const int tid = threadIdx.x, cc = tid % TX, t = tid / TX;
  const int kx = xcd_remap(bid, nblk) * TX + cc;
  const double2 *src = reinterpret_cast<const double2 *>(fk) + kx;
  FftTw<L, NT> T;
  T.load(twy, 1, t);
  fft_io<L, NT, true, TX, WAVE, false>(
      lds + cc, T, t, true,
      [&](int, int, int e) {
        const int ky = e <= hy ? e : L - e;
        if (e == hy) return make_double2(0.0, 0.0);
        const double2 ab = src[(size_t)(2 * ky) * H], cd = src[(size_t)(2 * ky + 1) * H];
        if (e == 0) return ab;
        return e < hy ? make_double2(ab.x - cd.y, cd.x + ab.y) : make_double2(ab.x + cd.y, -cd.x + ab.y);
      },
      [&](int, int, int e, double2 x) { out[(size_t)e * H + kx] = x; });
}
template <int HC, int NTC, int RPBC> struct RowsShape {
  static constexpr int H = HC, NT = NTC, RPB = RPBC, THREADS = NTC * RPBC;
  static constexpr size_t LDS = sizeof(double2) * padlen(HC) * RPBC;
};
template <int LC, int TXC, int NTC> struct ColsShape {
  static constexpr int L = LC, TX = TXC, NT = NTC, THREADS = TXC * NTC;
  static constexpr size_t LDS = sizeof(double2) * padlen(LC) * TXC;
};
template <class S>
__global__ void __launch_bounds__(S::THREADS) k_rows_fwd(const double *__restrict__ f, double2 *__restrict__ out,
                                                         const double2 *__restrict__ twx, int ny) {
  rows_fwd_body<S::H, S::NT, S::RPB>(f, out, twx, ny, blockIdx.x);
}
template <class S>
__global__ void __launch_bounds__(S::THREADS) k_rows_inv(const double2 *__restrict__ in, double *__restrict__ f,
                                                         const double2 *__restrict__ twx, int ny) {
  rows_inv_body<S::H, S::NT, S::RPB>(in, f, twx, ny, blockIdx.x);
}
template <class S>
__global__ void __launch_bounds__(S::THREADS) k_cols_fwd(const double2 *__restrict__ in, double *__restrict__ fk,
                                                         const double2 *__restrict__ twy, int H, double norm) {
  cols_fwd_body<S::L, S::TX, S::NT>(in, fk, twy, H, norm, blockIdx.x, gridDim.x);
}
template <class S>
__global__ void __launch_bounds__(S::THREADS) k_cols_inv(const double *__restrict__ fk, double2 *__restrict__ out,
                                                         const double2 *__restrict__ twy, int H) {
  cols_inv_body<S::L, S::TX, S::NT>(fk, out, twy, H, blockIdx.x, gridDim.x);
}

// A small grid in one workgroup: rows, transposition in LDS, columns.
// THREADS is a multiple of both NTX and NTY, each at most one wave.  f and fk
// may be the same array: all of the input is read before any output is written.
template <int H, int L, int NTX, int NTY, int THREADS>
__device__ __forceinline__ void fwd2d_body(const double *f, double *fk,
                                           const double2 *__restrict__ twx, const double2 *__restrict__ twy,
                                           double norm) {
  extern __shared__ double2 lds[];
  constexpr int PX = padlen(H), PY = padlen(L), GX = THREADS / NTX, GY = THREADS / NTY, hy = L / 2;
  double2 *cols = lds + GX * PX;
  {
    using Out = FftOut<H, NTX>;
    const int g = threadIdx.x / NTX, t = threadIdx.x - g * NTX;
    double2 *xb = lds + g * PX;
    FftTw<H, NTX> T;
    T.load(twx, 2, t);
#pragma unroll
    for (int y0 = 0; y0 < L; y0 += GX) {
      const int y = y0 + g;
      const bool act = L % GX == 0 || y < L;
      const double2 *src = reinterpret_cast<const double2 *>(f) + (size_t)y * H;
      double2 z[Out::N];
      fft_io<H, NTX, false, 1, true, false>(
          xb, T, t, act, [&](int, int, int e) { return src[e]; },
          [&](int i, int r, int, double2 x) { z[i * Out::R + r] = x; });
      grp_sync<true>();
#pragma unroll
      for (int i = 0; i < Out::ITEMS; ++i) {
        if (Out::M % NTX != 0 && t + i * NTX >= Out::M) continue;
#pragma unroll
        for (int r = 0; r < Out::R; ++r) xb[pidx(t + i * NTX + r * Out::M)] = z[i * Out::R + r];
      }
      grp_sync<true>();
      if (act)
#pragma unroll
        for (int i = 0; i < (H + NTX - 1) / NTX; ++i) {
          const int k = t + i * NTX;
          if (H % NTX != 0 && k >= H) continue;
          cols[k * PY + pidx(y)] = r2c_one(xb[pidx(k)], xb[pidx(k == 0 ? 0 : H - k)], twx[k]);
        }
      grp_sync<true>();
    }
  }
  __syncthreads();
  {
    using Out = FftOut<L, NTY>;
    const int g = threadIdx.x / NTY, t = threadIdx.x - g * NTY;
    FftTw<L, NTY> T;
    T.load(twy, 1, t);
#pragma unroll
    for (int k0 = 0; k0 < H; k0 += GY) {
      const int kx = k0 + g;
      const bool act = H % GY == 0 || kx < H;
      double2 *xb = cols + (act ? kx : 0) * PY;
      double2 z[Out::N];
      fft_io<L, NTY, false, 1, true, false>(
          xb, T, t, act, [&](int, int, int e) { return xb[pidx(e)]; },
          [&](int i, int r, int, double2 x) { z[i * Out::R + r] = x; });
      grp_sync<true>();
      if (act)
#pragma unroll
        for (int i = 0; i < Out::ITEMS; ++i) {
          if (Out::M % NTY != 0 && t + i * NTY >= Out::M) continue;
#pragma unroll
          for (int r = 0; r < Out::R; ++r) xb[pidx(t + i * NTY + r * Out::M)] = z[i * Out::R + r];
        }
    }
  }
  __syncthreads();
  for (int e = threadIdx.x; e < hy * H; e += THREADS) {
    const int ky = e / H, kx = e - ky * H;
    const double2 p = cols[kx * PY + pidx(ky)];
    double2 r0, r1;
    if (ky == 0) {
      r0 = make_double2(p.x * norm, p.y * norm);
      r1 = make_double2(0.0, 0.0);
    } else {
      const double2 m = cols[kx * PY + pidx(L - ky)];
      r0 = make_double2(0.5 * (p.x + m.x) * norm, 0.5 * (p.y + m.y) * norm);
      r1 = make_double2(0.5 * (p.y - m.y) * norm, 0.5 * (-p.x + m.x) * norm);
    }
    reinterpret_cast<double2 *>(fk)[(size_t)(2 * ky) * H + kx] = r0;
    reinterpret_cast<double2 *>(fk)[(size_t)(2 * ky + 1) * H + kx] = r1;
  }
}
template <int H, int L, int NTX, int NTY, int THREADS>
__device__ __forceinline__ void inv2d_body(const double *fk, double *f,
                                           const double2 *__restrict__ twx, const double2 *__restrict__ twy) {
  extern __shared__ double2 lds[];
  constexpr int PX = padlen(H), PY = padlen(L), GX = THREADS / NTX, GY = THREADS / NTY, hy = L / 2;
  double2 *rows = lds, *cols = lds + L * PX;
  for (int e = threadIdx.x; e < hy * H; e += THREADS) {
    const int ky = e / H, kx = e - ky * H;
    const double2 ab = reinterpret_cast<const double2 *>(fk)[(size_t)(2 * ky) * H + kx];
    const double2 cd = reinterpret_cast<const double2 *>(fk)[(size_t)(2 * ky + 1) * H + kx];
    double2 *c = cols + kx * PY;
    if (ky == 0) {
      c[0] = ab;
      c[pidx(hy)] = make_double2(0.0, 0.0);
    } else {
      c[pidx(ky)] = make_double2(ab.x - cd.y, cd.x + ab.y);
      c[pidx(L - ky)] = make_double2(ab.x + cd.y, -cd.x + ab.y);
    }
  }
  __syncthreads();
  {
    const int g = threadIdx.x / NTY, t = threadIdx.x - g * NTY;
    FftTw<L, NTY> T;
    T.load(twy, 1, t);
#pragma unroll
    for (int k0 = 0; k0 < H; k0 += GY) {
      const int kx = k0 + g;
      const bool act = H % GY == 0 || kx < H;
      double2 *xb = cols + (act ? kx : 0) * PY;
      fft_io<L, NTY, true, 1, true, false>(
          xb, T, t, act, [&](int, int, int e) { return xb[pidx(e)]; },
          [&](int, int, int e, double2 x) { rows[e * PX + pidx(kx)] = x; });
    }
  }
  __syncthreads();
  {
    const int g = threadIdx.x / NTX, t = threadIdx.x - g * NTX;
    FftTw<H, NTX> T;
    T.load(twx, 2, t);
#pragma unroll
    for (int y0 = 0; y0 < L; y0 += GX) {
      const int y = y0 + g;
      const bool act = L % GX == 0 || y < L;
      double2 *xb = rows + (act ? y : 0) * PX, *dst = reinterpret_cast<double2 *>(f) + (size_t)y * H;
      fft_io<H, NTX, true, 1, true, false>(
          xb, T, t, act,
          [&](int, int, int e) { return c2r_elem(xb[pidx(e)], xb[pidx(e == 0 ? 0 : H - e)], e, cconj(twx[e])); },
          [&](int, int, int e, double2 x) { dst[e] = x; });
    }
  }
}
template <int HC, int LC, int NTXC, int NTYC, int TH> struct SmallShape {
  static constexpr int H = HC, L = LC, NTX = NTXC, NTY = NTYC, THREADS = TH;
  static constexpr size_t LDSF = sizeof(double2) * ((TH / NTXC) * padlen(HC) + HC * padlen(LC));
  static constexpr size_t LDSI = sizeof(double2) * (LC * padlen(HC) + HC * padlen(LC));
};
template <class S>
__global__ void __launch_bounds__(S::THREADS) k_fwd2d(const double *f, double *fk,
                                                      const double2 *__restrict__ twx,
                                                      const double2 *__restrict__ twy, double norm) {
  fwd2d_body<S::H, S::L, S::NTX, S::NTY, S::THREADS>(f, fk, twx, twy, norm);
}
template <class S>
__global__ void __launch_bounds__(S::THREADS) k_inv2d(const double *fk, double *f,
                                                      const double2 *__restrict__ twx,
                                                      const double2 *__restrict__ twy) {
  inv2d_body<S::H, S::L, S::NTX, S::NTY, S::THREADS>(fk, f, twx, twy);
}

}  // namespace fsibe

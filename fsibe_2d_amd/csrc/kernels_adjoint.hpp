// kernels_adjoint.hpp -- the discrete adjoint of the fused fluid step for
// prescribed kinematics (no reference counterpart: the reference has no
// adjoint).  Each kernel is the transpose of one stage of kernels_step.hpp,
// run in reverse order, with the same FFT engine:
//
//   stage (forward)                       adjoint kernel (reverse order)
//   K6 rows  u = V(vortk(n1)), cal_drag   ak_rows_vel:  J-term, V^T rows
//   K5 cols  psi, i ky psi                ak_cols_ab2:  V^T columns, then
//   K4 cols  nlk, AB2 update                            the AB2 and nlk transposes
//   K2 rows  nonlinear + penalisation     ak_rows_nl:   products, masks
//   K1 cols  A, B of vortk(n0)            ak_cols_w0
//   K0 mask  create_mask                  ak_mask:      d(mask)/d(kinematics)
//
// The state of the reverse sweep: lW = dJ/d vortk (half spectrum), lNL =
// dJ/d nlk of the previous step, lu1/lu2 = dJ/du (physical).  Transposes
// over the real inner product of the stored arrays (the real and imaginary
// parts of each stored half-spectrum entry are two coordinates):
//   column inverse DFT (unnormalised)    -> column forward DFT (unnormalised)
//   column forward DFT x norm            -> norm x column inverse DFT
//   row c2r: f = Re X0 + 2 sum_k Re(Xk e^{i th})  -> X0 = R[f]_0, Xk = 2 R[f]_k
//   row r2c (unnormalised) R             -> f = c2r(Y), Y0 = X0, Yk = Xk / 2
//   spectral multiplier m                -> conj(m)
#pragma once
#include "kernels_fused.hpp"
#include "kernels_mask.hpp"
#include "kernels_step.hpp"

namespace fsibe {

// ---- ak_rows_vel (transpose of K6's velocity, plus the objective) ----------
// J = cJ sum_window m (u1 - vx) at this step; lu1 += cJ m on the window;
// lm = cJ (u1 - vx), lvx = -cJ m there (the mask adjoints are assigned here on
// the whole mask box and added to by ak_rows_nl).  Then Ta = R^T[lu1],
// Tb = i kx R^T[lu2] (u1 = R[Cpsiy] + U, u2 = -R[i kx Cpsi] + U).
template <class FX>
__global__ void __launch_bounds__(FX::LB) ak_rows_vel(const double *__restrict__ lu1, const double *__restrict__ lu2,
                                                      const double *__restrict__ u1n, MaskBox mb, Window win,
                                                      double cJ, double *__restrict__ lm, double *__restrict__ lvx,
                                                      double *__restrict__ lvy, double2 *__restrict__ Ta,
                                                      double2 *__restrict__ Tb, FX F,
                                                      const double2 *__restrict__ twx, StepConsts c) {
#pragma clang fp contract(off)
  extern __shared__ double2 lds[];
  const int H = F.H(), nx = 2 * H, tid = threadIdx.x, nt = blockDim.x, PL = padlen(H);
  const int y = blockIdx.x;
  double2 *f0 = lds, *f1 = lds + PL;
  const bool mrow = mb.x1 >= mb.x0 && y >= mb.y0 && y <= mb.y1;
  const bool wrow = y >= win.y0 && y <= win.y1;
  for (int n = tid; n < H; n += nt) {
    double2 a = reinterpret_cast<const double2 *>(lu1 + (size_t)y * nx)[n];
    const double2 b = reinterpret_cast<const double2 *>(lu2 + (size_t)y * nx)[n];
    if (mrow) {
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int x = 2 * n + h;
        if (!mb.inside(x, y)) continue;
        const size_t qq = (size_t)(y - mb.y0) * mb.w + (x - mb.x0);
        double gm = 0.0, gvx = 0.0;
        if (wrow && x >= win.x0 && x <= win.x1) {
          const double m = mb.m[qq];
          const double uu = h ? reinterpret_cast<const double2 *>(u1n + (size_t)y * nx)[n].y
                              : reinterpret_cast<const double2 *>(u1n + (size_t)y * nx)[n].x;
          gm = cJ * (uu - mb.vx[qq]);
          gvx = -(cJ * m);
          if (h) a.y += cJ * m; else a.x += cJ * m;
        }
        lm[qq] = gm;
        lvx[qq] = gvx;
        lvy[qq] = 0.0;
      }
    }
    f0[pidx(n)] = a;
    f1[pidx(n)] = b;
  }
  __syncthreads();
  F.template fft<false, 2>(lds, twx, tid, nt);
  rows_r2c_post(lds, 2, H, PL, twx, tid, nt);
  for (int k = tid; k < H; k += nt) {
    const double wk = k == 0 ? 1.0 : 2.0;
    const double2 xa = f0[pidx(k)], xb = f1[pidx(k)];
    const double kf = (double)k * c.sx;
    Ta[(size_t)y * H + k] = make_double2(wk * xa.x, wk * xa.y);
    // i kx (wk xb)
    Tb[(size_t)y * H + k] = make_double2(-(kf * (wk * xb.y)), kf * (wk * xb.x));
  }
}

// ---- ak_cols_ab2 (transposes of K5's psi columns, K4's AB2 and nlk) ---------
// lW holds dJ/d vortk(n1) from the later steps; on return it holds the part
// of dJ/d vortk(n0) that passes through the AB2 update, lNL the part of
// dJ/d nlk(n-1), and Tc, Td the row-pass adjoints of Rc, Rpx.
template <class FY>
__global__ void __launch_bounds__(FY::LB) ak_cols_ab2(const double2 *__restrict__ Ta, const double2 *__restrict__ Tb,
                                                      double2 *__restrict__ lW, double2 *__restrict__ lNL,
                                                      double2 *__restrict__ Tc, double2 *__restrict__ Td,
                                                      const DevScalars *__restrict__ st, int explicit_step, FY F,
                                                      const double2 *__restrict__ twy, StepConsts c) {
#pragma clang fp contract(off)
  extern __shared__ double2 lds[];
  const int ny = F.NY(), TX = F.tx(), H = c.H, tid = threadIdx.x, nt = blockDim.x;
  const int kx0 = xcd_remap(blockIdx.x, gridDim.x) * TX;
  const int TT = 2 * TX;
  for (int e = tid; e < ny * TX; e += nt) {
    const int y = e / TX, cc = e - y * TX;
    lds[pidx(y) * TT + cc] = Ta[(size_t)y * H + kx0 + cc];
    lds[pidx(y) * TT + TX + cc] = Tb[(size_t)y * H + kx0 + cc];
  }
  __syncthreads();
  F.template fft<false, 2, 2>(lds, twy, tid, nt);
  const DevScalars s = *st;
  const int hy = ny >> 1;
  for (int e = tid; e < ny * TX; e += nt) {
    const int idx = e / TX, cc = e - idx * TX, kx = kx0 + cc;
    const size_t g = (size_t)idx * H + kx;
    double2 lnl = make_double2(0.0, 0.0), lw0 = make_double2(0.0, 0.0), lnl1 = make_double2(0.0, 0.0);
    if (idx != hy) {
      const int ky = ky_signed(idx, ny);
      const int aky = ky < 0 ? -ky : ky;
      const double kyf = (double)ky * c.sy;
      const double2 ya = lds[pidx(idx) * TT + cc], yb = lds[pidx(idx) * TT + TX + cc];
      // d psi = -i ky Ya + Yb, then the Poisson factor (psi = W1 / |k|^2)
      double2 lpsi = make_double2(kyf * ya.y + yb.x, -(kyf * ya.x) + yb.y);
      double2 lw1 = lW[g];
      if (!(kx == 0 && ky == 0)) {
        const double quot = ((double)(kx * kx) * c.scalex + (double)(aky * aky) * c.scaley);
        lw1.x += lpsi.x / quot;
        lw1.y += lpsi.y / quot;
      }
      const double kx2 = (double)(kx * kx), ky2 = (double)(aky * aky);
      const double v1 = exp(s.cx1 * kx2 + s.cy1 * ky2);
      const double d = dealias(c, kx, aky);
      const double f = v1 * d;
      const double2 ln0 = lNL[g];
      lw0 = make_double2(f * lw1.x, f * lw1.y);
      lnl = make_double2(s.b10 * lw0.x + ln0.x, s.b10 * lw0.y + ln0.y);
      if (!explicit_step) {
        const double v0 = exp(s.cx0 * kx2 + s.cy0 * ky2);
        lnl1 = make_double2(s.b11 * v0 * lw0.x, s.b11 * v0 * lw0.y);
      }
    }
    lW[g] = lw0;
    lNL[g] = lnl1;
    // nl = norm Cfwd(Rc) - i ky norm Cfwd(Rpx):  dRc = norm Cinv(lnl), dRpx = norm Cinv(i ky lnl)
    const double kyf = (double)ky_signed(idx, ny) * c.sy;
    lds[pidx(idx) * TT + cc] = make_double2(c.norm * lnl.x, c.norm * lnl.y);
    lds[pidx(idx) * TT + TX + cc] = make_double2(c.norm * (-(kyf * lnl.y)), c.norm * (kyf * lnl.x));
  }
  __syncthreads();
  F.template fft<true, 2, 2>(lds, twy, tid, nt);
  for (int e = tid; e < ny * TX; e += nt) {
    const int y = e / TX, cc = e - y * TX;
    Tc[(size_t)y * H + kx0 + cc] = lds[pidx(y) * TT + cc];
    Td[(size_t)y * H + kx0 + cc] = lds[pidx(y) * TT + TX + cc];
  }
}

// ---- ak_rows_nl (transpose of K2) -------------------------------------------
// Forward values omega, omega_y, omega_x (c2r of A, B, i kx A) and the
// adjoints of the products lr, lpy, lpx (Rc = R[r] + i kx R[py], Rpx =
// R[px]) in one six-sequence transform; then the product rule, and the
// weighted r2c of l(omega), l(omega_x), l(omega_y):  Te = dA, Tf = dB.
// lu1, lu2 (dJ/du of this step's velocity) are assigned; the mask adjoints
// lm, lvx, lvy are added to.
template <class FX>
__global__ void __launch_bounds__(FX::LB) ak_rows_nl(const double2 *__restrict__ Tc, const double2 *__restrict__ Td,
                                                     const double2 *__restrict__ A, const double2 *__restrict__ B,
                                                     const double *__restrict__ u1, const double *__restrict__ u2,
                                                     const double *__restrict__ ms, MaskBox mb, int penal_on,
                                                     double *__restrict__ lu1, double *__restrict__ lu2,
                                                     double *__restrict__ lm, double *__restrict__ lvx,
                                                     double *__restrict__ lvy, double2 *__restrict__ Te,
                                                     double2 *__restrict__ Tf, FX F, const double2 *__restrict__ twx,
                                                     StepConsts c) {
#pragma clang fp contract(off)
  extern __shared__ double2 lds[];
  const int H = F.H(), nx = 2 * H, tid = threadIdx.x, nt = blockDim.x, PL = padlen(H);
  const int y = blockIdx.x;
  double2 *f0 = lds, *f1 = lds + PL, *f2 = lds + 2 * PL;
  double2 *g0 = lds + 3 * PL, *g1 = lds + 4 * PL, *g2 = lds + 5 * PL;
  for (int k = tid; k < H; k += nt) {
    const double2 a = live(A + (size_t)y * H, k, H, c.kc);
    const double kf = (double)k * c.sx;
    const int q = pidx(k);
    f0[q] = a;
    f1[q] = live(B + (size_t)y * H, k, H, c.kc);
    f2[q] = make_double2(-kf * a.y, kf * a.x);
    // transposes of the unnormalised r2c: Y0 = X0, Yk = Xk / 2 (k >= 1)
    const double hk = k == 0 ? 1.0 : 0.5;
    const double2 tc = Tc[(size_t)y * H + k], td = Td[(size_t)y * H + k];
    g0[q] = make_double2(hk * tc.x, hk * tc.y);                   // l(r)
    g1[q] = make_double2(hk * (kf * tc.y), hk * (-(kf * tc.x)));  // l(py) = -i kx Tc
    g2[q] = make_double2(hk * td.x, hk * td.y);                   // l(px)
  }
  __syncthreads();
  rows_c2r_pre(lds, 6, H, PL, twx, tid, nt);
  F.template fft<true, 6>(lds, twx, tid, nt);
  const bool prow = penal_on && mb.x1 >= mb.x0 && y >= mb.y0 && y <= mb.y1;
  for (int n = tid; n < H; n += nt) {
    const int q = pidx(n);
    const double2 w = f0[q], wy = f1[q], wx = f2[q];
    const double2 lr = g0[q], lpy = g1[q], lpx = g2[q];
    const double2 a1 = reinterpret_cast<const double2 *>(u1 + (size_t)y * nx)[n];
    const double2 a2 = reinterpret_cast<const double2 *>(u2 + (size_t)y * nx)[n];
    double2 s = make_double2(0.0, 0.0);
    if (ms) s = reinterpret_cast<const double2 *>(ms + (size_t)y * nx)[n];
    // r = -u1 wx - u2 wy - s w
    double2 lu1v = make_double2(-(wx.x * lr.x), -(wx.y * lr.y));
    double2 lu2v = make_double2(-(wy.x * lr.x), -(wy.y * lr.y));
    const double2 lw = make_double2(-(s.x * lr.x), -(s.y * lr.y));
    const double2 lwx = make_double2(-(a1.x * lr.x), -(a1.y * lr.y));
    const double2 lwy = make_double2(-(a2.x * lr.x), -(a2.y * lr.y));
    if (prow) {
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int x = 2 * n + h;
        if (!mb.inside(x, y)) continue;
        const size_t qq = (size_t)(y - mb.y0) * mb.w + (x - mb.x0);
        const double m = mb.m[qq], vx = mb.vx[qq], vy = mb.vy[qq];
        const double uu1 = h ? a1.y : a1.x, uu2 = h ? a2.y : a2.x;
        const double gpx = h ? lpx.y : lpx.x, gpy = h ? lpy.y : lpy.x;
        // px = -m (u1 - vx), py = -m (u2 - vy)
        if (h) { lu1v.y += -(m * gpx); lu2v.y += -(m * gpy); }
        else { lu1v.x += -(m * gpx); lu2v.x += -(m * gpy); }
        lvx[qq] += m * gpx;
        lvy[qq] += m * gpy;
        lm[qq] += -((uu1 - vx) * gpx) - (uu2 - vy) * gpy;
      }
    }
    reinterpret_cast<double2 *>(lu1 + (size_t)y * nx)[n] = lu1v;
    reinterpret_cast<double2 *>(lu2 + (size_t)y * nx)[n] = lu2v;
    g0[q] = lw;
    g1[q] = lwy;
    g2[q] = lwx;
  }
  __syncthreads();
  // weighted r2c (transpose of c2r) of l(omega), l(omega_y), l(omega_x)
  F.template fft<false, 3>(g0, twx, tid, nt);
  rows_r2c_post(g0, 3, H, PL, twx, tid, nt);
  for (int k = tid; k < H; k += nt) {
    const int q = pidx(k);
    const double wk = k == 0 ? 1.0 : 2.0;
    const double kf = (double)k * c.sx;
    const double2 xw = g0[q], xwy = g1[q], xwx = g2[q];
    // dA = R^T l(w) + conj(i kx) R^T l(wx), dB = R^T l(wy)
    Te[(size_t)y * H + k] = make_double2(wk * (xw.x + kf * xwx.y), wk * (xw.y - kf * xwx.x));
    Tf[(size_t)y * H + k] = make_double2(wk * xwy.x, wk * xwy.y);
  }
}

// ---- ak_cols_w0 (transpose of K1) -------------------------------------------
// lW += Cfwd(Te) - i ky Cfwd(Tf)  (A = Cinv(W0), B = Cinv(i ky W0))
template <class FY>
__global__ void __launch_bounds__(FY::LB) ak_cols_w0(const double2 *__restrict__ Te, const double2 *__restrict__ Tf,
                                                     double2 *__restrict__ lW, FY F,
                                                     const double2 *__restrict__ twy, StepConsts c) {
#pragma clang fp contract(off)
  extern __shared__ double2 lds[];
  const int ny = F.NY(), TX = F.tx(), H = c.H, tid = threadIdx.x, nt = blockDim.x;
  const int kx0 = xcd_remap(blockIdx.x, gridDim.x) * TX;
  const int TT = 2 * TX;
  for (int e = tid; e < ny * TX; e += nt) {
    const int y = e / TX, cc = e - y * TX;
    lds[pidx(y) * TT + cc] = Te[(size_t)y * H + kx0 + cc];
    lds[pidx(y) * TT + TX + cc] = Tf[(size_t)y * H + kx0 + cc];
  }
  __syncthreads();
  F.template fft<false, 2, 2>(lds, twy, tid, nt);
  const int hy = ny >> 1;
  for (int e = tid; e < ny * TX; e += nt) {
    const int idx = e / TX, cc = e - idx * TX, kx = kx0 + cc;
    const size_t g = (size_t)idx * H + kx;
    if (idx == hy) {
      lW[g] = make_double2(0.0, 0.0);
      continue;
    }
    const double kyf = (double)ky_signed(idx, ny) * c.sy;
    const double2 ye = lds[pidx(idx) * TT + cc], yf = lds[pidx(idx) * TT + TX + cc];
    const double2 l = lW[g];
    lW[g] = make_double2(l.x + (ye.x + kyf * yf.y), l.y + (ye.y - kyf * yf.x));
  }
}

// ---- the reverse step in two kernels ----------------------------------------
// Where the grid has the shapes: one row kernel takes ak_rows_nl of step j
// and ak_rows_vel of step j-1 (dJ/du passes in registers and LDS), one column
// kernel ak_cols_w0 of step j and ak_cols_ab2 of step j-1 (lW is read and
// written once).  Either half may be absent: the last step of a unit starts
// with the second halves alone, the first one ends with the first halves.
// Both are bound by the latency of their chains of transforms at 512^2: the
// four kernels took 12.8 + 8.5 and 6.9 + 14.0 us there, these two 16.9 and 12.8.
struct AdjRowArgs {
  // ak_rows_nl (Te null: absent)
  const double2 *Tc, *Td, *A, *B;
  const double *u1, *u2, *ms;
  MaskBox mb;
  int penal_on;
  double *lm, *lvx, *lvy;
  double2 *Te, *Tf;
  // dJ/du: written by the first half without the second, read by the second
  // without the first
  double *lu1, *lu2;
  // ak_rows_vel (Ta null: absent)
  const double *u1n;
  MaskBox mbv;
  Window win;
  double cJ;
  double *lmv, *lvxv, *lvyv;
  double2 *Ta, *Tb;
  // columns of the adjoint fields in use: dJ/d vortk of a mode that dealiasing
  // removes is multiplied by zero in the update before, so none is formed
  // for the columns beyond (H where one of the two kernels is not the fused one)
  int kl;
  StepConsts c;  // kc: of A, B
};

// one row by six slots of NT threads: the six inverse transforms, then the
// forward ones of dJ/du (slots 0, 1) and of l(omega), l(omega_y), l(omega_x)
template <int H, int NT>
__device__ __forceinline__ void adj_row_body(const AdjRowArgs &a, const double2 *__restrict__ twx, int y) {
#pragma clang fp contract(off)
  extern __shared__ double2 lds[];
  constexpr int PL = padlen(H), nx = 2 * H, NR = 6 * NT, PN = (H + NR - 1) / NR;
  constexpr bool WAVE = NR <= 64;
  using Out = FftOut<H, NT>;
  const int p = threadIdx.x, slot = p / NT, t = p - slot * NT;
  double2 *xb = lds + slot * PL;
  const size_t rowk = (size_t)y * H, rowx = (size_t)y * nx;
  const double sx = a.c.sx;
  const bool nl = a.Te != nullptr, vel = a.Ta != nullptr;
  FftTw<H, NT> T;
  T.load(twx, 2, t);
  double2 z[Out::N];
  auto put = [&]() {
#pragma unroll
    for (int i = 0; i < Out::ITEMS; ++i) {
      if (Out::M % NT != 0 && t + i * NT >= Out::M) continue;
#pragma unroll
      for (int r = 0; r < Out::R; ++r) xb[pidx(t + i * NT + r * Out::M)] = z[i * Out::R + r];
    }
  };
  if (nl) {
    const double2 *pA = a.A, *pB = a.B, *pC = a.Tc, *pD = a.Td;
    const double2 *src = (slot == 0 || slot == 2 ? pA : slot == 1 ? pB : slot == 5 ? pD : pC) + rowk;
    const int kc = slot < 3 ? a.c.kc : a.kl;
    auto at = [&](int k) {
      const double2 v = live(src, k, H, kc);
      const double kf = (double)k * sx;
      if (slot < 2) return v;
      if (slot == 2) return make_double2(-kf * v.y, kf * v.x);
      // transposes of the unnormalised r2c: Y0 = X0, Yk = Xk / 2 (k >= 1)
      const double hk = k == 0 ? 1.0 : 0.5;
      if (slot == 4) return make_double2(hk * (kf * v.y), hk * (-(kf * v.x)));
      return make_double2(hk * v.x, hk * v.y);
    };
    fft_io<H, NT, true, 1, WAVE, false>(
        xb, T, t, true,
        [&](int, int, int e) { return c2r_elem(at(e), at(e == 0 ? 0 : H - e), e, cconj(twx[e])); },
        [&](int i, int r, int, double2 x) { z[i * Out::R + r] = x; });
    grp_sync<WAVE>();
    put();
    grp_sync<WAVE>();
  }
  const MaskBox mb = a.mb, mbv = a.mbv;
  const bool prow = nl && a.penal_on && mb.x1 >= mb.x0 && y >= mb.y0 && y <= mb.y1;
  const bool mrow = vel && mbv.x1 >= mbv.x0 && y >= mbv.y0 && y <= mbv.y1;
  const bool wrow = y >= a.win.y0 && y <= a.win.y1;
#pragma unroll
  for (int k = 0; k < PN; ++k) {
    const int n = p + k * NR;
    if (H % NR != 0 && n >= H) continue;
    const int q = pidx(n);
    double2 lu1v, lu2v;
    if (nl) {
      const double2 w = lds[q], wy = lds[PL + q], wx = lds[2 * PL + q];
      const double2 lr = lds[3 * PL + q], lpy = lds[4 * PL + q], lpx = lds[5 * PL + q];
      const double2 a1 = reinterpret_cast<const double2 *>(a.u1 + rowx)[n];
      const double2 a2 = reinterpret_cast<const double2 *>(a.u2 + rowx)[n];
      double2 s = make_double2(0.0, 0.0);
      if (a.ms) s = reinterpret_cast<const double2 *>(a.ms + rowx)[n];
      (void)w;
      // r = -u1 wx - u2 wy - s w
      lu1v = make_double2(-(wx.x * lr.x), -(wx.y * lr.y));
      lu2v = make_double2(-(wy.x * lr.x), -(wy.y * lr.y));
      if (prow) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const int x = 2 * n + h;
          if (!mb.inside(x, y)) continue;
          const size_t qq = (size_t)(y - mb.y0) * mb.w + (x - mb.x0);
          const double m = mb.m[qq], vx = mb.vx[qq], vy = mb.vy[qq];
          const double uu1 = h ? a1.y : a1.x, uu2 = h ? a2.y : a2.x;
          const double gpx = h ? lpx.y : lpx.x, gpy = h ? lpy.y : lpy.x;
          // px = -m (u1 - vx), py = -m (u2 - vy)
          if (h) { lu1v.y += -(m * gpx); lu2v.y += -(m * gpy); }
          else { lu1v.x += -(m * gpx); lu2v.x += -(m * gpy); }
          a.lvx[qq] += m * gpx;
          a.lvy[qq] += m * gpy;
          a.lm[qq] += -((uu1 - vx) * gpx) - (uu2 - vy) * gpy;
        }
      }
      lds[3 * PL + q] = make_double2(-(s.x * lr.x), -(s.y * lr.y));
      lds[4 * PL + q] = make_double2(-(a2.x * lr.x), -(a2.y * lr.y));
      lds[5 * PL + q] = make_double2(-(a1.x * lr.x), -(a1.y * lr.y));
      if (!vel) {
        reinterpret_cast<double2 *>(a.lu1 + rowx)[n] = lu1v;
        reinterpret_cast<double2 *>(a.lu2 + rowx)[n] = lu2v;
      }
    } else {
      lu1v = reinterpret_cast<const double2 *>(a.lu1 + rowx)[n];
      lu2v = reinterpret_cast<const double2 *>(a.lu2 + rowx)[n];
    }
    if (vel) {
      if (mrow) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const int x = 2 * n + h;
          if (!mbv.inside(x, y)) continue;
          const size_t qq = (size_t)(y - mbv.y0) * mbv.w + (x - mbv.x0);
          double gm = 0.0, gvx = 0.0;
          if (wrow && x >= a.win.x0 && x <= a.win.x1) {
            const double m = mbv.m[qq], uu = a.u1n[rowx + x];
            gm = a.cJ * (uu - mbv.vx[qq]);
            gvx = -(a.cJ * m);
            if (h) lu1v.y += a.cJ * m; else lu1v.x += a.cJ * m;
          }
          a.lmv[qq] = gm;
          a.lvxv[qq] = gvx;
          a.lvyv[qq] = 0.0;
        }
      }
      lds[q] = lu1v;
      lds[PL + q] = lu2v;
    }
  }
  grp_sync<WAVE>();
  const bool act = slot < 2 ? vel : slot > 2 && nl;
  fft_io<H, NT, false, 1, WAVE, false>(
      xb, T, t, act, [&](int, int, int e) { return xb[pidx(e)]; },
      [&](int i, int r, int, double2 x) { z[i * Out::R + r] = x; });
  grp_sync<WAVE>();
  if (act) put();
  grp_sync<WAVE>();
#pragma unroll
  for (int i = 0; i < PN; ++i) {
    const int k = p + i * NR;
    if ((H % NR != 0 && k >= H) || k >= a.kl) continue;
    const int q = pidx(k), qm = pidx(k == 0 ? 0 : H - k);
    const double wk = k == 0 ? 1.0 : 2.0, kf = (double)k * sx;
    const double2 tw = twx[k];
    if (vel) {
      const double2 xa = r2c_one(lds[q], lds[qm], tw), xb2 = r2c_one(lds[PL + q], lds[PL + qm], tw);
      a.Ta[rowk + k] = make_double2(wk * xa.x, wk * xa.y);
      // i kx (wk xb)
      a.Tb[rowk + k] = make_double2(-(kf * (wk * xb2.y)), kf * (wk * xb2.x));
    }
    if (nl) {
      const double2 xw = r2c_one(lds[3 * PL + q], lds[3 * PL + qm], tw);
      const double2 xwy = r2c_one(lds[4 * PL + q], lds[4 * PL + qm], tw);
      const double2 xwx = r2c_one(lds[5 * PL + q], lds[5 * PL + qm], tw);
      // dA = R^T l(w) + conj(i kx) R^T l(wx), dB = R^T l(wy)
      a.Te[rowk + k] = make_double2(wk * (xw.x + kf * xwx.y), wk * (xw.y - kf * xwx.x));
      a.Tf[rowk + k] = make_double2(wk * xwy.x, wk * xwy.y);
    }
  }
}
template <int HC, int NTC> struct AdjRowShape {
  static constexpr int H = HC, NT = NTC, THREADS = 6 * NTC;
  static constexpr size_t LDS = sizeof(double2) * 6 * padlen(H);
};
template <class S>
__global__ void __launch_bounds__(S::THREADS) ak_row_step(AdjRowArgs a, const double2 *__restrict__ twx) {
  adj_row_body<S::H, S::NT>(a, twx, blockIdx.x);
}

struct AdjColArgs {
  const double2 *Te, *Tf;  // ak_cols_w0 (Te null: absent)
  const double2 *Ta, *Tb;  // ak_cols_ab2 (Ta null: absent)
  double2 *lW, *lNL, *Tc, *Td;
  const DevScalars *s;
  int explicit_step;
  StepConsts c;
};

// one column (of the kl in use) by four slots of NT threads: the four forward transforms, the
// spectral transposes, two inverse transforms
template <int L, int NT>
__device__ __forceinline__ void adj_col_body(const AdjColArgs &a, const double2 *__restrict__ twy, int bid, int nblk) {
#pragma clang fp contract(off)
  extern __shared__ double2 lds[];
  constexpr int PL = padlen(L), NTHR = 4 * NT, EL = (L + NTHR - 1) / NTHR;
  constexpr bool WAVE = NTHR <= 64;
  using Out = FftOut<L, NT>;
  const StepConsts &c = a.c;
  const int tid = threadIdx.x, H = c.H, slot = tid / NT, t = tid - slot * NT;
  const int kx = xcd_remap(bid, nblk);
  double2 *xb = lds + slot * PL;
  const bool w0 = a.Te != nullptr, ab2 = a.Ta != nullptr;
  FftTw<L, NT> T;
  T.load(twy, 1, t);
  double cx1 = 0.0, cy1 = 0.0, cx0 = 0.0, cy0 = 0.0, b10 = 0.0, b11 = 0.0;
  if (ab2) { cx1 = a.s->cx1; cy1 = a.s->cy1; cx0 = a.s->cx0; cy0 = a.s->cy0; b10 = a.s->b10; b11 = a.s->b11; }
  double2 lw[EL], ln[EL];
  double dl[EL];
  const double kx2 = (double)(kx * kx);
#pragma unroll
  for (int q = 0; q < EL; ++q) {
    const int idx = tid + q * NTHR;
    lw[q] = ln[q] = make_double2(0.0, 0.0);
    dl[q] = dealias_fast(c, kx, abs(ky_signed(idx, L)));  // 0: both are zero
    if (L % NTHR == 0 || idx < L) {
      const size_t g = (size_t)(dl[q] != 0.0 ? idx : 0) * H + kx;
      const double2 w = a.lW[g], n = a.lNL[g];
      if (dl[q] != 0.0) {
        lw[q] = w;
        if (ab2) ln[q] = n;
      }
    }
  }
  {
    double2 z[Out::N];
    const double2 *pe = a.Te, *pf = a.Tf, *pa = a.Ta, *pb = a.Tb;
    const double2 *src = slot == 0 ? pe : slot == 1 ? pf : slot == 2 ? pa : pb;
    const bool act = src != nullptr;
    fft_io<L, NT, false, 1, WAVE, false>(
        xb, T, t, act, [&](int, int, int e) { return src[(size_t)e * H + kx]; },
        [&](int i, int r, int, double2 x) { z[i * Out::R + r] = x; });
    grp_sync<WAVE>();
    if (act) {
#pragma unroll
      for (int i = 0; i < Out::ITEMS; ++i) {
        if (Out::M % NT != 0 && t + i * NT >= Out::M) continue;
#pragma unroll
        for (int r = 0; r < Out::R; ++r) xb[pidx(t + i * NT + r * Out::M)] = z[i * Out::R + r];
      }
    }
    grp_sync<WAVE>();
  }
  const bool same = cx0 == cx1 && cy0 == cy1;
#pragma unroll
  for (int q = 0; q < EL; ++q) {
    const int idx = tid + q * NTHR;
    if (L % NTHR != 0 && idx >= L) continue;
    const size_t g = (size_t)idx * H + kx;
    const int ky = ky_signed(idx, L), aky = ky < 0 ? -ky : ky;
    const double kyf = (double)ky * c.sy, ky2 = (double)(aky * aky);
    double2 *l0 = lds + pidx(idx);
    double2 l = lw[q];
    if (w0) {
      const double2 ye = l0[0], yf = l0[PL];
      l = idx == L / 2 ? make_double2(0.0, 0.0)
                       : make_double2(l.x + (ye.x + kyf * yf.y), l.y + (ye.y - kyf * yf.x));
    }
    if (!ab2) {
      a.lW[g] = l;
      continue;
    }
    double2 lnl = make_double2(0.0, 0.0), lw0 = lnl, lnl1 = lnl;
    if (idx != L / 2) {
      const double2 ya = l0[2 * PL], yb = l0[3 * PL];
      // d psi = -i ky Ya + Yb, then the Poisson factor (psi = W1 / |k|^2)
      const double2 lpsi = make_double2(kyf * ya.y + yb.x, -(kyf * ya.x) + yb.y);
      if (!(kx == 0 && ky == 0)) {
        const double quot = (kx2 * c.scalex + ky2 * c.scaley), rq = 1.0 / quot;
        const double2 d = div_by(lpsi, quot, rq);
        l.x += d.x;
        l.y += d.y;
      }
      const double v1 = exp(cx1 * kx2 + cy1 * ky2);
      const double f = v1 * dl[q];
      lw0 = make_double2(f * l.x, f * l.y);
      lnl = make_double2(b10 * lw0.x + ln[q].x, b10 * lw0.y + ln[q].y);
      if (!a.explicit_step) {
        const double v0 = same ? v1 : exp(cx0 * kx2 + cy0 * ky2);
        lnl1 = make_double2(b11 * v0 * lw0.x, b11 * v0 * lw0.y);
      }
    }
    a.lW[g] = lw0;
    a.lNL[g] = lnl1;
    // nl = norm Cfwd(Rc) - i ky norm Cfwd(Rpx):  dRc = norm Cinv(lnl), dRpx = norm Cinv(i ky lnl)
    l0[0] = make_double2(c.norm * lnl.x, c.norm * lnl.y);
    l0[PL] = make_double2(c.norm * (-(kyf * lnl.y)), c.norm * (kyf * lnl.x));
  }
  if (!ab2) return;
  grp_sync<WAVE>();
  double2 *oc = a.Tc, *od = a.Td;
  double2 *out = slot == 0 ? oc : od;
  fft_io<L, NT, true, 1, WAVE, false>(
      xb, T, t, slot < 2, [&](int, int, int e) { return xb[pidx(e)]; },
      [&](int, int, int e, double2 x) { out[(size_t)e * H + kx] = x; });
}
template <int LC, int NTC> struct AdjColShape {
  static constexpr int L = LC, NT = NTC, THREADS = 4 * NTC;
  static constexpr size_t LDS = sizeof(double2) * 4 * padlen(L);
};
template <class S>
__global__ void __launch_bounds__(S::THREADS) ak_col_step(AdjColArgs a, const double2 *__restrict__ twy) {
  adj_col_body<S::L, S::NT>(a, twy, blockIdx.x, gridDim.x);
}

// ---- ak_mask: d(mask)/d(kinematics) of a rigid beam -------------------------
// For prescribed motion with theta = 0 the beam is the straight line from
// the leading edge LE = (x0, LEy) at angle alpha; node i sits at
// LE + s_i t (t = (cos a, sin a)), with velocity (-at s_i sin a,
// hdot + at s_i cos a).  The pixel's value came from primitive `win`
// (create_mask's drawing order: segments 0..ns-2, hinges 1..ns-2, the
// leading-edge dot, the trailing-edge dot, after `off` fixed primitives).
// Sums over the tile of lm d(m)/dq + lvx d(vx)/dq + lvy d(vy)/dq for
// q = (LEy, alpha, hdot, alpha_t); one record of 4 partial sums per tile.
struct RigidBeam {
  double LEx, LEy, alpha, hdot, at;
  const double *s;  // s_i of the nodes (integrate_position's sums)
  int ns, off;
};

__device__ __forceinline__ double smooth_step_d(const MaskConsts &c, double x, double t) {
#pragma clang fp contract(off)
  if (c.sharp) return 0.0;
  const double delta = c.h * c.gerf;
  const double a = (x + t) / delta, b = (t - x) / delta;
  return (exp(-(a * a)) - exp(-(b * b))) / (delta * sqrt(c.pi));
}

__global__ void __launch_bounds__(256) ak_mask(const int *__restrict__ win, const double *__restrict__ lm,
                                               const double *__restrict__ lvx, const double *__restrict__ lvy,
                                               MaskConsts c, RigidBeam rb, int bx0, int by0, int bw, int bh,
                                               double *__restrict__ part) {
#pragma clang fp contract(off)
  __shared__ double red[4 * 4];
  const int npx = bw * bh;
  const double ca = cos(rb.alpha), sa = sin(rb.alpha);
  double g[4] = {0.0, 0.0, 0.0, 0.0};
  for (int q = blockIdx.x * blockDim.x + threadIdx.x; q < npx; q += gridDim.x * blockDim.x) {
    const int p = win[q];
    if (p < rb.off) continue;
    const int ly = q / bw, lx = q - ly * bw;
    const double x = (double)(bx0 + lx) * c.dx, y = (double)(by0 + ly) * c.dy;
    const double rx = x - rb.LEx, ry = y - rb.LEy;
    const double xi = ca * rx + sa * ry;    // along the beam
    const double d = -(sa * rx) + ca * ry;  // across the beam
    const double gm = lm[q] / c.eps, gvx = lvx[q], gvy = lvy[q];
    const int k = p - rb.off, ns = rb.ns;
    if (k <= ns - 2) {
      // segment: m = SS(|d|), (vx, vy) = v(xi)
      const double ad = fabs(d), sg = d < 0.0 ? -1.0 : 1.0;
      const double dv = smooth_step_d(c, ad, c.t) * sg;
      g[0] += gm * dv * (-ca) + gvx * (rb.at * sa * sa) + gvy * (-(rb.at * ca * sa));
      g[1] += gm * dv * (-xi) + gvx * (-(rb.at * (ca * xi + sa * d))) + gvy * (rb.at * (ca * d - sa * xi));
      g[2] += gvy;
      g[3] += gvx * (-(sa * xi)) + gvy * (ca * xi);
    } else {
      // hinge (node k - ns + 2) or dot (leading / trailing edge): m = SS(R)
      int node;
      if (k <= 2 * ns - 4) node = k - (ns - 1) + 1;
      else if (k == 2 * ns - 3) node = 0;
      else node = ns - 1;
      const double si = rb.s[node];
      const double px = rb.LEx + si * ca, py = rb.LEy + si * sa;
      const double ex = x - px, ey = y - py;
      const double R = sqrt(ex * ex + ey * ey);
      if (R > 0.0) {
        const double dv = smooth_step_d(c, R, c.t);
        // dR/dLEy = -ey / R, dR/dalpha = -(e . s_i n) / R with n = (-sa, ca)
        g[0] += gm * dv * (-ey / R);
        g[1] += gm * dv * (-(si * (-(sa * ex) + ca * ey)) / R);
      }
      g[1] += gvx * (-(rb.at * si * ca)) + gvy * (-(rb.at * si * sa));
      g[2] += gvy;
      g[3] += gvx * (-(si * sa)) + gvy * (si * ca);
    }
  }
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
#pragma unroll
  for (int i = 0; i < 4; ++i) g[i] = wave_sum(g[i]);
  if (lane == 0)
#pragma unroll
    for (int i = 0; i < 4; ++i) red[i * 4 + wid] = g[i];
  __syncthreads();
  if (threadIdx.x < 4) {
    const int i = threadIdx.x;
    part[(size_t)blockIdx.x * 4 + i] = ((red[i * 4] + red[i * 4 + 1]) + red[i * 4 + 2]) + red[i * 4 + 3];
  }
}

// device-to-device copies of n doubles (checkpoints, a tape's first velocity and scalars)
__global__ void ak_copy_d(const double *__restrict__ src, double *__restrict__ dst, long long n) {
  for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x)
    dst[i] = src[i];
}
__global__ void ak_zero(double *__restrict__ dst, long long n) {
  for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x)
    dst[i] = 0.0;
}

}  // namespace fsibe

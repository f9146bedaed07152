// kernels_fused.hpp -- the step's column and row stages fused across the
// boundaries of the kernels in kernels_step.hpp, on a transform that takes
// its input from and hands its output to the caller's registers.
//
//   column stage  K4 + K5 (+ the dw/dy column of the next step's K1):
//                 Rc, Rpx -> nlk, AB2 update -> omega, psi, i ky psi,
//                 -ky^2 psi (box rows), i ky omega, one read of the inputs
//   row stage     K6 + the convective part of the next step's K2: omega, u,
//                 diagnostics, pressure right-hand sides, and -u.grad(omega)
//                 - chi_s omega of the state just formed
//
// Every transform runs the radix passes of kernels_step.hpp's instances with
// the same twiddles (cp_radix, twiddle powers by binary splitting) and every
// elementwise formula is the same, so the fields are theirs bit for bit.
#pragma once
#include "kernels_step.hpp"

namespace fsibe {

// Orders the LDS accesses of the threads that share a transform's buffer:
// lanes of one wave (LDS instructions of a wave complete in order, so only
// the compiler has to be held back) or the whole workgroup.
template <bool WAVE>
__device__ __forceinline__ void grp_sync() {
  if constexpr (WAVE) {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  } else {
    __syncthreads();
  }
}

// The first twiddle of every butterfly of the later passes that thread t of
// NT takes part in, loaded once per kernel: a load between two passes would
// expose its latency in every transform.
template <int L, int NT> struct FftTw {
  static constexpr int NP = cp_np(L);
  static constexpr int items(int p) { return (L / cp_radix(L, p) + NT - 1) / NT; }
  static constexpr int off(int p) { return p <= 1 ? 0 : off(p - 1) + items(p - 1); }
  static constexpr int ns(int p) { return p == 0 ? 1 : ns(p - 1) * cp_radix(L, p - 1); }
  static constexpr int N = off(NP) > 0 ? off(NP) : 1;
  double2 w[N];
  template <int P = 1>
  __device__ __forceinline__ void load(const double2 *__restrict__ tw, int twm, int t) {
    if constexpr (P < NP) {
      constexpr int R = cp_radix(L, P), NS = ns(P);
#pragma unroll
      for (int i = 0; i < items(P); ++i) w[off(P) + i] = tw[((t + i * NT) % NS) * (L / (NS * R)) * twm];
      load<P + 1>(tw, twm, t);
    }
  }
};

// FFT of one sequence of length L by NT threads.  The first pass takes
// element e from ld(i, r, e), the last one hands it to st(i, r, e, x);
// between passes the data go through xb (element e at xb[pidx(e)*ES]).
// Threads with act = false only take part in the barriers.  Compared with
// fft_ct in LDS this saves the staging round trip of the first and the last
// pass and two barriers per pass.  xb may still be read by others at the
// call: the first write is behind a barrier.
template <int L, int NT, bool INV, int ES, bool WAVE, bool LEAN, int CH = 16, int P = 0, int NS = 1, class Ld, class St>
__device__ __forceinline__ void fft_io(double2 *xb, const FftTw<L, NT> &T, int t, bool act, const Ld &ld, const St &st) {
  // LEAN: the thread index and the twiddles are made opaque in every
  // transform.  The compiler otherwise keeps what depends on them (twiddle
  // powers, the caller's twiddles, addresses) in registers from one transform
  // to the next: faster where the registers are free, but 50 to 90 VGPRs
  if constexpr (LEAN && P == 0) asm volatile("" : "+v"(t));
  constexpr int NP = cp_np(L);
  constexpr int R = cp_radix(L, P), M = L / R, ITEMS = (M + NT - 1) / NT;
  constexpr bool LAST = P == NP - 1;
  double2 v[ITEMS][R];
#pragma unroll
  for (int i = 0; i < ITEMS; ++i) {
    const int j = t + i * NT;
    if (act && (M % NT == 0 || j < M)) {
#pragma unroll
      for (int r = 0; r < R; ++r) {
        if constexpr (P == 0) {
          // a bounded number of the caller's loads in flight per thread
          if (r % CH == 0 && r > 0) __builtin_amdgcn_sched_barrier(0);
          v[i][r] = ld(i, r, j + r * M);
        } else {
          v[i][r] = xb[pidx(j + r * M) * ES];
        }
      }
    }
  }
#pragma unroll
  for (int i = 0; i < ITEMS; ++i) {
    const int j = t + i * NT;
    if (act && (M % NT == 0 || j < M)) {
      if constexpr (NS > 1) {
        double2 w1 = T.w[FftTw<L, NT>::off(P) + i];
        if constexpr (LEAN) asm volatile("" : "+v"(w1.x), "+v"(w1.y));
        if (INV) w1.y = -w1.y;
        twiddle_row<R>(v[i], w1);
      }
      Dft<R, INV>::run(v[i]);
    }
  }
  if constexpr (LAST) {
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
      const int j = t + i * NT;
      if (act && (M % NT == 0 || j < M)) {
#pragma unroll
        for (int r = 0; r < R; ++r) st(i, r, j + r * M, v[i][r]);
      }
    }
  } else {
    grp_sync<WAVE>();
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
      const int j = t + i * NT;
      if (act && (M % NT == 0 || j < M)) {
        const int base = (j / NS) * NS * R + (j % NS);
#pragma unroll
        for (int r = 0; r < R; ++r) xb[pidx(base + r * NS) * ES] = v[i][r];
      }
    }
    grp_sync<WAVE>();
    fft_io<L, NT, INV, ES, WAVE, LEAN, CH, P + 1, NS * R>(xb, T, t, act, ld, st);
  }
}

// items and radix of the last pass: a thread's outputs are the NOUT values
// e = t + i NT + r (L / R)
template <int L, int NT> struct FftOut {
  static constexpr int R = cp_radix(L, cp_np(L) - 1), M = L / R, ITEMS = (M + NT - 1) / NT, N = ITEMS * R;
};

// ============================================================================
// Column stage
// ============================================================================
struct ColStepArgs {
  const double2 *Rc, *Rpx;   // Rpx null: no penalisation anywhere
  const double2 *W0, *NL1;
  double2 *NL0, *W1;
  double2 *o[5];             // omega, psi, i ky psi, -ky^2 psi, i ky omega (null: not wanted)
  const DevScalars *s;
  int explicit_step;
  int py0, py1;              // rows of Rpx that may be nonzero
  int r0, r1;                // rows of -ky^2 psi that are stored
  StepConsts c;
};

// a / b for a divisor b shared by many quotients, r = 1/b rounded: one
// Newton correction of a*r rounds as the division does while its remainder is
// exact, and the fixup takes zeros, infinities and NaN as the division does.
// The remainder of a dividend below 2^-1000 is a denormal number and rounds (up
// to 5 % of such quotients come out otherwise; a damped mode passes through
// that range), so where a wave meets a dividend below 2^-960 (div_small) it
// divides.  The choice is made once for all of a thread's quotients: a branch
// at each cost a coupled 256^2 step 0.7 % and two beams at 768 x 512 1 %.
__device__ __forceinline__ double2 div_fast(double2 a, double b, double r) {
  const double qx = a.x * r, qy = a.y * r;
  return make_double2(__builtin_amdgcn_div_fixup(fma(fma(-qx, b, a.x), r, qx), b, a.x),
                      __builtin_amdgcn_div_fixup(fma(fma(-qy, b, a.y), r, qy), b, a.y));
}
__device__ __forceinline__ bool div_small(double2 a) {
  const double x = fabs(a.x), y = fabs(a.y);
  return (x < 0x1p-960 && x != 0.0) || (y < 0x1p-960 && y != 0.0);
}
__device__ __forceinline__ double2 div_slow(double2 a, double b) { return make_double2(a.x / b, a.y / b); }
__device__ __forceinline__ double2 div_by(double2 a, double b, double r) {
  return __builtin_expect(div_small(a), 0) ? div_slow(a, b) : div_fast(a, b, r);
}

// dealias(c, kx, ky) with the divisions left to the modes on the ellipse's
// edge, where a product with the reciprocals could decide otherwise
__device__ __forceinline__ double dealias_fast(const StepConsts &c, int kx, int ky) {
  if (!c.idealis) return 1.0;
  const double a = (double)kx, b = (double)ky;
  const double q = a * a * c.rkxt2 + b * b * c.rkyt2;
  if (fabs(q - 1.0) < 1e-12) return dealias(c, kx, ky);
  return q >= 1.0 ? 0.0 : 1.0;
}

// Tile of workgroup bid when the first nl of nblk tiles are the ones with work
// (the others' columns are beyond the dealiasing ellipse): as xcd_remap, but
// each XCD gets its share of either kind.
__device__ __forceinline__ int live_remap(int bid, int nblk, int nl) {
  if (nblk % 8 != 0) return bid;
  nl = min((nl + 7) & ~7, nblk);
  const int x = bid & 7, i = bid >> 3, l = nl >> 3, d = (nblk - nl) >> 3;
  return i < l ? x * l + i : nl + x * d + (i - l);
}

// One workgroup per TX columns, NS slots of TX*NT threads.  Slots 0 and 1
// transform Rc and Rpx; all threads then form nlk and the AB2 update (W0
// and NL1 loaded before the transforms) and leave vortk(n1) and psi in the
// first two slots' buffers, from which the derived fields are transformed
// back, one per slot.  NS = 4: omega, psi, i ky psi, -ky^2 psi, then
// i ky omega in a second round of slot 0; NS = 2 (long columns, whose LDS
// leaves no room for four): slot 0 omega, i ky omega, slot 1 the others.
template <int L, int TX, int NT, int NS, bool LEAN>
__device__ __forceinline__ void col_step_body(const ColStepArgs &a, const double2 *__restrict__ twy, int bid, int nblk) {
  extern __shared__ double2 lds[];
  static_assert(NS == 2 || NS == 4, "slots");
  constexpr int PL = padlen(L), NTHR = NS * TX * NT, SB = TX * PL;
  constexpr int EL = (L * TX + NTHR - 1) / NTHR;
  static_assert(NTHR % TX == 0, "a thread stays on its column");
  using Out = FftOut<L, NT>;
  const StepConsts &c = a.c;
  const int tid = threadIdx.x, H = c.H;
  const int slot = tid / (TX * NT), w = tid - slot * (TX * NT), cc = w % TX, t = w / TX;
  const int kx0 = live_remap(bid, nblk, (c.kc + TX - 1) / TX) * TX;
  double2 *xb = lds + slot * SB + cc;
  const bool px_on = a.Rpx != nullptr;
  FftTw<L, NT> T;
  T.load(twy, 1, t);
  const double b10 = a.s->b10, b11 = a.s->b11, cx1 = a.s->cx1, cy1 = a.s->cy1, cx0 = a.s->cx0, cy0 = a.s->cy0;
  // the update's own operands, in flight during the forward transforms; a mode
  // that dealiasing removes needs none
  const int c2 = tid % TX, kx = kx0 + c2, i0 = tid / TX;  // rows i0 + q NTHR/TX of column kx
  constexpr bool PREF = EL <= 2;
  double2 w0[EL], n1[EL];
  double dl[EL];
  auto operands = [&](int q) {
    const int idx = i0 + q * (NTHR / TX);
    w0[q] = n1[q] = make_double2(0.0, 0.0);
    dl[q] = kx < c.kc ? dealias_fast(c, kx, abs(ky_signed(idx, L))) : 0.0;
    if (L * TX % NTHR == 0 || idx < L) {
      const size_t g = (size_t)(dl[q] != 0.0 ? idx : 0) * H + kx;
      const double2 w = a.W0[g], n = a.explicit_step ? w : a.NL1[g];
      if (dl[q] != 0.0) {
        w0[q] = w;
        if (!a.explicit_step) n1[q] = n;
      }
    }
  };
  if constexpr (PREF) {
#pragma unroll
    for (int q = 0; q < EL; ++q) operands(q);
  }
  {
    double2 z[Out::N];
    const double2 *src = slot == 0 ? a.Rc : a.Rpx;
    const int ya = slot == 0 ? 0 : a.py0, yb = slot == 0 ? L - 1 : a.py1;
    const bool act = slot == 0 || (slot == 1 && px_on);
    fft_io<L, NT, false, TX, false, LEAN>(
        xb, T, t, act,
        [&](int, int, int e) {
          return (e >= ya && e <= yb) ? src[(size_t)e * H + kx0 + cc] : make_double2(0.0, 0.0);
        },
        [&](int i, int r, int, double2 x) { z[i * Out::R + r] = x; });
    __syncthreads();
    if (act) {
#pragma unroll
      for (int i = 0; i < Out::ITEMS; ++i) {
        const int j = t + i * NT;
        if (Out::M % NT == 0 || j < Out::M) {
#pragma unroll
          for (int r = 0; r < Out::R; ++r) xb[pidx(j + r * Out::M) * TX] = z[i * Out::R + r];
        }
      }
    }
    __syncthreads();
  }
  {
    // a constant time step: both viscous factors are the same number
    const bool same = cx0 == cx1 && cy0 == cy1;
    const double kx2 = (double)(kx * kx);
    bool small = false;
    if constexpr (!PREF) {
#pragma unroll
      for (int q = 0; q < EL; ++q) operands(q);
    }
#pragma unroll
    for (int q = 0; q < EL; ++q) {
      const int idx = i0 + q * (NTHR / TX);
      if (L * TX % NTHR == 0 || idx < L) {
        double2 nl = make_double2(0.0, 0.0), w1 = nl, psi = nl;
        const double2 *l0 = lds + pidx(idx) * TX + c2;
        if (idx != L / 2) {
          const int ky = ky_signed(idx, L);
          const int aky = ky < 0 ? -ky : ky;
          const double kyf = (double)ky * c.sy;
          const double2 fc = *l0;
          const double2 fp = px_on ? l0[SB] : make_double2(0.0, 0.0);
          const double2 Fc = make_double2(fc.x * c.norm, fc.y * c.norm);
          const double2 Fp = make_double2(fp.x * c.norm, fp.y * c.norm);
          nl = make_double2(Fc.x + kyf * Fp.y, Fc.y - kyf * Fp.x);
          const double ky2 = (double)(aky * aky);
          const double v1 = exp(cx1 * kx2 + cy1 * ky2);
          const double d = dl[q];
          if (a.explicit_step) {
            w1.x = (w0[q].x + b10 * nl.x) * v1 * d;
            w1.y = (w0[q].y + b10 * nl.y) * v1 * d;
          } else {
            const double v0 = same ? v1 : exp(cx0 * kx2 + cy0 * ky2);
            const double2 n1v = make_double2(n1[q].x * v0, n1[q].y * v0);
            w1.x = ((w0[q].x + b10 * nl.x) + b11 * n1v.x) * v1 * d;
            w1.y = ((w0[q].y + b10 * nl.y) + b11 * n1v.y) * v1 * d;
          }
          if (kx != 0 || ky != 0) {
            const double quot = kx2 * c.scalex + ky2 * c.scaley, rq = 1.0 / quot;
            psi = div_fast(w1, quot, rq);
            small = small || div_small(w1);
          }
        }
        const size_t g = (size_t)idx * H + kx;
        a.NL0[g] = nl;
        a.W1[g] = w1;
        w0[q] = w1;
        n1[q] = psi;
      }
    }
    if (__builtin_expect(__any(small), 0)) {
#pragma unroll
      for (int q = 0; q < EL; ++q) {
        const int idx = i0 + q * (NTHR / TX), ky = ky_signed(idx, L);
        if (idx != L / 2 && (kx != 0 || ky != 0))
          n1[q] = div_slow(w0[q], kx2 * c.scalex + (double)(ky * ky) * c.scaley);
      }
    }
  }
  if (kx0 >= c.kc) return;  // vorticity and everything derived from it are zero, and not read
  // the derived fields, NS at a time: written to the slots' buffers by the
  // threads that hold the update, transformed back and stored
  auto derived = [&](int f, int q) {
    const double kyf = (double)ky_signed(i0 + q * (NTHR / TX), L) * c.sy;
    if (f == 0) return w0[q];
    if (f == 1) return n1[q];
    if (f == 3) return make_double2(-(kyf * kyf) * n1[q].x, -(kyf * kyf) * n1[q].y);
    const double2 v = f == 4 ? w0[q] : n1[q];
    return make_double2(-kyf * v.y, kyf * v.x);
  };
#pragma unroll
  for (int rd = 0; rd < (4 + NS) / NS; ++rd) {
    // the fields of this turn: omega, psi, i ky psi, -ky^2 psi, i ky omega
    // in this order for four slots; for two (omega, psi), (i ky psi, i ky
    // omega), (-ky^2 psi)
    constexpr int kF[5] = {0, 1, 2, NS == 2 ? 4 : 3, NS == 2 ? 3 : 4};
    bool any = false;
#pragma unroll
    for (int k = 0; k < NS; ++k)
      if (rd * NS + k < 5) any = any || a.o[kF[rd * NS + k]] != nullptr;
    if (!any) continue;
    if (rd > 0) __syncthreads();
#pragma unroll
    for (int q = 0; q < EL; ++q) {
      const int idx = i0 + q * (NTHR / TX);
      if (L * TX % NTHR == 0 || idx < L) {
#pragma unroll
        for (int k = 0; k < NS; ++k)
          if (rd * NS + k < 5) lds[k * SB + pidx(idx) * TX + c2] = derived(kF[rd * NS + k], q);
      }
    }
    __syncthreads();
    double2 *out = nullptr;
    int ya = 0, yb = L - 1;
#pragma unroll
    for (int k = 0; k < NS; ++k)
      if (rd * NS + k < 5 && slot == k) {
        out = a.o[kF[rd * NS + k]];
        if (kF[rd * NS + k] == 3) { ya = a.r0; yb = a.r1; }
      }
    fft_io<L, NT, true, TX, false, LEAN>(
        xb, T, t, out != nullptr, [&](int, int, int e) { return xb[pidx(e) * TX]; },
        [&](int, int, int e, double2 x) {
          if (e >= ya && e <= yb) out[(size_t)e * H + kx0 + cc] = x;
        });
  }
}

// The same stage for long columns, whose LDS holds one field of a tile: the
// fields follow one another, and a column's values stay in the registers of
// the threads that hold them (element t + NT q, the same in every radix of
// the plan), so the tile's buffer only serves the passes' exchanges.
template <int L, int TX, int NT, bool PX>
__device__ __forceinline__ void col_direct_body(const ColStepArgs &a, const double2 *__restrict__ twy, int bid, int nblk) {
  extern __shared__ double2 lds[];
  constexpr int E = L / NT, M0 = L / cp_radix(L, 0);
  using Out = FftOut<L, NT>;
  static_assert(Out::M == NT && M0 % NT == 0, "values stay in their thread");
  const StepConsts &c = a.c;
  const int tid = threadIdx.x, H = c.H, cc = tid % TX, t = tid / TX;
  const int kx = live_remap(bid, nblk, (c.kc + TX - 1) / TX) * TX + cc;
  double2 *xb = lds + cc;
  FftTw<L, NT> T;
  T.load(twy, 1, t);
  double2 P[PX ? E : 1], W[E];
  if constexpr (PX)
    fft_io<L, NT, false, TX, false, true>(
        xb, T, t, true,
        [&](int, int, int e) {
          return (e >= a.py0 && e <= a.py1) ? a.Rpx[(size_t)e * H + kx] : make_double2(0.0, 0.0);
        },
        [&](int, int r, int, double2 x) { P[r] = x; });
  fft_io<L, NT, false, TX, false, true>(
      xb, T, t, true, [&](int, int, int e) { return a.Rc[(size_t)e * H + kx]; },
      [&](int, int r, int, double2 x) { W[r] = x; });
  {
    const double b10 = a.s->b10, b11 = a.s->b11, cx1 = a.s->cx1, cy1 = a.s->cy1, cx0 = a.s->cx0, cy0 = a.s->cy0;
    const bool same = cx0 == cx1 && cy0 == cy1;
    const double kx2 = (double)(kx * kx);
#pragma unroll
    for (int q = 0; q < E; ++q) {
      if (q % 2 == 0) __builtin_amdgcn_sched_barrier(0);
      const int idx = t + NT * q;
      const size_t g = (size_t)idx * H + kx;
      double2 nl = make_double2(0.0, 0.0), w1 = nl;
      if (idx != L / 2) {
        const int ky = ky_signed(idx, L);
        const int aky = ky < 0 ? -ky : ky;
        const double kyf = (double)ky * c.sy;
        const double2 Fc = make_double2(W[q].x * c.norm, W[q].y * c.norm);
        double2 Fp = make_double2(0.0, 0.0);
        if constexpr (PX) Fp = make_double2(P[q].x * c.norm, P[q].y * c.norm);
        nl = make_double2(Fc.x + kyf * Fp.y, Fc.y - kyf * Fp.x);
        const double ky2 = (double)(aky * aky);
        const double v1 = exp(cx1 * kx2 + cy1 * ky2);
        const double d = kx < c.kc ? dealias_fast(c, kx, aky) : 0.0;
        const double2 zero = make_double2(0.0, 0.0);  // a mode that dealiasing removes needs no operands
        const double2 w0 = d != 0.0 ? a.W0[g] : zero;
        if (a.explicit_step) {
          w1.x = (w0.x + b10 * nl.x) * v1 * d;
          w1.y = (w0.y + b10 * nl.y) * v1 * d;
        } else {
          const double v0 = same ? v1 : exp(cx0 * kx2 + cy0 * ky2);
          const double2 n1 = d != 0.0 ? a.NL1[g] : zero;
          const double2 n1v = make_double2(n1.x * v0, n1.y * v0);
          w1.x = ((w0.x + b10 * nl.x) + b11 * n1v.x) * v1 * d;
          w1.y = ((w0.y + b10 * nl.y) + b11 * n1v.y) * v1 * d;
        }
      }
      a.NL0[g] = nl;
      a.W1[g] = w1;
      W[q] = w1;
    }
  }
  if (kx - cc >= c.kc) return;  // vorticity and everything derived from it are zero, and not read
  // omega, i ky omega, then W becomes psi: psi, i ky psi, -ky^2 psi
#pragma unroll
  for (int k = 0; k < 5; ++k) {
    constexpr int kF[5] = {0, 4, 1, 2, 3};
    const int f = kF[k];
    double2 *out = a.o[f];
    if (k == 2) {
      bool small = false;
#pragma unroll
      for (int q = 0; q < E; ++q) small = small || div_small(W[q]);
      auto psi = [&](auto slow) {
#pragma unroll
        for (int q = 0; q < E; ++q) {
          if (q % 2 == 0) __builtin_amdgcn_sched_barrier(0);
          const int idx = t + NT * q, ky = ky_signed(idx, L), aky = ky < 0 ? -ky : ky;
          if (idx != L / 2 && (kx != 0 || ky != 0)) {
            const double quot = (double)(kx * kx) * c.scalex + (double)(aky * aky) * c.scaley;
            if constexpr (decltype(slow)::value) W[q] = div_slow(W[q], quot);
            else W[q] = div_fast(W[q], quot, 1.0 / quot);
          } else {
            W[q] = make_double2(0.0, 0.0);
          }
        }
      };
      if (__builtin_expect(__any(small), 0)) psi(std::true_type{});
      else psi(std::false_type{});
    }
    if (!out) continue;
    const int ya = f == 3 ? a.r0 : 0, yb = f == 3 ? a.r1 : L - 1;
    fft_io<L, NT, true, TX, false, true>(
        xb, T, t, true,
        [&](int i, int r, int e) {
          const double2 v = W[i + r * (M0 / NT)];
          const double kyf = (double)ky_signed(e, L) * c.sy;
          if (f < 2) return v;
          if (f == 3) return make_double2(-(kyf * kyf) * v.x, -(kyf * kyf) * v.y);
          return make_double2(-kyf * v.y, kyf * v.x);
        },
        [&](int, int, int e, double2 x) {
          if (e >= ya && e <= yb) out[(size_t)e * H + kx] = x;
        });
  }
}

// The stage's shape for a column length: TX columns per workgroup, NT threads
// per column and slot, NS slots (0: the direct form, with PX for Rpx).
template <int LC, int TXC, int NTC, int NSC, bool LEANC> struct ColStepShape {
  static constexpr int L = LC, TX = TXC, NT = NTC, NS = NSC;
  static constexpr bool DIRECT = NSC == 0;
  static constexpr int THREADS = TX * NT * (DIRECT ? 1 : NS);
  static constexpr size_t LDS = sizeof(double2) * TX * padlen(L) * (DIRECT ? 1 : NS);
  static __device__ __forceinline__ void run(const ColStepArgs &a, const double2 *__restrict__ twy, int bid, int nblk) {
    if constexpr (DIRECT) col_direct_body<L, TX, NT, LEANC>(a, twy, bid, nblk);
    else col_step_body<L, TX, NT, NS, LEANC>(a, twy, bid, nblk);
  }
};
template <class S>
__global__ void __launch_bounds__(S::THREADS) k_col_step(ColStepArgs a, const double2 *__restrict__ twy) {
  S::run(a, twy, blockIdx.x, gridDim.x);
}

// ============================================================================
// Pressure stage (K7)
// ============================================================================
struct PressArgs {
  const double2 *Rq, *Rqy;
  double2 *Cq;
  int r0, r1;  // rows of the inverse transform that are stored
  StepConsts c;
};

// the right-hand side of q's equation at mode (kx, idx) from the transforms of
// its two parts (pressure, NavierStokes.f90:366-382), and |k|^2 in quot (1 at the
// modes that are zero)
template <int L>
__device__ __forceinline__ double2 press_rhs(const StepConsts &c, int kx, int idx, double2 a, double2 b, double &quot) {
  const int ky = ky_signed(idx, L);
  const int aky = ky < 0 ? -ky : ky;
  quot = 1.0;
  if (idx == L / 2 || (kx == 0 && ky == 0)) return make_double2(0.0, 0.0);
  const double kyf = (double)ky * c.sy;
  const double2 fa = make_double2(a.x * c.norm, a.y * c.norm);
  const double2 fb = make_double2(b.x * c.norm, b.y * c.norm);
  quot = ((double)(kx * kx) * c.scalex + (double)(aky * aky) * c.scaley);
  return make_double2(fa.x - kyf * fb.y, fa.y + kyf * fb.x);
}

// Two slots of TX*NT threads transform one right-hand side each straight from
// memory, all threads form q, slot 0 transforms it back into memory.  It
// reads two fields and stores a band of rows: bound by memory from about
// 1024^2, by the chain of two transforms below.  Against the stage that
// staged its columns in LDS first (compile-time plan, best width): 5.8 -> 5.1
// us at 256^2, 6.6 -> 5.5 at 512^2, 11.0 -> 9.3 at 1024^2, 19.8 -> 14.5 at
// 1024 x 1536.  Two columns per workgroup: one gives 5.1, 6.1, 11.3, 16.1 us.
template <int L, int TX, int NT>
__device__ __forceinline__ void press_step_body(const PressArgs &a, const double2 *__restrict__ twy, int bid, int nblk) {
  extern __shared__ double2 lds[];
  constexpr int PL = padlen(L), NTHR = 2 * TX * NT, SB = TX * PL;
  constexpr bool WAVE = NTHR <= 64;
  using Out = FftOut<L, NT>;
  const StepConsts &c = a.c;
  const int tid = threadIdx.x, H = c.H;
  const int slot = tid / (TX * NT), w = tid - slot * (TX * NT), cc = w % TX, t = w / TX;
  const int kx0 = xcd_remap(bid, nblk) * TX;
  double2 *xb = lds + slot * SB + cc;
  FftTw<L, NT> T;
  T.load(twy, 1, t);
  {
    double2 z[Out::N];
    const double2 *src = (slot == 0 ? a.Rq : a.Rqy) + kx0 + cc;
    fft_io<L, NT, false, TX, WAVE, false>(
        xb, T, t, true, [&](int, int, int e) { return src[(size_t)e * H]; },
        [&](int i, int r, int, double2 x) { z[i * Out::R + r] = x; });
    grp_sync<WAVE>();
#pragma unroll
    for (int i = 0; i < Out::ITEMS; ++i) {
      const int j = t + i * NT;
      if (Out::M % NT == 0 || j < Out::M) {
#pragma unroll
        for (int r = 0; r < Out::R; ++r) xb[pidx(j + r * Out::M) * TX] = z[i * Out::R + r];
      }
    }
    grp_sync<WAVE>();
  }
  {
    constexpr int EL = L * TX / NTHR;
    static_assert(L * TX % NTHR == 0, "every thread has as many modes");
    double2 rhs[EL];
    double quot[EL];
    bool small = false;
    auto at = [&](int q) { return lds + pidx((tid + q * NTHR) / TX) * TX + (tid + q * NTHR) % TX; };
#pragma unroll
    for (int q = 0; q < EL; ++q) {
      const int e = tid + q * NTHR;
      rhs[q] = press_rhs<L>(c, kx0 + e % TX, e / TX, at(q)[0], at(q)[SB], quot[q]);
      small = small || div_small(rhs[q]);
    }
    if (__builtin_expect(__any(small), 0)) {
#pragma unroll
      for (int q = 0; q < EL; ++q) *at(q) = div_slow(rhs[q], quot[q]);
    } else {
#pragma unroll
      for (int q = 0; q < EL; ++q) *at(q) = div_fast(rhs[q], quot[q], 1.0 / quot[q]);
    }
  }
  grp_sync<WAVE>();
  fft_io<L, NT, true, TX, WAVE, false>(
      xb, T, t, slot == 0, [&](int, int, int e) { return xb[pidx(e) * TX]; },
      [&](int, int, int e, double2 x) {
        if (e >= a.r0 && e <= a.r1) a.Cq[(size_t)e * H + kx0 + cc] = x;
      });
}

template <int LC, int TXC, int NTC> struct PressShape {
  static constexpr int L = LC, TX = TXC, NT = NTC, THREADS = 2 * TX * NT;
  static constexpr size_t LDS = sizeof(double2) * 2 * TX * padlen(L);
  static __device__ __forceinline__ void run(const PressArgs &a, const double2 *__restrict__ twy, int bid, int nblk) {
    press_step_body<L, TX, NT>(a, twy, bid, nblk);
  }
};
template <class S>
__global__ void __launch_bounds__(S::THREADS) k_press_step(PressArgs a, const double2 *__restrict__ twy) {
  S::run(a, twy, blockIdx.x, gridDim.x);
}

// ============================================================================
// Row stage
// ============================================================================
struct RowStepArgs {
  const double2 *Cw, *Cpsi, *Cpsiy, *Cwy;  // Cwy = Fy^-1[i ky omega] (NEXT)
  double *u1, *u2, *vor_mean;
  const double *ms;
  MaskBox mb;
  Window win, win2;
  double *sums, *umax_part;
  double2 *Rq, *Rqy, *Rc;
  const DevScalars *s;
  StepConsts c;
};

// sum / max over the NT lanes of a row (NT <= 64, a power of two)
template <int NT>
__device__ __forceinline__ double seg_sum(double v) {
  if constexpr (NT == 64) return wave_sum(v);
#pragma unroll
  for (int o = NT / 2; o > 0; o >>= 1) v += __shfl_xor(v, o);
  return v;
}
template <int NT>
__device__ __forceinline__ double seg_max(double v) {
  if constexpr (NT == 64) return wave_max(v);
#pragma unroll
  for (int o = NT / 2; o > 0; o >>= 1) v = fmax(v, __shfl_xor(v, o));
  return v;
}

// element e of the inverse row transform's input from the half spectrum's
// entries xa = X_e, xq = X_{H-e}
__device__ __forceinline__ double2 c2r_elem(double2 xa, double2 xq, int e, double2 wc) {
  if (e == 0) return make_double2(xa.x, xa.x);  // x-DC: real part only, x-Nyquist is zero
  return c2r_one(xa, xq, wc);
}
__device__ __forceinline__ double2 mul_ik(double2 a, double kf) { return make_double2(-kf * a.y, kf * a.x); }

// One row by four slots of NT threads, RPB rows per workgroup.  Inverse
// transforms of psi_y, psi_x, omega and (NEXT) omega_x, one per slot; then
// velocity, diagnostics and products; forward transforms of the pressure
// right-hand sides (PRES) beside the inverse one of omega_y (in slot 2, as
// the conjugate of a forward transform of the conjugate: the same
// operations); then the convective term's forward transform.
template <int H, int NT, int RPB, bool LEAN, bool PRES, bool NEXT>
__device__ __forceinline__ void row_step_body(const RowStepArgs &a, const double2 *__restrict__ twx, int bid) {
  extern __shared__ double2 lds[];
  constexpr int NS = 4, PL = padlen(H), nx = 2 * H, NR = NS * NT;  // NR threads per row
  constexpr bool WAVE = NR <= 64;
  constexpr int PN = (H + NR - 1) / NR;
  static_assert(!WAVE || (NR & (NR - 1)) == 0, "slots");
  static_assert(RPB == 1 || (WAVE && 64 % NR == 0), "several rows per workgroup: each within one wave");
  using Out = FftOut<H, NT>;
  const int tid = threadIdx.x, rr = RPB == 1 ? 0 : tid / NR, p = RPB == 1 ? tid : tid - rr * NR;
  const int slot = p / NT;
  int t = p - slot * NT;
  const int y = bid * RPB + rr;
  double2 *row = lds + rr * (NS * PL), *xb = row + slot * PL;
  const size_t rowk = (size_t)y * H, rowx = (size_t)y * nx;
  const double sx = a.c.sx;
  // the outputs of a slot's transform into its buffer, in natural order
  auto put = [&](const double2 *z) {
#pragma unroll
    for (int i = 0; i < Out::ITEMS; ++i) {
      if (Out::M % NT != 0 && t + i * NT >= Out::M) continue;
#pragma unroll
      for (int r = 0; r < Out::R; ++r) xb[pidx(t + i * NT + r * Out::M)] = z[i * Out::R + r];
    }
  };
  constexpr int R0 = cp_radix(H, 0), M0 = H / R0, IT0 = (M0 + NT - 1) / NT, NI = IT0 * R0;
  auto for_in = [&](auto fn) {
#pragma unroll
    for (int i = 0; i < IT0; ++i) {
      if (M0 % NT != 0 && t + i * NT >= M0) continue;
#pragma unroll
      for (int r = 0; r < R0; ++r) fn(i * R0 + r, t + i * NT + r * M0);
    }
  };
  // everything of the row that does not depend on the transforms, in flight
  // with their inputs: pass twiddles, mean vorticity, sponge
  FftTw<H, NT> T;
  T.load(twx, 2, t);
  const double UMx = a.s->UMx, UMy = a.s->UMy, Mx = a.s->Mx, My = a.s->My, time = a.s->time, dt1 = a.s->dt1;
  double2 vm[PN], ms[NEXT ? PN : 1];
#pragma unroll
  for (int k = 0; k < PN; ++k) {
    const int n = p + k * NR;
    if (H % NR != 0 && n >= H) continue;
    vm[k] = reinterpret_cast<const double2 *>(a.vor_mean + rowx)[n];
    if constexpr (NEXT)
      ms[k] = a.ms ? reinterpret_cast<const double2 *>(a.ms + rowx)[n] : make_double2(0.0, 0.0);
  }
  double2 z[Out::N];
  {
    const double2 *src = slot == 0 ? a.Cpsiy : slot == 1 ? a.Cpsi : a.Cw;
    const bool ik = slot == 1 || slot == 3;
    src += rowk;
    const int kc = a.c.kc;
    fft_io<H, NT, true, 1, WAVE, LEAN, LEAN ? 4 : 16>(
        xb, T, t, NEXT || slot < 3,
        [&](int, int, int e) {
          const int q = e == 0 ? 0 : H - e;
          double2 xa = live(src, e, H, kc), xq = live(src, q, H, kc);
          if (ik) { xa = mul_ik(xa, (double)e * sx); xq = mul_ik(xq, (double)q * sx); }
          return c2r_elem(xa, xq, e, cconj(twx[e]));
        },
        [&](int i, int r, int, double2 x) { z[i * Out::R + r] = x; });
  }
  grp_sync<WAVE>();
  if (NEXT || slot < 3) put(z);
  grp_sync<WAVE>();
  const MaskBox mb = a.mb;
  const Window win = a.win, win2 = a.win2;
  const bool mrow = mb.x1 >= mb.x0 && y >= mb.y0 && y <= mb.y1;
  const bool wrow = y >= win.y0 && y <= win.y1;
  const bool two = win2.x1 >= win2.x0;
  const bool wrow2 = two && y >= win2.y0 && y <= win2.y1;
  const double tsum = time + dt1, trcp = 1.0 / tsum;
  double um = 0.0, en[2] = {0.0, 0.0};
  bool small = false;
  double2 csw[NEXT ? PN : 1];
#pragma unroll
  for (int k = 0; k < PN; ++k) {
    const int n = p + k * NR;
    if (H % NR != 0 && n >= H) continue;
    if constexpr (LEAN) __builtin_amdgcn_sched_barrier(0);  // one element's temporaries at a time
    const int qn = pidx(n);
    const double2 uy1 = row[qn], gx = row[PL + qn], w = row[2 * PL + qn];
    double2 a1, a2;
    {
#pragma clang fp contract(off)
      a1 = make_double2(uy1.x + UMx, uy1.y + UMx);
      a2 = make_double2(-gx.x + UMy, -gx.y + UMy);
    }
    reinterpret_cast<double2 *>(a.u1 + rowx)[n] = a1;
    reinterpret_cast<double2 *>(a.u2 + rowx)[n] = a2;
    um = fmax(um, fmax(a1.x * a1.x + a2.x * a2.x, a1.y * a1.y + a2.y * a2.y));
    {
      const double2 m = make_double2(vm[k].x * time + dt1 * w.x, vm[k].y * time + dt1 * w.y);
      reinterpret_cast<double2 *>(a.vor_mean + rowx)[n] = div_fast(m, tsum, trcp);
      small = small || div_small(m);
    }
    en[0] += w.x * w.x + w.y * w.y;
    {
      const double u = a1.x - Mx, v = a2.x - My, r = a1.y - Mx, q = a2.y - My;
      en[1] += (u * u + v * v) + (r * r + q * q);
    }
    if constexpr (NEXT) {
      const double2 wx = row[3 * PL + qn];
      const double2 s = ms[k];
      const double2 cv = make_double2(-(a1.x * wx.x), -(a1.y * wx.y));
      const double2 sw = make_double2(s.x * w.x, s.y * w.y);
      row[3 * PL + qn] = cv;  // this thread takes it back below
      csw[k] = sw;
    }
    // penal(:,:,1) - vor*uy, penal(:,:,2) + vor*ux (:357-358); on the mask's
    // rows the velocity is left for the loop below, which adds the
    // penalisation
    if (mrow) {
      row[qn] = a1;
      row[PL + qn] = a2;
    } else if (PRES) {
      row[qn] = make_double2(0.0 - w.x * a2.x, 0.0 - w.y * a2.y);
      row[PL + qn] = make_double2(0.0 + w.x * a1.x, 0.0 + w.y * a1.y);
    }
  }
  if (__builtin_expect(__any(small), 0)) {
#pragma unroll
    for (int k = 0; k < PN; ++k) {
      const int n = p + k * NR;
      if (H % NR != 0 && n >= H) continue;
      const double2 w = row[2 * PL + pidx(n)];
      reinterpret_cast<double2 *>(a.vor_mean + rowx)[n] =
          div_slow(make_double2(vm[k].x * time + dt1 * w.x, vm[k].y * time + dt1 * w.y), tsum);
    }
  }
  // the mask's rows: penalisation p = chi (u - u_s), its sums, and the
  // pressure right-hand sides with it
  const int nv = !mrow ? 2 : two ? kNSUM : kNSUM1;
  double acc[kNSUM];
#pragma unroll
  for (int i = 0; i < kNSUM; ++i) acc[i] = i < 2 ? en[i] : 0.0;
  if (mrow) {
#pragma unroll
    for (int k = 0; k < PN; ++k) {
      const int n = p + k * NR;
      if (H % NR != 0 && n >= H) continue;
      __builtin_amdgcn_sched_barrier(0);
      const int qn = pidx(n), x = 2 * n;
      const double2 a1 = row[qn], a2 = row[PL + qn];
      double2 q1 = make_double2(0.0, 0.0), q2 = q1;
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        if (!mb.inside(x + h, y)) continue;
        const size_t qq = (size_t)(y - mb.y0) * mb.w + (x + h - mb.x0);
        const double m = mb.m[qq], vx = mb.vx[qq], vy = mb.vy[qq];
        const double uu1 = h ? a1.y : a1.x, uu2 = h ? a2.y : a2.x;
        const double r1 = uu1 - vx, r2 = uu2 - vy;
        const double p1 = m * r1, p2 = m * r2;
        acc[2] += m * (r1 * r1 + r2 * r2);
        acc[3] += m * (vx * r1 + vy * r2);
        acc[4] += Mx * p1 + My * p2;
        acc[5] += p1;
        acc[6] += p2;
        if (wrow && x + h >= win.x0 && x + h <= win.x1) {
          acc[7] += p1; acc[8] += p2; acc[9] += vx * m; acc[10] += vy * m;
        }
        if (wrow2 && x + h >= win2.x0 && x + h <= win2.x1) {
          acc[11] += p1; acc[12] += p2; acc[13] += vx * m; acc[14] += vy * m;
        }
        if (h) { q1.y = p1; q2.y = p2; } else { q1.x = p1; q2.x = p2; }
      }
      if constexpr (PRES) {
        const double2 w = row[2 * PL + qn];
        row[qn] = make_double2(q1.x - w.x * a2.x, q1.y - w.y * a2.y);
        row[PL + qn] = make_double2(q2.x + w.x * a1.x, q2.y + w.y * a1.y);
      }
    }
  }
  // the row sums and the row's CFL maximum
  {
    if constexpr (WAVE) {
      um = seg_max<NR>(um);
      if (p == 0) a.umax_part[y] = um;
      // every lane of the wave takes part in the exchange as long as one of
      // its rows has the sum; the others' are exactly 0
#pragma unroll
      for (int i = 0; i < kNSUM; ++i) {
        double s = 0.0;
        if (i < 2 || __any(i < nv)) s = seg_sum<NR>(acc[i]);
        if (p == 0) a.sums[(size_t)y * kNSUM + i] = s;
      }
    } else {
      constexpr int nw = (NR + 63) / 64;
      static_assert(NR % 64 == 0, "whole waves");
      __shared__ double red[(kNSUM + 1) * nw];
      const int lane = tid & 63, wid = tid >> 6;
      um = wave_max(um);
      if (lane == 0) red[wid] = um;
      if (nv == kNSUM) wave_sums<kNSUM>(acc, red + nw, lane, wid, nw);
      else if (nv == kNSUM1) wave_sums<kNSUM1>(acc, red + nw, lane, wid, nw);
      else wave_sums<2>(acc, red + nw, lane, wid, nw);
      __syncthreads();
      if (tid == 0) {
        double m = 0.0;
        for (int q = 0; q < nw; ++q) m = fmax(m, red[q]);
        a.umax_part[y] = m;
      }
      if (tid < kNSUM) {
        double q = 0.0;
        if (tid < nv)
          for (int k = 0; k < nw; ++k) q += red[nw + tid * nw + k];
        a.sums[(size_t)y * kNSUM + tid] = q;
      }
    }
  }
  if constexpr (!PRES && !NEXT) return;
  grp_sync<WAVE>();
  // post-processing of a forward transform in buffer b, over the row's threads
  auto post = [&](auto nfc, int b, auto out) {
    constexpr int NF = decltype(nfc)::value;
#pragma unroll
    for (int k = 0; k < PN; ++k) {
      const int n = p + k * NR;
      if (H % NR != 0 && n >= H) continue;
      const int q = n == 0 ? 0 : H - n;
      const double2 wk = twx[n];
      double2 x[NF];
#pragma unroll
      for (int f = 0; f < NF; ++f) x[f] = r2c_one(row[(b + f) * PL + pidx(n)], row[(b + f) * PL + pidx(q)], wk);
      out(n, x);
    }
  };
  using One = std::integral_constant<int, 1>;
  using Two = std::integral_constant<int, 2>;
  // second round: forward transforms of the pressure right-hand sides (slots
  // 0, 1), and slot 2 the inverse of omega_y
  {
    const bool inv = NEXT && slot == 2;
    const bool act = (PRES && slot < 2) || inv;
    double2 in[NI];
    if constexpr (LEAN) asm volatile("" : "+v"(t));
    if (inv) {
      for_in([&](int q, int e) {
        if (LEAN && q % 2 == 0) __builtin_amdgcn_sched_barrier(0);
        in[q] = cconj(c2r_elem(live(a.Cwy + rowk, e, H, a.c.kc),
                               live(a.Cwy + rowk, e == 0 ? 0 : H - e, H, a.c.kc), e, cconj(twx[e])));
      });
    } else if (act) {
      for_in([&](int q, int e) { in[q] = xb[pidx(e)]; });
    }
    fft_io<H, NT, false, 1, WAVE, LEAN>(
        xb, T, t, act, [&](int i, int r, int) { return in[i * R0 + r]; },
        [&](int i, int r, int, double2 x) { z[i * Out::R + r] = inv ? cconj(x) : x; });
    grp_sync<WAVE>();
    if (act) put(z);
    grp_sync<WAVE>();
  }
  if constexpr (PRES)
    post(Two{}, 0, [&](int k, const double2 *x) {
      a.Rq[rowk + k] = mul_ik(x[0], (double)k * sx);
      a.Rqy[rowk + k] = x[1];
    });
  if constexpr (NEXT) {
#pragma unroll
    for (int k = 0; k < PN; ++k) {
      const int n = p + k * NR;
      if (H % NR != 0 && n >= H) continue;
      const double2 wy = row[2 * PL + pidx(n)], cv = row[3 * PL + pidx(n)];
      const double2 a2 = reinterpret_cast<const double2 *>(a.u2 + rowx)[n];  // as this thread stored it
      row[3 * PL + pidx(n)] = make_double2((cv.x - a2.x * wy.x) - csw[k].x, (cv.y - a2.y * wy.y) - csw[k].y);
    }
    grp_sync<WAVE>();
    const bool act = slot == 3;
    fft_io<H, NT, false, 1, WAVE, LEAN>(
        xb, T, t, act, [&](int, int, int e) { return xb[pidx(e)]; },
        [&](int i, int r, int, double2 x) { z[i * Out::R + r] = x; });
    grp_sync<WAVE>();
    if (act) put(z);
    grp_sync<WAVE>();
    post(One{}, 3, [&](int k, const double2 *x) { a.Rc[rowk + k] = x[0]; });
  }
}

template <int HC, int NTC, int RPBC, bool LEANC> struct RowStepShape {
  static constexpr int H = HC, NT = NTC, NS = 4, RPB = RPBC;
  static constexpr bool LEAN = LEANC;
  static constexpr int THREADS = NS * NT * RPB;
  static constexpr size_t LDS = sizeof(double2) * NS * padlen(H) * RPB;
};
// a lean shape is held to 128 VGPRs, so that four waves per SIMD hold every
// row of the grid at once
template <class S, bool PRES, bool NEXT>
__global__ void __launch_bounds__(S::THREADS) __attribute__((amdgpu_waves_per_eu(S::LEAN ? 4 : 1, 8)))
k_row_step(RowStepArgs a, const double2 *__restrict__ twx) {
  row_step_body<S::H, S::NT, S::RPB, S::LEAN, PRES, NEXT>(a, twx, blockIdx.x);
}
struct RowStepRec {
  RowStepArgs a;
  int nblk, pad;
};
template <class S, bool PRES>
__global__ void __launch_bounds__(S::THREADS) __attribute__((amdgpu_waves_per_eu(S::LEAN ? 4 : 1, 8)))
kb_row_step(const RowStepRec *__restrict__ arr, const double2 *__restrict__ twx) {
  const RowStepRec &r = arr[blockIdx.y];
  if ((int)blockIdx.x >= r.nblk) return;
  row_step_body<S::H, S::NT, S::RPB, S::LEAN, PRES, false>(r.a, twx, blockIdx.x);
}

}  // namespace fsibe

// fsibe_hip.hip -- host side of libfsibe_hip.so (C ABI in include/fsibe_hip.h)
//
// One HIP stream per handle.  Tier A (fsibe_spectral) is the reference's FFT
// and operator plugin on the packed layout; Tier B (fsibe_sim) keeps the
// fluid state in HBM as half spectra and runs the fused step pipeline of
// kernels_step.hpp.  The host computes, with the same libm calls the
// reference makes, everything that depends only on the beam (mask primitive
// geometry, interpolation targets, bounding boxes), uploads it in one copy per
// step, and reads back one small result record per step.
#include <hip/hip_runtime.h>
#include <hip/hip_ext.h>

#include <algorithm>
#include <array>
#include <atomic>
#include <chrono>
#include <cmath>
#include <condition_variable>
#include <functional>
#include <map>
#include <mutex>
#include <thread>
#include <cstdarg>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <string>
#include <vector>

#include "../../include/fsibe_hip.h"
#include "kernels.hpp"
#include "kernels_mask.hpp"
#include "kernels_step.hpp"
#include "kernels_fused.hpp"
#include "kernels_spectral.hpp"
#include "transfer.hpp"
#include "kernels_adjoint.hpp"
#include "kinematics.hpp"
#include "solid.hpp"
#include "wait.hpp"

using namespace fsibe;

// ---------------------------------------------------------------------------
// errors
// ---------------------------------------------------------------------------
static thread_local std::string g_err;

static int set_err(int code, const char *fmt, ...) {
  char buf[512];
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(buf, sizeof(buf), fmt, ap);
  va_end(ap);
  g_err = buf;
  return code;
}

extern "C" const char *fsibe_last_error(void) { return g_err.c_str(); }

#define HIPCHK(call)                                                                        \
  do {                                                                                      \
    hipError_t e_ = (call);                                                                 \
    if (e_ != hipSuccess)                                                                   \
      return set_err(FSIBE_EHIP, "%s failed: %s (%s:%d)", #call, hipGetErrorString(e_),    \
                     __FILE__, __LINE__);                                                   \
  } while (0)

#define CHK(call)                  \
  do {                             \
    int r_ = (call);               \
    if (r_ != FSIBE_OK) return r_; \
  } while (0)

// ---------------------------------------------------------------------------
// planning
// ---------------------------------------------------------------------------
// radices for length L: 3s, then a 16, 2 or 4 for the power of two left
// after the eights, then 8s (cp_radix); false if unsupported
static bool make_plan(int L, FftPlan &p) {
  p = FftPlan{};
  p.L = L;
  if (L < 1) return false;
  int m = L, n3 = 0, e2 = 0;
  while (m % 3 == 0) { m /= 3; ++n3; }
  while (m % 2 == 0) { m /= 2; ++e2; }
  if (m != 1) return false;
  std::vector<int> r;
  for (int i = 0; i < n3; ++i) r.push_back(3);
  int a = e2 / 3, b = e2 % 3;
  if (b == 1 && a >= 1) { a -= 1; r.push_back(16); }
  else if (b == 1) r.push_back(2);
  else if (b == 2) r.push_back(4);
  for (int i = 0; i < a; ++i) r.push_back(8);
  if ((int)r.size() > 16) return false;
  p.np = (int)r.size();
  for (int i = 0; i < p.np; ++i) p.r[i] = r[i];
  p.code = 0;
  for (int i = 0; i < p.np; ++i) p.code |= (unsigned long long)radix_code(r[i]) << (4 * i);
  return true;
}

static std::vector<double2> twiddles(int n) {
  std::vector<double2> t(n);
  const long double twopi = 6.283185307179586476925286766559005768L;
  for (int k = 0; k < n; ++k) {
    long double a = twopi * (long double)k / (long double)n;
    t[k] = make_double2((double)cosl(a), (double)(-sinl(a)));
  }
  return t;
}

// Launch shape of a transform kernel holding `elems` complex values in LDS:
// the workgroup grows to 1024 threads while every thread still holds at least
// 4 values (more waves per CU to hide LDS and memory latency); EMAX is the
// per-thread bound rounded up to an instantiated value.
struct Shape {
  int nt, emax;
};

static bool has_radix16(const FftPlan &p) {
  for (int i = 0; i < p.np; ++i)
    if (p.r[i] == 16) return true;
  return false;
}

static Shape shape_of(long long elems, bool r16) {
  // one radix-8 butterfly per thread: nt ~ elems / 8, between 256 and 1024;
  // a plan with a radix-16 pass runs on the 256-thread instances (EMAX 16
  // or 32), the only ones whose passes include the 16-point butterfly
  if (r16) {
    const long long e = (elems + kNT - 1) / kNT;
    return Shape{kNT, e <= 16 ? 16 : e <= 32 ? 32 : -1};
  }
  int nt = kNT;
  while (nt < 1024 && elems >= 16LL * nt) nt *= 2;
  long long e = (elems + nt - 1) / nt;
  int em = e <= 4 ? 4 : e <= 8 ? 8 : e <= 16 ? 16 : e <= 32 ? 32 : -1;
  if (em > 8 && nt > kNT) {  // EMAX 16/32 instances are bounded to 256 threads
    nt = kNT;
    e = (elems + nt - 1) / nt;
    em = e <= 16 ? 16 : e <= 32 ? 32 : -1;
  }
  return Shape{nt, em};
}

static int lds_limit() {
  static int lim = -1;
  if (lim < 0) {
    int dev = 0, v = 0;
    (void)hipGetDevice(&dev);
    if (hipDeviceGetAttribute(&v, hipDeviceAttributeMaxSharedMemoryPerBlock, dev) != hipSuccess || v <= 0)
      v = 65536;
    lim = v;
  }
  return lim;
}

template <typename K>
static int prep_lds(K kernel, size_t lds) {
  if (lds > (size_t)lds_limit())
    return set_err(FSIBE_ESIZE, "tile needs %zu bytes of LDS (limit %d)", lds, lds_limit());
  if (lds > 65536) {
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(kernel),
                                       hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return set_err(FSIBE_EHIP, "hipFuncSetAttribute: %s", hipGetErrorString(e));
  }
  return FSIBE_OK;
}

// ---- policy dispatch --------------------------------------------------------
// Sizes with a compile-time plan: the transform's index arithmetic folds to
// constants.  Other sizes (any 2^a 3^b) run the runtime-plan kernels.
constexpr int ct_nt(int butterflies, int cap) {
  int nt = 64;
  while (nt < butterflies && nt < cap) nt *= 2;
  return nt;
}
constexpr int ct_tx(int ny) { return (ny == 1024 || ny == 2048) ? 2 : 1; }

// threads of a row workgroup: one per radix-8 butterfly, at most 256, or
// at most 1024 for rows of 1024 complex values and more, whose LDS
// footprint (three sequences: 55-110 KB) leaves room for one or two
// workgroups per CU, which then need enough waves of their own
constexpr int row_nt(int H, int nseq) { return ct_nt(H * nseq / 8, H >= 1024 ? 1024 : 256); }

// fn(policy, nthreads) for row transforms of length H holding NSEQ sequences
template <int NSEQ, class Fn>
static int with_rows(const FftPlan &px, Fn &&fn) {
  switch (px.L) {
#define ROWCASE(HH) \
    case HH: return fn(RowCT<HH, row_nt(HH, NSEQ)>{px}, row_nt(HH, NSEQ));
    ROWCASE(64) ROWCASE(128) ROWCASE(192) ROWCASE(256) ROWCASE(384) ROWCASE(512) ROWCASE(1024) ROWCASE(2048)
#undef ROWCASE
    default: break;
  }
  const Shape sh = shape_of((long long)NSEQ * px.L, has_radix16(px));
  switch (sh.emax) {
    case 4: return fn(RowRT<4>{px}, sh.nt);
    case 8: return fn(RowRT<8>{px}, sh.nt);
    case 16: return fn(RowRT<16>{px}, sh.nt);
    case 32: return fn(RowRT<32>{px}, sh.nt);
    default: return set_err(FSIBE_ESIZE, "row transform of %d x %d too large", NSEQ, px.L);
  }
}

// fn(policy, nthreads, TX) for column tiles of length NY, BM fields per tile
template <int BM, class Fn>
static int with_cols(const FftPlan &py, int H, int rt_tx, Fn &&fn) {
  switch (py.L) {
#define COLCASE(NN)                                                                              \
    case NN:                                                                                     \
      if (H % ct_tx(NN) == 0)                                                                    \
        return fn(ColCT<NN, ct_tx(NN), ct_nt(NN * ct_tx(NN) * BM / 8, 1024)>{py, ct_tx(NN)},     \
                  ct_nt(NN * ct_tx(NN) * BM / 8, 1024), ct_tx(NN));                              \
      break;
    COLCASE(128) COLCASE(256) COLCASE(384) COLCASE(512) COLCASE(768) COLCASE(1024) COLCASE(2048) COLCASE(4096)
#undef COLCASE
    default: break;
  }
  const Shape sh = shape_of((long long)BM * rt_tx * py.L, has_radix16(py));
  switch (sh.emax) {
    case 4: return fn(ColRT<4>{py, rt_tx}, sh.nt, rt_tx);
    case 8: return fn(ColRT<8>{py, rt_tx}, sh.nt, rt_tx);
    case 16: return fn(ColRT<16>{py, rt_tx}, sh.nt, rt_tx);
    case 32: return fn(ColRT<32>{py, rt_tx}, sh.nt, rt_tx);
    default: return set_err(FSIBE_ESIZE, "column tile of %d x %d too large", BM * rt_tx, py.L);
  }
}

// A launch choice of a column stage: the compile-time plan (ct = 1) or the
// runtime plan (ct = 0), with tx columns per tile.  Every choice runs the
// same radix passes with the same twiddles on each column, so the choice
// changes the speed, never the result.
struct ColSel {
  int ct, tx;
};

// compile-time instances with other tile widths than ct_tx: the grid sizes
// of uneven batches, where the best width depends on how many simulations
// share a launch
constexpr bool ct_extra(int ny, int tx) {
  return ((ny == 256 || ny == 384 || ny == 512 || ny == 768) && (tx == 2 || tx == 4)) ||
         (ny == 1024 && (tx == 1 || tx == 4)) || (ny == 2048 && tx == 1) || (ny == 4096 && tx == 2);
}

static bool col_sel_valid(int ny, int H, int bm, ColSel c) {
  if (c.tx < 1 || H % c.tx) return false;
  if ((size_t)c.tx * bm * padlen(ny) * sizeof(double2) > (size_t)lds_limit()) return false;
  if (c.ct) {
    switch (ny) {
      case 128: case 256: case 384: case 512: case 768: case 1024: case 2048: case 4096: break;
      default: return false;
    }
    return c.tx == ct_tx(ny) || ct_extra(ny, c.tx);
  }
  FftPlan pl;
  make_plan(ny, pl);
  return shape_of((long long)bm * c.tx * ny, has_radix16(pl)).emax > 0;
}

// K4 (launched through with_cols_sel<2>) holds two fields per column when
// some member has penalisation (px), else one: its tiles' LDS is sized by
// that, and a runtime-plan choice must also have a launch shape for two
static bool k4_sel_valid(int ny, int H, bool px, ColSel c) {
  if (!col_sel_valid(ny, H, px ? 2 : 1, c)) return false;
  if (c.ct) return true;
  FftPlan pl;
  make_plan(ny, pl);
  return shape_of(2LL * c.tx * ny, has_radix16(pl)).emax > 0;
}
static size_t k4_lds(int ny, bool px, int TX) { return sizeof(double2) * (px ? 2 : 1) * TX * padlen(ny); }

// fn(policy, nthreads, TX) for the column stage launch choice `sel`
// (col_sel_valid must hold)
template <int BM, class Fn>
static int with_cols_sel(const FftPlan &py, int H, ColSel sel, Fn &&fn) {
  if (sel.ct && sel.tx == ct_tx(py.L) && H % sel.tx == 0) return with_cols<BM>(py, H, sel.tx, fn);
  if (sel.ct) {
    switch (py.L * 8 + sel.tx) {
#define COLSEL(NN, TT) \
      case NN * 8 + TT: return fn(ColCT<NN, TT, ct_nt(NN * TT * BM / 8, 1024)>{py, TT}, ct_nt(NN * TT * BM / 8, 1024), TT);
      COLSEL(256, 2) COLSEL(256, 4) COLSEL(384, 2) COLSEL(384, 4) COLSEL(512, 2) COLSEL(512, 4) COLSEL(768, 2)
      COLSEL(768, 4) COLSEL(1024, 1) COLSEL(1024, 4) COLSEL(2048, 1) COLSEL(4096, 2)
#undef COLSEL
      default: return set_err(FSIBE_ESIZE, "no compile-time column plan for %d x %d", py.L, sel.tx);
    }
  }
  const Shape sh = shape_of((long long)BM * sel.tx * py.L, has_radix16(py));
  switch (sh.emax) {
    case 4: return fn(ColRT<4>{py, sel.tx}, sh.nt, sel.tx);
    case 8: return fn(ColRT<8>{py, sel.tx}, sh.nt, sel.tx);
    case 16: return fn(ColRT<16>{py, sel.tx}, sh.nt, sel.tx);
    case 32: return fn(ColRT<32>{py, sel.tx}, sh.nt, sel.tx);
    default: return set_err(FSIBE_ESIZE, "column tile of %d x %d too large", BM * sel.tx, py.L);
  }
}

// Kernel timing (fsibe_profile_enable): a profiled region arms its event pair
// here, and its first KLAUNCH launches with hipExtLaunchKernelGGL, which
// records the pair at the kernel's own start and end.  An event pair
// recorded around a launch would also time the launch's dispatch.  A region
// with one launch is timed by the kernel alone; with several, from the
// first kernel's start to an event after the last launch.
static thread_local hipEvent_t t_prof_start = nullptr, t_prof_stop = nullptr;
static thread_local int t_prof_launches = 0;

#define KLAUNCH(KT, grid, nt, lds, st, ...)                                                             \
  do {                                                                                                  \
    CHK(prep_lds(KT, lds));                                                                             \
    if (t_prof_start && t_prof_launches++ == 0)                                                         \
      hipExtLaunchKernelGGL(KT, dim3(grid), dim3(nt), (std::uint32_t)(lds), st, t_prof_start, t_prof_stop, \
                            0u, __VA_ARGS__);                                                           \
    else                                                                                                \
      KT<<<grid, nt, lds, st>>>(__VA_ARGS__);                                                           \
    HIPCHK(hipGetLastError());                                                                          \
  } while (0)

// KLAUNCH whose kernel also records `ev` at its end, carried by its own
// dispatch: an event recorded between two kernels is a marker that stalls
// the queue until the first has drained (~5.6 us per marker measured in the
// step's kernel traces).  Under kernel timing the launch keeps KLAUNCH's
// events and `ev` is recorded after it.
#define KLAUNCH_EV(KT, grid, nt, lds, st, ev, ...)                                                      \
  do {                                                                                                  \
    if (t_prof_start) {                                                                                 \
      KLAUNCH(KT, grid, nt, lds, st, __VA_ARGS__);                                                      \
      HIPCHK(hipEventRecord(ev, st));                                                                   \
    } else {                                                                                            \
      CHK(prep_lds(KT, lds));                                                                           \
      hipExtLaunchKernelGGL(KT, dim3(grid), dim3(nt), (std::uint32_t)(lds), st, nullptr, ev, 0u, __VA_ARGS__); \
      HIPCHK(hipGetLastError());                                                                        \
    }                                                                                                   \
  } while (0)

static int env_int(const char *name, int dflt) {
  const char *v = getenv(name);
  return v ? atoi(v) : dflt;
}

// columns per tile for a column kernel holding `nfld` fields of length ny
static int pick_tx(int H, int ny, int nfld, int split) {
  int forced = env_int("FSIBE_TX", 0);
  if (forced > 0 && H % forced == 0 && (long long)forced * nfld * ny <= 32LL * kNT) return forced;
  int best = 1;
  for (int tx = 1; tx <= 16; tx *= 2) {
    if (H % tx) break;
    if ((long long)tx * nfld * ny > 32LL * kNT) break;
    if ((size_t)tx * nfld * padlen(ny) * sizeof(double2) > (size_t)lds_limit()) break;
    if ((long long)(H / tx) * split < 256 && tx > 1) break;
    if (tx > 1 && (size_t)tx * nfld * padlen(ny) * sizeof(double2) > 73728) break;
    best = tx;
  }
  return best;
}

static bool size_ok(int nx, int ny) {
  FftPlan a, b;
  return nx >= 4 && ny >= 4 && nx % 2 == 0 && ny % 2 == 0 && make_plan(nx / 2, a) && make_plan(ny, b);
}

// fn(shape) for the fused column stage (K4, K5 and the dw/dy column) of
// columns of length ny; false if the grid has none (the separate stages run).
// The shapes follow from what a workgroup holds: four slots of one column up
// to 512 points, of two columns (32-byte row pieces) at 768 and 1024, two
// slots of two columns at 1536, and one buffer of two columns beyond, where
// the fields follow one another.  Both sides measured on square grids (one
// simulation, K4 + K5 with four fields + the dw/dy column of K1, us):
// 256^2 19.0 -> 7.2, 384^2 22.9 -> 11.3, 512^2 21.3 -> 11.7, 768^2 30.7 ->
// 22.1, 1024^2 37.9 -> 26.0, 2048^2 131 -> 125.
// Columns of 4096 points, where px leaves no room: two columns a workgroup
// with their fields one after another are too few workgroups below 192
// columns, where the separate stages spread the fields over more.  A step of a
// flow without a body, with the stages separate and fused, us: 64 columns 104
// and 113 (one step a call: 127 and 144), 128 columns 127 and 129 (151 and
// 160), 192 columns 139 and 127 (163 and 158).  next: the next step's terms are
// formed too, which pays below 192 columns as well where the rows would need a
// run-time plan for them (32 columns 108 and 85, 96: 138 and 102, 108: 177
// and 157; 16 and 24: 200 and 204, 139 and 143).
template <class Fn>
static bool with_col_step(int ny, int H, bool px, bool next, Fn &&fn) {
  switch (ny) {
    case 64: fn(ColStepShape<64, 1, 8, 4, false>{}); return true;
    case 96: fn(ColStepShape<96, 1, 12, 4, false>{}); return true;
    case 128: fn(ColStepShape<128, 1, 16, 4, false>{}); return true;
    case 192: fn(ColStepShape<192, 1, 24, 4, false>{}); return true;
    case 256: fn(ColStepShape<256, 1, 32, 4, false>{}); return true;
    case 384: fn(ColStepShape<384, 1, 48, 4, false>{}); return true;
    case 512: fn(ColStepShape<512, 1, 64, 4, false>{}); return true;
    default: break;
  }
  if (H % 2) return false;
  switch (ny) {
    case 768: fn(ColStepShape<768, 2, 96, 4, true>{}); return true;
    case 1024: fn(ColStepShape<1024, 2, 128, 4, true>{}); return true;
    case 1536: fn(ColStepShape<1536, 2, 192, 2, true>{}); return true;
    case 2048:
      if (px) fn(ColStepShape<2048, 2, 256, 0, true>{});
      else fn(ColStepShape<2048, 2, 256, 0, false>{});
      return true;
    case 4096:
      if (px || (H < 192 && !(next && H >= 32 && H != 64 && H != 128))) return false;
      fn(ColStepShape<4096, 2, 512, 0, false>{});
      return true;
    default: return false;
  }
}

// fn(shape) for the pressure stage (K7) of columns of ny values; false if
// there is none (odd H, other lengths, and columns whose two buffers leave
// one workgroup on a CU)
template <class Fn>
static bool with_press_step(int ny, int H, Fn &&fn) {
  if (H % 2) return false;
  switch (ny) {
    case 64: fn(PressShape<64, 2, 8>{}); return true;
    case 96: fn(PressShape<96, 2, 12>{}); return true;
    case 128: fn(PressShape<128, 2, 16>{}); return true;
    case 192: fn(PressShape<192, 2, 24>{}); return true;
    case 256: fn(PressShape<256, 2, 32>{}); return true;
    case 384: fn(PressShape<384, 2, 48>{}); return true;
    case 512: fn(PressShape<512, 2, 64>{}); return true;
    case 768: fn(PressShape<768, 2, 96>{}); return true;
    case 1024: fn(PressShape<1024, 2, 128>{}); return true;
    case 1536: fn(PressShape<1536, 2, 192>{}); return true;
    default: return false;
  }
}

// transform lengths that a policy fixes at compile time (0: a runtime plan),
// so that the fallbacks below are not instantiated where they cannot run
template <class F> struct fixed_len { static constexpr int v = 0; };
template <int H, int NT> struct fixed_len<RowCT<H, NT>> { static constexpr int v = H; };
template <int NY, int TX, int NT> struct fixed_len<ColCT<NY, TX, NT>> { static constexpr int v = NY; };
constexpr bool always_col_step(int ny) { return ny == 128 || ny == 256 || ny == 384 || ny == 512; }
constexpr bool always_row_step(int H) { return H == 192 || H == 256; }

// fn(shape) for the fused row stage (K6 and, with NEXT, the convective part of
// the next K2) of rows of H complex values on ny rows; false if there is none.
// Rows of 128 without NEXT: the stage's one wave a row, of which a quarter
// has no transform then, against K6 alone, us, 256, 1024, 2048 and 4096 rows:
// 8.3, 11.1, 16.5, 25.4 and 7.3, 9.5, 14.8, 23.6; with the pressure (pres) 11.6, 15.2,
// 20.8, 31.0 and 11.4, 14.5, 20.6, 25.2, where only the last shows in a step.
// Rows of 512 without NEXT: four workgroups of the stage fit a CU, six of K6
// alone, so that beyond 1024 rows the stage goes in rounds.  Without the
// pressure that is slower, with it where the last round is a quarter or
// less.  Stage and K6 alone at 1024, 1152, 1296, 2048, 2304 and 4096 rows: 15.6, 19.3,
// 20.2, 27.6, -, 51.9 and 16.3, 17.1, 20.6, 25.9, -, 49.9; with the pressure 20.4, 25.1,
// 27.4, 36.8, 41.6, 69.7 and 22.6, 23.4, 28.5, 37.6, 39.2, 70.3.
// Lengths without a shape: 384, 37 us against 30 of K6 and K2 at 768 x 768; 1024
// and more, whose four buffers leave one or two rows on a CU (2048^2: 112 to 200 us
// in the shapes tried, K6 80 and K2 54); 48, 768 and lengths with a 9: not tried.
template <bool NEXT, class Fn>
static bool with_row_step(int H, int ny, bool pres, Fn &&fn) {
  switch (H) {
    case 32:
      if (ny % 4) return false;
      fn(RowStepShape<32, 4, 4, false>{});
      return true;
    case 64:
      if (ny % 2) return false;
      fn(RowStepShape<64, 8, 2, false>{});
      return true;
    case 96: fn(RowStepShape<96, 16, 1, false>{}); return true;
    case 128:
      if (!NEXT && (!pres || ny > 2048)) return false;
      fn(RowStepShape<128, 16, 1, false>{});
      return true;
    case 192: fn(RowStepShape<192, 32, 1, false>{}); return true;
    case 256: fn(RowStepShape<256, 32, 1, false>{}); return true;
    case 512:
      if (!NEXT && ny > 1024 && (!pres || (ny - 1) % 1024 < 256)) return false;
      fn(RowStepShape<512, 64, 1, true>{});
      return true;
    default: return false;
  }
}

// ---------------------------------------------------------------------------
// Tier A
// ---------------------------------------------------------------------------
struct fsibe_spectral {
  int nx, ny, H;
  double xl, yl, nu, pi, scalex, scaley;
  FftPlan px, py;
  hipStream_t stream;
  double2 *twx, *twy, *tmp;
  double *hbuf_in, *hbuf_out;  // device staging for host-pointer calls
};

static PackedDims packed_dims(const fsibe_spectral *c) {
  PackedDims d;
  d.nx = c->nx; d.ny = c->ny;
  d.sx = 2.0 * c->pi / c->xl;
  d.sy = 2.0 * c->pi / c->yl;
  d.scalex = c->scalex; d.scaley = c->scaley;
  return d;
}

extern "C" int fsibe_spectral_create(int nx, int ny, double xl, double yl, double nu, fsibe_spectral **out) {
  if (!out) return set_err(FSIBE_EARG, "out is NULL");
  *out = nullptr;
  if (!size_ok(nx, ny))
    return set_err(FSIBE_ESIZE, "grid %dx%d not supported (even sizes, nx/2 and ny = 2^a 3^b)", nx, ny);
  if (!(xl > 0.0) || !(yl > 0.0)) return set_err(FSIBE_EARG, "domain size must be positive");
  fsibe_spectral *c = new fsibe_spectral();
  c->nx = nx; c->ny = ny; c->H = nx / 2;
  c->xl = xl; c->yl = yl; c->nu = nu;
  c->pi = 4.0 * atan(1.0);
  { double a = 2.0 * c->pi / xl; c->scalex = a * a; }
  { double a = 2.0 * c->pi / yl; c->scaley = a * a; }
  make_plan(c->H, c->px);
  make_plan(ny, c->py);
  HIPCHK(hipStreamCreate(&c->stream));
  auto tx = twiddles(nx), ty = twiddles(ny);
  HIPCHK(hipMalloc(&c->twx, sizeof(double2) * nx));
  HIPCHK(hipMalloc(&c->twy, sizeof(double2) * ny));
  HIPCHK(hipMemcpy(c->twx, tx.data(), sizeof(double2) * nx, hipMemcpyHostToDevice));
  HIPCHK(hipMemcpy(c->twy, ty.data(), sizeof(double2) * ny, hipMemcpyHostToDevice));
  size_t N = (size_t)nx * ny;
  HIPCHK(hipMalloc(&c->tmp, sizeof(double2) * (N / 2)));
  HIPCHK(hipMalloc(&c->hbuf_in, sizeof(double) * N));
  HIPCHK(hipMalloc(&c->hbuf_out, sizeof(double) * N));
  *out = c;
  return FSIBE_OK;
}

extern "C" int fsibe_spectral_destroy(fsibe_spectral *c) {
  if (!c) return FSIBE_OK;
  (void)hipStreamSynchronize(c->stream);
  (void)hipFree(c->twx); (void)hipFree(c->twy); (void)hipFree(c->tmp);
  (void)hipFree(c->hbuf_in); (void)hipFree(c->hbuf_out);
  (void)hipStreamDestroy(c->stream);
  delete c;
  return FSIBE_OK;
}

// fn(shape) for row transforms of H complex values; false if there is none.
// Threads and rows per workgroup are the fastest measured: H/4 threads a row up
// to 256 values and H/8 from 512 on, H/3 or H/6 where the length holds a 3.
template <class Fn>
static bool with_rows_io(int H, Fn &&fn) {
  switch (H) {
    case 32: fn(RowsShape<32, 8, 8>{}); return true;
    case 48: fn(RowsShape<48, 16, 4>{}); return true;
    case 64: fn(RowsShape<64, 16, 4>{}); return true;
    case 96: fn(RowsShape<96, 32, 2>{}); return true;
    case 128: fn(RowsShape<128, 32, 2>{}); return true;
    case 192: fn(RowsShape<192, 32, 2>{}); return true;
    case 256: fn(RowsShape<256, 64, 1>{}); return true;
    case 384: fn(RowsShape<384, 64, 1>{}); return true;
    case 512: fn(RowsShape<512, 64, 1>{}); return true;
    case 768: fn(RowsShape<768, 256, 1>{}); return true;
    case 1024: fn(RowsShape<1024, 128, 1>{}); return true;
    default: return false;
  }
}
// fixed-length row policies whose length always has such a shape
constexpr bool always_rows_io(int H) {
  return H == 64 || H == 128 || H == 192 || H == 256 || H == 384 || H == 512 || H == 1024;
}

// fn(shape) for column transforms of ny values; false if there is none.  Two
// columns per workgroup, except where four were faster (384: 17.2 against
// 20.0 us for both directions of 384^2).
template <class Fn>
static bool with_cols_io(int ny, int H, Fn &&fn) {
  if (H % 4 == 0 && ny == 384) { fn(ColsShape<384, 4, 48>{}); return true; }
  if (H % 2) return false;
  switch (ny) {
    case 64: fn(ColsShape<64, 2, 16>{}); return true;
    case 96: fn(ColsShape<96, 2, 24>{}); return true;
    case 128: fn(ColsShape<128, 2, 32>{}); return true;
    case 192: fn(ColsShape<192, 2, 24>{}); return true;
    case 256: fn(ColsShape<256, 2, 32>{}); return true;
    case 512: fn(ColsShape<512, 2, 64>{}); return true;
    case 768: fn(ColsShape<768, 2, 96>{}); return true;
    case 1024: fn(ColsShape<1024, 2, 128>{}); return true;
    case 1536: fn(ColsShape<1536, 2, 192>{}); return true;
    case 2048: fn(ColsShape<2048, 2, 256>{}); return true;
    default: return false;
  }
}

// fn(shape) for a grid in one workgroup, 64 x 64, 128 x 32 and 64 x 32; false for
// the others (twice the entries gain nothing: kernels_spectral.hpp)
template <class Fn>
static bool with_small(int H, int ny, Fn &&fn) {
  if (H == 32 && ny == 64) { fn(SmallShape<32, 64, 4, 8, 512>{}); return true; }
  if (H == 64 && ny == 32) { fn(SmallShape<64, 32, 8, 4, 512>{}); return true; }
  if (H == 32 && ny == 32) { fn(SmallShape<32, 32, 4, 4, 256>{}); return true; }
  return false;
}

// real rows -> half spectrum (unnormalised)
static int rows_r2c(int nx, int ny, const FftPlan &px, const double2 *twx, const double *f, double2 *out,
                    hipStream_t st) {
  int rc = FSIBE_OK;
  if (with_rows_io(nx / 2, [&](auto S) {
        using ST = decltype(S);
        rc = [&]() -> int {
          KLAUNCH(k_rows_fwd<ST>, (ny + ST::RPB - 1) / ST::RPB, ST::THREADS, ST::LDS, st, f, out, twx, ny);
          return FSIBE_OK;
        }();
      }))
    return rc;
  const size_t lds = sizeof(double2) * padlen(nx / 2);
  return with_rows<1>(px, [&](auto F, int nt) -> int {
    if constexpr (!always_rows_io(fixed_len<decltype(F)>::v)) KLAUNCH(k_rows_r2c<decltype(F)>, ny, nt, lds, st, f, out, F, twx);
    return FSIBE_OK;
  });
}

static int rows_c2r(int nx, int ny, const FftPlan &px, const double2 *twx, const double2 *in, double *f,
                    hipStream_t st) {
  int rc = FSIBE_OK;
  if (with_rows_io(nx / 2, [&](auto S) {
        using ST = decltype(S);
        rc = [&]() -> int {
          KLAUNCH(k_rows_inv<ST>, (ny + ST::RPB - 1) / ST::RPB, ST::THREADS, ST::LDS, st, in, f, twx, ny);
          return FSIBE_OK;
        }();
      }))
    return rc;
  const size_t lds = sizeof(double2) * padlen(nx / 2);
  return with_rows<1>(px, [&](auto F, int nt) -> int {
    if constexpr (!always_rows_io(fixed_len<decltype(F)>::v)) KLAUNCH(k_rows_c2r<decltype(F)>, ny, nt, lds, st, in, f, F, twx);
    return FSIBE_OK;
  });
}

// columns of the half spectrum in -> packed layout, and back
static int cols_pack(int H, int ny, const FftPlan &py, const double2 *twy, const double2 *in, double *fk,
                     hipStream_t st) {
  const double norm = 1.0 / ((double)(2 * H) * (double)ny);
  int rc = FSIBE_OK;
  if (with_cols_io(ny, H, [&](auto S) {
        using ST = decltype(S);
        rc = [&]() -> int {
          KLAUNCH(k_cols_fwd<ST>, H / ST::TX, ST::THREADS, ST::LDS, st, in, fk, twy, H, norm);
          return FSIBE_OK;
        }();
      }))
    return rc;
  return with_cols<1>(py, H, pick_tx(H, ny, 1, 1), [&](auto F, int nt, int TX) -> int {
    const size_t lds = sizeof(double2) * TX * padlen(ny);
    KLAUNCH(k_cols_fwd_pack<decltype(F)>, H / TX, nt, lds, st, in, fk, F, twy, H, norm);
    return FSIBE_OK;
  });
}
static int cols_unpack(int H, int ny, const FftPlan &py, const double2 *twy, const double *fk, double2 *out,
                       hipStream_t st) {
  int rc = FSIBE_OK;
  if (with_cols_io(ny, H, [&](auto S) {
        using ST = decltype(S);
        rc = [&]() -> int {
          KLAUNCH(k_cols_inv<ST>, H / ST::TX, ST::THREADS, ST::LDS, st, fk, out, twy, H);
          return FSIBE_OK;
        }();
      }))
    return rc;
  return with_cols<1>(py, H, pick_tx(H, ny, 1, 1), [&](auto F, int nt, int TX) -> int {
    const size_t lds = sizeof(double2) * TX * padlen(ny);
    KLAUNCH(k_cols_unpack_inv<decltype(F)>, H / TX, nt, lds, st, fk, out, F, twy, H);
    return FSIBE_OK;
  });
}

static int dev_coftxy(fsibe_spectral *c, const double *f, double *fk, hipStream_t st) {
  int rc = FSIBE_OK;
  if (with_small(c->H, c->ny, [&](auto S) {
        using ST = decltype(S);
        rc = [&]() -> int {
          KLAUNCH(k_fwd2d<ST>, 1, ST::THREADS, ST::LDSF, st, f, fk, c->twx, c->twy,
                  1.0 / ((double)c->nx * (double)c->ny));
          return FSIBE_OK;
        }();
      }))
    return rc;
  CHK(rows_r2c(c->nx, c->ny, c->px, c->twx, f, c->tmp, st));
  return cols_pack(c->H, c->ny, c->py, c->twy, c->tmp, fk, st);
}

static int dev_cofitxy(fsibe_spectral *c, const double *fk, double *f, hipStream_t st) {
  int rc = FSIBE_OK;
  if (with_small(c->H, c->ny, [&](auto S) {
        using ST = decltype(S);
        rc = [&]() -> int {
          KLAUNCH(k_inv2d<ST>, 1, ST::THREADS, ST::LDSI, st, fk, f, c->twx, c->twy);
          return FSIBE_OK;
        }();
      }))
    return rc;
  CHK(cols_unpack(c->H, c->ny, c->py, c->twy, fk, c->tmp, st));
  return rows_c2r(c->nx, c->ny, c->px, c->twx, c->tmp, f, st);
}

static int grid1d(size_t n) { return (int)std::min<size_t>((n + 255) / 256, 4096); }

static int dev_op(fsibe_spectral *c, int which, const double *in, double *out, hipStream_t st) {
  PackedDims d = packed_dims(c);
  if (which == 0) {
    k_cofdx<<<grid1d((size_t)c->H * c->ny), 256, 0, st>>>(in, out, d);
  } else if (which == 1) {
    k_cofdy<<<grid1d((size_t)c->nx * (c->ny / 2)), 256, 0, st>>>(in, out, d);
  } else if (which >= 2 && which <= 5) {
    k_block_op<<<grid1d((size_t)c->H * (c->ny / 2)), 256, 0, st>>>(in, out, d, which);
  } else {
    return set_err(FSIBE_EARG, "unknown operator %d", which);
  }
  HIPCHK(hipGetLastError());
  return FSIBE_OK;
}

static int dev_vis(fsibe_spectral *c, double dt, double *work, hipStream_t st) {
  PackedDims d = packed_dims(c);
  const double coefx = -(dt * c->nu * c->scalex), coefy = -(dt * c->nu * c->scaley);
  k_vis<<<grid1d((size_t)c->H * (c->ny / 2)), 256, 0, st>>>(work, d, coefx, coefy);
  HIPCHK(hipGetLastError());
  return FSIBE_OK;
}

static hipStream_t pick_stream(fsibe_spectral *c, void *s) { return s ? (hipStream_t)s : c->stream; }

extern "C" int fsibe_dev_coftxy(fsibe_spectral *c, const double *d_f, double *d_fk, void *s) {
  if (!c || !d_f || !d_fk) return set_err(FSIBE_EARG, "null argument");
  return dev_coftxy(c, d_f, d_fk, pick_stream(c, s));
}
extern "C" int fsibe_dev_cofitxy(fsibe_spectral *c, const double *d_fk, double *d_f, void *s) {
  if (!c || !d_f || !d_fk) return set_err(FSIBE_EARG, "null argument");
  return dev_cofitxy(c, d_fk, d_f, pick_stream(c, s));
}
extern "C" int fsibe_dev_spectral_op(fsibe_spectral *c, int which, const double *d_in, double *d_out, void *s) {
  if (!c || !d_in || !d_out) return set_err(FSIBE_EARG, "null argument");
  return dev_op(c, which, d_in, d_out, pick_stream(c, s));
}
extern "C" int fsibe_dev_vis(fsibe_spectral *c, double dt, double *d_work, void *s) {
  if (!c || !d_work) return set_err(FSIBE_EARG, "null argument");
  return dev_vis(c, dt, d_work, pick_stream(c, s));
}
extern "C" int fsibe_spectral_sync(fsibe_spectral *c) {
  if (!c) return set_err(FSIBE_EARG, "null context");
  HIPCHK(hipStreamSynchronize(c->stream));
  return FSIBE_OK;
}

// ---- coftxy without allocation ----------------------------------------------
// For callers that cannot allocate device memory (code under HIP graph
// capture, serving loops, harnesses that forbid hipMalloc):
// fsibe_dev_coftxy_noalloc runs the kernels of fsibe_dev_coftxy with the
// intermediate half spectrum and the two twiddle tables in `scratch`, a
// static device array of the library (each GPU holds its own copy until the
// process ends).  Layout in double2 elements: the half spectrum
// [0, kNaMaxPoints/2), then the x table (nx values), then the y table (ny
// values).  Every element the kernels read is written first by the same
// call, so nothing needs clearing.  Calls that overlap on one GPU race on it.
static constexpr long long kNaMaxPoints = 2048LL * 2048LL;  // nx * ny
static constexpr int kNaMaxLen = 4096;                       // nx and ny each
static constexpr size_t kNaElems = (size_t)(kNaMaxPoints / 2) + 2 * (size_t)kNaMaxLen;
static __device__ __align__(256) double2 scratch[kNaElems];

// the device address of `scratch` per device (hipGetSymbolAddress once per
// device, with that device current); the array's name is only a host-side
// stand-in and is never passed to a kernel or copy
static std::mutex g_na_mu;
static std::map<int, double2 *> g_na_ptr;
// the sizes whose twiddle tables a device's scratch holds (so repeated calls
// of one size upload them once)
static std::map<int, std::pair<int, int>> g_na_tw;

static int noalloc_scratch(int dev, double2 **out) {
  std::lock_guard<std::mutex> g(g_na_mu);
  auto it = g_na_ptr.find(dev);
  if (it != g_na_ptr.end()) {
    *out = it->second;
    return FSIBE_OK;
  }
  double2 *ptr = nullptr;
  const hipError_t e = hipGetSymbolAddress(reinterpret_cast<void **>(&ptr), HIP_SYMBOL(scratch));
  if (e != hipSuccess || !ptr)
    return set_err(FSIBE_EHIP, "hipGetSymbolAddress(scratch) on device %d: %s", dev, hipGetErrorString(e));
  g_na_ptr[dev] = ptr;
  *out = ptr;
  return FSIBE_OK;
}

extern "C" int fsibe_dev_coftxy_noalloc(int nx, int ny, const double *d_f, double *d_fk, void *s) {
  if (!d_f || !d_fk) return set_err(FSIBE_EARG, "null argument");
  if (!size_ok(nx, ny))
    return set_err(FSIBE_ESIZE, "grid %dx%d not supported (even sizes, nx/2 and ny = 2^a 3^b)", nx, ny);
  if ((long long)nx * ny > kNaMaxPoints || nx > kNaMaxLen || ny > kNaMaxLen)
    return set_err(FSIBE_ESIZE, "grid %dx%d exceeds the static buffer of fsibe_dev_coftxy_noalloc "
                   "(nx*ny <= %lld, nx, ny <= %d)", nx, ny, kNaMaxPoints, kNaMaxLen);
  int dev = 0;
  HIPCHK(hipGetDevice(&dev));
  double2 *ptr = nullptr;
  CHK(noalloc_scratch(dev, &ptr));
  const hipStream_t st = (hipStream_t)s;
  double2 *tmp = ptr, *twx = ptr + kNaMaxPoints / 2, *twy = twx + kNaMaxLen;
  FftPlan px, py;
  make_plan(nx / 2, px);
  make_plan(ny, py);
  {
    std::lock_guard<std::mutex> g(g_na_mu);
    auto it = g_na_tw.find(dev);
    if (it == g_na_tw.end() || it->second != std::make_pair(nx, ny)) {
      // the tables of fsibe_spectral_create, so the results are those of
      // fsibe_dev_coftxy bit for bit; copied synchronously from host memory
      const auto tx = twiddles(nx), ty = twiddles(ny);
      HIPCHK(hipMemcpyAsync(twx, tx.data(), sizeof(double2) * nx, hipMemcpyHostToDevice, st));
      HIPCHK(hipMemcpyAsync(twy, ty.data(), sizeof(double2) * ny, hipMemcpyHostToDevice, st));
      HIPCHK(hipStreamSynchronize(st));
      g_na_tw[dev] = std::make_pair(nx, ny);
    }
  }
  CHK(rows_r2c(nx, ny, px, twx, d_f, tmp, st));
  return cols_pack(nx / 2, ny, py, twy, tmp, d_fk, st);
}

// host-pointer wrappers: copy in, run, copy out
static int host_call(fsibe_spectral *c, const double *in, double *out, int kind, int which, double dt) {
  if (!c || !out || (kind != 3 && !in)) return set_err(FSIBE_EARG, "null argument");
  const size_t bytes = sizeof(double) * (size_t)c->nx * c->ny;
  if (kind != 3) HIPCHK(Transfer::get().upload(c->hbuf_in, in, bytes, c->stream));
  if (kind == 0) CHK(dev_coftxy(c, c->hbuf_in, c->hbuf_out, c->stream));
  else if (kind == 1) CHK(dev_cofitxy(c, c->hbuf_in, c->hbuf_out, c->stream));
  else if (kind == 2) CHK(dev_op(c, which, c->hbuf_in, c->hbuf_out, c->stream));
  else CHK(dev_vis(c, dt, c->hbuf_out, c->stream));
  HIPCHK(Transfer::get().download(out, c->hbuf_out, bytes, c->stream));
  return FSIBE_OK;
}

extern "C" int fsibe_coftxy(fsibe_spectral *c, const double *f, double *fk) { return host_call(c, f, fk, 0, 0, 0); }
extern "C" int fsibe_cofitxy(fsibe_spectral *c, const double *fk, double *f) { return host_call(c, fk, f, 1, 0, 0); }
extern "C" int fsibe_cofdx(fsibe_spectral *c, const double *a, double *b) { return host_call(c, a, b, 2, 0, 0); }
extern "C" int fsibe_cofdy(fsibe_spectral *c, const double *a, double *b) { return host_call(c, a, b, 2, 1, 0); }
extern "C" int fsibe_cofdxdx(fsibe_spectral *c, const double *a, double *b) { return host_call(c, a, b, 2, 2, 0); }
extern "C" int fsibe_cofdydy(fsibe_spectral *c, const double *a, double *b) { return host_call(c, a, b, 2, 3, 0); }
extern "C" int fsibe_cofdxdy(fsibe_spectral *c, const double *a, double *b) { return host_call(c, a, b, 2, 4, 0); }
extern "C" int fsibe_poisson(fsibe_spectral *c, const double *a, double *b) { return host_call(c, a, b, 2, 5, 0); }
extern "C" int fsibe_vis(fsibe_spectral *c, double dt, double *w) { return host_call(c, nullptr, w, 3, 0, dt); }

// dealiase_mask.f90:1-33 (host; the 0/1 pattern is computed once per run)
static void dealias_host(int nx, int ny, double *d) {
  const int kx_max = nx / 2 - 1, ky_max = ny / 2 - 1;
  const double kx_trunc = 2.0 / 3.0 * (double)kx_max, ky_trunc = 2.0 / 3.0 * (double)ky_max;
  for (size_t i = 0; i < (size_t)nx * ny; ++i) d[i] = 1.0;
  for (int ky = 0; ky <= ky_max; ++ky)
    for (int kx = 0; kx <= kx_max; ++kx) {
      const double a = (double)kx, b = (double)ky;
      if (a * a / (kx_trunc * kx_trunc) + b * b / (ky_trunc * ky_trunc) >= 1.0) {
        d[(size_t)(2 * ky) * nx + 2 * kx] = 0.0;
        d[(size_t)(2 * ky) * nx + 2 * kx + 1] = 0.0;
        d[(size_t)(2 * ky + 1) * nx + 2 * kx] = 0.0;
        d[(size_t)(2 * ky + 1) * nx + 2 * kx + 1] = 0.0;
      }
    }
}

extern "C" int fsibe_dealiase_mask(fsibe_spectral *c, double *d) {
  if (!c || !d) return set_err(FSIBE_EARG, "null argument");
  dealias_host(c->nx, c->ny, d);
  return FSIBE_OK;
}

// ---- 1-D transforms of the FFT plugin (cofts / cofits) ---------------------
// Host-side: their only caller is the beam-curvature filter of the host solid
// solver (SolidSolver.f90:1388,1417) on L = ns + 2 n_ext points, far too
// small for a device launch.  Each column is a real DFT of length L summed in
// long double with twiddles exp(-2 pi i jk/L) from a table of L entries.
static void twiddle_table(int L, std::vector<long double> &c, std::vector<long double> &s) {
  const long double pi = 3.141592653589793238462643383279502884L;
  c.resize(L);
  s.resize(L);
  for (int m = 0; m < L; ++m) {
    c[m] = cosl(2.0L * pi * (long double)m / (long double)L);
    s[m] = sinl(2.0L * pi * (long double)m / (long double)L);
  }
}

extern "C" int fsibe_cofts(const double *f, double *fk, int L, int n) {
  if (!f || !fk || L < 1 || n < 0) return set_err(FSIBE_EARG, "cofts: bad argument");
  std::vector<long double> c, s;
  twiddle_table(L, c, s);
  std::vector<double> ft((size_t)L + 2);
  for (int j = 0; j < n; ++j) {
    const double *x = f + (size_t)j * L;
    // ft = r2c(x) as interleaved (Re, Im) for k = 0 .. L/2
    for (int k = 0; k <= L / 2; ++k) {
      long double re = 0.0L, im = 0.0L;
      for (int m = 0; m < L; ++m) {
        const int q = (int)(((long long)k * m) % L);
        re += (long double)x[m] * c[q];
        im -= (long double)x[m] * s[q];
      }
      ft[2 * k] = (double)re;
      ft[2 * k + 1] = (double)im;
    }
    // fk = ft(0:L-1) / L: the highest coefficient pair is cut (cof_fftw33.f90:277-285)
    const double norm = 1.0 / (double)L;
    for (int m = 0; m < L; ++m) fk[(size_t)j * L + m] = ft[m] * norm;
  }
  return FSIBE_OK;
}

extern "C" int fsibe_cofits(const double *fk, double *f, int L, int n) {
  if (!f || !fk || L < 1 || n < 0) return set_err(FSIBE_EARG, "cofits: bad argument");
  std::vector<long double> c, s;
  twiddle_table(L, c, s);
  std::vector<double> ft((size_t)L + 2);
  for (int j = 0; j < n; ++j) {
    // ft(0:L-1) = fk, ft(L:L+1) = 0 (cof_fftw33.f90:311-316), then the
    // unnormalised c2r, which reads Re only of the k = 0 (and, for even L,
    // the k = L/2) coefficient
    for (int m = 0; m < L; ++m) ft[m] = fk[(size_t)j * L + m];
    ft[L] = 0.0;
    ft[L + 1] = 0.0;
    const int K = L / 2;  // last index of the half spectrum
    for (int m = 0; m < L; ++m) {
      long double acc = (long double)ft[0];
      for (int k = 1; k <= K; ++k) {
        const int q = (int)(((long long)k * m) % L);
        const long double re = ft[2 * k], im = ft[2 * k + 1];
        const long double t = re * c[q] - im * s[q];
        acc += (2 * k == L) ? (long double)re * c[q] : 2.0L * t;
      }
      f[(size_t)j * L + m] = (double)acc;
    }
  }
  return FSIBE_OK;
}

extern "C" int fsibe_mouvement(const fsibe_params *p, int im, double x0, double y0, double angle, double phase,
                               double time, double *alpha, double *alpha_t, double *alpha_tt, double LE[6]) {
  if (!p || !alpha || !alpha_t || !alpha_tt || !LE) return set_err(FSIBE_EARG, "null argument");
  mouvement_host(*p, im, x0, y0, angle, phase, time, *alpha, *alpha_t, *alpha_tt, LE);
  return FSIBE_OK;
}

extern "C" int fsibe_integrate_position(const fsibe_params *p, int im, double time, const double *theta,
                                        const double *theta_dot, double *x, double *y, double *vx, double *vy) {
  if (!p || !theta || !theta_dot || !x || !y || !vx || !vy) return set_err(FSIBE_EARG, "null argument");
  if (p->ns < 2) return set_err(FSIBE_EARG, "ns must be >= 2");
  integrate_position_host(*p, im, time, theta, theta_dot, x, y, vx, vy);
  return FSIBE_OK;
}

extern "C" int fsibe_beam_placement(const fsibe_params *p, int ib, double *x0, double *y0, double *phase) {
  if (!p || !x0 || !y0 || !phase) return set_err(FSIBE_EARG, "null argument");
  if (ib < 0 || ib > 1 || !beam_placement(*p, ib, *x0, *y0, *phase))
    return set_err(FSIBE_EARG, "error...iMotion bad bad: beam %d needs iMotion 300..307 (init_beam.f90:55-74)",
                   ib + 1);
  return FSIBE_OK;
}

extern "C" int fsibe_integrate_position_beam(const fsibe_params *p, int ib, double time, const double *theta,
                                             const double *theta_dot, double *x, double *y, double *vx,
                                             double *vy) {
  if (!p || !theta || !theta_dot || !x || !y || !vx || !vy) return set_err(FSIBE_EARG, "null argument");
  if (p->ns < 2) return set_err(FSIBE_EARG, "ns must be >= 2");
  double x0 = 0.0, y0 = 0.0, ph = 0.0;
  CHK(fsibe_beam_placement(p, ib, &x0, &y0, &ph));
  integrate_position_host(*p, p->iMotion, x0, y0, ph, time, theta, theta_dot, x, y, vx, vy);
  return FSIBE_OK;
}

// ---------------------------------------------------------------------------
// host solid solver (solid.hpp)
// ---------------------------------------------------------------------------
struct fsibe_solid {
  ibes::Solver sv;
  ibes::Beam b;
};

extern "C" int fsibe_solid_create(const fsibe_params *p, fsibe_solid **out) {
  return fsibe_solid_create_beam(p, 0, out);
}

extern "C" int fsibe_solid_create_beam(const fsibe_params *p, int ib, fsibe_solid **out) {
  if (!p || !out) return set_err(FSIBE_EARG, "null argument");
  *out = nullptr;
  if (p->iBeam < 1) return set_err(FSIBE_EARG, "the solid solver needs a beam (iBeam >= 1)");
  if (!(p->length > 0.0)) return set_err(FSIBE_EARG, "beam length must be > 0");
  double x0 = 0.0, y0 = 0.0, ph = 0.0;
  if (ib < 0 || ib >= p->iBeam || !beam_placement(*p, ib, x0, y0, ph))
    return set_err(FSIBE_EARG, "beam %d of %d: the second beam needs iMotion 300..307 (init_beam.f90:55-74)",
                   ib + 1, p->iBeam);
  fsibe_solid *b = new fsibe_solid();
  if (!b->sv.init(*p)) {
    const std::string e = b->sv.err;
    delete b;
    return set_err(FSIBE_EARG, "%s", e.c_str());
  }
  b->sv.x0 = x0; b->sv.y0 = y0; b->sv.phase = ph;
  ibes::init_beam(*p, b->b, x0, y0, ph);
  *out = b;
  return FSIBE_OK;
}

extern "C" int fsibe_solid_destroy(fsibe_solid *b) {
  delete b;
  return FSIBE_OK;
}

static std::vector<double> *solid_array(fsibe_solid *b, int which) {
  ibes::Beam &m = b->b;
  std::vector<double> *v[FSIBE_SOLID_OLDOLD + 1] = {&m.x, &m.y, &m.vx, &m.vy, &m.theta, &m.theta_dot, &m.ax,
                                                    &m.ay, &m.pressure_old, &m.pressure_new, &m.tau_old,
                                                    &m.tau_new, &m.oldold};
  return (which >= 0 && which <= FSIBE_SOLID_OLDOLD) ? v[which] : nullptr;
}

extern "C" int fsibe_solid_get(fsibe_solid *b, int which, double *out) {
  if (!b || !out) return set_err(FSIBE_EARG, "null argument");
  std::vector<double> *v = solid_array(b, which);
  if (!v) return set_err(FSIBE_EARG, "unknown solid array %d", which);
  std::copy(v->begin(), v->end(), out);
  return FSIBE_OK;
}

extern "C" int fsibe_solid_set(fsibe_solid *b, int which, const double *in) {
  if (!b || !in) return set_err(FSIBE_EARG, "null argument");
  std::vector<double> *v = solid_array(b, which);
  if (!v) return set_err(FSIBE_EARG, "unknown solid array %d", which);
  std::copy(in, in + v->size(), v->begin());
  b->sv.pre_ok_ = false;
  return FSIBE_OK;
}

extern "C" int fsibe_solid_get_info(fsibe_solid *b, fsibe_solid_info *o) {
  if (!b || !o) return set_err(FSIBE_EARG, "null argument");
  const ibes::Beam &m = b->b;
  o->dt_old = m.dt_old;
  o->grav = b->sv.grav;
  o->E_kinetic = m.E_kinetic;
  o->E_pot = m.E_pot;
  o->E_elastic = m.E_elastic;
  o->Inertial_Force[0] = m.Inertial_Force[0];
  o->Inertial_Force[1] = m.Inertial_Force[1];
  o->StartupStep = m.StartupStep ? 1 : 0;
  o->iter = b->sv.iter;
  o->brake = b->sv.brake ? 1 : 0;
  o->method = b->sv.step_method(m);
  return FSIBE_OK;
}

extern "C" int fsibe_solid_set_info(fsibe_solid *b, const fsibe_solid_info *in) {
  if (!b || !in) return set_err(FSIBE_EARG, "null argument");
  b->b.dt_old = in->dt_old;
  b->sv.grav = in->grav;
  b->b.StartupStep = in->StartupStep != 0;
  b->sv.pre_ok_ = false;
  return FSIBE_OK;
}

extern "C" int fsibe_solid_step(fsibe_solid *b, double time, double dt) {
  if (!b) return set_err(FSIBE_EARG, "null solid");
  if (!(dt > 0.0)) return set_err(FSIBE_EARG, "dt must be > 0");
  if (time > b->sv.p.T_release && b->sv.step_method(b->b) == ibes::kBDF2 && !(b->b.dt_old > 0.0))
    return set_err(FSIBE_ESTATE, "BDF2 step without a previous step (dt_old = 0)");
  if (!b->sv.step(time, dt, b->b)) return set_err(FSIBE_EDOMAIN, "%s", b->sv.err.c_str());
  return FSIBE_OK;
}

extern "C" int fsibe_solid_wrapper(fsibe_solid *b, double time, double dt) {
  if (!b) return set_err(FSIBE_EARG, "null solid");
  if (!(dt > 0.0)) return set_err(FSIBE_EARG, "dt must be > 0");
  if (time > b->sv.p.T_release && b->sv.step_method(b->b) == ibes::kBDF2 && !(b->b.dt_old > 0.0))
    return set_err(FSIBE_ESTATE, "BDF2 step without a previous step (dt_old = 0)");
  if (!b->sv.wrapper(time, dt, b->b)) return set_err(FSIBE_EDOMAIN, "%s", b->sv.err.c_str());
  return FSIBE_OK;
}

extern "C" int fsibe_gravity_impulse(const fsibe_params *p, double time, double *grav) {
  if (!p || !grav) return set_err(FSIBE_EARG, "null argument");
  *grav = ibes::Solver::gravity_at(p->iImpulse, time, *grav);
  return FSIBE_OK;
}

// context of the next step without taking it (test hooks)
static int solid_context(fsibe_solid *b, double time, double dt) {
  if (!(dt > 0.0)) return set_err(FSIBE_EARG, "dt must be > 0");
  const int m = b->sv.step_method(b->b);
  if (m == ibes::kBDF2 && !(b->b.dt_old > 0.0)) return set_err(FSIBE_ESTATE, "BDF2 step without dt_old");
  if (!b->sv.begin(time, dt, b->b, m)) return set_err(FSIBE_EDOMAIN, "%s", b->sv.err.c_str());
  return FSIBE_OK;
}

extern "C" int fsibe_solid_guess(fsibe_solid *b, double time, double dt, double *x) {
  if (!b || !x) return set_err(FSIBE_EARG, "null argument");
  if (!(dt > 0.0)) return set_err(FSIBE_EARG, "dt must be > 0");
  if (!b->sv.guess(time, dt, b->b, x)) return set_err(FSIBE_EDOMAIN, "%s", b->sv.err.c_str());
  return FSIBE_OK;
}

extern "C" int fsibe_solid_residual(fsibe_solid *b, double time, double dt, const double *x, double *F) {
  if (!b || !x || !F) return set_err(FSIBE_EARG, "null argument");
  CHK(solid_context(b, time, dt));
  b->sv.residual(x, [&](int k, double v) { F[k - 1] = v; });
  return FSIBE_OK;
}

extern "C" int fsibe_solid_jacobian(fsibe_solid *b, double time, double dt, const double *x, double *J) {
  if (!b || !x || !J) return set_err(FSIBE_EARG, "null argument");
  CHK(solid_context(b, time, dt));
  const size_t n = (size_t)b->sv.nx;
  std::fill(J, J + n * n, 0.0);
  b->sv.jacobian(x, [&](int k, int l, double v) { J[(size_t)(k - 1) * n + (l - 1)] = v; });
  return FSIBE_OK;
}

extern "C" int fsibe_solid_rhs(fsibe_solid *b, double time, const double *theta, const double *theta_dot,
                               const double *pressure, const double *tau, double *theta_t, double *theta_tt,
                               double *T) {
  if (!b || !theta || !theta_dot || !pressure || !tau || !theta_t || !theta_tt || !T)
    return set_err(FSIBE_EARG, "null argument");
  const int ns = b->sv.ns;
  std::copy(theta, theta + ns, theta_t);
  std::copy(theta_dot, theta_dot + ns, theta_tt);
  if (!b->sv.rhs_beameqn(time, theta_t, theta_tt, pressure, tau, T))
    return set_err(FSIBE_EDOMAIN, "%s", b->sv.err.c_str());
  return FSIBE_OK;
}

// ---------------------------------------------------------------------------
// Tier B
// ---------------------------------------------------------------------------
static constexpr int kNC = 128;  // BeamSurfaceIntegral circle points (BeamForces.f90:311)

struct Box {
  int x0 = 0, x1 = -1, y0 = 0, y1 = -1;
  int w() const { return x1 >= x0 ? x1 - x0 + 1 : 0; }
  int h() const { return y1 >= y0 ? y1 - y0 + 1 : 0; }
  bool empty() const { return x1 < x0 || y1 < y0; }
  void add(int a0, int a1, int b0, int b1) {
    if (a1 < a0 || b1 < b0) return;
    if (empty()) { x0 = a0; x1 = a1; y0 = b0; y1 = b1; return; }
    x0 = std::min(x0, a0); x1 = std::max(x1, a1); y0 = std::min(y0, b0); y1 = std::max(y1, b1);
  }
};

// kernel classes timed by fsibe_profile_* (HIP events on the sim's stream)
enum ProfKernel {
  P_MASK = 0, P_VEL, P_COLS_W0, P_ROWS_NL, P_SCALARS, P_COLS_AB2, P_COLS_W1, P_ROWS_PRESS, P_REDUCE,
  P_COLS_PRESS, P_ROWS_BOX, P_INTERP, P_FORCES, P_NK
};

struct Prof {
  bool on = false;
  unsigned mask = 0;  // kernel classes that are timed
  hipEvent_t ev[P_NK][2] = {};
  bool rec[P_NK] = {};
  double ms[P_NK] = {};
  long long cnt[P_NK] = {};
};

struct fsibe_sim {
  Prof prof;
  fsibe_params p;
  int nx, ny, H, ns;
  // beams (iBeam <= 2, init_beam.f90:48-76): their count, and per beam the
  // leading edge (x0, y0) and the phase of mouvement; the beam arrays below
  // hold nb * ns values, beam ib at offset ib * ns
  int nb = 0;
  double bx0[2] = {0, 0}, by0[2] = {0, 0}, bphase[2] = {0, 0};
  double pi, dx, dy, ds, scalex, scaley, gerf;
  bool sharp, penal_on, sponge_on, pressure_on, forces_on, visc;
  StepConsts sc;
  FlowParams fp;
  FftPlan px, py;
  hipStream_t stream;
  // bit b: a copy from host staging buffer b may still be running (cleared
  // by every wait that follows the copies)
  int upload_pending = 0;
  double2 *twx, *twy;
  char *fields = nullptr;  // the allocation that holds the fields of the grid below
  double2 *W[2], *NL[2], *T[9];
  double *u1, *u2, *vor_mean, *ms, *wallrow;
  double *frame = nullptr;   // iSponge = 22: the frame mask (SmoothFrameAroundDomain), full grid
  double *rowpen = nullptr;  // iMeanVelocity = 11: row sums of the penalisation term (2 per row)
  fsibe_spectral *spec = nullptr;  // packed-layout operators for pressure snapshots (made on first use)
  double *snap = nullptr;          // their scratch, 9 fields
  double *umax_part;
  DevScalars *dscal;
  double *mask_m, *mask_vx, *mask_vy;
  int *mask_win = nullptr;  // winning primitive per mask pixel (adjoint runs only)
  double *fb_p, *fb_sa, *fb_sb;
  // per-step upload area: prims | targets | node data | circle data | vals.
  // Two host buffers, written in turn: the host builds step n+1's geometry
  // in one while the copy of step n may still read the other, so no event
  // marks a copy's end (the loops' own waits follow every copy).
  char *h_stage = nullptr, *d_stage;
  char *m_stage = nullptr;  // device address of h_stage (mapped)
  char *h_stage_b[2] = {nullptr, nullptr}, *m_stage_b[2] = {nullptr, nullptr};
  int stage_cur = 0;        // the buffer h_stage / m_stage point to
  // coupled loop: the next step's record copy, queued before the beam solve
  // behind a gate in host memory that the upload opens (k_stage_copy_gated)
  long long *h_gate = nullptr, *m_gate = nullptr;
  long long gate_seq = 0, gate_ticks = 0;
  long long gate_opened = 0;  // the last gate an upload opened (checked after the step's wait)
  bool gate_armed = false;
  size_t stage_bytes;
  // two result slots (StepOutDev, p_beam[nsb], tau_beam[nsb]) in pinned,
  // host-coherent memory that the kernels write directly; d_res is the
  // device address of h_res
  char *h_res = nullptr, *d_res = nullptr;
  size_t res_stride = 0;
  int slot = 0;
  bool res_pending = false;  // pipelined run: results of the previous step not yet read
  // coupled run: the slot whose row sums (energies, cal_drag) are read after
  // the next step's launches, off the beam solve's path (-1: none)
  int rows_pending = -1;
  bool pipe = false;         // record ev_dt after the nonlinear-term kernel
  hipEvent_t ev_dt;
  hipEvent_t ev_step;        // after a step's last kernel (iFLUSI=1 loop)
  // the next step's first column pass (it reads only vortk) already runs:
  // launched for time level k1_level before the host solves the beam, or
  // part of the previous step's fused column stage.  Its dw/dy column is in
  // Bp (T[1] or T[7]), its omega column in T[0]
  bool k1_ready = false;
  // K2's convective part of every row went ahead too (the iFLUSI=1 loop's
  // launch, or the previous step's fused row stage), into Rcp (T[2] or T[8])
  bool k2_ready = false;
  double2 *Bp = nullptr, *Rcp = nullptr;
  int kcA = 0;  // the columns of both beyond are zero and not stored
  // launch choices of the column stages K1, K4, K5, K7 (the autotuner's,
  // once fsibe_run has measured them for this grid; else the static ones)
  ColSel csel[4];
  bool csel_ready = false;
  int k1_level = -1;
  // what each slot holds: the fluid step's row sums, the force terms
  bool slot_fluid[2] = {false, false}, slot_forces[2] = {false, false};
  int slot_units[2] = {0, 0};
  // cal_drag's previous penalisation sums per beam (type Solid
  // drag_unst_old, lift_unst_old, UnsteadyCorrectionsReady;
  // NavierStokes.f90:579-589)
  double drag_unst_old[2] = {0, 0}, lift_unst_old[2] = {0, 0};
  bool unst_ready[2] = {false, false};
  int n0 = 0, n1 = 1;
  // geometry of the current step (set by create_mask)
  bool have_beam = false, sponge_done = false;
  // mouvement(time_mask) per beam: alpha, LeadingEdge(1:6)
  double time_mask = 0.0, alpha[2] = {0, 0}, LE[2][6] = {{0, 0, 0, 0, 0, 0}, {0, 0, 0, 0, 0, 0}};
  std::vector<double> bx, by, bvx, bvy, btheta, btheta_dot;
  std::vector<double> seg_ang, seg_c, seg_s;  // mask geometry scratch, one per segment
  Box mbox, fbox;
  Window win[2];  // cal_drag's window per beam
  int nprim = 0, ntg = 0;
  size_t off_prim = 0, off_beam = 0, off_tg = 0, off_nd = 0, off_cd = 0, off_val = 0;
  int nprim_cap = 0;  // room for mask primitives in the staging buffer
  ForceGeom fg;
  bool forces_ready = false;
  bool press_box_valid = false;
  // time loop state (fsibe_run)
  double time = 0.0, dt0 = 0.0, dt1 = 0.0;
  int it = 0;
  bool startup_done = false;
  fsibe_step_out last;       // the last step's results; the per-beam fields of the first beam
  fsibe_step_out last_b[2];  // the per-beam fields (Force ... fx_int, ibes_iter) of each beam
  std::vector<double> pbeam, tbeam;
  // the spectral and mask arrays of the field record of the last
  // fsibe_backup_read (vortk, nlk, workvis at both levels, mask, maskvx,
  // maskvy; packed layout), kept until the state changes (a step, a new
  // mask, a level swap, new vorticity): the device holds the spectra as half
  // spectra, whose conversion back is exact only to rounding, and neither
  // the scaled nlk(n0) nor workvis(n1) of the AB2 history, so a backup
  // written before the next step writes these verbatim
  std::vector<double> restored;
  fsibe_solid *solid[2] = {nullptr, nullptr};  // iFLUSI=1: the beams solved by the library (fsibe_run)
  // time of the kinematics in the beam arrays (integrate_position's time)
  double beam_time = 0.0;
  // sums of -Force(1) dt1 and dt1 over the steps read so far (the objective
  // of the adjoint, J = (1/T) sum (-Force(1)) dt)
  double jsum_f = 0.0, jsum_t = 0.0;
  struct AdjTape *tape = nullptr;  // records the forward data of each step for the adjoint
};

static void tape_mask_place(fsibe_sim *s);
static void tape_k1_place(fsibe_sim *s);
static void tape_mask(fsibe_sim *s);
static int tape_fluid(fsibe_sim *s, bool explicit_step);

static double now_ms();

// host phases timed with the steady clock into the otherwise unused classes
// wait for an event by polling: the waiting thread stays on its core, so the
// host work that follows (the beam solve, the next geometry) starts at once
// and with warm caches, where a blocking wait may let the core sleep.  The
// poll has a deadline (wait.hpp): FSIBE_EHIP naming `stage` if the event has
// not completed by then.
static int wait_event(hipEvent_t ev, const char *stage) {
  hipError_t err = hipSuccess;
  std::string msg;
  const int rc = bounded_wait(
      [&] {
        err = hipEventQuery(ev);
        return err == hipSuccess ? Poll::Done : err == hipErrorNotReady ? Poll::Busy : Poll::Failed;
      },
      now_ms, [&] { return hipGetErrorString(err); }, wait_timeout_ms(), stage, msg);
  return rc == FSIBE_OK ? FSIBE_OK : set_err(rc, "%s", msg.c_str());
}

static double now_ms() {
  return std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now().time_since_epoch()).count();
}
static void prof_host(fsibe_sim *s, int k, double t0) {
  if (s->prof.on && (s->prof.mask >> k & 1u)) {
    s->prof.ms[k] += now_ms() - t0;
    s->prof.cnt[k] += 1;
  }
}

// the host-written part of the geometry record (primitives, beam block)
// into device memory, on the step's stream; the builders then write the
// other host buffer.  No event marks the copy's end: an event between two
// kernels stalls the queue until the first has drained (~5 us here, before
// the mask kernel could start), and the loops wait for a later kernel of
// the same step anyway.
static int upload_geometry(fsibe_sim *s) {
  const int n = (int)(s->off_tg / sizeof(double2));
  if (s->gate_armed) {
    // the copy from this buffer is queued: the record is written, open it
    __atomic_store_n(s->h_gate, s->gate_seq, __ATOMIC_RELEASE);
    s->gate_armed = false;
    s->gate_opened = s->gate_seq;
  } else if (n > 0) {
    const int blocks = std::min(64, (n + 255) / 256);
    k_stage_copy<<<blocks, 256, 0, s->stream>>>(reinterpret_cast<const double2 *>(s->m_stage),
                                              reinterpret_cast<double2 *>(s->d_stage), n);
    HIPCHK(hipGetLastError());
  }
  s->upload_pending |= 1 << s->stage_cur;
  s->stage_cur ^= 1;
  s->h_stage = s->h_stage_b[s->stage_cur];
  s->m_stage = s->m_stage_b[s->stage_cur];
  return FSIBE_OK;
}

// Coupled loop, before the beam solve: queue the next step's record copy
// (from the buffer the builders write next) behind the gate, so that after
// the solve the host only opens the gate instead of launching the copy into
// an idle queue.  The stream's later work waits behind it, so every path
// that leaves the loop opens it (open_gate).
static int arm_upload(fsibe_sim *s) {
  const int n = (int)(s->off_tg / sizeof(double2));
  if (n <= 0 || s->gate_armed || !s->h_gate || (s->upload_pending >> s->stage_cur & 1)) return FSIBE_OK;
  const long long seq = ++s->gate_seq;
  const int blocks = std::min(64, (n + 255) / 256);
  k_stage_copy_gated<<<blocks, 256, 0, s->stream>>>(reinterpret_cast<const double2 *>(s->m_stage),
                                                    reinterpret_cast<double2 *>(s->d_stage), n, s->m_gate, seq,
                                                    s->gate_ticks);
  HIPCHK(hipGetLastError());
  s->gate_armed = true;
  return FSIBE_OK;
}

// after a wait that follows the copy: a gate that timed out copied a stale
// record, so the step's mask is wrong
static int gate_check(fsibe_sim *s) {
  if (s->gate_opened && __atomic_load_n(s->h_gate + 1, __ATOMIC_ACQUIRE) == s->gate_opened)
    return set_err(FSIBE_EHIP, "the geometry copy stopped waiting for its record (2 s) and copied a stale one");
  return FSIBE_OK;
}

// a queued copy that no upload will open: open it (it copies a stale
// record, overwritten by the next upload before any mask kernel reads it);
// the builders wait for it before writing that buffer again
static void open_gate(fsibe_sim *s) {
  if (!s->gate_armed) return;
  __atomic_store_n(s->h_gate, s->gate_seq, __ATOMIC_RELEASE);
  s->gate_armed = false;
  s->upload_pending |= 1 << s->stage_cur;
}

// before the builders write h_stage: a copy still reading it (two uploads
// without a wait in between, e.g. repeated fsibe_create_mask calls) ends first
static int stage_writable(fsibe_sim *s) {
  if (s->upload_pending >> s->stage_cur & 1) {
    HIPCHK(hipStreamSynchronize(s->stream));
    s->upload_pending = 0;
  }
  return FSIBE_OK;
}

// the force kernel's tables, built by the mask kernel beside its tiles
static BeamGeo beam_geo(const fsibe_sim *s, int nthreads) {
  BeamGeo g;
  g.beam = reinterpret_cast<const double *>(s->d_stage + s->off_beam);
  g.ns = s->ns; g.nb = s->nb;
  g.pi = s->pi;
  const bool bsi = s->visc && s->p.iCylinder == 0;
  g.nc = bsi ? kNC : 0;
  g.rr = s->p.t_beam + s->p.N_smooth * std::max(s->dy, s->dx);
  g.r1 = s->p.t_beam - 0.0 * s->p.N_smooth * std::max(s->dy, s->dx);
  g.dphi = s->pi / (double)(kNC - 1);
  g.tg = reinterpret_cast<double *>(s->d_stage + s->off_tg);
  g.nd = reinterpret_cast<double *>(s->d_stage + s->off_nd);
  g.cd = reinterpret_cast<double *>(s->d_stage + s->off_cd);
  const int items = s->nb * (s->ns + 2 * g.nc);
  g.fwg = (s->forces_on && s->nb > 0) ? (items + nthreads - 1) / nthreads : 0;
  return g;
}

// The start event is also recorded here, for regions whose kernels are not
// launched through KLAUNCH (their interval then includes the dispatch).
static void prof_begin(fsibe_sim *s, int k) {
  if (s->prof.on && (s->prof.mask >> k & 1u)) {
    (void)hipEventRecord(s->prof.ev[k][0], s->stream);
    t_prof_start = s->prof.ev[k][0];
    t_prof_stop = s->prof.ev[k][1];
    t_prof_launches = 0;
  }
}
static void prof_end(fsibe_sim *s, int k) {
  if (s->prof.on && (s->prof.mask >> k & 1u)) {
    if (t_prof_launches != 1) (void)hipEventRecord(s->prof.ev[k][1], s->stream);
    s->prof.rec[k] = true;
    t_prof_start = t_prof_stop = nullptr;
    t_prof_launches = 0;
  }
}
// disarms the kernel timing at the end of the enclosing scope, so that a
// region left by an error return (before its prof_end) leaves no armed
// events for a later launch
struct ProfDisarm {
  ~ProfDisarm() {
    t_prof_start = t_prof_stop = nullptr;
    t_prof_launches = 0;
  }
};
#define PROF_CAT2(a, b) a##b
#define PROF_CAT(a, b) PROF_CAT2(a, b)
#define PROF_BEGIN(s, k) \
  prof_begin(s, k);      \
  ProfDisarm PROF_CAT(prof_disarm_, __LINE__)
// after a stream synchronisation: accumulate the recorded intervals
static void prof_collect(fsibe_sim *s) {
  if (!s->prof.on) return;
  for (int k = 0; k < P_NK; ++k) {
    if (!s->prof.rec[k]) continue;
    float ms = 0.0f;
    if (hipEventElapsedTime(&ms, s->prof.ev[k][0], s->prof.ev[k][1]) == hipSuccess) {
      s->prof.ms[k] += ms;
      s->prof.cnt[k] += 1;
    }
    s->prof.rec[k] = false;
  }
}

// device addresses of the result slot k
static StepOutDev *res_dev(const fsibe_sim *s, int k) {
  return reinterpret_cast<StepOutDev *>(s->d_res + (size_t)k * s->res_stride);
}
static double *pbeam_dev(const fsibe_sim *s, int k) {
  return reinterpret_cast<double *>(s->d_res + (size_t)k * s->res_stride + sizeof(StepOutDev));
}
// beam nodes of all beams (at least 1: the size of the per-node arrays)
static int nodes_all(const fsibe_sim *s) { return std::max(s->nb * s->ns, 1); }
static size_t rows_off(const fsibe_sim *s) { return sizeof(StepOutDev) + sizeof(double) * 2 * nodes_all(s); }
static size_t parts_off(const fsibe_sim *s) { return rows_off(s) + sizeof(double) * (size_t)s->ny * kNSUM; }
static double *rows_dev(const fsibe_sim *s, int k) {
  return reinterpret_cast<double *>(s->d_res + (size_t)k * s->res_stride + rows_off(s));
}
static double *parts_dev(const fsibe_sim *s, int k) {
  return reinterpret_cast<double *>(s->d_res + (size_t)k * s->res_stride + parts_off(s));
}

static double smooth_step_host(const fsibe_sim *s, double x, double t, double h) {
  if (!s->sharp) {
    const double delta = h * s->gerf;
    return 0.5 * (erf((t - x) / delta) + erf((x + t) / delta));
  }
  return x <= t ? 1.0 : 0.0;
}

static inline int fnint(double x) { return (int)lround(x); }

// SmoothFrameAroundDomain, create_mask.f90:370-463: a level set phi of the
// distance to the domain's edges, with corners rounded to radius
// 2 thickness (thickness = 4 t_beam), and the cosine step SmoothStep2
// (:523-544) of phi over thickness/2; phi stays 1000 where no loop sets it
static void frame_host(const fsibe_sim *s, std::vector<double> &fr) {
  const int nx = s->nx, ny = s->ny;
  const double dx = s->dx, dy = s->dy, xl = s->p.xl, yl = s->p.yl, pi = s->pi;
  std::vector<double> phi((size_t)nx * ny, 1000.0);
  const double thickness = 4.0 * s->p.t_beam, R1 = 0.0, R2 = 2.0 * thickness, RR = R1 + R2;
  const int ixmin = fnint(RR / dx), ixmax = nx - fnint(RR / dx);
  const int iymin = fnint(RR / dy), iymax = ny - fnint(RR / dy);
  auto P = [&](int ix, int iy) -> double & { return phi[(size_t)iy * nx + ix]; };
  for (int ix = std::max(ixmin, 0); ix <= std::min(ixmax, nx - 1); ++ix)
    for (int iy = 0; iy < ny; ++iy) {
      const double y = (double)iy * dy;
      const double m = std::min(P(ix, iy), std::min(fabs(y - R1), fabs(y - (yl - R1))));
      P(ix, iy) = (iy <= fnint(R1 / dy) || iy >= ny - 1 - fnint(R1 / dy)) ? -m : m;
    }
  for (int ix = 0; ix < nx; ++ix)
    for (int iy = std::max(iymin, 0); iy <= std::min(iymax, ny - 1); ++iy) {
      const double x = (double)ix * dx;
      const double m = std::min(P(ix, iy), std::min(fabs(x - R1), fabs(x - (xl - R1))));
      P(ix, iy) = (ix <= fnint(R1 / dx) || ix >= nx - 1 - fnint(R1 / dx)) ? -m : m;
    }
  const double cxs[4] = {RR, RR, xl - RR, xl - RR}, cys[4] = {RR, yl - RR, yl - RR, RR};
  const int xa[4] = {0, 0, ixmax, ixmax}, xb[4] = {ixmin, ixmin, nx - 1, nx - 1};
  const int ya[4] = {0, iymax, iymax, 0}, yb[4] = {iymin, ny - 1, ny - 1, iymin};
  for (int c = 0; c < 4; ++c)
    for (int ix = std::max(xa[c], 0); ix <= std::min(xb[c], nx - 1); ++ix)
      for (int iy = std::max(ya[c], 0); iy <= std::min(yb[c], ny - 1); ++iy) {
        const double a = (double)ix * dx - cxs[c], b = (double)iy * dy - cys[c];
        P(ix, iy) = std::min(P(ix, iy), -(sqrt(a * a + b * b) - R2));
      }
  const double t = thickness / 2., h = thickness / 2.;
  fr.resize(phi.size());
  for (size_t k = 0; k < phi.size(); ++k) {
    const double x = phi[k];
    if (x <= t - h) fr[k] = 1.0;
    else if ((t - h) < x && x < (t + h)) fr[k] = 0.5 * (1. + cos((x - t + h) * pi / (2.0 * h)));
    else fr[k] = 0.0;
  }
}

// Mean_ux, Mean_uy (mean_velocity.f90) at `time` on the host; case 11
// (u_mean) is the device's state and reads as 0 here
static void mean_u_host(const FlowParams &f, double time, double &mx, double &my) {
  double tf = 1.0;
  switch (f.iMeanVelocity) {
    case 1:
      if (time < f.T_fullspeed) {
        const double t1 = f.T_fullspeed;
        tf = (time * time * time) / (-0.5 * t1 * t1 * t1) + 3 * (time * time) / (t1 * t1);
      }
      mx = cos(f.theta_inf) * tf; my = sin(f.theta_inf) * tf; break;
    case 2:
      if (time < f.T_fullspeed) tf = 0.5 * (1.0 - cos(0.5 * f.pi * time / f.T_fullspeed));
      mx = cos(f.theta_inf) * tf; my = sin(f.theta_inf) * tf; break;
    case 3: mx = cos(f.theta_inf); my = sin(f.theta_inf); break;
    case 6: mx = time; my = 0.0; break;
    case 22: mx = 0.1; my = 0.0; break;
    default: mx = 0.0; my = 0.0; break;
  }
}

// create_sponge_mask, create_mask.f90:223-364 (types 0,1,2,3,10,22)
static void sponge_host(const fsibe_sim *s, const double *mask_full, std::vector<double> &ms) {
  const int nx = s->nx, ny = s->ny;
  const double dx = s->dx, dy = s->dy, N = s->p.N_smooth, xl = s->p.xl, yl = s->p.yl;
  ms.assign((size_t)nx * ny, 0.0);
  const int isp = s->p.iSponge;
  if (isp == 1) {
    const double sss = s->p.SpongeSize, ssz = sss - 2.0 * N * dx, sb = xl - sss;
    int ixmax = fnint((xl - 0.5 * sss) / dx), ixmin = fnint(sb / dx);
    for (int ix = ixmin; ix <= ixmax; ++ix) {
      const double tmp = smooth_step_host(s, xl - 0.5 * sss - (double)ix * dx, ssz * 0.5, N * dx);
      for (int iy = 0; iy < ny; ++iy) ms[(size_t)iy * nx + ix] = tmp;
    }
    ixmin = fnint((xl - 0.5 * sss) / dx);
    ixmax = nx - 1;
    for (int ix = ixmin; ix <= ixmax; ++ix) {
      const double tmp = smooth_step_host(s, (double)ix * dx - xl + 0.5 * sss - 1.0 * dx, ssz * 0.4, N * dx);
      for (int iy = 0; iy < ny; ++iy) ms[(size_t)iy * nx + ix] = tmp;
    }
  } else if (isp == 22) {
    // :333-349: 1 outside the inner rectangle, 0 inside and wherever the
    // startup mask (frame included) is positive
    const int ixmin = fnint(s->p.SpongeSize / dx), iymin = fnint(s->p.SpongeSize / dy);
    const int ixmax = fnint((xl - s->p.SpongeSize) / dx), iymax = fnint((yl - s->p.SpongeSize) / dy);
    for (auto &v : ms) v = 1.0;
    for (int iy = std::max(iymin, 0); iy <= std::min(iymax, ny - 1); ++iy)
      for (int ix = std::max(ixmin, 0); ix <= std::min(ixmax, nx - 1); ++ix) ms[(size_t)iy * nx + ix] = 0.0;
    if (mask_full)
      for (size_t k = 0; k < ms.size(); ++k)
        if (mask_full[k] > 0.0) ms[k] = 0.0;
  } else if (isp == 10) {
    const int ixmin = fnint((xl - s->p.SpongeSize) / dx);
    for (int ix = std::max(ixmin, 0); ix < nx; ++ix)
      for (int iy = 0; iy < ny; ++iy) ms[(size_t)iy * nx + ix] = 1.0;
  } else if (isp == 2) {
    const double sss = s->p.SpongeSize, ssz = sss - 2.0 * N * dx;
    int ixmax = fnint((0.5 * sss) / dx);
    for (int ix = 0; ix <= ixmax; ++ix) {
      const double tmp = smooth_step_host(s, 0.5 * sss - (double)ix * dx, ssz * 0.5, N * dx);
      for (int iy = 0; iy < ny; ++iy) ms[(size_t)iy * nx + ix] = tmp;
    }
    const int ixmin = fnint((0.5 * sss) / dx);
    ixmax = fnint((1.0 * sss) / dx);
    for (int ix = ixmin; ix <= ixmax; ++ix) {
      const double tmp = smooth_step_host(s, (double)ix * dx - 0.5 * sss, ssz * 0.5, N * dx);
      for (int iy = 0; iy < ny; ++iy) ms[(size_t)iy * nx + ix] = tmp;
    }
    for (int ix = 0; ix <= ixmax; ++ix)
      for (int iy = 0; iy < ny; ++iy) {
        const size_t k = (size_t)iy * nx + ix;
        const double m = mask_full ? mask_full[k] : 0.0;
        if (m * s->p.eps > 0.0) ms[k] = ms[k] * (1.0 - m * s->p.eps);
      }
  } else if (isp == 3) {
    const double ssz = s->p.SpongeSize - N * dx;
    for (int ix = 0; ix < nx; ++ix)
      for (int iy = 0; iy < ny; ++iy) {
        const double t1 = smooth_step_host(s, (double)ix * dx, ssz, N * dx);
        const double t2 = smooth_step_host(s, xl - (double)ix * dx, ssz, N * dx);
        const double t3 = smooth_step_host(s, (double)iy * dy, ssz, N * dy);
        const double t4 = smooth_step_host(s, yl - (double)iy * dy, ssz, N * dy);
        double v = t1 + t2 + t3 + t4;
        if (v > 1.0) v = 1.0;
        ms[(size_t)iy * nx + ix] = v;
      }
  }
  for (auto &v : ms) v = v / s->p.eps_sponge;
}

extern "C" void *fsibe_sim_stream(fsibe_sim *s) { return s ? (void *)s->stream : nullptr; }

extern "C" int fsibe_sim_destroy(fsibe_sim *s) {
  if (!s) return FSIBE_OK;
  open_gate(s);
  (void)hipStreamSynchronize(s->stream);
  void *ptrs[] = {s->twx, s->twy, s->fields, s->ms, s->wallrow, s->umax_part, s->dscal, s->d_stage, s->frame,
                  s->rowpen, s->snap};
  if (s->spec) fsibe_spectral_destroy(s->spec);
  for (void *q : ptrs)
    if (q) (void)hipFree(q);
  for (int b = 0; b < 2; ++b)
    if (s->h_stage_b[b]) (void)hipHostFree(s->h_stage_b[b]);
  if (s->h_gate) (void)hipHostFree(s->h_gate);
  if (s->h_res) (void)hipHostFree(s->h_res);
  (void)hipEventDestroy(s->ev_dt);
  (void)hipEventDestroy(s->ev_step);
  for (int k = 0; k < P_NK; ++k)
    for (int j = 0; j < 2; ++j)
      if (s->prof.ev[k][j]) (void)hipEventDestroy(s->prof.ev[k][j]);
  (void)hipStreamDestroy(s->stream);
  delete s->solid[0];
  delete s->solid[1];
  if (s->mask_win) (void)hipFree(s->mask_win);
  delete s;
  return FSIBE_OK;
}

extern "C" int fsibe_sim_create(const fsibe_params *pp, fsibe_sim **out) {
  if (!pp || !out) return set_err(FSIBE_EARG, "null argument");
  *out = nullptr;
  const fsibe_params &p = *pp;
  if (!size_ok(p.nx, p.ny))
    return set_err(FSIBE_ESIZE, "grid %dx%d not supported (even sizes, nx/2 and ny = 2^a 3^b)", p.nx, p.ny);
  if (!(p.iSponge >= 0 && p.iSponge <= 4) && p.iSponge != 10 && p.iSponge != 22)
    return set_err(FSIBE_EUNSUPPORTED, "iSponge=%d is not a sponge type of create_mask.f90", p.iSponge);
  if (p.iBeam < 0 || p.iBeam > 2) return set_err(FSIBE_EUNSUPPORTED, "iBeam=%d: at most two beams", p.iBeam);
  // the second beam's phase exists for the dragonfly motions only; the
  // reference stops otherwise (init_beam.f90:72-73)
  if (p.iBeam == 2 && !(p.iMotion >= 300 && p.iMotion <= 307))
    return set_err(FSIBE_EARG, "error...iMotion bad bad: two beams need iMotion 300..307 (init_beam.f90:55-74)");
  if (p.iBeam > 0 && p.ns < 3) return set_err(FSIBE_EARG, "ns must be >= 3");
  if (p.iBeam > 0 && 2 * p.iBeam * p.ns + 8 > kMaxTilePrims)
    return set_err(FSIBE_EUNSUPPORTED, "ns=%d: at most %d beam nodes per beam", p.ns,
                   (kMaxTilePrims - 8) / (2 * p.iBeam));
  if (!(p.eps > 0.0) || !(p.xl > 0.0) || !(p.yl > 0.0)) return set_err(FSIBE_EARG, "eps, xl, yl must be > 0");
  if (((p.iSponge > 0 && p.iSponge < 4) || p.iSponge == 10 || p.iSponge == 22) && !(p.eps_sponge > 0.0))
    return set_err(FSIBE_EARG, "vorticity sponge needs eps_sponge > 0 (params.f90:185-188)");
  fsibe_sim *s = new fsibe_sim();
  s->p = p;
  s->nx = p.nx; s->ny = p.ny; s->H = p.nx / 2; s->ns = p.iBeam ? p.ns : 0;
  s->nb = p.iBeam;
  s->pi = 4.0 * atan(1.0);
  s->dx = p.xl / (double)p.nx;
  s->dy = p.yl / (double)p.ny;
  s->ds = p.ns > 1 ? p.length / (double)(p.ns - 1) : 0.0;
  { double a = 2.0 * s->pi / p.xl; s->scalex = a * a; }
  { double a = 2.0 * s->pi / p.yl; s->scaley = a * a; }
  s->gerf = fabs((exp(-(2.0 * 1.0) * (2.0 * 1.0)) - 1.0) / sqrt(s->pi));
  s->sharp = fabs(p.N_smooth) < 1e-4;
  if (s->p.U_mean_true == 0.0) s->p.U_mean_true = 1.0;
  // cal_nlk's penalisation term (NavierStokes.f90:88) and vorticity sponge
  // (:142); the time-step limit 0.9 eps leaves iSponge = 22 out (:71)
  s->penal_on = p.iBeam > 0 || p.iWalls > 0 || p.iCylinder > 0 || p.iSponge == 22;
  s->sponge_on = (p.iSponge > 0 && p.iSponge < 4) || p.iSponge == 22;
  s->pressure_on = p.iFLUSI == 1 || p.iSaveBeam > 0;
  s->forces_on = s->pressure_on && p.iBeam > 0;
  s->visc = p.iViscous == 1;
  make_plan(s->H, s->px);
  make_plan(s->ny, s->py);
  StepConsts &c = s->sc;
  c.nx = s->nx; c.ny = s->ny; c.H = s->H;
  c.sx = 2.0 * s->pi / p.xl; c.sy = 2.0 * s->pi / p.yl;
  c.scalex = s->scalex; c.scaley = s->scaley;
  c.norm = 1.0 / ((double)s->nx * (double)s->ny);
  {
    const double kxt = 2.0 / 3.0 * (double)(s->nx / 2 - 1), kyt = 2.0 / 3.0 * (double)(s->ny / 2 - 1);
    c.kxt2 = kxt * kxt; c.kyt2 = kyt * kyt;
    c.rkxt2 = 1.0 / c.kxt2; c.rkyt2 = 1.0 / c.kyt2;
  }
  c.idealis = p.idealis == 1;
  c.kc = s->H;
  for (int k = s->H - 1; k >= 0 && c.idealis && s->H > kCutH && (double)k * (double)k / c.kxt2 + 0.0 / c.kyt2 >= 1.0; --k) c.kc = k;
  c.nu = p.nu; c.eps = p.eps; c.dx = s->dx; c.dy = s->dy;
  FlowParams &f = s->fp;
  f.iMeanVelocity = p.iMeanVelocity; f.penal_on = p.iBeam > 0 || p.iWalls > 0 || p.iCylinder > 0;
  f.theta_inf = p.theta_inf; f.T_fullspeed = p.T_fullspeed; f.U_mean_true = s->p.U_mean_true;
  f.cfl = p.cfl; f.eps = p.eps; f.dt_fixed = p.dt_fixed; f.Time_end = p.Time_end; f.pi = s->pi;
  f.dx = s->dx; f.dy = s->dy; f.nu = p.nu; f.scalex = s->scalex; f.scaley = s->scaley;

  int rc = FSIBE_OK;
  auto fail = [&](int code) { fsibe_sim_destroy(s); return code; };
#define SIMCHK(call)                                                                    \
  do {                                                                                  \
    hipError_t e_ = (call);                                                             \
    if (e_ != hipSuccess) {                                                             \
      rc = set_err(FSIBE_EHIP, "%s failed: %s", #call, hipGetErrorString(e_));          \
      return fail(rc);                                                                  \
    }                                                                                   \
  } while (0)
  SIMCHK(hipStreamCreate(&s->stream));
  SIMCHK(hipEventCreate(&s->ev_dt));  // bound to K2's dispatch in the pipelined loop
  SIMCHK(hipEventCreate(&s->ev_step));  // bound to the force kernel's dispatch in the coupled loop
  const size_t N = (size_t)s->nx * s->ny, NH = (size_t)s->H * s->ny;
  auto tx = twiddles(s->nx), ty = twiddles(s->ny);
  SIMCHK(hipMalloc(&s->twx, sizeof(double2) * s->nx));
  SIMCHK(hipMalloc(&s->twy, sizeof(double2) * s->ny));
  SIMCHK(hipMemcpy(s->twx, tx.data(), sizeof(double2) * s->nx, hipMemcpyHostToDevice));
  SIMCHK(hipMemcpy(s->twy, ty.data(), sizeof(double2) * s->ny, hipMemcpyHostToDevice));
  {
    // every field of the grid in one allocation (22 of them: each call of
    // the allocator costs more than the fields' clearing), the ones that
    // are read before they are written cleared.  Fields at a distance
    // of exactly a power of two meet in the same memory channels: 4 KiB and 256 B
    // more between them took a step with a body at 4096^2 from 1930 to 1826 us, at
    // 1024 x 4096 from 416 to 409 (without a body 243 to 225), at 2048^2 from 325
    // to 317, at 1024^2 from 98.5 to 96.6, a gradient at 512^2 from 23.8 to 23.6 ms
    const size_t fld = ((sizeof(double2) * NH + 255) & ~(size_t)255) + 4096 + 256;
    SIMCHK(hipMalloc(&s->fields, 22 * fld));
    SIMCHK(hipMemset(s->fields, 0, 14 * fld));
    char *q = s->fields;
    auto take = [&](auto &dst) { dst = reinterpret_cast<std::remove_reference_t<decltype(dst)>>(q); q += fld; };
    for (int i = 0; i < 2; ++i) { take(s->W[i]); take(s->NL[i]); }
    for (int i = 0; i < 7; ++i) take(s->T[i]);
    take(s->u1); take(s->u2); take(s->vor_mean);
    take(s->T[7]); take(s->T[8]);
    take(s->mask_m); take(s->mask_vx); take(s->mask_vy);
    take(s->fb_p); take(s->fb_sa); take(s->fb_sb);
  }
  SIMCHK(hipMalloc(&s->umax_part, sizeof(double) * s->ny));
  SIMCHK(hipMemset(s->umax_part, 0, sizeof(double) * s->ny));
  SIMCHK(hipMalloc(&s->dscal, sizeof(DevScalars)));
  SIMCHK(hipMemset(s->dscal, 0, sizeof(DevScalars)));
  const int nsb0 = std::max(s->nb * s->ns, 1), nb1 = std::max(s->nb, 1);
  // slot: StepOutDev | p_beam[nsb] | tau_beam[nsb] | row sums[ny][kNSUM] |
  // force terms[8][nsb + nb kNC] (nsb = nb ns: every beam's nodes)
  const size_t res_bytes = sizeof(StepOutDev) + sizeof(double) * (2 * nsb0 + (size_t)s->ny * kNSUM +
                                                                   8 * (size_t)(nsb0 + nb1 * kNC));
  s->res_stride = (res_bytes + 255) & ~(size_t)255;
  SIMCHK(hipHostMalloc((void **)&s->h_res, 2 * s->res_stride, hipHostMallocMapped | hipHostMallocCoherent));
  memset(s->h_res, 0, 2 * s->res_stride);
  SIMCHK(hipHostGetDevicePointer((void **)&s->d_res, s->h_res, 0));
  const int nsb = std::max(s->nb * s->ns, 1);
  // staging layout
  {
    size_t off = 0;
    auto al = [&](size_t b) { size_t o = off; off += (b + 255) & ~(size_t)255; return o; };
    const int nprim_max = 2 * nsb + 8;
    const int ntg_max = 6 * nsb + 6 * kNC * nb1;
    s->nprim_cap = nprim_max;
    // host-written part: the primitives and the beam block X, Y, TH, alpha;
    // device-only: the force kernel's tables (built by the mask kernel) and
    // the interpolated values
    s->off_prim = al(sizeof(Prim) * nprim_max);
    s->off_beam = al(sizeof(double) * (3 * (size_t)nsb + 2));
    s->off_tg = al(sizeof(double) * 3 * ntg_max);
    s->off_nd = al(sizeof(double) * 4 * nsb);
    s->off_cd = al(sizeof(double) * 4 * 2 * kNC * nb1);
    s->off_val = al(sizeof(double) * ntg_max);
    s->stage_bytes = off;
  }
  for (int b = 0; b < 2; ++b) {
    SIMCHK(hipHostMalloc((void **)&s->h_stage_b[b], s->stage_bytes, hipHostMallocMapped | hipHostMallocCoherent));
    SIMCHK(hipHostGetDevicePointer((void **)&s->m_stage_b[b], s->h_stage_b[b], 0));
  }
  s->h_stage = s->h_stage_b[0];
  s->m_stage = s->m_stage_b[0];
  SIMCHK(hipHostMalloc((void **)&s->h_gate, 256, hipHostMallocMapped | hipHostMallocCoherent));
  SIMCHK(hipHostGetDevicePointer((void **)&s->m_gate, s->h_gate, 0));
  s->h_gate[0] = 0;
  s->h_gate[1] = 0;
  {
    int khz = 0, dev = 0;
    SIMCHK(hipGetDevice(&dev));
    SIMCHK(hipDeviceGetAttribute(&khz, hipDeviceAttributeWallClockRate, dev));
    s->gate_ticks = 2000LL * (long long)std::max(khz, 1000);  // 2 s of the wall clock
    // a shorter bound (wall-clock ticks) lets a test take the timeout path
    if (const char *e = getenv("FSIBE_GATE_TICKS")) s->gate_ticks = std::max(0LL, atoll(e));
  }
  SIMCHK(hipMalloc(&s->d_stage, s->stage_bytes));
  SIMCHK(hipMemset(s->d_stage, 0, s->stage_bytes));
  s->ms = nullptr;
  s->wallrow = nullptr;
  if (p.iWalls > 0) {
    std::vector<double> wr(s->ny, 0.0);
    const double N_ = p.N_smooth, h_star = p.h_channel + N_ * s->dy;
    const int iymax = fnint(h_star / s->dy);
    for (int j = 0; j <= iymax && j < s->ny; ++j) wr[j] = smooth_step_host(s, (double)j * s->dy, p.h_channel, N_ * s->dy);
    const int iymin = fnint((p.yl - h_star) / s->dy);
    for (int j = s->ny - 1; j >= iymin && j >= 0; --j)
      wr[j] = smooth_step_host(s, fabs((double)j * s->dy - p.yl), p.h_channel, N_ * s->dy);
    SIMCHK(hipMalloc(&s->wallrow, sizeof(double) * s->ny));
    SIMCHK(hipMemcpy(s->wallrow, wr.data(), sizeof(double) * s->ny, hipMemcpyHostToDevice));
  }
  if (p.iSponge == 22) {
    std::vector<double> fr;
    frame_host(s, fr);
    SIMCHK(hipMalloc(&s->frame, sizeof(double) * fr.size()));
    SIMCHK(hipMemcpy(s->frame, fr.data(), sizeof(double) * fr.size(), hipMemcpyHostToDevice));
  }
  if (p.iMeanVelocity == 11) {
    SIMCHK(hipMalloc(&s->rowpen, sizeof(double) * 2 * s->ny));
    SIMCHK(hipMemset(s->rowpen, 0, sizeof(double) * 2 * s->ny));
  }
  s->bx.assign(nsb, 0.0); s->by.assign(nsb, 0.0); s->bvx.assign(nsb, 0.0); s->bvy.assign(nsb, 0.0);
  s->btheta.assign(nsb, 0.0); s->btheta_dot.assign(nsb, 0.0);
  s->seg_ang.assign(nsb, 0.0); s->seg_c.assign(nsb, 0.0); s->seg_s.assign(nsb, 0.0);
  s->pbeam.assign(nsb, 0.0); s->tbeam.assign(nsb, 0.0);
  memset(&s->last, 0, sizeof(s->last));
  memset(s->last_b, 0, sizeof(s->last_b));
  s->win[0] = s->win[1] = Window{0, -1, 0, -1};
  // init_beam.f90:48-76: the first beam at (x0, y0), phase 0; the second at
  // (x0 + 1.25, y0) with the dragonfly phase (iMotion - 300) pi / 4
  for (int ib = 0; ib < s->nb; ++ib) {
    s->bx0[ib] = p.x0 + (ib == 1 ? 1.25 : 0.0);
    s->by0[ib] = p.y0;
    s->bphase[ib] = ib == 1 ? 0.25 * (double)(p.iMotion - 300) * s->pi : 0.0;
  }
#undef SIMCHK
  *out = s;
  return FSIBE_OK;
}

extern "C" int fsibe_set_vortk(fsibe_sim *s, const double *vk) {
  if (!s || !vk) return set_err(FSIBE_EARG, "null argument");
  const size_t N = (size_t)s->nx * s->ny;
  HIPCHK(Transfer::get().upload(s->fb_p, vk, sizeof(double) * N, s->stream));
  k_packed_to_half<<<grid1d((size_t)s->H * (s->ny / 2)), 256, 0, s->stream>>>(s->fb_p, s->W[s->n0], s->nx, s->ny);
  HIPCHK(hipGetLastError());
  HIPCHK(hipStreamSynchronize(s->stream));
  s->press_box_valid = false;
  std::vector<double>().swap(s->restored);
  return FSIBE_OK;
}

extern "C" int fsibe_swap_levels(fsibe_sim *s) {
  if (!s) return set_err(FSIBE_EARG, "null argument");
  std::swap(s->n0, s->n1);
  std::vector<double>().swap(s->restored);
  return FSIBE_OK;
}

// ---- geometry of one step (host) ------------------------------------------
static void add_prim(fsibe_sim *s, Prim &P, int &np) {
  Prim *dst = reinterpret_cast<Prim *>(s->h_stage + s->off_prim);
  if (np < s->nprim_cap) dst[np] = P;  // the caller checks the count
  ++np;
}

// the mask's primitives and box, and the cal_drag window (create_mask.f90)
static int build_mask_geometry(fsibe_sim *s) {
  const int nx = s->nx, ny = s->ny, ns = s->ns;
  const double dx = s->dx, dy = s->dy, N = s->p.N_smooth, t = s->p.t_beam;
  const double mdx = std::max(dx, dy);
  int np = 0;
  Box mb;
  if (s->p.iWalls > 0) {
    const double h_star = s->p.h_channel + N * dy;
    mb.add(0, nx - 1, 0, std::min(ny - 1, fnint(h_star / dy)));
    mb.add(0, nx - 1, std::max(0, fnint((s->p.yl - h_star) / dy)), ny - 1);
  }
  // the velocity sponge's columns (create_mask.f90:137-180) and the frame
  // (:187-202) on every row
  if (s->p.iSponge == 4) mb.add(0, std::min(nx - 1, fnint((1.0 * s->p.SpongeSize) / dx)), 0, ny - 1);
  if (s->p.iSponge == 22) mb.add(0, nx - 1, 0, ny - 1);
  const double delta = N * mdx * s->gerf;
  // segments and hinges: create_mask's t* = t + 2 N max(dx,dy), or with
  // iSmoothCutoff = 1 the end dots' reach t + 7 delta (smooth step < 1e-22)
  const double t_cut = s->p.iSmoothCutoff ? t + 7.0 * delta : t + 2.0 * N * mdx;
  auto dot = [&](double px_, double py_, double vx_, double vy_, double tt) {
    Prim P{};
    P.type = PRIM_DOT;
    const double r = s->sharp ? tt + mdx : tt + 7.0 * delta + mdx;
    P.ix0 = std::max(0, (int)floor((px_ - r) / dx) - 1);
    P.ix1 = std::min(nx - 1, (int)ceil((px_ + r) / dx) + 1);
    P.iy0 = std::max(0, (int)floor((py_ - r) / dy) - 1);
    P.iy1 = std::min(ny - 1, (int)ceil((py_ + r) / dy) + 1);
    P.a[0] = px_; P.a[1] = py_; P.a[2] = vx_; P.a[3] = vy_; P.a[4] = tt;
    add_prim(s, P, np);
    mb.add(P.ix0, P.ix1, P.iy0, P.iy1);
  };
  if (s->p.iCylinder == 1) dot(s->p.x0 - s->p.R_cylinder, s->p.y0, 0.0, 0.0, s->p.R_cylinder);
  // beam after beam (create_mask.f90:74-119): each primitive overwrites
  // where its value is strictly larger, so the list order is the drawing order
  for (int ib = 0; ib < s->nb; ++ib) {
    const int o = ib * ns;
    const double *X = s->bx.data() + o, *Y = s->by.data() + o, *VX = s->bvx.data() + o, *VY = s->bvy.data() + o;
    const double *TH = s->btheta.data() + o;
    const double t_star = t_cut;
    // the segments' directions atan2(dy, dx), shared by the hinges (DrawHinge
    // takes the same atan2 of the same differences, create_mask.f90:104-105)
    double *seg_ang = s->seg_ang.data() + o, *seg_c = s->seg_c.data() + o, *seg_s = s->seg_s.data() + o;
    for (int i = 0; i <= ns - 2; ++i) {  // DrawBeamSegment :740-761
      Prim P{};
      P.type = PRIM_SEG;
      const double p1x = X[i], p1y = Y[i], p2x = X[i + 1], p2y = Y[i + 1];
      seg_ang[i] = atan2((p2y - p1y), (p2x - p1x));
      const double al = -seg_ang[i];
      P.ix0 = std::max(fnint((std::min(p1x, p2x) - t_star) / dx), 0);
      P.ix1 = std::min(fnint((std::max(p1x, p2x) + t_star) / dx), nx - 1);
      P.iy0 = std::max(fnint((std::min(p1y, p2y) - t_star) / dy), 0);
      P.iy1 = std::min(fnint((std::max(p1y, p2y) + t_star) / dy), ny - 1);
      double ca, sa;
      sincos(al, &sa, &ca);  // glibc's sincos returns sin and cos bit for bit
      seg_c[i] = ca;
      seg_s[i] = -sa;
      P.a[0] = ca * p1x - sa * p1y; P.a[1] = sa * p1x + ca * p1y;
      P.a[2] = ca * p2x - sa * p2y; P.a[3] = sa * p2x + ca * p2y;
      P.a[4] = ca; P.a[5] = sa; P.a[6] = t_star;
      P.a[7] = VX[i]; P.a[8] = VY[i]; P.a[9] = VX[i + 1]; P.a[10] = VY[i + 1];
      add_prim(s, P, np);
      mb.add(P.ix0, P.ix1, P.iy0, P.iy1);
    }
    if (s->p.iSharpTrailing == 1) {  // DrawSharpEnd :796-822
      Prim P{};
      P.type = PRIM_SHARP;
      const double al = TH[ns - 1] + s->alpha[ib];
      const double pex = X[ns - 1], pey = Y[ns - 1];
      double ca, sa;
      sincos(al, &sa, &ca);
      const double p1x = pex - 2.0 * mdx * ca, p1y = pey - 2.0 * mdx * sa;
      const double p2x = pex + 4.0 * mdx * ca, p2y = pey + 4.0 * mdx * sa;
      P.ix0 = std::max(fnint((std::min(p1x, p2x) - t_star) / dx), 0);
      P.ix1 = std::min(fnint((std::max(p1x, p2x) + t_star) / dx), nx - 1);
      P.iy0 = std::max(fnint((std::min(p1y, p2y) - t_star) / dy), 0);
      P.iy1 = std::min(fnint((std::max(p1y, p2y) + t_star) / dy), ny - 1);
      P.a[0] = ca * p1x + sa * p1y; P.a[1] = -sa * p1x + ca * p1y;
      P.a[2] = ca * p2x + sa * p2y; P.a[3] = -sa * p2x + ca * p2y;
      P.a[4] = ca; P.a[5] = sa; P.a[6] = t_star; P.a[7] = VX[ns - 1]; P.a[8] = VY[ns - 1]; P.a[9] = mdx;
      add_prim(s, P, np);
      mb.add(P.ix0, P.ix1, P.iy0, P.iy1);
    }
    for (int i = 1; i <= ns - 2; ++i) {  // DrawHinge :579-592 via create_mask :103-107
      Prim P{};
      P.type = PRIM_HINGE;
      const double a1 = seg_ang[i - 1], a2 = seg_ang[i];
      const double ts2 = t_cut;
      P.ix0 = std::max(fnint((X[i] - ts2) / dx), 0);
      P.ix1 = std::min(fnint((X[i] + ts2) / dx), nx - 1);
      P.iy0 = std::max(fnint((Y[i] - ts2) / dy), 0);
      P.iy1 = std::min(fnint((Y[i] + ts2) / dy), ny - 1);
      const double c1 = a1 < 0.0 ? 2.0 * s->pi + a1 : a1, c2 = a2 < 0.0 ? 2.0 * s->pi + a2 : a2;
      P.a[0] = X[i]; P.a[1] = Y[i];
      P.a[2] = c1 * 180.0 / s->pi; P.a[3] = c2 * 180.0 / s->pi;
      P.a[4] = ts2; P.a[5] = VX[i]; P.a[6] = VY[i];
      // unit directions of the two segments, for the sector pre-test only
      P.a[8] = seg_c[i - 1]; P.a[9] = seg_s[i - 1]; P.a[10] = seg_c[i]; P.a[11] = seg_s[i];
      add_prim(s, P, np);
      mb.add(P.ix0, P.ix1, P.iy0, P.iy1);
    }
    if (Y[0] < 0.0) return set_err(FSIBE_EDOMAIN, "Mask:: Beam Hinge. Index out of region (create_mask.f90:685-688)");
    dot(X[0], Y[0], VX[0], VY[0], t);
    if (s->p.iSharpTrailing == 0) dot(X[ns - 1], Y[ns - 1], VX[ns - 1], VY[ns - 1], t);
  }
  // the beam block the device reads: X, Y, TH of every beam, then alpha
  {
    double *bb = reinterpret_cast<double *>(s->h_stage + s->off_beam);
    const int nsb = s->nb * ns;
    for (int i = 0; i < nsb; ++i) { bb[i] = s->bx[i]; bb[nsb + i] = s->by[i]; bb[2 * nsb + i] = s->btheta[i]; }
    for (int ib = 0; ib < s->nb; ++ib) bb[3 * nsb + ib] = s->alpha[ib];
  }
  if (np > s->nprim_cap) return set_err(FSIBE_ESIZE, "mask: %d primitives, room for %d", np, s->nprim_cap);
  s->nprim = np;
  s->mbox = mb;

  // cal_drag window of each beam (NavierStokes.f90:528-564); without a beam
  // the whole grid
  for (int ib = 0; ib < std::max(s->nb, 1); ++ib) {
    int ixmin, ixmax, iymin, iymax;
    const double *X = s->bx.data() + ib * ns, *Y = s->by.data() + ib * ns;
    const double *LE = s->LE[ib];
    if (s->p.iBeam > 0) {
      double ymax = Y[0], ymin = Y[0], xmin = X[0], xmax = X[0];
      for (int i = 1; i < ns; ++i) {
        ymax = std::max(ymax, Y[i]); ymin = std::min(ymin, Y[i]);
        xmin = std::min(xmin, X[i]); xmax = std::max(xmax, X[i]);
      }
      const double tb = s->p.t_beam, rc = s->p.R_cylinder;
      iymax = (int)((std::max(ymax + 1.5 * tb, LE[1] + 2.0 * rc)) / dy);
      iymin = (int)((std::min(ymin - 1.5 * tb, LE[1] - 2.0 * rc)) / dy);
      ixmin = (int)(std::min((LE[0] - std::max(2.5 * rc, 1.5 * tb)), (xmin - 1.5 * tb)) / dx);
      ixmax = (int)((xmax + 1.5 * tb) / dx);
    } else {
      iymax = ny - 1; iymin = 0; ixmax = nx - 1; ixmin = 0;
    }
    if (s->p.iBeam > 0 && s->p.iSmoothCutoff) {
      // every pixel within t + 7 delta + max(dx,dy) of a node
      double ymax = Y[0], ymin = Y[0], xmin = X[0], xmax = X[0];
      for (int i = 1; i < ns; ++i) {
        ymax = std::max(ymax, Y[i]); ymin = std::min(ymin, Y[i]);
        xmin = std::min(xmin, X[i]); xmax = std::max(xmax, X[i]);
      }
      const double r = t + 7.0 * delta + mdx;
      ixmin = std::min(ixmin, fnint((xmin - r) / dx));
      ixmax = std::max(ixmax, fnint((xmax + r) / dx));
      iymin = std::min(iymin, fnint((ymin - r) / dy));
      iymax = std::max(iymax, fnint((ymax + r) / dy));
    }
    const double h_star = s->p.h_channel + s->p.N_smooth * dy;
    if (s->p.iWalls > 0) {
      if (ixmin < 0) ixmin = 0;
      if (ixmax > nx - 1) ixmax = nx - 1;
      if (iymin < fnint(h_star / dy) + 2) iymin = fnint(h_star / dy) + 2;
      if (iymax > fnint((s->p.yl - h_star) / dy) - 2) iymax = fnint((s->p.yl - h_star) / dy) - 2;
    }
    ixmin = std::max(ixmin, 0); ixmax = std::min(ixmax, nx - 1);
    iymin = std::max(iymin, 0); iymax = std::min(iymax, ny - 1);
    s->win[ib] = Window{ixmin, ixmax, iymin, iymax};
  }
  if (s->nb < 2) s->win[1] = Window{0, -1, 0, -1};
  return FSIBE_OK;
}

// interpolation targets (BeamForces.f90:150-165, :351-362, :389-400), node
// and circle data of GetForces, and the pressure box they need
// the interpolation targets of every beam as the force kernel forms them
// (BeamForces.f90:150-165, :351-362, :389-400), here only to decide whether
// one leaves the field and to bound their stencils; the host needs them only
// where the bound from the nodes alone does not settle it (near the edges)
static void exact_target_box(const fsibe_sim *s, double rr, double r1, bool bsi, double dxi, double dyi, Box &fb,
                             bool &bad) {
  const int nx = s->nx, ny = s->ny, ns = s->ns;
  const double x2 = s->p.xl - s->dx, y2 = s->p.yl - s->dy;
  auto target = [&](double xt, double yt) {
    if (xt > x2 || xt < 0.0 || yt > y2 || yt < 0.0) bad = true;
    const int i = (int)((xt - 0.0) / dxi), j = (int)((yt - 0.0) / dyi);
    if (i - 4 < 0 || i + 4 > nx - 1 || j - 4 < 0 || j + 4 > ny - 1) bad = true;
    fb.add(i - 4, i + 4, j - 4, j + 4);
  };
  for (int ib = 0; ib < s->nb; ++ib) {
    const double *X = s->bx.data() + ib * ns, *Y = s->by.data() + ib * ns, *TH = s->btheta.data() + ib * ns;
    const double alpha = s->alpha[ib];
    for (int n = 0; n < ns; ++n) {
      const double th = TH[n] + alpha;
      const double st = sin(th), ct = cos(th);
      target(X[n] - r1 * st, Y[n] + r1 * ct);
      target(X[n] + r1 * st, Y[n] - r1 * ct);
      target(X[n] - rr * st, Y[n] + rr * ct);
      target(X[n] + rr * st, Y[n] - rr * ct);
    }
    if (bsi) {
      const double dphi = s->pi / (double)(kNC - 1);
      for (int i = 0; i < kNC; ++i) {
        const double phi = -(0.5 * s->pi - (TH[ns - 1] + alpha)) + (double)i * dphi;
        target(X[ns - 1] + rr * cos(phi), Y[ns - 1] + rr * sin(phi));
        const double phl = (0.5 * s->pi + (TH[1] + alpha)) + (double)i * dphi;
        target(X[0] + rr * cos(phl), Y[0] + rr * sin(phl));
      }
    }
  }
}

// The force kernel builds the interpolation targets itself from the beam
// block.  Every target lies within rr of a node (rr >= r1), so the nodes'
// box grown by rr bounds them, and their 9 x 9 stencils (plus one cell for
// the rounding of the device's target coordinates) bound the pressure box.
// Where that bound reaches the field's edge the exact targets decide the
// reference's error (Interpolation.f90:19-24).
static int build_force_geometry(fsibe_sim *s, double time) {
  const int nx = s->nx, ny = s->ny, ns = s->ns;
  const double dx = s->dx, dy = s->dy;
  s->forces_ready = false;
  s->ntg = 0;
  Box fb;
  if (s->forces_on) {
    const double x2 = s->p.xl - dx, y2 = s->p.yl - dy;
    const double dxi = (x2 - 0.0) / (double)(nx - 1), dyi = (y2 - 0.0) / (double)(ny - 1);
    const double rr = s->p.t_beam + s->p.N_smooth * std::max(dy, dx);
    const double r1 = s->p.t_beam - 0.0 * s->p.N_smooth * std::max(dy, dx);
    const bool bsi = s->visc && s->p.iCylinder == 0;
    const int nsb = s->nb * ns;
    double xmin = s->bx[0], xmax = s->bx[0], ymin = s->by[0], ymax = s->by[0];
    for (int i = 1; i < nsb; ++i) {
      xmin = std::min(xmin, s->bx[i]); xmax = std::max(xmax, s->bx[i]);
      ymin = std::min(ymin, s->by[i]); ymax = std::max(ymax, s->by[i]);
    }
    // a margin of a hundredth of a cell covers the rounding of the targets
    const double mx = 0.01 * dxi, my = 0.01 * dyi;
    const double xa = xmin - rr - mx, xb = xmax + rr + mx, ya = ymin - rr - my, yb = ymax + rr + my;
    const bool inside = xa >= 0.0 && ya >= 0.0 && xb <= x2 && yb <= y2;
    int i0 = 0, i1 = -1, j0 = 0, j1 = -1;
    if (inside) {
      i0 = (int)(xa / dxi); i1 = (int)(xb / dxi); j0 = (int)(ya / dyi); j1 = (int)(yb / dyi);
    }
    if (inside && i0 - 4 >= 0 && i1 + 4 <= nx - 1 && j0 - 4 >= 0 && j1 + 4 <= ny - 1) {
      fb.add(i0 - 4, i1 + 4, j0 - 4, j1 + 4);
    } else {
      bool bad = false;
      exact_target_box(s, rr, r1, bsi, dxi, dyi, fb, bad);
      if (bad) return set_err(FSIBE_EDOMAIN, "DeltaInterpolation: target coordinates not in the field "
                                             "(Interpolation.f90:19-24) or stencil leaves the grid");
    }
    // one more cell each side for the device's rounding, inside the grid
    fb.x0 = std::max(fb.x0 - 1, 0); fb.x1 = std::min(fb.x1 + 1, nx - 1);
    fb.y0 = std::max(fb.y0 - 1, 0); fb.y1 = std::min(fb.y1 + 1, ny - 1);
    const int nc = bsi ? kNC : 0;
    s->ntg = s->nb * (6 * ns + 6 * nc);
    ForceGeom &g = s->fg;
    g.ns = ns; g.nc = nc; g.nt = s->ntg;
    g.bx0 = fb.x0; g.by0 = fb.y0; g.bw = fb.w(); g.bh = fb.h();
    g.dxi = dxi; g.dyi = dyi; g.pi = s->pi; g.ds = s->ds;
    g.dL = (s->pi / (double)(kNC - 1)) * rr;
    g.visc = s->visc; g.bsi_on = bsi;
    g.nb = s->nb; g.nx = nx; g.ny = ny; g.pad = 0;
    g.rr = rr; g.r1 = r1; g.dphi = s->pi / (double)(kNC - 1);
    // soft startup (BeamForces.f90:246-252)
    const double Tr = s->p.T_release, tau = tau_eff(s->p);
    double soft;
    if (time <= Tr) soft = 0.0;
    else if (time > Tr && time < (Tr + tau)) {
      const double a = time - Tr;
      soft = (a * a * a) / (-0.5 * (tau * tau * tau)) + 3. * (a * a) / (tau * tau);
    } else soft = 1.0;
    g.soft = soft;
    s->fbox = fb;
    s->forces_ready = true;
  } else if (s->pressure_on) {
    s->fbox = Box();
  }
  return FSIBE_OK;
}

static int build_geometry(fsibe_sim *s, double time) {
  CHK(build_mask_geometry(s));
  return build_force_geometry(s, time);
}

// rows of Rpx (K2's penalisation spectrum, the input of K4) that may be
// nonzero: the mask box's rows (K2 writes 0 on the others), or every row
// when the iSponge = 10 term adds to it
static void rpx_rows(const fsibe_sim *s, const MaskBox &mb, int &py0, int &py1) {
  if (s->p.iSponge == 10) {
    py0 = 0;
    py1 = s->ny - 1;
  } else if (mb.x1 >= mb.x0) {
    py0 = mb.y0;
    py1 = mb.y1;
  } else {
    py0 = 1;
    py1 = 0;
  }
}

// rows of -ky^2 psi (K5's field 3) that K8 reads: the force box's, once the
// force geometry of the step is built (else every row)
static void stress_rows(const fsibe_sim *s, int &r0, int &r1) {
  if (s->forces_ready && !s->fbox.empty()) {
    r0 = s->fbox.y0;
    r1 = s->fbox.y1;
  } else {
    r0 = 0;
    r1 = s->ny - 1;
  }
}

static MaskBox mask_box(const fsibe_sim *s) {
  MaskBox m;
  m.x0 = s->mbox.x0; m.x1 = s->mbox.x1; m.y0 = s->mbox.y0; m.y1 = s->mbox.y1; m.w = s->mbox.w();
  if (s->mbox.empty()) { m.x0 = 0; m.x1 = -1; m.y0 = 0; m.y1 = -1; m.w = 0; }
  m.m = s->mask_m; m.vx = s->mask_vx; m.vy = s->mask_vy;
  return m;
}

static int ensure_sponge(fsibe_sim *s) {
  if (s->sponge_done) return FSIBE_OK;
  s->sponge_done = true;
  if (!s->sponge_on && s->p.iSponge != 10) return FSIBE_OK;
  std::vector<double> mfull;
  if (s->p.iSponge == 2 || s->p.iSponge == 22) {
    mfull.assign((size_t)s->nx * s->ny, 0.0);
    if (!s->mbox.empty()) {
      std::vector<double> mb((size_t)s->mbox.w() * s->mbox.h());
      HIPCHK(hipMemcpyAsync(mb.data(), s->mask_m, sizeof(double) * mb.size(), hipMemcpyDeviceToHost, s->stream));
      HIPCHK(hipStreamSynchronize(s->stream));
      for (int y = 0; y < s->mbox.h(); ++y)
        for (int x = 0; x < s->mbox.w(); ++x)
          mfull[(size_t)(y + s->mbox.y0) * s->nx + x + s->mbox.x0] = mb[(size_t)y * s->mbox.w() + x];
    }
  }
  std::vector<double> ms;
  sponge_host(s, mfull.empty() ? nullptr : mfull.data(), ms);
  HIPCHK(hipMalloc(&s->ms, sizeof(double) * ms.size()));
  HIPCHK(hipMemcpy(s->ms, ms.data(), sizeof(double) * ms.size(), hipMemcpyHostToDevice));
  return FSIBE_OK;
}

// with_forces = false: only the mask's part of the geometry is built and
// uploaded; the caller builds and uploads the force part (force_geometry)
// before the pressure and force kernels
// beam arrays of nb ns values (beam ib's nodes from ib ns), alpha[nb],
// LE[6 nb] (NULL: zeros)
static int create_mask_impl(fsibe_sim *s, double time, const double *x, const double *y, const double *vx,
                            const double *vy, const double *theta, const double *alpha, const double *LE,
                            bool with_forces);

extern "C" int fsibe_create_mask(fsibe_sim *s, double time, const double *x, const double *y, const double *vx,
                                 const double *vy, const double *theta, double alpha, const double LE[6]) {
  if (s && s->nb > 1)
    return set_err(FSIBE_EARG, "%d beams: fsibe_create_mask_beams takes every beam's kinematics", s->nb);
  return create_mask_impl(s, time, x, y, vx, vy, theta, &alpha, LE, true);
}

extern "C" int fsibe_create_mask_beams(fsibe_sim *s, double time, const double *x, const double *y,
                                       const double *vx, const double *vy, const double *theta,
                                       const double *alpha, const double *LE) {
  if (s && s->nb > 0 && !alpha) return set_err(FSIBE_EARG, "null alpha");
  return create_mask_impl(s, time, x, y, vx, vy, theta, alpha, LE, true);
}

static int force_geometry(fsibe_sim *s, double time) {
  const double th0 = now_ms();
  CHK(build_force_geometry(s, time));  // host scalars and box only: the kernel builds its targets
  prof_host(s, P_REDUCE, th0);
  return FSIBE_OK;
}

static int create_mask_impl(fsibe_sim *s, double time, const double *x, const double *y, const double *vx,
                            const double *vy, const double *theta, const double *alpha, const double *LE,
                            bool with_forces) {
  if (!s) return set_err(FSIBE_EARG, "null sim");
  if (s->ns > 0 && (!x || !y || !vx || !vy || !theta)) return set_err(FSIBE_EARG, "null beam array");
  std::vector<double>().swap(s->restored);
  CHK(stage_writable(s));
  for (int i = 0; i < s->nb * s->ns; ++i) {
    s->bx[i] = x[i]; s->by[i] = y[i]; s->bvx[i] = vx[i]; s->bvy[i] = vy[i]; s->btheta[i] = theta[i];
  }
  for (int ib = 0; ib < 2; ++ib) {
    const bool have = ib < s->nb || (ib == 0 && alpha);
    s->alpha[ib] = have && alpha ? alpha[ib] : 0.0;
    for (int i = 0; i < 6; ++i) s->LE[ib][i] = have && LE ? LE[6 * ib + i] : 0.0;
  }
  s->time_mask = time;
  s->have_beam = true;
  const double th0 = now_ms();
  if (with_forces) {
    CHK(build_geometry(s, time));
  } else {
    CHK(build_mask_geometry(s));
    s->forces_ready = false;
  }
  CHK(upload_geometry(s));
  prof_host(s, P_REDUCE, th0);
  if (s->tape) tape_mask_place(s);
  if (!s->mbox.empty()) {
    MaskConsts mc;
    mc.dx = s->dx; mc.dy = s->dy; mc.t = s->p.t_beam; mc.h = s->p.N_smooth * std::max(s->dx, s->dy);
    mc.gerf = s->gerf; mc.inv_eps_unused = 0.0; mc.ds = s->ds; mc.pi = s->pi; mc.sharp = s->sharp;
    mc.eps = s->p.eps;
    if (s->p.iSponge == 4 || s->p.iSponge == 22) {
      mean_u_host(s->fp, time, mc.mux, mc.muy);
      if (s->p.iMeanVelocity == 11)  // device address of DevScalars::u_mean
        mc.mean_dev = reinterpret_cast<const double *>(reinterpret_cast<const char *>(s->dscal) +
                                                        offsetof(DevScalars, u_mean));
      mc.N = s->p.N_smooth;
    }
    if (s->p.iSponge == 4) {
      const double S = s->p.SpongeSize;
      mc.vs4 = 1;
      mc.vs_S = S;
      mc.vs_ssz = S - 2.0 * s->p.N_smooth * s->dx;
      mc.vs_Heff = s->p.yl - 2.0 * s->p.h_channel;
      mc.h_channel = s->p.h_channel;
      mc.vs_ixmid = fnint((0.5 * S) / s->dx);
      mc.vs_ixmax = fnint((1.0 * S) / s->dx);
    }
    if (s->p.iSponge == 22) {
      mc.frame = s->frame;
      mc.nx_frame = s->nx;
      mc.frame_M = std::max(1.0e-3, s->p.eps);
    }
    const BeamGeo bg = beam_geo(s, kMaskThreads);
    const int tiles_x = (s->mbox.w() + kMaskTile - 1) / kMaskTile, tiles_y = (s->mbox.h() + kMaskTile - 1) / kMaskTile;
    // one more row of workgroups builds the force tables beside the tiles
    dim3 blk(kMaskThreads);
    dim3 grd(std::max(tiles_x, bg.fwg), tiles_y + (bg.fwg > 0 ? 1 : 0));
    PROF_BEGIN(s, P_MASK);
    k_mask<<<grd, blk, 0, s->stream>>>(
        reinterpret_cast<const Prim *>(s->d_stage + s->off_prim), s->nprim, s->wallrow ? s->wallrow + 0 : nullptr, mc,
        bg, tiles_y, s->mbox.x0, s->mbox.y0, s->mbox.w(), s->mbox.h(), s->mask_m, s->mask_vx, s->mask_vy,
        s->mask_win);
    HIPCHK(hipGetLastError());
    prof_end(s, P_MASK);
  }
  if (s->tape) tape_mask(s);
  CHK(ensure_sponge(s));
  return FSIBE_OK;
}

// ---- fluid step ----------------------------------------------------------
static ColSel static_sel(const fsibe_sim *s, int bm, int split);

// launch choice of column stage `which` (0: K1 and the other inverse
// transforms of one level, 1: K4, 2: K5, 3: K7) of a kernel over `split`
// fields
static ColSel sim_sel(const fsibe_sim *s, int which, int split) {
  if (s->csel_ready) return s->csel[which];
  return static_sel(s, (which == 1 || which == 3) ? 2 : 1, split);
}

// (fields -ky^2 psi are stored on rows r0_3 .. r1_3 only)
static int cols_inv_fields(fsibe_sim *s, const double2 *W, double2 *const *outs, const int *fsel, int nf,
                           int which = 0, int r0_3 = 0, int r1_3 = 1 << 30) {
  double2 *o[4] = {outs[0], nf > 1 ? outs[1] : nullptr, nf > 2 ? outs[2] : nullptr, nf > 3 ? outs[3] : nullptr};
  int f[4] = {fsel[0], nf > 1 ? fsel[1] : 0, nf > 2 ? fsel[2] : 0, nf > 3 ? fsel[3] : 0};
  return with_cols_sel<1>(s->py, s->H, sim_sel(s, which, nf), [&](auto F, int nt, int TX) -> int {
    const size_t lds = sizeof(double2) * TX * padlen(s->ny);
    const int grid = (s->H / TX) * nf;
    KLAUNCH(k_cols_inv_fields<decltype(F)>, grid, nt, lds, s->stream, W, o[0], o[1], o[2], o[3], f[0], f[1], f[2],
            f[3], nf, F, s->twy, s->sc, r0_3, r1_3);
    return FSIBE_OK;
  });
}

// u = cal_velocity(time, vortk(n0)) and the CFL maxima (EvolveFluidExplicit :440)
static int velocity_only(fsibe_sim *s, double time) {
  double2 *outs[2] = {s->T[1], s->T[2]};
  const int fsel[2] = {1, 2};
  CHK(cols_inv_fields(s, s->W[s->n0], outs, fsel, 2));
  const size_t lds = sizeof(double2) * 3 * padlen(s->H);
  double mx, my;
  {
    // Mean_ux/Mean_uy at `time`; only the startup step comes here, when
    // case 11's u_mean is still 0
    mean_u_host(s->fp, time, mx, my);
  }
  const double UMx = s->p.U_mean_true * mx, UMy = s->p.U_mean_true * my;
  MaskBox mb = mask_box(s);
  StepConsts c = s->sc;
  c.kc = s->H;  // a spectrum that no update has dealiased
  return with_rows<3>(s->px, [&](auto F, int nt) -> int {
    KLAUNCH(k_rows_press<decltype(F)>, s->ny, nt, lds, s->stream, nullptr, s->T[1], s->T[2], s->u1, s->u2,
            s->vor_mean, mb, s->win[0], s->win[1], rows_dev(s, s->slot), s->umax_part, s->T[4], s->T[5], s->dscal, UMx,
            UMy, 0, 0,
            F, s->twx,
            c);
    return FSIBE_OK;
  });
}

// K1: A = Fy^-1[W0], B = Fy^-1[i ky W0] (and Fy^-1[i ky psi] for iSponge =
// 10, whose outflow sponge acts inside the penalisation term).  It reads only
// the vorticity of time level `level`.  have_a: T[0] holds that level's
// omega column already (the column stage just before wrote it).
static int launch_k1(fsibe_sim *s, int level, bool have_a = false) {
  const bool sp10 = s->p.iSponge == 10 && s->penal_on && s->ms;
  double2 *outs[3] = {s->T[0], s->T[1], s->T[4]};
  const int fsel[3] = {0, 4, 2};
  const int f0 = have_a && !sp10 ? 1 : 0;
  PROF_BEGIN(s, P_COLS_W0);
  CHK(cols_inv_fields(s, s->W[level], outs + f0, fsel + f0, (sp10 ? 3 : 2) - f0));
  prof_end(s, P_COLS_W0);
  s->Bp = s->T[1];
  s->kcA = have_a ? s->sc.kc : s->H;
  return FSIBE_OK;
}

// K2's instance for rows by F: rows of at most kCutH entries are never cut, longer
// ones whole only on a call's first step or without dealiasing, where the selects
// cost little of the call with a compile-time plan (1024 rows of 512: 18.3 us and
// 17.1 without) and 2 % of a step with a run-time one
template <class F> static auto nl_kernel(const fsibe_sim *s) {
  constexpr int H = fixed_len<F>::v;
  if constexpr (H > 0) return &k_rows_nl<F, (H > kCutH)>;
  else return s->kcA < s->H ? &k_rows_nl<F, true> : &k_rows_nl<F, false>;
}

// the constants of K2: columns of A, B beyond kcA are zero and not stored
static StepConsts nl_consts(const fsibe_sim *s) {
  StepConsts c = s->sc;
  c.kc = s->kcA;
  return c;
}

// K2 of the next step without the penalisation term, on every row: it reads
// K1's output, the velocity and the sponge, none of which the beam solve
// changes (empty mask box: Rc = Fx[r], Rpx = 0, row sums 0).  evolve_fluid
// then adds the penalisation on the rows of the new mask box (k_rows_pen,
// which also computes the K3 scalars).
static int launch_k2_ahead(fsibe_sim *s) {
  s->k2_ready = false;
  if (s->mbox.empty() || !s->penal_on) return FSIBE_OK;
  const int na = s->ny, nb = 0, b1 = s->ny - 1;
  MaskBox none;
  none.x0 = 0; none.x1 = -1; none.y0 = 0; none.y1 = -1; none.w = 0;
  none.m = none.vx = none.vy = nullptr;
  const size_t lds = sizeof(double2) * 3 * padlen(s->H);
  CHK(with_rows<3>(s->px, [&](auto F, int nt) -> int {
    auto *kern = nl_kernel<decltype(F)>(s);
    KLAUNCH(kern, na + nb, nt, lds, s->stream, s->T[0], s->Bp, s->u1, s->u2,
            s->sponge_on ? s->ms : nullptr, none, (int)s->penal_on, s->T[2], s->penal_on ? s->T[3] : nullptr,
            F, s->twx, nl_consts(s),
            s->umax_part, s->ny, s->dscal, s->fp, 0.0, 0.0, 0, res_dev(s, s->slot), 0, na, b1 + 1, 0,
            s->penal_on ? s->rowpen : nullptr, (int)(s->p.iSponge == 10));
    return FSIBE_OK;
  }));
  s->Rcp = s->T[2];
  s->k2_ready = true;
  return FSIBE_OK;
}

static RowStepArgs row_step_args(const fsibe_sim *s, const MaskBox &mb) {
  RowStepArgs a;
  a.Cw = s->T[0]; a.Cpsi = s->T[1]; a.Cpsiy = s->T[2]; a.Cwy = s->T[7];
  a.u1 = s->u1; a.u2 = s->u2; a.vor_mean = s->vor_mean; a.ms = s->sponge_on ? s->ms : nullptr;
  a.mb = mb; a.win = s->win[0]; a.win2 = s->win[1];
  a.sums = rows_dev(s, s->slot); a.umax_part = s->umax_part;
  a.Rq = s->T[4]; a.Rqy = s->T[5]; a.Rc = s->T[8];
  a.s = s->dscal; a.c = s->sc;
  return a;
}
static ColStepArgs col_step_args(const fsibe_sim *s, const MaskBox &mb, const double2 *Rc, bool explicit_step,
                                 bool next) {
  ColStepArgs a;
  // without penalisation K2 leaves Rpx unwritten (it is 0) and the stage skips it
  a.Rc = Rc; a.Rpx = s->penal_on ? s->T[3] : nullptr;
  a.W0 = s->W[s->n0]; a.NL1 = s->NL[s->n1]; a.NL0 = s->NL[s->n0]; a.W1 = s->W[s->n1];
  a.o[0] = s->T[0]; a.o[1] = s->T[1]; a.o[2] = s->T[2];
  a.o[3] = s->forces_on && s->visc ? s->T[3] : nullptr;
  a.o[4] = next ? s->T[7] : nullptr;
  a.s = s->dscal; a.explicit_step = explicit_step;
  rpx_rows(s, mb, a.py0, a.py1);
  stress_rows(s, a.r0, a.r1);
  a.c = s->sc;
  return a;
}

// K1 .. K6 of a step: the new vorticity, velocity, pressure right-hand
// sides and the row sums.  next: another step follows in the same call, and
// its dw/dy column and convective term are formed here, where their inputs
// are at hand
static int evolve_fluid(fsibe_sim *s, double time, double dt0, bool explicit_step, bool next = false) {
  if (s->p.iBeam > 0 && !s->have_beam) return set_err(FSIBE_ESTATE, "fsibe_create_mask must be called first");
  std::vector<double>().swap(s->restored);
  if (!s->have_beam)  // no beam: walls / cylinder only (create_mask.f90:34-69)
    CHK(fsibe_create_mask(s, time, nullptr, nullptr, nullptr, nullptr, nullptr, 0.0, nullptr));
  const int n0 = s->n0, n1 = s->n1;
  if (explicit_step) {
    PROF_BEGIN(s, P_VEL);
    CHK(velocity_only(s, time));
    prof_end(s, P_VEL);
  }
  const bool sp10 = s->p.iSponge == 10 && s->penal_on && s->ms;
  const bool k2_ahead = s->k2_ready && s->k1_ready && s->k1_level == n0;
  s->k2_ready = false;
  if (s->k1_ready && s->k1_level == n0) {
    s->k1_ready = false;  // K1 of this step was launched ahead (run_one)
  } else {
    s->k1_ready = false;
    if (s->tape) tape_k1_place(s);
    CHK(launch_k1(s, n0));
  }
  MaskBox mb = mask_box(s);
  if (!k2_ahead) s->Rcp = s->T[2];
  // K2 (block 0 also computes the K3 scalars from the previous u_max partials).
  // When the convective part of every row went ahead, the penalisation of
  // this mask box's rows remains.
  {
    const size_t lds = sizeof(double2) * 3 * padlen(s->H);
    PROF_BEGIN(s, P_ROWS_NL);
    if (k2_ahead) {
      const int y0 = mb.x1 >= mb.x0 ? mb.y0 : 0, nrow = mb.x1 >= mb.x0 ? mb.y1 - mb.y0 + 1 : 0;
      CHK(with_rows<3>(s->px, [&](auto F, int nt) -> int {
        if (s->pipe)
          KLAUNCH_EV(k_rows_pen<decltype(F)>, nrow + 1, nt, lds, s->stream, s->ev_dt, s->u1, s->u2, mb, s->Rcp, s->T[3],
                     F, s->twx, s->sc, y0, nrow, s->rowpen, s->umax_part, s->ny, s->dscal, s->fp, time, dt0,
                     (int)explicit_step, res_dev(s, s->slot));
        else
          KLAUNCH(k_rows_pen<decltype(F)>, nrow + 1, nt, lds, s->stream, s->u1, s->u2, mb, s->Rcp, s->T[3],
                  F, s->twx, s->sc, y0, nrow, s->rowpen, s->umax_part, s->ny, s->dscal, s->fp, time, dt0,
                  (int)explicit_step, res_dev(s, s->slot));
        return FSIBE_OK;
      }));
    } else if (s->pipe) {
      // ev_dt at K2's end: the host reads dt1 and then the previous step's
      // results (kernels before this one in the stream)
      CHK(with_rows<3>(s->px, [&](auto F, int nt) -> int {
        auto *kern = nl_kernel<decltype(F)>(s);
        KLAUNCH_EV(kern, s->ny, nt, lds, s->stream, s->ev_dt, s->T[0], s->Bp, s->u1, s->u2,
                   s->sponge_on ? s->ms : nullptr, mb, (int)s->penal_on, s->T[2], s->penal_on ? s->T[3] : nullptr,
                   F, s->twx, nl_consts(s),
                   s->umax_part, s->ny, s->dscal, s->fp, time, dt0, (int)explicit_step, res_dev(s, s->slot), 0,
                   s->ny, 0, 1, s->penal_on ? s->rowpen : nullptr, (int)(s->p.iSponge == 10));
        return FSIBE_OK;
      }));
    } else {
      CHK(with_rows<3>(s->px, [&](auto F, int nt) -> int {
        auto *kern = nl_kernel<decltype(F)>(s);
        KLAUNCH(kern, s->ny, nt, lds, s->stream, s->T[0], s->Bp, s->u1, s->u2,
                s->sponge_on ? s->ms : nullptr, mb, (int)s->penal_on, s->T[2], s->penal_on ? s->T[3] : nullptr,
                F, s->twx, nl_consts(s),
                s->umax_part, s->ny, s->dscal, s->fp, time, dt0, (int)explicit_step, res_dev(s, s->slot), 0, s->ny,
                0, 1, s->penal_on ? s->rowpen : nullptr, (int)(s->p.iSponge == 10));
        return FSIBE_OK;
      }));
    }
    prof_end(s, P_ROWS_NL);
  }
  if (s->tape) CHK(tape_fluid(s, explicit_step));
  if (s->p.iMeanVelocity == 11) {
    k_mean11<<<1, 256, 0, s->stream>>>(s->penal_on ? s->rowpen : nullptr, s->ny,
                                       1.0 / ((double)s->nx * (double)s->ny), s->dscal, n0, n1, (int)explicit_step,
                                       s->p.U_mean_true);
    HIPCHK(hipGetLastError());
  }
  if (sp10) {
    // NavierStokes.f90:108-109: ixmin = nint((xl - SpongeSize)/dx), ixmax = nx - 1 - 15
    const int ixmin = (int)lround((s->p.xl - s->p.SpongeSize) / s->dx), ixmax = s->nx - 1 - 15;
    if (ixmin < 0) return set_err(FSIBE_EARG, "iSponge=10: SpongeSize exceeds the domain");
    if (ixmin <= ixmax) {
      const size_t lds = sizeof(double2) * 2 * padlen(s->H);
      CHK(with_rows<1>(s->px, [&](auto F, int nt) -> int {
        KLAUNCH(k_rows_sponge10<decltype(F)>, s->ny, nt, lds, s->stream, s->T[4], s->ms, s->T[3], ixmin, ixmax, F,
                s->twx, s->sc);
        return FSIBE_OK;
      }));
    }
  }
  // K4, K5: the fused column stage where the grid has one
  next = next && !sp10 && s->p.iMeanVelocity != 11;
  int rc = FSIBE_OK;
  PROF_BEGIN(s, P_COLS_AB2);
  const bool fused_cols = with_col_step(s->ny, s->H, s->penal_on, next, [&](auto S) {
    using ST = decltype(S);
    rc = [&]() -> int {
      KLAUNCH(k_col_step<ST>, s->H / ST::TX, ST::THREADS, ST::LDS, s->stream,
              col_step_args(s, mb, s->Rcp, explicit_step, next), s->twy);
      return FSIBE_OK;
    }();
  });
  CHK(rc);
  if (!fused_cols) {
    CHK(with_cols_sel<2>(s->py, s->H, sim_sel(s, 1, 1), [&](auto F, int nt, int TX) -> int {
      const size_t lds = k4_lds(s->ny, s->penal_on, TX);
      int py0, py1;
      rpx_rows(s, mb, py0, py1);
      // without penalisation K2 leaves Rpx unwritten (it is 0) and K4 skips it
      if constexpr (!always_col_step(fixed_len<decltype(F)>::v))
        KLAUNCH(k_cols_ab2<decltype(F)>, s->H / TX, nt, lds, s->stream, s->Rcp, s->penal_on ? s->T[3] : nullptr,
                s->W[n0], s->NL[n1],
                s->NL[n0], s->W[n1], s->dscal, (int)explicit_step, F, s->twy, s->sc, py0, py1);
      return FSIBE_OK;
    }));
  }
  prof_end(s, P_COLS_AB2);
  if (!fused_cols) {
    // K5: omega, psi, i ky psi (, -ky^2 psi) of vortk(n1)
    const bool st = s->forces_on && s->visc;
    double2 *outs[4] = {s->T[0], s->T[1], s->T[2], s->T[3]};
    const int fsel[4] = {0, 1, 2, 3};
    int r0_3, r1_3;
    stress_rows(s, r0_3, r1_3);
    PROF_BEGIN(s, P_COLS_W1);
    CHK(cols_inv_fields(s, s->W[n1], outs, fsel, st ? 4 : 3, 2, r0_3, r1_3));
    prof_end(s, P_COLS_W1);
  }
  // K6, with the next step's convective term where the grid has the fused
  // row stage and the column stage left it the dw/dy column
  bool conv = false;
  {
    const size_t lds = sizeof(double2) * 3 * padlen(s->H);
    PROF_BEGIN(s, P_ROWS_PRESS);
    auto launch = [&](auto nx) {
      constexpr bool NEXT = decltype(nx)::value;
      return with_row_step<NEXT>(s->H, s->ny, s->pressure_on, [&](auto S) {
        using ST = decltype(S);
        auto *kern = s->pressure_on ? &k_row_step<ST, true, NEXT> : &k_row_step<ST, false, NEXT>;
        rc = [&]() -> int {
          KLAUNCH(kern, s->ny / ST::RPB, ST::THREADS, ST::LDS, s->stream, row_step_args(s, mb), s->twx);
          return FSIBE_OK;
        }();
      });
    };
    conv = next && fused_cols && launch(std::true_type{});
    const bool fused_rows = conv || launch(std::false_type{});
    CHK(rc);
    if (!fused_rows)
      CHK(with_rows<3>(s->px, [&](auto F, int nt) -> int {
        // the step's instances: mode 1, with or without the pressure rhs
        using FT = decltype(F);
        if constexpr (!always_row_step(fixed_len<FT>::v)) {
          auto *kern = s->pressure_on ? &k_rows_press<FT, 1, 1> : &k_rows_press<FT, 1, 0>;
          KLAUNCH(kern, s->ny, nt, lds, s->stream, s->T[0], s->T[1], s->T[2], s->u1, s->u2, s->vor_mean, mb, s->win[0],
                  s->win[1], rows_dev(s, s->slot), s->umax_part, s->T[4], s->T[5], s->dscal, 0.0, 0.0, 1,
                  (int)s->pressure_on, F, s->twx, s->sc);
        }
        return FSIBE_OK;
      }));
    prof_end(s, P_ROWS_PRESS);
  }
  if (next && fused_cols) {
    s->k1_ready = true;
    s->k1_level = n1;
    s->Bp = s->T[7];
    s->kcA = s->sc.kc;
    if (conv) {
      s->k2_ready = true;
      s->Rcp = s->T[8];
    }
  }
  s->slot_fluid[s->slot] = true;  // the host adds the row sums of K6
  return FSIBE_OK;
}

// K7: the inverse column transform of the pressure (T4, T5) on rows r0 .. r1, into T6
static int launch_press(fsibe_sim *s, int r0, int r1) {
  int rc = FSIBE_OK;
  const bool fast = with_press_step(s->ny, s->H, [&](auto S) {
    using ST = decltype(S);
    PressArgs a;
    a.Rq = s->T[4]; a.Rqy = s->T[5]; a.Cq = s->T[6]; a.r0 = r0; a.r1 = r1; a.c = s->sc;
    rc = [&]() -> int {
      KLAUNCH(k_press_step<ST>, s->H / ST::TX, ST::THREADS, ST::LDS, s->stream, a, s->twy);
      return FSIBE_OK;
    }();
  });
  if (fast) return rc;
  return with_cols_sel<2>(s->py, s->H, sim_sel(s, 3, 1), [&](auto F, int nt, int TX) -> int {
    const size_t lds = sizeof(double2) * 2 * TX * padlen(s->ny);
    KLAUNCH(k_cols_press<decltype(F)>, s->H / TX, nt, lds, s->stream, s->T[4], s->T[5], s->T[6], r0, r1, F, s->twy,
            s->sc);
    return FSIBE_OK;
  });
}

// K7 + K8: the static pressure and the stresses on the rows/columns the
// interpolation needs (the box of the force geometry)
static int evolve_pressure_box(fsibe_sim *s) {
  s->press_box_valid = false;
  if (s->forces_on && s->forces_ready && !s->fbox.empty()) {
    const Box &fb = s->fbox;
    {
      PROF_BEGIN(s, P_COLS_PRESS);
      CHK(launch_press(s, fb.y0, fb.y1));
      prof_end(s, P_COLS_PRESS);
    }
    {
      const size_t lds = sizeof(double2) * 3 * padlen(s->H);
      PROF_BEGIN(s, P_ROWS_BOX);
      CHK(with_rows<3>(s->px, [&](auto F, int nt) -> int {
        KLAUNCH(k_rows_box<decltype(F)>, fb.h(), nt, lds, s->stream, s->T[6], s->T[1], s->T[2], s->T[3], s->u1,
                s->u2, s->fb_p, s->fb_sa, s->fb_sb, fb.y0, fb.x0, fb.x1, fb.w(), (int)s->visc, F, s->twx, s->sc);
        return FSIBE_OK;
      }));
      prof_end(s, P_ROWS_BOX);
    }
    s->press_box_valid = true;
  }
  return FSIBE_OK;
}

static int evolve(fsibe_sim *s, double time, double dt0, bool explicit_step, bool next = false) {
  CHK(evolve_fluid(s, time, dt0, explicit_step, next));
  return evolve_pressure_box(s);
}

// end_ev (optional): recorded at the force kernel's end by its own dispatch;
// *recorded tells whether it was (no launch, or kernel timing: it was not)
static int launch_forces(fsibe_sim *s, hipEvent_t end_ev = nullptr, bool *recorded = nullptr) {
  if (recorded) *recorded = false;
  if (!s->forces_on || !s->forces_ready || !s->press_box_valid) return FSIBE_OK;
  const double *tg = reinterpret_cast<const double *>(s->d_stage + s->off_tg);
  double *val = reinterpret_cast<double *>(s->d_stage + s->off_val);
  if (s->ntg <= 0) return set_err(FSIBE_ESTATE, "no interpolation targets");
  // one block per beam node and per pair of circle points, beam after beam
  const int units = s->nb * (s->fg.ns + s->fg.nc);
  if (s->ntg != s->nb * (6 * s->fg.ns + 3 * 2 * s->fg.nc) || s->fg.nc > kNC)
    return set_err(FSIBE_ESTATE, "interpolation targets do not match the beam");
  PROF_BEGIN(s, P_INTERP);
  const double *nd = reinterpret_cast<const double *>(s->d_stage + s->off_nd);
  const double *cd = reinterpret_cast<const double *>(s->d_stage + s->off_cd);
  if (end_ev && !t_prof_start) {
    hipExtLaunchKernelGGL(k_forces, dim3(units), dim3(kForceThreads), 0u, s->stream, nullptr, end_ev, 0u, tg, s->fb_p,
                          s->fb_sa, s->fb_sb, s->fg, val, nd, cd, pbeam_dev(s, s->slot),
                          pbeam_dev(s, s->slot) + nodes_all(s), parts_dev(s, s->slot));
    if (recorded) *recorded = true;
  } else {
    k_forces<<<units, kForceThreads, 0, s->stream>>>(tg, s->fb_p, s->fb_sa, s->fb_sb, s->fg, val, nd, cd,
                                                     pbeam_dev(s, s->slot), pbeam_dev(s, s->slot) + nodes_all(s),
                                                     parts_dev(s, s->slot));
  }
  HIPCHK(hipGetLastError());
  prof_end(s, P_INTERP);
  s->slot_forces[s->slot] = true;
  s->slot_units[s->slot] = units;
  return FSIBE_OK;
}

// the first beam's per-beam fields of last_b into last
static void sync_last(fsibe_sim *s) {
  const fsibe_step_out &b = s->last_b[0];
  fsibe_step_out &r = s->last;
  for (int i = 0; i < 2; ++i) {
    r.Force[i] = b.Force[i]; r.Force_unst[i] = b.Force_unst[i]; r.Force_press[i] = b.Force_press[i];
  }
  for (int i = 2; i < 10; ++i) r.bsi[i] = b.bsi[i];
  r.fx_int = b.fx_int; r.fy_int = b.fy_int;
  r.ibes_iter = b.ibes_iter;
}

// Result slot k's head: dt1, u_max and the node loads, the part the beam
// solve needs (GetForces' p_beam, tau_beam)
static void parse_head(fsibe_sim *s, int k) {
  const int nsb = nodes_all(s), nb = s->nb, nr = std::max(nb, 1);
  const char *base = s->h_res + (size_t)k * s->res_stride;
  const StepOutDev *o = reinterpret_cast<const StepOutDev *>(base);
  fsibe_step_out &r = s->last;
  r.dt1 = o->dt1;
  r.u_max = o->u_max;
  r.status = 0;
  r.ibes_iter = 0;
  if (s->slot_forces[k]) {
    const double *pb = reinterpret_cast<const double *>(base + sizeof(StepOutDev));
    for (int i = 0; i < s->nb * s->ns; ++i) { s->pbeam[i] = pb[i]; s->tbeam[i] = pb[nsb + i]; }
  }
  for (int ib = 0; ib < nr; ++ib) {
    fsibe_step_out &rb = s->last_b[ib];
    rb.dt1 = r.dt1; rb.u_max = r.u_max; rb.status = 0; rb.ibes_iter = 0;
  }
}

// Result slot k's row sums of the fluid step (energies cal_energy
// NavierStokes.f90:236-256, cal_drag Force / Force_unst :567-589,
// BeamSurfaceIntegral drag/lift BeamForces.f90:483-486) added over rows in
// order; completes s->last (after parse_head of the same slot and the beam
// solve, whose iteration count it keeps)
static void parse_rows(fsibe_sim *s, int k) {
  const int nb = s->nb, nr = std::max(nb, 1);
  const char *base = s->h_res + (size_t)k * s->res_stride;
  // the force kernel's per-unit terms: Force_press and the surface
  // integrals (not needed by the beam solve, which takes p_beam, tau_beam)
  if (s->slot_forces[k]) {
    s->slot_forces[k] = false;
    const double *part = reinterpret_cast<const double *>(base + parts_off(s));
    const int per = s->slot_units[k] / nr;
    for (int ib = 0; ib < nr; ++ib) {
      fsibe_step_out &rb = s->last_b[ib];
      double tot[8] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
      for (int u = ib * per; u < (ib + 1) * per; ++u)
        for (int i = 0; i < 8; ++i) tot[i] += part[8 * u + i];
      rb.Force_press[0] = tot[0];
      rb.Force_press[1] = tot[1];
      rb.fx_int = tot[0];
      rb.fy_int = tot[1];
      if (s->fg.bsi_on) {
        rb.bsi[2] = tot[2] + tot[4] + tot[6];
        rb.bsi[3] = tot[3] + tot[5] + tot[7];
        rb.bsi[4] = tot[2]; rb.bsi[5] = tot[4]; rb.bsi[6] = tot[6];
        rb.bsi[7] = tot[3]; rb.bsi[8] = tot[5]; rb.bsi[9] = tot[7];
      }
    }
  }
  const StepOutDev *o = reinterpret_cast<const StepOutDev *>(base);
  fsibe_step_out &r = s->last;
  const double dxdy = s->dx * s->dy;
  if (s->slot_fluid[k]) {
    s->slot_fluid[k] = false;
    const double *rows = reinterpret_cast<const double *>(base + rows_off(s));
    double tot[kNSUM];
    for (int i = 0; i < kNSUM; ++i) tot[i] = 0.0;
    for (int y = 0; y < s->ny; ++y)
      for (int i = 0; i < kNSUM; ++i) tot[i] += rows[(size_t)y * kNSUM + i];
    r.energies[0] = dxdy * sqrt(tot[0]);
    r.energies[1] = 0.5 * dxdy * tot[1];
    r.energies[2] = s->p.nu * dxdy * tot[0];
    r.energies[3] = dxdy * tot[2];
    r.energies[4] = dxdy * tot[3];
    r.energies[5] = dxdy * s->p.U_mean_true * tot[4];
    // BeamSurfaceIntegral's drag and lift are whole-grid sums, the same for
    // every beam (BeamForces.f90:483-486)
    r.bsi[0] = tot[5] * dxdy;
    r.bsi[1] = tot[6] * dxdy;
    // cal_drag per beam over its own window (NavierStokes.f90:528-589)
    for (int ib = 0; ib < nb; ++ib) {
      fsibe_step_out &rb = s->last_b[ib];
      const double *t = tot + 7 + 4 * ib;
      rb.Force[0] = t[0] * dxdy;
      rb.Force[1] = t[1] * dxdy;
      const double dn = t[2] * dxdy * s->p.eps, ln = t[3] * dxdy * s->p.eps;
      if (s->unst_ready[ib]) {
        rb.Force_unst[0] = (dn - s->drag_unst_old[ib]) / o->dt1;
        rb.Force_unst[1] = (ln - s->lift_unst_old[ib]) / o->dt1;
      } else {
        rb.Force_unst[0] = 0.0;
        rb.Force_unst[1] = 0.0;
      }
      s->drag_unst_old[ib] = dn;
      s->lift_unst_old[ib] = ln;
      s->unst_ready[ib] = true;
    }
    if (nb > 0) {
      s->jsum_f += -s->last_b[0].Force[0] * o->dt1;
      s->jsum_t += o->dt1;
    }
  }
  // each beam's record carries the step's common fields; s->last the first
  // beam's per-beam fields
  for (int ib = 0; ib < nr; ++ib) {
    fsibe_step_out &rb = s->last_b[ib];
    for (int i = 0; i < 6; ++i) rb.energies[i] = r.energies[i];
    rb.bsi[0] = r.bsi[0]; rb.bsi[1] = r.bsi[1];
  }
  sync_last(s);
}

// Read result slot k (its kernels have finished) into s->last: the head
// (dt1, u_max, the force terms of k_forces, Force_press :261-267 and the
// surface integrals :485-496, added over units in order, and p_beam /
// tau_beam), then the row sums.  Each part is read once per step.
static void parse_results(fsibe_sim *s, int k) {
  parse_head(s, k);
  parse_rows(s, k);
}

// the coupled loop's deferred row sums of the previous step, if any
static void flush_rows(fsibe_sim *s) {
  if (s->rows_pending < 0) return;
  parse_rows(s, s->rows_pending);
  s->rows_pending = -1;
}

static int fetch_results(fsibe_sim *s) {
  HIPCHK(hipStreamSynchronize(s->stream));
  s->upload_pending = 0;
  prof_collect(s);
  parse_results(s, s->slot);
  return FSIBE_OK;
}

extern "C" int fsibe_evolve_explicit(fsibe_sim *s, double time, double *dt1) {
  if (!s) return set_err(FSIBE_EARG, "null sim");
  CHK(evolve(s, time, 0.0, true));
  CHK(fetch_results(s));
  if (dt1) *dt1 = s->last.dt1;
  return FSIBE_OK;
}

extern "C" int fsibe_evolve_ab2(fsibe_sim *s, double time, double dt0, double *dt1) {
  if (!s) return set_err(FSIBE_EARG, "null sim");
  if (!(dt0 > 0.0)) return set_err(FSIBE_EARG, "dt0 must be > 0 (take the startup step first)");
  CHK(evolve(s, time, dt0, false));
  CHK(fetch_results(s));
  if (dt1) *dt1 = s->last.dt1;
  return FSIBE_OK;
}

extern "C" int fsibe_get_forces(fsibe_sim *s, double time, double *pressure_beam, double *tau_beam,
                                double Force_press[2]) {
  (void)time;  // the soft-startup factor uses the time given to fsibe_create_mask
  if (!s) return set_err(FSIBE_EARG, "null sim");
  if (!s->forces_on) return set_err(FSIBE_ESTATE, "forces need iSaveBeam>0 (pressure is not computed otherwise)");
  if (!s->press_box_valid) return set_err(FSIBE_ESTATE, "no pressure of the current step (evolve first)");
  CHK(launch_forces(s));
  CHK(fetch_results(s));
  for (int i = 0; i < s->nb * s->ns; ++i) {
    if (pressure_beam) pressure_beam[i] = s->pbeam[i];
    if (tau_beam) tau_beam[i] = s->tbeam[i];
  }
  if (Force_press)
    for (int ib = 0; ib < std::max(s->nb, 1); ++ib) {
      Force_press[2 * ib] = s->last_b[ib].Force_press[0];
      Force_press[2 * ib + 1] = s->last_b[ib].Force_press[1];
    }
  return FSIBE_OK;
}

extern "C" int fsibe_get_step_out(fsibe_sim *s, fsibe_step_out *out) {
  if (!s || !out) return set_err(FSIBE_EARG, "null argument");
  *out = s->last;
  return FSIBE_OK;
}

extern "C" int fsibe_get_step_out_beam(fsibe_sim *s, int ib, fsibe_step_out *out) {
  if (!s || !out) return set_err(FSIBE_EARG, "null argument");
  if (ib < 0 || ib >= std::max(s->nb, 1)) return set_err(FSIBE_EARG, "beam %d of %d", ib, s->nb);
  *out = s->last_b[ib];
  out->status = s->last.status;
  return FSIBE_OK;
}

// ---- time loop (time_step.f90:120-162, :178-341) ---------------------------
// the beam of the library's solid solver, for iFLUSI=1
static int ensure_solid(fsibe_sim *s) {
  if (s->p.iBeam < 1) return set_err(FSIBE_EARG, "iFLUSI=1 without a beam");
  for (int ib = 0; ib < s->nb; ++ib)
    if (!s->solid[ib]) CHK(fsibe_solid_create_beam(&s->p, ib, &s->solid[ib]));
  return FSIBE_OK;
}

static void beam_from_solid(fsibe_sim *s) {
  const int ns = s->ns;
  for (int ib = 0; ib < s->nb; ++ib) {
    const ibes::Beam &b = s->solid[ib]->b;
    const size_t o = (size_t)ib * ns;
    std::copy(b.x.begin(), b.x.end(), s->bx.begin() + o);
    std::copy(b.y.begin(), b.y.end(), s->by.begin() + o);
    std::copy(b.vx.begin(), b.vx.end(), s->bvx.begin() + o);
    std::copy(b.vy.begin(), b.vy.end(), s->bvy.begin() + o);
    std::copy(b.theta.begin(), b.theta.end(), s->btheta.begin() + o);
    std::copy(b.theta_dot.begin(), b.theta_dot.end(), s->btheta_dot.begin() + o);
  }
}

// GetForces' loads -> GravityImpulse + SolidSolverWrapper(time, dt1), one
// IBES solve per beam (SolidSolver.f90:25-27) -> pressure_old = pressure_new
// (time_step.f90:199-228).  The emergency brake of any beam ends the run.
static int solid_step(fsibe_sim *s) {
  int brake = 0;
  for (int ib = 0; ib < s->nb; ++ib) {
    fsibe_solid *sd = s->solid[ib];
    ibes::Beam &b = sd->b;
    const int o = ib * s->ns;
    for (int i = 0; i < s->ns; ++i) { b.pressure_new[i] = s->pbeam[o + i]; b.tau_new[i] = s->tbeam[o + i]; }
    if (!sd->sv.step(s->time, s->dt1, b))
      return set_err(FSIBE_EDOMAIN, "beam %d: %s", ib + 1, sd->sv.err.c_str());
    s->last_b[ib].ibes_iter = sd->sv.iter;
    brake |= sd->sv.brake ? 1 : 0;
  }
  beam_from_solid(s);
  s->last.ibes_iter = s->last_b[0].ibes_iter;
  s->last.status = brake;
  return FSIBE_OK;
}

extern "C" int fsibe_sim_solid(fsibe_sim *s, fsibe_solid **out) {
  return fsibe_sim_solid_beam(s, 0, out);
}

extern "C" int fsibe_sim_solid_beam(fsibe_sim *s, int ib, fsibe_solid **out) {
  if (!s || !out) return set_err(FSIBE_EARG, "null argument");
  if (ib < 0 || ib >= std::max(s->nb, 1)) return set_err(FSIBE_EARG, "beam %d of %d", ib, s->nb);
  CHK(ensure_solid(s));
  *out = s->solid[ib];
  return FSIBE_OK;
}

// mouvement(time) of every beam (create_mask.f90:77): alpha[ib], LE[6 ib ..]
static void motion_all(const fsibe_sim *s, double time, double *alpha, double *LE) {
  for (int ib = 0; ib < s->nb; ++ib) {
    double x0 = 0.0, y0 = 0.0, ph = 0.0, at, att;
    beam_placement(s->p, ib, x0, y0, ph);
    mouvement_host(s->p, s->p.iMotion, x0, y0, s->p.AngleBeam, ph, time, alpha[ib], at, att, LE + 6 * ib);
  }
}

// integrate_position(time, beams(i)) of every beam (time_step.f90:215-217)
static void integrate_all(fsibe_sim *s, double time) {
  for (int ib = 0; ib < s->nb; ++ib) {
    double x0 = 0.0, y0 = 0.0, ph = 0.0;
    beam_placement(s->p, ib, x0, y0, ph);
    const size_t o = (size_t)ib * s->ns;
    integrate_position_host(s->p, s->p.iMotion, x0, y0, ph, time, s->btheta.data() + o, s->btheta_dot.data() + o,
                            s->bx.data() + o, s->by.data() + o, s->bvx.data() + o, s->bvy.data() + o);
  }
}

// One step of the loop.  pipe: do not wait for the step to finish; wait only
// for dt1 (written by the nonlinear-term kernel), read the previous step's
// results, and return so that the host prepares the next step's geometry
// while this one runs.  next (pipe): another step follows in this call.
static int run_one(fsibe_sim *s, bool pipe, bool k1_ahead, bool next = false) {
  s->pipe = pipe;
  const fsibe_params &p = s->p;
  const bool moving = (p.iSponge >= 4 && s->time < p.T_fullspeed) || p.iFLUSI == 1 || p.iMotion > 0;
  // iFLUSI=1 waits for every step: the mask's record goes up (and its copy
  // starts) before the host bounds the force box (the device builds the
  // interpolation targets), which K5 and the pressure box need
  const bool split = !pipe && p.iFLUSI == 1 && p.iBeam > 0 && s->forces_on;
  if (p.iBeam > 0 && (moving || !s->have_beam)) {
    double alpha[2], LE[12];
    motion_all(s, s->time, alpha, LE);
    CHK(create_mask_impl(s, s->time, s->bx.data(), s->by.data(), s->bvx.data(), s->bvy.data(),
                         s->btheta.data(), alpha, LE, !split));
  } else if (p.iBeam > 0) {
    // soft-startup factor follows time
    CHK(stage_writable(s));
    CHK(build_geometry(s, s->time));
    CHK(upload_geometry(s));
  }
  if (s->startup_done) s->dt0 = s->dt1;
  if (split) {
    // the force box first: K5 stores -ky^2 psi on its rows only
    CHK(force_geometry(s, s->time));
    CHK(evolve_fluid(s, s->time, s->startup_done ? s->dt0 : 0.0, !s->startup_done));
    CHK(evolve_pressure_box(s));
  } else {
    CHK(evolve(s, s->time, s->startup_done ? s->dt0 : 0.0, !s->startup_done, pipe && next));
  }
  // iFLUSI=1 with the next step ahead: ev_step at the force kernel's end,
  // carried by its dispatch (a marker after it would idle the queue first)
  bool step_recorded = false;
  if (s->forces_on) CHK(launch_forces(s, (!pipe && k1_ahead) ? s->ev_step : nullptr, &step_recorded));
  if (!pipe && k1_ahead) {
    // iFLUSI=1: the next step's K1 runs while the host solves the beam
    if (!step_recorded) HIPCHK(hipEventRecord(s->ev_step, s->stream));
    CHK(launch_k1(s, s->n1, true));
    s->k1_ready = true;
    s->k1_level = s->n1;
    CHK(launch_k2_ahead(s));
    CHK(arm_upload(s));
    // the beam solver's predictor needs only the state at t_n: it runs while
    // the step's fluid kernels finish
    if (p.iFLUSI == 1 && p.iBeam > 0 && s->time > p.T_release)
      for (int ib = 0; ib < s->nb; ++ib)
        if (s->solid[ib]) (void)s->solid[ib]->sv.predict(s->time, s->solid[ib]->b);
    // the previous step's row sums while this step's kernels run
    flush_rows(s);
    CHK(wait_event(s->ev_step, "the step's results (pressure and force kernels)"));
    s->upload_pending = 0;
    CHK(gate_check(s));
    // the beam solve needs the head; the row sums are read during the next
    // step, which writes the other slot
    parse_head(s, s->slot);
    s->dt1 = s->last.dt1;
    s->rows_pending = s->slot;
    s->slot ^= 1;
  } else if (!pipe) {
    flush_rows(s);
    const double th0 = now_ms();
    CHK(fetch_results(s));
    CHK(gate_check(s));
    prof_host(s, P_FORCES, th0);
    s->dt1 = s->last.dt1;
  } else {
    CHK(wait_event(s->ev_dt, "the step's time step dt1 (nonlinear-term kernel)"));
    s->upload_pending = 0;  // the geometry upload precedes the nonlinear-term kernel
    s->dt1 = *reinterpret_cast<volatile const double *>(s->h_res + (size_t)s->slot * s->res_stride);
    if (s->res_pending) parse_results(s, s->slot ^ 1);  // finished before this step started
    s->res_pending = true;
    s->slot ^= 1;
  }
  if (p.iFLUSI == 1 && p.iBeam > 0) {
    const double th0 = now_ms();
    CHK(solid_step(s));
    prof_host(s, P_SCALARS, th0);
  } else if (p.iFLUSI == 0 && p.iMotion > 0 && p.iBeam > 0) {
    integrate_all(s, s->time);
    s->beam_time = s->time;
  }
  std::swap(s->n0, s->n1);
  s->time = s->time + s->dt1;
  if (s->startup_done) s->it++;
  s->startup_done = true;
  return FSIBE_OK;
}

static void init_beam_host(fsibe_sim *s) {
  // init_beam.f90:130-167 for every beam
  double alpha[2], LE[12];
  motion_all(s, 0.0, alpha, LE);
  for (int ib = 0; ib < s->nb; ++ib)
    for (int n = 0; n < s->ns; ++n) {
      const int i = ib * s->ns + n;
      s->bx[i] = LE[6 * ib] + (double)n * s->ds;
      s->by[i] = LE[6 * ib + 1];
      s->bvx[i] = 0.0; s->bvy[i] = 0.0; s->btheta[i] = 0.0; s->btheta_dot[i] = 0.0;
    }
  integrate_all(s, 0.0);
  s->beam_time = 0.0;
}

static int sim_tune_cols(fsibe_sim *s);

extern "C" int fsibe_run(fsibe_sim *s, int nsteps, fsibe_step_out *out) {
  if (!s) return set_err(FSIBE_EARG, "null sim");
  if (nsteps > 0) CHK(sim_tune_cols(s));
  const bool fsi = s->p.iFLUSI == 1 && s->p.iBeam > 0;
  if (fsi) {
    CHK(ensure_solid(s));
    if (!s->startup_done && !s->have_beam) beam_from_solid(s);
  } else if (!s->startup_done && s->time == 0.0 && s->p.iBeam > 0 && !s->have_beam) {
    init_beam_host(s);
  }
  // kernel timing needs a synchronisation per step; so does the solid
  // solver, which needs the step's loads before the next step's mask
  const bool pipe = !s->prof.on && !fsi;
  int rc = FSIBE_OK;
  for (int k = 0; k < nsteps; ++k) {
    if (!(s->time < s->p.Time_end)) break;
    // the next step's first kernel goes ahead of the host's beam solve when
    // there is a next step in this call (event timing keeps the plain order)
    const bool ahead = fsi && !s->prof.on && k + 1 < nsteps;
    rc = run_one(s, pipe, ahead, k + 1 < nsteps);
    if (rc != FSIBE_OK) break;
    if (s->last.status == 1) break;  // continue_timestep = .false.
  }
  open_gate(s);
  s->k1_ready = false;
  s->k2_ready = false;
  s->pipe = false;
  flush_rows(s);
  if (s->res_pending) {
    HIPCHK(hipStreamSynchronize(s->stream));
    s->upload_pending = 0;
    parse_results(s, s->slot ^ 1);
    s->res_pending = false;
  }
  if (rc != FSIBE_OK) return rc;
  if (out) *out = s->last;
  return FSIBE_OK;
}

extern "C" int fsibe_get_time(fsibe_sim *s, double *time, double *dt1, int *it) {
  if (!s) return set_err(FSIBE_EARG, "null sim");
  if (time) *time = s->time;
  if (dt1) *dt1 = s->dt1;
  if (it) *it = s->it;
  return FSIBE_OK;
}

extern "C" int fsibe_get_beam(fsibe_sim *s, double *x, double *y, double *vx, double *vy, double *theta,
                              double *pressure_new, double *tau_new) {
  if (!s) return set_err(FSIBE_EARG, "null sim");
  for (int i = 0; i < s->nb * s->ns; ++i) {
    if (x) x[i] = s->bx[i];
    if (y) y[i] = s->by[i];
    if (vx) vx[i] = s->bvx[i];
    if (vy) vy[i] = s->bvy[i];
    if (theta) theta[i] = s->btheta[i];
    if (pressure_new) pressure_new[i] = s->pbeam[i];
    if (tau_new) tau_new[i] = s->tbeam[i];
  }
  return FSIBE_OK;
}

// ---- field download --------------------------------------------------------
static int box_to_full(fsibe_sim *s, const double *box, const Box &b, double *host) {
  const size_t N = (size_t)s->nx * s->ny;
  std::vector<double> tmp((size_t)std::max(1, b.w() * b.h()));
  if (!b.empty()) {
    HIPCHK(hipMemcpyAsync(tmp.data(), box, sizeof(double) * (size_t)b.w() * b.h(), hipMemcpyDeviceToHost, s->stream));
    HIPCHK(hipStreamSynchronize(s->stream));
  }
  memset(host, 0, sizeof(double) * N);
  for (int y = 0; y < b.h(); ++y)
    memcpy(host + (size_t)(y + b.y0) * s->nx + b.x0, tmp.data() + (size_t)y * b.w(), sizeof(double) * b.w());
  return FSIBE_OK;
}

extern "C" int fsibe_get_field(fsibe_sim *s, int which, double *out) {
  if (!s || !out) return set_err(FSIBE_EARG, "null argument");
  const size_t N = (size_t)s->nx * s->ny;
  const int g = grid1d((size_t)s->H * (s->ny / 2));
  switch (which) {
    case FSIBE_FIELD_VORTK:
    case FSIBE_FIELD_NLK: {
      const double2 *src = which == FSIBE_FIELD_VORTK ? s->W[s->n0] : s->NL[s->n0];
      k_half_to_packed<<<g, 256, 0, s->stream>>>(src, s->fb_p, s->nx, s->ny);
      HIPCHK(hipGetLastError());
      HIPCHK(Transfer::get().download(out, s->fb_p, sizeof(double) * N, s->stream));
      s->press_box_valid = false;
      break;
    }
    case FSIBE_FIELD_U1: HIPCHK(Transfer::get().download(out, s->u1, sizeof(double) * N, s->stream)); break;
    case FSIBE_FIELD_U2: HIPCHK(Transfer::get().download(out, s->u2, sizeof(double) * N, s->stream)); break;
    case FSIBE_FIELD_VOR_MEAN:
      HIPCHK(Transfer::get().download(out, s->vor_mean, sizeof(double) * N, s->stream));
      break;
    case FSIBE_FIELD_MASK_SPONGE:
      if (s->ms) HIPCHK(Transfer::get().download(out, s->ms, sizeof(double) * N, s->stream));
      else memset(out, 0, sizeof(double) * N);
      break;
    case FSIBE_FIELD_MASK: return box_to_full(s, s->mask_m, s->mbox, out);
    case FSIBE_FIELD_MASKVX: return box_to_full(s, s->mask_vx, s->mbox, out);
    case FSIBE_FIELD_MASKVY: return box_to_full(s, s->mask_vy, s->mbox, out);
    case FSIBE_FIELD_VORT: {
      double2 *outs[1] = {s->T[6]};
      const int fsel[1] = {0};
      CHK(cols_inv_fields(s, s->W[s->n0], outs, fsel, 1));
      CHK(rows_c2r(s->nx, s->ny, s->px, s->twx, s->T[6], s->fb_sb, s->stream));
      HIPCHK(Transfer::get().download(out, s->fb_sb, sizeof(double) * N, s->stream));
      s->press_box_valid = false;
      break;
    }
    case FSIBE_FIELD_PRESS: {
      if (!s->pressure_on) { memset(out, 0, sizeof(double) * N); break; }
      // full-grid pressure from the last step's right-hand side (T4, T5)
      CHK(launch_press(s, 0, s->ny - 1));
      const size_t lds2 = sizeof(double2) * 3 * padlen(s->H);
      CHK(with_rows<3>(s->px, [&](auto F, int nt) -> int {
        KLAUNCH(k_rows_box<decltype(F)>, s->ny, nt, lds2, s->stream, s->T[6], s->T[1], s->T[2], s->T[3], s->u1,
                s->u2, s->fb_sb, s->fb_sa, s->fb_sa, 0, 0, s->nx - 1, s->nx, 0, F, s->twx, s->sc);
        return FSIBE_OK;
      }));
      HIPCHK(Transfer::get().download(out, s->fb_sb, sizeof(double) * N, s->stream));
      s->press_box_valid = false;
      break;
    }
    default: return set_err(FSIBE_EARG, "unknown field %d", which);
  }
  HIPCHK(hipStreamSynchronize(s->stream));
  return FSIBE_OK;
}

extern "C" int fsibe_get_box(fsibe_sim *s, int which, double *out, int box[4]) {
  if (!s || !box) return set_err(FSIBE_EARG, "null argument");
  const Box &b = which < 3 ? s->fbox : s->mbox;
  box[0] = b.x0; box[1] = b.x1; box[2] = b.y0; box[3] = b.y1;
  if (!out || b.empty()) return FSIBE_OK;
  const double *src = nullptr;
  switch (which) {
    case 0: src = s->fb_p; break;
    case 1: src = s->fb_sa; break;
    case 2: src = s->fb_sb; break;
    case 3: src = s->mask_m; break;
    case 4: src = s->mask_vx; break;
    case 5: src = s->mask_vy; break;
    default: return set_err(FSIBE_EARG, "unknown box field %d", which);
  }
  if (which < 3 && !s->press_box_valid) return set_err(FSIBE_ESTATE, "no pressure box of the current step");
  HIPCHK(hipMemcpyAsync(out, src, sizeof(double) * (size_t)b.w() * b.h(), hipMemcpyDeviceToHost, s->stream));
  HIPCHK(hipStreamSynchronize(s->stream));
  return FSIBE_OK;
}

extern "C" int fsibe_profile_enable(fsibe_sim *s, int classes) {
  if (!s) return set_err(FSIBE_EARG, "null sim");
  HIPCHK(hipStreamSynchronize(s->stream));
  for (int k = 0; k < P_NK; ++k) {
    for (int j = 0; j < 2; ++j)
      if (!s->prof.ev[k][j]) HIPCHK(hipEventCreate(&s->prof.ev[k][j]));
    s->prof.ms[k] = 0.0;
    s->prof.cnt[k] = 0;
    s->prof.rec[k] = false;
  }
  s->prof.on = classes != 0;
  s->prof.mask = (unsigned)classes & ((1u << P_NK) - 1u);
  return FSIBE_OK;
}

extern "C" int fsibe_profile_read(fsibe_sim *s, double *total_ms, long long *count, int n) {
  if (!s || !total_ms || !count) return set_err(FSIBE_EARG, "null argument");
  for (int k = 0; k < n && k < P_NK; ++k) {
    total_ms[k] = s->prof.ms[k];
    count[k] = s->prof.cnt[k];
  }
  return P_NK;
}

// ===========================================================================
// Batched simulations (no reference counterpart: the reference runs
// simulations one after another, dns.f90:70-101).  A batch owns ordinary
// simulations grouped by grid size.  Each member takes its startup step on
// its own; every AB2 step after that is one launch per stage and size group,
// with one argument record per member at blockIdx.y (kb_* kernels).  Members
// keep their own time, dt, beam and parameters.  Each size group runs its
// own chain of steps on its own stream (batch_run_groups).
// ===========================================================================
// A few host threads for the per-member host work of a batch step (beam
// geometry, reading results): for(i = 0 .. n-1) fn(i), spread over the pool
// and the calling thread.  Each member's host state is touched by one thread.
class HostPool {
 public:
  explicit HostPool(int nthreads) {
    for (int t = 0; t < nthreads; ++t) workers_.emplace_back([this] { loop(); });
  }
  ~HostPool() {
    {
      std::lock_guard<std::mutex> g(mu_);
      stop_ = true;
    }
    cv_.notify_all();
    for (auto &w : workers_) w.join();
  }
  void run(int n, const std::function<void(int)> &fn) {
    if (workers_.empty() || n <= 1) {
      for (int i = 0; i < n; ++i) fn(i);
      return;
    }
    {
      std::lock_guard<std::mutex> g(mu_);
      fn_ = &fn;
      n_ = n;
      next_.store(0);
      active_ = (int)workers_.size();
      ++gen_;
    }
    cv_.notify_all();
    work();
    std::unique_lock<std::mutex> g(mu_);
    done_cv_.wait(g, [this] { return active_ == 0; });
    fn_ = nullptr;
  }

 private:
  void work() {
    for (int i = next_.fetch_add(1); i < n_; i = next_.fetch_add(1)) (*fn_)(i);
  }
  void loop() {
    unsigned long long seen = 0;
    for (;;) {
      {
        std::unique_lock<std::mutex> g(mu_);
        cv_.wait(g, [&] { return stop_ || gen_ != seen; });
        if (stop_) return;
        seen = gen_;
      }
      work();
      std::lock_guard<std::mutex> g(mu_);
      if (--active_ == 0) done_cv_.notify_one();
    }
  }
  std::vector<std::thread> workers_;
  std::mutex mu_;
  std::condition_variable cv_, done_cv_;
  const std::function<void(int)> *fn_ = nullptr;
  std::atomic<int> next_{0};
  int n_ = 0, active_ = 0;
  unsigned long long gen_ = 0;
  bool stop_ = false;
};

enum BatchStage { B_MASK, B_K1, B_K2, B_K4, B_K5, B_K6, B_K7, B_K8, B_K10, B_NST };

static const size_t kBatchArgSize[B_NST] = {sizeof(MaskArgs),      sizeof(ColsInvArgs),   sizeof(RowsNlArgs),
                                            sizeof(ColsAb2Args),   sizeof(ColsInvArgs),
                                            std::max(sizeof(RowsPressArgs), sizeof(RowStepRec)),
                                            sizeof(ColsPressArgs), sizeof(RowsBoxArgs),   sizeof(ForcesArgs)};

struct BatchGroup {
  int nx, ny, H, nf5;
  bool pres;
  // some member has penalisation: K4's tiles hold two fields (Rc, Rpx);
  // without, one (members without penalisation pass no Rpx)
  bool px = false;
  std::vector<int> mem;
  hipStream_t stream = nullptr;  // each group runs its stages on its own stream
  hipEvent_t ev_dt = nullptr;    // after the group's nonlinear-term stage
  size_t off[B_NST];  // argument arrays in the batch's argument buffer
  int tx[B_NST];      // columns per tile of the column stages
  ColSel sel[B_NST];  // launch choice of the column stages
  float tune_us[B_NST], base_us[B_NST];  // measured time of the choice and of the static one (0: not tuned)
  int ncand[B_NST];   // choices measured
  int cap[B_NST];     // grid.x of the stage in the captured step (0: stage left out)
  // the group's stages as two captured graphs (up to the nonlinear term, and
  // the rest), replayed on the group's stream
  hipGraph_t graph[2] = {nullptr, nullptr};
  hipGraphExec_t gexec[2] = {nullptr, nullptr};
};

struct fsibe_batch {
  std::vector<fsibe_sim *> m;
  std::vector<BatchGroup> groups;
  char *h_args = nullptr, *d_args = nullptr, *m_args = nullptr;  // m_args: device address of h_args
  size_t args_bytes = 0;
  bool fsi = false;  // some member's beam is solved (iFLUSI=1): every step waits for its loads
  HostPool *pool = nullptr;
  // each group's stages replayed from captured graphs while every stage
  // fits the captured grids
  bool use_graph = true;
  int captures = 0, replays = 0;
  bool tuned = false;
};

static void drop_graphs(fsibe_batch *b) {
  for (auto &g : b->groups)
    for (int i = 0; i < 2; ++i) {
      if (g.gexec[i]) (void)hipGraphExecDestroy(g.gexec[i]);
      if (g.graph[i]) (void)hipGraphDestroy(g.graph[i]);
      g.gexec[i] = nullptr;
      g.graph[i] = nullptr;
    }
}

extern "C" int fsibe_batch_destroy(fsibe_batch *b) {
  if (!b) return FSIBE_OK;
  for (auto &g : b->groups) {
    if (g.stream) (void)hipStreamSynchronize(g.stream);
    if (g.stream) (void)hipStreamDestroy(g.stream);
    if (g.ev_dt) (void)hipEventDestroy(g.ev_dt);
  }
  drop_graphs(b);
  for (fsibe_sim *s : b->m) fsibe_sim_destroy(s);
  if (b->h_args) (void)hipHostFree(b->h_args);
  if (b->d_args) (void)hipFree(b->d_args);
  delete b->pool;
  delete b;
  return FSIBE_OK;
}

// the single path's launch choice of a column stage holding `bm` fields per
// tile, of a kernel over `split` fields
static ColSel static_sel(const fsibe_sim *s, int bm, int split) {
  // the first column stage (two fields of one spectrum) of 1024-point
  // columns: 4 columns per tile as the static choice (its LDS accesses see
  // 64 bank-conflict cycles per wave against 192 with 2); the two are
  // within a few percent in time and the tuner keeps whichever it measures
  // 2% faster
  if (bm == 1 && split == 2 && s->ny == 1024) {
    const ColSel c4{1, 4};
    if (col_sel_valid(s->ny, s->H, bm, c4)) return c4;
  }
  const ColSel c{1, ct_tx(s->ny)};
  if (col_sel_valid(s->ny, s->H, bm, c)) return c;
  return ColSel{0, pick_tx(s->H, s->ny, bm, split)};
}

static const int kColStages[4] = {B_K1, B_K4, B_K5, B_K7};

// Argument records of column stage k for every member of g with tile width
// tx, for the autotuner: the inputs are the members' own fields (read
// only), and every output goes to the tuner's scratch, four fields of
// H ny per member from scr, so timing a stage leaves every simulation as it
// was (the temporaries T also hold the last step's pressure inputs).
static size_t tune_records(const fsibe_batch *b, const BatchGroup &g, int k, int tx, double2 *scr, char *h,
                           int *nblk_max) {
  const int nm = (int)g.mem.size();
  *nblk_max = 0;
  for (int j = 0; j < nm; ++j) {
    const fsibe_sim *s = b->m[g.mem[j]];
    const size_t NH = (size_t)s->H * s->ny;
    double2 *o = scr + (size_t)j * 4 * NH;
    int nb = 0;
    if (k == B_K1 || k == B_K5) {
      ColsInvArgs &a = reinterpret_cast<ColsInvArgs *>(h)[j];
      a = ColsInvArgs{};
      const int nf = k == B_K1 ? 2 : g.nf5;
      a.W = s->W[k == B_K1 ? s->n0 : s->n1];
      for (int q = 0; q < 4; ++q) {
        a.o[q] = q < nf ? o + q * NH : nullptr;
        a.fsel[q] = k == B_K1 ? (q == 1 ? 4 : 0) : (q < nf ? q : 0);
      }
      a.nfield = nf;
      a.r0_3 = 0; a.r1_3 = s->ny - 1;
      a.nblk = nb = (s->H / tx) * nf;
      a.c = s->sc;
    } else if (k == B_K4) {
      ColsAb2Args &a = reinterpret_cast<ColsAb2Args *>(h)[j];
      a = ColsAb2Args{};
      a.Rc = s->T[2]; a.Rpx = s->penal_on ? s->T[3] : nullptr; a.W0 = s->W[s->n0]; a.NL1 = s->NL[s->n1];
      a.NL0 = o; a.W1 = o + NH;
      a.s = s->dscal; a.explicit_step = 0; a.nblk = nb = s->H / tx; a.c = s->sc;
      a.py0 = 0; a.py1 = s->ny - 1;
    } else {
      ColsPressArgs &a = reinterpret_cast<ColsPressArgs *>(h)[j];
      a = ColsPressArgs{};
      a.Rq = s->T[4]; a.Rqy = s->T[5]; a.Cq = o; a.r0 = 0; a.r1 = s->ny - 1;
      a.nblk = nb = s->H / tx; a.c = s->sc;
    }
    *nblk_max = std::max(*nblk_max, nb);
  }
  const size_t rec = (k == B_K1 || k == B_K5) ? sizeof(ColsInvArgs) : k == B_K4 ? sizeof(ColsAb2Args) : sizeof(ColsPressArgs);
  return rec * nm;
}

// one launch of column stage k of group g with launch choice c over the
// records at d (reps times)
static int tune_launch(const fsibe_batch *b, const BatchGroup &g, int k, ColSel c, const char *d, int gx, int reps) {
  const fsibe_sim *s0 = b->m[g.mem[0]];
  const int nm = (int)g.mem.size();
  if (k == B_K1 || k == B_K5)
    return with_cols_sel<1>(s0->py, s0->H, c, [&](auto F, int nt, int TX) -> int {
      const size_t lds = sizeof(double2) * TX * padlen(s0->ny);
      CHK(prep_lds(kb_cols_inv_fields<decltype(F)>, lds));
      for (int r = 0; r < reps; ++r)
        kb_cols_inv_fields<decltype(F)><<<dim3(gx, nm), nt, lds, g.stream>>>(reinterpret_cast<const ColsInvArgs *>(d), F, s0->twy);
      HIPCHK(hipGetLastError());
      return FSIBE_OK;
    });
  if (k == B_K4)
    return with_cols_sel<2>(s0->py, s0->H, c, [&](auto F, int nt, int TX) -> int {
      const size_t lds = k4_lds(s0->ny, g.px, TX);
      CHK(prep_lds(kb_cols_ab2<decltype(F)>, lds));
      for (int r = 0; r < reps; ++r)
        kb_cols_ab2<decltype(F)><<<dim3(gx, nm), nt, lds, g.stream>>>(reinterpret_cast<const ColsAb2Args *>(d), F, s0->twy);
      HIPCHK(hipGetLastError());
      return FSIBE_OK;
    });
  return with_cols_sel<2>(s0->py, s0->H, c, [&](auto F, int nt, int TX) -> int {
    const size_t lds = sizeof(double2) * 2 * TX * padlen(s0->ny);
    CHK(prep_lds(kb_cols_press<decltype(F)>, lds));
    for (int r = 0; r < reps; ++r)
      kb_cols_press<decltype(F)><<<dim3(gx, nm), nt, lds, g.stream>>>(reinterpret_cast<const ColsPressArgs *>(d), F, s0->twy);
    HIPCHK(hipGetLastError());
    return FSIBE_OK;
  });
}

// Autotuner of a batch's column stages (the FFT passes along y, fused with
// their spectral operators).  For each size group and stage, every valid
// launch choice (compile-time or runtime plan, 1 .. 16 columns per tile) is
// timed on the group's own members with HIP events, two rounds of 4
// launches each after a warm-up launch, and the fastest is kept; the single
// path's choice stays unless another is more than 2 % faster.  No choice
// changes a result (ColSel), so the members stay bit-identical to their own
// runs whatever the measurements say.  Stages whose bit is set in `skip` keep
// their static choice untimed.
static int tune_batch(fsibe_batch *b, unsigned skip = 0) {
  for (fsibe_sim *s : b->m) HIPCHK(hipStreamSynchronize(s->stream));
  size_t bytes = 0;
  for (auto &g : b->groups)
    bytes = std::max(bytes, g.mem.size() * std::max(sizeof(ColsInvArgs), std::max(sizeof(ColsAb2Args), sizeof(ColsPressArgs))));
  std::vector<char> h(bytes);
  char *d = nullptr;
  hipEvent_t e0 = nullptr, e1 = nullptr;
  int rc = FSIBE_OK;
  if (hipMalloc(&d, bytes) != hipSuccess || hipEventCreate(&e0) != hipSuccess || hipEventCreate(&e1) != hipSuccess)
    rc = set_err(FSIBE_EHIP, "batch autotuner: allocation failed");
  for (size_t gi = 0; rc == FSIBE_OK && gi < b->groups.size(); ++gi) {
    BatchGroup &g = b->groups[gi];
    const fsibe_sim *s0 = b->m[g.mem[0]];
    double2 *scr = nullptr;  // the stages' outputs while they are timed
    if (hipMalloc(&scr, sizeof(double2) * 4 * (size_t)s0->H * s0->ny * g.mem.size()) != hipSuccess) {
      rc = set_err(FSIBE_EHIP, "batch autotuner: allocation failed");
      break;
    }
    for (int k : kColStages) {
      if (skip >> k & 1u) continue;
      const int bm = (k == B_K4 || k == B_K7) ? 2 : 1;
      std::vector<ColSel> cand;
      for (int ct = 1; ct >= 0; --ct)
        for (int tx = 1; tx <= 16; tx *= 2) {
          const ColSel c{ct, tx};
          if (k == B_K4 ? k4_sel_valid(s0->ny, s0->H, g.px, c) : col_sel_valid(s0->ny, s0->H, bm, c)) cand.push_back(c);
        }
      std::vector<float> best(cand.size(), 1e30f);
      for (int round = 0; rc == FSIBE_OK && round < 2; ++round)
        for (size_t ci = 0; rc == FSIBE_OK && ci < cand.size(); ++ci) {
          int gx = 0;
          const size_t nb = tune_records(b, g, k, cand[ci].tx, scr, h.data(), &gx);
          if (hipStreamSynchronize(g.stream) != hipSuccess || hipMemcpy(d, h.data(), nb, hipMemcpyHostToDevice) != hipSuccess) {
            rc = set_err(FSIBE_EHIP, "batch autotuner: upload failed");
            break;
          }
          rc = tune_launch(b, g, k, cand[ci], d, gx, 1);
          if (rc != FSIBE_OK) break;
          const int reps = 4;
          float ms = 0.0f;
          if (hipEventRecord(e0, g.stream) != hipSuccess) { rc = set_err(FSIBE_EHIP, "batch autotuner: event"); break; }
          rc = tune_launch(b, g, k, cand[ci], d, gx, reps);
          if (rc != FSIBE_OK) break;
          if (hipEventRecord(e1, g.stream) != hipSuccess || hipEventSynchronize(e1) != hipSuccess ||
              hipEventElapsedTime(&ms, e0, e1) != hipSuccess) {
            rc = set_err(FSIBE_EHIP, "batch autotuner: timing failed");
            break;
          }
          best[ci] = std::min(best[ci], 1000.0f * ms / reps);
        }
      if (rc != FSIBE_OK) break;
      size_t bi = 0, si = 0;
      for (size_t ci = 0; ci < cand.size(); ++ci) {
        if (best[ci] < best[bi]) bi = ci;
        if (cand[ci].ct == g.sel[k].ct && cand[ci].tx == g.sel[k].tx) si = ci;
      }
      if (!(best[bi] < 0.98f * best[si])) bi = si;
      g.sel[k] = cand[bi];
      g.tx[k] = cand[bi].tx;
      g.tune_us[k] = best[bi];
      g.base_us[k] = best[si];
      g.ncand[k] = (int)cand.size();
    }
    (void)hipStreamSynchronize(g.stream);
    (void)hipFree(scr);
  }
  if (d) (void)hipFree(d);
  if (e0) (void)hipEventDestroy(e0);
  if (e1) (void)hipEventDestroy(e1);
  if (rc == FSIBE_OK) b->tuned = true;
  return rc;
}

// The single path's column stages take the autotuner's choices too:
// measured once per process and grid (nx, ny, fields of K5) on a batch of
// that one simulation at its first fsibe_run, and kept for every
// simulation of that grid.
static std::mutex g_csel_mu;
static std::map<std::array<int, 4>, std::array<ColSel, 4>> g_csel;

static int sim_tune_cols(fsibe_sim *s) {
  if (s->csel_ready) return FSIBE_OK;
  if (env_int("FSIBE_AUTOTUNE", 1) == 0) return FSIBE_OK;  // the static choices (reproducible profiles)
  const int nf5 = (s->forces_on && s->visc) ? 4 : 3;
  const std::array<int, 4> key{s->nx, s->ny, nf5, s->penal_on ? 1 : 0};
  std::lock_guard<std::mutex> lock(g_csel_mu);
  auto it = g_csel.find(key);
  if (it == g_csel.end()) {
    fsibe_batch t;  // borrows the simulation; releases nothing of it
    t.m.push_back(s);
    BatchGroup g;
    g.nx = s->nx; g.ny = s->ny; g.H = s->H; g.nf5 = nf5; g.pres = s->pressure_on; g.px = s->penal_on;
    g.mem.push_back(0);
    g.stream = s->stream;
    g.sel[B_K1] = static_sel(s, 1, 2);
    g.sel[B_K4] = static_sel(s, 2, 1);
    g.sel[B_K5] = static_sel(s, 1, nf5);
    g.sel[B_K7] = static_sel(s, 2, 1);
    t.groups.push_back(g);
    // only what this grid launches: K4, K5 and K7 are not where the fused
    // column stage and the pressure stage replace them
    unsigned skip = 0;
    if (with_col_step(s->ny, s->H, s->penal_on, false, [](auto) {})) skip |= 1u << B_K4 | 1u << B_K5;
    if (with_press_step(s->ny, s->H, [](auto) {})) skip |= 1u << B_K7;
    const int rc = tune_batch(&t, skip);
    const std::array<ColSel, 4> sel{t.groups[0].sel[B_K1], t.groups[0].sel[B_K4], t.groups[0].sel[B_K5],
                                    t.groups[0].sel[B_K7]};
    t.groups[0].stream = nullptr;
    t.m.clear();
    t.groups.clear();
    if (rc != FSIBE_OK) return rc;
    it = g_csel.emplace(key, sel).first;
  }
  for (int q = 0; q < 4; ++q) s->csel[q] = it->second[q];
  s->csel_ready = true;
  return FSIBE_OK;
}

extern "C" int fsibe_batch_create(const fsibe_params *params, int n, const double *const *vortk,
                                  fsibe_batch **out) {
  if (!params || !out || n < 1) return set_err(FSIBE_EARG, "batch: bad argument");
  *out = nullptr;
  for (int i = 0; i < n; ++i) {
    const fsibe_params &p = params[i];
    if (p.iSponge == 10 || p.iSponge == 4 || p.iSponge == 22 || p.iMeanVelocity == 11)
      return set_err(FSIBE_EUNSUPPORTED, "batch member %d: iSponge=%d / iMeanVelocity=%d is not batched", i,
                     p.iSponge, p.iMeanVelocity);
  }
  fsibe_batch *b = new fsibe_batch();
  auto fail = [&](int rc) { fsibe_batch_destroy(b); return rc; };
  for (int i = 0; i < n; ++i) {
    fsibe_sim *s = nullptr;
    int rc = fsibe_sim_create(&params[i], &s);
    if (rc != FSIBE_OK) return fail(rc);
    b->m.push_back(s);
    if (vortk && vortk[i]) {
      rc = fsibe_set_vortk(s, vortk[i]);
      if (rc != FSIBE_OK) return fail(rc);
    }
    if (s->p.iFLUSI == 1 && s->p.iBeam > 0) {
      rc = ensure_solid(s);
      if (rc != FSIBE_OK) return fail(rc);
      b->fsi = true;
    }
  }
  // groups: same grid and the same launch shapes
  for (int i = 0; i < n; ++i) {
    const fsibe_sim *s = b->m[i];
    const int nf5 = (s->forces_on && s->visc) ? 4 : 3;
    BatchGroup *g = nullptr;
    for (auto &q : b->groups)
      if (q.nx == s->nx && q.ny == s->ny && q.nf5 == nf5 && q.pres == s->pressure_on) g = &q;
    if (!g) {
      b->groups.push_back(BatchGroup{});
      g = &b->groups.back();
      g->nx = s->nx; g->ny = s->ny; g->H = s->H; g->nf5 = nf5; g->pres = s->pressure_on;
    }
    g->px = g->px || s->penal_on;
    g->mem.push_back(i);
  }
  size_t off = 0;
  for (auto &g : b->groups)
    for (int k = 0; k < B_NST; ++k) {
      g.off[k] = off;
      off += (kBatchArgSize[k] * g.mem.size() + 255) & ~(size_t)255;
    }
  b->args_bytes = off;
  for (auto &g : b->groups)
    if (hipStreamCreate(&g.stream) != hipSuccess || hipEventCreateWithFlags(&g.ev_dt, hipEventDisableTiming) != hipSuccess)
      return fail(set_err(FSIBE_EHIP, "batch: stream creation failed"));
  if (hipHostMalloc((void **)&b->h_args, off, hipHostMallocMapped | hipHostMallocCoherent) != hipSuccess ||
      hipHostGetDevicePointer((void **)&b->m_args, b->h_args, 0) != hipSuccess ||
      hipMalloc(&b->d_args, off) != hipSuccess)
    return fail(set_err(FSIBE_EHIP, "batch: allocation failed"));
  memset(b->h_args, 0, off);
  {
    // host threads: FSIBE_HOST_THREADS, else up to 15 helpers beside the caller
    const int hw = (int)std::thread::hardware_concurrency();
    int nt = env_int("FSIBE_HOST_THREADS", std::min(16, std::max(1, hw))) - 1;
    nt = std::max(0, std::min(nt, n - 1));
    b->pool = new HostPool(nt);
  }
  // launch choices of the column stages: the single path's, then the
  // autotuner's measurements
  for (auto &g : b->groups) {
    const fsibe_sim *s = b->m[g.mem[0]];
    g.sel[B_K1] = static_sel(s, 1, 2);
    g.sel[B_K4] = static_sel(s, 2, 1);
    g.sel[B_K5] = static_sel(s, 1, g.nf5);
    g.sel[B_K7] = static_sel(s, 2, 1);
    for (int k = 0; k < B_NST; ++k) {
      g.tx[k] = g.sel[k].tx;
      g.tune_us[k] = g.base_us[k] = 0.0f;
      g.ncand[k] = 0;
      g.cap[k] = 0;
    }
  }
  if (env_int("FSIBE_AUTOTUNE", 1) != 0) {
    const int rc = tune_batch(b);
    if (rc != FSIBE_OK) return fail(rc);
  }
  *out = b;
  return FSIBE_OK;
}

// the host part of fsibe_create_mask: beam state and geometry for `time`
static int stage_geometry(fsibe_sim *s, double time) {
  const fsibe_params &p = s->p;
  const bool moving = (p.iSponge >= 4 && s->time < p.T_fullspeed) || p.iFLUSI == 1 || p.iMotion > 0;
  if (p.iBeam > 0 && moving) {
    motion_all(s, time, s->alpha, &s->LE[0][0]);
    s->time_mask = time;
  }
  return build_geometry(s, time);
}

static void fill_batch_args(fsibe_batch *b, BatchGroup &g, int j, fsibe_sim *s, int maxblk[B_NST]) {
  char *A = b->h_args;
  const int n0 = s->n0, n1 = s->n1;
  const MaskBox mb = mask_box(s);
  {  // create_mask
    MaskArgs &a = reinterpret_cast<MaskArgs *>(A + g.off[B_MASK])[j];
    a.prims = reinterpret_cast<const Prim *>(s->d_stage + s->off_prim);
    a.np = s->nprim;
    a.wallrow = s->wallrow;
    a.om = s->mask_m; a.ovx = s->mask_vx; a.ovy = s->mask_vy;
    MaskConsts &mc = a.c;
    mc.dx = s->dx; mc.dy = s->dy; mc.t = s->p.t_beam; mc.h = s->p.N_smooth * std::max(s->dx, s->dy);
    mc.gerf = s->gerf; mc.inv_eps_unused = 0.0; mc.ds = s->ds; mc.pi = s->pi; mc.sharp = s->sharp;
    mc.eps = s->p.eps;
    a.bx0 = s->mbox.x0; a.by0 = s->mbox.y0; a.bw = s->mbox.w(); a.bh = s->mbox.h();
    a.tiles_x = (a.bw + kMaskTile - 1) / kMaskTile;
    a.tiles = s->mbox.empty() ? 0 : a.tiles_x * ((a.bh + kMaskTile - 1) / kMaskTile);
    a.bg = beam_geo(s, kMaskThreadsBatch);
    if (s->mbox.empty()) a.bg.fwg = 0;
    maxblk[B_MASK] = std::max(maxblk[B_MASK], a.tiles + a.bg.fwg);
  }
  {  // K1: A = Fy^-1[W0], B = Fy^-1[i ky W0]
    ColsInvArgs &a = reinterpret_cast<ColsInvArgs *>(A + g.off[B_K1])[j];
    a.W = s->W[n0]; a.o[0] = s->T[0]; a.o[1] = s->T[1]; a.o[2] = nullptr; a.o[3] = nullptr;
    a.fsel[0] = 0; a.fsel[1] = 4; a.fsel[2] = 0; a.fsel[3] = 0; a.nfield = 2;
    a.r0_3 = 0; a.r1_3 = s->ny - 1;
    a.nblk = (s->H / g.tx[B_K1]) * 2;
    a.c = s->sc;
    maxblk[B_K1] = std::max(maxblk[B_K1], a.nblk);
  }
  {  // K2 + K3
    RowsNlArgs &a = reinterpret_cast<RowsNlArgs *>(A + g.off[B_K2])[j];
    a.A = s->T[0]; a.B = s->T[1]; a.u1 = s->u1; a.u2 = s->u2; a.ms = s->sponge_on ? s->ms : nullptr;
    a.mb = mb; a.penal_on = s->penal_on; a.nparts = s->ny; a.explicit_step = 0; a.nblk = s->ny;
    a.Rc = s->T[2]; a.Rpx = s->T[3]; a.c = s->sc; a.c.kc = s->H; a.umax_part = s->umax_part; a.sc = s->dscal; a.fl = s->fp;
    a.time = s->time; a.dt0 = s->dt0; a.res = res_dev(s, s->slot);
    a.rpx_zero = s->p.iSponge == 10 ? 1 : 0;
    maxblk[B_K2] = std::max(maxblk[B_K2], a.nblk);
  }
  {  // K4
    ColsAb2Args &a = reinterpret_cast<ColsAb2Args *>(A + g.off[B_K4])[j];
    a.Rc = s->T[2]; a.Rpx = s->penal_on ? s->T[3] : nullptr; a.W0 = s->W[n0]; a.NL1 = s->NL[n1]; a.NL0 = s->NL[n0];
    a.W1 = s->W[n1];
    a.s = s->dscal; a.explicit_step = 0; a.nblk = s->H / g.tx[B_K4]; a.c = s->sc;
    rpx_rows(s, mb, a.py0, a.py1);
    maxblk[B_K4] = std::max(maxblk[B_K4], a.nblk);
  }
  {  // K5
    ColsInvArgs &a = reinterpret_cast<ColsInvArgs *>(A + g.off[B_K5])[j];
    a.W = s->W[n1];
    for (int k = 0; k < 4; ++k) { a.o[k] = k < g.nf5 ? s->T[k] : nullptr; a.fsel[k] = k < g.nf5 ? k : 0; }
    a.nfield = g.nf5; a.nblk = (s->H / g.tx[B_K5]) * g.nf5; a.c = s->sc;
    stress_rows(s, a.r0_3, a.r1_3);
    maxblk[B_K5] = std::max(maxblk[B_K5], a.nblk);
  }
  // K6: the record of the row stage the single path launches
  const bool rs = with_row_step<false>(s->H, s->ny, g.pres, [&](auto S) {
    RowStepRec &r = reinterpret_cast<RowStepRec *>(A + g.off[B_K6])[j];
    r.a = row_step_args(s, mb);
    r.nblk = s->ny / decltype(S)::RPB;
    r.pad = 0;
    maxblk[B_K6] = std::max(maxblk[B_K6], r.nblk);
  });
  if (!rs) {
    RowsPressArgs &a = reinterpret_cast<RowsPressArgs *>(A + g.off[B_K6])[j];
    a.Cw = s->T[0]; a.Cpsi = s->T[1]; a.Cpsiy = s->T[2]; a.u1 = s->u1; a.u2 = s->u2; a.vor_mean = s->vor_mean;
    a.sums = rows_dev(s, s->slot); a.umax_part = s->umax_part; a.mb = mb; a.win = s->win[0];
    a.win2 = s->win[1];
    a.Rq = s->T[4]; a.Rqy = s->T[5]; a.s = s->dscal; a.UMx0 = 0.0; a.UMy0 = 0.0; a.mode = 1;
    a.pres = s->pressure_on; a.nblk = s->ny; a.c = s->sc;
    maxblk[B_K6] = std::max(maxblk[B_K6], a.nblk);
  }
  s->slot_fluid[s->slot] = true;
  const bool fz = s->forces_on && s->forces_ready && !s->fbox.empty();
  const Box &fb = s->fbox;
  {  // K7
    ColsPressArgs &a = reinterpret_cast<ColsPressArgs *>(A + g.off[B_K7])[j];
    a.Rq = s->T[4]; a.Rqy = s->T[5]; a.Cq = s->T[6]; a.r0 = fb.y0; a.r1 = fb.y1;
    a.nblk = fz ? s->H / g.tx[B_K7] : 0; a.c = s->sc;
    maxblk[B_K7] = std::max(maxblk[B_K7], a.nblk);
  }
  {  // K8
    RowsBoxArgs &a = reinterpret_cast<RowsBoxArgs *>(A + g.off[B_K8])[j];
    a.Cq = s->T[6]; a.Cpsi = s->T[1]; a.Cpsiy = s->T[2]; a.Cpsiyy = s->T[3]; a.u1 = s->u1; a.u2 = s->u2;
    a.press = s->fb_p; a.sa = s->fb_sa; a.sb = s->fb_sb; a.r0 = fb.y0; a.bx0 = fb.x0; a.bx1 = fb.x1;
    a.bw = fb.w(); a.visc = s->visc; a.nblk = fz ? fb.h() : 0; a.c = s->sc;
    maxblk[B_K8] = std::max(maxblk[B_K8], a.nblk);
  }
  s->press_box_valid = fz;
  {  // K10
    ForcesArgs &a = reinterpret_cast<ForcesArgs *>(A + g.off[B_K10])[j];
    const bool ok = fz && s->ntg > 0 && s->ntg == s->nb * (6 * s->fg.ns + 6 * s->fg.nc);
    a.tg = reinterpret_cast<const double *>(s->d_stage + s->off_tg);
    a.nd = reinterpret_cast<const double *>(s->d_stage + s->off_nd);
    a.cd = reinterpret_cast<const double *>(s->d_stage + s->off_cd);
    a.press = s->fb_p; a.sa = s->fb_sa; a.sb = s->fb_sb;
    a.val = reinterpret_cast<double *>(s->d_stage + s->off_val);
    a.pbeam = pbeam_dev(s, s->slot); a.tbeam = pbeam_dev(s, s->slot) + nodes_all(s);
    a.part = parts_dev(s, s->slot); a.g = s->fg;
    a.nblk = ok ? s->nb * (s->fg.ns + s->fg.nc) : 0;
    maxblk[B_K10] = std::max(maxblk[B_K10], a.nblk);
    s->slot_forces[s->slot] = ok;
    s->slot_units[s->slot] = a.nblk;
  }
}

// how batch_stages launches: eager (set the LDS limit, then launch), only
// set the LDS limits (before a capture), or only launch (under capture)
enum StageLaunch { SL_EAGER, SL_PREP, SL_CAPTURE };

#define SLAUNCH(KT, gx, gy, nt, lds, st, mode, ...)                \
  do {                                                              \
    if ((gx) > 0) {                                                 \
      if ((mode) != SL_CAPTURE) CHK(prep_lds(KT, lds));             \
      if ((mode) != SL_PREP) {                                      \
        KT<<<dim3((gx), (gy)), nt, lds, st>>>(__VA_ARGS__);         \
        HIPCHK(hipGetLastError());                                  \
      }                                                             \
    }                                                               \
  } while (0)

// stages [k0, k1) of every group, stage by stage, each group on its own
// stream, with grid.x = grids[group][stage] (0: the stage is skipped)
static int batch_stages(fsibe_batch *b, const std::vector<std::array<int, B_NST>> &grids, int k0, int k1,
                        StageLaunch mode, int only = -1) {
  auto arr = [&](const BatchGroup &g, int k) { return b->d_args + g.off[k]; };
  for (int k = k0; k < k1; ++k)
    for (size_t gi = 0; gi < b->groups.size(); ++gi) {
      if (only >= 0 && (int)gi != only) continue;
      const BatchGroup &g = b->groups[gi];
      const fsibe_sim *s0 = b->m[g.mem[0]];
      const int nm = (int)g.mem.size();
      const int gx = grids[gi][k];
      if (gx <= 0) continue;
      switch (k) {
        case B_MASK:
          SLAUNCH(kb_mask, gx, nm, kMaskThreadsBatch, 0, g.stream, mode,
                  reinterpret_cast<const MaskArgs *>(arr(g, B_MASK)));
          break;
        case B_K1:
        case B_K5:
          CHK(with_cols_sel<1>(s0->py, s0->H, g.sel[k], [&](auto F, int nt, int TX) -> int {
            SLAUNCH(kb_cols_inv_fields<decltype(F)>, gx, nm, nt, sizeof(double2) * TX * padlen(s0->ny), g.stream, mode,
                    reinterpret_cast<const ColsInvArgs *>(arr(g, k)), F, s0->twy);
            return FSIBE_OK;
          }));
          break;
        case B_K2:
          CHK(with_rows<3>(s0->px, [&](auto F, int nt) -> int {
            SLAUNCH(kb_rows_nl<decltype(F)>, gx, nm, nt, sizeof(double2) * 3 * padlen(s0->H), g.stream, mode,
                    reinterpret_cast<const RowsNlArgs *>(arr(g, B_K2)), F, s0->twx);
            return FSIBE_OK;
          }));
          break;
        case B_K4:
          CHK(with_cols_sel<2>(s0->py, s0->H, g.sel[B_K4], [&](auto F, int nt, int TX) -> int {
            SLAUNCH(kb_cols_ab2<decltype(F)>, gx, nm, nt, k4_lds(s0->ny, g.px, TX), g.stream, mode,
                    reinterpret_cast<const ColsAb2Args *>(arr(g, B_K4)), F, s0->twy);
            return FSIBE_OK;
          }));
          break;
        case B_K6: {
          int rc = FSIBE_OK;
          const bool rs = with_row_step<false>(s0->H, s0->ny, g.pres, [&](auto S) {
            using ST = decltype(S);
            auto *kern = g.pres ? &kb_row_step<ST, true> : &kb_row_step<ST, false>;
            rc = [&]() -> int {
              SLAUNCH(kern, gx, nm, ST::THREADS, ST::LDS, g.stream, mode,
                      reinterpret_cast<const RowStepRec *>(arr(g, B_K6)), s0->twx);
              return FSIBE_OK;
            }();
          });
          CHK(rc);
          if (rs) break;
          CHK(with_rows<3>(s0->px, [&](auto F, int nt) -> int {
            if constexpr (!always_row_step(fixed_len<decltype(F)>::v))
              SLAUNCH(kb_rows_press<decltype(F)>, gx, nm, nt, sizeof(double2) * 3 * padlen(s0->H), g.stream, mode,
                      reinterpret_cast<const RowsPressArgs *>(arr(g, B_K6)), F, s0->twx);
            return FSIBE_OK;
          }));
          break;
        }
        case B_K7:
          CHK(with_cols_sel<2>(s0->py, s0->H, g.sel[B_K7], [&](auto F, int nt, int TX) -> int {
            SLAUNCH(kb_cols_press<decltype(F)>, gx, nm, nt, sizeof(double2) * 2 * TX * padlen(s0->ny), g.stream, mode,
                    reinterpret_cast<const ColsPressArgs *>(arr(g, B_K7)), F, s0->twy);
            return FSIBE_OK;
          }));
          break;
        case B_K8:
          CHK(with_rows<3>(s0->px, [&](auto F, int nt) -> int {
            SLAUNCH(kb_rows_box<decltype(F)>, gx, nm, nt, sizeof(double2) * 3 * padlen(s0->H), g.stream, mode,
                    reinterpret_cast<const RowsBoxArgs *>(arr(g, B_K8)), F, s0->twx);
            return FSIBE_OK;
          }));
          break;
        case B_K10:
          SLAUNCH(kb_forces, gx, nm, kForceThreads, 0, g.stream, mode, reinterpret_cast<const ForcesArgs *>(arr(g, B_K10)));
          break;
        default:
          break;
      }
    }
  return FSIBE_OK;
}

// Captures part 0 (mask, K1, K2) or part 1 (K4 .. K10) of one group's
// step into a graph with the grids g.cap.  Every stage reads its argument
// records from fixed device addresses (refreshed by the gather kernel each
// step), so one capture serves every step whose blocks fit the captured
// grids.  Kernel nodes only, in one chain on the group's stream.
static int capture_part(fsibe_batch *b, int gi, int part) {
  BatchGroup &g = b->groups[gi];
  const int k0 = part == 0 ? B_MASK : B_K4, k1 = part == 0 ? B_K4 : B_NST;
  std::vector<std::array<int, B_NST>> caps(b->groups.size());
  for (int k = 0; k < B_NST; ++k) caps[gi][k] = g.cap[k];
  CHK(batch_stages(b, caps, k0, k1, SL_PREP, gi));
  HIPCHK(hipStreamBeginCapture(g.stream, hipStreamCaptureModeRelaxed));
  const int rc = batch_stages(b, caps, k0, k1, SL_CAPTURE, gi);
  hipGraph_t gr = nullptr;
  const hipError_t e = hipStreamEndCapture(g.stream, &gr);
  if (rc != FSIBE_OK || e != hipSuccess) {
    if (gr) (void)hipGraphDestroy(gr);
    return rc != FSIBE_OK ? rc : set_err(FSIBE_EHIP, "hipStreamEndCapture: %s", hipGetErrorString(e));
  }
  hipGraphExec_t ex = nullptr;
  const hipError_t e2 = hipGraphInstantiate(&ex, gr, nullptr, nullptr, 0);
  if (e2 != hipSuccess) {
    (void)hipGraphDestroy(gr);
    return set_err(FSIBE_EHIP, "hipGraphInstantiate: %s", hipGetErrorString(e2));
  }
  if (g.gexec[part]) (void)hipGraphExecDestroy(g.gexec[part]);
  if (g.graph[part]) (void)hipGraphDestroy(g.graph[part]);
  g.graph[part] = gr;
  g.gexec[part] = ex;
  b->captures++;
  return FSIBE_OK;
}

// Launches group gi's stages of a step from its graphs (after the gather).
// A stage whose blocks no longer fit its captured grid (the mask box, the
// force window and the beam's force units grow and shrink as the beam
// moves) is captured again with a quarter more room; blocks beyond a
// member's own count return at once.
static int group_graph_stages(fsibe_batch *b, int gi, const std::array<int, B_NST> &need) {
  BatchGroup &g = b->groups[gi];
  bool fits[2] = {g.gexec[0] != nullptr, g.gexec[1] != nullptr};
  for (int k = 0; k < B_NST; ++k)
    if (need[k] > g.cap[k]) {
      const bool grows = k == B_MASK || k == B_K8 || k == B_K10;
      g.cap[k] = grows ? need[k] + need[k] / 4 : need[k];
      fits[k < B_K4 ? 0 : 1] = false;
    }
  for (int part = 0; part < 2; ++part)
    if (!fits[part]) CHK(capture_part(b, gi, part));
  HIPCHK(hipGraphLaunch(g.gexec[0], g.stream));
  HIPCHK(hipGraphLaunch(g.gexec[1], g.stream));
  HIPCHK(hipEventRecord(g.ev_dt, g.stream));
  return FSIBE_OK;
}

// ---- one chain of steps per size group --------------------------------------
// A member's host work (reading its results, the beam solve of a coupled
// member or the leading edge's motion of a prescribed one, the next
// geometry) sits between two of its steps.  Each size group runs its own
// chain: when a group's step ends, the pool does its members' host work and
// the group's next step is launched while the other groups' steps keep the
// GPU busy.  Members never wait for another group, and each stays
// bit-identical to its own run.

// geometry and argument records of group gi's next step; need = its grids
static int group_prepare(fsibe_batch *b, int gi, std::array<int, B_NST> &need) {
  BatchGroup &g = b->groups[gi];
  for (int i : g.mem)
    if (!(b->m[i]->time < b->m[i]->p.Time_end)) return set_err(FSIBE_ESTATE, "batch: a member reached Time_end");
  std::atomic<int> bad{-1};
  std::vector<std::string> errs(g.mem.size());
  b->pool->run((int)g.mem.size(), [&](int j) {
    fsibe_sim *s = b->m[g.mem[j]];
    s->dt0 = s->dt1;
    if (stage_geometry(s, s->time) != FSIBE_OK) {
      errs[j] = fsibe_last_error();
      bad.store(j);
    }
  });
  if (bad.load() >= 0)
    return set_err(FSIBE_EDOMAIN, "batch member %d: %s", g.mem[bad.load()], errs[bad.load()].c_str());
  int mx[B_NST] = {};
  for (size_t j = 0; j < g.mem.size(); ++j) fill_batch_args(b, g, (int)j, b->m[g.mem[j]], mx);
  for (int k = 0; k < B_NST; ++k) need[k] = mx[k];
  return FSIBE_OK;
}

// group gi's argument records and its members' geometry, copied on its stream
static int group_gather(fsibe_batch *b, int gi) {
  const BatchGroup &g = b->groups[gi];
  const size_t nm = g.mem.size();
  const size_t a0 = g.off[0], a1 = g.off[B_NST - 1] + ((kBatchArgSize[B_NST - 1] * nm + 255) & ~(size_t)255);
  std::vector<StageSeg> segs;
  segs.push_back(StageSeg{reinterpret_cast<const double2 *>(b->m_args + a0), reinterpret_cast<double2 *>(b->d_args + a0),
                          (long long)((a1 - a0) / sizeof(double2))});
  for (int i : g.mem) {
    const fsibe_sim *s = b->m[i];
    segs.push_back(StageSeg{reinterpret_cast<const double2 *>(s->m_stage), reinterpret_cast<double2 *>(s->d_stage),
                            (long long)(s->off_tg / sizeof(double2))});
  }
  for (size_t k0 = 0; k0 < segs.size(); k0 += kMaxStageSegs) {
    StageSegs ss{};
    const int ns = (int)std::min(segs.size() - k0, (size_t)kMaxStageSegs);
    for (int k = 0; k < ns; ++k) ss.s[k] = segs[k0 + k];
    k_stage_gather<<<dim3(8, ns), 256, 0, g.stream>>>(ss);
    HIPCHK(hipGetLastError());
  }
  return FSIBE_OK;
}

// prepare and launch group gi's next step; g.ev_dt marks its end
static int group_start(fsibe_batch *b, int gi) {
  std::array<int, B_NST> need{};
  CHK(group_prepare(b, gi, need));
  CHK(group_gather(b, gi));
  if (b->use_graph) {
    CHK(group_graph_stages(b, gi, need));
  } else {
    std::vector<std::array<int, B_NST>> grids(b->groups.size());
    grids[gi] = need;
    CHK(batch_stages(b, grids, B_MASK, B_NST, SL_EAGER, gi));
    HIPCHK(hipEventRecord(b->groups[gi].ev_dt, b->groups[gi].stream));
  }
  return FSIBE_OK;
}

// after group gi's step: each member reads its results, and its beam is
// solved (or moved); time and levels advance
static int group_finish(fsibe_batch *b, int gi) {
  BatchGroup &g = b->groups[gi];
  std::atomic<int> bad{-1};
  std::vector<std::string> errs(g.mem.size());
  b->pool->run((int)g.mem.size(), [&](int j) {
    fsibe_sim *s = b->m[g.mem[j]];
    s->upload_pending = 0;
    parse_results(s, s->slot);
    s->dt1 = s->last.dt1;
    s->slot ^= 1;
    const fsibe_params &p = s->p;
    if (p.iFLUSI == 1 && p.iBeam > 0) {
      if (solid_step(s) != FSIBE_OK) {
        errs[j] = fsibe_last_error();
        bad.store(j);
      }
    } else if (p.iMotion > 0 && p.iBeam > 0) {
      integrate_all(s, s->time);
    }
    std::swap(s->n0, s->n1);
    s->time = s->time + s->dt1;
    s->it++;
  });
  if (bad.load() >= 0)
    return set_err(FSIBE_EDOMAIN, "batch member %d: %s", g.mem[bad.load()], errs[bad.load()].c_str());
  return FSIBE_OK;
}

// nsteps AB2 steps of every group of a batch.  A member whose
// emergency brake trips stops its group after that step; the other groups
// finish the step they are running and take no further one.
static int batch_run_groups(fsibe_batch *b, int nsteps) {
  const int ng = (int)b->groups.size();
  std::vector<int> left(ng, nsteps);
  std::vector<char> busy(ng, 0);
  int rc = FSIBE_OK;
  bool stop = false;
  for (int gi = 0; gi < ng && rc == FSIBE_OK; ++gi) {
    rc = group_start(b, gi);
    if (rc == FSIBE_OK) busy[gi] = 1;
  }
  const double timeout = wait_timeout_ms();
  for (;;) {
    // the next group whose step has written its dt1, polled with the
    // deadline of wait.hpp (a group that never completes is an error)
    int gi = -1;
    bool any = false;
    for (int k = 0; k < ng; ++k) any = any || busy[k];
    if (!any) break;
    hipError_t herr = hipSuccess;
    std::string msg;
    const int rw = bounded_wait(
        [&] {
          for (int k = 0; k < ng; ++k) {
            if (!busy[k]) continue;
            herr = hipEventQuery(b->groups[k].ev_dt);
            if (herr == hipSuccess) {
              gi = k;
              return Poll::Done;
            }
            if (herr != hipErrorNotReady) return Poll::Failed;
          }
          return Poll::Busy;
        },
        now_ms, [&] { return hipGetErrorString(herr); }, timeout, "a batch step (nonlinear-term kernel)", msg);
    if (rw != FSIBE_OK) return set_err(rw, "batch: %s", msg.c_str());
    busy[gi] = 0;
    --left[gi];
    const int rf = group_finish(b, gi);
    if (rf != FSIBE_OK && rc == FSIBE_OK) rc = rf;
    for (int i : b->groups[gi].mem) stop = stop || b->m[i]->last.status == 1;
    if (rc == FSIBE_OK && !stop && left[gi] > 0) {
      rc = group_start(b, gi);
      if (rc == FSIBE_OK) busy[gi] = 1;
    }
  }
  if (b->use_graph && ng > 0) b->replays += nsteps - left[0];  // steps of the first group
  return rc;
}

extern "C" int fsibe_batch_run(fsibe_batch *b, int nsteps) {
  if (!b) return set_err(FSIBE_EARG, "null batch");
  // the startup (Euler) step of members that have not taken it, on their
  // own; it counts as the first of the nsteps steps
  int done = 0;
  if (nsteps > 0) {
    bool any = false;
    for (fsibe_sim *s : b->m)
      if (!s->startup_done) {
        CHK(fsibe_run(s, 1, nullptr));
        any = true;
      }
    done = any ? 1 : 0;
  }
  for (fsibe_sim *s : b->m) HIPCHK(hipStreamSynchronize(s->stream));
  return nsteps > done ? batch_run_groups(b, nsteps - done) : FSIBE_OK;
}

extern "C" int fsibe_batch_size(fsibe_batch *b) { return b ? (int)b->m.size() : 0; }

extern "C" fsibe_sim *fsibe_batch_member(fsibe_batch *b, int i) {
  if (!b || i < 0 || i >= (int)b->m.size()) return nullptr;
  return b->m[i];
}

// Step mode and autotuning of a batch.  use_graph: 1 replays captured
// graphs, 0 launches every stage eagerly, < 0 keeps the mode.  autotune: 1
// times the column stages' launch choices again and keeps the fastest, 0
// returns to the single path's choices, < 0 keeps them.  Neither changes a
// result.
extern "C" int fsibe_batch_configure(fsibe_batch *b, int use_graph, int autotune) {
  if (!b) return set_err(FSIBE_EARG, "null batch");
  for (auto &g : b->groups) HIPCHK(hipStreamSynchronize(g.stream));
  if (autotune >= 0) {
    drop_graphs(b);
    for (auto &g : b->groups) {
      const fsibe_sim *s = b->m[g.mem[0]];
      g.sel[B_K1] = static_sel(s, 1, 2);
      g.sel[B_K4] = static_sel(s, 2, 1);
      g.sel[B_K5] = static_sel(s, 1, g.nf5);
      g.sel[B_K7] = static_sel(s, 2, 1);
      for (int k = 0; k < B_NST; ++k) {
        g.tx[k] = g.sel[k].tx;
        g.tune_us[k] = g.base_us[k] = 0.0f;
        g.ncand[k] = 0;
        g.cap[k] = 0;
      }
    }
    b->tuned = false;
    if (autotune > 0) CHK(tune_batch(b));
  }
  if (use_graph >= 0) b->use_graph = use_graph != 0;
  return FSIBE_OK;
}

// Pins the launch choice of one column stage of one size group (stage 1,
// 4, 5 or 7 for K1, K4, K5, K7; groups in the order fsibe_batch_describe
// lists them): a compile-time plan (ct = 1) or the runtime plan (ct = 0)
// with tx columns per tile.  For reusing measured choices without
// measuring again; no choice changes a result.
extern "C" int fsibe_batch_set_tiles(fsibe_batch *b, int group, int stage, int ct, int tx) {
  if (!b || group < 0 || group >= (int)b->groups.size()) return set_err(FSIBE_EARG, "bad batch or group");
  const int k = stage == 1 ? B_K1 : stage == 4 ? B_K4 : stage == 5 ? B_K5 : stage == 7 ? B_K7 : -1;
  if (k < 0) return set_err(FSIBE_EARG, "stage must be 1, 4, 5 or 7");
  BatchGroup &g = b->groups[group];
  const int bm = (k == B_K4 || k == B_K7) ? 2 : 1;
  const ColSel c{ct ? 1 : 0, tx};
  if (!(k == B_K4 ? k4_sel_valid(g.ny, g.H, g.px, c) : col_sel_valid(g.ny, g.H, bm, c)))
    return set_err(FSIBE_EARG, "%s plan with %d columns per tile is not a launch choice for %d x %d",
                   c.ct ? "compile-time" : "runtime", tx, g.nx, g.ny);
  for (auto &q : b->groups) HIPCHK(hipStreamSynchronize(q.stream));
  drop_graphs(b);
  for (auto &q : b->groups)
    for (int j = 0; j < B_NST; ++j) q.cap[j] = 0;
  g.sel[k] = c;
  g.tx[k] = tx;
  g.tune_us[k] = g.base_us[k] = 0.0f;
  return FSIBE_OK;
}

// The batch's groups, launch choices and step mode as one JSON object.
extern "C" int fsibe_batch_describe(fsibe_batch *b, char *buf, size_t len) {
  if (!b || !buf || len == 0) return set_err(FSIBE_EARG, "bad argument");
  static const char *kName[B_NST] = {"mask", "K1", "K2", "K4", "K5", "K6", "K7", "K8", "K10"};
  std::string o;
  char t[512];
  snprintf(t, sizeof t, "{\"graph\": %d, \"tuned\": %d, \"captures\": %d, \"graph_steps\": %d, \"groups\": [",
           b->use_graph ? 1 : 0, b->tuned ? 1 : 0, b->captures, b->replays);
  o += t;
  for (size_t gi = 0; gi < b->groups.size(); ++gi) {
    const BatchGroup &g = b->groups[gi];
    snprintf(t, sizeof t, "%s{\"nx\": %d, \"ny\": %d, \"members\": %d, \"column_stages\": {", gi ? ", " : "", g.nx,
             g.ny, (int)g.mem.size());
    o += t;
    for (int q = 0; q < 4; ++q) {
      const int k = kColStages[q];
      snprintf(t, sizeof t,
               "%s\"%s\": {\"plan\": \"%s\", \"tx\": %d, \"us\": %.2f, \"static_us\": %.2f, \"candidates\": %d}",
               q ? ", " : "", kName[k], g.sel[k].ct ? "compile-time" : "runtime", g.sel[k].tx, g.tune_us[k],
               g.base_us[k], g.ncand[k]);
      o += t;
    }
    o += "}, \"graph_grids\": {";
    for (int k = 0; k < B_NST; ++k) {
      snprintf(t, sizeof t, "%s\"%s\": %d", k ? ", " : "", kName[k], g.cap[k]);
      o += t;
    }
    o += "}}";
  }
  o += "]}";
  const size_t n = std::min(o.size(), len - 1);
  memcpy(buf, o.data(), n);
  buf[n] = '\0';
  if (o.size() >= len) return set_err(FSIBE_ESIZE, "batch description needs %zu bytes", o.size() + 1);
  return FSIBE_OK;
}

// ---- discrete adjoint (fsibe_adjoint_*) -------------------------------------
#include "adjoint_host.hpp"
#include "backup_host.hpp"
#include "outputs_host.hpp"

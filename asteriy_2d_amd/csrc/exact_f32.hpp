// exact_f32.hpp -- the exact Riemann face flux of the fast path.
//
// Godunov_Solver_Alexashov (kernel.cu:128-570) in FP32: the same side swap
// (pI <= pII), the same wave-pattern test on Uud/Urz/Uvk, the same sampling
// at the face (w = 0) with the reference's region edges, and the same flux
// and dt -- with the p* solve adapted to FP32:
//  * two shocks: the root of newton's equation (kernel.cu:635-680) by Newton
//    in sqrt(p), to FP32 resolution, from the reference's PVRS-type estimate
//    or a learned guess;
//  * shock + rarefaction: the root of lev (kernel.cu:751-765) on the same
//    bracket [pI, pII] as devtwo's bisection (kernel.cu:682-749), found by a
//    bracket-safeguarded Newton iteration in (p/pII)^((g-1)/2g);
//  * FP64 islands: near vacuum and in strong rarefactions the p* equation
//    subtracts two nearly equal numbers, and FP32 would lose the digits of
//    p* there.  That difference -- and only it: every other term of these
//    equations is a sum of like-signed terms -- is formed in FP64 from FP64
//    sound speeds; the solve then runs in FP32 to FP32 accuracy.
//      two rarefactions, (Udf-Uvk)/(Urz-Uvk) < 0.05: the numerator
//        Udf - Uvk = (enI - enII) + 2/(g-1) (cI + cII);
//      shock + rarefaction, pI < 1e-4 pII: the constant D = c2 + du of the
//        pressure equation fI(p) + c2 q(p) - D = 0 (c2 = 2 cII/(g-1),
//        du = enI - enII, q = (p/pII)^((g-1)/2g)).
//    Counted in ast_stats_t.fp64_faces.  (No FP64 pow: the islands keep the
//    kernel's register budget, and so its occupancy, at the FP32 level.)
// Bound: vector instructions.  Against the same solves in p (seven
// transcendental operations a step, a pow among them, stopped at 1e-6) and a
// sampling per pattern: 2^24 faces 345 -> 187 us, the step at 2047x1021
// 41.5 -> 38.5; the error against 64 bits is the same (3.6e-8 of the flux, 99%
// of the values within 3.5e-6 of theirs, was 3.6e-6).
#pragma once
#include <hip/hip_runtime.h>
#include <math.h>

#include "fast_flux.hpp"
#include "mlp.hpp"
#include "dev.hpp"

namespace ast {

struct ExactCtx {
  float g, g1, g2, gp, gm, igm, ig1, c2g1, g1g2, c2g2;
  double gd, c2g1d;  // gamma, 2/(gamma - 1)
  int n;  // 1/gm = 2 gamma/(gamma - 1) when that is an integer in [1, 16] (5 for
          // gamma = 5/3, 7 for 7/5), else 0
  const unsigned char* mlp;  // learned-guess block (ast_mlp_t) in device memory, or null
  // When set, the kernel ORs 1 into *strong when it meets a strong two-shock
  // face (the runtime's learned mode, time_slots.h).
  uint32_t* strong;
  AST_DEV int order() const { return n; }
};
// The same with n known when the code is compiled: the powers are then
// straight-line products without the scalar tests and branches of the other
// orders (a fifth of the solver's code; the step at 2047x1021 36.4 -> 33.9 us,
// 2^24 fluxes 190 -> 183).  n = 5 only, gamma = 5/3; the kernels that count or
// serve the learned start, and the batch's, keep the general code.  Measured
// at gamma = 5/3 / 7/5 / 1.3: the step at 1021x509 15.4 / 16.4 / 16.1 us, 2^21
// fluxes 31 / 35 / 34.
struct ExactCtx5 : ExactCtx {
  AST_DEV explicit ExactCtx5(const ExactCtx& e) : ExactCtx(e) {}
  AST_DEV static constexpr int order() { return 5; }
};

static inline ExactCtx make_exact_ctx(double gamma, const void* mlp) {
  ExactCtx e;
  const double g1 = gamma - 1.0, g2 = gamma + 1.0;
  const double gp = (g2 / gamma) / 2.0, gm = (g1 / gamma) / 2.0;
  e.g = (float)gamma;
  e.g1 = (float)g1;
  e.g2 = (float)g2;
  e.gp = (float)gp;
  e.gm = (float)gm;
  e.igm = (float)(1.0 / gm);
  e.ig1 = (float)(1.0 / g1);
  e.c2g1 = (float)(2.0 / g1);
  e.g1g2 = (float)(g1 / g2);
  e.c2g2 = (float)(2.0 / g2);
  e.gd = gamma;
  e.c2g1d = 2.0 / g1;
  const double ig = 1.0 / gm, ni = floor(ig + 0.5);
  // (an FP32 gamma of 5/3 or 7/5 still counts: 1e-6 is its resolution)
  e.n = (fabs(ig - ni) <= 1e-6 * ig && ni >= 1.0 && ni <= 16.0) ? (int)ni : 0;
  e.mlp = (const unsigned char*)mlp;
  e.strong = nullptr;
  return e;
}

// x^y for x > 0 via the hardware log2/exp2 (about 1 ulp of FP32 each)
AST_DEV float fpow(float x, float y) { return __builtin_amdgcn_exp2f(y * __builtin_amdgcn_logf(x)); }

// For an integer n = 1/gm (e.n, wave-uniform): x^n by products and the
// geometric sum 1 + x + ... + x^(n-1) by Horner's rule, straight-line for
// n = 5 (gamma 5/3) and n = 7 (gamma 7/5), a loop otherwise.
AST_DEV float ipow(float x, int n) {
  if (n == 5) {
    const float x2 = x * x;
    return x2 * x2 * x;
  }
  if (n == 7) {
    const float x3 = x * x * x;
    return x3 * x3 * x;
  }
  float p = x;
  for (int k = 1; k < n; k++) p *= x;
  return p;
}
AST_DEV float geom_sum(float x, int n) {
  if (n == 5) return fmaf(fmaf(fmaf(fmaf(x, 1.f, 1.f), x, 1.f), x, 1.f), x, 1.f);
  if (n == 7)
    return fmaf(fmaf(fmaf(fmaf(fmaf(fmaf(x, 1.f, 1.f), x, 1.f), x, 1.f), x, 1.f), x, 1.f), x, 1.f);
  float s = 1.f;
  for (int k = 1; k < n; k++) s = fmaf(s, x, 1.f);
  return s;
}
// x^(1/gm): exact products for an integer 1/gm, else exp2/log2
template <class E>
AST_DEV float pow_igm(const E& e, float x) {
  return e.order() ? ipow(x, e.order()) : fpow(x, e.igm);
}

// x^(1/gm - 1), the same way
template <class E>
AST_DEV float pow_igm1(const E& e, float x) {
  if (e.order() == 5) {
    const float x2 = x * x;
    return x2 * x2;
  }
  if (e.order() == 7) {
    const float x2 = x * x;
    return x2 * x2 * x2;
  }
  return e.order() ? ipow(x, e.order() - 1) : fpow(x, e.igm - 1.f);
}
AST_DEV float frsq(float x) { return __builtin_amdgcn_rsqf(x); }

// What the exact solver did on one face (pat: -1 vacuum, 0 two
// rarefactions, 1 shock + rarefaction, 2 two shocks; kNoFace: not an exact
// face, e.g. a low-order face of the window).
constexpr int kNoFace = -3;
constexpr int kNoPattern = -9;  // an exact face whose input matches no wave pattern (NaN)
struct FaceInfo {
  int pat, it;
  bool capped, island, learned;
  bool strong;  // a strong two-shock face (the learned start's gate), when detected
};

AST_DEV uint32_t wcount(bool c) {
  return (uint32_t)__builtin_popcountll(__builtin_amdgcn_ballot_w64(c));
}

// The counter type of kernels that count nothing (counting costs the exact
// kernels a third of their time, so it is compiled only into the variants
// that are asked for counters).
struct NoStats {
  AST_DEV void clear() {}
  AST_DEV void add(const struct FaceInfo&) {}
  AST_DEV bool any_strong() const { return false; }
};
// Only whether the wave met a strong two-shock face (gated launches).
struct StrongStats {
  uint32_t strong;
  AST_DEV void clear() { strong = 0; }
  AST_DEV void add(const FaceInfo& f) { strong += wcount(f.strong); }
  AST_DEV bool any_strong() const { return strong != 0; }
};

// Solver counters of the FP32 exact solver.  Face counts are per wave
// (ballot + popcount: wave-uniform, kept in scalar registers), the iteration
// sums per lane.  Per-lane face counters would hold ten vector registers for
// the whole strip and cost the kernel a wave of occupancy.  add() runs in
// converged code (every lane of the wave active), after the face calls.
struct StatsF32 {
  uint32_t exact, newton, bisect, raref, vacuum, capped, fp64, mlp, strong;  // per wave
  uint32_t newton_it, bisect_it;                                             // per lane
  AST_DEV void clear() {
    exact = newton = bisect = raref = vacuum = capped = fp64 = mlp = strong = 0;
    newton_it = bisect_it = 0;
  }
  AST_DEV bool any_strong() const { return strong != 0; }
  AST_DEV void add(const FaceInfo& f) {
    strong += wcount(f.strong);
    exact += wcount(f.pat != kNoFace);
    raref += wcount(f.pat == 0);
    vacuum += wcount(f.pat == -1);
    bisect += wcount(f.pat == 1);
    newton += wcount(f.pat == 2);
    bisect_it += f.pat == 1 ? f.it : 0;
    newton_it += f.pat == 2 ? f.it : 0;
    capped += wcount(f.capped);
    fp64 += wcount(f.island);
    mlp += wcount(f.learned);
  }
};

// Adds a block's StatsF32 to *stats (ast_stats_t order); full workgroup.
template <int NT>
AST_DEV void block_stats_f32_to(const StatsF32& st, uint32_t* red, ast_stats_t* stats) {
  constexpr int NW = NT / 64;
  const uint32_t v[10] = {st.exact, st.newton, wave_sum(st.newton_it), st.bisect,
                          wave_sum(st.bisect_it), st.raref, st.vacuum, st.capped, st.fp64,
                          st.mlp};
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if (lane == 0)
    for (int i = 0; i < 10; i++) red[wave * 10 + i] = v[i];
  __syncthreads();
  if (threadIdx.x < 10) {
    unsigned long long t = 0;
    for (int w = 0; w < NW; w++) t += red[w * 10 + threadIdx.x];
    if (t) atomicAdd(reinterpret_cast<unsigned long long*>(stats) + threadIdx.x, t);
  }
}

constexpr float kBracket = 2e-7f;  // a bracket of y this narrow holds its root to 1e-6 in p
// a two-shock face is served by the learned guess when the PVRS start is
// poor: PVRS estimate above kStrongShock * pII (strong shocks)
constexpr float kStrongShock = 3.f;
constexpr float kVacuumIsland = 0.05f;
constexpr float kRarefIsland = 1e-4f;

// A Newton step stops the iterations below once it is at most kStep of the
// iterate: its own remainder is then below kStep^2 (both equations bend by
// less than that, curvature x / (2 slope) < 1), under the FP32 resolution.
constexpr float kStep = 1e-4f;

// Two shocks: the root of kernel.cu:635-680's equation
//   fI(p) + fII(p) = enI - enII,  fK = (p - pK) hK,
//   1/hK = zK sqrt(gp p/pK + gm),  zK = rK cK
// by Newton in w = sqrt(p): a strong shock's fK grows like sqrt(p), which is
// linear in w, so strong faces need no more steps than weak ones.  With sK =
// (gp p/pK + gm)^-1/2, dfK/dp = hK (1 + sK^2)/2: three transcendental
// operations a step.  In ratios of pressures, not as rK ((g+1) p + (g-1) pK)/2:
// that product leaves the FP32 range first (r = 1e-24, p = 1e-14), and a
// side without pressure has no p* here, as in the reference; the times are
// the same.  pee: the PVRS-type estimate, kernel.cu:640, the start unless a
// learned guess is used.  Every iterate is kept at or above pII (p* > pII in
// this pattern); a NaN stays one.
AST_DEV float newton_f32(const ExactCtx& e, float du, float pI, float rI, float cI, float pII,
                         float rII, float cII, float guess, bool use_guess, int& iters,
                         bool& capped) {
  const float zI = rI * cI, zII = rII * cII;
  const float pee = (pI * zII + pII * zI + du * zI * zII) * frcp(zI + zII);
  const float gI = e.gp * frcp(pI), gII = e.gp * frcp(pII), iI = frcp(zI), iII = frcp(zII);
  const float wlo = fsqrt(pII);
  float w = fmaxf(fsqrt(use_guess ? guess : pee), wlo);
  float p, dw;
  int k = 0;
  for (;;) {
    p = w * w;
    k++;
    const float sI = frsq(fmaf(gI, p, e.gm)), sII = frsq(fmaf(gII, p, e.gm));
    const float hI = iI * sI, hII = iII * sII;
    const float f = fmaf(p - pI, hI, fmaf(p - pII, hII, -du));
    // 2 df/dp
    const float d = fmaf(hI, fmaf(sI, sI, 1.f), hII * fmaf(sII, sII, 1.f));
    dw = -f * frcp(w * d);  // df/dw = w d
    if (!(fabsf(dw) > kStep * w)) break;
    if (k >= AST_ITER_CAP) { capped = true; break; }
    w = fmaxf(w + dw, wlo);
  }
  iters = k;
  const float pn = fmaf(dw, fmaf(2.f, w, dw), p);  // (w + dw)^2
  return pn < pII ? pII : pn;
}

// Shock + rarefaction: the root of lev (kernel.cu:751-765) on devtwo's
// bracket [pI, pII] (kernel.cu:682-749) by safeguarded Newton in
// y = (p/pII)^gm, in which the rarefaction is linear and p = pII y^n,
// n = 1/gm (5 for gamma 5/3: products, no power function).  With x = p/pII,
// xI = pI/pII and the shock's 1/hI = (rI pII ((g+1) x + (g-1) xI)/2)^1/2,
//   (rI/pII)^-1/2 (x - xI) s + c2 y - D = 0,  s = (((g+1) x + (g-1) xI)/2)^-1/2,
//   c2 = 2 cII/(g - 1),  D = c2 + enI - enII
// (D from the caller: FP64-formed in strong rarefactions); d/dx of (x - xI) s is
// s (1 + g xI s^2)/2, dx/dy = n x/y: two transcendental operations a step.
// q = (pI/pII)^gm; the start takes side I as a rarefaction too, whose root is
// (cI + cII + (g-1)/2 du)/(cI/q + cII).  Returns y and p.
template <class E>
AST_DEV float shock_raref_f32(const E& e, float du, float D, float pI, float rI, float cI,
                              float pII, float cII, float q, float& p, int& iters, bool& capped) {
  const float xI = pI * frcp(pII), k2 = 0.5f * e.g2, j = 0.5f * e.g1 * xI, gx = e.g * xI;
  const float A = fsqrt(pII) * frsq(rI), c2 = e.c2g1 * cII, hn = 0.5f * e.igm * A;
  float lo = q, hi = 1.f;
  float y = q * fmaf(0.5f * e.g1, du, cI + cII) * frcp(fmaf(q, cII, cI));
  y = fminf(fmaxf(y, lo), hi);
  if (!(y > 0.f)) y = 0.5f;  // pI / pII under the FP32 range
  int k = 0;
  for (;;) {
    k++;
    const float m = pow_igm1(e, y);  // x/y
    const float x = m * y;
    const float s = frsq(fmaf(k2, x, j));
    const float f = fmaf(x - xI, A * s, fmaf(c2, y, -D));
    const float df = fmaf(hn * m * s, fmaf(gx * s, s, 1.f), c2);
    const float dy = -f * frcp(df);
    if (f < 0.f) lo = y;
    else hi = y;
    float yn = y + dy;
    if (!(fabsf(dy) > kStep * y)) {
      y = fminf(fmaxf(yn, lo), hi);
      break;
    }
    if (!(yn > lo && yn < hi)) yn = 0.5f * (lo + hi);
    y = yn;
    if (!(hi - lo > kBracket * y)) break;
    if (k >= AST_ITER_CAP) { capped = true; break; }
  }
  iters = k;
  p = pII * pow_igm1(e, y) * y;
  return y;
}

// A face with its sides swapped so that pI <= pII (kernel.cu:156-184; u turns
// with them), the sides' sound speeds and q = (pI/pII)^gm.
struct ExactFace {
  float rI, pI, enI, teI, rII, pII, enII, teII, cI, cII, q;
  bool sw;
};
AST_DEV ExactFace exact_sides(const PrimF& L, const PrimF& R, const ExactCtx& e) {
  const bool sw = L.p > R.p;
  ExactFace f;
  f.sw = sw;
  f.rI = sw ? R.r : L.r;
  f.pI = sw ? R.p : L.p;
  f.enI = sw ? -R.u : L.u;
  f.teI = sw ? R.v : L.v;
  f.rII = sw ? L.r : R.r;
  f.pII = sw ? L.p : R.p;
  f.enII = sw ? -L.u : R.u;
  f.teII = sw ? L.v : R.v;
  f.cI = fsqrt(e.g * f.pI * frcp(f.rI));
  f.cII = fsqrt(e.g * f.pII * frcp(f.rII));
  f.q = fpow(f.pI * frcp(f.pII), e.gm);
  return f;
}

// The wave pattern: vacuum, two rarefactions, shock + rarefaction or two
// shocks.  Each pattern's whole interval is tested, so NaN input matches none.
// Four lane masks, which live in scalar registers.
struct WavePattern {
  bool vac, rr, sr, ss;
  // FaceInfo's number
  AST_DEV int number() const { return vac ? -1 : rr ? 0 : sr ? 1 : ss ? 2 : kNoPattern; }
};
AST_DEV WavePattern wave_pattern(const ExactFace& f, const ExactCtx& e) {
  const float Uud = (f.pII - f.pI) * frsq(f.rI * (e.g2 * f.pII + e.g1 * f.pI) * 0.5f);
  const float Urz = -e.c2g1 * f.cII * (1.f - f.q);
  const float Uvk = -e.c2g1 * (f.cII + f.cI);
  const float Udf = f.enI - f.enII;
  WavePattern w;
  w.vac = Udf < Uvk;
  w.rr = Udf >= Uvk && Udf <= Urz;
  w.sr = Udf > Urz && Udf <= Uud;
  w.ss = Udf > Uud;
  if (w.vac) w.rr = w.sr = w.ss = false;  // the first pattern that matches
  if (w.rr) w.sr = w.ss = false;
  if (w.sr) w.ss = false;
  return w;
}
// A two-shock face whose PVRS estimate is above kStrongShock * pII: the
// learned start's faces.
AST_DEV bool strong_shocks(const ExactFace& f) {
  const float zI = f.rI * f.cI, zII = f.rII * f.cII;
  return (f.pI * zII + f.pII * zI + (f.enI - f.enII) * zI * zII) * frcp(zI + zII) >
         kStrongShock * f.pII;
}

// A face's schedule key for sorting faces by pattern: 0 vacuum, 1 two
// rarefactions, 2 shock + rarefaction, 3 two shocks, 4 (STRONG) strong two
// shocks, 5 no pattern (NaN).
constexpr int kPatternKeys = 6;
template <bool STRONG>
AST_DEV int pattern_key(const ExactFace& f, const WavePattern& w) {
  return w.vac ? 0 : w.rr ? 1 : w.sr ? 2 : w.ss ? (STRONG && strong_shocks(f) ? 4 : 3) : 5;
}

// FP64 sound speed of an FP32 state (for the FP64-formed differences), c its
// FP32 value: 1/r and the root refined from the FP32 ones by Newton steps
// (1e-7 -> 1e-14 -> the last bits), a third of the double divide and square
// root's instructions.
AST_DEV double sound_speed_d(double g, float p, float r, float c) {
  const double rd = r, i0 = frcp(r);
  const double e0 = fma(-rd, i0, 1.0);
  const double x = g * (double)p * fma(i0, fma(e0, e0, e0), i0);
  const double h = c > 0.f ? 0.5f * frcp(c) : 0.f;
  double cd = c;
  cd = fma(fma(-cd, cd, x), h, cd);
  return fma(fma(-cd, cd, x), h, cd);
}

// The flux of a face of pattern w (kernel.cu:128-570 in FP32, see the
// header), as the physical flux of the state it samples at the face, written
// in that state's frame (FaceF: m = r un, w = (un, ut), gn = p, gt = 0, ge =
// un p/(g-1)); UU is the largest |wave speed| used for dt; fi reports the
// iterations and flags.  `guess` (finite, > 0) seeds newton.
//
// The patterns differ only in their p* solve: the sampling (kernel.cu:
// 234-544) is one code for all, with the side that holds w = 0 mirrored onto
// side I, so that lanes of different patterns and regions share it.  Faces
// outside both rarefactions take a side's state without a p*.
template <class E>
AST_DEV FaceF exact_solve_f32(const ExactFace& s, const WavePattern& w, const E& e,
                              float& UU, FaceInfo& fi, float guess) {
  const float g = e.g, g1 = e.g1, g2 = e.g2, gm = e.gm;
  const float enI = s.enI, enII = s.enII, pI = s.pI, pII = s.pII, rI = s.rI, rII = s.rII;
  const float cI = s.cI, cII = s.cII, Udf = enI - enII;
  // heads of the waves, the rarefactions' until a shock is found; the tails
  // lie between them, so the largest |speed| is a head's
  float dI = enI - cI, dII = enII + cII;
  // two rarefactions: t = (p/pI)^gm; Urz - Uvk = 2/(g-1) (cII q + cI) (no
  // cancellation)
  const float iden = frcp(e.c2g1 * fmaf(cII, s.q, cI));
  float t = (Udf + e.c2g1 * (cII + cI)) * iden;
  bool island = (w.rr && t < kVacuumIsland) || (w.sr && pI < kRarefIsland * pII);
  int it = 0;
  bool capped = false, learned = false;
  const bool shock = w.sr || w.ss;
  const bool outI = 0.f <= dI;
  bool one = outI;
  float en = outI ? enI : -enII, pp = outI ? pI : pII, r = outI ? rI : rII;
  bool empty = false;
  if (shock || !(outI || dII <= 0.f)) {
    const float zI = rI * cI, zII = rII * cII;
    float p = 0.f, aI = zI, aII = zII, y = 0.f;
    if (w.rr) {
      if (island) {  // FP64 island: near vacuum
        const double num = fma(e.c2g1d, sound_speed_d(e.gd, pI, rI, cI) +
                                        sound_speed_d(e.gd, pII, rII, cII),
                               (double)enI - (double)enII);
        t = fmaxf((float)num, 0.f) * iden;
      }
      y = t * s.q;
      p = pI * pow_igm(e, t);
    }
    if (w.sr) {
      float D = fmaf(e.c2g1, cII, Udf);
      if (island)  // FP64 island: strong rarefaction
        D = (float)fma(e.c2g1d, sound_speed_d(e.gd, pII, rII, cII), (double)enI - (double)enII);
      y = shock_raref_f32(e, Udf, D, pI, rI, cI, pII, cII, s.q, p, it, capped);
    }
    if (w.ss) {
      learned = guess > 0.f && guess < 3.0e38f;
      p = newton_f32(e, Udf, pI, rI, cI, pII, rII, cII, guess, learned, it, capped);
    }
    // impedances: shocks aK^2 = rK ((g+1) p + (g-1) pK)/2, speed enI - aI/rI
    // (enII + aII/rII); rarefactions (kernel.cu:369-388) aK = gm rK cK
    // (1 - x)/(1 - x^gm), x = p/pK, with x^gm = t (side I) and y (side II):
    // a geometric sum for an integer 1/gm
    const float hp = 0.5f * g2 * p;
    if (shock) {
      aI = fsqrt(rI * fmaf(0.5f * g1, pI, hp));
      dI = enI - aI * frcp(rI);
    } else if (e.order()) {
      aI = gm * zI * geom_sum(t, e.order());
    } else if (!(fabsf(p - pI) < 1e-6f * pI)) {
      aI = gm * zI * (1.f - p * frcp(pI)) * frcp(1.f - t);
    }
    if (w.ss) {
      aII = fsqrt(rII * fmaf(0.5f * g1, pII, hp));
      dII = enII + aII * frcp(rII);
    } else if (e.order()) {
      aII = gm * zII * geom_sum(y, e.order());
    } else if (!(fabsf(p - pII) < 1e-6f * pII)) {
      aII = gm * zII * (1.f - p * frcp(pII)) * frcp(1.f - y);
    }
    const float u = (aI * enI + aII * enII + pI - pII) * frcp(aI + aII);
    // rarefactions' tails; a vacuum's edges
    const float hg = 0.5f * g1;
    const float tI = w.vac ? fmaf(e.c2g1, cI, enI) : u - fmaf(hg, enI - u, cI);
    const float tII = w.vac ? fmaf(-e.c2g1, cII, enII) : u + fmaf(hg, u - enII, cII);
    // the side of the face, mirrored onto side I
    one = 0.f <= dI || (!shock && 0.f < tI) || (!w.vac && 0.f <= u);
    const float en0 = one ? enI : -enII, c0 = one ? cI : cII, us = one ? u : -u;
    const float head = one ? dI : -dII, tail = one ? tI : -tII;
    const bool sh0 = one ? shock : w.ss;
    en = en0;
    pp = one ? pI : pII;
    r = one ? rI : rII;
    if (head < 0.f) {  // (a NaN speed: the side's state)
      if (sh0) {
        const float a0 = one ? aI : aII;
        r = r * a0 * frcp(a0 - r * (en0 - us));
        en = us;
        pp = p;
      } else {
        const bool fan = 0.f < tail;
        const float ce = fan ? fmaf(e.g1g2, en0, e.c2g2 * c0) : fmaf(hg, en0 - us, c0);
        en = fan ? ce : us;
        pp = fan ? pp * pow_igm(e, ce * frcp(c0)) : p;
        r = g * pp * frcp(ce * ce);
        empty = w.vac && !one && !fan;  // between a vacuum's edges
      }
    }
  }
  fi.pat = w.number();
  fi.it = it;
  fi.capped = capped;
  fi.island = island;
  fi.learned = learned;
  UU = fmaxf(fabsf(dI), fabsf(dII));
  float te = one ? s.teI : s.teII;
  if (empty) en = pp = r = te = 0.f;
  if (!(w.vac || w.rr || shock)) {  // no pattern (NaN input): NaN fluxes, dt 0
    UU = INFINITY;
    en = pp = r = te = __int_as_float(0x7fc00000);
  }
  if (!(UU > 1e-7f)) UU = 1e-7f;  // eps8 floor of the reference's dt, kernel.cu:246-253
  if (one == s.sw) en = -en;      // side II mirrored, sides swapped: either turns u
  FaceF f;
  f.m = r * en;
  f.wn = en;
  f.wt = te;
  f.gn = pp;
  f.gt = 0.f;
  f.ge = en * pp * e.ig1;
  return f;
}

// The exact face flux of two states in the face frame (u normal, v tangential).
// LEARNED (compiled only into the kernels that serve a learned guess; its
// network needs registers the plain solver does not) with e.mlp set: the
// caller guarantees a full wave (EXEC all ones); if any lane of the wave
// holds a strong two-shock face, the wave evaluates the learned guess for
// all its lanes on MFMA (a wave-uniform branch) and those lanes start
// newton from it.
// DETECT: report strong two-shock faces (fi.strong) without the network.
template <bool LEARNED, bool DETECT = false, class E>
AST_DEV FaceF exact_frame_f32(const PrimF& L, const PrimF& R, const E& e, float& UU,
                              FaceInfo& fi, float guess = -1.f) {
  const ExactFace s = exact_sides(L, R, e);
  const WavePattern w = wave_pattern(s, e);
  // strong two-shock face (the learned kernel needs it for its wave ballot)
  bool strong = false;
  if constexpr (LEARNED || DETECT) strong = w.ss && strong_shocks(s);
  if (LEARNED && e.mlp != nullptr) {
    if (__builtin_amdgcn_ballot_w64(strong) != 0) {  // wave-uniform
      float fe[mlp::IN];
      const float lp = mlp::features<float>(s.rI, s.pI, s.enI, s.rII, s.pII, s.enII, e.g, fe);
      const float y = mlp::forward_wave_bf16(e.mlp, fe);
      if (strong) guess = __expf(y + lp);
    }
  }
  fi.strong = strong;
  return exact_solve_f32(s, w, e, UU, fi, guess);
}

// The same flux in the lab frame (face-frame axes).
template <bool LEARNED, bool DETECT = false, class E>
AST_DEV FluxF exact_f32(const PrimF& L, const PrimF& R, const E& e, float& UU,
                        FaceInfo& fi, float guess = -1.f) {
  return lab_flux(exact_frame_f32<LEARNED, DETECT>(L, R, e, UU, fi, guess));
}

}  // namespace ast

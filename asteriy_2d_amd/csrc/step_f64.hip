// step_f64.hip -- the FP64 step, the drop-in for the reference's Kernel_TVD
// (kernel.cu:2513-3073; axisymmetric update KorolkovSolver.cu:13-32) on
// gfx950: face-centric wave strips in IEEE double.
//
// A wave owns 64 consecutive columns (60 output columns and 2 halo columns on
// each side) and walks the rows [m0, m1) of its strip top to bottom.  Per row
// each lane
//  * takes its x-neighbours' states from the adjacent lanes (DPP wave shifts),
//    forms the minmod face values of its cell, and solves its WEST face once;
//    its east flux is the west flux of the next lane (another shift);
//  * solves the NORTH face of its cell from the rows m-1 .. m+2 it holds in
//    registers; the south flux is the north flux of the row before;
//  * updates its cell from the four fluxes (conservative update, the
//    r-weighted source in axisymmetric geometry, the reference's floors).
// So every face of the grid is solved once (the reference solves each
// interior face twice, once per cell, kernel.cu:2799-2857), with no LDS and no
// barrier inside the strip.  Slopes are the minmod of neighbour differences,
// c +- minmod(c - a, b - c)/2, which is the reference's coordinate-difference
// form (linear/linear2, kernel.cu:35-50) on a uniform grid without its
// divisions.
//
// The state stays in the reference's layout (two planes of double pairs);
// loads and stores are 16-byte accesses of consecutive columns.  Row m+3 is
// fetched while row m is computed.  Ghost cells follow the rules of
// fetch_cell (common.hpp), split so that they cost the other cells nothing:
// each lane loads the column its x rule names and each ghost row the row its
// y rule names, and the rule's transform (mirrored, clamped or fixed state)
// is applied a row later, when the fetch has arrived, under wave-uniform
// branches that only the bands and rows with ghosts take.  Frozen cells are
// looked for only by waves whose columns and rows can meet the region.  dt: each
// wave keeps the largest |wave speed| of the faces it solved for each
// direction, turns them into dt once, and workgroup minima lower *T with one
// 64-bit atomicMin on the IEEE bits (positive doubles order like their
// bits): the exact minimum over all faces, independent of the order.  The
// runtime spreads these atomics over 64 slots and lets the next step fold
// them and advance the time (time_slots.h), so that a step is one kernel:
// funk_time as a kernel of its own took 4.8 us of a step
// (Sod 256x128: 13.0 -> 9.5 us a step, 2048x1024 HLLC 51.3 -> 49.0,
// both with the fold under the first rows' loads).
#include <algorithm>
#include <type_traits>

#include "common.hpp"
#include "flux64.hpp"

namespace ast {
namespace s64 {

using namespace d64;

constexpr int WOUT = 60;  // output columns per wave
constexpr int WPB = 4;    // waves (stacked strips) per workgroup
constexpr int NT = 64 * WPB;

struct Q {
  double r, p, vx, vy;
};

AST_DEV Q q_sub(const Q& a, const Q& b) { return Q{a.r - b.r, a.p - b.p, a.vx - b.vx, a.vy - b.vy}; }

// lane i <- lane i - 1 (lane 0 keeps its own value) and lane i <- lane i + 1
// (lane 63 keeps its own): wave shifts by DPP on the two halves of a double.
AST_DEV double from_left(double v) {
  const int lo = __double2loint(v), hi = __double2hiint(v);
  return __hiloint2double(__builtin_amdgcn_update_dpp(hi, hi, 0x138, 0xf, 0xf, false),
                          __builtin_amdgcn_update_dpp(lo, lo, 0x138, 0xf, 0xf, false));
}
AST_DEV double from_right(double v) {
  const int lo = __double2loint(v), hi = __double2hiint(v);
  return __hiloint2double(__builtin_amdgcn_update_dpp(hi, hi, 0x130, 0xf, 0xf, false),
                          __builtin_amdgcn_update_dpp(lo, lo, 0x130, 0xf, 0xf, false));
}
AST_DEV Q from_left(const Q& q) {
  return Q{from_left(q.r), from_left(q.p), from_left(q.vx), from_left(q.vy)};
}
AST_DEV Q from_right(const Q& q) {
  return Q{from_right(q.r), from_right(q.p), from_right(q.vx), from_right(q.vy)};
}
AST_DEV FluxD from_right(const FluxD& f) {
  return FluxD{from_right(f.m), from_right(f.e), from_right(f.un), from_right(f.ut)};
}
AST_DEV bool from_left(bool b) {
  const int v = b ? 1 : 0;
  return __builtin_amdgcn_update_dpp(v, v, 0x138, 0xf, 0xf, false) != 0;
}

// minmod(a, b) (kernel.cu:22-33): the one of a, b nearer zero when they have
// the same sign, else 0 -- the median of a, b and 0.
AST_DEV double minmod(double a, double b) { return fmax(fmin(a, b), fmin(fmax(a, b), 0.0)); }

// Face values c + s and c - s with s = minmod(c - a, b - c)/2 (dl = c - a,
// dr = b - c).  A density or pressure face value <= 0 falls back to the cell
// value (kernel.cu:2706-2788); that can only happen for a cell state that is
// itself not positive, so the four tests run only in waves where one of the
// face values is not positive (c - |s| <= 0; wave-uniform).
AST_DEV void face_values(const Q& c, const Q& dl, const Q& dr, Q& hi, Q& lo) {
  const double sr = minmod(dl.r, dr.r), sp = minmod(dl.p, dr.p);
  const double sx = minmod(dl.vx, dr.vx), sy = minmod(dl.vy, dr.vy);
  // 0.5 s is exact: one fma rounds as c +- (0.5 s) does
  hi = Q{fma(0.5, sr, c.r), fma(0.5, sp, c.p), fma(0.5, sx, c.vx), fma(0.5, sy, c.vy)};
  lo = Q{fma(-0.5, sr, c.r), fma(-0.5, sp, c.p), fma(-0.5, sx, c.vx), fma(-0.5, sy, c.vy)};
  const bool low = fma(-0.5, fabs(sr), c.r) <= 0.0 || fma(-0.5, fabs(sp), c.p) <= 0.0;
  if (__builtin_amdgcn_ballot_w64(low) != 0) {
    if (hi.r <= 0.0) hi.r = c.r;
    if (hi.p <= 0.0) hi.p = c.p;
    if (lo.r <= 0.0) lo.r = c.r;
    if (lo.p <= 0.0) lo.p = c.p;
  }
}

// The column lane `n` of a row loads: itself, its ghost rule's source for
// the two ghost columns of a side, else the nearest grid column (columns
// past the halo of a partial band, read by no output cell).
AST_DEV int source_column(const ast_grid_t& g, int n) {
  if (n < 0) return g.bc[AST_XLO] == AST_BC_REFLECT ? -1 - n : 0;
  if (n < g.N) return n;
  return n <= g.N + 1 && g.bc[AST_XHI] == AST_BC_REFLECT ? 2 * g.N - 1 - n : g.N - 1;
}
// The row that row m loads, the same way (m >= -2; wave-uniform).
AST_DEV int source_row(const ast_grid_t& g, int m) {
  if (m < 0) return g.bc[AST_YLO] == AST_BC_REFLECT ? -1 - m : 0;
  if (m < g.M) return m;
  return m <= g.M + 1 && g.bc[AST_YHI] == AST_BC_REFLECT ? 2 * g.M - 1 - m : g.M - 1;
}

// The ghost rules' transforms of a loaded cell of row m (kernel.cu:2549-2698,
// 2328-2377): x_ghosts: the wave's band has ghost columns (wave-uniform).
// Corner ghosts, read by no cell, may take both.
AST_DEV void apply_ghost_rules(const ast_grid_t& g, Q& q, int n, int m, bool x_ghosts,
                               double pulse) {
  if (x_ghosts) {
    auto side = [&](int k, bool here) {
      const int bc = g.bc[k];  // wave-uniform
      if (bc == AST_BC_DIRICHLET || bc == AST_BC_DIRICHLET_PULSED) {
        const double r = bc == AST_BC_DIRICHLET_PULSED && pulsed_row(g, m)
                             ? g.bc_state[k][0] * pulse : g.bc_state[k][0];
        q.r = here ? r : q.r;
        q.p = here ? g.bc_state[k][1] : q.p;
        q.vx = here ? g.bc_state[k][2] : q.vx;
        q.vy = here ? g.bc_state[k][3] : q.vy;
      } else if (bc == AST_BC_REFLECT) {
        q.vx = here ? -q.vx : q.vx;
      } else if (bc == AST_BC_OUTFLOW_CLAMPED) {
        const double c = g.bc_vclamp[k];
        q.vx = here && (k == AST_XLO ? q.vx > c : q.vx < c) ? c : q.vx;
      }
    };
    side(AST_XLO, n < 0);
    side(AST_XHI, n >= g.N && n <= g.N + 1);
  }
  if (m < 0 || m >= g.M) {
    const int k = m < 0 ? AST_YLO : AST_YHI, bc = g.bc[k];
    if (bc == AST_BC_DIRICHLET || bc == AST_BC_DIRICHLET_PULSED) {
      const double r = bc == AST_BC_DIRICHLET_PULSED && pulsed_row(g, m)
                           ? g.bc_state[k][0] * pulse : g.bc_state[k][0];
      q = Q{r, g.bc_state[k][1], g.bc_state[k][2], g.bc_state[k][3]};
    } else if (bc == AST_BC_REFLECT) {
      q.vy = -q.vy;
    } else if (bc == AST_BC_OUTFLOW_CLAMPED) {
      const double c = g.bc_vclamp[k];
      if (k == AST_YLO ? q.vy > c : q.vy < c) q.vy = c;
    }
  }
}

// Can any cell of columns [n0, n1] x rows [m0, m1] lie in the frozen
// ellipse?  (wave-uniform; with a margin, so that rounding cannot matter)
AST_DEV bool frozen_possible(const ast_grid_t& g, int n0, int n1, int m0, int m1) {
  if (!(g.frozen_ax > 0.0)) return false;
  const double x0 = g.x_min + n0 * g.dx, x1 = g.x_min + n1 * g.dx;
  const double y0 = g.y_min + m0 * g.dy, y1 = g.y_min + m1 * g.dy;
  const double ax = g.frozen_ax * 1.01, ay = fabs(g.frozen_ay) * 1.01;
  return x1 >= g.frozen_x0 - ax && x0 <= g.frozen_x0 + ax && y1 >= -ay && y0 <= ay;
}

// Exact-solver counters of one lane (the STATS kernels), ast_stats_t order.
struct Counters {
  uint32_t v[10];
  AST_DEV void clear() {
    for (int k = 0; k < 10; k++) v[k] = 0;
  }
  AST_DEV void add(const ExactInfo& e, bool counted) {
    if (!counted || e.pat == -3) return;
    v[0] += 1;
    if (e.pat == 2) { v[1] += 1; v[2] += e.it; }
    if (e.pat == 1) { v[3] += 1; v[4] += e.it; }
    if (e.pat == 0) v[5] += 1;
    if (e.pat == -1) v[6] += 1;
    if (e.capped) v[7] += 1;
    if (e.guessed && e.pat == 2) v[9] += 1;
  }
};

// Adds a workgroup's counters to *stats.
AST_DEV void block_counters_to(const Counters& c, uint32_t* red, ast_stats_t* stats) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  for (int k = 0; k < 10; k++) {
    const uint32_t w = wave_sum(c.v[k]);
    if (lane == 0) red[wave * 10 + k] = w;
  }
  __syncthreads();
  if (threadIdx.x < 10) {
    unsigned long long t = 0;
    for (int w = 0; w < WPB; w++) t += red[w * 10 + threadIdx.x];
    if (t) atomicAdd(reinterpret_cast<unsigned long long*>(stats) + threadIdx.x, t);
  }
}

// The face between states l (left/below) and r (right/above) for a normal
// along x (NX) or y: high order -- the method on the reconstructed values lv,
// rv -- or, outside the high-order window, HLL on the cell states
// (kernel.cu:2812, 2838-2839, 2856).  Returns the flux in the face frame
// (un: momentum along the normal, ut: along the other axis) and the face's
// largest |wave speed|.
template <int METHOD, bool WINDOW, bool NX, class G>
AST_DEV FluxD face(const Q& lv, const Q& rv, const Q& l, const Q& r, bool ho, const G& a,
                   double& UU, ExactInfo& info) {
  info.pat = -3;  // no exact solve
  if (WINDOW && !ho) {
    const PrimD L = NX ? PrimD{l.r, l.p, l.vx, l.vy} : PrimD{l.r, l.p, l.vy, l.vx};
    const PrimD R = NX ? PrimD{r.r, r.p, r.vx, r.vy} : PrimD{r.r, r.p, r.vy, r.vx};
    return hll(L, R, a, UU);
  }
  const PrimD L = NX ? PrimD{lv.r, lv.p, lv.vx, lv.vy} : PrimD{lv.r, lv.p, lv.vy, lv.vx};
  const PrimD R = NX ? PrimD{rv.r, rv.p, rv.vx, rv.vy} : PrimD{rv.r, rv.p, rv.vy, rv.vx};
  return face_flux<METHOD>(L, R, a, UU, info);
}

struct StepArgs {
  ast_grid_t g;
  GasD gas;
  const double2* s;
  const double2* u;
  double2* s2;
  double2* u2;
  double* T;
  const double* T_do;
  const double* TT;  // simulation time (read only with a pulsed side; else null)
  KTime kt;          // the runtime's time protocol (time_slots.h), or all null
  ast_stats_t* stats;
  // neutral-H source planes of add_MK (kernel.cu:2495-2498), null when absent:
  // nn2 3 doubles per cell (x, y used), nn3 one
  const double* nn2;
  const double* nn3;
  double kmom, ken;
  int rows;    // rows per strip, or -S strips per band (strip_of)
  int nbands;  // bands of WOUT columns
  int nwg;     // workgroups
};

// The band and rows [m0, m1) of wave `wave` of workgroup `wg` (wave-uniform).
// rows > 0: strips of `rows` rows, WPB of them stacked per workgroup.  rows =
// -S: every band cut into S strips of equal height (to one row), the waves
// of all workgroups numbered band by band, so that the launch can hold
// exactly the waves that are resident at once; waves past the last band get
// no rows (m0 = M).
AST_DEV void strip_of(int M, int nbands, int rows, int wg, int wave, int& band, int& m0, int& m1) {
  if (rows > 0) {
    band = wg % nbands;
    m0 = ((wg / nbands) * WPB + wave) * rows;
    m1 = min(m0 + rows, M);
  } else {
    const int S = -rows, gw = wg * WPB + wave;
    band = gw / S;
    const int k = gw - band * S, h = M / S, r = M - h * S;
    m0 = k * h + min(k, r);
    m1 = m0 + h + (k < r ? 1 : 0);
    if (band >= nbands) {
      band = nbands - 1;
      m0 = m1 = M;
    }
  }
}

// G: the gas, with its order 1/gm compiled in (the exact solver) or not.
// Three waves a SIMD; the exact solver with the general power (232 VGPRs)
// would spill 244 B a lane for the third, so it keeps two.
template <int METHOD, class G>
constexpr int step_waves() {
  return METHOD == AST_EXACT && std::is_same<G, GasD>::value ? 2 : 3;
}
template <int METHOD, int GEOM, bool WINDOW, bool STATS, class G>
__global__ __launch_bounds__(NT, (step_waves<METHOD, G>())) void strip_kernel(StepArgs A) {
  __shared__ double red[WPB];
  __shared__ uint32_t redc[WPB * 10];
  const ast_grid_t& g = A.g;
  const G gas(A.gas);
  const int lane = threadIdx.x & 63;
  // wave index made explicitly uniform: rows and the loop stay scalar
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wg = xcd_tile(blockIdx.x, A.nwg);
  int band, m0, m1;
  strip_of(g.M, A.nbands, A.rows, wg, wave, band, m0, m1);
  const int n = band * WOUT + lane - 2;
  const bool out_col = (lane >= 2) & (lane < 2 + WOUT) & (n < g.N);
  // the west face of this lane's column is a face of an output cell
  const bool west_face = (lane >= 2) & (lane <= 2 + WOUT) & (n <= g.N);
  const double x = g.x_min + n * g.dx;
  const bool ho_x = high_order(g, x - g.dx / 2.0);  // west face (kernel.cu:2843)
  const bool ho_y = high_order(g, x);               // y faces: the cell x (kernel.cu:2816)
  const double dt_loaded = step_dt_load(A.T_do, A.kt);
  // pulsed Dirichlet sides: the density factor at the time before the step.
  // With the runtime's slots workgroup 0 advances TT during this step, so
  // the step takes the time the previous step of its run used (word 2 of
  // that step's slot set) plus its own dt -- the sum TT receives -- and
  // records its own; the first step of a run reads TT.
  double pulse = 1.0;
  if (A.TT != nullptr) {  // wave-uniform
    const double tt = A.kt.prev != nullptr ? A.kt.prev[2] + step_dt_fold(A.kt, dt_loaded) : *A.TT;
    if (A.kt.cur != nullptr && blockIdx.x == 0 && threadIdx.x == 0) A.kt.cur[2] = tt;
    pulse = pulse_factor(g, tt);
  }
  const bool any_out = m0 < g.M;  // wave-uniform (every band holds columns)
  // frozen grid cells are copied (kernel.cu:2317-2324); a face votes for dt
  // when one of its cells is a grid cell that is not frozen (frozen cells
  // return before their faces).  Without frozen cells that is every face of
  // an output cell, so the lanes are masked once, after the rows.
  const bool frz = any_out && frozen_possible(g, band * WOUT - 3, band * WOUT + 62, m0 - 1, m1);
  auto in_grid = [&](int nn, int mm) { return nn >= 0 && nn < g.N && mm >= 0 && mm < g.M; };
  auto frozen = [&](int nn, int mm) {
    return frz && in_grid(nn, mm) && is_frozen(g, g.x_min + nn * g.dx, g.y_min + mm * g.dy);
  };
  double UUx = 0.0, UUy = 0.0;
  Counters cnt;
  if constexpr (STATS) cnt.clear();

  if (any_out) {  // wave-uniform
    const bool x_ghosts = band * WOUT < 2 || band * WOUT + 61 >= g.N;
    const unsigned off = (unsigned)source_column(g, n);
    const unsigned out_off = (unsigned)max(n, 0);
    const int last = m1 + 1;  // the last row a fetch may name
    auto fetch = [&](int m) {
      const size_t row = (size_t)source_row(g, m) * g.N;
      const double2 a = A.s[row + off], b = A.u[row + off];
      return Q{a.x, a.y, b.x, b.y};
    };
    auto ghosts = [&](Q& q, int m) { apply_ghost_rules(g, q, n, m, x_ghosts, pulse); };
    // prologue: rows m0-2 .. m0+1 and the fetch of m0+2; the south face of
    // row m0.  w[k & 3] holds row m0 + k: the window slides by a change of
    // names in the unrolled rows below
    Q w[4], vn[2], dd[2];
    FluxD Gf[2];
    bool fr[2] = {false, false};
    double T_do;
    {
      Q qa = fetch(m0 - 2), qb = fetch(m0 - 1);
      w[0] = fetch(m0);
      w[1] = fetch(m0 + 1);
      w[2] = fetch(min(m0 + 2, last));
      __builtin_amdgcn_sched_barrier(0);  // the fetches go out before the dt fold waits
      T_do = step_dt_fold(A.kt, dt_loaded);
      step_dt_commit(A.T, A.kt, T_do);  // (by wave 0 of workgroup 0, which has rows)
      ghosts(qa, m0 - 2);
      ghosts(qb, m0 - 1);
      ghosts(w[0], m0);
      ghosts(w[1], m0 + 1);
      dd[0] = q_sub(w[1], w[0]);
      const Q db = q_sub(w[0], qb);
      Q nb, sb, s0;
      face_values(qb, q_sub(qb, qa), db, nb, sb);
      face_values(w[0], db, dd[0], vn[0], s0);
      double uu;
      ExactInfo ei;
      Gf[0] = face<METHOD, WINDOW, false>(nb, s0, qb, w[0], ho_y, gas, uu, ei);
      if (frz) {
        fr[0] = frozen(n, m0);
        const bool vote = (in_grid(n, m0 - 1) && !frozen(n, m0 - 1)) || (in_grid(n, m0) && !fr[0]);
        if (vote) UUy = fmax(UUy, uu);
      } else {
        UUy = fmax(UUy, uu);
      }
      if constexpr (STATS) cnt.add(ei, out_col && m0 == 0);
    }
    const double kx = div64(T_do, g.dx), ky = div64(T_do, g.dy);
    // T_do/y of the r-source: row m0 + 64 j + k in lane k, read back per row
    double tyl = 0.0;

    auto row = [&](auto tag, int m) {
      constexpr int J = decltype(tag)::value;
      const Q& q0 = w[J & 3];
      const Q& q1 = w[(J + 1) & 3];
      Q& q2 = w[(J + 2) & 3];
      ghosts(q2, min(m + 2, last));
      w[(J + 3) & 3] = fetch(min(m + 3, last));  // for the next row
      // y: face values of row m+1; the north face of row m
      const Q d2 = q_sub(q2, q1);
      Q vn1, vs1;
      face_values(q1, dd[J & 1], d2, vn1, vs1);
      dd[(J + 1) & 1] = d2;
      double uuy;
      ExactInfo eiy;
      const FluxD Gn = face<METHOD, WINDOW, false>(vn[J & 1], vs1, q0, q1, ho_y, gas, uuy, eiy);
      vn[(J + 1) & 1] = vn1;
      const FluxD Gs = Gf[J & 1];
      Gf[(J + 1) & 1] = Gn;
      // x: face values of row m; the west face (left value from lane - 1)
      const Q ql = from_left(q0);
      const Q dl = q_sub(q0, ql);
      Q ve, vw;
      face_values(q0, dl, from_right(dl), ve, vw);
      double uux;
      ExactInfo eix;
      const FluxD Fw = face<METHOD, WINDOW, true>(from_left(ve), vw, ql, q0, ho_x, gas, uux, eix);
      const FluxD Fe = from_right(Fw);
      // votes
      const bool fr_m = fr[J & 1];
      if (frz) {
        const bool fr_up = frozen(n, m + 1);
        const bool vote_here = in_grid(n, m) && !fr_m;
        const bool vote_up = in_grid(n, m + 1) && !fr_up;
        const bool vote_left = from_left(vote_here);
        if (vote_here || vote_up) UUy = fmax(UUy, uuy);
        if (vote_here || vote_left) UUx = fmax(UUx, uux);
        fr[(J + 1) & 1] = fr_up;
      } else {
        UUy = fmax(UUy, uuy);
        UUx = fmax(UUx, uux);
      }
      if constexpr (STATS) {
        cnt.add(eiy, out_col);
        cnt.add(eix, west_face);
      }
      // conservative update (kernel.cu:3027-3032, 3059-3073): dU = -T_do/dx
      // (F_e - F_w) - T_do/dy (G_n - G_s)
      double dr = -kx * (Fe.m - Fw.m) - ky * (Gn.m - Gs.m);
      double dE = -kx * (Fe.e - Fw.e) - ky * (Gn.e - Gs.e);
      double dmx = -kx * (Fe.un - Fw.un) - ky * (Gn.ut - Gs.ut);
      double dmy = -kx * (Fe.ut - Fw.ut) - ky * (Gn.un - Gs.un);
      const double ke = 0.5 * q0.r * (q0.vx * q0.vx + q0.vy * q0.vy);
      const double mx = q0.r * q0.vx, my = q0.r * q0.vy;
      if constexpr (GEOM == AST_AXISYMMETRIC) {
        // KorolkovSolver.cu:13-32: -(T_do/y) v {rho, rho u, rho v, gamma p/(g-1) + KE}
        const int k = (m - m0) & 63;
        if (k == 0) tyl = div64(T_do, g.y_min + (m + lane) * g.dy);
        const double ty = __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(tyl), k),
                                           __builtin_amdgcn_readlane(__double2loint(tyl), k));
        const double tr = ty * my;
        dr -= tr;
        dmx -= tr * q0.vx;
        dmy -= tr * q0.vy;
        dE -= ty * q0.vy * (gas.g * gas.ig1 * q0.p + ke);
      }
      const size_t rowk = (size_t)m * g.N;
      if (A.nn2 != nullptr || A.nn3 != nullptr) {  // wave-uniform
        // neutral-H sources (kernel.cu:2495-2498): momentum T_do (rho kmom)
        // nn2.{x,y}, energy T_do ken nn3; output cells only (in bounds)
        const size_t k = out_col ? rowk + out_off : 0;
        if (A.nn2 != nullptr) {
          const double tk = T_do * (q0.r * A.kmom);
          dmx += tk * (out_col ? A.nn2[3 * k] : 0.0);
          dmy += tk * (out_col ? A.nn2[3 * k + 1] : 0.0);
        }
        if (A.nn3 != nullptr) dE += (T_do * A.ken) * (out_col ? A.nn3[k] : 0.0);
      }
      // density floor (kernel.cu:3060-3064): a non-positive density keeps
      // the old one, and the kinetic energy of the new state uses it
      const bool rfloor = q0.r + dr <= 0.0;
      const double drf = rfloor ? 0.0 : dr;
      const double r2 = q0.r + drf;
      const double ir2 = rcp64(r2);  // shared by the three quotients
      const double vx2 = div64(mx + dmx, r2, ir2);
      const double vy2 = div64(my + dmy, r2, ir2);
      // p' = (E' - rho'|u'|^2/2)(g-1) with the O(E) terms cancelled exactly:
      // KE' - KE = (m.dm + |dm|^2/2 - KE dr)/rho'
      const double dke =
          div64(mx * dmx + my * dmy + 0.5 * (dmx * dmx + dmy * dmy) - ke * drf, r2, ir2);
      double p2 = q0.p + gas.g1 * (dE - dke);
      if (p2 <= 0.0) p2 = 0.000001;  // kernel.cu:3070-3073
      if (out_col) {
        double2 so = make_double2(r2, p2), uo = make_double2(vx2, vy2);
        if (frz && fr_m) {  // frozen: copied (kernel.cu:2317-2324)
          so = make_double2(q0.r, q0.p);
          uo = make_double2(q0.vx, q0.vy);
        }
        A.s2[rowk + out_off] = so;
        A.u2[rowk + out_off] = uo;
      }
    };
    // four rows a trip, so that the window slides by names; the exact solver
    // (two inlined solvers a row, ~40 KB of code) takes one row a trip and
    // moves the window
    if constexpr (METHOD == AST_EXACT) {
      for (int m = m0; m < m1; m++) {
        row(std::integral_constant<int, 0>{}, m);
        for (int k = 0; k < 3; k++) w[k] = w[k + 1];
        vn[0] = vn[1];
        dd[0] = dd[1];
        Gf[0] = Gf[1];
        fr[0] = fr[1];
      }
    } else {
      for (int m = m0; m < m1; m += 4) {
        // wave priority falls with the fraction of the strip done, so that
        // the waves of a SIMD end together (a SIMD issues for its oldest
        // wave first, and the last would run alone)
        const int q = (4 * (m - m0)) / (m1 - m0);  // wave-uniform, 0..3
        if (q == 0) __builtin_amdgcn_s_setprio(3);
        else if (q == 1) __builtin_amdgcn_s_setprio(2);
        else if (q == 2) __builtin_amdgcn_s_setprio(1);
        else __builtin_amdgcn_s_setprio(0);
        row(std::integral_constant<int, 0>{}, m);
        if (m + 1 >= m1) break;
        row(std::integral_constant<int, 1>{}, m + 1);
        if (m + 2 >= m1) break;
        row(std::integral_constant<int, 2>{}, m + 2);
        if (m + 3 >= m1) break;
        row(std::integral_constant<int, 3>{}, m + 3);
      }
    }
  }
  // per-face dt = krit*rad/UU (monotone in UU), capped at 1000 (kernel.cu:2530)
  UUx = wave_max(west_face ? UUx : 0.0);
  UUy = wave_max(out_col ? UUy : 0.0);
  double tmin = any_out ? 1000.0 : INFINITY;
  if (UUx > 0.0) tmin = fmin(tmin, g.krit * g.dx / UUx);
  if (UUy > 0.0) tmin = fmin(tmin, g.krit * g.dy / UUy);
  tmin = first_step_min(tmin, A.T, A.kt);
  block_min_uniform<NT>(tmin, red, A.kt.cur ? A.kt.cur : A.T, A.kt.cur ? A.kt.nslots : 0);
  if constexpr (STATS) block_counters_to(cnt, redc, A.stats);
}

template <int METHOD, int GEOM, bool WINDOW>
static int launch3(const StepArgs& a, bool stats, hipStream_t st) {
  auto kernel = strip_kernel<METHOD, GEOM, WINDOW, false, GasD>;
  if constexpr (METHOD == AST_EXACT) {
    using G5 = GasN<5>;
    if (a.gas.n == 5)
      kernel = stats ? strip_kernel<METHOD, GEOM, WINDOW, true, G5>
                     : strip_kernel<METHOD, GEOM, WINDOW, false, G5>;
    else if (stats)
      kernel = strip_kernel<METHOD, GEOM, WINDOW, true, GasD>;
  }
  hipLaunchKernelGGL(kernel, dim3(a.nwg), dim3(NT), 0, st, a);
  AST_LAUNCH_CHECK("ast_step_f64 launch");
  return AST_OK;
}

template <int METHOD>
static int launch(const StepArgs& a, bool stats, bool window, hipStream_t st) {
  const bool axi = a.g.geometry == AST_AXISYMMETRIC;
  if (axi)
    return window ? launch3<METHOD, AST_AXISYMMETRIC, true>(a, stats, st)
                  : launch3<METHOD, AST_AXISYMMETRIC, false>(a, stats, st);
  return window ? launch3<METHOD, AST_PLANAR, true>(a, stats, st)
                : launch3<METHOD, AST_PLANAR, false>(a, stats, st);
}

}  // namespace s64
}  // namespace ast

// The default strip tiling (ast_step_f64_rows, rows = 0; strip_of's
// convention).  A wave's row is one chain of dependent FP64 operations, and a
// SIMD holds three waves, so the launch is cut into S equal strips a band
// that give every SIMD the same 1, 2 or 3 waves, or whole rounds of 3: few
// waves of many rows leave the chains exposed, many short strips pay their
// prologue (south face, first fetches) and the rounds' changes.  The rule
// takes the count with the least time fitted to the measured ones (us, h the
// tallest strip's rows): 1.5 h + 6, 1.85 h + 8 and 2.7 h + 8 for 1, 2 and 3
// waves a SIMD, 2.6 r h + 4 r + 4 for r rounds of 3.
// Measured, us a step (HLLC; the rule / 6-row strips): 256x128 8.0 / 14.7,
// 512x256 10.7 / 15.7, 1024x512 17.5 / 19.4, 1500x750 26.5 / 34.3, 2048x1024
// 39.3 / 46.6, 8192x400 60.7 / 73.0, 4096x2048 135 / 166, 32000x400 216 / 257.
// The exact solver's rows differ by tens of times between waves (its
// patterns and iterations diverge), so its strips stay short until 16384 of
// them share the load: 256x128 26.0 (1 row) / 95.7, 1500x750 56.6 (2) / 106.4,
// 2048x1024 82.1 (3) / 109.1, 4096x2048 about 243 (9) / 246.5.
int ast_step_f64_default_tile(const ast_grid_t* g, int method) {
  const long long nbands = (g->N + ast::s64::WOUT - 1) / ast::s64::WOUT, M = g->M;
  if (method == AST_EXACT) return (int)std::min((nbands * M + 16383) / 16384, 32LL);
  int best = 32;
  double cost = INFINITY;
  for (int waves = 1; waves <= 192; waves += waves < 3 ? 1 : 3) {
    const long long S = std::min(M, waves * 1024 / nbands);
    if (S < 1) continue;
    const double h = (double)((M + S - 1) / S), r = waves / 3;
    const double c = waves == 1   ? 1.5 * h + 6.0
                     : waves == 2 ? 1.85 * h + 8.0
                     : waves == 3 ? 2.7 * h + 8.0
                                  : 2.6 * r * h + 4.0 * r + 4.0;
    if (c < cost) {
      cost = c;
      best = (int)-S;
    }
  }
  return best;
}

// The step with a given strip tiling (strip_of; 0 = the default) and
// optional neutral-H source planes (src may be null).  tm (may be null): the
// runtime's time protocol (time_slots.h); null: the reference protocol (the
// step lowers *T, dt is *T_do).
int ast_step_f64_rows(const ast_grid_t* g, const double* s, const double* u, double* s2,
                      double* u2, double* T, const double* T_do, const double* TT, int method,
                      ast_stats_t* stats, int rows, const ast::StepTime* tm,
                      const ast_sources_t* src, void* stream) {
  using namespace ast::s64;
  int rc = ast_grid_check(g);
  if (rc != AST_OK) return rc;
  if (!s || !u || !s2 || !u2 || !T || !T_do)
    return ast_fail(AST_ERR_ARG, "ast_step_f64: null state or time pointer");
  if (s == s2 || u == u2 || s == u2 || u == s2)
    return ast_fail(AST_ERR_ARG, "ast_step_f64: output planes must not alias the input planes");
  if (rows == 0) rows = ast_step_f64_default_tile(g, method);
  if (rows == 0 || rows > 4096 || rows < -g->M) return ast_fail(AST_ERR_ARG, "ast_step_f64: %d rows per strip", rows);
  StepArgs a;
  a.g = *g;
  a.gas = ast::d64::make_gas(g->gamma);
  a.s = (const double2*)s;
  a.u = (const double2*)u;
  a.s2 = (double2*)s2;
  a.u2 = (double2*)u2;
  a.T = T;
  a.T_do = T_do;
  bool pulsed = false;
  for (int k = 0; k < 4; k++) pulsed |= g->bc[k] == AST_BC_DIRICHLET_PULSED;
  if (pulsed && !TT)
    return ast_fail(AST_ERR_ARG, "ast_step_f64: a pulsed Dirichlet side needs the time TT");
  a.TT = pulsed ? TT : nullptr;
  a.kt = ast::KTime{nullptr, nullptr, nullptr, 0};
  if (tm != nullptr) {
    if (tm->nslots < 1 || tm->nslots > ast::kMaxSlots || tm->cur == nullptr)
      return ast_fail(AST_ERR_ARG, "ast_step_f64: %d dt slots", tm->nslots);
    a.kt = ast::KTime{tm->prev, tm->cur, tm->rst, tm->nslots};
  }
  a.stats = stats;
  a.nn2 = src ? src->nn2 : nullptr;
  a.nn3 = src ? src->nn3 : nullptr;
  a.kmom = src ? src->kmom : 0.0;
  a.ken = src ? src->ken : 0.0;
  if (a.nn2 == s || a.nn2 == u || a.nn3 == s || a.nn3 == u)
    return ast_fail(AST_ERR_ARG, "ast_step_f64: a source plane aliases a state plane");
  a.rows = rows;
  a.nbands = (g->N + WOUT - 1) / WOUT;
  const long long nwg = rows > 0
      ? (long long)a.nbands * (((g->M + rows - 1) / rows + WPB - 1) / WPB)
      : ((long long)a.nbands * -(long long)rows + WPB - 1) / WPB;
  if (nwg > 0x7fffffffLL) return ast_fail(AST_ERR_SIZE, "ast_step_f64: grid too large");
  a.nwg = (int)nwg;
  const bool window = !(g->ho_lo == -INFINITY && g->ho_hi == INFINITY);
  const bool st = stats != nullptr;
  hipStream_t hs = (hipStream_t)stream;
  switch (method) {
    case AST_HLL: return launch<AST_HLL>(a, st, window, hs);
    case AST_HLLC: return launch<AST_HLLC>(a, st, window, hs);
    case AST_EXACT: return launch<AST_EXACT>(a, st, window, hs);
    case AST_HLLC_A: return launch<AST_HLLC_A>(a, st, window, hs);
    default:
      return ast_fail(AST_ERR_ARG,
                      "ast_step_f64: method %d is not AST_HLL/AST_HLLC/AST_EXACT/AST_HLLC_A",
                      method);
  }
}

extern "C" int ast_step_f64(const ast_grid_t* g, const double* s, const double* u, double* s2,
                            double* u2, double* T, const double* T_do, double* TT, int method,
                            ast_stats_t* stats, void* stream) {
  // TT is read only with a pulsed Dirichlet side (unused by the reference's
  // live body)
  return ast_step_f64_rows(g, s, u, s2, u2, T, T_do, TT, method, stats, 0, nullptr, nullptr,
                           stream);
}

extern "C" int ast_step_f64_src(const ast_grid_t* g, const double* s, const double* u,
                                double* s2, double* u2, double* T, const double* T_do, double* TT,
                                int method, const ast_sources_t* src, ast_stats_t* stats,
                                void* stream) {
  return ast_step_f64_rows(g, s, u, s2, u2, T, T_do, TT, method, stats, 0, nullptr, src, stream);
}

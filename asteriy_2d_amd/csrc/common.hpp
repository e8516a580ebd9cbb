// common.hpp -- shared device/host helpers of the HIP kernels: error
// reporting of the C-ABI, the XCD-aware tile order, the ghost-cell rules,
// and the deterministic block reductions (dt min).
#pragma once
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>

#include "../../include/asteriy.h"
#include "dev.hpp"
#include "time_slots.h"

// ---- host side: status + message of the last failure (api.cpp) ----------
int ast_fail(int code, const char* fmt, ...);
int ast_hip_fail(hipError_t e, const char* where);
#define AST_HIP_CHECK(call)                                   \
  do {                                                        \
    hipError_t _e = (call);                                   \
    if (_e != hipSuccess) return ast_hip_fail(_e, #call);     \
  } while (0)
#define AST_LAUNCH_CHECK(where)                               \
  do {                                                        \
    hipError_t _e = hipGetLastError();                        \
    if (_e != hipSuccess) return ast_hip_fail(_e, where);     \
  } while (0)

namespace ast {

// The hardware hands workgroup i to XCD (i mod 8).  Remap so that each XCD
// receives one contiguous run of tiles: neighbouring tiles share halo rows
// and then meet in the same XCD's L2.
AST_DEV int xcd_tile(int bid, int ntiles) {
  const int nx = 8;
  int q = ntiles / nx, r = ntiles % nx;
  int xcd = bid % nx, local = bid / nx;
  return xcd * q + (xcd < r ? xcd : r) + local;
}

// Density factor of AST_BC_DIRICHLET_PULSED sides at simulation time TT
// (add2's inflow perturbation, kernel.cu:2022-2025): 1 + a sin(w TT) while
// TT < t_lim, else 1.
AST_DEV double pulse_factor(const ast_grid_t& g, double TT) {
  return TT < g.bc_pulse[3] ? 1.0 + g.bc_pulse[0] * sin(TT * g.bc_pulse[1]) : 1.0;
}

// Does row m (ghost rows included) have its centre below the pulsed sides'
// y_lim?  The sum is formed unfused, as the host forms it.
__host__ __device__ __forceinline__ bool pulsed_row(const ast_grid_t& g, int m) {
#pragma clang fp contract(off)
  return g.y_min + m * g.dy < g.bc_pulse[2];
}

// Cell (n, m) of a state plane with the ghost rules of Kernel_TVD
// (kernel.cu:2549-2698) and add_MK (kernel.cu:2328-2377).  Indices may lie
// up to 2 cells outside the grid on at most one axis; anything else
// (corners, beyond the halo of a partial tile) is never read by a cell and
// returns zeros.  pulse: the density factor of pulsed Dirichlet ghosts whose
// centre lies below y_lim (pulse_factor).
template <typename P>
AST_DEV void fetch_cell(const ast_grid_t& g, const P* __restrict__ s, const P* __restrict__ u,
                        int n, int m, P& so, P& uo, double pulse = 1.0) {
  const int N = g.N, M = g.M;
  const bool xin = (n >= 0) & (n < N), yin = (m >= 0) & (m < M);
  if (xin & yin) {
    so = s[(size_t)m * N + n];
    uo = u[(size_t)m * N + n];
    return;
  }
  so.x = so.y = uo.x = uo.y = 0;
  if ((!xin & !yin) | (n < -2) | (n > N + 1) | (m < -2) | (m > M + 1)) return;
  int side, in_n = n, in_m = m;
  if (n < 0) { side = AST_XLO; in_n = -1 - n; }
  else if (n >= N) { side = AST_XHI; in_n = 2 * N - 1 - n; }
  else if (m < 0) { side = AST_YLO; in_m = -1 - m; }
  else { side = AST_YHI; in_m = 2 * M - 1 - m; }
  const int bc = g.bc[side];
  if (bc == AST_BC_DIRICHLET || bc == AST_BC_DIRICHLET_PULSED) {
    so.x = g.bc_state[side][0];
    so.y = g.bc_state[side][1];
    uo.x = g.bc_state[side][2];
    uo.y = g.bc_state[side][3];
    if (bc == AST_BC_DIRICHLET_PULSED && pulsed_row(g, m))
      so.x = (decltype(so.x))(g.bc_state[side][0] * pulse);
    return;
  }
  if (bc == AST_BC_REFLECT) {
    size_t k = (size_t)in_m * N + in_n;
    so = s[k];
    uo = u[k];
    if (side <= AST_XHI) uo.x = -uo.x;
    else uo.y = -uo.y;
    return;
  }
  int en = n < 0 ? 0 : (n >= N ? N - 1 : n);
  int em = m < 0 ? 0 : (m >= M ? M - 1 : m);
  size_t k = (size_t)em * N + en;
  so = s[k];
  uo = u[k];
  if (bc == AST_BC_OUTFLOW_CLAMPED) {
    // kernel.cu:2347-2350 caps the lo-side normal velocity from above; the
    // hi side is the mirror image.
    const auto c = (decltype(uo.x))g.bc_vclamp[side];
    if (side == AST_XLO) { if (uo.x > c) uo.x = c; }
    else if (side == AST_XHI) { if (uo.x < c) uo.x = c; }
    else if (side == AST_YLO) { if (uo.y > c) uo.y = c; }
    else { if (uo.y < c) uo.y = c; }
  }
}

// Frozen region of add_MK (kernel.cu:2317-2324) as an ellipse.
AST_DEV bool is_frozen(const ast_grid_t& g, double x, double y) {
  if (!(g.frozen_ax > 0.0)) return false;
  double dxr = x - g.frozen_x0;
  double d = (dxr * dxr) / (g.frozen_ax * g.frozen_ax) + (y * y) / (g.frozen_ay * g.frozen_ay);
  return d < 1.0;
}

AST_DEV bool high_order(const ast_grid_t& g, double xf) { return xf > g.ho_lo && xf < g.ho_hi; }

// ---- wave64 / block reductions ------------------------------------------

// v of the lane DPP control CTRL names, in the rows of ROWS (a lane without
// a source, or in another row, keeps its own).
template <int CTRL, int ROWS>
AST_DEV double dpp64(double v) {
  const int lo = __double2loint(v), hi = __double2hiint(v);
  return __hiloint2double(__builtin_amdgcn_update_dpp(hi, hi, CTRL, ROWS, 0xf, false),
                          __builtin_amdgcn_update_dpp(lo, lo, CTRL, ROWS, 0xf, false));
}
// The minimum / maximum over the wave, wave-uniform (every lane active): row
// shifts by 1, 2, 4, 8 leave each row's result in its lane 15, row_bcast:15
// and :31 carry them to lane 63.  Six register moves in place of six rounds
// through the LDS permute.
template <class F>
AST_DEV double wave_reduce(double v, F f) {
  v = f(v, dpp64<0x111, 0xf>(v));
  v = f(v, dpp64<0x112, 0xf>(v));
  v = f(v, dpp64<0x114, 0xf>(v));
  v = f(v, dpp64<0x118, 0xf>(v));
  v = f(v, dpp64<0x142, 0xa>(v));
  v = f(v, dpp64<0x143, 0xc>(v));
  return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), 63),
                          __builtin_amdgcn_readlane(__double2loint(v), 63));
}
AST_DEV double wave_min(double v) {
  return wave_reduce(v, [](double a, double b) { return fmin(a, b); });
}
AST_DEV double wave_max(double v) {
  return wave_reduce(v, [](double a, double b) { return fmax(a, b); });
}
AST_DEV uint32_t wave_sum(uint32_t v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  return v;
}

// Lowers *T to the block minimum of tmin, which is uniform across each wave.
// Positive IEEE doubles order like their bit patterns, so one 64-bit
// atomicMin on the bits gives the exact, order-independent minimum (the
// reference's store, kernel.cu:3013-3017, is racy).  `red` is LDS of at least
// nwaves doubles.  With nslots > 0, T is a set of dt slots (time_slots.h) and
// workgroup b lowers slot (b mod nslots), so that no single address takes
// every workgroup's atomic; the time advance folds the slots.  Without
// slots the atomics of one address follow each other (about 17 ns each, and
// workgroups of equal strips end together), so a workgroup looks first
// whether *T is already as low, as it is for nearly all.
template <int NT>
AST_DEV void block_min_uniform(double tmin, double* red, double* T, int nslots) {
  constexpr int NW = NT / 64;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if (lane == 0) red[wave] = tmin;
  __syncthreads();
  if (threadIdx.x == 0) {
    double t = red[0];
#pragma unroll
    for (int i = 1; i < NW; i++) t = fmin(t, red[i]);
    double* dst = nslots > 0 ? T + kSlotStride * (int)(blockIdx.x % (unsigned)nslots) : T;
    auto* word = reinterpret_cast<unsigned long long*>(dst);
    const auto bits = (unsigned long long)__double_as_longlong(t);
    const bool lower = nslots > 0 || __hip_atomic_load(word, __ATOMIC_RELAXED,
                                                       __HIP_MEMORY_SCOPE_AGENT) > bits;
    if (t < INFINITY && lower) atomicMin(word, bits);
  }
}

// The time arguments of one step launch (time_slots.h): prev, the slot set
// of the previous step (null: dt is *T_do); cur, the set this step lowers
// (null: *T itself); rst, a set to clear (may be null).
struct KTime {
  const double* prev;
  double* cur;
  double* rst;
  int nslots;
};

// dt of this step, in three parts.  With a previous slot set dt is the
// minimum of its slots (every wave folds them itself: no workgroup waits for
// another), else *T_do: step_dt_load issues the loads, step_dt_fold takes
// the minimum, where the kernel first needs it, so that the strip's own
// first loads are under way meanwhile.  step_dt_commit (the writes): with a
// previous set, wave 0 of workgroup 0 performs the previous step's
// time advance, funk_time of kernel.cu:1525-1536 (T_do = that minimum,
// TT += T_do, i += 1; T stays at its reset value); it clears the set `rst`
// for the step after.
AST_DEV double step_dt_load(const double* T_do, const KTime& kt) {
  const int lane = threadIdx.x & 63;
  if (kt.prev != nullptr) return lane < kt.nslots ? kt.prev[kSlotStride * lane] : INFINITY;
  return *T_do;
}
AST_DEV double step_dt_fold(const KTime& kt, double loaded) {
  return kt.prev != nullptr ? wave_min(loaded) : loaded;
}
AST_DEV void step_dt_commit(double* T, const KTime& kt, double t) {
  const int lane = threadIdx.x & 63;
  if (blockIdx.x == 0 && threadIdx.x < 64) {
    if (kt.rst != nullptr) {
      if (lane < kt.nslots) kt.rst[kSlotStride * lane] = kSlotEmpty;
      if (lane == 0) reinterpret_cast<uint32_t*>(kt.rst + 1)[0] = 0u;
    }
    if (kt.prev != nullptr && lane == 0) {
      T[1] = t;
      T[2] = T[2] + t;
      int* i = reinterpret_cast<int*>(T + 3);
      *i = *i + 1;
    }
  }
}

// The wave's dt candidate after the T that the first step of a run finds:
// that step lowers T (set_time may have left one below the step's own
// minimum), so its slots start from it and T[0] is reset, by wave 0 of
// workgroup 0 (every lane active).  Compared as the atomics compare, by the
// IEEE bits: a T that is negative or NaN limits nothing.
AST_DEV double lower_of(double t, double T) {
  const auto a = (unsigned long long)__double_as_longlong(t);
  const auto b = (unsigned long long)__double_as_longlong(T);
  return b < a ? T : t;
}
AST_DEV double first_step_min(double tmin, double* T, const KTime& kt) {
  if (kt.cur != nullptr && kt.prev == nullptr && blockIdx.x == 0 && threadIdx.x < 64) {
    tmin = lower_of(tmin, T[0]);
    if ((threadIdx.x & 63) == 0) T[0] = kSlotEmpty;
  }
  return tmin;
}

}  // namespace ast

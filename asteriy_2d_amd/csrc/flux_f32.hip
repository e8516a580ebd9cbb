// flux_f32.hip -- batched FP32 face-flux operators over SoA face arrays:
// HLL, HLLC (both wave-speed estimates) and the exact solver (FP64 islands)
// of the fast path applied to
// n independent faces with a common normal (n1, n2).  52 B/face of
// algorithmic traffic (8 words in, 5 out).
#include <type_traits>

#include "common.hpp"
#include "exact_f32.hpp"
#include "fast_flux.hpp"

namespace ast {
namespace f32 {

constexpr int FNT = 256;

// E: the exact solver's constants, with gamma = 5/3 compiled in or not.
template <int METHOD, class E>
__global__ __launch_bounds__(FNT) void flux_kernel(size_t n, const float* __restrict__ in,
                                                   float n1, float n2, float krad,
                                                   ExactCtx ex0, float* __restrict__ out) {
  const E ex(ex0);
  const size_t stride = (size_t)gridDim.x * FNT;
  for (size_t i = (size_t)blockIdx.x * FNT + threadIdx.x; i < n; i += stride) {
    const float rl = in[i], pl = in[n + i], vxl = in[2 * n + i], vyl = in[3 * n + i];
    const float rr = in[4 * n + i], pr = in[5 * n + i], vxr = in[6 * n + i], vyr = in[7 * n + i];
    // face frame: normal (n1, n2), tangent (-n2, n1)
    const PrimF L = {rl, pl, vxl * n1 + vyl * n2, -vxl * n2 + vyl * n1};
    const PrimF R = {rr, pr, vxr * n1 + vyr * n2, -vxr * n2 + vyr * n1};
    float UU;
    FluxF f;
    FaceInfo fi;
    if constexpr (METHOD == AST_HLL) f = hll_f32(L, R, ex.g, ex.ig1, UU);
    else if constexpr (METHOD == AST_HLLC) f = hllc_f32<false>(L, R, ex.g, ex.ig1, UU);
    else if constexpr (METHOD == AST_HLLC_A) f = hllc_f32<true>(L, R, ex.g, ex.ig1, UU);
    else f = exact_f32<false>(L, R, ex, UU, fi);
    out[i] = f.m;
    out[n + i] = f.e;
    out[2 * n + i] = f.un * n1 - f.ut * n2;
    out[3 * n + i] = f.un * n2 + f.ut * n1;
    out[4 * n + i] = krad * frcp(UU);
  }
}

// ---- the exact solver on pattern-sorted faces ------------------------------
//
// Faces of one wave that take different wave patterns (and different
// iteration counts) run their branches one after another with most lanes
// masked.  Here each workgroup takes a tile of STILE faces, classifies them
// (pattern_key: vacuum, two rarefactions, shock + rarefaction, two shocks,
// strong two shocks, no pattern), orders the tile's faces by that key with a
// counting sort in LDS, and then solves them in that order, so that the 64
// lanes of a wave mostly hold faces of one pattern.  Results depend only on
// each face's own data: the order changes no bit.
//
// Bound: the solver's vector instructions (about 90% of issue at 2^24 faces,
// 400 a face and wave; the 52 B a face take 155 us at a copy's rate).
//
// The tile's faces are kept in LDS from the classifying (coalesced) loads on,
// swapped and with the sound speeds and the power the classes needed: the
// solve reads its permuted faces there and leaves its fluxes there, and the
// tile's fluxes go out with coalesced stores.  Measured at 2^24 faces: 345 us
// with the p* solves and a sampling per pattern of before, 200 us with
// exact_f32.hpp's, 188 us with the classes' values kept as well; re-reading
// the faces from global memory in sorted order, 32 scattered loads per lane
// and tile, took 60% of the kernel's time.
//
// With the learned newton start, a first kernel (kGuessPass) evaluates the
// network for the strong two-shock faces only -- they are contiguous after
// the sort, so its waves are full of faces that use the guess -- and leaves
// each guess in the face's dt slot of `out`; the solve kernel
// (kSolveGuessed) reads it there before it writes the dt.  The solver kernel
// thus carries no network registers, and the network's own kernel runs only
// on the faces it serves.
constexpr int SORT_NT = 256;
constexpr int SORT_PER = 2;                  // faces per thread per tile
constexpr int STILE = SORT_NT * SORT_PER;    // faces per tile
constexpr int kSolve = 0, kGuessPass = 1, kSolveGuessed = 2;

// The face's eight words (rhoL, pL, vxL, vyL, rhoR, pR, vxR, vyR) in the
// frame of the normal (n1, n2).
AST_DEV void face_frame(const float* w, float n1, float n2, PrimF& L, PrimF& R) {
  L = PrimF{w[0], w[1], w[2] * n1 + w[3] * n2, -w[2] * n2 + w[3] * n1};
  R = PrimF{w[4], w[5], w[6] * n1 + w[7] * n2, -w[6] * n2 + w[7] * n1};
}

template <bool STATS, int MODE, class E = ExactCtx>
__global__ __launch_bounds__(SORT_NT) void exact_sorted_kernel(size_t n,
                                                               const float* __restrict__ in,
                                                               float n1, float n2, float krad,
                                                               ExactCtx ex0, float* out,
                                                               ast_stats_t* stats,
                                                               int* __restrict__ info) {
  const E ex(ex0);
  constexpr bool STRONG = MODE != kSolve;  // strong faces form a group of their own
  __shared__ uint32_t redi[(SORT_NT / 64) * 10];
  // slot -> face of the tile (low bits), its key and its swap
  static_assert(STILE <= 1 << 9 && kPatternKeys < 8, "perm's fields");
  __shared__ unsigned short perm[STILE];
  __shared__ int cnt[kPatternKeys + 1], cur[kPatternKeys + 1];
  __shared__ float stage[11][STILE];  // the tile's ExactFaces, then (5 planes) its fluxes
  typename std::conditional<STATS, StatsF32, NoStats>::type st;
  st.clear();
  auto staged = [&](int li) {
    return ExactFace{stage[0][li], stage[1][li], stage[2][li], stage[3][li], stage[4][li],
                     stage[5][li], stage[6][li], stage[7][li], stage[8][li], stage[9][li],
                     stage[10][li], false};
  };
  const size_t ntiles = (n + STILE - 1) / STILE;
  for (size_t tile = blockIdx.x; tile < ntiles; tile += gridDim.x) {  // workgroup-uniform
    const size_t base = tile * STILE;
    const int nv = (int)min((size_t)STILE, n - base);
    if (threadIdx.x <= kPatternKeys) cnt[threadIdx.x] = 0;
    __syncthreads();
    // classify (coalesced loads) and count
    unsigned tag[SORT_PER];  // perm's entry
#pragma unroll
    for (int j = 0; j < SORT_PER; j++) {
      const int li = j * SORT_NT + threadIdx.x;
      unsigned key = kPatternKeys;  // past the end of the batch
      bool sw = false;
      if (li < nv) {
        float w[8];
#pragma unroll
        for (int k = 0; k < 8; k++) w[k] = in[k * n + base + li];
        PrimF L, R;
        face_frame(w, n1, n2, L, R);
        const ExactFace f = exact_sides(L, R, ex);
        const float v[11] = {f.rI, f.pI, f.enI, f.teI, f.rII, f.pII, f.enII, f.teII, f.cI, f.cII,
                             f.q};
#pragma unroll
        for (int k = 0; k < 11; k++) stage[k][li] = v[k];
        key = pattern_key<STRONG>(f, wave_pattern(f, ex));
        sw = f.sw;
      }
      tag[j] = (unsigned)li | key << 9 | (sw ? 1u << 12 : 0u);
      atomicAdd(&cnt[key], 1);
    }
    __syncthreads();
    if (threadIdx.x == 0) {
      int s = 0;
      for (int k = 0; k <= kPatternKeys; k++) {
        cur[k] = s;
        s += cnt[k];
      }
      cnt[0] = cur[4];             // first strong face
      cnt[1] = cur[5];             // one past the last strong face
      cnt[2] = cur[kPatternKeys];  // the tile's faces of the batch
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < SORT_PER; j++) {
      const int slot = atomicAdd(&cur[tag[j] >> 9 & 7], 1);
      perm[slot] = (unsigned short)tag[j];
    }
    __syncthreads();
    const int s0 = cnt[0], s1 = cnt[1], nfaces = cnt[2];
    if constexpr (MODE == kGuessPass) {
      // the network on the strong faces, whole waves of them (EXEC full)
      const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
      for (int w0 = s0 + 64 * wave; w0 < s1; w0 += SORT_NT) {  // wave-uniform
        const int li = perm[min(w0 + lane, s1 - 1)] & (STILE - 1);
        const ExactFace f = staged(li);
        float fe[mlp::IN];
        const float lp =
            mlp::features<float>(f.rI, f.pI, f.enI, f.rII, f.pII, f.enII, ex.g, fe);
        const float y = mlp::forward_wave_bf16(ex.mlp, fe);
        if (w0 + lane < s1) out[4 * n + base + li] = __expf(y + lp);
      }
    } else {
      // solve in sorted order
#pragma unroll 1
      for (int j = 0; j < SORT_PER; j++) {  // uniform
        const int pos = j * SORT_NT + threadIdx.x;
        FaceInfo fi{kNoFace, 0, false, false, false, false};
        if (pos < nfaces) {
          const unsigned tg = perm[pos];
          const int li = tg & (STILE - 1), key = tg >> 9 & 7;
          const size_t i = base + li;
          ExactFace f = staged(li);
          f.sw = (tg >> 12) != 0;
          const WavePattern wp{key == 0, key == 1, key == 2, key == 3 || key == 4};
          const float g = (MODE == kSolveGuessed && pos >= s0 && pos < s1) ? out[4 * n + i] : -1.f;
          float UU;
          const FluxF q = lab_flux(exact_solve_f32(f, wp, ex, UU, fi, g));
          // this lane alone holds face li: its words are read, its fluxes
          // take their place
          stage[0][li] = q.m;
          stage[1][li] = q.e;
          stage[2][li] = q.un * n1 - q.ut * n2;
          stage[3][li] = q.un * n2 + q.ut * n1;
          stage[4][li] = krad * frcp(UU);
          if (info) {
            info[2 * i] = fi.it;
            info[2 * i + 1] = (fi.pat == kNoPattern ? -1 : fi.pat + 1) | (fi.capped ? 8 : 0) |
                              (fi.island ? 16 : 0);
          }
        }
        st.add(fi);
      }
      __syncthreads();
      // the tile's fluxes, coalesced
#pragma unroll
      for (int j = 0; j < SORT_PER; j++) {
        const int li = j * SORT_NT + threadIdx.x;
        if (li < nv) {
#pragma unroll
          for (int k = 0; k < 5; k++) out[k * n + base + li] = stage[k][li];
        }
      }
    }
    __syncthreads();  // stage, perm and the counters are reused by the next tile
  }
  if constexpr (STATS) block_stats_f32_to<SORT_NT>(st, redi, stats);
}

template <int METHOD>
static int launch(size_t n, const float* in, float n1, float n2, float krad, const ExactCtx& ex,
                  float* out, ast_stats_t* stats, int* info, hipStream_t stream) {
  // The sort pays where the solver's instructions bound the kernel; a launch
  // that leaves the chip part idle waits for its longest chain instead, which
  // the sort and its barriers lengthen.  Measured, exact, us (face order /
  // sorted), gamma = 5/3: 50001 faces 6.1 / 6.4, 200000 6.7 / 7.6, 400000 9.1 /
  // 10.3, 1000001 17.4 / 18.0, 1200001 19.9 / 20.9, 2000003 29.3 / 28.9, 2^24
  // 220 / 207; gamma = 7/5: 50001 6.1 / 7.4, 1000001 18.9 / 20.0, 2000003 31.3 /
  // 31.7, 2^24 230 / 220.
  const bool plain = METHOD != AST_EXACT ||
                     (n <= (size_t(1) << 20) && ex.mlp == nullptr && !stats && !info);
  if (plain) {
    size_t blocks = (n + FNT - 1) / FNT;
    if (blocks > 256 * 64) blocks = 256 * 64;
    const auto kernel = METHOD == AST_EXACT && ex.n == 5 ? flux_kernel<METHOD, ExactCtx5>
                                                         : flux_kernel<METHOD, ExactCtx>;
    hipLaunchKernelGGL(kernel, dim3((unsigned)blocks), dim3(FNT), 0, stream, n, in, n1, n2, krad,
                       ex, out);
    AST_LAUNCH_CHECK("ast_flux_f32 launch");
    return AST_OK;
  }
  if constexpr (METHOD == AST_EXACT) {
    // one tile per workgroup (measured on 2^24 faces, before the solver's
    // present form: 512-face tiles, one per workgroup, 346 us; 1024-face tiles
    // 367-403 us; 4096 workgroups looping over the tiles 389-427 us), a loop
    // over tiles beyond 2^20 workgroups
    size_t blocks = (n + STILE - 1) / STILE;
    if (blocks > (size_t(1) << 20)) blocks = size_t(1) << 20;
    const dim3 gr((unsigned)blocks), bl(SORT_NT);
    const bool st = stats != nullptr;
    if (ex.mlp != nullptr) {
      hipLaunchKernelGGL((exact_sorted_kernel<false, kGuessPass>), gr, bl, 0, stream, n, in, n1,
                         n2, krad, ex, out, nullptr, nullptr);
      AST_LAUNCH_CHECK("ast_flux_f32 guess launch");
      if (st)
        hipLaunchKernelGGL((exact_sorted_kernel<true, kSolveGuessed>), gr, bl, 0, stream, n, in,
                           n1, n2, krad, ex, out, stats, info);
      else
        hipLaunchKernelGGL((exact_sorted_kernel<false, kSolveGuessed>), gr, bl, 0, stream, n, in,
                           n1, n2, krad, ex, out, stats, info);
    } else if (st) {
      hipLaunchKernelGGL((exact_sorted_kernel<true, kSolve>), gr, bl, 0, stream, n, in, n1, n2,
                         krad, ex, out, stats, info);
    } else if (ex.n == 5) {
      hipLaunchKernelGGL((exact_sorted_kernel<false, kSolve, ExactCtx5>), gr, bl, 0, stream, n, in,
                         n1, n2, krad, ex, out, stats, info);
    } else {
      hipLaunchKernelGGL((exact_sorted_kernel<false, kSolve>), gr, bl, 0, stream, n, in, n1, n2,
                         krad, ex, out, stats, info);
    }
    AST_LAUNCH_CHECK("ast_flux_f32 launch");
  }
  return AST_OK;
}

}  // namespace f32
}  // namespace ast

extern "C" int ast_flux_f32_info(int method, size_t n, const float* in, float n1, float n2,
                                 float rad, float gamma, float krit, const ast_mlp_t* mlp,
                                 float* out, ast_stats_t* stats, int* info, void* stream) {
  using namespace ast::f32;
  if (n == 0) return AST_OK;
  if (!in || !out) return ast_fail(AST_ERR_ARG, "ast_flux_f32: null in/out");
  if (!(gamma > 1.0f)) return ast_fail(AST_ERR_ARG, "ast_flux_f32: gamma must be > 1");
  const ast::ExactCtx ex = ast::make_exact_ctx((double)gamma, mlp);
  const float krad = krit * rad;
  hipStream_t st = (hipStream_t)stream;
  switch (method) {
    case AST_HLL: return launch<AST_HLL>(n, in, n1, n2, krad, ex, out, stats, nullptr, st);
    case AST_HLLC: return launch<AST_HLLC>(n, in, n1, n2, krad, ex, out, stats, nullptr, st);
    case AST_EXACT: return launch<AST_EXACT>(n, in, n1, n2, krad, ex, out, stats, info, st);
    case AST_HLLC_A: return launch<AST_HLLC_A>(n, in, n1, n2, krad, ex, out, stats, nullptr, st);
    default: return ast_fail(AST_ERR_ARG, "ast_flux_f32: unknown method %d", method);
  }
}

extern "C" int ast_flux_f32(int method, size_t n, const float* in, float n1, float n2, float rad,
                            float gamma, float krit, float* out, ast_stats_t* stats,
                            void* stream) {
  return ast_flux_f32_info(method, n, in, n1, n2, rad, gamma, krit, nullptr, out, stats, nullptr,
                           stream);
}

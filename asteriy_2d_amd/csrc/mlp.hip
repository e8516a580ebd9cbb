// mlp.hip -- training and inference kernels of the learned p* guess.
//
//  * features: the solver's own face log.  For each face of a batch the FP64
//    exact solver's classification and newton (kernel.cu:200-231, 635-680)
//    run at the reference tolerance; two-shock faces get mask 1 and the
//    target log(p*/p_ref).
//  * forward: FP32 masters on the vector ALU (one sample per lane), or the
//    BF16 MFMA path (one 64-sample tile per wave, mlp.hpp).
//  * loss + gradient: mean squared error over the masked rows, forward and
//    backward on FP32 MFMA, per-workgroup partials summed in a fixed order by
//    a second kernel (deterministic).
//  * Adam on the FP32 masters, the BF16 MFMA operands rebuilt with it.
#include "common.hpp"
#include "flux64.hpp"
#include "mlp.hpp"

namespace ast {
namespace mlp {

// ---- features from the FP64 exact solve ---------------------------------
__global__ void features_kernel(size_t n, const double* __restrict__ in, double n1, double n2,
                                d64::GasD gas, float* __restrict__ feats,
                                float* __restrict__ target, unsigned char* __restrict__ mask) {
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (size_t)gridDim.x * blockDim.x) {
    const double rL = in[i], pL = in[n + i], uL = in[2 * n + i] * n1 + in[3 * n + i] * n2;
    const double rR = in[4 * n + i], pR = in[5 * n + i],
                 uR = in[6 * n + i] * n1 + in[7 * n + i] * n2;
    // post-swap states, kernel.cu:156-184
    const bool sw = pL > pR;
    const double enI = sw ? -uR : uL, enII = sw ? -uL : uR;
    const double pI = sw ? pR : pL, pII = sw ? pL : pR, rI = sw ? rR : rL, rII = sw ? rL : rR;
    float f[IN];
    const float lp = features<double>(rI, pI, enI, rII, pII, enII, gas.g, f);
    for (int k = 0; k < IN; k++) feats[k * n + i] = f[k];
    // two shocks when the closing speed exceeds f_I(p_II) (kernel.cu:200-231)
    const double du = enI - enII;
    const bool two_shock = du > (pII - pI) / sqrt(0.5 * rI * (gas.g2 * pII + gas.g1 * pI));
    if (mask) mask[i] = two_shock ? 1 : 0;
    if (target) {
      float t = 0.f;
      if (two_shock) {
        int it;
        bool capped = false;
        const double zI = rI * sqrt(gas.g * pI / rI), zII = rII * sqrt(gas.g * pII / rII);
        const double p =
            d64::two_shock_root(gas, du, pI, rI, zI, pII, rII, zII, -1.0, false, it, capped);
        t = (float)(log(p) - (double)lp);
      }
      target[i] = t;
    }
  }
}

// ---- forward ----------------------------------------------------------------
__global__ void forward_f32_kernel(const float* __restrict__ P, size_t n,
                                   const float* __restrict__ feats, float* __restrict__ pred) {
  __shared__ float Ps[NP];
  for (int k = threadIdx.x; k < NP; k += blockDim.x) Ps[k] = P[k];
  __syncthreads();
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (size_t)gridDim.x * blockDim.x) {
    float x[IN];
    for (int k = 0; k < IN; k++) x[k] = feats[k * n + i];
    pred[i] = forward_f32(Ps, x);
  }
}

// every wave walks whole 64-sample tiles (EXEC stays full for the MFMAs);
// lanes past n compute on clamped rows and do not store
__global__ void forward_bf16_kernel(const unsigned char* __restrict__ buf, size_t n,
                                    const float* __restrict__ feats, float* __restrict__ pred) {
  const size_t waves = (size_t)gridDim.x * (blockDim.x / 64);
  const size_t w0 = (size_t)blockIdx.x * (blockDim.x / 64) + (threadIdx.x >> 6);
  const size_t tiles = (n + 63) / 64;
  for (size_t t = w0; t < tiles; t += waves) {
    const size_t i = t * 64 + (threadIdx.x & 63);
    const size_t ic = i < n ? i : n - 1;
    float x[IN];
    for (int k = 0; k < IN; k++) x[k] = feats[k * n + ic];
    const float y = forward_wave_bf16(buf, x);
    if (i < n) pred[i] = y;
  }
}

// ---- loss and gradient -----------------------------------------------------
//
// Every product of the network runs on FP32 MFMA (FP32 operands, products
// and accumulation).  A wave takes 16 samples at a time in the transposed
// form of mlp.hpp, H_out^T = W H_in^T, on v_mfma_f32_16x16x4: lane (q, j) of
// the accumulators holds the units 4q..4q+3 and 16+4q..16+4q+3 (slot_unit)
// of sample j, which is the B operand of the next product as it stands when
// that product's k index runs over the units in the same order -- forward
// (W) and backward (W^T) alike, so activations and deltas never move between
// lanes.  The weight gradients contract over samples instead,
// dW[a][k] = sum_s g[s][a] h[s][k], so deltas and activations pass through a
// wave-private LDS tile once and accumulate on v_mfma_f32_32x32x2.
//
// About 13 kflop a sample, bound by the FP32 MFMA issue (3456 cycles a block)
// and, at the training batch of 65536 samples, by the start and the end of
// the waves, which take two blocks each: 20 us with a trace on (78 us with
// products on the vector ALU and weight gradients that each re-read 128
// samples from LDS), 9.9 us more for every 65536 samples beyond.
constexpr int GWAVES = 8;            // waves of a workgroup (two a SIMD)
constexpr int GNT = 64 * GWAVES;
constexpr int GBLOCKS = 256;         // most workgroups: partial gradients to reduce
constexpr int PW = NP + 2;           // partial: gradient, loss sum, row count
constexpr int TS = 36;               // row stride of the LDS tiles (16 samples x 32 units)

typedef float f32x16 __attribute__((ext_vector_type(16)));

// v of lane l + the DPP row shifts' sums: lane 15 of each 16-lane row ends
// with the row's sum
AST_DEV float row_sum15(float v) {
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x111, 0xf, 0xf, true));
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x112, 0xf, 0xf, true));
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x114, 0xf, 0xf, true));
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x118, 0xf, 0xf, true));
  return v;
}

// orders a wave's LDS accesses before and after it (one wave's run in order)
AST_DEV void wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// the two 16-unit tiles of W x (A: 8 k-steps a tile; B: a unit vector in
// slot order), added to c
AST_DEV void product32(const float* A, const float* B, f32x4* c) {
#pragma unroll
  for (int k = 0; k < 8; k++) {
    c[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(A[k], B[k], c[0], 0, 0, 0);
    c[1] = __builtin_amdgcn_mfma_f32_16x16x4f32(A[8 + k], B[k], c[1], 0, 0, 0);
  }
}

__global__ __launch_bounds__(GNT, 2) void grad_kernel(const float* __restrict__ P, size_t n,
                                                      const float* __restrict__ feats,
                                                      const float* __restrict__ target,
                                                      const unsigned char* __restrict__ mask,
                                                      float* __restrict__ partial) {
  // the waves' tiles (deltas, activations), then four partial gradients
  constexpr int kTileFloats = 2 * 16 * TS;
  constexpr int kShared = GWAVES * kTileFloats > 4 * PW ? GWAVES * kTileFloats : 4 * PW;
  __shared__ __align__(16) float sh[kShared];
  // W1, the biases and w4, read from here where they are used
  constexpr int vB2 = oW2, vB3 = vB2 + H, vW4 = vB3 + H;
  __shared__ __align__(16) float vec[vW4 + H];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, q = lane >> 4, j = lane & 15;
  float* tg = sh + wave * kTileFloats;
  float* th = tg + 16 * TS;
  // operands: A[8 t + k] = row 16 t + j of the matrix, unit slot_unit(8 q + k),
  // gathered from an LDS copy of the masters whose rows are padded to 33
  constexpr int HP = H + 1, kW2 = 0, kW3 = kW2 + H * HP;
  static_assert(kW3 + H * HP <= kShared, "staged masters fit the tiles' space");
  // a block's inputs, fetched a block ahead: the features of sample s0 + j
  // for layer 1 (x0, x1), those of dW1's B operand (lane (q, j): feature j of
  // sample s0 + 4 k + q, and a column of ones that sums db1), the target
  const size_t blocks = (n + 15) / 16;
  const size_t first = (size_t)blockIdx.x * GWAVES + wave, stride = (size_t)gridDim.x * GWAVES;
  float x0 = 0.f, x1 = 0.f, xb[4] = {0.f, 0.f, 0.f, 0.f}, tv = 0.f;
  bool valid = false;
  auto fetch = [&](size_t blk) {
    const size_t s0 = blk * 16, s = s0 + j, sc = s < n ? s : n - 1;
    valid = s < n && (mask == nullptr || mask[s]);
    x0 = feats[(size_t)q * n + sc];
    x1 = q < IN - 4 ? feats[(size_t)(4 + q) * n + sc] : 0.f;
#pragma unroll
    for (int k = 0; k < 4; k++) {
      const size_t ss = s0 + 4 * k + q;
      xb[k] = j < IN ? feats[(size_t)j * n + (ss < n ? ss : n - 1)] : (j == IN ? 1.f : 0.f);
    }
    tv = target[sc];
  };
  if (first < blocks) fetch(first);
  float A2[16], A3[16], A2t[16], A3t[16];
  for (int p = threadIdx.x; p < vW4 + H; p += GNT)
    vec[p] = P[p < vB2 ? p : p < vB3 ? oB2 + (p - vB2) : p < vW4 ? oB3 + (p - vB3) : oW4 + (p - vW4)];
  for (int p = threadIdx.x; p < H * H; p += GNT) {
    sh[kW2 + (p >> 5) * HP + (p & 31)] = P[oW2 + p];
    sh[kW3 + (p >> 5) * HP + (p & 31)] = P[oW3 + p];
  }
  __syncthreads();
#pragma unroll
  for (int t = 0; t < 2; t++) {
#pragma unroll
    for (int k = 0; k < 8; k++) {
      const int u = slot_unit(8 * q + k), r = 16 * t + j;
      A2[8 * t + k] = sh[kW2 + r * HP + u];
      A3[8 * t + k] = sh[kW3 + r * HP + u];
      A2t[8 * t + k] = sh[kW2 + u * HP + r];
      A3t[8 * t + k] = sh[kW3 + u * HP + r];
    }
  }
  __syncthreads();
  const float b4 = P[oB4];
  auto units = [&](int off, f32x4* c) {  // a unit vector of vec, in slot order
    c[0] = *reinterpret_cast<const f32x4*>(vec + off + 4 * q);
    c[1] = *reinterpret_cast<const f32x4*>(vec + off + 16 + 4 * q);
  };
  f32x16 dW3 = {0.f}, dW2 = {0.f};
  f32x4 dW1[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
  float s3[8], s2[8], s4[8], sb4 = 0.f, lsum = 0.f, cnt = 0.f;
#pragma unroll
  for (int k = 0; k < 8; k++) s3[k] = s2[k] = s4[k] = 0.f;

  for (size_t blk = first; blk < blocks; blk += stride) {  // wave-uniform: EXEC stays full
    f32x4 c[2];
    float h1[8], h2[8], h3[8], g[8];
    units(oB1, c);
#pragma unroll
    for (int t = 0; t < 2; t++) {
      const float* r = vec + oW1 + (16 * t + j) * IN;
      c[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(r[q], x0, c[t], 0, 0, 0);
      c[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(q < IN - 4 ? r[4 + q] : 0.f, x1, c[t], 0, 0, 0);
    }
#pragma unroll
    for (int k = 0; k < 8; k++) h1[k] = tanh_f(c[k >> 2][k & 3]);
    units(vB2, c);
    product32(A2, h1, c);
#pragma unroll
    for (int k = 0; k < 8; k++) h2[k] = tanh_f(c[k >> 2][k & 3]);
    units(vB3, c);
    product32(A3, h2, c);
    float y = 0.f;
    f32x4 w4[2];
    units(vW4, w4);
#pragma unroll
    for (int k = 0; k < 8; k++) {
      h3[k] = tanh_f(c[k >> 2][k & 3]);
      y += w4[k >> 2][k & 3] * h3[k];
    }
    y += __shfl_xor(y, 16, 64);
    y += __shfl_xor(y, 32, 64);
    y += b4;
    const float e = valid ? y - tv : 0.f;
    if (q == 0) {
      lsum += e * e;
      cnt += valid ? 1.f : 0.f;
    }
    const float dy = 2.f * e;  // d(e^2)/dy; the mean is taken in the reduction
    if (q == 0) sb4 += dy;
    float xw[4];
#pragma unroll
    for (int k = 0; k < 4; k++) xw[k] = xb[k];
    if (blk + stride < blocks) fetch(blk + stride);
    // dW = sum over the block's samples of (the tile tg)^T th
    auto contract = [&](f32x16& dW) {
      const int half = lane >> 5, col = lane & 31;
#pragma unroll
      for (int k = 0; k < 8; k++)
        dW = __builtin_amdgcn_mfma_f32_32x32x2f32(tg[(2 * k + half) * TS + col],
                                                  th[(2 * k + half) * TS + col], dW, 0, 0, 0);
    };
    auto put = [&](float* T, const float* v) {  // sample j, units 4q.. and 16+4q..
      *reinterpret_cast<f32x4*>(T + j * TS + 4 * q) = f32x4{v[0], v[1], v[2], v[3]};
      *reinterpret_cast<f32x4*>(T + j * TS + 16 + 4 * q) = f32x4{v[4], v[5], v[6], v[7]};
    };
    // layer-3 deltas
#pragma unroll
    for (int k = 0; k < 8; k++) {
      s4[k] += dy * h3[k];
      g[k] = dy * w4[k >> 2][k & 3] * (1.f - h3[k] * h3[k]);
      s3[k] += g[k];
    }
    put(tg, g);
    put(th, h2);
    wave_lds_fence();
    contract(dW3);
    // layer-2 deltas: (W3^T g3) (1 - h2^2)
    c[0] = c[1] = f32x4{0.f, 0.f, 0.f, 0.f};
    product32(A3t, g, c);
#pragma unroll
    for (int k = 0; k < 8; k++) {
      g[k] = c[k >> 2][k & 3] * (1.f - h2[k] * h2[k]);
      s2[k] += g[k];
    }
    wave_lds_fence();
    put(tg, g);
    put(th, h1);
    wave_lds_fence();
    contract(dW2);
    // layer-1 deltas: (W2^T g2) (1 - h1^2)
    c[0] = c[1] = f32x4{0.f, 0.f, 0.f, 0.f};
    product32(A2t, g, c);
#pragma unroll
    for (int k = 0; k < 8; k++) g[k] = c[k >> 2][k & 3] * (1.f - h1[k] * h1[k]);
    wave_lds_fence();
    put(tg, g);
    wave_lds_fence();
#pragma unroll
    for (int t = 0; t < 2; t++)
#pragma unroll
      for (int k = 0; k < 4; k++)
        dW1[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(tg[(4 * k + q) * TS + 16 * t + j], xw[k],
                                                      dW1[t], 0, 0, 0);
    wave_lds_fence();
  }

  // this workgroup's partial gradient: four waves leave theirs in LDS, the
  // others add theirs, and the four are summed in order
  lsum = row_sum15(lsum);
  cnt = row_sum15(cnt);
  sb4 = row_sum15(sb4);
#pragma unroll
  for (int k = 0; k < 8; k++) {
    s3[k] = row_sum15(s3[k]);
    s2[k] = row_sum15(s2[k]);
    s4[k] = row_sum15(s4[k]);
  }
  float* R = sh + (wave & 3) * PW;
  auto leave = [&](bool add) {
    auto at = [&](int p, float v) { R[p] = add ? R[p] + v : v; };
#pragma unroll
    for (int r = 0; r < 16; r++) {
      const int row = 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3), col = lane & 31;
      at(oW3 + row * H + col, dW3[r]);
      at(oW2 + row * H + col, dW2[r]);
    }
#pragma unroll
    for (int t = 0; t < 2; t++)
#pragma unroll
      for (int v = 0; v < 4; v++) {
        const int row = 16 * t + 4 * q + v;
        if (j < IN) at(oW1 + row * IN + j, dW1[t][v]);
        else if (j == IN) at(oB1 + row, dW1[t][v]);
      }
    if (j == 15) {
#pragma unroll
      for (int k = 0; k < 8; k++) {
        const int u = slot_unit(8 * q + k);
        at(oB3 + u, s3[k]);
        at(oB2 + u, s2[k]);
        at(oW4 + u, s4[k]);
      }
      if (q == 0) {
        at(oB4, sb4);
        at(NP, lsum);
        at(NP + 1, cnt);
      }
    }
  };
  __syncthreads();
  if (wave >= 4) leave(false);
  __syncthreads();
  if (wave < 4) leave(true);
  __syncthreads();
  float* out = partial + (size_t)blockIdx.x * PW;
  for (int p = threadIdx.x; p < PW; p += GNT)
    out[p] = (sh[p] + sh[PW + p]) + (sh[2 * PW + p] + sh[3 * PW + p]);
}

// Sums the workgroups' partials in a fixed order; grad = sum / count, loss =
// mean.  A workgroup takes RCOLS entries, each summed by RSLICES threads over
// every RSLICES-th partial (75 workgroups; one thread an entry over all
// partials, 10 workgroups, took 114 us of latency for 256 of them).
constexpr int RCOLS = 32, RSLICES = 16, RNT = RCOLS * RSLICES;

__global__ __launch_bounds__(RNT) void grad_reduce_kernel(const float* __restrict__ partial,
                                                          int nblocks, float* __restrict__ grad,
                                                          float* __restrict__ loss) {
  __shared__ float part[RSLICES][RCOLS], cpart[RNT];
  const int col = threadIdx.x % RCOLS, slice = threadIdx.x / RCOLS;
  const int k = blockIdx.x * RCOLS + col;
  float s = 0.f, cnt = 0.f;
  if (k < NP + 1) {
#pragma unroll 8
    for (int b = slice; b < nblocks; b += RSLICES) s += partial[(size_t)b * PW + k];
  }
  for (int b = threadIdx.x; b < nblocks; b += RNT) cnt += partial[(size_t)b * PW + NP + 1];
  part[slice][col] = s;
  cpart[threadIdx.x] = cnt;
  __syncthreads();
  for (int w = RNT / 2; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) cpart[threadIdx.x] += cpart[threadIdx.x + w];
    __syncthreads();
  }
  if (slice == 0 && k < NP + 1) {
    float t = part[0][col];
#pragma unroll
    for (int i = 1; i < RSLICES; i++) t += part[i][col];
    const float inv = cpart[0] > 0.f ? 1.f / cpart[0] : 0.f;
    if (k < NP) grad[k] = t * inv;
    else if (loss) *loss = t * inv;
  }
}

// The master parameter behind element v of lane `lane` of MFMA operand `op`
// (-1: none, the element is zero).  No two elements share a parameter.
AST_DEV int operand_param(int op, int lane, int v) {
  const int i = lane & 15, s = 8 * (lane >> 4) + v;
  if (op < 2) return s < IN ? oW1 + (op * 16 + i) * IN + s : -1;  // layer 1: feature slots 0..5
  if (op < 6) {  // layers 2, 3: permuted hidden slots
    const int off = op < 4 ? oW2 : oW3, mb = (op - 2) % 2;
    return off + (mb * 16 + i) * H + slot_unit(s);
  }
  return i == 0 ? oW4 + slot_unit(s) : -1;  // output: row 0 = w4
}
constexpr int OPELEMS = OPS * 64 * 8;

// rebuilds the BF16 MFMA operands from the FP32 masters
__global__ void refresh_bf16_kernel(unsigned char* buf) {
  const float* P = (const float*)buf;
  __bf16* A = (__bf16*)(buf + BF_OFF);
  for (int e = blockIdx.x * blockDim.x + threadIdx.x; e < OPELEMS; e += gridDim.x * blockDim.x) {
    const int k = operand_param(e >> 9, (e >> 3) & 63, e & 7);
    A[e] = (__bf16)(k >= 0 ? P[k] : 0.f);
  }
}

// One Adam step on the masters and the rebuilt MFMA operands in one kernel:
// thread e < OPELEMS owns operand element e and the parameter behind it, the
// threads after them the biases, which have no operand.
__global__ void adam_kernel(unsigned char* buf, const float* __restrict__ g,
                            float* __restrict__ st, int step, float lr) {
  float* P = (float*)buf;
  __bf16* A = (__bf16*)(buf + BF_OFF);
  const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
  const float c1 = 1.f - powf(b1, (float)step), c2 = 1.f - powf(b2, (float)step);
  auto update = [&](int k) {
    float m = st[k], v = st[NP + k];
    m = b1 * m + (1.f - b1) * g[k];
    v = b2 * v + (1.f - b2) * g[k] * g[k];
    st[k] = m;
    st[NP + k] = v;
    const float p = P[k] - lr * (m / c1) / (sqrtf(v / c2) + eps);
    P[k] = p;
    return p;
  };
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e < OPELEMS) {
    const int k = operand_param(e >> 9, (e >> 3) & 63, e & 7);
    A[e] = (__bf16)(k >= 0 ? update(k) : 0.f);
  } else {
    const int b = e - OPELEMS;
    if (b < 3 * H) update((b < H ? oB1 : b < 2 * H ? oB2 : oB3) + b % H);
    else if (b == 3 * H) update(oB4);
  }
}
constexpr int ADAM_THREADS = OPELEMS + 3 * H + 1;

}  // namespace mlp
}  // namespace ast

using namespace ast;
using namespace ast::mlp;

extern "C" size_t ast_mlp_bytes(void) { return (size_t)BYTES; }
extern "C" size_t ast_mlp_work_floats(void) { return (size_t)GBLOCKS * PW; }

extern "C" int ast_mlp_features(size_t n, const double* in, double n1, double n2, double gamma,
                                float* feats, float* target, unsigned char* mask, void* stream) {
  if (n == 0) return AST_OK;
  if (!in || !feats) return ast_fail(AST_ERR_ARG, "ast_mlp_features: null pointer");
  if (!(gamma > 1.0)) return ast_fail(AST_ERR_ARG, "ast_mlp_features: gamma must be > 1");
  const d64::GasD gas = d64::make_gas(gamma);
  size_t blocks = (n + 255) / 256;
  if (blocks > 16384) blocks = 16384;
  hipLaunchKernelGGL(features_kernel, dim3((unsigned)blocks), dim3(256), 0, (hipStream_t)stream, n,
                     in, n1, n2, gas, feats, target, mask);
  AST_LAUNCH_CHECK("ast_mlp_features launch");
  return AST_OK;
}

extern "C" int ast_mlp_forward(const ast_mlp_t* mlp, size_t n, const float* feats, float* pred,
                               int precision, void* stream) {
  if (n == 0) return AST_OK;
  if (!mlp || !feats || !pred) return ast_fail(AST_ERR_ARG, "ast_mlp_forward: null pointer");
  hipStream_t st = (hipStream_t)stream;
  if (precision == 0) {
    size_t blocks = (n + 255) / 256;
    if (blocks > 4096) blocks = 4096;
    hipLaunchKernelGGL(forward_f32_kernel, dim3((unsigned)blocks), dim3(256), 0, st,
                       (const float*)mlp, n, feats, pred);
  } else if (precision == 1) {
    size_t tiles = (n + 63) / 64, blocks = (tiles + 3) / 4;
    if (blocks > 4096) blocks = 4096;
    hipLaunchKernelGGL(forward_bf16_kernel, dim3((unsigned)blocks), dim3(256), 0, st,
                       (const unsigned char*)mlp, n, feats, pred);
  } else {
    return ast_fail(AST_ERR_ARG, "ast_mlp_forward: precision %d (0 FP32, 1 BF16 MFMA)", precision);
  }
  AST_LAUNCH_CHECK("ast_mlp_forward launch");
  return AST_OK;
}

extern "C" int ast_mlp_loss_grad(const ast_mlp_t* mlp, size_t n, const float* feats,
                                 const float* target, const unsigned char* mask, float* grad,
                                 float* loss, float* work, void* stream) {
  if (!mlp || !feats || !target || !grad || !work)
    return ast_fail(AST_ERR_ARG, "ast_mlp_loss_grad: null pointer");
  hipStream_t st = (hipStream_t)stream;
  const size_t groups = (n + 16 * GWAVES - 1) / (16 * GWAVES);
  const int wgs = groups < 1 ? 1 : groups > GBLOCKS ? GBLOCKS : (int)groups;
  hipLaunchKernelGGL(grad_kernel, dim3(wgs), dim3(GNT), 0, st, (const float*)mlp, n, feats, target,
                     mask, work);
  AST_LAUNCH_CHECK("ast_mlp_loss_grad launch");
  hipLaunchKernelGGL(grad_reduce_kernel, dim3((NP + RCOLS) / RCOLS), dim3(RNT), 0, st, work, wgs,
                     grad, loss);
  AST_LAUNCH_CHECK("ast_mlp_loss_grad reduce");
  return AST_OK;
}

extern "C" int ast_mlp_refresh(ast_mlp_t* mlp, void* stream) {
  if (!mlp) return ast_fail(AST_ERR_ARG, "ast_mlp_refresh: null pointer");
  hipLaunchKernelGGL(refresh_bf16_kernel, dim3((OPELEMS + 255) / 256), dim3(256), 0,
                     (hipStream_t)stream, (unsigned char*)mlp);
  AST_LAUNCH_CHECK("ast_mlp_refresh launch");
  return AST_OK;
}

extern "C" int ast_mlp_adam(ast_mlp_t* mlp, const float* grad, float* state, int step, float lr,
                            void* stream) {
  if (!mlp || !grad || !state || step < 1) return ast_fail(AST_ERR_ARG, "ast_mlp_adam: bad argument");
  hipLaunchKernelGGL(adam_kernel, dim3((ADAM_THREADS + 255) / 256), dim3(256), 0,
                     (hipStream_t)stream, (unsigned char*)mlp, grad, state, step, lr);
  AST_LAUNCH_CHECK("ast_mlp_adam launch");
  return AST_OK;
}

extern "C" int ast_mlp_set_params(ast_mlp_t* mlp, const float* host_params, void* stream) {
  if (!mlp || !host_params) return ast_fail(AST_ERR_ARG, "ast_mlp_set_params: null pointer");
  hipStream_t st = (hipStream_t)stream;
  AST_HIP_CHECK(hipMemcpyAsync(mlp, host_params, NP * sizeof(float), hipMemcpyHostToDevice, st));
  int rc = ast_mlp_refresh(mlp, stream);
  if (rc != AST_OK) return rc;
  AST_HIP_CHECK(hipStreamSynchronize(st));
  return AST_OK;
}

extern "C" int ast_mlp_get_params(const ast_mlp_t* mlp, float* host_params, void* stream) {
  if (!mlp || !host_params) return ast_fail(AST_ERR_ARG, "ast_mlp_get_params: null pointer");
  hipStream_t st = (hipStream_t)stream;
  AST_HIP_CHECK(hipMemcpyAsync(host_params, mlp, NP * sizeof(float), hipMemcpyDeviceToHost, st));
  AST_HIP_CHECK(hipStreamSynchronize(st));
  return AST_OK;
}

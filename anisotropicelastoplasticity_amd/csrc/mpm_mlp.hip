// mpm_mlp.hip -- the learned Drucker-Prager return-map surrogate: a 5 -> 128 -> 128 -> 128 -> 128 -> 3
// MLP with SiLU, BF16 weights and activations and FP32 accumulation, evaluated and trained with
// v_mfma_f32_16x16x32_bf16 (CDNA4).
//
// Network input (one row per particle): the trial Hencky principal strains eps_1 >= eps_2 >= eps_3,
// the friction angle phi (degrees) and the ratio of bulk to shear modulus K/mu, normalised as
//   x = (eps / EPS_SCALE, (phi - PHI_MID) / PHI_SPAN, (K/mu - KMU_MID) / KMU_SPAN).
// Output: the plastic correction y = (H - eps) / CORR_SCALE of the projected strains H.
// The exact return map (HybridSolver.cpp:646-673) produces the training pairs and remains the
// fallback whenever the prediction fails the yield-residual gate.
//
// Layout. Layer l has weights W_l stored [N_l][K_l] (out x in, row-major) and bias b_l; the padded
// shapes are N = (128,128,128,128,16), K = (32,128,128,128,128): input columns 5..31 and output
// rows 3..15 are zero and stay zero (their gradients are masked). FP32 master weights live in one
// flat vector; the BF16 copies are regenerated after every optimiser step.
//
// MFMA lane layout (16x16x32 bf16): lane i holds A[i%16][8*(i/16) .. +8] and B[8*(i/16) .. +8][i%16];
// the 16x16 FP32 result gives lane i the rows 4*(i/16) .. +4 of column i%16.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "mpm_mlp_device.hpp"

namespace mpm {

// ------------------------------------------------------------------ batch forward (inference / training)
// in: n x 5 raw inputs (row-major), out: n x 3 normalised outputs; zsave (optional): per 16-row block b,
// 4 x 16 x 128 FP32 pre-activations at zsave + b * 4 * 16 * 128. Each wave evaluates 64 rows.
__global__ __launch_bounds__(MLP_FWD_THREADS) void k_mlp_forward(const uint16_t* __restrict__ wbf,
                                                                 const float* __restrict__ master,
                                                                 const float* __restrict__ in, float* __restrict__ out,
                                                                 int n, float* __restrict__ zsave) {
  extern __shared__ __align__(16) unsigned char smem[];
  MLPShared& s = *reinterpret_cast<MLPShared*>(smem);
  stage_weights(s, wbf, master);
  __syncthreads();
  const int nw = blockDim.x >> 6, w = threadIdx.x >> 6, lane = threadIdx.x & 63;
  for (int g = blockIdx.x * nw + w; (int64_t)g * 64 < n; g += gridDim.x * nw) {
    const int64_t r = (int64_t)g * 64 + lane;
    float x[5] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
    if (r < n)
      for (int c = 0; c < 5; ++c) x[c] = in[r * 5 + c];
    float y[3];
    wave_forward64<MLP_FWD_TILES>(s, x, y, zsave, (int64_t)g * 64, n);
    if (r < n)
      for (int c = 0; c < 3; ++c) out[r * 3 + c] = y[c];
  }
}

// ------------------------------------------------------------------ forward of a small batch
// The same network for few rows (a training or gradient batch). k_mlp_forward copies all weights
// (121 KB) into the LDS of every workgroup and gives a wave 64 rows, so 4096 rows keep 6 of the 256
// CUs busy. Here a workgroup of 8 waves takes 32 rows and wave w the 16 output features 16 w .. 16 w + 15
// of every layer: a wave reads only its own weight rows, once, straight into registers (all layers'
// loads are issued before the first product), and the activations pass through LDS in the operand
// order of the next layer (the slot order of MLPShared). Every product has the operands, the K order
// and the rounding of k_mlp_forward, so the results are the same bits. What bounds it is the chain of
// five layers, each LDS read -> MFMA -> SiLU -> LDS write -> barrier.
// Measured on MI355X at 4096 rows: 15 us, against 32 us alone and 53 us behind an Adam step for
// k_mlp_forward.
constexpr int SMALL_PER_CU = 2;                      // small-batch workgroups per CU up to which it is used
constexpr int SMALL_ROWS = 32;                       // rows per workgroup
constexpr int SMALL_THREADS = 64 * MLP_HIDDEN / 16;  // one wave per output tile

__global__ __launch_bounds__(SMALL_THREADS) void k_mlp_forward_small(const uint16_t* __restrict__ wbf,
                                                                     const float* __restrict__ master,
                                                                     const float* __restrict__ in, float* __restrict__ out,
                                                                     int n, float* __restrict__ zsave) {
  constexpr int NT = SMALL_ROWS / 16;
  __shared__ __align__(16) uint16_t s_act[2][SMALL_ROWS][LDW_H];
  const int w = (int)threadIdx.x >> 6, lane = (int)threadIdx.x & 63, c = lane & 15, q = lane >> 4;
  const int64_t row0 = (int64_t)blockIdx.x * SMALL_ROWS;
  auto frag = [&](const uint16_t* rows, int K, int s) {  // 8 inputs of output feature row `rows` in slot order
    const uint2 lo = *reinterpret_cast<const uint2*>(rows + K * c + 32 * s + 4 * q);
    const uint2 hi = *reinterpret_cast<const uint2*>(rows + K * c + 32 * s + 16 + 4 * q);
    return __builtin_bit_cast(bf16x8, make_uint4(lo.x, lo.y, hi.x, hi.y));
  };
  float v[NT][5];  // (rows past n repeat the last one and are not stored)
#pragma unroll
  for (int T = 0; T < NT; ++T) {
    const int64_t r = min(row0 + 16 * T + c, (int64_t)n - 1);
#pragma unroll
    for (int k = 0; k < 5; ++k) v[T][k] = in[r * 5 + k];
  }
  asm volatile("" ::: "memory");  // the inputs are loaded first, then the weights in layer order
  bf16x8 a1 = frag(wbf + MLP_BF_W1 + 16 * w * MLP_IN_PAD, MLP_IN_PAD, 0), ah[3][4], a5[4];
  f32x4 bias[4], bias5;
#pragma unroll
  for (int l = 0; l < 3; ++l)
#pragma unroll
    for (int s = 0; s < 4; ++s)
      ah[l][s] = frag(wbf + MLP_BF_WH + l * MLP_HIDDEN * MLP_HIDDEN + 16 * w * MLP_HIDDEN, MLP_HIDDEN, s);
#pragma unroll
  for (int s = 0; s < 4; ++s) a5[s] = frag(wbf + MLP_BF_W5, MLP_HIDDEN, s);
#pragma unroll
  for (int l = 0; l < 4; ++l)
#pragma unroll
    for (int j = 0; j < 4; ++j) bias[l][j] = master[mlp_bias_offset(l) + 16 * w + 4 * q + j] * MLP_LOG2E;
#pragma unroll
  for (int j = 0; j < 4; ++j) bias5[j] = master[mlp_bias_offset(4) + 4 * q + j];
  f32x4 acc[NT];
#pragma unroll
  for (int T = 0; T < NT; ++T) {
    const float x[5] = {v[T][0] * (1.0f / MLP_EPS_SCALE), v[T][1] * (1.0f / MLP_EPS_SCALE),
                        v[T][2] * (1.0f / MLP_EPS_SCALE), (v[T][3] - MLP_PHI_MID) * (1.0f / MLP_PHI_SPAN),
                        (v[T][4] - MLP_KMU_MID) * (1.0f / MLP_KMU_SPAN)};
    bf16x8 o;
#pragma unroll
    for (int j = 0; j < 8; ++j) o[j] = (__bf16)0.0f;
    if (q == 0) {
#pragma unroll
      for (int j = 0; j < 4; ++j) o[j] = (__bf16)x[j];
    } else if (q == 1) {
      o[0] = (__bf16)x[4];
    }
    acc[T] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a1, o, bias[0], 0, 0, 0);
  }
#pragma unroll
  for (int l = 0; l < 4; ++l) {
    // layer l's pre-activations are in acc: save, SiLU, and into the next layer's operand rows
    uint16_t(*act)[LDW_H] = s_act[l & 1];
#pragma unroll
    for (int T = 0; T < NT; ++T) {
      const int64_t r = row0 + 16 * T + c;
      if (zsave && r < n)
        *reinterpret_cast<f32x4*>(zsave + (((r >> 4) * 4 + l) * 16 + (r & 15)) * MLP_HIDDEN + 16 * w + 4 * q) =
            acc[T] * MLP_LN2;
      typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
      bf16x4 o;
#pragma unroll
      for (int j = 0; j < 4; ++j) o[j] = (__bf16)silu_log2(acc[T][j]);
      *reinterpret_cast<bf16x4*>(&act[16 * T + c][32 * (w >> 1) + 8 * q + 4 * (w & 1)]) = o;
    }
    __syncthreads();  // the other buffer was last read before this barrier
    if (l < 3) {
#pragma unroll
      for (int T = 0; T < NT; ++T) {
        acc[T] = bias[l + 1];
#pragma unroll
        for (int s = 0; s < 4; ++s) {
          const bf16x8 b = *reinterpret_cast<const bf16x8*>(&act[16 * T + c][32 * s + 8 * q]);
          acc[T] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah[l][s], b, acc[T], 0, 0, 0);
        }
      }
    } else if (w < NT) {  // output layer: wave T takes sample tile T
      f32x4 o = bias5;
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        const bf16x8 b = *reinterpret_cast<const bf16x8*>(&act[16 * w + c][32 * s + 8 * q]);
        o = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a5[s], b, o, 0, 0, 0);
      }
      const int64_t r = row0 + 16 * w + c;
      if (q == 0 && r < n) {
#pragma unroll
        for (int k = 0; k < 3; ++k) out[r * 3 + k] = o[k];
      }
    }
  }
}

// ------------------------------------------------------------------ backward
// One workgroup (8 waves) processes 64 consecutive rows per iteration and writes the weight gradients
// of its rows; the loss is L = sum over rows and outputs of (y - t)^2 / n, t = (H - eps) / CORR_SCALE.
// Partial gradients are written per workgroup (grad_part + blockIdx.x * MLP_NPARAM, every entry) and
// summed in workgroup order by k_mlp_reduce, so training is deterministic.
//
// Per layer L, from the output down: dW_L = dZ_L^T A_{L-1} and db_L from the rows' dZ_L, then
// dA_{L-1} = dZ_L W_L and dZ_{L-1} = dA_{L-1} SiLU'(Z_{L-1}). Wave w owns the 16 input features of
// tile w: it reads its column tile of Z_{L-1} once (the next layer's while this one is computed) for
// both SiLU (the operand A_{L-1}^T) and SiLU', and its 16 rows of W_L^T straight into registers. The
// kernel is bound by the chain of layers (few workgroups: 64 for a 4096-row batch), so its steps hold
// no strided gather and, for a workgroup's first group, no global read-modify-write (later groups, in batches of
// more than 1024 x 64 rows, add to its gradients in memory).
// Measured on MI355X at 4096 rows: 30 us; with 4 waves, gradients accumulated in global memory and each
// Z element gathered by row (64 cache lines per load) it took 152 us.
constexpr int BWD_THREADS = 512;
struct BackShared {
  float dz[64][MLP_HIDDEN + 4];      // dZ of the current layer, rows of the 64-row group (FP32)
  uint16_t dzt[MLP_HIDDEN][64 + 8];  // dZ^T (bf16), feature-major
  uint16_t at[MLP_HIDDEN][64 + 8];   // A_prev^T (bf16), feature-major
  uint16_t dzb[64][LDA];             // dZ rows (bf16): the A operand of dA = dZ W
};

// One 64-row group: its gradient entries are stored (FIRST: the workgroup's first group) or added.
template <bool FIRST>
__device__ __forceinline__ float backward_group(BackShared& s, const uint16_t* __restrict__ wbft,
                                                const float* __restrict__ in, const float* __restrict__ y,
                                                const float* __restrict__ H, const float* __restrict__ zsave, int n, int grp,
                                                float* __restrict__ g, float lsum) {
  const int tid = threadIdx.x, w = tid >> 6, lane = tid & 63;
  const int col = lane & 15, rq = (lane >> 4) * 4, kq = (lane >> 4) * 8;
  const int f = 16 * w + col;  // this lane's input feature
  const int row0 = grp * 64;
  auto put = [&](int i, float v) { g[i] = FIRST ? v : g[i] + v; };
  // All bits for the rows before n, none past it: rows past n contribute exact zeros (their loads
  // repeat the last row's values; a mask, unlike a branch per value, keeps the loads together).
  uint32_t ok[4];
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    ok[t] = 0;
#pragma unroll
    for (int j = 0; j < 4; ++j) ok[t] |= row0 + 16 * t + rq + j < n ? 1u << j : 0u;
  }
  auto mask = [&](int t, int j) { return 0u - ((ok[t] >> j) & 1u); };
  // this lane's 16 entries of Z_l: rows 16 t + rq + j, feature f
  auto load_z = [&](int l, float (&z)[4][4]) {
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int r = min(row0 + 16 * t + rq + j, n - 1);
        z[t][j] = zsave[(((size_t)(r >> 4) * 4 + l) * 16 + (r & 15)) * MLP_HIDDEN + f];
      }
  };
  {
    float z[4][4];
    load_z(3, z);
    // dZ of the output layer: 2 (y - t) / n in the first 3 features, zero in the padding up to 32
    for (int i = tid; i < 64 * 32; i += BWD_THREADS) {
      const int r = i >> 5, o = i & 31;
      float d = 0.0f, e = 0.0f;
      if (o < 3 && row0 + r < n) {
        const size_t rr = (size_t)(row0 + r);
        e = y[rr * 3 + o] - (H[rr * 3 + o] - in[rr * 5 + o]) / MLP_CORR_SCALE;
        d = 2.0f * e / (float)n;
      }
      if (o < MLP_OUT_PAD) {
        s.dz[r][o] = d;
        s.dzt[o][r] = f2bf(d);
      }
      s.dzb[r][o] = f2bf(d);
      if (o < 3) s.dz[r][64 + o] = e;  // the errors, for the loss
    }
    __syncthreads();
    if (tid < 64) {
      if (row0 + tid < n)
        for (int c = 0; c < 3; ++c) lsum += s.dz[tid][64 + c] * s.dz[tid][64 + c];
    }
#pragma unroll 1
    for (int L = 4; L >= 0; --L) {
      const int nout = (L == 4) ? MLP_OUT_PAD : MLP_HIDDEN;
      const int nin = (L == 0) ? MLP_IN_PAD : MLP_HIDDEN;
      // A_prev^T (feature-major, bf16): SiLU(Z_{L-1}), or the normalised inputs for L = 0
      float zn[4][4];
      bf16x8 bw[4];
      if (L > 0) {
        if (L > 1) load_z(L - 2, zn);  // the next layer's, under this layer's products
        const uint16_t* wt = wbft + mlp_t_offset(L) + (size_t)f * (L == 4 ? 32 : MLP_HIDDEN);
        bw[0] = *reinterpret_cast<const bf16x8*>(wt + kq);
#pragma unroll
        for (int ss = 1; ss < 4; ++ss) bw[ss] = *reinterpret_cast<const bf16x8*>(wt + (L == 4 ? 0 : 32 * ss) + kq);
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          uint16_t o[4];
#pragma unroll
          for (int j = 0; j < 4; ++j) o[j] = (uint16_t)(f2bf(silu(z[t][j])) & mask(t, j));
          *reinterpret_cast<uint2*>(&s.at[f][16 * t + rq]) =
              make_uint2((uint32_t)o[0] | ((uint32_t)o[1] << 16), (uint32_t)o[2] | ((uint32_t)o[3] << 16));
        }
      } else {
        for (int i = tid; i < MLP_IN_PAD * 64; i += BWD_THREADS) {
          const int fi = i >> 6, r = i & 63;
          float a = 0.0f;
          if (fi < 5 && row0 + r < n) {
            const float x = in[(size_t)(row0 + r) * 5 + fi];
            a = fi < 3 ? x * (1.0f / MLP_EPS_SCALE)
                       : (fi == 3 ? (x - MLP_PHI_MID) * (1.0f / MLP_PHI_SPAN) : (x - MLP_KMU_MID) * (1.0f / MLP_KMU_SPAN));
          }
          s.at[fi][r] = f2bf(a);
        }
      }
      __syncthreads();
      // dW_L[o][k] = sum over the rows of dZ[r][o] A_prev[r][k]: K = 64 rows = 2 MFMA steps. Wave w takes
      // output tile w and every input tile (L = 4: the one output tile and input tile w).
      {
        const int woff = mlp_weight_offset(L), o0 = L == 4 ? 0 : 16 * w;
        const int t0 = L == 4 ? w : 0, t1 = L == 4 ? w + 1 : nin / 16;
        const bf16x8 a0 = *reinterpret_cast<const bf16x8*>(&s.dzt[o0 + col][kq]);
        const bf16x8 a1 = *reinterpret_cast<const bf16x8*>(&s.dzt[o0 + col][32 + kq]);
        for (int t = t0; t < t1; ++t) {
          const bf16x8 b0 = *reinterpret_cast<const bf16x8*>(&s.at[16 * t + col][kq]);
          const bf16x8 b1 = *reinterpret_cast<const bf16x8*>(&s.at[16 * t + col][32 + kq]);
          f32x4 acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a0, b0, f32x4{0, 0, 0, 0}, 0, 0, 0);
          acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a1, b1, acc, 0, 0, 0);
#pragma unroll
          for (int j = 0; j < 4; ++j) put(woff + (o0 + rq + j) * nin + 16 * t + col, acc[j]);
        }
      }
      // db_L = sum over the rows of dZ[r][o], rows ascending
      if (tid < nout) {
        float sb = 0.0f;
#pragma unroll 16
        for (int r = 0; r < 64; ++r) sb += s.dz[r][tid];
        put(mlp_bias_offset(L) + tid, sb);
      }
      if (L == 0) break;
      // dA_{L-1} = dZ_L W_L for the wave's input features and the four row tiles (W_L^T [in][out], zero
      // padded to 32 outputs for the output layer), then dZ_{L-1} = dA_{L-1} SiLU'(Z_{L-1})
      f32x4 acc[4];
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        acc[t] = f32x4{0, 0, 0, 0};
#pragma unroll
        for (int ss = 0; ss < 4; ++ss) {
          if (L == 4 && ss > 0) break;
          const bf16x8 a = *reinterpret_cast<const bf16x8*>(&s.dzb[16 * t + col][32 * ss + kq]);
          acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, bw[ss], acc[t], 0, 0, 0);
        }
      }
      __syncthreads();  // every wave has read dZ_L
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        uint16_t o[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int r = 16 * t + rq + j;
          const float d = __uint_as_float(__float_as_uint(acc[t][j] * dsilu(z[t][j])) & mask(t, j));
          o[j] = f2bf(d);
          s.dz[r][f] = d;
          s.dzb[r][f] = o[j];
        }
        *reinterpret_cast<uint2*>(&s.dzt[f][16 * t + rq]) =
            make_uint2((uint32_t)o[0] | ((uint32_t)o[1] << 16), (uint32_t)o[2] | ((uint32_t)o[3] << 16));
      }
      if (L > 1) {
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
          for (int j = 0; j < 4; ++j) z[t][j] = zn[t][j];
      }
    }
    __syncthreads();  // the next group rewrites the shared arrays
  }
  return lsum;
}

__global__ __launch_bounds__(BWD_THREADS) void k_mlp_backward(const uint16_t* __restrict__ wbft,
                                                              const float* __restrict__ in, const float* __restrict__ y,
                                                              const float* __restrict__ H, const float* __restrict__ zsave,
                                                              int n, float* __restrict__ grad_part,
                                                              float* __restrict__ loss) {
  extern __shared__ __align__(16) unsigned char smem[];
  BackShared& s = *reinterpret_cast<BackShared*>(smem);
  float* g = grad_part + (size_t)blockIdx.x * MLP_NPARAM;
  const int ngrp = (n + 63) / 64;  // at least one per workgroup
  float lsum = backward_group<true>(s, wbft, in, y, H, zsave, n, blockIdx.x, g, 0.0f);
  for (int grp = blockIdx.x + gridDim.x; grp < ngrp; grp += gridDim.x)
    lsum = backward_group<false>(s, wbft, in, y, H, zsave, n, grp, g, lsum);
  // the loss terms are in the first wave's lanes
  if (threadIdx.x < 64) {
    for (int off = 32; off > 0; off >>= 1) lsum += __shfl_xor(lsum, off);
    if (threadIdx.x == 0) loss[blockIdx.x] = lsum;
  }
}

// Sum of the per-workgroup partial gradients in workgroup order (deterministic), 16 loads in flight
// (one load at a time took 18 us for 64 partials, 16 take 8 us with the Adam update). The sum either goes to grad or straight into the Adam
// update of its parameter, which saves a launch and a round trip through memory per training batch.
// Block 0 also sums the workgroups' losses: added to *loss_acc (training) or, over n, into *loss_mean.
struct AdamArgs {
  float *master, *m1, *m2;
  uint16_t *wbf, *wbft;
  float lr, beta1, beta2, eps;
  int step;
};
__device__ __forceinline__ void mlp_adam(const AdamArgs& p, int i, float grad);

template <bool ADAM>
__global__ __launch_bounds__(256) void k_mlp_reduce(const float* __restrict__ part, int nparts, float* __restrict__ grad,
                                                    const float* __restrict__ loss_part, float* __restrict__ loss_acc,
                                                    float* __restrict__ loss_mean, int n, AdamArgs adam) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i == 0) {
    float l = 0.0f;
    for (int p = 0; p < nparts; ++p) l += loss_part[p];
    if (loss_acc) *loss_acc += l;
    if (loss_mean) *loss_mean = l / (float)n;
  }
  if (i >= MLP_NPARAM) return;
  float s = 0.0f;
  int p = 0;
  for (; p + 16 <= nparts; p += 16) {
    float v[16];
#pragma unroll
    for (int k = 0; k < 16; ++k) v[k] = part[(size_t)(p + k) * MLP_NPARAM + i];
#pragma unroll
    for (int k = 0; k < 16; ++k) s += v[k];
  }
  for (; p < nparts; ++p) s += part[(size_t)p * MLP_NPARAM + i];
  if constexpr (ADAM) mlp_adam(adam, i, s);
  else grad[i] = s;
}

// BF16 copies of master entry i: forward [N][K] and, for layers 1..4, transposed [K][N'].
__device__ __forceinline__ void mlp_store_bf16(int i, float wv, uint16_t* wbf, uint16_t* wbft) {
  for (int l = 0; l < 5; ++l) {
    const int w0 = mlp_weight_offset(l), b0 = mlp_bias_offset(l);
    if (i >= w0 && i < b0) {
      const int K = mlp_K(l), o = (i - w0) / K, k = (i - w0) % K;
      const int fo = l == 0 ? MLP_BF_W1 : (l == 4 ? MLP_BF_W5 : MLP_BF_WH + (l - 1) * MLP_HIDDEN * MLP_HIDDEN);
      // forward copy in the log2(e)-scaled convention (MLP_LOG2E); the backward's transposed copy unscaled
      wbf[fo + o * K + k] = f2bf(l == 0 ? wv * MLP_LOG2E : (l == 4 ? wv * MLP_LN2 : wv));
      if (l >= 1) wbft[mlp_t_offset(l) + k * (l == 4 ? 32 : MLP_HIDDEN) + o] = f2bf(wv);
      return;
    }
  }
}

// Adam (Kingma & Ba 2015) on FP32 master weight i; padded entries stay zero; BF16 copies refreshed.
__device__ __forceinline__ void mlp_adam(const AdamArgs& p, int i, float grad) {
  const bool act = mlp_param_active(i);
  const float gi = act ? grad : 0.0f;
  // fused in this form, so that the moments do not depend on the compiler's choice
  const float a = __builtin_fmaf(1.0f - p.beta1, gi, p.beta1 * p.m1[i]);
  const float b = __builtin_fmaf(gi, (1.0f - p.beta2) * gi, p.beta2 * p.m2[i]);
  p.m1[i] = a;
  p.m2[i] = b;
  const float ah = a / (1.0f - powf(p.beta1, (float)p.step));
  const float bh = b / (1.0f - powf(p.beta2, (float)p.step));
  const float wv = act ? p.master[i] - p.lr * ah / (sqrtf(bh) + p.eps) : 0.0f;
  p.master[i] = wv;
  mlp_store_bf16(i, wv, p.wbf, p.wbft);
}

__global__ __launch_bounds__(256) void k_mlp_to_bf16(const float* __restrict__ master, uint16_t* __restrict__ wbf,
                                                     uint16_t* __restrict__ wbft) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= MLP_NPARAM) return;
  mlp_store_bf16(i, mlp_param_active(i) ? master[i] : 0.0f, wbf, wbft);
}

size_t mlp_forward_smem() { return sizeof(MLPShared); }
size_t mlp_backward_smem() { return sizeof(BackShared); }

void mlp_set_smem_limits() {
  (void)hipFuncSetAttribute(reinterpret_cast<const void*>(&k_mlp_forward), hipFuncAttributeMaxDynamicSharedMemorySize,
                            (int)mlp_forward_smem());
  (void)hipFuncSetAttribute(reinterpret_cast<const void*>(&k_mlp_backward), hipFuncAttributeMaxDynamicSharedMemorySize,
                            (int)mlp_backward_smem());
}

// Which forward: the small-batch kernel re-reads the weights for every 32 rows, the other one stages them
// once per workgroup and CU. Up to two small workgroups per CU the first is faster (4096 rows 14 against
// 32 us, 16384 rows 22 against 32 us); from four per CU on the second (32768 rows 37 against 33 us, 65536
// rows 69 against 34 us).
void launch_mlp_forward(hipStream_t s, const uint16_t* wbf, const float* master, const float* in, float* out, int n,
                        float* zsave, int n_cu) {
  if (n <= 0) return;
  if (n <= SMALL_PER_CU * SMALL_ROWS * n_cu) {
    hipLaunchKernelGGL(k_mlp_forward_small, dim3((n + SMALL_ROWS - 1) / SMALL_ROWS), dim3(SMALL_THREADS), 0, s, wbf,
                       master, in, out, n, zsave);
    return;
  }
  // one workgroup per CU at most: each stages the weights once and its waves take 64 rows at a time
  const int grid = (int)std::min<int64_t>(n_cu, ((int64_t)n + MLP_FWD_THREADS - 1) / MLP_FWD_THREADS);
  hipLaunchKernelGGL(k_mlp_forward, dim3(grid), dim3(MLP_FWD_THREADS), mlp_forward_smem(), s, wbf, master, in, out, n,
                     zsave);
}

void launch_mlp_backward(hipStream_t s, const uint16_t* wbft, const float* in, const float* y, const float* H,
                         const float* zsave, int n, float* grad_part, float* loss, int grid) {
  hipLaunchKernelGGL(k_mlp_backward, dim3(grid), dim3(BWD_THREADS), mlp_backward_smem(), s, wbft, in, y, H, zsave, n,
                     grad_part, loss);
}

void launch_mlp_reduce(hipStream_t s, const float* part, int nparts, float* grad, const float* loss_part,
                       float* loss_acc, float* loss_mean, int n) {
  hipLaunchKernelGGL(k_mlp_reduce<false>, dim3((MLP_NPARAM + 255) / 256), dim3(256), 0, s, part, nparts, grad, loss_part,
                     loss_acc, loss_mean, n, AdamArgs{});
}

void launch_mlp_reduce_adam(hipStream_t s, const float* part, int nparts, const float* loss_part, float* loss_acc,
                            float* master, float* m1, float* m2, uint16_t* wbf, uint16_t* wbft, float lr, int step) {
  const AdamArgs adam{master, m1, m2, wbf, wbft, lr, 0.9f, 0.999f, 1e-8f, step};
  hipLaunchKernelGGL(k_mlp_reduce<true>, dim3((MLP_NPARAM + 255) / 256), dim3(256), 0, s, part, nparts, nullptr,
                     loss_part, loss_acc, nullptr, 0, adam);
}

void launch_mlp_to_bf16(hipStream_t s, const float* master, uint16_t* wbf, uint16_t* wbft) {
  hipLaunchKernelGGL(k_mlp_to_bf16, dim3((MLP_NPARAM + 255) / 256), dim3(256), 0, s, master, wbf, wbft);
}

}  // namespace mpm

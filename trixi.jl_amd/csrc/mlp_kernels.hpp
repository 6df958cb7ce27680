// mlp_kernels.hpp -- the launches of the learned troubled-cell indicator's
// network (mlp.hpp): parameter packing, inference over a feature matrix,
// loss gradient, the fixed-order reduction of its partial rows, one from each
// workgroup, and Adam. Included by the one translation unit that launches them (the element
// kernels include only mlp.hpp's device functions).
#pragma once
#include "mlp.hpp"

namespace trixi_hip {
namespace mlp {

// FP32 parameters -> images (one thread for each parameter, then the padded features).
constexpr int PACK_BLOCKS = (NP + NH * (KF - NF) + 255) / 256;
__global__ __launch_bounds__(256) void mlp_pack_kernel(const float *__restrict__ w, TrainImage *__restrict__ img) {
  const int p = blockIdx.x * 256 + threadIdx.x;
  const int i = p - NP;
  if (p < NP) pack_param(*img, p, w[p]);
  else if (i < NH * (KF - NF)) img->infer.w1f[frag_index<2>(i / (KF - NF), NF + i % (KF - NF))] = 0;
  if (p < 3) img->infer.pad[p] = 0.f;
}

// Inference over E elements: alpha_raw[e] = hg_clip(alpha_max * y(features[e])),
// or the HG value (alpha_hg, clipped by the HG kernel) when a feature lies
// outside [lo, hi] or y is not finite (fallback != 0); with fallback == 0 the
// network output is always used.
__global__ __launch_bounds__(NTHR) void mlp_infer_kernel(const float *__restrict__ w, const float *__restrict__ x,
                                                         const float *__restrict__ lo, const float *__restrict__ hi,
                                                         const double *__restrict__ alpha_hg, double alpha_max,
                                                         double alpha_min, int fallback, int E,
                                                         double *__restrict__ alpha_raw, float *__restrict__ y_out) {
  __shared__ __attribute__((aligned(16))) WeightsLDS s;
  load_weights(w, s);
  __syncthreads();
  const int wave = threadIdx.x >> 6, l = threadIdx.x & 63;
  const int ntiles = (E + 15) / 16;
  for (int tile = blockIdx.x * WAVES + wave; tile < ntiles; tile += gridDim.x * WAVES) {
    Tile t;
    load_tile(x, E, tile, t);
    forward_layers(s, t);
    const int e = tile * 16 + l;
    if (l < 16 && e < E) {
      if (y_out) y_out[e] = t.y;
      if (alpha_raw) {
        bool use_nn = true;
        if (fallback) {
          use_nn = isfinite(t.y);
          for (int f = 0; f < NF; ++f) {
            const float v = x[(size_t)e * KF + f];
            use_nn = use_nn && v >= lo[f] && v <= hi[f];
          }
        }
        alpha_raw[e] = use_nn ? hg_clip(alpha_max * (double)t.y, alpha_min, alpha_max) : alpha_hg[e];
      }
    }
  }
}

// Sum over the 16 lanes of a row group, in every lane: the pairs of a butterfly
// over lane bits 0..3 in DPP moves (quads, then mirrored halves and rows: after
// two steps the lanes of a quad agree, so a mirrored lane holds what the lane with
// one bit flipped does).
template <int CTRL> __device__ __forceinline__ float dpp_move(float x) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), CTRL, 0xf, 0xf, true));
}
__device__ __forceinline__ float row_sum(float x) {
  x += dpp_move<0xB1>(x);   // quad_perm 1 0 3 2
  x += dpp_move<0x4E>(x);   // quad_perm 2 3 0 1
  x += dpp_move<0x141>(x);  // row_half_mirror
  x += dpp_move<0x140>(x);  // row_mirror
  return x;
}

// Loss L = sum_e (y_e - target_e)^2 / n and its gradient. Workgroup b of B
// handles tiles b, b + B, ... and writes one partial row [NPL] (gradient, then
// loss) to partial[b]; mlp_reduce_kernel sums the rows.
//
// A minibatch has few tiles (512 of them at 8192 elements), so a launch lasts as
// long as one wavefront's chain of instructions and memory round trips. Hence four
// wavefronts to a tile: each runs the forward pass, then wavefront w takes hidden rows
// 16 w .. 16 w + 15 of both layers' gradients (and wavefront 0 the scalars). The
// weights are loaded as fragments from the image into registers, all at once. 8192
// elements: 25.2 us with one wavefront to a tile, four to a workgroup that converted
// the FP32 weights into LDS first; 13.9 us with one, weights from the image; 13.3 us
// with four.
__global__ __launch_bounds__(256) void mlp_grad_kernel(const TrainImage *__restrict__ img, const float *__restrict__ x,
                                                       const float *__restrict__ target, int n,
                                                       float *__restrict__ partial) {
  // transposes [hidden or feature][element], BF16, of each wavefront
  __shared__ __attribute__((aligned(16))) uint16_t s_x[4][KF * 16];
  __shared__ __attribute__((aligned(16))) uint16_t s_h1[4][NH * 16];
  __shared__ __attribute__((aligned(16))) uint16_t s_d2[4][16 * 16];
  __shared__ __attribute__((aligned(16))) uint16_t s_d1[4][16 * 16];
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), l = threadIdx.x & 63;
  const int g = l >> 4, c = l & 15;
  const int ntiles = (n + 15) / 16;
  const float inv_n = 1.f / (float)n;
  WeightRegs wr;
  load_weight_regs(img->infer, wr);
  bf16x4 w2t[4];  // of input rows 16 w ..
#pragma unroll
  for (int ob = 0; ob < 4; ++ob) w2t[ob] = lds4(&img->w2tf[((w * 4 + ob) * 64 + l) * 4]);

  f32x4 gW1[2], gW2[4];
#pragma unroll
  for (int b = 0; b < 2; ++b) gW1[b] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int b = 0; b < 4; ++b) gW2[b] = f32x4{0.f, 0.f, 0.f, 0.f};
  float gb1[4], gb2[4], gw3[4];  // per lane: hidden 16 w + 4 g + r
#pragma unroll
  for (int r = 0; r < 4; ++r) gb1[r] = gb2[r] = gw3[r] = 0.f;
  float gb3 = 0.f, loss = 0.f;

  for (int tile = blockIdx.x; tile < ntiles; tile += gridDim.x) {
    Tile t;
    load_tile(x, n, tile, t);
    const int e = tile * 16 + c;
    const bool ok = e < n;
    const float tgt = ok ? target[e] : 0.f;
    forward_layers_regs(wr, t);
    const float res = ok ? t.y - tgt : 0.f;
    if (g == 0) {
      loss += res * res * inv_n;
      gb3 += 2.f * res * t.y * (1.f - t.y) * inv_n;
    }
    const float dout = 2.f * res * t.y * (1.f - t.y) * inv_n;  // dL/do for element c
    // layer 3 and layer 2 backward (C layout)
    bf16x4 d2b[4], d2w = {0, 0, 0, 0};
#pragma unroll
    for (int ob = 0; ob < 4; ++ob) {
      float d2[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) d2[r] = t.z2[ob][r] > 0.f ? wr.w3[ob][r] * dout : 0.f;
      d2b[ob] = pack4(d2[0], d2[1], d2[2], d2[3]);
      if (ob == w) {
        d2w = d2b[ob];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const float z = t.z2[ob][r];
          gw3[r] += dout * (z > 0.f ? z : 0.f);
          gb2[r] += d2[r];
        }
      }
    }
    // rows 16 w .. of dH1^T = W2^T dZ2^T, then through the first ReLU
    f32x4 acc = {0.f, 0.f, 0.f, 0.f}, z1 = t.z1[0];
#pragma unroll
    for (int ob = 0; ob < 4; ++ob) acc = mfma(w2t[ob], d2b[ob], acc);
#pragma unroll
    for (int b = 1; b < 4; ++b)
      if (b == w) z1 = t.z1[b];
    float d1[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      d1[r] = z1[r] > 0.f ? acc[r] : 0.f;
      gb1[r] += d1[r];
    }
    // transposes: [hidden][element] images of X, H1, dZ2, dZ1 (BF16)
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
      for (int j = 0; j < 4; ++j) s_x[w][(kb * 16 + 4 * g + j) * 16 + c] = (uint16_t)t.xb[kb][j];
#pragma unroll
    for (int b = 0; b < 4; ++b)
#pragma unroll
      for (int j = 0; j < 4; ++j) s_h1[w][(b * 16 + 4 * g + j) * 16 + c] = (uint16_t)t.h1b[b][j];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      s_d2[w][(4 * g + j) * 16 + c] = (uint16_t)d2w[j];
      s_d1[w][(4 * g + j) * 16 + c] = to_bf16(d1[j]);
    }
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    // dW2 (out x in) += dZ2^T H1: A = dZ2^T rows, B = H1 columns, K = element
    const bf16x4 a2 = lds4(&s_d2[w][c * 16 + 4 * g]);
#pragma unroll
    for (int ib = 0; ib < 4; ++ib) gW2[ib] = mfma(a2, lds4(&s_h1[w][(ib * 16 + c) * 16 + 4 * g]), gW2[ib]);
    // dW1 (hidden x feature) += dZ1^T X
    const bf16x4 a1 = lds4(&s_d1[w][c * 16 + 4 * g]);
#pragma unroll
    for (int fb = 0; fb < 2; ++fb) gW1[fb] = mfma(a1, lds4(&s_x[w][(fb * 16 + c) * 16 + 4 * g]), gW1[fb]);
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
  }

  float *row = partial + (size_t)blockIdx.x * NPL;
  // accumulator layout: row 4g + r, column c of each 16 x 16 tile
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int h = w * 16 + 4 * g + r;
#pragma unroll
    for (int fb = 0; fb < 2; ++fb)
      if (fb * 16 + c < NF) row[OFF_W1 + h * NF + fb * 16 + c] = gW1[fb][r];
#pragma unroll
    for (int ib = 0; ib < 4; ++ib) row[OFF_W2 + h * NH + ib * 16 + c] = gW2[ib][r];
    // per-lane vectors summed over the 16 lanes of a row group (elements)
    const float s1 = row_sum(gb1[r]), s2 = row_sum(gb2[r]), s3 = row_sum(gw3[r]);
    if (c == 0) {
      row[OFF_B1 + h] = s1;
      row[OFF_B2 + h] = s2;
      row[OFF_W3 + h] = s3;
    }
  }
  if (w == 0) {
    const float s = row_sum(gb3), ls = row_sum(loss);
    if (l == 0) {
      row[OFF_B3] = s;
      row[NP] = ls;
    }
  }
}

// out[p] = sum over rows of partial[row][p], p < NPL, in a fixed order: a
// workgroup takes RED_COLS consecutive columns; its RED_SPLIT row groups sum
// rows g, g + RED_SPLIT, ... in row order (each load instruction of a
// wavefront reads two rows of 32 consecutive columns), then the group sums are
// added in group order. Bound by the latency of the rows, which other XCDs wrote:
// RED_BATCH loads are in flight at a time (rows past the end add +0, which
// leaves a sum that began at +0 as it is).
//
// STEP: also one Adam step (Kingma & Ba 2015; step = 1, 2, ...) on the FP32 master
// weights w with the moments m and v, and the new weight into the images, by the
// thread that holds the gradient's sum. As four launches (reduction with two
// loads in flight, Adam, packing by one workgroup) a training step on 8192
// elements took 58 us, with this 24 us (the
// reduction alone 19.9 and 6.3 us). Same weights, bit for bit.
constexpr int RED_COLS = 32, RED_SPLIT = 8, RED_BATCH = 32;
struct AdamArgs {
  float *w, *m, *v;
  TrainImage *img;
  float lr, beta1, beta2, eps;
  int step;
};
template <bool STEP>
__global__ __launch_bounds__(RED_COLS *RED_SPLIT) void mlp_reduce_kernel(const float *__restrict__ partial, int rows,
                                                                         float *__restrict__ out, AdamArgs a) {
  __shared__ float s_part[RED_SPLIT][RED_COLS];
  const int c = threadIdx.x % RED_COLS, g = threadIdx.x / RED_COLS;
  const int p = blockIdx.x * RED_COLS + c;
  float mi = 0.f, vi = 0.f, wi = 0.f;
  if (STEP && g == 0 && p < NP) {
    mi = a.m[p];
    vi = a.v[p];
    wi = a.w[p];
  }
  float acc = 0.f;
  if (p < NPL) {
    for (int r0 = g; r0 < rows; r0 += RED_SPLIT * RED_BATCH) {
      float x[RED_BATCH];
#pragma unroll
      for (int i = 0; i < RED_BATCH; ++i) {
        const int r = r0 + RED_SPLIT * i;
        x[i] = r < rows ? partial[(size_t)r * NPL + p] : 0.f;
      }
#pragma unroll
      for (int i = 0; i < RED_BATCH; ++i) acc += x[i];
    }
  }
  s_part[g][c] = acc;
  __syncthreads();
  if (g == 0 && p < NPL) {
    float t = s_part[0][c];
#pragma unroll
    for (int k = 1; k < RED_SPLIT; ++k) t += s_part[k][c];
    out[p] = t;
    if (STEP && p < NP) {
      // the roundings written out: Adam divides by the gradient's size, so that one of
      // another order shows in the weights after a few steps
      mi = __builtin_fmaf(1.f - a.beta1, t, a.beta1 * mi);
      vi = __builtin_fmaf((1.f - a.beta2) * t, t, a.beta2 * vi);
      a.m[p] = mi;
      a.v[p] = vi;
      const float mh = mi / (1.f - powf(a.beta1, (float)a.step));
      const float vh = vi / (1.f - powf(a.beta2, (float)a.step));
      wi -= a.lr * mh / (sqrtf(vh) + a.eps);
      a.w[p] = wi;
      pack_param(*a.img, p, wi);
    }
  }
}

}  // namespace mlp
}  // namespace trixi_hip

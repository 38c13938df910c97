// oic_mlp.h -- the learned cost model: a 12 -> 64 -> 64 -> 2 ReLU MLP in FP32 on gfx950.
//
// Parameter vector (OIC_NPARAM floats): W1[64][12] b1[64] W2[64][64] b2[64] W3[2][64] b3[2].
// Inputs are standardised features z = (x - mu) / sd; outputs are log(1 + DP cells) and the
// exit diagonal / 1000.  Loss per sample: 0.5 (y0 - t0)^2 + 0.5 w_exit (y1 - t1)^2, averaged.
//
// Kernels: the forward pass runs one thread per sample with the weights in LDS.  The gradient runs four
// wavefronts over MLP_CHUNK samples, one per 16 hidden units, on the FP32 matrix cores; each workgroup writes its
// sums once, and the kernel of the weight update adds them up.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#define MLP_IN  12
#define MLP_H   64
#define MLP_OUT 2
#define MLP_OFF_W1 0
#define MLP_OFF_B1 (MLP_OFF_W1 + MLP_H * MLP_IN)
#define MLP_OFF_W2 (MLP_OFF_B1 + MLP_H)
#define MLP_OFF_B2 (MLP_OFF_W2 + MLP_H * MLP_H)
#define MLP_OFF_W3 (MLP_OFF_B2 + MLP_H)
#define MLP_OFF_B3 (MLP_OFF_W3 + MLP_OUT * MLP_H)
#define MLP_NPARAM (MLP_OFF_B3 + MLP_OUT)

__device__ __forceinline__ float wave_sum_f(float v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
  return v;
}

// y[i] = MLP(x[i]) with x standardised by (mu, sd) when mu != nullptr
__global__ void __launch_bounds__(256) k_mlp_forward(const float *__restrict__ X, uint64_t n, const float *__restrict__ P,
                                                     const float *__restrict__ mu, const float *__restrict__ sd,
                                                     float *__restrict__ Y) {
  __shared__ float w[MLP_NPARAM];
  for (int i = threadIdx.x; i < MLP_NPARAM; i += blockDim.x) w[i] = P[i];
  __syncthreads();
  const uint64_t s = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= n) return;
  float z[MLP_IN];
#pragma unroll
  for (int i = 0; i < MLP_IN; i++) {
    const float x = X[s * MLP_IN + i];
    z[i] = mu ? (x - mu[i]) / sd[i] : x;
  }
  float h1[MLP_H];
#pragma unroll
  for (int j = 0; j < MLP_H; j++) {
    float a = w[MLP_OFF_B1 + j];
#pragma unroll
    for (int i = 0; i < MLP_IN; i++) a += w[MLP_OFF_W1 + j * MLP_IN + i] * z[i];
    h1[j] = a > 0.f ? a : 0.f;
  }
  float y0 = w[MLP_OFF_B3], y1 = w[MLP_OFF_B3 + 1];
  for (int k = 0; k < MLP_H; k++) {
    float a = w[MLP_OFF_B2 + k];
#pragma unroll
    for (int j = 0; j < MLP_H; j++) a += w[MLP_OFF_W2 + k * MLP_H + j] * h1[j];
    const float h2 = a > 0.f ? a : 0.f;
    y0 += w[MLP_OFF_W3 + k] * h2;
    y1 += w[MLP_OFF_W3 + MLP_H + k] * h2;
  }
  Y[s * MLP_OUT] = y0;
  Y[s * MLP_OUT + 1] = y1;
}

typedef float f32x4 __attribute__((ext_vector_type(4)));

// sum over each 16 lanes, in all of them
__device__ __forceinline__ float row_sum_f(float v) {
#define OIC_RSUM(ctl)                                                                                              \
  v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int32_t, v), ctl, 0xF, 0xF, false));
  OIC_RSUM(0x128)   // row_ror:8, 4, 2, 1
  OIC_RSUM(0x124)
  OIC_RSUM(0x122)
  OIC_RSUM(0x121)
#undef OIC_RSUM
  return v;
}

// Gradient of the mean loss over samples idx[0..n) (or 0..n when idx is null); Z is standardised.  Workgroup b
// writes the sums of its chunks, in the parameters' order, and its sum of losses to part[b * MLP_PART ..].
//
// The products are v_mfma_f32_16x16x4_f32 (FP32 in, FP32 sums).  Lane (g, c) = (lane / 16, lane % 16) of wavefront
// w gives A[row c][slot g] and B[slot g][column c] and receives D[rows 4 g .. 4 g + 3][column c].  Rows are
// samples, columns the wavefront's units u = 16 w + c, so a lane keeps the activations and gradients of unit u at
// samples 4 g + r in registers from the forward pass to the end: they are the mask of the backward pass and,
// as they are, the A operand of dW2 = G2^T H1 and dW1 = G1^T Z (slot g of step r is sample 4 g + r).  The order in
// which a product's slots run over its inner index is free, so a lane reads 16 neighbours of an LDS row.
// Only H1 and G2 go through LDS.  Rows of 68 words: b128 reads of 16 rows, and dword reads and writes of rows
// 4 g + r, touch each bank once.
//
// Bound by latency at the batches in use: 128 workgroups at 4096 samples, each one chunk: 4 barriers and about
// 110 matrix instructions of 32 cycles a wavefront.  The form before it (one wavefront per 64 samples, lane =
// sample, then lane = unit, on the vector unit with one operand of each product from LDS, 256 VGPRs, an atomic per
// wavefront and parameter) took 257 us a batch, this one 10; training on 60 000 samples for 2 epochs took 8.9 ms as a
// whole, now 1.2 ms: about half are the 30 dependent steps (this kernel, 10 us, k_mlp_adam, 6, and 2 us gaps), the rest
// the host's sums and shuffles, buffers and copies.
#define MLP_TILES 2                       // of 16 samples
#define MLP_CHUNK (16 * MLP_TILES)
#define MLP_LD    (MLP_H + 4)
#define MLP_PART  (MLP_NPARAM + 2)        // the loss behind the parameters, an even stride
#define MLP_WG    512                     // most workgroups, and rows of part
__global__ void __launch_bounds__(256) k_mlp_grad(const float *__restrict__ Z, const float *__restrict__ Tg,
                                                  const uint32_t *__restrict__ idx, uint64_t n, const float *__restrict__ P,
                                                  float w_exit, float inv_n, float *__restrict__ part) {
  __shared__ __attribute__((aligned(16))) float H1[MLP_CHUNK * MLP_LD], G2[MLP_CHUNK * MLP_LD];
  __shared__ float Y[4][MLP_CHUNK][2], G3[MLP_CHUNK][2];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, g = lane >> 4, c = lane & 15, u = 16 * w + c;
  float w1[3], w2[16], w2t[16];
#pragma unroll
  for (int i = 0; i < 3; i++) w1[i] = P[MLP_OFF_W1 + u * MLP_IN + 3 * g + i];
#pragma unroll
  for (int i = 0; i < 16; i++) {
    w2[i] = P[MLP_OFF_W2 + u * MLP_H + 16 * g + i];
    w2t[i] = P[MLP_OFF_W2 + (16 * g + i) * MLP_H + u];
  }
  const float b1 = P[MLP_OFF_B1 + u], b2 = P[MLP_OFF_B2 + u], w30 = P[MLP_OFF_W3 + u], w31 = P[MLP_OFF_W3 + MLP_H + u];
  const float b30 = P[MLP_OFF_B3], b31 = P[MLP_OFF_B3 + 1];
  f32x4 dw1 = {0.f, 0.f, 0.f, 0.f}, dw2[4];
#pragma unroll
  for (int i = 0; i < 4; i++) dw2[i] = dw1;
  float db1 = 0.f, db2 = 0.f, dw30 = 0.f, dw31 = 0.f, db30 = 0.f, db31 = 0.f, loss = 0.f;

  for (uint64_t c0 = (uint64_t)blockIdx.x * MLP_CHUNK; c0 < n; c0 += (uint64_t)gridDim.x * MLP_CHUNK) {
    // features 3 g .. 3 g + 2 of sample 16 t + c; feature c of samples 16 t + 4 g + r; the targets
    float z[MLP_TILES][3], zc[MLP_TILES][4], t0 = 0.f, t1 = 0.f;
#pragma unroll
    for (int t = 0; t < MLP_TILES; t++) {
      const uint64_t si = c0 + 16 * t + c;
      const bool in = si < n;
      const float *zs = Z + (in ? (idx ? idx[si] : si) : 0) * MLP_IN + 3 * g;
#pragma unroll
      for (int i = 0; i < 3; i++) z[t][i] = in ? zs[i] : 0.f;
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const uint64_t sr = c0 + 16 * t + 4 * g + r;
        zc[t][r] = sr < n && c < MLP_IN ? Z[(idx ? idx[sr] : sr) * MLP_IN + c] : 0.f;
      }
    }
    const uint64_t st = c0 + threadIdx.x;
    const bool own = threadIdx.x < MLP_CHUNK && st < n;
    if (own) {
      const float *ts = Tg + (idx ? idx[st] : st) * MLP_OUT;
      t0 = ts[0];
      t1 = ts[1];
    }
    f32x4 h1[MLP_TILES], h2[MLP_TILES];
#pragma unroll
    for (int t = 0; t < MLP_TILES; t++) {
      h1[t] = (f32x4){b1, b1, b1, b1};
#pragma unroll
      for (int i = 0; i < 3; i++) h1[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(z[t][i], w1[i], h1[t], 0, 0, 0);
#pragma unroll
      for (int r = 0; r < 4; r++) {
        h1[t][r] = h1[t][r] > 0.f ? h1[t][r] : 0.f;
        H1[(16 * t + 4 * g + r) * MLP_LD + u] = h1[t][r];
      }
      h2[t] = (f32x4){b2, b2, b2, b2};
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < 4; q++)
#pragma unroll
      for (int t = 0; t < MLP_TILES; t++) {
        const f32x4 a = *(const f32x4 *)&H1[(16 * t + c) * MLP_LD + 16 * g + 4 * q];
#pragma unroll
        for (int i = 0; i < 4; i++) h2[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i], w2[4 * q + i], h2[t], 0, 0, 0);
      }
#pragma unroll
    for (int t = 0; t < MLP_TILES; t++)
#pragma unroll
      for (int r = 0; r < 4; r++) {
        h2[t][r] = h2[t][r] > 0.f ? h2[t][r] : 0.f;
        const float y0 = row_sum_f(w30 * h2[t][r]), y1 = row_sum_f(w31 * h2[t][r]);
        if (c == 0) {
          Y[w][16 * t + 4 * g + r][0] = y0;
          Y[w][16 * t + 4 * g + r][1] = y1;
        }
      }
    __syncthreads();
    if (threadIdx.x < MLP_CHUNK) {
      const int s = threadIdx.x;
      const float e0 = b30 + ((Y[0][s][0] + Y[1][s][0]) + (Y[2][s][0] + Y[3][s][0])) - t0;
      const float e1 = b31 + ((Y[0][s][1] + Y[1][s][1]) + (Y[2][s][1] + Y[3][s][1])) - t1;
      const float g0 = own ? e0 * inv_n : 0.f, g1 = own ? w_exit * e1 * inv_n : 0.f;
      if (own) loss += 0.5f * e0 * e0 + 0.5f * w_exit * e1 * e1;
      db30 += g0;
      db31 += g1;
      G3[s][0] = g0;
      G3[s][1] = g1;
    }
    __syncthreads();
    f32x4 g2[MLP_TILES];
#pragma unroll
    for (int t = 0; t < MLP_TILES; t++)
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const int s = 16 * t + 4 * g + r;
        const float g0 = G3[s][0], g1 = G3[s][1], h = h2[t][r];
        dw30 += g0 * h;
        dw31 += g1 * h;
        g2[t][r] = h > 0.f ? w30 * g0 + w31 * g1 : 0.f;
        db2 += g2[t][r];
        G2[s * MLP_LD + u] = g2[t][r];
      }
#pragma unroll
    for (int t = 0; t < MLP_TILES; t++)
#pragma unroll
      for (int r = 0; r < 4; r++)
#pragma unroll
        for (int j = 0; j < 4; j++)
          dw2[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(g2[t][r], H1[(16 * t + 4 * g + r) * MLP_LD + 16 * j + c], dw2[j], 0, 0, 0);
    __syncthreads();   // H1 is free from here, G2 until the next chunk's third barrier
    f32x4 g1[MLP_TILES];
#pragma unroll
    for (int t = 0; t < MLP_TILES; t++) g1[t] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int q = 0; q < 4; q++)
#pragma unroll
      for (int t = 0; t < MLP_TILES; t++) {
        const f32x4 a = *(const f32x4 *)&G2[(16 * t + c) * MLP_LD + 16 * g + 4 * q];
#pragma unroll
        for (int i = 0; i < 4; i++) g1[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i], w2t[4 * q + i], g1[t], 0, 0, 0);
      }
#pragma unroll
    for (int t = 0; t < MLP_TILES; t++)
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const float v = h1[t][r] > 0.f ? g1[t][r] : 0.f;
        db1 += v;
        dw1 = __builtin_amdgcn_mfma_f32_16x16x4f32(v, zc[t][r], dw1, 0, 0, 0);
      }
  }

  float *out = part + (uint64_t)blockIdx.x * MLP_PART;
#pragma unroll
  for (int r = 0; r < 4; r++) {
    const int k = 16 * w + 4 * g + r;
    if (c < MLP_IN) out[MLP_OFF_W1 + k * MLP_IN + c] = dw1[r];
#pragma unroll
    for (int j = 0; j < 4; j++) out[MLP_OFF_W2 + k * MLP_H + 16 * j + c] = dw2[j][r];
  }
#pragma unroll
  for (int o = 16; o <= 32; o <<= 1) {
    db1 += __shfl_xor(db1, o);
    db2 += __shfl_xor(db2, o);
    dw30 += __shfl_xor(dw30, o);
    dw31 += __shfl_xor(dw31, o);
  }
  if (g == 0) {
    out[MLP_OFF_B1 + u] = db1;
    out[MLP_OFF_B2 + u] = db2;
    out[MLP_OFF_W3 + u] = dw30;
    out[MLP_OFF_W3 + MLP_H + u] = dw31;
  }
  if (w == 0) {
    db30 = wave_sum_f(db30);
    db31 = wave_sum_f(db31);
    loss = wave_sum_f(loss);
    if (lane == 0) {
      out[MLP_OFF_B3] = db30;
      out[MLP_OFF_B3 + 1] = db31;
      out[MLP_NPARAM] = loss;
    }
  }
}

// Sum of the workgroups' rows, 64 parameters a workgroup and a quarter of the rows a wavefront.  The sum of
// losses goes to *loss, or is added there.
__device__ __forceinline__ bool mlp_sum(const float *__restrict__ part, uint32_t rows, float *__restrict__ loss, bool add_loss,
                                        int &p, float &sum) {
  __shared__ float q[4][64];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  p = blockIdx.x * 64 + lane;
  float s[4] = {0.f, 0.f, 0.f, 0.f};
  if (p <= MLP_NPARAM) {
    uint32_t b = w;
    for (; b + 28 < rows; b += 32) {
      float v[8];
#pragma unroll
      for (int i = 0; i < 8; i++) v[i] = part[(uint64_t)(b + 4 * i) * MLP_PART + p];
#pragma unroll
      for (int i = 0; i < 8; i++) s[i & 3] += v[i];
    }
    for (; b < rows; b += 4) s[0] += part[(uint64_t)b * MLP_PART + p];
  }
  q[w][lane] = (s[0] + s[1]) + (s[2] + s[3]);
  __syncthreads();
  sum = (q[0][lane] + q[1][lane]) + (q[2][lane] + q[3][lane]);
  if (w == 0 && p == MLP_NPARAM) *loss = add_loss ? *loss + sum : sum;
  return w == 0 && p < MLP_NPARAM;
}

__global__ void __launch_bounds__(256) k_mlp_sum(const float *__restrict__ part, uint32_t rows, float *__restrict__ grad,
                                                 float *__restrict__ loss) {
  int p;
  float sum;
  if (mlp_sum(part, rows, loss, false, p, sum)) grad[p] = sum;
}

// Adam (Kingma & Ba 2015) with bias correction, on the summed gradient; the first step starts m and v
__global__ void __launch_bounds__(256) k_mlp_adam(const float *__restrict__ part, uint32_t rows, float *__restrict__ P,
                                                  float *__restrict__ m, float *__restrict__ v, bool first, float lr, float b1,
                                                  float b2, float eps, float c1, float c2, float *__restrict__ loss, bool add_loss) {
  int i;
  float gi;
  if (!mlp_sum(part, rows, loss, add_loss, i, gi)) return;
  const float mi = b1 * (first ? 0.f : m[i]) + (1.f - b1) * gi;
  const float vi = b2 * (first ? 0.f : v[i]) + (1.f - b2) * gi * gi;
  m[i] = mi;
  v[i] = vi;
  const float mh = mi / c1, vh = vi / c2;
  P[i] -= lr * mh / (sqrtf(vh) + eps);
}

// z = (x - mu) / sd over n samples, in place
__global__ void k_standardise(float *__restrict__ Z, uint64_t n, const float *__restrict__ mu, const float *__restrict__ sd) {
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n * MLP_IN; i += (uint64_t)gridDim.x * blockDim.x)
    Z[i] = (Z[i] - mu[i % MLP_IN]) / sd[i % MLP_IN];
}

// the 12 features of a candidate pair: log1p of S length, T length, seed hits, match nodes;
// min and max node diagonal / 1000; log1p diagonal spread; log1p max k-mer multiplicity;
// consistent flag; orientation; log1p shorter read length; log1p longest node length
__global__ void k_pair_features(const PairRec *__restrict__ pairs, uint64_t np, const int32_t *__restrict__ len,
                                float *__restrict__ X) {
  const uint64_t p = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= np) return;
  const PairRec pr = pairs[p];
  const double sl = len[pr.s_id], tl = len[pr.t_id];
  float *x = X + p * MLP_IN;
  x[0] = (float)log1p(sl);
  x[1] = (float)log1p(tl);
  x[2] = (float)log1p((double)(pr.he - pr.hb));
  x[3] = (float)log1p((double)pr.nnodes);
  x[4] = (float)(pr.dmin / 1000.0);
  x[5] = (float)(pr.dmax / 1000.0);
  x[6] = (float)log1p((double)pr.dmax - (double)pr.dmin);
  x[7] = (float)log1p((double)pr.max_mult);
  x[8] = (float)pr.consistent;
  x[9] = (float)pr.dir;
  x[10] = (float)log1p(sl < tl ? sl : tl);
  x[11] = (float)log1p((double)pr.longest);
}

// Learned initial guess for the mixed-cell closure: a small MLP predicts the
// equilibrium volume fractions and log temperature of a cell from its inputs;
// the FP64 Newton solver starts from that guess when it lowers the initial
// residual and from its own guess otherwise, so results keep the solver's
// 1e-10 accuracy either way.
//
// Network: 64 inputs (per material slot s < 6: one-hot of the material id,
// alpha, ln rho, ln T; per cell: asinh(sie_tot / 1e10), ln rho_total; padded
// from 56) -> 128 -> 128 -> 128 (GELU, tanh form) -> 16 outputs (6 slot
// logits, masked softmax over the cell's materials; standardized ln T; 9
// padding). BF16 weights and activations, FP32 accumulation on the matrix
// cores (gfx950's v_mfma_f32_16x16x32_bf16), FP32 master weights, Adam.
//
// Work split: a wave computes 16 rows (cells) x all columns of a layer with
// 16x16 MFMA tiles and keeps its rows in LDS from layer to layer. Inference:
// blocks of 8 waves with every layer's weights in LDS. Training: blocks of 4
// waves, the weights of the layer being applied in LDS ([out][in] for the
// forward, [in][out] for the input-gradient product).
#include "sgm_internal.hpp"

#include <cmath>
#include <cstring>
#include <random>
#include <vector>

namespace sgm {
namespace mlp {

constexpr int KIN = 64, H = 128, KOUT = 16, SLOTS = 6, NFEAT = 9 * SLOTS + 2;
constexpr int ROWS = 64;  // rows per block
// flat parameter layout (FP32 master, gradients, Adam moments)
constexpr int OW1 = 0, OB1 = OW1 + H * KIN, OW2 = OB1 + H, OB2 = OW2 + H * H, OW3 = OB2 + H,
              OB3 = OW3 + H * H, OW4 = OB3 + H, OB4 = OW4 + KOUT * H, NPARAM = OB4 + KOUT;
// bf16 weight layout (no biases): W1 [128x64], W2, W3 [128x128], W4 [16x128]
constexpr int QW1 = 0, QW2 = QW1 + H * KIN, QW3 = QW2 + H * H, QW4 = QW3 + H * H,
              NQ = QW4 + KOUT * H;

typedef short s4 __attribute__((ext_vector_type(4)));
typedef __bf16 b8 __attribute__((ext_vector_type(8)));
typedef float f4 __attribute__((ext_vector_type(4)));
typedef unsigned short bf16;

__host__ __device__ inline bf16 f2bf(float x) {  // round to nearest even
  unsigned u;
  std::memcpy(&u, &x, 4);
  if ((u & 0x7f800000u) == 0x7f800000u) return (bf16)((u >> 16) | ((u & 0xffff) ? 0x40 : 0));
  u += 0x7fffu + ((u >> 16) & 1u);
  return (bf16)(u >> 16);
}
__host__ __device__ inline float bf2f(bf16 h) {
  const unsigned u = (unsigned)h << 16;
  float x;
  std::memcpy(&x, &u, 4);
  return x;
}
// One wave: acc[j] (+)= A[16 rows x K] * Bt[16 cols of tile j x K]^T, bf16 in
// LDS. A row-major with stride lda; Bt row-major ([N][K]) with stride ldb
// (16-byte aligned rows). gfx950's 16x16x32 step: lane l holds
// A[l%16][8(l/16)..+7] and Bt[l%16][8(l/16)..+7]; a K that leaves 16 over
// (the 16-wide output layer's gradient product) ends with one 16x16x16 step,
// lane l holding 4(l/16)..+3 of those 16. D[4(l/16)+i][l%16] comes back in
// acc[j][i].
template <int NT>
__device__ inline void wave_gemm(const bf16 *A, int lda, const bf16 *Bt, int ldb, int K,
                                 f4 (&acc)[NT]) {
  const int l = threadIdx.x & 63;
  const int r = l & 15;
  int k0 = 0;
  for (; k0 + 32 <= K; k0 += 32) {
    const int q = (l >> 4) * 8;
    const b8 a = *reinterpret_cast<const b8 *>(A + r * lda + k0 + q);
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      const b8 b = *reinterpret_cast<const b8 *>(Bt + (j * 16 + r) * ldb + k0 + q);
      acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, acc[j], 0, 0, 0);
    }
  }
  if (k0 < K) {
    const int q = (l >> 4) * 4;
    const s4 a = *reinterpret_cast<const s4 *>(A + r * lda + k0 + q);
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      const s4 b = *reinterpret_cast<const s4 *>(Bt + (j * 16 + r) * ldb + k0 + q);
      acc[j] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, acc[j], 0, 0, 0);
    }
  }
}

constexpr int LDK = KIN + 8, LDH = H + 8, LDR = ROWS + 8;  // padded LDS strides
constexpr int MAXPART = 256;  // training blocks: one per CU

typedef unsigned u4 __attribute__((ext_vector_type(4)));
// a [rows][COLS] bf16 matrix from global memory to LDS (stride ld) through
// registers, 16 bytes a load, so that the loads of the next layer's weights
// run under this layer's products
template <int N>
__device__ __forceinline__ void w_load(u4 (&r)[N], const bf16 *src) {
#pragma unroll
  for (int i = 0; i < N; ++i)
    r[i] = reinterpret_cast<const u4 *>(src)[i * blockDim.x + threadIdx.x];
}
template <int COLS, int N>
__device__ __forceinline__ void w_store(const u4 (&r)[N], bf16 *dst, int ld) {
#pragma unroll
  for (int i = 0; i < N; ++i) {
    const int c = i * blockDim.x + threadIdx.x;
    *reinterpret_cast<u4 *>(dst + (c / (COLS / 8)) * ld + (c % (COLS / 8)) * 8) = r[i];
  }
}
// LDS written by some lanes of a wave before it, read by others after it. The
// barrier alone orders no memory for the compiler; the fences do, and cost no
// instruction (a wave's LDS operations execute in order).
__device__ __forceinline__ void wave_handover() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}
// 16 features of a row: two 16-byte loads, or, where the caller's matrix is not
// on a 16-byte boundary, one by one
__device__ __forceinline__ void load_features(const bf16 *p, bool aligned, u4 (&x)[2]) {
  if (aligned) {
    x[0] = reinterpret_cast<const u4 *>(p)[0];
    x[1] = reinterpret_cast<const u4 *>(p)[1];
    return;
  }
#pragma unroll
  for (int i = 0; i < 8; ++i)
    x[i >> 2][i & 3] = (unsigned)p[2 * i] | ((unsigned)p[2 * i + 1] << 16);
}
template <int N>
__device__ __forceinline__ void zero_acc(f4 (&acc)[N]) {
#pragma unroll
  for (int j = 0; j < N; ++j) acc[j] = f4{0, 0, 0, 0};
}

// One hidden layer of a wave's 16 rows: product, bias, GELU. The activations
// go back to the wave's rows of `row` (in place) as bf16; TRAIN also writes
// them transposed ([column][row], the weight gradient's operand) and keeps
// GELU' of each value, so that the backward pass needs neither the
// pre-activations nor a second tanh.
template <bool TRAIN>
__device__ __forceinline__ void hidden_layer(bf16 *row, const bf16 *w, int ldw, int kin,
                                             const float *__restrict__ bias, bf16 *at, int rbase,
                                             f4 *gd) {
  const int l = threadIdx.x & 63;
  f4 acc[H / 16];
  zero_acc(acc);
  wave_gemm<H / 16>(row, LDH, w, ldw, kin, acc);
#pragma unroll
  for (int j = 0; j < H / 16; ++j) {
    const int cc = j * 16 + (l & 15), r0 = (l >> 4) * 4;
    const float bz = bias[cc];
    bf16 a[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float z = acc[j][i] + bz;
      const float k = 0.7978845608028654f, c = 0.044715f;
      const float t = tanhf(k * (z + c * z * z * z));
      a[i] = f2bf(0.5f * z * (1.0f + t));
      if constexpr (TRAIN)
        gd[j][i] = 0.5f * (1.0f + t) + 0.5f * z * (1.0f - t * t) * k * (1.0f + 3.0f * c * z * z);
      row[(r0 + i) * LDH + cc] = a[i];
    }
    if constexpr (TRAIN)
      *reinterpret_cast<s4 *>(at + cc * LDR + rbase + r0) =
          s4{(short)a[0], (short)a[1], (short)a[2], (short)a[3]};
  }
}

// The rows of one inference block: 8 waves of 16, all weights in LDS, staged
// once; a wave's tiles need nothing from the other waves.
constexpr int IROWS = 128;
struct InferLds {
  __attribute__((aligned(16))) bf16 w1[H * LDK], w2[H * LDH], w3[H * LDH], w4[KOUT * LDH];
  __attribute__((aligned(16))) bf16 row[IROWS * LDH];
  float y[IROWS * (KOUT + 1)];
  int nm[IROWS];
};
__device__ __forceinline__ void infer_stage(InferLds &L, const bf16 *__restrict__ wq) {
  u4 r1[2], r2[4], r3[4];
  w_load(r1, wq + QW1);
  w_load(r2, wq + QW2);
  w_load(r3, wq + QW3);
  w_store<KIN>(r1, L.w1, LDK);
  w_store<H>(r2, L.w2, LDH);
  w_store<H>(r3, L.w3, LDH);
  const int c = threadIdx.x;
  if (c < KOUT * H / 8)
    *reinterpret_cast<u4 *>(L.w4 + (c / (H / 8)) * LDH + (c % (H / 8)) * 8) =
        reinterpret_cast<const u4 *>(wq + QW4)[c];
  __syncthreads();
}
// the four layers of the wave's 16 rows (L.row holds the inputs): outputs in L.y
__device__ __forceinline__ void infer_rows(InferLds &L, const float *__restrict__ P) {
  const int w = threadIdx.x >> 6, l = threadIdx.x & 63;
  bf16 *row = L.row + w * 16 * LDH;
  hidden_layer<false>(row, L.w1, LDK, KIN, P + OB1, nullptr, 0, nullptr);
  wave_handover();
  hidden_layer<false>(row, L.w2, LDH, H, P + OB2, nullptr, 0, nullptr);
  wave_handover();
  hidden_layer<false>(row, L.w3, LDH, H, P + OB3, nullptr, 0, nullptr);
  wave_handover();
  f4 acc[1] = {f4{0, 0, 0, 0}};
  wave_gemm<1>(row, LDH, L.w4, LDH, H, acc);
  const float b = P[OB4 + (l & 15)];
#pragma unroll
  for (int i = 0; i < 4; ++i)
    L.y[(w * 16 + (l >> 4) * 4 + i) * (KOUT + 1) + (l & 15)] = acc[0][i] + b;
  wave_handover();
}

// outputs of rows idx[0..B) of the feature matrix Xall [N][KIN]
__global__ void __launch_bounds__(512, 1) fwd_kernel(const bf16 *__restrict__ wq,
                                                     const float *__restrict__ P,
                                                     const bf16 *__restrict__ Xall,
                                                     const int *__restrict__ idx, long B,
                                                     float *__restrict__ Y) {
  __shared__ InferLds L;
  infer_stage(L, wq);
  const int w = threadIdx.x >> 6, l = threadIdx.x & 63;
  const bool aligned = (reinterpret_cast<uintptr_t>(Xall) & 15) == 0;
  for (long t = (long)blockIdx.x * 8 + w; t * 16 < B; t += (long)gridDim.x * 8) {
    const long r = t * 16 + (l >> 2);
    u4 x[2] = {u4{0, 0, 0, 0}, u4{0, 0, 0, 0}};
    if (r < B) load_features(Xall + (long)idx[r] * KIN + (l & 3) * 16, aligned, x);
    u4 *d = reinterpret_cast<u4 *>(L.row + (w * 16 + (l >> 2)) * LDH + (l & 3) * 16);
    d[0] = x[0];
    d[1] = x[1];
    wave_handover();
    infer_rows(L, P);
    for (int k = l; k < 16 * KOUT; k += 64) {
      const long rr = t * 16 + k / KOUT;
      if (rr < B) Y[rr * KOUT + k % KOUT] = L.y[(w * 16 + k / KOUT) * (KOUT + 1) + k % KOUT];
    }
    wave_handover();
  }
}

// Loss of one row: squared error of the log volume fractions (log-softmax of
// the slot logits over the cell's materials, targets floored at 1e-8) + wT
// times the squared error of the standardized ln T; y is replaced with the
// gradient of the batch mean. Target row: [alpha0..alpha5, lnT_std, nmat (0 =
// row excluded)]
__device__ __forceinline__ float row_loss(float *y, const float *__restrict__ t, float wT,
                                          float inv_b) {
  float yv[SLOTS + 1];
#pragma unroll
  for (int c = 0; c < SLOTS + 1; ++c) yv[c] = y[c];
#pragma unroll
  for (int c = 0; c < KOUT; ++c) y[c] = 0.f;
  const int nm = t ? (int)t[7] : 0;
  if (nm < 2 || nm > SLOTS) return 0.f;
  float mx = -1e30f;
#pragma unroll
  for (int s = 0; s < SLOTS; ++s)
    if (s < nm) mx = fmaxf(mx, yv[s]);
  float p[SLOTS], sum = 0.f;
#pragma unroll
  for (int s = 0; s < SLOTS; ++s) {
    p[s] = s < nm ? expf(yv[s] - mx) : 0.f;
    sum += p[s];
  }
  const float lse = mx + logf(sum);
  float L = 0.f, e[SLOTS], esum = 0.f;
#pragma unroll
  for (int s = 0; s < SLOTS; ++s) {
    e[s] = 0.f;
    if (s >= nm) continue;
    p[s] /= sum;
    e[s] = (yv[s] - lse) - logf(fmaxf(t[s], 1e-8f));
    L += e[s] * e[s];
    esum += e[s];
  }
  // d/dy_j sum_s e_s^2 = 2 (e_j - p_j sum_s e_s)
#pragma unroll
  for (int s = 0; s < SLOTS; ++s)
    if (s < nm) y[s] = inv_b * 2.f * (e[s] - p[s] * esum);
  const float et = yv[6] - t[6];
  L += wT * et * et;
  y[6] = inv_b * 2.f * wT * et;
  return L;
}

// dz of a layer from its rows' gradient (acc x GELU'): bf16 into the wave's
// rows and transposed into dzt, column sums (the bias gradient, fp32) added
// to db
__device__ __forceinline__ void put_dz(const f4 (&acc)[H / 16], const f4 (&gd)[H / 16], bf16 *row,
                                       bf16 *dzt, int rbase, float (&db)[H / 16]) {
  const int l = threadIdx.x & 63;
#pragma unroll
  for (int j = 0; j < H / 16; ++j) {
    const int cc = j * 16 + (l & 15), r0 = (l >> 4) * 4;
    float s = 0.f;
    bf16 v[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float d = acc[j][i] * gd[j][i];
      s += d;
      v[i] = f2bf(d);
      row[(r0 + i) * LDH + cc] = v[i];
    }
    *reinterpret_cast<s4 *>(dzt + cc * LDR + rbase + r0) =
        s4{(short)v[0], (short)v[1], (short)v[2], (short)v[3]};
    s += __shfl_xor(s, 16, 64);
    s += __shfl_xor(s, 32, 64);
    db[j] += s;
  }
}

// Forward, loss and backward of 64-row tiles in one kernel: a wave's 16 rows
// stay in its registers and LDS from the features to the last gradient, and
// every weight gradient accumulates in the wave's private values over the
// block's tiles (of these 366 a lane are in scratch memory, the 512 registers of
// one wave per SIMD being in use); a block writes its partial sums once. What bounded the step before was eight
// launches, each reading and writing every activation, pre-activation and
// gradient in global memory and staging weights two bytes at a time.
// One gradient call, batch 8192: 298 -> 115 us; 32,768: 638 -> 208 us.
struct TrainLds {
  __attribute__((aligned(16))) bf16 row[ROWS * LDH], wl[H * LDH];
  __attribute__((aligned(16))) bf16 xt[KIN * LDR], at[3][H * LDR], dzt[H * LDR];
  float y[ROWS * (KOUT + 1)];
  float db[4][H];
};
__global__ void __launch_bounds__(256, 1)
    train_kernel(const bf16 *__restrict__ wq, const bf16 *__restrict__ wq_io,
                 const float *__restrict__ P, const bf16 *__restrict__ Xall,
                 const float *__restrict__ tgt, const int *__restrict__ idx, long B, int ntile,
                 float wT, float inv_b, float *__restrict__ part, float *__restrict__ loss) {
  __shared__ TrainLds L;
  const int w = threadIdx.x >> 6, l = threadIdx.x & 63, rb = w * 16;
  const bool aligned = (reinterpret_cast<uintptr_t>(Xall) & 15) == 0;
  bf16 *row = L.row + rb * LDH;
  f4 dw1[2][KIN / 16], dw2[2][H / 16], dw3[2][H / 16], dw4[2];
  float db1[H / 16], db2[H / 16], db3[H / 16], db4 = 0.f;
#pragma unroll
  for (int m = 0; m < 2; ++m) {
    zero_acc(dw1[m]);
    zero_acc(dw2[m]);
    zero_acc(dw3[m]);
  }
  zero_acc(dw4);
#pragma unroll
  for (int j = 0; j < H / 16; ++j) db1[j] = db2[j] = db3[j] = 0.f;
  u4 wr[8];
  for (int tile = blockIdx.x; tile < ntile; tile += gridDim.x) {
    const long row0 = (long)tile * ROWS;
    const int nrow = (int)((B - row0) < ROWS ? (B - row0) : ROWS);
    u4 w1r[4];
    w_load(w1r, wq + QW1);
    {
      // features: thread (row, quarter): 16 values, row-major and transposed
      const int r = threadIdx.x >> 2, q = (threadIdx.x & 3) * 16;
      union {
        u4 v[2];
        bf16 h[16];
      } x;
      x.v[0] = x.v[1] = u4{0, 0, 0, 0};
      if (r < nrow) load_features(Xall + (long)idx[row0 + r] * KIN + q, aligned, x.v);
      u4 *d = reinterpret_cast<u4 *>(L.row + r * LDH + q);
      d[0] = x.v[0];
      d[1] = x.v[1];
#pragma unroll
      for (int i = 0; i < 16; ++i) L.xt[(q + i) * LDR + r] = x.h[i];
    }
    w_store<KIN>(w1r, L.wl, LDH);
    __syncthreads();
    w_load(wr, wq + QW2);
    f4 gd1[H / 16], gd2[H / 16], gd3[H / 16];
    hidden_layer<true>(row, L.wl, LDH, KIN, P + OB1, L.at[0], rb, gd1);
    __syncthreads();
    w_store<H>(wr, L.wl, LDH);
    __syncthreads();
    w_load(wr, wq + QW3);
    hidden_layer<true>(row, L.wl, LDH, H, P + OB2, L.at[1], rb, gd2);
    __syncthreads();
    w_store<H>(wr, L.wl, LDH);
    __syncthreads();
    u4 w4r[1], w4t[1];
    w_load(w4r, wq + QW4);
    w_load(w4t, wq_io + QW4);
    hidden_layer<true>(row, L.wl, LDH, H, P + OB3, L.at[2], rb, gd3);
    __syncthreads();
    w_store<H>(w4r, L.wl, LDH);
    __syncthreads();
    {
      f4 acc[1] = {f4{0, 0, 0, 0}};
      wave_gemm<1>(row, LDH, L.wl, LDH, H, acc);
      const float b = P[OB4 + (l & 15)];
#pragma unroll
      for (int i = 0; i < 4; ++i)
        L.y[(rb + (l >> 4) * 4 + i) * (KOUT + 1) + (l & 15)] = acc[0][i] + b;
    }
    __syncthreads();
    w_store<KOUT>(w4t, L.wl, LDH);
    if (l < 16) {
      const int r = rb + l;
      float *y = L.y + r * (KOUT + 1);
      const float Lr =
          row_loss(y, r < nrow ? tgt + (long)idx[row0 + r] * 8 : nullptr, wT, inv_b);
      if (loss && r < nrow) loss[row0 + r] = Lr;
#pragma unroll
      for (int c = 0; c < KOUT; ++c) {
        const bf16 v = f2bf(y[c]);
        L.row[r * LDH + c] = v;
        L.dzt[c * LDR + r] = v;
      }
    }
    w_load(wr, wq_io + QW3);
    __syncthreads();
    f4 acc[H / 16];
    zero_acc(acc);
    wave_gemm<H / 16>(row, LDH, L.wl, LDH, KOUT, acc);
    wave_gemm<2>(L.dzt, LDR, L.at[2] + w * 32 * LDR, LDR, ROWS, dw4);
    if (threadIdx.x < KOUT)
      for (int r = 0; r < ROWS; ++r) db4 += L.y[r * (KOUT + 1) + threadIdx.x];
    __syncthreads();
    put_dz(acc, gd3, row, L.dzt, rb, db3);
    w_store<H>(wr, L.wl, LDH);
    w_load(wr, wq_io + QW2);
    __syncthreads();
#pragma unroll
    for (int m = 0; m < 2; ++m)
      wave_gemm<H / 16>(L.dzt + (w * 2 + m) * 16 * LDR, LDR, L.at[1], LDR, ROWS, dw3[m]);
    zero_acc(acc);
    wave_gemm<H / 16>(row, LDH, L.wl, LDH, H, acc);
    __syncthreads();
    put_dz(acc, gd2, row, L.dzt, rb, db2);
    w_store<H>(wr, L.wl, LDH);
    __syncthreads();
#pragma unroll
    for (int m = 0; m < 2; ++m)
      wave_gemm<H / 16>(L.dzt + (w * 2 + m) * 16 * LDR, LDR, L.at[0], LDR, ROWS, dw2[m]);
    zero_acc(acc);
    wave_gemm<H / 16>(row, LDH, L.wl, LDH, H, acc);
    __syncthreads();
    put_dz(acc, gd1, row, L.dzt, rb, db1);
    __syncthreads();
#pragma unroll
    for (int m = 0; m < 2; ++m)
      wave_gemm<KIN / 16>(L.dzt + (w * 2 + m) * 16 * LDR, LDR, L.xt, LDR, ROWS, dw1[m]);
    __syncthreads();
  }
  float *out = part + (long)blockIdx.x * NPARAM;
#pragma unroll
  for (int m = 0; m < 2; ++m)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int n = (w * 2 + m) * 16 + (l >> 4) * 4 + i, c = l & 15;
#pragma unroll
      for (int j = 0; j < H / 16; ++j) {
        out[OW3 + n * H + j * 16 + c] = dw3[m][j][i];
        out[OW2 + n * H + j * 16 + c] = dw2[m][j][i];
        if (j < KIN / 16) out[OW1 + n * KIN + j * 16 + c] = dw1[m][j < KIN / 16 ? j : 0][i];
      }
      out[OW4 + ((l >> 4) * 4 + i) * H + (w * 2 + m) * 16 + c] = dw4[m][i];
    }
  // bias gradients: the waves' column sums
  const int ob[3] = {OB1, OB2, OB3};
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    __syncthreads();
    if (l < 16)
#pragma unroll
      for (int j = 0; j < H / 16; ++j)
        L.db[w][j * 16 + l] = k == 0 ? db1[j] : k == 1 ? db2[j] : db3[j];
    __syncthreads();
    if (threadIdx.x < H)
      out[ob[k] + threadIdx.x] = (L.db[0][threadIdx.x] + L.db[1][threadIdx.x]) +
                                 (L.db[2][threadIdx.x] + L.db[3][threadIdx.x]);
  }
  if (threadIdx.x < KOUT) out[OB4 + threadIdx.x] = db4;
}

// sum over blocks of the partials of parameter p, eight at a time
__device__ __forceinline__ float part_sum(const float *__restrict__ part, int nblocks, int p) {
  float s = 0.f;
  int b = 0;
  for (; b + 8 <= nblocks; b += 8) {
    float v[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) v[k] = part[(long)(b + k) * NPARAM + p];
    s += ((v[0] + v[1]) + (v[2] + v[3])) + ((v[4] + v[5]) + (v[6] + v[7]));
  }
  for (; b < nblocks; ++b) s += part[(long)b * NPARAM + p];
  return s;
}
__global__ void __launch_bounds__(64) reduce_kernel(const float *__restrict__ part, int nblocks,
                                                    float *__restrict__ grad) {
  const int p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p < NPARAM) grad[p] = part_sum(part, nblocks, p);
}

// bf16 copies of the weights in both layouts
__device__ inline void write_bf(bf16 *wq, bf16 *wq_io, int p, float v) {
  int q, nout, nin, local;
  if (p < OB1) { q = QW1; nout = H; nin = KIN; local = p - OW1; }
  else if (p >= OW2 && p < OB2) { q = QW2; nout = H; nin = H; local = p - OW2; }
  else if (p >= OW3 && p < OB3) { q = QW3; nout = H; nin = H; local = p - OW3; }
  else if (p >= OW4 && p < OB4) { q = QW4; nout = KOUT; nin = H; local = p - OW4; }
  else return;
  const int n = local / nin, k = local - n * nin;
  const bf16 h = f2bf(v);
  wq[q + local] = h;
  wq_io[q + k * nout + n] = h;
}

// the gradient's last sum and the Adam step
__global__ void __launch_bounds__(64)
    adam_kernel(float *P, float *m, float *v, const float *__restrict__ part, int nblocks,
                bf16 *wq, bf16 *wq_io, float lr, float b1, float b2, float eps, float c1,
                float c2) {
  const int p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= NPARAM) return;
  const float gp = part_sum(part, nblocks, p);
  const float mp = b1 * m[p] + (1.f - b1) * gp;
  const float vp = b2 * v[p] + (1.f - b2) * gp * gp;
  m[p] = mp;
  v[p] = vp;
  const float x = P[p] - lr * (mp / c1) / (sqrtf(vp / c2) + eps);
  P[p] = x;
  write_bf(wq, wq_io, p, x);
}

__global__ void sync_bf_kernel(const float *P, bf16 *wq, bf16 *wq_io) {
  const int p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p < NPARAM) write_bf(wq, wq_io, p, P[p]);
}

// Features of cell c (CSR inputs) -> raw[64]; returns nmat if the cell can be
// described (2..6 materials, registry ids < 6), else 0.
__device__ inline int cell_features(const PteArgs &a, long c, float *raw) {
  for (int i = 0; i < KIN; ++i) raw[i] = 0.f;
  const long o0 = a.offsets[c], o1 = a.offsets[c + 1];
  if (!(o0 >= 0 && o1 >= o0 && o1 <= a.nnz)) return 0;
  const int nm = (int)(o1 - o0);
  if (nm < 2 || nm > SLOTS) return 0;
  double rt = 0;
  for (int s = 0; s < nm; ++s) {
    const int m = a.mat_ids[o0 + s];
    if (m >= SLOTS) return 0;
    const double r = a.rho[o0 + s], al = a.vfrac[o0 + s], T = a.temp[o0 + s];
    if (!(r > 0) || !(al > 0) || !(T > 0)) return 0;
    raw[9 * s + m] = 1.f;
    raw[9 * s + 6] = (float)al;
    raw[9 * s + 7] = (float)log(r);
    raw[9 * s + 8] = (float)log(T);
    rt += r * al;
  }
  raw[54] = (float)asinh(a.sie_tot[c] * 1e-10);
  raw[55] = (float)log(rt);
  return nm;
}

// normalized feature row: active slots and the cell features standardized,
// inactive slots exactly zero
__device__ inline void normalize(const float *raw, int nm, const float *mu, const float *sg,
                                 bf16 *out) {
  for (int i = 0; i < KIN; ++i) {
    const bool on = i < 9 * nm || i == 54 || i == 55;
    out[i] = on && i < NFEAT ? f2bf((raw[i] - mu[i]) / sg[i]) : (bf16)0;
  }
}

__global__ void features_kernel(PteArgs a, const float *mu, const float *sg, float *raw_out,
                                bf16 *X, int *nmat) {
  const long c = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= a.ncell) return;
  float raw[KIN];
  const int nm = cell_features(a, c, raw);
  nmat[c] = nm;
  if (raw_out)
    for (int i = 0; i < KIN; ++i) raw_out[c * KIN + i] = raw[i];
  if (X) {
    bf16 row[KIN];
    normalize(raw, nm, mu, sg, row);
    for (int i = 0; i < KIN; ++i) X[c * KIN + i] = row[i];
  }
}

// training targets from a solved closure: converged alphas per slot (over
// vfrac_tot) and the standardized ln T; nmat 0 for cells left out
__global__ void targets_kernel(PteArgs a, const int *nmat_feat, const int *conv, float t_mu,
                               float t_sg, float *tgt) {
  const long c = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= a.ncell) return;
  float *t = tgt + c * 8;
  for (int i = 0; i < 8; ++i) t[i] = 0.f;
  const int nm = nmat_feat[c];
  if (nm == 0 || !conv[c]) return;
  const long o0 = a.offsets[c];
  const double vt = a.vfrac_tot[c];
  for (int s = 0; s < nm; ++s) t[s] = (float)(a.vfrac[o0 + s] / vt);
  t[6] = ((float)log(a.temp[o0]) - t_mu) / t_sg;
  t[7] = (float)nm;
}

// inference: features, the four layers, softmax -> guesses for the closure.
// A wave takes 16 cells at a time: a lane per cell checks it and forms the
// cell's own features, then a lane per (cell, slot) the slot's; the weights
// stay in LDS for all of the block's tiles (before, a block staged every
// layer's weights for each 64 cells, two bytes at a time, and 64 of its 256
// threads formed the features). 2^18 cells: 1195 -> 203 us.
__global__ void __launch_bounds__(512, 1)
    guess_kernel(PteArgs a, const bf16 *__restrict__ wq, const float *__restrict__ P,
                 const float *__restrict__ mu, const float *__restrict__ sg, float t_mu,
                 float t_sg, double *gv, double *gT) {
  __shared__ InferLds L;
  infer_stage(L, wq);
  const int w = threadIdx.x >> 6, l = threadIdx.x & 63;
  bf16 *row = L.row + w * 16 * LDH;
  for (long t = (long)blockIdx.x * 8 + w; t * 16 < a.ncell; t += (long)gridDim.x * 8) {
    // inactive slots and the padding are zero
    for (int k = l; k < 16 * (KIN / 8); k += 64)
      *reinterpret_cast<u4 *>(row + (k / (KIN / 8)) * LDH + (k % (KIN / 8)) * 8) =
          u4{0, 0, 0, 0};
    wave_handover();
    if (l < 16) {
      const long c = t * 16 + l;
      int nm = 0;
      if (c < a.ncell) {
        const long o0 = a.offsets[c], o1 = a.offsets[c + 1];
        if (o0 >= 0 && o1 >= o0 && o1 <= a.nnz && o1 - o0 >= 2 && o1 - o0 <= SLOTS) {
          nm = (int)(o1 - o0);
          double rt = 0;
          bool ok = true;
          for (int s = 0; s < nm; ++s) {
            const double r = a.rho[o0 + s], al = a.vfrac[o0 + s], T = a.temp[o0 + s];
            ok = ok && a.mat_ids[o0 + s] < SLOTS && r > 0 && al > 0 && T > 0;
            rt += r * al;
          }
          if (ok) {
            row[l * LDH + 54] =
                f2bf(((float)asinh(a.sie_tot[c] * 1e-10) - mu[54]) / sg[54]);
            row[l * LDH + 55] = f2bf(((float)log(rt) - mu[55]) / sg[55]);
          } else {
            nm = 0;
          }
        }
      }
      L.nm[w * 16 + l] = nm;
    }
    wave_handover();
    for (int k = l; k < 16 * SLOTS; k += 64) {
      const int q = k / SLOTS, s = k % SLOTS;
      if (s >= L.nm[w * 16 + q]) continue;
      const long e = a.offsets[t * 16 + q] + s;
      const int m = a.mat_ids[e], f = 9 * s;
      bf16 *x = row + q * LDH + f;
      for (int i = 0; i < SLOTS; ++i)
        x[i] = f2bf(((i == m ? 1.f : 0.f) - mu[f + i]) / sg[f + i]);
      x[6] = f2bf(((float)a.vfrac[e] - mu[f + 6]) / sg[f + 6]);
      x[7] = f2bf(((float)log(a.rho[e]) - mu[f + 7]) / sg[f + 7]);
      x[8] = f2bf(((float)log(a.temp[e]) - mu[f + 8]) / sg[f + 8]);
    }
    wave_handover();
    infer_rows(L, P);
    if (l < 16 && t * 16 + l < a.ncell) {
      const long c = t * 16 + l;
      const int nm = L.nm[w * 16 + l];
      const float *y = L.y + (w * 16 + l) * (KOUT + 1);
      if (nm == 0) {
        gT[c] = __builtin_nan("");
      } else {
        float mx = -1e30f;
        for (int s = 0; s < nm; ++s) mx = fmaxf(mx, y[s]);
        float p[SLOTS], sum = 0.f;
#pragma unroll
        for (int s = 0; s < SLOTS; ++s) {
          p[s] = s < nm ? expf(y[s] - mx) : 0.f;
          sum += p[s];
        }
        const long o0 = a.offsets[c];
        const double vt = a.vfrac_tot[c];
#pragma unroll
        for (int s = 0; s < SLOTS; ++s)
          if (s < nm) gv[o0 + s] = (double)(p[s] / sum) * vt;
        gT[c] = exp((double)(t_mu + t_sg * y[6]));
      }
    }
    wave_handover();
  }
}

} // namespace mlp
} // namespace sgm

using namespace sgm;
using namespace sgm::mlp;

struct sgm_mlp {
  float *P = nullptr, *m = nullptr, *v = nullptr;
  bf16 *wq = nullptr, *wq_io = nullptr;
  float *mu = nullptr, *sg = nullptr;  // [KIN]
  float t_mu = 0.f, t_sg = 1.f;
  int step = 0;
  float *part = nullptr;  // training: the blocks' partial gradients
  int cap = 0;            // blocks it holds
};

namespace {
template <class T>
bool dalloc(T *&p, size_t n) {
  return hipMalloc((void **)&p, sizeof(T) * n) == hipSuccess;
}
void free_ws(sgm_mlp *M) {
  if (M->part) (void)hipFree(M->part);
  M->part = nullptr;
  M->cap = 0;
}
bool ensure_ws(sgm_mlp *M, int nb) {
  if (nb <= M->cap) return true;
  free_ws(M);
  if (!dalloc(M->part, nb * (size_t)NPARAM)) return false;
  M->cap = nb;
  return true;
}
PteArgs csr_args(sgm_ctx *ctx, long ncell, long nnz, const int *off, const uint8_t *mat,
                 const double *rho, const double *vfrac, const double *temp,
                 const double *vfrac_tot, const double *sie_tot) {
  PteArgs a{};
  a.d_eos = ctx ? ctx->d_eos : nullptr;
  a.nreg = ctx ? ctx->nmat : 0;
  a.ncell = ncell;
  a.nnz = nnz;
  a.offsets = off;
  a.mat_ids = mat;
  a.rho = const_cast<double *>(rho);
  a.vfrac = const_cast<double *>(vfrac);
  a.temp = const_cast<double *>(temp);
  a.vfrac_tot = vfrac_tot;
  a.sie_tot = sie_tot;
  return a;
}
int grid1(long n, int bs = 256) { return (int)((n + bs - 1) / bs); }

// forward + loss + backward over rows idx[0..B) into nb partial gradients
int gradients(sgm_mlp *M, const bf16 *X, const float *tgt, const int *idx, long B, float wT,
              float *loss, int &nb, hipStream_t s) {
  const int ntile = (int)((B + ROWS - 1) / ROWS);
  nb = ntile < MAXPART ? ntile : MAXPART;
  if (!ensure_ws(M, nb)) return SGM_E_HIP;
  train_kernel<<<nb, 256, 0, s>>>(M->wq, M->wq_io, M->P, X, tgt, idx, B, ntile, wT,
                                  1.0f / (float)B, M->part, loss);
  return hipGetLastError() == hipSuccess ? SGM_OK : SGM_E_HIP;
}
// blocks of the inference kernels: 128 rows a block and pass, one block a CU
int infer_grid(long n) {
  const long need = (n + IROWS - 1) / IROWS, ncu = device_cu_count();
  return (int)(need < ncu ? need : ncu);
}
} // namespace

extern "C" {

int sgm_mlp_create(uint64_t seed, sgm_mlp **out) {
  if (!out) return SGM_E_ARG;
  *out = nullptr;
  int nd = 0;
  if (hipGetDeviceCount(&nd) != hipSuccess || nd < 1) return SGM_E_NOGPU;
  auto *M = new sgm_mlp();
  bool ok = dalloc(M->P, NPARAM) && dalloc(M->m, NPARAM) && dalloc(M->v, NPARAM) &&
            dalloc(M->wq, NQ) && dalloc(M->wq_io, NQ) &&
            dalloc(M->mu, KIN) && dalloc(M->sg, KIN);
  // He-uniform weights, zero biases
  std::vector<float> h(NPARAM, 0.f), zero(NPARAM, 0.f), ones(KIN, 1.f), zk(KIN, 0.f);
  std::mt19937_64 rng(seed);
  auto fill = [&](int off, int nout, int nin) {
    const double b = std::sqrt(6.0 / nin);
    for (int i = 0; i < nout * nin; ++i) {
      const double u = (double)(rng() >> 11) * (1.0 / 9007199254740992.0);
      h[off + i] = (float)((2 * u - 1) * b);
    }
  };
  fill(OW1, H, KIN);
  fill(OW2, H, H);
  fill(OW3, H, H);
  fill(OW4, KOUT, H);
  ok = ok && hipMemcpy(M->P, h.data(), 4 * NPARAM, hipMemcpyHostToDevice) == hipSuccess &&
       hipMemcpy(M->m, zero.data(), 4 * NPARAM, hipMemcpyHostToDevice) == hipSuccess &&
       hipMemcpy(M->v, zero.data(), 4 * NPARAM, hipMemcpyHostToDevice) == hipSuccess &&
       hipMemcpy(M->mu, zk.data(), 4 * KIN, hipMemcpyHostToDevice) == hipSuccess &&
       hipMemcpy(M->sg, ones.data(), 4 * KIN, hipMemcpyHostToDevice) == hipSuccess;
  if (ok) {
    sync_bf_kernel<<<grid1(NPARAM), 256>>>(M->P, M->wq, M->wq_io);
    ok = hipDeviceSynchronize() == hipSuccess;
  }
  if (!ok) {
    sgm_mlp_destroy(M);
    return SGM_E_HIP;
  }
  *out = M;
  return SGM_OK;
}

int sgm_mlp_destroy(sgm_mlp *M) {
  if (!M) return SGM_E_ARG;
  (void)hipDeviceSynchronize();
  free_ws(M);
  for (float *p : {M->P, M->m, M->v, M->mu, M->sg})
    if (p) (void)hipFree(p);
  if (M->wq) (void)hipFree(M->wq);
  if (M->wq_io) (void)hipFree(M->wq_io);
  delete M;
  return SGM_OK;
}

int sgm_mlp_nparam(void) { return NPARAM; }

int sgm_mlp_params(sgm_mlp *M, float *host_out, const float *host_in) {
  if (!M) return SGM_E_ARG;
  if (host_out && hipMemcpy(host_out, M->P, 4 * NPARAM, hipMemcpyDeviceToHost) != hipSuccess)
    return SGM_E_HIP;
  if (host_in) {
    if (hipMemcpy(M->P, host_in, 4 * NPARAM, hipMemcpyHostToDevice) != hipSuccess)
      return SGM_E_HIP;
    sync_bf_kernel<<<grid1(NPARAM), 256>>>(M->P, M->wq, M->wq_io);
    if (hipDeviceSynchronize() != hipSuccess) return SGM_E_HIP;
  }
  return SGM_OK;
}

int sgm_mlp_set_norm(sgm_mlp *M, const float *mu, const float *sg, float t_mu, float t_sg) {
  if (!M || !mu || !sg || !(t_sg > 0)) return SGM_E_ARG;
  for (int i = 0; i < KIN; ++i)
    if (!(sg[i] > 0)) return SGM_E_ARG;
  if (hipMemcpy(M->mu, mu, 4 * KIN, hipMemcpyHostToDevice) != hipSuccess ||
      hipMemcpy(M->sg, sg, 4 * KIN, hipMemcpyHostToDevice) != hipSuccess)
    return SGM_E_HIP;
  M->t_mu = t_mu;
  M->t_sg = t_sg;
  return SGM_OK;
}

int sgm_mlp_features(sgm_mlp *M, long ncell, long nnz, const int *offsets,
                     const uint8_t *mat_ids, const double *rho, const double *vfrac,
                     const double *temp, const double *sie_tot, float *raw_out, void *X_out,
                     int *nmat_out, sgm_stream_t stream) {
  if (!M || ncell < 0 || !offsets || !mat_ids || !rho || !vfrac || !temp || !sie_tot ||
      !nmat_out)
    return SGM_E_ARG;
  if (ncell == 0) return SGM_OK;
  PteArgs a = csr_args(nullptr, ncell, nnz, offsets, mat_ids, rho, vfrac, temp, nullptr,
                       sie_tot);
  features_kernel<<<grid1(ncell), 256, 0, (hipStream_t)stream>>>(a, M->mu, M->sg, raw_out,
                                                                  (bf16 *)X_out, nmat_out);
  return hipGetLastError() == hipSuccess ? SGM_OK : SGM_E_HIP;
}

int sgm_mlp_targets(sgm_mlp *M, long ncell, long nnz, const int *offsets, const double *vfrac,
                    const double *temp, const double *vfrac_tot, const int *nmat,
                    const int *converged, float *targets, sgm_stream_t stream) {
  if (!M || ncell < 0 || !offsets || !vfrac || !temp || !vfrac_tot || !nmat || !converged ||
      !targets)
    return SGM_E_ARG;
  if (ncell == 0) return SGM_OK;
  PteArgs a = csr_args(nullptr, ncell, nnz, offsets, nullptr, nullptr, vfrac, temp, vfrac_tot,
                       nullptr);
  targets_kernel<<<grid1(ncell), 256, 0, (hipStream_t)stream>>>(a, nmat, converged, M->t_mu,
                                                                 M->t_sg, targets);
  return hipGetLastError() == hipSuccess ? SGM_OK : SGM_E_HIP;
}

int sgm_mlp_gradients(sgm_mlp *M, const void *X, const float *targets, const int *idx,
                      long batch, float wT, float *grad_out, float *loss_out,
                      sgm_stream_t stream) {
  if (!M || !X || !targets || !idx || batch < 1 || batch > (1L << 24)) return SGM_E_ARG;
  hipStream_t s = (hipStream_t)stream;
  int nb = 0;
  const int rc = gradients(M, (const bf16 *)X, targets, idx, batch, wT, loss_out, nb, s);
  if (rc != SGM_OK) return rc;
  if (grad_out) reduce_kernel<<<grid1(NPARAM, 64), 64, 0, s>>>(M->part, nb, grad_out);
  return hipGetLastError() == hipSuccess ? SGM_OK : SGM_E_HIP;
}

int sgm_mlp_train_step(sgm_mlp *M, const void *X, const float *targets, const int *idx,
                       long batch, float wT, float lr, float *loss_out, sgm_stream_t stream) {
  if (!M || !X || !targets || !idx || batch < 1 || batch > (1L << 24) || !(lr >= 0))
    return SGM_E_ARG;
  hipStream_t s = (hipStream_t)stream;
  int nb = 0;
  const int rc = gradients(M, (const bf16 *)X, targets, idx, batch, wT, loss_out, nb, s);
  if (rc != SGM_OK) return rc;
  ++M->step;
  const float b1 = 0.9f, b2 = 0.999f;
  const float c1 = 1.f - std::pow(b1, (float)M->step), c2 = 1.f - std::pow(b2, (float)M->step);
  adam_kernel<<<grid1(NPARAM, 64), 64, 0, s>>>(M->P, M->m, M->v, M->part, nb, M->wq, M->wq_io,
                                               lr, b1, b2, 1e-8f, c1, c2);
  return hipGetLastError() == hipSuccess ? SGM_OK : SGM_E_HIP;
}

int sgm_mlp_forward(sgm_mlp *M, const void *X, const int *idx, long batch, float *Y_out,
                    sgm_stream_t stream) {
  if (!M || !X || !idx || batch < 1 || batch > (1L << 24) || !Y_out) return SGM_E_ARG;
  fwd_kernel<<<infer_grid(batch), 512, 0, (hipStream_t)stream>>>(M->wq, M->P, (const bf16 *)X,
                                                                 idx, batch, Y_out);
  return hipGetLastError() == hipSuccess ? SGM_OK : SGM_E_HIP;
}

int sgm_mlp_guess(sgm_mlp *M, sgm_ctx *ctx, long ncell, long nnz, const int *offsets,
                  const uint8_t *mat_ids, const double *rho, const double *vfrac,
                  const double *temp, const double *vfrac_tot, const double *sie_tot,
                  double *guess_vfrac, double *guess_T, sgm_stream_t stream) {
  if (!M || !ctx || ncell < 0 || !offsets || !mat_ids || !rho || !vfrac || !temp ||
      !vfrac_tot || !sie_tot || !guess_vfrac || !guess_T)
    return SGM_E_ARG;
  if (ctx->host_only) return SGM_E_NOGPU;
  if (ncell == 0) return SGM_OK;
  PteArgs a = csr_args(ctx, ncell, nnz, offsets, mat_ids, rho, vfrac, temp, vfrac_tot, sie_tot);
  guess_kernel<<<infer_grid(ncell), 512, 0, (hipStream_t)stream>>>(
      a, M->wq, M->P, M->mu, M->sg, M->t_mu, M->t_sg, guess_vfrac, guess_T);
  return hipGetLastError() == hipSuccess ? SGM_OK : SGM_E_HIP;
}

} // extern "C"

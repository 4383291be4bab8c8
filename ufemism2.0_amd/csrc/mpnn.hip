// Mesh message-passing network on the triangle graph: the learned Picard
// initial guess.  Inference and training run on the device with hand-written
// kernels; the dense layers use BF16 matrix-core instructions
// (gfx950's mfma_f32_16x16x32_bf16; 16x16x16bf16_1k for the 16-wide layers)
// with FP32 accumulation, everything else is FP32.
//
// Network (nodes = triangles, neighbours = TriC, mean aggregation):
//   h0  = relu(X We + be)                                   X [N,16]  We [16,64]
//   h_l = h_{l-1} + relu([h_{l-1} | mean_nb h_{l-1}] W_l + b_l)    W_l [128,64], l = 1..3
//   y   = h_3 Wd + bd                                       Wd [64,16], outputs 0..2 used
// The outputs are log10 of the speed (m/yr) and the flow direction (x, y;
// normalised when applied), so members whose speeds differ by orders of
// magnitude (A and beta_sq vary over decades) share one scale.  Training
// minimises sum_i ||y_i[0:3] - t_i||^2 / N with Adam (full batch over the
// disjoint union of the training graphs).
//
// Kernels (one workgroup = 4 wavefronts = 64-row tiles, grid-stride; operands
// are converted to bf16 in LDS with the reduction index contiguous, so each
// lane reads its 8 (or 4) consecutive operands with one LDS load):
//   k_layer_fwd     one message-passing layer: the rows of h and the means over
//       the neighbours are gathered straight into the LDS tile of [h | mean];
//       keeps one bit per output for the backward pass (pre-activation > 0)
//   k_rowgemm       encoder and decoder
//   k_decoder_back  loss, dY, gradient of Wd and bd, dH of the last layer
//   k_layer_back    one layer backward: dH (the previous kernel's own part plus
//       the gather of its neighbour part, the adjoint of the mean), dZ, weight
//       and bias gradient of the layer and both parts of the next dH, from one
//       tile; [h | mean] is gathered again instead of being kept
//   k_encoder_back  the same end for the encoder
//   k_reduce_parts  adds the workgroups' partial gradients in a fixed order
// Bound: HBM passes over the [N, 64] fields.  A layer reads and writes two
// fields forward and reads three and writes two backward (N = 160k: 41 MB each);
// with a kernel per operation and Cat, Z, dZ and dCat in memory one gradient took
// 2.66 ms of kernel time at N = 160k, now 0.62 ms (one layer: forward 45 us against
// 144 us, backward 127 us against 495 us).
#include <algorithm>
#include <cmath>
#include <cstring>
#include <memory>
#include <vector>

#include "krylov.h"
#include "ufe_internal.h"

namespace ufe {
namespace mp {

constexpr int kFin = 16, kHid = 64, kFout = 16, kLayers = 3;
constexpr int kTargets = 3;  // trained outputs: log10 speed, direction (x, y)
constexpr int kRows = 64;  // rows per workgroup tile

typedef short bf16x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

// One 16x16 FP32 tile += A (16 x KS) B (KS x 16) on the matrix cores, KS = 32
// (gfx950's v_mfma_f32_16x16x32_bf16: lane l holds A[l % 16][8 (l / 16) ..
// +7] and B[8 (l / 16) .. +7][l % 16]) or KS = 16 (the 16x16x16 shape, for
// the 16-wide layers: lane l holds 4 values from 4 (l / 16)).  p and q point
// at lane l's first A and B values in LDS (16- and 8-byte aligned).
template <int KS>
__device__ __forceinline__ f32x4 mfma_tile(const unsigned short *p, const unsigned short *q, f32x4 acc) {
  if constexpr (KS == 32) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(*reinterpret_cast<const bf16x8 *>(p),
                                                   *reinterpret_cast<const bf16x8 *>(q), acc, 0, 0, 0);
  } else {
    return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(*reinterpret_cast<const bf16x4 *>(p),
                                                     *reinterpret_cast<const bf16x4 *>(q), acc, 0, 0, 0);
  }
}

// float32 -> bfloat16, round to nearest even (gfx950 converts in hardware)
__device__ __forceinline__ unsigned short f2bf(float f) { return __builtin_bit_cast(unsigned short, (__bf16)f); }

// Four consecutive rows of 4 columns (one float4 per row) -> bf16, row-major
// tile of pitch P at (row 4 rg, column 4 c4).
template <int P>
__device__ __forceinline__ void put_rows(unsigned short *t, int rg, int c4, const float4 (&v)[4]) {
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const bf16x4 o = {(short)f2bf(v[q].x), (short)f2bf(v[q].y), (short)f2bf(v[q].z), (short)f2bf(v[q].w)};
    *reinterpret_cast<bf16x4 *>(&t[(4 * rg + q) * P + 4 * c4]) = o;
  }
}

// The same values transposed: column-major tile of pitch P (rows contiguous).
template <int P>
__device__ __forceinline__ void put_cols(unsigned short *t, int rg, int c4, const float4 (&v)[4]) {
  const bf16x4 o0 = {(short)f2bf(v[0].x), (short)f2bf(v[1].x), (short)f2bf(v[2].x), (short)f2bf(v[3].x)};
  const bf16x4 o1 = {(short)f2bf(v[0].y), (short)f2bf(v[1].y), (short)f2bf(v[2].y), (short)f2bf(v[3].y)};
  const bf16x4 o2 = {(short)f2bf(v[0].z), (short)f2bf(v[1].z), (short)f2bf(v[2].z), (short)f2bf(v[3].z)};
  const bf16x4 o3 = {(short)f2bf(v[0].w), (short)f2bf(v[1].w), (short)f2bf(v[2].w), (short)f2bf(v[3].w)};
  *reinterpret_cast<bf16x4 *>(&t[(4 * c4 + 0) * P + 4 * rg]) = o0;
  *reinterpret_cast<bf16x4 *>(&t[(4 * c4 + 1) * P + 4 * rg]) = o1;
  *reinterpret_cast<bf16x4 *>(&t[(4 * c4 + 2) * P + 4 * rg]) = o2;
  *reinterpret_cast<bf16x4 *>(&t[(4 * c4 + 3) * P + 4 * rg]) = o3;
}

__device__ __forceinline__ void add4(float4 &a, const float4 &b) { a.x += b.x; a.y += b.y; a.z += b.z; a.w += b.w; }

// The rows r0 + 4 rg .. + 3 of h and the means over their valid neighbours
// (summed in list order), 4 columns each; zero past the last row.
__device__ __forceinline__ void load_cat(int N, int r0, int rg, int c4, const float4 *__restrict__ H,
                                         const int *__restrict__ nb, float4 (&h)[4], float4 (&m)[4]) {
  int j[4][3];
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int row = r0 + 4 * rg + q;
#pragma unroll
    for (int n = 0; n < 3; ++n) j[q][n] = row < N ? nb[3 * row + n] : -1;
    h[q] = row < N ? H[(size_t)row * (kHid / 4) + c4] : float4{0.0f, 0.0f, 0.0f, 0.0f};
  }
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    float4 s{0.0f, 0.0f, 0.0f, 0.0f};
    int d = 0;
#pragma unroll
    for (int n = 0; n < 3; ++n)
      if (j[q][n] >= 0) {
        add4(s, H[(size_t)j[q][n] * (kHid / 4) + c4]);
        ++d;
      }
    const float f = (float)d;
    m[q] = d ? float4{s.x / f, s.y / f, s.z / f, s.w / f} : float4{0.0f, 0.0f, 0.0f, 0.0f};
  }
}

// Signs of the pre-activations of one wavefront's 16 rows: bit c of mask[row]
// is z(row, c) > 0; pos[t][i] belongs to row 4 (lane / 16) + i, column 16 t +
// lane % 16.  mask is one 64-bit word per row, stored as four 16-bit parts.
__device__ __forceinline__ void put_mask(int N, int row0, int lane, const bool (&pos)[4][4],
                                         unsigned short *__restrict__ mask) {
  const int g = lane >> 4, part = lane & 15;
  unsigned int mine = 0;
#pragma unroll
  for (int t = 0; t < 4; ++t)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const unsigned long long b = __ballot(pos[t][i]);
      if (part == 4 * i + t) mine = (unsigned int)(b >> (16 * g)) & 0xffffu;
    }
  const int row = row0 + 4 * g + (part >> 2);
  if (row < N) mask[4 * (size_t)row + (part & 3)] = (unsigned short)mine;
}

enum { EPI_ENC = 0, EPI_LIN = 2 };

// Out[N,NO] = epi(A[N,K] W + bias); Wt = W^T in bf16, [NO][K].
template <int K, int NO, int EPI>
__global__ void __launch_bounds__(256) k_rowgemm(int N, const float4 *__restrict__ A,
                                                 const unsigned short *__restrict__ Wt,
                                                 const float *__restrict__ bias, unsigned short *__restrict__ mask,
                                                 float *__restrict__ Out) {
  // K steps of 32 where K allows (gfx950's 16x16x32 shape), else of 16; row
  // pitch K + 8 keeps every lane's 16-byte operand aligned and the 16 rows of
  // a step on distinct LDS banks
  constexpr int KS = K % 32 == 0 ? 32 : 16;
  constexpr int KP = K + 8;
  __shared__ __align__(16) unsigned short sA[kRows * KP];
  __shared__ __align__(16) unsigned short sW[NO * KP];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  for (int e = tid; e < NO * K; e += 256) sW[(e / K) * KP + (e % K)] = Wt[e];
  const int ar = wave * 16 + (lane & 15);
  const int kq = (KS / 4) * (lane >> 4);
  for (int tile = blockIdx.x; tile * kRows < N; tile += gridDim.x) {
    const int r0 = tile * kRows;
    __syncthreads();
#pragma unroll
    for (int e = tid; e < kRows * K / 4; e += 256) {
      const int r = e / (K / 4), c4 = e % (K / 4), row = r0 + r;
      const float4 v = row < N ? A[(size_t)row * (K / 4) + c4] : float4{0.0f, 0.0f, 0.0f, 0.0f};
      const bf16x4 o = {(short)f2bf(v.x), (short)f2bf(v.y), (short)f2bf(v.z), (short)f2bf(v.w)};
      *reinterpret_cast<bf16x4 *>(&sA[r * KP + 4 * c4]) = o;
    }
    __syncthreads();
    f32x4 acc[NO / 16];
#pragma unroll
    for (int t = 0; t < NO / 16; ++t) acc[t] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int kb = 0; kb < K; kb += KS) {
#pragma unroll
      for (int t = 0; t < NO / 16; ++t)
        acc[t] = mfma_tile<KS>(&sA[ar * KP + kb + kq], &sW[(t * 16 + (lane & 15)) * KP + kb + kq], acc[t]);
    }
    // lane holds rows 4*(lane/16)+i, column lane%16 of each 16x16 tile
    [[maybe_unused]] bool pos[4][4];
#pragma unroll
    for (int t = 0; t < NO / 16; ++t) {
      const int col = t * 16 + (lane & 15);
      const float bc = bias[col];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int row = r0 + wave * 16 + 4 * (lane >> 4) + i;
        const float z = acc[t][i] + bc;
        if constexpr (EPI == EPI_ENC) pos[t][i] = z > 0.0f;
        if (row < N) Out[(size_t)row * NO + col] = EPI == EPI_ENC ? fmaxf(z, 0.0f) : z;
      }
    }
    if constexpr (EPI == EPI_ENC) put_mask(N, r0 + wave * 16, lane, pos, mask);
  }
}

// Out = H + relu([H | mean_nb H] W + b), mask = signs of the pre-activations;
// Wt = W^T in bf16, [64][128].
__global__ void __launch_bounds__(256) k_layer_fwd(int N, const float4 *__restrict__ H, const int *__restrict__ nb,
                                                   const unsigned short *__restrict__ Wt,
                                                   const float *__restrict__ bias, unsigned short *__restrict__ mask,
                                                   float *__restrict__ Out) {
  constexpr int K = 2 * kHid, KP = K + 8;
  __shared__ __align__(16) unsigned short sA[kRows * KP];
  __shared__ __align__(16) unsigned short sW[kHid * KP];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, rg = tid >> 4, c4 = tid & 15;
  for (int e = tid; e < kHid * K / 8; e += 256)
    *reinterpret_cast<bf16x8 *>(&sW[(e / (K / 8)) * KP + 8 * (e % (K / 8))]) =
        reinterpret_cast<const bf16x8 *>(Wt)[e];
  const int ar = wave * 16 + (lane & 15), kq = 8 * (lane >> 4);
  const float *Hf = reinterpret_cast<const float *>(H);
  for (int tile = blockIdx.x; tile * kRows < N; tile += gridDim.x) {
    const int r0 = tile * kRows;
    float4 h[4], m[4];
    load_cat(N, r0, rg, c4, H, nb, h, m);
    __syncthreads();  // the previous tile's operand reads
    put_rows<KP>(sA, rg, c4, h);
    put_rows<KP>(sA + kHid, rg, c4, m);
    __syncthreads();
    f32x4 acc[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) acc[t] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int kb = 0; kb < K; kb += 32)
#pragma unroll
      for (int t = 0; t < 4; ++t)
        acc[t] = mfma_tile<32>(&sA[ar * KP + kb + kq], &sW[(t * 16 + (lane & 15)) * KP + kb + kq], acc[t]);
    bool pos[4][4];
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const int col = t * 16 + (lane & 15);
      const float bc = bias[col];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int row = r0 + wave * 16 + 4 * (lane >> 4) + i;
        const float z = acc[t][i] + bc;
        pos[t][i] = z > 0.0f;
        const size_t o = (size_t)row * kHid + col;
        if (row < N) Out[o] = Hf[o] + fmaxf(z, 0.0f);
      }
    }
    put_mask(N, r0 + wave * 16, lane, pos, mask);
  }
}

// Accumulates A^T B over a tile's 64 rows into this wavefront's 16x16 tiles of
// the K x NO product; At [K][RP] and Bt [NO][RP] hold the rows contiguously.
constexpr int kRP = kRows + 8;
template <int K, int NO>
constexpr int col_tiles() { return ((K / 16) * (NO / 16) + 3) / 4; }
template <int K, int NO>
__device__ __forceinline__ void col_product(const unsigned short *At, const unsigned short *Bt, int wave, int lane,
                                            f32x4 (&acc)[col_tiles<K, NO>()]) {
  constexpr int TN = NO / 16, TT = (K / 16) * TN, PER = col_tiles<K, NO>();
#pragma unroll
  for (int q = 0; q < PER; ++q) {
    const int t = wave * PER + q;
    if (t < TT) {
      const int tm = t / TN, tn = t % TN, kq = 8 * (lane >> 4);
#pragma unroll
      for (int rb = 0; rb < kRows; rb += 32)
        acc[q] = mfma_tile<32>(&At[(tm * 16 + (lane & 15)) * kRP + rb + kq],
                               &Bt[(tn * 16 + (lane & 15)) * kRP + rb + kq], acc[q]);
    }
  }
}

// This workgroup's partial gradient: [K * NO] weights, then NO column sums
// (col[c] summed over the workgroup's 16 row groups through LDS).
template <int K, int NO>
__device__ __forceinline__ void put_partial(int wave, int lane, const f32x4 (&acc)[col_tiles<K, NO>()], float4 bsum,
                                            float *red /* [16][NO] LDS */, float *__restrict__ part) {
  constexpr int TN = NO / 16, TT = (K / 16) * TN, PER = col_tiles<K, NO>();
  const int tid = threadIdx.x, rg = tid / (NO / 4), c4 = tid % (NO / 4);
  float *out = part + (size_t)blockIdx.x * (K * NO + NO);
#pragma unroll
  for (int q = 0; q < PER; ++q) {
    const int t = wave * PER + q;
    if (t < TT) {
      const int tm = t / TN, tn = t % TN;
#pragma unroll
      for (int i = 0; i < 4; ++i) out[(tm * 16 + 4 * (lane >> 4) + i) * NO + tn * 16 + (lane & 15)] = acc[q][i];
    }
  }
  constexpr int RG = 256 / (NO / 4);  // row groups
  __syncthreads();
  *reinterpret_cast<float4 *>(&red[rg * NO + 4 * c4]) = bsum;
  __syncthreads();
  if (tid < NO) {
    float t = 0.0f;
    for (int q = 0; q < RG; ++q) t += red[q * NO + tid];
    out[K * NO + tid] = t;
  }
}

// Loss, decoder gradient and dH of the last layer: dY = 2 (Y[:, 0:3] - T) / N
// (other columns 0), partial sums of Wd's gradient H^T dY and of the squared
// error, dH = dY Wd^T.  Wn = Wd in bf16, [64][16].
__global__ void __launch_bounds__(256) k_decoder_back(int N, const float4 *__restrict__ Y, const float *__restrict__ T,
                                                      const float4 *__restrict__ H,
                                                      const unsigned short *__restrict__ Wn, float *__restrict__ dH,
                                                      float *__restrict__ part, float *__restrict__ lpart) {
  constexpr int YP = kFout + 8;
  __shared__ __align__(16) unsigned short sY[kRows * YP], sYt[kFout * kRP], sHt[kHid * kRP], sW[kHid * YP];
  __shared__ __align__(16) float red[64 * kFout];
  __shared__ float sl[4];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, rg = tid >> 4, c4 = tid & 15;
  for (int e = tid; e < kHid * kFout; e += 256) sW[(e / kFout) * YP + (e % kFout)] = Wn[e];
  const float s = 2.0f / (float)N;
  f32x4 acc[col_tiles<kHid, kFout>()];
  acc[0] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  float4 bsum{0.0f, 0.0f, 0.0f, 0.0f};
  float se = 0.0f;
  for (int tile = blockIdx.x; tile * kRows < N; tile += gridDim.x) {
    const int r0 = tile * kRows;
    float4 h[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int row = r0 + 4 * rg + q;
      h[q] = row < N ? H[(size_t)row * (kHid / 4) + c4] : float4{0.0f, 0.0f, 0.0f, 0.0f};
    }
    // one thread per (row, four outputs)
    const int yr = tid >> 2, yc = tid & 3, yrow = r0 + yr;
    float4 d{0.0f, 0.0f, 0.0f, 0.0f};
    if (yc == 0 && yrow < N) {
      const float4 y = Y[(size_t)yrow * (kFout / 4)];
      const float *t = T + (size_t)kTargets * yrow;
      const float d0 = y.x - t[0], d1 = y.y - t[1], d2 = y.z - t[2];
      se += d0 * d0 + d1 * d1 + d2 * d2;
      d = float4{s * d0, s * d1, s * d2, 0.0f};
    }
    add4(bsum, d);
    __syncthreads();
    put_cols<kRP>(sHt, rg, c4, h);
    const unsigned short b0 = f2bf(d.x), b1 = f2bf(d.y), b2 = f2bf(d.z), b3 = f2bf(d.w);
    const bf16x4 o = {(short)b0, (short)b1, (short)b2, (short)b3};
    *reinterpret_cast<bf16x4 *>(&sY[yr * YP + 4 * yc]) = o;
    sYt[(4 * yc + 0) * kRP + yr] = b0;
    sYt[(4 * yc + 1) * kRP + yr] = b1;
    sYt[(4 * yc + 2) * kRP + yr] = b2;
    sYt[(4 * yc + 3) * kRP + yr] = b3;
    __syncthreads();
    col_product<kHid, kFout>(sHt, sYt, wave, lane, acc);
#pragma unroll
    for (int t = 0; t < kHid / 16; ++t) {
      const f32x4 z = mfma_tile<16>(&sY[(wave * 16 + (lane & 15)) * YP + 4 * (lane >> 4)],
                                    &sW[(t * 16 + (lane & 15)) * YP + 4 * (lane >> 4)], f32x4{0.0f, 0.0f, 0.0f, 0.0f});
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int row = r0 + wave * 16 + 4 * (lane >> 4) + i;
        if (row < N) dH[(size_t)row * kHid + t * 16 + (lane & 15)] = z[i];
      }
    }
  }
  se = wave_sum(se);
  if (lane == 0) sl[wave] = se;
  put_partial<kHid, kFout>(wave, lane, acc, bsum, red, part);
  if (tid == 0) lpart[blockIdx.x] = sl[0] + sl[1] + sl[2] + sl[3];
}

// dH of the rows r0 + 4 rg .. + 3: the own part plus, from the second layer on,
// the neighbours' parts G (already divided by their degrees) in list order.
template <bool HAS_G>
__device__ __forceinline__ void load_dh(int N, int r0, int rg, int c4, const float4 *__restrict__ dH,
                                        const float4 *__restrict__ G, const int *__restrict__ nb, float4 (&v)[4]) {
  int j[4][3];
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int row = r0 + 4 * rg + q;
    v[q] = row < N ? dH[(size_t)row * (kHid / 4) + c4] : float4{0.0f, 0.0f, 0.0f, 0.0f};
    if (HAS_G)
#pragma unroll
      for (int n = 0; n < 3; ++n) j[q][n] = row < N ? nb[3 * row + n] : -1;
  }
  if (HAS_G)
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
      for (int n = 0; n < 3; ++n)
        if (j[q][n] >= 0) add4(v[q], G[(size_t)j[q][n] * (kHid / 4) + c4]);
}

// dZ = dH where the pre-activation was positive
__device__ __forceinline__ void apply_mask(int N, int r0, int rg, int c4, const unsigned short *__restrict__ mask,
                                           float4 (&v)[4]) {
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int row = r0 + 4 * rg + q;
    const unsigned int b = row < N ? mask[4 * (size_t)row + (c4 >> 2)] >> (4 * (c4 & 3)) : 0u;
    v[q].x = b & 1u ? v[q].x : 0.0f;
    v[q].y = b & 2u ? v[q].y : 0.0f;
    v[q].z = b & 4u ? v[q].z : 0.0f;
    v[q].w = b & 8u ? v[q].w : 0.0f;
  }
}

// One layer backward (file comment).  Wn = W in bf16, [128][64]; dHout = dH +
// dCat[:, 0:64], Gout = dCat[:, 64:128] / degree.
template <bool HAS_G>
__global__ void __launch_bounds__(256) k_layer_back(int N, const float4 *__restrict__ dH, const float4 *__restrict__ G,
                                                    const int *__restrict__ nb,
                                                    const unsigned short *__restrict__ mask,
                                                    const float4 *__restrict__ H,
                                                    const unsigned short *__restrict__ Wn, float *__restrict__ dHout,
                                                    float *__restrict__ Gout, float *__restrict__ part) {
  constexpr int K = 2 * kHid, ZP = kHid + 8, DP = kHid + 4;
  __shared__ __align__(16) unsigned short sW[K * ZP], sZ[kRows * ZP], sZt[kHid * kRP], sCt[K * kRP];
  __shared__ __align__(16) float sD[kRows * DP];
  __shared__ float sdeg[kRows];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, rg = tid >> 4, c4 = tid & 15;
  for (int e = tid; e < K * kHid / 8; e += 256)
    *reinterpret_cast<bf16x8 *>(&sW[(e / (kHid / 8)) * ZP + 8 * (e % (kHid / 8))]) =
        reinterpret_cast<const bf16x8 *>(Wn)[e];
  f32x4 acc[col_tiles<K, kHid>()];
#pragma unroll
  for (int q = 0; q < col_tiles<K, kHid>(); ++q) acc[q] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  float4 bsum{0.0f, 0.0f, 0.0f, 0.0f};
  for (int tile = blockIdx.x; tile * kRows < N; tile += gridDim.x) {
    const int r0 = tile * kRows;
    float4 v[4], h[4], m[4];
    load_dh<HAS_G>(N, r0, rg, c4, dH, G, nb, v);
    load_cat(N, r0, rg, c4, H, nb, h, m);
    __syncthreads();  // the previous tile's reads
    if (tid < kRows) {
      const int row = r0 + tid;
      int d = 0;
      if (row < N)
        for (int n = 0; n < 3; ++n) d += nb[3 * row + n] >= 0;
      sdeg[tid] = (float)d;
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) *reinterpret_cast<float4 *>(&sD[(4 * rg + q) * DP + 4 * c4]) = v[q];
    apply_mask(N, r0, rg, c4, mask, v);
#pragma unroll
    for (int q = 0; q < 4; ++q) add4(bsum, v[q]);
    put_rows<ZP>(sZ, rg, c4, v);
    put_cols<kRP>(sZt, rg, c4, v);
    put_cols<kRP>(sCt, rg, c4, h);
    put_cols<kRP>(sCt + kHid * kRP, rg, c4, m);
    __syncthreads();
    col_product<K, kHid>(sCt, sZt, wave, lane, acc);
    const int ar = wave * 16 + (lane & 15), kq = 8 * (lane >> 4);
#pragma unroll
    for (int t = 0; t < K / 16; ++t) {
      f32x4 z = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int kb = 0; kb < kHid; kb += 32)
        z = mfma_tile<32>(&sZ[ar * ZP + kb + kq], &sW[(t * 16 + (lane & 15)) * ZP + kb + kq], z);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int r = wave * 16 + 4 * (lane >> 4) + i, row = r0 + r;
        if (row >= N) continue;
        if (t < kHid / 16) {
          const int c = t * 16 + (lane & 15);
          dHout[(size_t)row * kHid + c] = sD[r * DP + c] + z[i];
        } else {
          // a node without neighbours is read by none
          Gout[(size_t)row * kHid + (t - kHid / 16) * 16 + (lane & 15)] = sdeg[r] > 0.0f ? z[i] / sdeg[r] : 0.0f;
        }
      }
    }
  }
  put_partial<K, kHid>(wave, lane, acc, bsum, sD, part);
}

// Encoder gradient: dZ from the first layer's dH, X^T dZ and its column sums.
__global__ void __launch_bounds__(256) k_encoder_back(int N, const float4 *__restrict__ dH,
                                                      const float4 *__restrict__ G, const int *__restrict__ nb,
                                                      const unsigned short *__restrict__ mask,
                                                      const float4 *__restrict__ X, float *__restrict__ part) {
  __shared__ __align__(16) unsigned short sXt[kFin * kRP], sZt[kHid * kRP];
  __shared__ __align__(16) float red[16 * kHid];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, rg = tid >> 4, c4 = tid & 15;
  f32x4 acc[col_tiles<kFin, kHid>()];
  acc[0] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  float4 bsum{0.0f, 0.0f, 0.0f, 0.0f};
  for (int tile = blockIdx.x; tile * kRows < N; tile += gridDim.x) {
    const int r0 = tile * kRows;
    float4 v[4];
    load_dh<true>(N, r0, rg, c4, dH, G, nb, v);
    apply_mask(N, r0, rg, c4, mask, v);
#pragma unroll
    for (int q = 0; q < 4; ++q) add4(bsum, v[q]);
    const int xr = tid >> 2, xc = tid & 3;
    const float4 x = r0 + xr < N ? X[(size_t)(r0 + xr) * (kFin / 4) + xc] : float4{0.0f, 0.0f, 0.0f, 0.0f};
    __syncthreads();
    put_cols<kRP>(sZt, rg, c4, v);
    sXt[(4 * xc + 0) * kRP + xr] = f2bf(x.x);
    sXt[(4 * xc + 1) * kRP + xr] = f2bf(x.y);
    sXt[(4 * xc + 2) * kRP + xr] = f2bf(x.z);
    sXt[(4 * xc + 3) * kRP + xr] = f2bf(x.w);
    __syncthreads();
    col_product<kFin, kHid>(sXt, sZt, wave, lane, acc);
  }
  put_partial<kFin, kHid>(wave, lane, acc, bsum, red, part);
}

// Sum over the workgroups' partials part[p * len + e]: elements below n go to
// w[e], the rest to b[e - n].  A wavefront takes 64 elements of every 16th
// partial, the 16 sums are added in order.
constexpr int kReduceWaves = 16;
__global__ void __launch_bounds__(64 * kReduceWaves) k_reduce_parts(int nparts, int len, int n,
                                                                    const float *__restrict__ part,
                                                                    float *__restrict__ w, float *__restrict__ b) {
  __shared__ float red[kReduceWaves][64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, e = blockIdx.x * 64 + lane;
  float s = 0.0f;
  if (e < len) {
#pragma unroll 8
    for (int p = wave; p < nparts; p += kReduceWaves) s += part[(size_t)p * len + e];
  }
  red[wave][lane] = s;
  __syncthreads();
  if (wave == 0 && e < len) {
    float t = 0.0f;
    for (int q = 0; q < kReduceWaves; ++q) t += red[q][lane];
    if (e < n) w[e] = t;
    else b[e - n] = t;
  }
}

// Neighbour lists must be symmetric (j in nb(i) <=> i in nb(j)) and in range:
// the gathers rely on it, so this runs before any of them.
__global__ void __launch_bounds__(256) k_check_graph(int N, const int *__restrict__ nb, int *__restrict__ bad) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= N) return;
  bool ok = true;
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    const int j = nb[3 * i + a];
    if (j < -1 || j >= N) {
      ok = false;
    } else if (j >= 0) {
      ok = ok && (nb[3 * j] == i || nb[3 * j + 1] == i || nb[3 * j + 2] == i);
    }
  }
  if (!ok) *bad = 1;
}

// W [K, NO] fp32 -> Wt [NO][K] bf16 (forward operand) and Wn [K][NO] bf16
// (operand of the input-gradient product)
__global__ void __launch_bounds__(256) k_weights_bf16(int K, int NO, const float *__restrict__ W,
                                                      unsigned short *__restrict__ Wt, unsigned short *__restrict__ Wn) {
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= K * NO) return;
  const int k = e / NO, n = e % NO;
  const unsigned short b = f2bf(W[e]);
  Wt[n * K + k] = b;
  Wn[e] = b;
}

__global__ void __launch_bounds__(256) k_adam(int n, float *__restrict__ w, const float *__restrict__ g,
                                              float *__restrict__ m, float *__restrict__ v, float lr, float b1,
                                              float b2, float eps, float c1, float c2) {
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= n) return;
  const float gi = g[e];
  const float mi = b1 * m[e] + (1.0f - b1) * gi;
  const float vi = b2 * v[e] + (1.0f - b2) * gi * gi;
  m[e] = mi;
  v[e] = vi;
  w[e] -= lr * (mi / c1) / (sqrtf(vi / c2) + eps);
}

// ---------------------------------------------------------------------------
// Host side
// ---------------------------------------------------------------------------

// Parameter layout in one fp32 vector.
struct Layout {
  size_t We, be, W[kLayers], b[kLayers], Wd, bd, total;
  Layout() {
    size_t o = 0;
    We = o; o += kFin * kHid;
    be = o; o += kHid;
    for (int l = 0; l < kLayers; ++l) {
      W[l] = o; o += 2 * kHid * kHid;
      b[l] = o; o += kHid;
    }
    Wd = o; o += kHid * kFout;
    bd = o; o += kFout;
    total = o;
  }
};

// persistent workgroups of the tile kernels: k_layer_back's 71 KB of LDS
// (72,960 bytes) leave room for two per CU, and each adds one partial gradient
// to sum
constexpr int kMaxParts = 512;
inline int grid_rows(int N) { return std::max(1, std::min((N + kRows - 1) / kRows, 4 * kMaxParts)); }
inline int grid_parts(int N) { return std::min(grid_rows(N), kMaxParts); }
inline int grid_elems(long n) { return (int)std::max<long>(1, (n + 255) / 256); }

}  // namespace mp
}  // namespace ufe

using namespace ufe;
using namespace ufe::mp;

struct ufe_mpnn {
  int device = 0;
  hipStream_t s = nullptr;
  Layout L;
  DBuf w, g, m, v, wt16, wn16, part;
  int step = 0;
  // graph buffers (sized for the largest N seen)
  int cap = 0;
  DBuf X, nb, T, H[kLayers + 1], mask[kLayers + 1], Y, dH[2], G[2], lpart;
  int *bad = nullptr;  // pinned: set by the graph check
  std::string err;
  ~ufe_mpnn() {
    if (bad) (void)hipHostFree(bad);
  }

  size_t wt_off(size_t woff) const { return woff; }  // bf16 copies share the fp32 offsets

  void ensure(int N) {
    if (N <= cap) return;
    cap = N;
    size_t n = (size_t)N;
    X.alloc(n * kFin * 4);
    nb.alloc(n * 3 * 4);
    T.alloc(n * kTargets * 4);
    for (auto &b : H) b.alloc(n * kHid * 4);
    for (auto &b : mask) b.alloc(n * kHid / 8);
    Y.alloc(n * kFout * 4);
    for (auto &b : dH) b.alloc(n * kHid * 4);
    for (auto &b : G) b.alloc(n * kHid * 4);
    lpart.alloc(kMaxParts * 4);
  }

  void refresh_bf16() {
    auto conv = [&](size_t off, int K, int NO) {
      hipLaunchKernelGGL(k_weights_bf16, dim3(grid_elems((long)K * NO)), dim3(256), 0, s, K, NO,
                         w.as<float>() + off, wt16.as<unsigned short>() + off, wn16.as<unsigned short>() + off);
      UFE_LAUNCH_CHECK();
    };
    conv(L.We, kFin, kHid);
    for (int l = 0; l < kLayers; ++l) conv(L.W[l], 2 * kHid, kHid);
    conv(L.Wd, kHid, kFout);
  }

  const unsigned short *wt(size_t off) const { return wt16.as<unsigned short>() + off; }
  const unsigned short *wn(size_t off) const { return wn16.as<unsigned short>() + off; }
  const float *wf(size_t off) const { return w.as<float>() + off; }

  // forward over N nodes already in X / nb
  void forward(int N) {
    const int *n3 = nb.as<int>();
    const int gr = grid_rows(N);
    hipLaunchKernelGGL((k_rowgemm<kFin, kHid, EPI_ENC>), dim3(gr), dim3(256), 0, s, N, X.as<float4>(), wt(L.We),
                       wf(L.be), mask[0].as<unsigned short>(), H[0].as<float>());
    UFE_LAUNCH_CHECK();
    for (int l = 0; l < kLayers; ++l) {
      hipLaunchKernelGGL(k_layer_fwd, dim3(gr), dim3(256), 0, s, N, H[l].as<float4>(), n3, wt(L.W[l]), wf(L.b[l]),
                         mask[l + 1].as<unsigned short>(), H[l + 1].as<float>());
      UFE_LAUNCH_CHECK();
    }
    hipLaunchKernelGGL((k_rowgemm<kHid, kFout, EPI_LIN>), dim3(gr), dim3(256), 0, s, N, H[kLayers].as<float4>(),
                       wt(L.Wd), wf(L.bd), (unsigned short *)nullptr, Y.as<float>());
    UFE_LAUNCH_CHECK();
  }

  // gradient of a K x NO weight block and its bias from the workgroups' partials
  void reduce(int nparts, int K, int NO, size_t woff, size_t boff) {
    const int len = K * NO + NO;
    hipLaunchKernelGGL(k_reduce_parts, dim3((len + 63) / 64), dim3(64 * kReduceWaves), 0, s, nparts, len, K * NO,
                       part.as<float>(), g.as<float>() + woff, g.as<float>() + boff);
    UFE_LAUNCH_CHECK();
  }

  // loss and gradient for the N nodes in X / nb / T; returns the loss
  float loss_grad(int N) {
    forward(N);
    const int gp = grid_parts(N);
    const int *n3 = nb.as<int>();
    float *pt = part.as<float>();
    hipLaunchKernelGGL(k_decoder_back, dim3(gp), dim3(256), 0, s, N, Y.as<float4>(), T.as<float>(),
                       H[kLayers].as<float4>(), wn(L.Wd), dH[0].as<float>(), pt, lpart.as<float>());
    UFE_LAUNCH_CHECK();
    reduce(gp, kHid, kFout, L.Wd, L.bd);
    int cur = 0;
    for (int l = kLayers - 1; l >= 0; --l, cur ^= 1) {
      const unsigned short *mk = mask[l + 1].as<unsigned short>();
      if (l == kLayers - 1)
        hipLaunchKernelGGL(k_layer_back<false>, dim3(gp), dim3(256), 0, s, N, dH[cur].as<float4>(),
                           (const float4 *)nullptr, n3, mk, H[l].as<float4>(), wn(L.W[l]), dH[cur ^ 1].as<float>(),
                           G[cur ^ 1].as<float>(), pt);
      else
        hipLaunchKernelGGL(k_layer_back<true>, dim3(gp), dim3(256), 0, s, N, dH[cur].as<float4>(),
                           G[cur].as<float4>(), n3, mk, H[l].as<float4>(), wn(L.W[l]), dH[cur ^ 1].as<float>(),
                           G[cur ^ 1].as<float>(), pt);
      UFE_LAUNCH_CHECK();
      reduce(gp, 2 * kHid, kHid, L.W[l], L.b[l]);
    }
    hipLaunchKernelGGL(k_encoder_back, dim3(gp), dim3(256), 0, s, N, dH[cur].as<float4>(), G[cur].as<float4>(), n3,
                       mask[0].as<unsigned short>(), X.as<float4>(), pt);
    UFE_LAUNCH_CHECK();
    reduce(gp, kFin, kHid, L.We, L.be);
    float lp[kMaxParts];
    UFE_HIP(hipMemcpyAsync(lp, lpart.p, sizeof(float) * gp, hipMemcpyDeviceToHost, s));
    UFE_HIP(hipStreamSynchronize(s));
    double tot = 0.0;
    for (int i = 0; i < gp; ++i) tot += lp[i];
    return (float)(tot / N);
  }

  void adam(float lr) {
    ++step;
    const float b1 = 0.9f, b2 = 0.999f;
    const float c1 = 1.0f - std::pow(b1, (float)step), c2 = 1.0f - std::pow(b2, (float)step);
    hipLaunchKernelGGL(k_adam, dim3(grid_elems((long)L.total)), dim3(256), 0, s, (int)L.total, w.as<float>(),
                       g.as<float>(), m.as<float>(), v.as<float>(), lr, b1, b2, 1e-8f, c1, c2);
    UFE_LAUNCH_CHECK();
    refresh_bf16();
  }

  void upload_graph(int N, const float *Xh, const int *nbh, const float *Th) {
    ensure(N);
    UFE_HIP(hipMemcpyAsync(X.p, Xh, sizeof(float) * kFin * (size_t)N, hipMemcpyHostToDevice, s));
    UFE_HIP(hipMemcpyAsync(nb.p, nbh, sizeof(int) * 3 * (size_t)N, hipMemcpyHostToDevice, s));
    if (Th) UFE_HIP(hipMemcpyAsync(T.p, Th, sizeof(float) * kTargets * (size_t)N, hipMemcpyHostToDevice, s));
  }

  // whether the neighbour lists in nb are in range and symmetric
  bool graph_ok(int N) {
    *bad = 0;
    hipLaunchKernelGGL(k_check_graph, dim3(grid_elems(N)), dim3(256), 0, s, N, nb.as<int>(), bad);
    UFE_LAUNCH_CHECK();
    UFE_HIP(hipStreamSynchronize(s));
    return *bad == 0;
  }
};

namespace {

int mp_fail(ufe_mpnn *n, int code, const std::string &msg) {
  if (n) n->err = msg;
  set_global_error(msg);
  return code;
}

template <typename F>
int mp_guard(ufe_mpnn *n, F &&f) {
  try {
    return f();
  } catch (const HipError &e) {
    return mp_fail(n, UFE_ERR_DEVICE, e.what());
  } catch (const std::exception &e) {
    return mp_fail(n, UFE_ERR_ARGUMENT, e.what());
  }
}

constexpr const char *kBadGraph = "neighbour lists must be in range and symmetric";

}  // namespace

extern "C" int ufe_mpnn_num_weights(void) { return (int)Layout().total; }

extern "C" int ufe_mpnn_create(ufe_mpnn **out, int device, const float *weights) {
  if (!out) return mp_fail(nullptr, UFE_ERR_ARGUMENT, "null argument");
  auto n = std::make_unique<ufe_mpnn>();
  int rc = mp_guard(n.get(), [&]() -> int {
    n->device = device;
    UFE_HIP(hipSetDevice(device));
    UFE_HIP(hipStreamCreateWithFlags(&n->s, hipStreamNonBlocking));
    const size_t P = n->L.total;
    n->w.alloc(P * 4);
    n->g.alloc(P * 4);
    n->m.alloc(P * 4);
    n->v.alloc(P * 4);
    n->wt16.alloc(P * 2);
    n->wn16.alloc(P * 2);
    // partials: the largest block (128x64 + 64) of every workgroup
    n->part.alloc(sizeof(float) * (size_t)kMaxParts * (2 * kHid * kHid + kHid));
    UFE_HIP(hipHostMalloc((void **)&n->bad, sizeof(int), hipHostMallocDefault));
    UFE_HIP(hipMemsetAsync(n->g.p, 0, P * 4, n->s));
    UFE_HIP(hipMemsetAsync(n->m.p, 0, P * 4, n->s));
    UFE_HIP(hipMemsetAsync(n->v.p, 0, P * 4, n->s));
    if (weights) UFE_HIP(hipMemcpyAsync(n->w.p, weights, P * 4, hipMemcpyHostToDevice, n->s));
    else UFE_HIP(hipMemsetAsync(n->w.p, 0, P * 4, n->s));
    n->refresh_bf16();
    UFE_HIP(hipStreamSynchronize(n->s));
    return UFE_OK;
  });
  if (rc != UFE_OK) return rc;
  *out = n.release();
  return UFE_OK;
}

extern "C" int ufe_mpnn_destroy(ufe_mpnn *n) {
  if (!n) return UFE_OK;
  (void)hipSetDevice(n->device);
  if (n->s) (void)hipStreamSynchronize(n->s);
  hipStream_t s = n->s;
  delete n;
  if (s) (void)hipStreamDestroy(s);
  return UFE_OK;
}

extern "C" int ufe_mpnn_get_weights(ufe_mpnn *n, float *weights) {
  if (!n || !weights) return mp_fail(n, UFE_ERR_ARGUMENT, "null argument");
  return mp_guard(n, [&]() -> int {
    UFE_HIP(hipSetDevice(n->device));
    UFE_HIP(hipMemcpyAsync(weights, n->w.p, n->L.total * 4, hipMemcpyDeviceToHost, n->s));
    UFE_HIP(hipStreamSynchronize(n->s));
    return UFE_OK;
  });
}

extern "C" int ufe_mpnn_forward(ufe_mpnn *n, int N, const float *X, const int *nb, float *Y) {
  if (!n || N < 1 || !X || !nb || !Y) return mp_fail(n, UFE_ERR_ARGUMENT, "invalid argument");
  return mp_guard(n, [&]() -> int {
    UFE_HIP(hipSetDevice(n->device));
    n->upload_graph(N, X, nb, nullptr);
    if (!n->graph_ok(N)) return mp_fail(n, UFE_ERR_ARGUMENT, kBadGraph);
    n->forward(N);
    UFE_HIP(hipMemcpyAsync(Y, n->Y.p, sizeof(float) * kFout * (size_t)N, hipMemcpyDeviceToHost, n->s));
    UFE_HIP(hipStreamSynchronize(n->s));
    return UFE_OK;
  });
}

extern "C" int ufe_mpnn_loss_grad(ufe_mpnn *n, int N, const float *X, const int *nb, const float *T, float *loss,
                                  float *grad) {
  if (!n || N < 1 || !X || !nb || !T || !loss) return mp_fail(n, UFE_ERR_ARGUMENT, "invalid argument");
  return mp_guard(n, [&]() -> int {
    UFE_HIP(hipSetDevice(n->device));
    n->upload_graph(N, X, nb, T);
    if (!n->graph_ok(N)) return mp_fail(n, UFE_ERR_ARGUMENT, kBadGraph);
    *loss = n->loss_grad(N);
    if (grad) {
      UFE_HIP(hipMemcpyAsync(grad, n->g.p, n->L.total * 4, hipMemcpyDeviceToHost, n->s));
      UFE_HIP(hipStreamSynchronize(n->s));
    }
    return UFE_OK;
  });
}

extern "C" int ufe_mpnn_train(ufe_mpnn *n, int N, const float *X, const int *nb, const float *T, int steps,
                              float lr, float *loss_history) {
  if (!n || N < 1 || !X || !nb || !T || steps < 0 || !(lr > 0.0f))
    return mp_fail(n, UFE_ERR_ARGUMENT, "invalid argument");
  return mp_guard(n, [&]() -> int {
    UFE_HIP(hipSetDevice(n->device));
    n->upload_graph(N, X, nb, T);
    if (!n->graph_ok(N)) return mp_fail(n, UFE_ERR_ARGUMENT, kBadGraph);
    for (int it = 0; it < steps; ++it) {
      float l = n->loss_grad(N);
      if (loss_history) loss_history[it] = l;
      if (!std::isfinite(l)) return mp_fail(n, UFE_ERR_DIVERGED, "training loss is not finite");
      n->adam(lr);
    }
    UFE_HIP(hipStreamSynchronize(n->s));
    return UFE_OK;
  });
}

// ---------------------------------------------------------------------------
// Inference inside a solver context (features from the uploaded inputs).
// ---------------------------------------------------------------------------
namespace ufe {
namespace mp {
int ctx_features(ufe_ctx *c, float *X_dev, int *nb_dev, hipStream_t *s_out, int *N_out);
int ctx_set_guess(ufe_ctx *c, const float *Y_dev);
}  // namespace mp
}  // namespace ufe

extern "C" int ufe_mpnn_initial_guess(ufe_ctx *c, ufe_mpnn *n) {
  if (!c || !n) return mp_fail(n, UFE_ERR_ARGUMENT, "null argument");
  return mp_guard(n, [&]() -> int {
    UFE_HIP(hipSetDevice(n->device));
    int N = 0;
    hipStream_t cs;
    // first call sizes the buffers
    int rc = ufe::mp::ctx_features(c, nullptr, nullptr, &cs, &N);
    if (rc != UFE_OK) return rc;
    n->ensure(N);
    UFE_HIP(hipStreamSynchronize(n->s));
    rc = ufe::mp::ctx_features(c, n->X.as<float>(), n->nb.as<int>(), &cs, &N);
    if (rc != UFE_OK) return rc;
    UFE_HIP(hipStreamSynchronize(cs));
    n->forward(N);
    UFE_HIP(hipStreamSynchronize(n->s));
    return ufe::mp::ctx_set_guess(c, n->Y.as<float>());
  });
}

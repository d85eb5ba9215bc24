// Neural radiance cache MLP on the gfx950 matrix cores.
//
// Fully fused: one wave runs a tile of queries through every layer, the
// activations staying in registers between layers (training, which needs
// them again, keeps them in LDS).  Every product is a
// v_mfma_f32_16x16x32_bf16 (16x16 tile, K = 32, bf16 operands, fp32
// accumulation).  Operand layout of that instruction, lane l = 16 g + r:
//   A (16 x 32): row r, k = 8 g .. 8 g + 7      (one 16-byte load)
//   B (32 x 16): column r, k = 8 g .. 8 g + 7   (one 16-byte load)
//   D (16 x 16): column r, rows 4 g .. 4 g + 3  (4 fp32 registers)
// so an operand is read where its K index is contiguous: weights
// row-major (out, in) for the forward pass, their transposes for the
// backward pass, activations query-major [q][n] as the B operand of the
// next layer and neuron-major [n][q] (K = queries) for the weight
// gradients.
//
// Network (include/ospray_hip/hip_nrc.h): 160 -> 64 -> 64 -> 64 -> 64 -> 3,
// ReLU, no biases (input 156 is a constant 1).  Loss: relative L2,
// mean over queries and channels of (y - t)^2 / (y^2 + 0.01), the
// denominator held constant.  Training writes one gradient row per tile;
// the Adam kernel sums the rows in tile order (deterministic).
#include <hip/hip_runtime.h>

#include "ospray_hip/hip_nrc.h"
#include "pt_math.h"

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kIn = HPT_NRC_INPUTS, kH = HPT_NRC_HIDDEN, kOP = 16, kP = HPT_NRC_PARAMS;
// element offsets of W0..W4 in the weights, of W1^T..W4^T in the transposes
__constant__ const int kOff[5] = {0, 10240, 14336, 18432, 22528};
__constant__ const int kOffT[4] = {0, 4096, 8192, 12288};
constexpr int kS = 72; // LDS row stride (bf16) of 64-wide rows: 144 B, 16-byte aligned
constexpr int kDyS = 40; // row stride of the query-major output gradient (32 used)
constexpr float kLossEps = 0.01f;

__device__ __forceinline__ f32x4 mma(const bf16x8 &a, const bf16x8 &b, const f32x4 &c)
{
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ bf16x8 ld8(const __bf16 *p) { return *reinterpret_cast<const bf16x8 *>(p); }
__device__ __forceinline__ bf16x8 zero8()
{
  bf16x8 z;
  for (int i = 0; i < 8; i++)
    z[i] = (__bf16)0.f;
  return z;
}
__device__ __forceinline__ f32x4 zero4() { return f32x4{0.f, 0.f, 0.f, 0.f}; }

// max(x, 0), 0 for a NaN, in one instruction: fmaxf quiets x in another one
// first, and so does a median with a bound that the compiler sees as infinity
__device__ __forceinline__ float relu(float x)
{
  float inf = __builtin_inff();
  asm("" : "+s"(inf));
  return __builtin_amdgcn_fmed3f(x, 0.f, inf);
}

// The D operand that a product leaves in lane (r, g) holds rows 16 nt + 4 g ..
// + 3 of its A operand, and the next product takes from that lane the neurons
// 32 kb + 8 g .. + 7.  The weight rows of layers 0..3 are therefore handed to
// the matrix cores in this order: row s is neuron rowNeuron(s), so that tiles
// 2 kb and 2 kb + 1 leave a lane its eight neurons, and no activation goes
// through LDS.  Each sum runs over its inputs in their own order, as in the
// training kernel.
__device__ __forceinline__ int rowNeuron(int s) { return (s & 32) + ((s & 12) << 1) + ((s & 16) >> 2) + (s & 3); }
__device__ __forceinline__ int neuronRow(int n) { return (n & 32) + ((n & 4) << 2) + ((n & 24) >> 1) + (n & 3); }

// x of the lane N further on in the row of 16
template <int N>
__device__ __forceinline__ float rotated(float x)
{
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x120 + N, 0xf, 0xf, false)); // row_ror
}

// Layers 1..4 of the forward pass in registers.
// acc[nt][qt]: layer 0's sums in, o[qt]: W4 (16 x 64) x h4; rows 0..2 are
// the outputs.  wf(layer, nt, kb) loads an A operand (of W4: nt 0, its own
// rows).
template <int QT, typename WF>
__device__ __forceinline__ void forwardTail(const WF &wf, f32x4 (&acc)[4][QT], f32x4 (&o)[QT])
{
  bf16x8 h[2][QT];
#pragma unroll
  for (int l = 1; l <= 4; l++) {
    for (int kb = 0; kb < 2; kb++)
      for (int qt = 0; qt < QT; qt++)
        for (int e = 0; e < 4; e++) {
          h[kb][qt][e] = (__bf16)relu(acc[2 * kb][qt][e]);
          h[kb][qt][4 + e] = (__bf16)relu(acc[2 * kb + 1][qt][e]);
        }
    if (l == 4)
      break;
    for (int nt = 0; nt < 4; nt++) {
      for (int qt = 0; qt < QT; qt++)
        acc[nt][qt] = zero4();
      for (int kb = 0; kb < 2; kb++) {
        const bf16x8 a = wf(l, nt, kb);
        for (int qt = 0; qt < QT; qt++)
          acc[nt][qt] = mma(a, h[kb][qt], acc[nt][qt]);
      }
    }
  }
  for (int qt = 0; qt < QT; qt++)
    o[qt] = zero4();
  for (int kb = 0; kb < 2; kb++) {
    const bf16x8 a = wf(4, 0, kb);
    for (int qt = 0; qt < QT; qt++)
      o[qt] = mma(a, h[kb][qt], o[qt]);
  }
}

__global__ __launch_bounds__(64) void k_nrc_infer(HptNrc N, const __bf16 *X, int n, float *out)
{
  const int lane = threadIdx.x, r = lane & 15, g = lane >> 4;
  const __bf16 *W = reinterpret_cast<const __bf16 *>(N.w);
  const auto wf = [&](int l, int nt, int kb) {
    return ld8(W + kOff[l] + (l < 4 ? rowNeuron(nt * 16 + r) : r) * kH + kb * 32 + g * 8);
  };
  for (int tile = blockIdx.x; tile * 64 < n; tile += gridDim.x) {
    const int q0 = tile * 64;
    f32x4 acc[4][4];
    for (int nt = 0; nt < 4; nt++)
      for (int qt = 0; qt < 4; qt++)
        acc[nt][qt] = zero4();
    for (int kb = 0; kb < kIn / 32; kb++) {
      bf16x8 b[4];
      for (int qt = 0; qt < 4; qt++) {
        const int q = q0 + qt * 16 + r;
        b[qt] = q < n ? ld8(X + (size_t)q * kIn + kb * 32 + g * 8) : zero8();
      }
      for (int nt = 0; nt < 4; nt++) {
        const bf16x8 a = ld8(W + rowNeuron(nt * 16 + r) * kIn + kb * 32 + g * 8);
        for (int qt = 0; qt < 4; qt++)
          acc[nt][qt] = mma(a, b[qt], acc[nt][qt]);
      }
    }
    f32x4 o[4];
    forwardTail<4>(wf, acc, o);
    if (g == 0)
      for (int qt = 0; qt < 4; qt++) {
        const int q = q0 + qt * 16 + r;
        if (q < n) {
          out[3 * (size_t)q] = o[qt][0];
          out[3 * (size_t)q + 1] = o[qt][1];
          out[3 * (size_t)q + 2] = o[qt][2];
        }
      }
  }
}

// One tile of 64 (features, target) pairs per block iteration: forward,
// relative-L2 gradient, backward; the tile's weight gradients go to row
// `tile` of N.partial, its loss to N.tileLoss[tile].
//
// A training step has few tiles (256 for 16,384 records, one a CU), so a
// tile's chain of layers sets its time: four waves share a tile, wave w
// owning rows 16 w .. 16 w + 15 of every layer (queries 16 w .. of the
// output layer), with every weight fragment it will need, forward and
// transposed, loaded before the first layer.  Each output element's sums, and
// the tile's loss, run over the same operands in the same order as with one
// wave.  256 tiles:
// 39.8 -> 21.8 us.
constexpr int kSX = 168; // LDS row stride (bf16) of the query-major features
__global__ __launch_bounds__(256) void k_nrc_train(HptNrc N, const __bf16 *X, const float *T, int n)
{
  __shared__ __attribute__((aligned(16))) __bf16 xq[64 * kSX]; // [q][k]
  __shared__ __attribute__((aligned(16))) __bf16 xT[kIn * kS]; // [k][q]
  __shared__ __attribute__((aligned(16))) __bf16 hT[4][kH * kS]; // h1..h4, [n][q]
  __shared__ __attribute__((aligned(16))) __bf16 act[64 * kS]; // [q][n]; backward: dz [q][n]
  __shared__ __attribute__((aligned(16))) __bf16 dzT[kH * kS]; // [n][q]
  __shared__ __attribute__((aligned(16))) __bf16 dyT[kOP * kS]; // [c][q]
  __shared__ __attribute__((aligned(16))) __bf16 dy[64 * kDyS]; // [q][c], c < 32
  __shared__ float lossTerms[3 * 64]; // [q][c]
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
  const __bf16 *W = reinterpret_cast<const __bf16 *>(N.w);
  const __bf16 *WT = reinterpret_cast<const __bf16 *>(N.wT);
  const float scale = 1.f / (3.f * (float)n);
  const int row = wave * 16 + r; // this lane's weight row in the A operands
  bf16x8 w0[kIn / 32], wh[3][2], wo[2], wt[3][2], wt4;
  for (int kb = 0; kb < kIn / 32; kb++)
    w0[kb] = ld8(W + row * kIn + kb * 32 + g * 8);
  for (int l = 0; l < 3; l++)
    for (int kb = 0; kb < 2; kb++) {
      wh[l][kb] = ld8(W + kOff[l + 1] + row * kH + kb * 32 + g * 8);
      wt[l][kb] = ld8(WT + kOffT[l] + row * kH + kb * 32 + g * 8);
    }
  for (int kb = 0; kb < 2; kb++)
    wo[kb] = ld8(W + kOff[4] + r * kH + kb * 32 + g * 8);
  wt4 = ld8(WT + kOffT[3] + row * 32 + g * 8);
  // relu(acc) of this wave's 16 neurons in bf16 to act[q][n] and hl[n][q]
  const int n0 = wave * 16 + 4 * g;
  auto store = [&](const f32x4 (&acc)[4], __bf16 *hl) {
    for (int qt = 0; qt < 4; qt++) {
      const int q = qt * 16 + r;
      bf16x4 v;
      for (int e = 0; e < 4; e++) {
        v[e] = (__bf16)fmaxf(acc[qt][e], 0.f);
        hl[(n0 + e) * kS + q] = v[e];
      }
      *reinterpret_cast<bf16x4 *>(act + q * kS + n0) = v;
    }
  };
  for (int tile = blockIdx.x; tile * 64 < n; tile += gridDim.x) {
    const int q0 = tile * 64;
    float *grad = N.partial + (size_t)tile * kP;
    { // the tile's features, query-major and transposed
      const int q = threadIdx.x >> 2, qg = q0 + q;
      for (int j = 0; j < kIn / 32; j++) {
        const int c = (threadIdx.x & 3) + 4 * j;
        const bf16x8 v = qg < n ? ld8(X + (size_t)qg * kIn + c * 8) : zero8();
        *reinterpret_cast<bf16x8 *>(xq + q * kSX + c * 8) = v;
        for (int i = 0; i < 8; i++)
          xT[(c * 8 + i) * kS + q] = v[i];
      }
    }
    // the targets of this wave's output queries
    const int qo = wave * 16 + r, qog = q0 + qo;
    float t3[3] = {0.f, 0.f, 0.f};
    if (g == 0 && qog < n)
      for (int e = 0; e < 3; e++)
        t3[e] = T[3 * (size_t)qog + e];
    __syncthreads();
    // forward
    f32x4 acc[4];
    for (int qt = 0; qt < 4; qt++) {
      acc[qt] = zero4();
      for (int kb = 0; kb < kIn / 32; kb++)
        acc[qt] = mma(w0[kb], ld8(xq + (qt * 16 + r) * kSX + kb * 32 + g * 8), acc[qt]);
    }
    store(acc, hT[0]);
    __syncthreads();
    for (int l = 0; l < 3; l++) {
      for (int qt = 0; qt < 4; qt++) {
        acc[qt] = zero4();
        for (int kb = 0; kb < 2; kb++)
          acc[qt] = mma(wh[l][kb], ld8(act + (qt * 16 + r) * kS + kb * 32 + g * 8), acc[qt]);
      }
      __syncthreads();
      store(acc, hT[l + 1]);
      __syncthreads();
    }
    // output gradient dy = 2 (y - t) / (y^2 + eps) / (3 n) in rows 0..2
    {
      f32x4 o = zero4();
      for (int kb = 0; kb < 2; kb++)
        o = mma(wo[kb], ld8(act + qo * kS + kb * 32 + g * 8), o);
      bf16x4 dv;
      for (int e = 0; e < 4; e++) {
        float d = 0.f, loss = 0.f;
        if (g == 0 && e < 3 && qog < n) {
          const float y = o[e], t = t3[e];
          const float den = y * y + kLossEps;
          d = 2.f * (y - t) / den * scale;
          loss = (y - t) * (y - t) / den * scale;
        }
        if (g == 0 && e < 3)
          lossTerms[3 * qo + e] = loss;
        dv[e] = (__bf16)d;
        dyT[(4 * g + e) * kS + qo] = dv[e];
        dy[qo * kDyS + 16 + 4 * g + e] = (__bf16)0.f;
      }
      *reinterpret_cast<bf16x4 *>(dy + qo * kDyS + 4 * g) = dv;
    }
    __syncthreads();
    if (threadIdx.x < 16) { // the tile's loss: queries r, r + 16, .. in order, then r + 8, 4, 2, 1
      float loss = 0.f;
      for (int qt = 0; qt < 4; qt++)
        for (int e = 0; e < 3; e++)
          loss += lossTerms[3 * (qt * 16 + r) + e];
      loss += rotated<8>(loss);
      loss += rotated<4>(loss);
      loss += rotated<2>(loss);
      loss += rotated<1>(loss);
      if (r == 0)
        N.tileLoss[tile] = loss;
    }
    { // dW4 (16 x 64) = dy^T h4: this wave's 16 columns
      f32x4 a4 = zero4();
      for (int kb = 0; kb < 2; kb++)
        a4 = mma(ld8(dyT + r * kS + kb * 32 + g * 8), ld8(hT[3] + row * kS + kb * 32 + g * 8), a4);
      for (int e = 0; e < 4; e++)
        grad[kOff[4] + (4 * g + e) * kH + row] = a4[e];
    }
    // dz4 = (W4^T dy) * [h4 > 0]
    for (int qt = 0; qt < 4; qt++)
      acc[qt] = mma(wt4, ld8(dy + (qt * 16 + r) * kDyS + g * 8), zero4());
#pragma unroll
    for (int l = 3; l >= 0; l--) {
      // mask with the layer's input activation, store dz both ways (the
      // previous layer's readers of act and dzT are behind a barrier)
      for (int qt = 0; qt < 4; qt++) {
        const int q = qt * 16 + r;
        bf16x4 v;
        for (int e = 0; e < 4; e++) {
          const float h = (float)hT[l][(n0 + e) * kS + q];
          v[e] = (__bf16)(h > 0.f ? acc[qt][e] : 0.f);
          dzT[(n0 + e) * kS + q] = v[e];
        }
        *reinterpret_cast<bf16x4 *>(act + q * kS + n0) = v;
      }
      __syncthreads();
      // dh_l = W_l^T dz, masked by h_l in the next iteration
      if (l > 0)
        for (int qt = 0; qt < 4; qt++) {
          acc[qt] = zero4();
          for (int kb = 0; kb < 2; kb++)
            acc[qt] = mma(wt[l - 1][kb], ld8(act + (qt * 16 + r) * kS + kb * 32 + g * 8), acc[qt]);
        }
      // dW_l (64 x K_in) = dz h_l^T, h_0 = x: this wave's 16 rows
      const int kin = l ? kH : kIn;
      const __bf16 *hin = l ? hT[l ? l - 1 : 0] : xT;
      bf16x8 z[2];
      for (int kb = 0; kb < 2; kb++)
        z[kb] = ld8(dzT + row * kS + kb * 32 + g * 8);
      for (int jt = 0; jt < kin / 16; jt++) {
        f32x4 a4 = zero4();
        for (int kb = 0; kb < 2; kb++)
          a4 = mma(z[kb], ld8(hin + (jt * 16 + r) * kS + kb * 32 + g * 8), a4);
        for (int e = 0; e < 4; e++)
          grad[kOff[l] + (n0 + e) * kin + jt * 16 + r] = a4[e];
      }
      __syncthreads();
    }
  }
}

// parameter p of the flat layout -> (layer, row, column)
__device__ __forceinline__ void paramIndex(int p, int &l, int &row, int &col)
{
  l = p < 10240 ? 0 : (p < 14336 ? 1 : (p < 18432 ? 2 : (p < 22528 ? 3 : 4)));
  const int k = l ? kH : kIn;
  const int o = p - kOff[l];
  row = o / k;
  col = o - row * k;
}

__device__ __forceinline__ void writeWeight(const HptNrc &N, int p, float w)
{
  int l, row, col;
  paramIndex(p, l, row, col);
  if (l == 4 && row >= HPT_NRC_OUTPUTS)
    w = 0.f; // padded output rows stay zero
  N.master[p] = w;
  const __bf16 b = (__bf16)w;
  reinterpret_cast<__bf16 *>(N.w)[p] = b;
  if (l >= 1) // transposes: W_l^T [in][out], W4^T [64][32]
    reinterpret_cast<__bf16 *>(N.wT)[kOffT[l - 1] + col * (l == 4 ? 32 : kH) + row] = b;
}

__global__ __launch_bounds__(256) void k_nrc_init(HptNrc N, uint32_t seed)
{
  for (int p = blockIdx.x * blockDim.x + threadIdx.x; p < kP; p += gridDim.x * blockDim.x) {
    int l, row, col;
    paramIndex(p, l, row, col);
    // PCG-style hash of (seed, p) -> uniform [0, 1)
    uint64_t s = (uint64_t)seed * 0x9E3779B97F4A7C15ull + (uint64_t)p * 0xD1B54A32D192ED03ull + 1442695040888963407ull;
    s ^= s >> 33;
    s *= 0xff51afd7ed558ccdull;
    s ^= s >> 33;
    s *= 0xc4ceb9fe1a85ec53ull;
    s ^= s >> 33;
    const float u = (float)(uint32_t)(s >> 40) * (1.f / 16777216.f);
    const float lim = sqrtf(6.f / (float)(l ? kH : kIn));
    N.adamM[p] = 0.f;
    N.adamV[p] = 0.f;
    writeWeight(N, p, (2.f * u - 1.f) * lim);
  }
  // W4^T columns 16..31: zero
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < kH * 16; i += gridDim.x * blockDim.x)
    reinterpret_cast<__bf16 *>(N.wT)[kOffT[3] + (i / 16) * 32 + 16 + (i & 15)] = (__bf16)0.f;
}

// 64 parameters per block.  Their sums over the tiles' gradient rows run in a
// fixed order: of four groups, group k adds tiles k, k + 4, ... in turn, then
// (0 + 1) + (2 + 3).  The rows (94 KB a tile) come from HBM, and with one wave
// a group (64 rows each of 256 tiles, a few in flight) a step took 35.2 us,
// 0.69 TB/s.  Four waves share a group: each has kAdamRows of its rows in
// flight at once, and they add theirs to the group's sum one after another,
// which keeps the order and costs a barrier each: 6.9 us, 3.5 TB/s (sixteen
// groups, an order of their own, 6.4).
constexpr int kAdamGroups = 4, kAdamSegs = 4, kAdamRows = 16;
__global__ __launch_bounds__(64 * kAdamGroups * kAdamSegs) void k_nrc_adam(HptNrc N, int tiles, float lr, float bc1, float bc2)
{
  __shared__ float part[kAdamGroups][64];
  const int col = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int grp = wave % kAdamGroups, seg = wave / kAdamGroups;
  if (blockIdx.x == kP / 64) { // the last block: the tiles' losses in order
    constexpr int kLosses = 64 * kAdamGroups * kAdamSegs;
    __shared__ float losses[kLosses];
    float L = 0.f;
    for (int t0 = 0; t0 < tiles; t0 += kLosses) {
      const int t = t0 + (int)threadIdx.x;
      losses[threadIdx.x] = t < tiles ? N.tileLoss[t] : 0.f;
      __syncthreads();
      if (wave == 0)
        for (int k = 0; k < min(kLosses, tiles - t0); k += 64) {
          const int x = __float_as_int(losses[k + col]);
#pragma unroll
          for (int i = 0; i < 64; i++) // (a lane past the last tile adds 0)
            L += __int_as_float(__builtin_amdgcn_readlane(x, i));
        }
      __syncthreads();
    }
    if (threadIdx.x == 0)
      N.loss[0] = L;
    return;
  }
  const int p = blockIdx.x * 64 + col;
  float m0 = 0.f, v0 = 0.f, w0 = 0.f; // on their way beside the rows
  if (wave == 0) {
    m0 = N.adamM[p];
    v0 = N.adamV[p];
    w0 = N.master[p];
  }
  for (int t0 = 0; t0 < tiles; t0 += kAdamGroups * kAdamSegs * kAdamRows) {
    const int first = t0 + seg * kAdamGroups * kAdamRows + grp;
    float x[kAdamRows] = {};
    if (first < tiles) {
#pragma unroll
      for (int i = 0; i < kAdamRows; i++) { // loads without a branch between them
        const int t = first + kAdamGroups * i;
        const float v = N.partial[(size_t)min(t, tiles - 1) * kP + p];
        x[i] = t < tiles ? v : 0.f;
      }
    }
    for (int s = 0; s < kAdamSegs && t0 + s * kAdamGroups * kAdamRows < tiles; s++) {
      if (t0 + s > 0)
        __syncthreads();
      if (seg == s) {
        float gs = t0 + s > 0 ? part[grp][col] : 0.f;
#pragma unroll
        for (int i = 0; i < kAdamRows; i++)
          gs += x[i];
        part[grp][col] = gs;
      }
    }
  }
  __syncthreads();
  if (wave == 0) {
    const float g = (part[0][col] + part[1][col]) + (part[2][col] + part[3][col]);
    const float m = 0.9f * m0 + 0.1f * g;
    const float v = 0.99f * v0 + 0.01f * g * g;
    N.adamM[p] = m;
    N.adamV[p] = v;
    writeWeight(N, p, w0 - lr * (m / bc1) / (sqrtf(v / bc2) + 1e-8f));
  }
}

// feature group j (0..19: 8 features) of a query whose raw inputs are
// position, direction, normal, albedo (raw12): groups 0..17 hold 4 bands
// x (sin, cos) of coordinate j / 3 (position mapped over [lo, hi], then
// direction); 18 and 19 the albedo, normal, mapped position, direction, 1.
// j may differ across lanes: the coordinate is picked by selects, so the
// raw inputs stay in registers.
__device__ __forceinline__ bf16x8 encodeGroup(const float (&raw12)[12], int j, const float lo[3], const float inv[3])
{
  const float px = (raw12[0] - lo[0]) * inv[0], py = (raw12[1] - lo[1]) * inv[1], pz = (raw12[2] - lo[2]) * inv[2];
  bf16x8 v;
  if (j < 18) {
    const int d = j / 3, h = j - 3 * d;
    float c = px;
    c = d == 1 ? py : c;
    c = d == 2 ? pz : c;
    c = d == 3 ? raw12[3] : c;
    c = d == 4 ? raw12[4] : c;
    c = d == 5 ? raw12[5] : c;
    // band 4h directly, the next three by the double-angle formulas
    // sin 2x = 2 sin x cos x, cos 2x = (cos x - sin x)(cos x + sin x)
    float sn, cs;
    hpt::fsincos((float)(1 << (4 * h)) * hpt::kPi * c, sn, cs);
    for (int b = 0; b < 4; b++) {
      v[2 * b] = (__bf16)sn;
      v[2 * b + 1] = (__bf16)cs;
      const float s2 = 2.f * sn * cs, c2 = (cs - sn) * (cs + sn);
      sn = s2;
      cs = c2;
    }
    return v;
  }
  const bool first = j == 18;
  const float t[8] = {first ? raw12[9] : pz, first ? raw12[10] : raw12[3], first ? raw12[11] : raw12[4],
      first ? raw12[6] : raw12[5], first ? raw12[7] : 1.f, first ? raw12[8] : 0.f, first ? px : 0.f,
      first ? py : 0.f};
  for (int b = 0; b < 8; b++)
    v[b] = (__bf16)t[b];
  return v;
}

__global__ __launch_bounds__(256) void k_nrc_encode(const float *raw, int n, float lx, float ly, float lz, float hx,
    float hy, float hz, __bf16 *X)
{
  const float lo[3] = {lx, ly, lz}, inv[3] = {1.f / (hx - lx), 1.f / (hy - ly), 1.f / (hz - lz)};
  for (int q = blockIdx.x * blockDim.x + threadIdx.x; q < n; q += gridDim.x * blockDim.x) {
    float rq[12];
    for (int k = 0; k < 12; k++)
      rq[k] = raw[12 * (size_t)q + k];
    bf16x8 *out = reinterpret_cast<bf16x8 *>(X + (size_t)q * kIn);
    for (int j = 0; j < kIn / 8; j++)
      out[j] = encodeGroup(rq, j, lo, inv);
  }
}

// The path tracer's cache queries in one kernel: gather the queued vertex
// records (per path slot: P, thr.x | wo, thr.y | Ns, thr.z | albedo, -),
// encode them in registers, run the network with the weights staged once
// per block in LDS, and add throughput * max(prediction, 0) to the path's
// contribution.  A wave takes 16 queries at a time.
//
// The encoding's VALU work bounds it.  LDS holds the weights only, their
// rows padded (16 rows of one K chunk on distinct banks), so three blocks of
// eight waves fit a CU, and a wave's 16 queries keep a short call short.
// 573,245 queries: with activations in LDS (one block a CU), 64 queries a
// wave and unpadded rows 98.7 us; without the three 64 queries 63.7, 32
// queries 46.4, 16 queries 42.9.  1,000 queries: 18.6, 12.6, 8.5, 5.7.
constexpr int kQueryWaves = 8, kQueryBlocks = 3; // waves a block, blocks a CU
constexpr int kW0S = 168, kWS = 72; // LDS row strides (bf16) of W0 and of W1..W4
__global__ __launch_bounds__(64 * kQueryWaves, 6) void k_nrc_query(HptNrc N, const float *rec16, const uint32_t *queue,
    int n, float lx, float ly, float lz, float hx, float hy, float hz, float *contrib4)
{
  __shared__ __attribute__((aligned(16))) __bf16 wl[64 * kW0S + 208 * kWS];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
  {
    const bf16x8 *src = reinterpret_cast<const bf16x8 *>(N.w);
    for (int i = threadIdx.x; i < kP / 8; i += 64 * kQueryWaves) {
      const bf16x8 v = src[i];
      if (i < kH * kIn / 8) {
        const int row = i / (kIn / 8);
        *reinterpret_cast<bf16x8 *>(wl + neuronRow(row) * kW0S + (i - row * (kIn / 8)) * 8) = v;
      } else { // W1..W4: 208 rows of 64, W4's as they are
        const int j = i - kH * kIn / 8, row = j >> 3;
        const int at = row < 3 * kH ? (row & ~(kH - 1)) + neuronRow(row & (kH - 1)) : row;
        *reinterpret_cast<bf16x8 *>(wl + 64 * kW0S + at * kWS + (j & 7) * 8) = v;
      }
    }
  }
  __syncthreads();
  const auto wf = [&](int l, int nt, int kb) {
    return ld8(wl + 64 * kW0S + ((l - 1) * kH + nt * 16 + r) * kWS + kb * 32 + g * 8);
  };
  const float lo[3] = {lx, ly, lz}, inv[3] = {1.f / (hx - lx), 1.f / (hy - ly), 1.f / (hz - lz)};
  const int step = gridDim.x * kQueryWaves * 16;
  int q0 = (blockIdx.x * kQueryWaves + wave) * 16;
  uint32_t pNext = q0 < n ? queue[min(q0 + r, n - 1)] : 0u;
  for (; q0 < n; q0 += step) {
    asm volatile("" ::: "memory"); // weights stay in LDS: in registers they leave two waves a SIMD
    const int q = q0 + r; // this lane's query (column r of the products)
    const bool valid = q < n;
    const uint32_t p = pNext;
    if (q0 + step < n)
      pNext = queue[min(q + step, n - 1)];
    const float *rec = rec16 + 16 * (size_t)p;
    float raw[12], thr[3];
    for (int k = 0; k < 4; k++) {
      const float4 v = *reinterpret_cast<const float4 *>(rec + 4 * k);
      raw[3 * k] = v.x;
      raw[3 * k + 1] = v.y;
      raw[3 * k + 2] = v.z;
      if (k < 3)
        thr[k] = v.w;
    }
    f32x4 acc[4][1];
    for (int nt = 0; nt < 4; nt++)
      acc[nt][0] = zero4();
    for (int kb = 0; kb < kIn / 32; kb++) {
      const bf16x8 b = encodeGroup(raw, 4 * kb + g, lo, inv);
      for (int nt = 0; nt < 4; nt++)
        acc[nt][0] = mma(ld8(wl + (nt * 16 + r) * kW0S + kb * 32 + g * 8), b, acc[nt][0]);
    }
    f32x4 o[1];
    forwardTail<1>(wf, acc, o);
    if (g == 0 && valid) {
      float *c = contrib4 + 4 * (size_t)p;
      for (int k = 0; k < 3; k++)
        c[k] = c[k] + thr[k] * fmaxf(o[0][k], 0.f);
    }
  }
}

int gridFor(long long n, int per, int cap)
{
  const long long b = (n + per - 1) / per;
  return (int)(b < 1 ? 1 : (b > cap ? cap : b));
}

} // namespace

extern "C" {

hipError_t hpt_nrc_init(const HptNrc *N, uint32_t seed, hipStream_t s)
{
  hipLaunchKernelGGL(k_nrc_init, dim3(gridFor(kP, 256, 1024)), dim3(256), 0, s, *N, seed);
  return hipGetLastError();
}

hipError_t hpt_nrc_encode(const float *raw12, int n, const float *lo3, const float *hi3, uint16_t *features, hipStream_t s)
{
  if (n <= 0)
    return hipSuccess;
  hipLaunchKernelGGL(k_nrc_encode, dim3(gridFor(n, 256, 8192)), dim3(256), 0, s, raw12, n, lo3[0], lo3[1], lo3[2],
      hi3[0], hi3[1], hi3[2], reinterpret_cast<__bf16 *>(features));
  return hipGetLastError();
}

hipError_t hpt_nrc_query(const HptNrc *N, const float *rec16, const uint32_t *queue, int n, const float *lo3,
    const float *hi3, float *contrib4, hipStream_t s)
{
  if (n <= 0)
    return hipSuccess;
  hipLaunchKernelGGL(k_nrc_query, dim3(gridFor(n, 16 * kQueryWaves, 256 * kQueryBlocks)), dim3(64 * kQueryWaves), 0, s, *N, rec16,
      queue, n, lo3[0], lo3[1], lo3[2], hi3[0], hi3[1], hi3[2], contrib4);
  return hipGetLastError();
}

hipError_t hpt_nrc_infer(const HptNrc *N, const uint16_t *features, int n, float *out3, hipStream_t s)
{
  if (n <= 0)
    return hipSuccess;
  hipLaunchKernelGGL(k_nrc_infer, dim3(gridFor(n, 64, 8192)), dim3(64), 0, s, *N,
      reinterpret_cast<const __bf16 *>(features), n, out3);
  return hipGetLastError();
}

hipError_t hpt_nrc_train(const HptNrc *N, const uint16_t *features, const float *target3, int n, hipStream_t s)
{
  if (n <= 0)
    return hipSuccess;
  if ((n + 63) / 64 > N->maxTiles)
    return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_nrc_train, dim3(gridFor(n, 64, N->maxTiles)), dim3(256), 0, s, *N,
      reinterpret_cast<const __bf16 *>(features), target3, n);
  return hipGetLastError();
}

hipError_t hpt_nrc_adam(const HptNrc *N, int n, float lr, int step, hipStream_t s)
{
  const int tiles = (n + 63) / 64;
  if (tiles <= 0 || tiles > N->maxTiles || step < 1)
    return hipErrorInvalidValue;
  const float bc1 = 1.f - powf(0.9f, (float)step), bc2 = 1.f - powf(0.99f, (float)step);
  hipLaunchKernelGGL(k_nrc_adam, dim3(kP / 64 + 1), dim3(64 * kAdamGroups * kAdamSegs), 0, s, *N, tiles, lr, bc1, bc2);
  return hipGetLastError();
}

} // extern "C"

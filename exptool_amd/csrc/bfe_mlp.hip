// MLP neural field x, y, z -> (Phi, F_R, F_phi, F_z): 3 -> 128 -> 128 -> 128 -> 128 -> 4,
// SiLU activations.  Training and inference kernels for gfx950.
//
// Precision: the 3 -> 128 input layer and the 128 -> 4 output layer run in
// float32 on the vector ALUs (positions are never rounded to bf16); the three
// 128 x 128 layers run on v_mfma_f32_16x16x32_bf16 with bf16 weights and
// activations and float32 accumulation.  Master weights and Adam moments are
// float32.
//
// MFMA operand layout (16x16x32, wave64): lane l, g = l / 16, c = l % 16
//   A (16 x 32):  A[c][8g + j], j < 8        B (32 x 16): B[8g + j][c]
//   D (16 x 16):  D[4g + i][c], i < 4
// Activations are kept "neuron x point": M = output neurons, N = points,
// K = input neurons.  Lane l of an output tile (mt, nt) holds neurons
// 16 mt + 4 g + i of point 16 nt + c; the next layer's B operand for K-step
// kk takes the 8 values of tiles 2kk and 2kk+1, i.e. logical k = 32kk + 8g + j
// stands for neuron pi(k) = 32kk + 4g + j (j < 4) or 32kk + 16 + 4g + j - 4.
// The weights are stored permuted along K by the same pi, so no shuffle is
// needed between layers.  The same holds for the backward chain with the
// transposed weights.
#include <math.h>

#include <vector>

#include "bfe_field.hpp"

namespace bfe {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float floatx4 __attribute__((ext_vector_type(4)));

constexpr int kH = 128;
constexpr int kNIn = 3;
constexpr int kNOut = 4;
// parameter offsets (float32 master vector)
constexpr int kOffW0 = 0;                       // [128][3]
constexpr int kOffB0 = kOffW0 + kH * kNIn;       // [128]
constexpr int kOffW1 = kOffB0 + kH;              // [128][128]
constexpr int kOffB1 = kOffW1 + kH * kH;
constexpr int kOffW2 = kOffB1 + kH;
constexpr int kOffB2 = kOffW2 + kH * kH;
constexpr int kOffW3 = kOffB2 + kH;
constexpr int kOffB3 = kOffW3 + kH * kH;
constexpr int kOffW4 = kOffB3 + kH;              // [4][128]
constexpr int kOffB4 = kOffW4 + kNOut * kH;      // [4]
constexpr int kNParams = kOffB4 + kNOut;         // 50564
static_assert(kNParams == BFE_MLP_NPARAMS, "parameter count");
constexpr int kHidOff[3] = {kOffW1, kOffW2, kOffW3};
constexpr int kSmallFloats = kH * kNIn + 4 * kH + kNOut * kH + kNOut;  // W0, b0..b3, W4, b4
#ifndef BFE_MLP_NT
#define BFE_MLP_NT 2
#endif
#ifndef BFE_MLP_BLOCK
#define BFE_MLP_BLOCK 512
#endif
constexpr int kNT = BFE_MLP_NT;                  // 16-point N-tiles per wave
constexpr int kWaveTile = 16 * kNT;              // points per wave
// Threads per block of the inference and integrator kernels: 8 waves on one
// copy of the LDS weights (two waves per SIMD hide the SiLU latency).
constexpr int kBlockInf = BFE_MLP_BLOCK;
static_assert(kBlockInf == 512 && kNT == 2, "mlp_leap_launch");
constexpr int kInfPts = kWaveTile * kBlockInf / 64;   // points per block
// The conservative-field kernels carry three tangent operand sets beside the
// activations (192 registers): eight waves per block, two per SIMD, so that one
// wave's activations cover the other's products.  Inference of 1M points 667 ->
// 458 us against four waves (no spills; 422 with the point work once per point);
// the integrator, which holds its state as well and spills 39 registers, 55.7 ->
// 37.5 ms per 100 steps of 1M orbits.  Few orbits take four waves, one per SIMD, with
// nothing spilled (mlp_leap_launch).
constexpr int kBlockGrad = 512;
constexpr int kBlockGradSmall = 256;
// LDS copy of the three hidden weight matrices: rows of kH bf16 padded to
// kLdsRow.  A lane reads 16 bytes of row 16 mt + c; unpadded (256-byte)
// rows put the rows that one read cycle serves on the same four banks, with
// 16 bytes of padding they cover every bank once.
constexpr int kLdsRow = kH + 8;
constexpr int kLdsLayer = kH * kLdsRow;
constexpr size_t kLdsWBytes = 3 * kLdsLayer * sizeof(__bf16);
constexpr size_t kLdsBytes = kLdsWBytes + kSmallFloats * sizeof(float);

__device__ __forceinline__ floatx4 mfma16(bf16x8 a, bf16x8 b, floatx4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

__host__ __device__ __forceinline__ int pi_neuron(int kk, int g, int j) {
  return 32 * kk + (j < 4 ? 4 * g + j : 16 + 4 * g + (j - 4));
}
// inverse of pi within a 32-block: neuron n -> logical k
__host__ __device__ __forceinline__ int pi_inverse(int n) {
  const int kk = n >> 5, r = n & 31;
  const int hi = r >> 4, q = r & 15;
  return 32 * kk + 8 * (q >> 2) + 4 * hi + (q & 3);
}

// SiLU and its derivative with the hardware reciprocal (about 1 ulp).
__device__ __forceinline__ float sigmoid(float z) { return __builtin_amdgcn_rcpf(1.f + __expf(-z)); }
__device__ __forceinline__ float silu(float z) { return z * sigmoid(z); }
__device__ __forceinline__ float dsilu(float z) {
  const float s = sigmoid(z);
  return s * (1.f + z * (1.f - s));
}

// Analytic base of the field: the network predicts the field minus this
// model (all zero: no base).  Up to kMaxMN Miyamoto-Nagai discs
// Phi = -M / sqrt(R^2 + (a + sqrt(z^2 + b^2))^2) and one Hernquist sphere
// Phi = -Mh / (r + ah), plus a constant; evaluated in float64.
struct MLPBase {
  int nmn;
  double M[kMaxMN], a[kMaxMN], b[kMaxMN];
  double mh, ah, phi0;
};

struct MLPCfg {
  float sxy;        // feature 0,1 = x/sxy, y/sxy
  float hz, wz;     // feature 2 = asinh(z/hz)/wz
  float os[4];      // physical output k = os[k] * y_k + ob[k] + base_k
  float ob[4];
  MLPBase base;
  int conservative; // forces are -grad of the potential output (mlp_tile_grad)
  float lw[4];      // training loss weight of output k
};

// (Phi, F_R, F_phi = 0, F_z) of the analytic base at (R, z).
__device__ __forceinline__ void mlp_base_eval(const MLPBase& B, float Rf, float zf, float out[4]) {
  const double R = Rf, z = zf, R2 = R * R, z2 = z * z;
  double pot = B.phi0, fR = 0.0, fz = 0.0;
  for (int k = 0; k < B.nmn; ++k) {
    const double bz = sqrt(z2 + B.b[k] * B.b[k]);
    const double s = B.a[k] + bz;
    const double id = 1.0 / sqrt(R2 + s * s);
    const double m3 = B.M[k] * id * id * id;
    pot -= B.M[k] * id;
    fR -= m3 * R;
    fz -= m3 * z * s / bz;
  }
  if (B.mh != 0.0) {
    const double r = sqrt(R2 + z2);
    const double ir = 1.0 / (r + B.ah);
    pot -= B.mh * ir;
    // -Mh / (r + a)^2 along r-hat; r = 0 gives no force
    const double g = r > 0.0 ? B.mh * ir * ir / r : 0.0;
    fR -= g * R;
    fz -= g * z;
  }
  out[0] = (float)pot;
  out[1] = (float)fR;
  out[2] = 0.f;
  out[3] = (float)fz;
}

__device__ __forceinline__ void mlp_features(const MLPCfg& c, float x, float y, float z, float f[3]) {
  f[0] = x / c.sxy;
  f[1] = y / c.sxy;
  f[2] = asinhf(z / c.hz) / c.wz;
}

struct MLPKArgs {
  const float* x;
  const float* y;
  const float* z;
  int64_t n;
  float* out;            // [4][n] physical outputs
  const float* params;
  const __bf16* Wp;      // [3][128][128] forward A operands (K-permuted)
  MLPCfg cfg;
};

__device__ __forceinline__ void load_small(const float* __restrict__ params, float* s_small) {
  // W0, b0, b1, b2, b3, W4, b4 into LDS
  for (int t = threadIdx.x; t < kSmallFloats; t += blockDim.x) {
    int src;
    if (t < kH * kNIn + kH) src = t;                                       // W0, b0
    else if (t < kH * kNIn + 2 * kH) src = kOffB1 + (t - kH * kNIn - kH);
    else if (t < kH * kNIn + 3 * kH) src = kOffB2 + (t - kH * kNIn - 2 * kH);
    else if (t < kH * kNIn + 4 * kH) src = kOffB3 + (t - kH * kNIn - 3 * kH);
    else src = kOffW4 + (t - kH * kNIn - 4 * kH);                          // W4, b4
    s_small[t] = params[src];
  }
}

__device__ __forceinline__ void load_weights(const __bf16* __restrict__ W, __bf16* s_w) {
  constexpr int kRow16 = kH / 8, kLds16 = kLdsRow / 8;   // 16-byte chunks per row
  const uint4* src = reinterpret_cast<const uint4*>(W);
  uint4* dst = reinterpret_cast<uint4*>(s_w);
  for (int t = threadIdx.x; t < 3 * kH * kRow16; t += blockDim.x)
    dst[(t / kRow16) * kLds16 + t % kRow16] = src[t];
}

// Hidden layer: acc[mt][nt] = bias + W (K-permuted, LDS) x B[kk][nt].
template <int NT>
__device__ __forceinline__ void hidden_mfma(const __bf16* __restrict__ sW, const float* bias,
                                            const bf16x8 (&B)[4][NT], floatx4 (&acc)[8][NT],
                                            int g, int c) {
#pragma unroll
  for (int mt = 0; mt < 8; ++mt)
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
#pragma unroll
      for (int i = 0; i < 4; ++i) acc[mt][nt][i] = bias ? bias[16 * mt + 4 * g + i] : 0.f;
#pragma unroll
  for (int kk = 0; kk < 4; ++kk) {
    // keep the operand loads of one K-step in flight at a time (register budget)
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int mt = 0; mt < 8; ++mt) {
      const bf16x8 a = *reinterpret_cast<const bf16x8*>(sW + (16 * mt + c) * kLdsRow + 32 * kk + 8 * g);
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) acc[mt][nt] = mfma16(a, B[kk][nt], acc[mt][nt]);
    }
  }
}

// SiLU of a hidden layer's pre-activations acc: into the next layer's bf16
// operands B, or (LAST) in place as float32 for the output layer.
template <bool LAST>
__device__ __forceinline__ void forward_activate(floatx4 (&acc)[8][kNT], bf16x8 (&B)[4][kNT]) {
#pragma unroll
  for (int mt = 0; mt < 8; ++mt)
#pragma unroll
    for (int nt = 0; nt < kNT; ++nt)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float hh = silu(acc[mt][nt][i]);
        if (LAST) acc[mt][nt][i] = hh;
        else B[mt >> 1][nt][(mt & 1) * 4 + i] = (__bf16)hh;
      }
}

// Forward pass of one wave tile (kNT x 16 points, column c of lane group g):
// features f -> normalised outputs yk (all four lane groups of a column end
// with the same yk).
__device__ __forceinline__ void mlp_tile_forward(const __bf16* __restrict__ sW,
                                                 const float* __restrict__ sS,
                                                 const float (&f)[kNT][3], float (&yk)[kNT][4],
                                                 int g, int c) {
  const float* sW0 = sS;
  const float* sB0 = sS + kH * kNIn;
  const float* sBh = sS + kH * kNIn + kH;           // b1, b2, b3
  const float* sW4 = sS + kH * kNIn + 4 * kH;
  const float* sB4 = sW4 + kNOut * kH;
  // layer 0 (float32): each lane evaluates the 32 neurons it feeds to layer 1
  bf16x8 B[4][kNT];
#pragma unroll
  for (int kk = 0; kk < 4; ++kk)
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int nr = pi_neuron(kk, g, j);
      const float w0 = sW0[nr * 3], w1 = sW0[nr * 3 + 1], w2 = sW0[nr * 3 + 2], b = sB0[nr];
#pragma unroll
      for (int nt = 0; nt < kNT; ++nt) {
        const float zz = fmaf(w0, f[nt][0], fmaf(w1, f[nt][1], fmaf(w2, f[nt][2], b)));
        B[kk][nt][j] = (__bf16)silu(zz);
      }
    }
  floatx4 acc[8][kNT];
  // layers 1 and 2 feed the next layer's operands; the last layer is peeled
  // so that no activation carries a branch on the layer
#pragma unroll 1
  for (int layer = 0; layer < 2; ++layer) {
    hidden_mfma(sW + layer * kLdsLayer, sBh + layer * kH, B, acc, g, c);
    forward_activate<false>(acc, B);
  }
  hidden_mfma(sW + 2 * kLdsLayer, sBh + 2 * kH, B, acc, g, c);
  forward_activate<true>(acc, B);
  // output layer (float32): partial sums over this lane's neurons, then
  // reduce over the four lane groups that hold the same point column
#pragma unroll
  for (int nt = 0; nt < kNT; ++nt)
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      float s = 0.f;
#pragma unroll
      for (int mt = 0; mt < 8; ++mt)
#pragma unroll
        for (int i = 0; i < 4; ++i) s = fmaf(sW4[k * kH + 16 * mt + 4 * g + i], acc[mt][nt][i], s);
      s += __shfl_xor(s, 16);
      s += __shfl_xor(s, 32);
      yk[nt][k] = s + sB4[k];
    }
}

// Forward pass of one wave tile for the potential output y0 and its
// derivatives dy0/df_k along the three features, by forward-mode tangents:
// t_1^k = silu'(z_1) W0[:, k], t_{l+1}^k = silu'(z_{l+1}) (W_l t_l^k), each
// W_l t_l^k one more bf16 MFMA pass over the layer's LDS weights (float32
// accumulation, tangents rounded to bf16 as the activations are), and
// dy0/df_k = W4[0] . t_4^k.  Layout as mlp_tile_forward; NT 16-point tiles.
//
// One hidden layer W of it, 32 output neurons (one operand of the next layer) at
// a time: each A fragment is read from LDS once and multiplied into the
// activations (acc[0], from the bias) and the three tangents (acc[1..3], from
// zero).  The activations of one group (B2, T2; LAST: into the sums ys, ds of the
// potential row) run on the vector ALUs while the products of the next are on the
// matrix cores: the scheduling groups place three vector instructions behind each
// product, which is about what both units take.
template <int NT, bool LAST>
__device__ __forceinline__ void grad_layer(const __bf16* __restrict__ W, const float* bias,
                                           const float* __restrict__ sW4,
                                           const bf16x8 (&B)[4][NT], const bf16x8 (&T)[3][4][NT],
                                           bf16x8 (&B2)[4][NT], bf16x8 (&T2)[3][4][NT],
                                           float (&ys)[NT], float (&ds)[NT][3], int g, int c) {
  floatx4 acc[2][4][2][NT];
  const floatx4 zero = {0.f, 0.f, 0.f, 0.f};
  auto products = [&](int mp, floatx4 (&ac)[4][2][NT]) {
#pragma unroll
    for (int kk = 0; kk < 4; ++kk)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int mt = 2 * mp + h;
        const bf16x8 a = *reinterpret_cast<const bf16x8*>(W + (16 * mt + c) * kLdsRow + 32 * kk + 8 * g);
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
          if (kk == 0) {
            floatx4 b0;
#pragma unroll
            for (int i = 0; i < 4; ++i) b0[i] = bias[16 * mt + 4 * g + i];
            ac[0][h][nt] = mfma16(a, B[0][nt], b0);
#pragma unroll
            for (int k = 0; k < 3; ++k) ac[1 + k][h][nt] = mfma16(a, T[k][0][nt], zero);
          } else {
            ac[0][h][nt] = mfma16(a, B[kk][nt], ac[0][h][nt]);
#pragma unroll
            for (int k = 0; k < 3; ++k) ac[1 + k][h][nt] = mfma16(a, T[k][kk][nt], ac[1 + k][h][nt]);
          }
        }
      }
  };
  auto activate = [&](int mp, const floatx4 (&ac)[4][2][NT]) {
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int nt = 0; nt < NT; ++nt)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int mt = 2 * mp + h;
          const float zz = ac[0][h][nt][i];
          const float sg = sigmoid(zz);
          const float hh = zz * sg;
          const float dsl = sg * (1.f + zz * (1.f - sg));
          if (LAST) ys[nt] = fmaf(sW4[16 * mt + 4 * g + i], hh, ys[nt]);
          else B2[mp][nt][h * 4 + i] = (__bf16)hh;
#pragma unroll
          for (int k = 0; k < 3; ++k) {
            const float tt = dsl * ac[1 + k][h][nt][i];
            if (LAST) ds[nt][k] = fmaf(sW4[16 * mt + 4 * g + i], tt, ds[nt][k]);
            else T2[k][mp][nt][h * 4 + i] = (__bf16)tt;
          }
        }
  };
  products(0, acc[0]);
#pragma unroll
  for (int mp = 0; mp < 4; ++mp) {
    __builtin_amdgcn_sched_barrier(0);
    if (mp < 3) products(mp + 1, acc[(mp + 1) & 1]);
    activate(mp, acc[mp & 1]);
    if (mp < 3) {
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);   // an LDS read
#pragma unroll
        for (int k = 0; k < 4 * NT; ++k) {
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);   // a product
          __builtin_amdgcn_sched_group_barrier(0x002, 3, 0);   // three vector instructions
        }
      }
    }
  }
}

template <int NT>
__device__ __forceinline__ void mlp_tile_grad(const __bf16* __restrict__ sW,
                                              const float* __restrict__ sS,
                                              const float (&f)[NT][3], float (&y0)[NT],
                                              float (&dy)[NT][3], int g, int c) {
  const float* sW0 = sS;
  const float* sB0 = sS + kH * kNIn;
  const float* sBh = sS + kH * kNIn + kH;
  const float* sW4 = sS + kH * kNIn + 4 * kH;
  const float* sB4 = sW4 + kNOut * kH;
  bf16x8 B[4][NT];
  bf16x8 T[3][4][NT];
#pragma unroll
  for (int kk = 0; kk < 4; ++kk)
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int nr = pi_neuron(kk, g, j);
      const float w0 = sW0[nr * 3], w1 = sW0[nr * 3 + 1], w2 = sW0[nr * 3 + 2], b = sB0[nr];
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) {
        const float zz = fmaf(w0, f[nt][0], fmaf(w1, f[nt][1], fmaf(w2, f[nt][2], b)));
        const float sg = sigmoid(zz);
        const float d = sg * (1.f + zz * (1.f - sg));
        B[kk][nt][j] = (__bf16)(zz * sg);
        T[0][kk][nt][j] = (__bf16)(d * w0);
        T[1][kk][nt][j] = (__bf16)(d * w1);
        T[2][kk][nt][j] = (__bf16)(d * w2);
      }
    }
  float ys[NT], ds[NT][3];
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) {
    ys[nt] = 0.f;
    ds[nt][0] = ds[nt][1] = ds[nt][2] = 0.f;
  }
  bf16x8 B2[4][NT];
  bf16x8 T2[3][4][NT];
  grad_layer<NT, false>(sW, sBh, sW4, B, T, B2, T2, ys, ds, g, c);
  grad_layer<NT, false>(sW + kLdsLayer, sBh + kH, sW4, B2, T2, B, T, ys, ds, g, c);
  grad_layer<NT, true>(sW + 2 * kLdsLayer, sBh + 2 * kH, sW4, B, T, B2, T2, ys, ds, g, c);
  // sums over the four lane groups that hold the same point column
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) {
    float v = ys[nt];
    v += __shfl_xor(v, 16);
    v += __shfl_xor(v, 32);
    y0[nt] = v + sB4[0];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      float w = ds[nt][k];
      w += __shfl_xor(w, 16);
      w += __shfl_xor(w, 32);
      dy[nt][k] = w;
    }
  }
}

// Potential and Cartesian force of the conservative field at (x, y, z): the
// network's potential os0 y0 + ob0 plus the base, F = -grad of it (chain rule
// through the features f = (x/sxy, y/sxy, asinh(z/hz)/wz)).
__device__ __forceinline__ void conservative_field(const MLPCfg& cf, float x, float y, float z,
                                                   float y0, const float (&dy)[3], float& fx,
                                                   float& fy, float& fz, float& pot) {
  const float R = sqrtf(x * x + y * y);
  float bv[4];
  mlp_base_eval(cf.base, R, z, bv);
  const float cp = R > 0.f ? x / R : 1.f, sp = R > 0.f ? y / R : 0.f;
  const float zh = z / cf.hz;
  const float dfz = 1.f / (cf.wz * cf.hz * sqrtf(1.f + zh * zh));
  fx = -cf.os[0] * dy[0] / cf.sxy + bv[1] * cp;
  fy = -cf.os[0] * dy[1] / cf.sxy + bv[1] * sp;
  fz = -cf.os[0] * dy[2] * dfz + bv[3];
  pot = cf.os[0] * y0 + cf.ob[0] + bv[0];
}

// Forward pass over 32-point tiles per wave.
__global__ __launch_bounds__(kBlockInf) void mlp_fwd_kernel(MLPKArgs a) {
  extern __shared__ __align__(16) unsigned char smem[];
  __bf16* sW = reinterpret_cast<__bf16*>(smem);
  float* sS = reinterpret_cast<float*>(smem + kLdsWBytes);
  load_small(a.params, sS);
  load_weights(a.Wp, sW);
  __syncthreads();

  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int g = lane >> 4, c = lane & 15;
  const int64_t ntiles = (a.n + kInfPts - 1) / kInfPts;
  for (int64_t tile = blockIdx.x; tile < ntiles; tile += gridDim.x) {
    const int64_t base = tile * kInfPts + wave * kWaveTile;
    int64_t pid[kNT];
    bool valid[kNT];
    float f[kNT][3];
#pragma unroll
    for (int nt = 0; nt < kNT; ++nt) {
      pid[nt] = base + 16 * nt + c;
      valid[nt] = pid[nt] < a.n;
      const int64_t q = valid[nt] ? pid[nt] : 0;
      mlp_features(a.cfg, a.x[q], a.y[q], a.z[q], f[nt]);
    }
    float yk[kNT][4];
    mlp_tile_forward(sW, sS, f, yk, g, c);
#pragma unroll
    for (int nt = 0; nt < kNT; ++nt)
      if (valid[nt] && g == 0) {
        const float px = a.x[pid[nt]], py = a.y[pid[nt]];
        float bv[4];
        mlp_base_eval(a.cfg.base, sqrtf(px * px + py * py), a.z[pid[nt]], bv);
#pragma unroll
        for (int k = 0; k < 4; ++k)
          a.out[(size_t)k * a.n + pid[nt]] = a.cfg.os[k] * yk[nt][k] + a.cfg.ob[k] + bv[k];
      }
  }
}

// Inference of the conservative field: out = Phi, F_R, F_phi, F_z with
// F = -grad Phi (mlp_tile_grad).  The first `waves` waves of a block take `per`
// 16-point tiles (1 to 4) each at a time (mlp_grad_launch): the features and the force of the base model, a fifth of the vector work
// when every lane group of a tile repeats them, are then evaluated one point per
// lane, and the tiles' features and results pass through the lanes.
__global__ __launch_bounds__(kBlockGrad) void mlp_fwd_grad_kernel(MLPKArgs a, int waves, int per) {
  constexpr int NT = 1;
  extern __shared__ __align__(16) unsigned char smem[];
  __bf16* sW = reinterpret_cast<__bf16*>(smem);
  float* sS = reinterpret_cast<float*>(smem + kLdsWBytes);
  load_small(a.params, sS);
  load_weights(a.Wp, sW);
  __syncthreads();
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int g = lane >> 4, c = lane & 15;
  const int pts = 16 * per;            // points of a wave
  if (wave >= waves) return;
  for (int64_t base = ((int64_t)blockIdx.x * waves + wave) * pts; base < a.n;
       base += (int64_t)gridDim.x * waves * pts) {
    const int64_t p = base + lane;
    const bool valid = lane < pts && p < a.n;
    const int64_t q = valid ? p : base;
    const float x = a.x[q], y = a.y[q], z = a.z[q];
    float fl[3], y0 = 0.f, dy[3] = {0.f, 0.f, 0.f};
    mlp_features(a.cfg, x, y, z, fl);
#pragma unroll 1
    for (int t = 0; t < per; ++t) {
      float f[NT][3], yt[NT], dt[NT][3];
#pragma unroll
      for (int k = 0; k < 3; ++k) f[0][k] = __shfl(fl[k], 16 * t + c, 64);
      mlp_tile_grad<NT>(sW, sS, f, yt, dt, g, c);
      if (g == t) {   // all four lane groups hold the tile's results
        y0 = yt[0];
#pragma unroll
        for (int k = 0; k < 3; ++k) dy[k] = dt[0][k];
      }
    }
    if (valid) {
      float fx, fy, fz, pot;
      conservative_field(a.cfg, x, y, z, y0, dy, fx, fy, fz, pot);
      const float R = sqrtf(x * x + y * y);
      const float cp = R > 0.f ? x / R : 1.f, sp = R > 0.f ? y / R : 0.f;
      a.out[p] = pot;
      a.out[a.n + p] = fx * cp + fy * sp;
      a.out[2 * a.n + p] = fy * cp - fx * sp;
      a.out[3 * a.n + p] = fz;
    }
  }
}

// ---------------------------------------------------------------------------
// Training: one kernel takes tiles of 128 points through the forward pass, the
// loss, the backward chain and the weight gradients; a second one reduces the
// blocks' partial sums.
//
// Eight waves of 16 points.  The pre-activations of the four layers stay in
// registers (float32, 128 per lane: nothing but partial sums goes to memory;
// as global arrays they were 134 MB written and read twice per 65 536 points).
// The six weight operands W1, W2, W3, W3^T, W2^T, W1^T pass through two LDS
// buffers, the next copied (global to LDS directly) while one is multiplied:
// 16-byte chunk q of row r lies at q ^ (r mod 16), so the 16 rows a read
// touches are on different banks without padding.
// dW_l = gZ_{l+1} H_l^T sums over points, whose values lie across lanes: gZ
// and H go to LDS as bf16 [point][neuron] and come back transposed
// (ds_read_tr16: of a 16-lane group's 16 chunks of four neurons, lane l gets
// neuron l of four points).  Wave w makes output rows 16 w .. 16 w + 15.  The
// k order of the products is point 4 g + j, then 16 + 4 g + j, for lane group
// g, in both operands.  The sums run in float32 over a tile and in float64
// over tiles.  b0..b3, W0 and W4 gradients: products and sums over points in
// float64 throughout (reduce_rows).
// Measured for 65 536 points: 910 us as separate forward, backward, weight
// gradient and reduction kernels (72 + 200 + 337 + 63 + 197 + 41), 86 us for
// this one and 16 for the reduction (100 MB of partial sums; 82 with float32 small
// sums); about half of a tile's 41 us is vector-ALU issue (SiLUs and the sums over lanes), the rest
// waits of two waves per SIMD at 256 registers.
constexpr int kTrainThreads = 512;
constexpr int kTrainPts = 128;
constexpr int kStageRow = kH + 16;   // bf16 per stage row: 8-row stride of 64 banks
constexpr int kStageElems = kTrainPts * kStageRow;
constexpr int kNSmall = kH * kNIn + 4 * kH + kNOut * kH + kNOut;   // gradients outside W1..W3
constexpr int kSmallRow = kNSmall + 1;                             // and the loss
constexpr size_t kTrainLds = (2 * (size_t)kH * kH + 2 * (size_t)kStageElems) * sizeof(__bf16) +
                             kSmallFloats * sizeof(float);

struct MLPTrainArgs {
  const float* x;
  const float* y;
  const float* z;
  const float* target;   // [4][n] normalised targets
  const float* weight;   // [n] per-point loss weight or NULL
  int64_t n;
  int tiles;             // 128-point tiles per block
  float inv_n;
  const float* params;
  const __bf16* Wp;
  const __bf16* Wt;
  float* dwpart;         // [tile][3][128][128]
  double* small_wave;    // [block][8 waves][11][128]
  double* small_part;    // [block][kSmallRow]: dW0[d][nr], db0..db3, dW4, db4, loss
  MLPCfg cfg;
};

typedef const void __attribute__((address_space(1)))* GlobalPtr;
typedef void __attribute__((address_space(3)))* LdsPtr;
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef s16x4 __attribute__((address_space(3)))* LdsS4;

// Starts the copy of one 128 x 128 weight operand into an LDS buffer (every
// thread calls it; waited for by train_sync).
__device__ __forceinline__ void train_load(const __bf16* __restrict__ W, __bf16* buf, int wave,
                                           int lane) {
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const int row = 16 * wave + 4 * k + (lane >> 4), q = (lane & 15) ^ (row & 15);
    __builtin_amdgcn_global_load_lds((GlobalPtr)(W + row * kH + 8 * q),
                                     (LdsPtr)(buf + (16 * wave + 4 * k) * kH), 16, 0, 0);
  }
}

// The block's copies and stage writes have arrived, and every wave is done
// with the buffers they replace.
__device__ __forceinline__ void train_sync() {
  __builtin_amdgcn_sched_barrier(0);
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
  __syncthreads();
  __builtin_amdgcn_sched_barrier(0);
}

// Four consecutive floats of the small parameters (16-byte aligned: every
// array there starts at a multiple of four).
__device__ __forceinline__ float4 small4(const float* p) {
  return *reinterpret_cast<const float4*>(__builtin_assume_aligned(p, 16));
}

// acc = bias + W x B for one 16-point tile, W in a swizzled LDS buffer (BIAS
// false: no bias).
template <bool BIAS>
__device__ __forceinline__ void train_mfma(const __bf16* __restrict__ sW, const float* bias,
                                           const bf16x8 (&B)[4], floatx4 (&acc)[8], int g, int c) {
#pragma unroll
  for (int mt = 0; mt < 8; ++mt) {
    if constexpr (BIAS) {
      const float4 b = small4(bias + 16 * mt + 4 * g);
      acc[mt] = floatx4{b.x, b.y, b.z, b.w};
    } else {
      acc[mt] = floatx4{0.f, 0.f, 0.f, 0.f};
    }
  }
#pragma unroll
  for (int kk = 0; kk < 4; ++kk) {
    // two K-steps' operand reads in flight at a time (register budget)
    if (kk == 2) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int mt = 0; mt < 8; ++mt) {
      const bf16x8 a = *reinterpret_cast<const bf16x8*>(sW + (16 * mt + c) * kH + (((4 * kk + g) ^ c) << 3));
      acc[mt] = mfma16(a, B[kk], acc[mt]);
    }
  }
  __builtin_amdgcn_sched_barrier(0);
}

// The lane's 32 values (neuron 16 mt + 4 g + i at v[4 mt + i]) as bf16 into
// row p of a stage.
__device__ __forceinline__ void train_stage(__bf16* st, int p, int g, const float (&v)[32]) {
  typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
#pragma unroll
  for (int mt = 0; mt < 8; ++mt) {
    bf16x4 b;
#pragma unroll
    for (int i = 0; i < 4; ++i) b[i] = (__bf16)v[4 * mt + i];
    *reinterpret_cast<bf16x4*>(st + p * kStageRow + 16 * mt + 4 * g) = b;
  }
}

// K-step ks (points 32 ks ..) of the neurons n0 .. n0 + 15 as an MFMA operand.
__device__ __forceinline__ bf16x8 train_operand(const __bf16* st, int ks, int n0, int g, int c) {
  const __bf16* p = st + (32 * ks + 4 * g + (c >> 2)) * kStageRow + n0 + 4 * (c & 3);
  union {
    s16x4 h[2];
    bf16x8 v;
  } u;
  u.h[0] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LdsS4)p);
  u.h[1] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LdsS4)(p + 16 * kStageRow));
  return u.v;
}

// The staged points' product G H^T, rows 16 wave .. of part ([128][128]).
__device__ __forceinline__ void train_dw(const __bf16* sG, const __bf16* sH, float* __restrict__ part,
                                         int wave, int g, int c) {
  floatx4 acc[8];
  float* o = part + (16 * wave + 4 * g) * kH + c;
#pragma unroll
  for (int b = 0; b < 8; ++b) acc[b] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int ks = 0; ks < kTrainPts / 32; ++ks) {
    const bf16x8 a = train_operand(sG, ks, 16 * wave, g, c);
#pragma unroll
    for (int b = 0; b < 8; ++b) acc[b] = mfma16(a, train_operand(sH, ks, 16 * b, g, c), acc[b]);
  }
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int b = 0; b < 8; ++b)
#pragma unroll
    for (int i = 0; i < 4; ++i) o[i * kH + 16 * b] = acc[b][i];
}

// Keeps the compiler from holding what it computed from z (the sigmoids, one
// register a value) until they are needed again: recomputed they cost two
// transcendentals, held they spill.
__device__ __forceinline__ void forget(floatx4 (&z)[8]) {
#pragma unroll
  for (int k = 0; k < 8; ++k) asm volatile("" : "+v"(z[k]));
}

template <int CTRL>
__device__ __forceinline__ int dpp_get(int v) {
  return __builtin_amdgcn_update_dpp(0, v, CTRL, 0xf, 0xf, true);
}
template <int CTRL>
__device__ __forceinline__ float dpp_get(float v) {
  return __int_as_float(dpp_get<CTRL>(__float_as_int(v)));
}

template <int CTRL>
__device__ __forceinline__ double dpp_get(double v) {
  return __hiloint2double(dpp_get<CTRL>(__double2hiint(v)), dpp_get<CTRL>(__double2loint(v)));
}

// Sums of a lane's 32 values over the 16 lanes of a row (one point each), products
// and sums in float64.  Each exchange halves the values a lane keeps; lane c ends
// with the sums of values 2 c and 2 c + 1.  The first exchange passes the float32
// values, kept in v[0..15] and received in v[16..31], once for several factors.
__device__ __forceinline__ void rows_exchange(float (&v)[32], int c) {
  const bool b3 = c & 8;
#pragma unroll
  for (int k = 0; k < 16; ++k) {
    const float keep = b3 ? v[k + 16] : v[k], send = b3 ? v[k] : v[k + 16];
    v[k] = keep;
    v[k + 16] = dpp_get<0x140>(send);   // row_mirror: lane 15 - c
  }
}
// The sums of the exchanged values times the lanes' factors m (MUL).
template <bool MUL>
__device__ __forceinline__ void reduce_rows(const float (&v)[32], float m, int c, double (&s)[2]) {
  const bool b2 = c & 4, b1 = c & 2, b0 = c & 1;
  const double mk = m, mo = dpp_get<0x140>(m);
  double t[16];
#pragma unroll
  for (int k = 0; k < 16; ++k)
    t[k] = MUL ? fma((double)v[k], mk, (double)v[k + 16] * mo) : (double)v[k] + (double)v[k + 16];
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    const double keep = b2 ? t[k + 8] : t[k], send = b2 ? t[k] : t[k + 8];
    t[k] = keep + dpp_get<0x141>(send);   // row_half_mirror
  }
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const double keep = b1 ? t[k + 4] : t[k], send = b1 ? t[k] : t[k + 4];
    t[k] = keep + dpp_get<0x4E>(send);    // lanes 2 apart
  }
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    const double keep = b0 ? t[k + 2] : t[k], send = b0 ? t[k] : t[k + 2];
    s[k] = keep + dpp_get<0xB1>(send);    // neighbours
  }
}

// z = Z[l] and Z[l] = z for a uniform l that is not known at compile time.
__device__ __forceinline__ void layer_get(const floatx4 (&Z)[4][8], int l, floatx4 (&z)[8]) {
#pragma unroll
  for (int k = 0; k < 4; ++k)
    if (l == k) {
#pragma unroll
      for (int j = 0; j < 8; ++j) z[j] = Z[k][j];
    }
}
__device__ __forceinline__ void layer_put(floatx4 (&Z)[4][8], int l, const floatx4 (&z)[8]) {
#pragma unroll
  for (int k = 0; k < 4; ++k)
    if (l == k) {
#pragma unroll
      for (int j = 0; j < 8; ++j) Z[k][j] = z[j];
    }
}
__device__ __forceinline__ float pick4(const float (&v)[4], int k) {
  return k == 0 ? v[0] : k == 1 ? v[1] : k == 2 ? v[2] : v[3];
}

// Sums over the wave's 16 points of m v (MUL) or v, v exchanged (rows_exchange), to
// the wave's row of small sums, added to what an earlier tile left there: lane c of
// group g has neurons 16 (c / 2) + 4 g + 2 (c & 1) + {0, 1}.
template <bool MUL>
__device__ __forceinline__ void small_sums(const float (&v)[32], float m, double* __restrict__ row,
                                           bool first, int g, int c) {
  double2* o = reinterpret_cast<double2*>(row + 16 * (c >> 1) + 4 * g + 2 * (c & 1));
  const double2 old = first ? make_double2(0.0, 0.0) : *o;
  double s[2];
  reduce_rows<MUL>(v, m, c, s);
  *o = make_double2(old.x + s[0], old.y + s[1]);
}

__global__ __launch_bounds__(kTrainThreads) void mlp_train_kernel(MLPTrainArgs a) {
  extern __shared__ __align__(16) unsigned char smem[];
  __bf16* buf = reinterpret_cast<__bf16*>(smem);   // two operands of kH * kH
  __bf16* sG = buf + 2 * kH * kH;
  __bf16* sH = sG + kStageElems;
  float* sS = reinterpret_cast<float*>(sH + kStageElems);
  __shared__ double s_loss[8][5];
  const float* sW0 = sS;
  const float* sB0 = sS + kH * kNIn;
  const float* sBh = sB0 + kH;
  const float* sW4 = sS + kH * kNIn + 4 * kH;
  const float* sB4 = sW4 + kNOut * kH;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int g = lane >> 4, c = lane & 15;
  train_load(a.Wp, buf, wave, lane);
  load_small(a.params, sS);
  if (lane < 5) s_loss[wave][lane] = 0.0;          // the wave's loss and db4
  double* rows = a.small_wave + ((size_t)blockIdx.x * 8 + wave) * 11 * kH;   // dW0 (3), db0..3, dW4 (4)
#pragma unroll 1
  for (int t = 0; t < a.tiles; ++t) {
    const int64_t tile = (int64_t)blockIdx.x * a.tiles + t;
    const int64_t p0 = tile * kTrainPts;
    if (p0 >= a.n) break;
    float* part = a.dwpart + (size_t)tile * 3 * kH * kH;
    const int row = 16 * wave + c;   // the lane's point in the tile
    const int64_t p = p0 + row;
    const bool valid = p < a.n;
    const int64_t q = valid ? p : 0;
    float f[4], tg[4];
    {
      float f3[3];
      mlp_features(a.cfg, a.x[q], a.y[q], a.z[q], f3);
      f[0] = f3[0]; f[1] = f3[1]; f[2] = f3[2];
      f[3] = 1.f;
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) tg[k] = a.target[(size_t)k * a.n + q];
    const float wt = valid ? (a.weight ? a.weight[q] : 1.f) : 0.f;
    floatx4 Z[4][8], z[8];
    bf16x8 B[4];
    float v[32];
    train_sync();   // W1 (and the small parameters)
#pragma unroll
    for (int mt = 0; mt < 8; ++mt) {
      const int nr = 16 * mt + 4 * g;
      const float4 w0 = small4(sW0 + 3 * nr), w1 = small4(sW0 + 3 * nr + 4), w2 = small4(sW0 + 3 * nr + 8);
      const float4 b = small4(sB0 + nr);
      const float w[12] = {w0.x, w0.y, w0.z, w0.w, w1.x, w1.y, w1.z, w1.w, w2.x, w2.y, w2.z, w2.w};
      const float bb[4] = {b.x, b.y, b.z, b.w};
#pragma unroll
      for (int i = 0; i < 4; ++i)
        Z[0][mt][i] = fmaf(w[3 * i], f[0], fmaf(w[3 * i + 1], f[1], fmaf(w[3 * i + 2], f[2], bb[i])));
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) z[j] = Z[0][j];
    // layers as loops: unrolled, the kernel's 60 KB of code were read from
    // the L2 once per tile, which took longer than running them
#pragma unroll 1
    for (int l = 0; l < 3; ++l) {
#pragma unroll
      for (int j = 0; j < 32; ++j) B[j >> 3][j & 7] = (__bf16)silu(z[j >> 2][j & 3]);
      if (l > 0) train_sync();   // W_{l+1}; then the next operand into the other buffer
      train_load(l < 2 ? a.Wp + (l + 1) * kH * kH : a.Wt + 2 * kH * kH, buf + ((l + 1) & 1) * kH * kH,
                 wave, lane);
      train_mfma<true>(buf + (l & 1) * kH * kH, sBh + l * kH, B, z, g, c);
      layer_put(Z, l + 1, z);
    }
    // output layer and loss (all four lane groups hold the same point)
    float gy[4];
#pragma unroll
    for (int k = 0; k < 32; ++k) v[k] = silu(z[k >> 2][k & 3]);
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      float s = 0.f;
#pragma unroll
      for (int mt = 0; mt < 8; ++mt) {
        const float4 w = small4(sW4 + k * kH + 16 * mt + 4 * g);
        s = fmaf(w.x, v[4 * mt], s);
        s = fmaf(w.y, v[4 * mt + 1], s);
        s = fmaf(w.z, v[4 * mt + 2], s);
        s = fmaf(w.w, v[4 * mt + 3], s);
      }
      s += __shfl_xor(s, 16);
      s += __shfl_xor(s, 32);
      const float d = valid ? s + sB4[k] - tg[k] : 0.f;
      gy[k] = 2.f * wt * a.cfg.lw[k] * d * a.inv_n;
      // the same in the four lane groups: over the 16 points in float64
      double ls = (double)(wt * a.cfg.lw[k] * d * d), bs = (double)gy[k];
#pragma unroll
      for (int off = 8; off > 0; off >>= 1) {
        ls += __shfl_xor(ls, off);
        bs += __shfl_xor(bs, off);
      }
      if (lane == 0) {
        s_loss[wave][0] += ls;
        s_loss[wave][1 + k] += bs;
      }
    }
    rows_exchange(v, c);
#pragma unroll 1
    for (int k = 0; k < 4; ++k) small_sums<true>(v, pick4(gy, k), rows + (7 + k) * kH, t == 0, g, c);
    // gZ_4, and down the chain gZ_l = (W_l^T gZ_{l+1}) silu'(Z_l)
    asm volatile("" ::: "memory");   // W4 is read again, not kept
    forget(z);
#pragma unroll
    for (int mt = 0; mt < 8; ++mt) {
      float gh[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const float4 w = small4(sW4 + k * kH + 16 * mt + 4 * g);
        gh[0] = fmaf(w.x, gy[k], gh[0]);
        gh[1] = fmaf(w.y, gy[k], gh[1]);
        gh[2] = fmaf(w.z, gy[k], gh[2]);
        gh[3] = fmaf(w.w, gy[k], gh[3]);
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) v[4 * mt + i] = gh[i] * dsilu(z[mt][i]);
    }
#pragma unroll 1
    for (int l = 2; l >= 0; --l) {
      // v = gZ_{l+2}: operand of the chain, of dW_{l+1}, and its bias sums
#pragma unroll
      for (int j = 0; j < 32; ++j) B[j >> 3][j & 7] = (__bf16)v[j];
      train_stage(sG, row, g, v);
      rows_exchange(v, c);
      small_sums<false>(v, 1.f, rows + (4 + l) * kH, t == 0, g, c);
      layer_get(Z, l, z);
#pragma unroll
      for (int j = 0; j < 32; ++j) v[j] = silu(z[j >> 2][j & 3]);
      train_stage(sH, row, g, v);
      forget(z);
      train_sync();   // the stages and W_{l+1}^T
      // next operand: W^T of the layer below, or W1 of the next tile
      train_load(l > 0 ? a.Wt + (l - 1) * kH * kH : a.Wp, buf + (l & 1) * kH * kH, wave, lane);
      train_dw(sG, sH, part + l * kH * kH, wave, g, c);
      floatx4 acc[8];
      train_mfma<false>(buf + ((l + 1) & 1) * kH * kH, nullptr, B, acc, g, c);
#pragma unroll
      for (int j = 0; j < 32; ++j) v[j] = acc[j >> 2][j & 3] * dsilu(z[j >> 2][j & 3]);
      __syncthreads();   // every wave has read the stages
    }
    rows_exchange(v, c);
#pragma unroll 1
    for (int d = 0; d < 4; ++d) small_sums<true>(v, pick4(f, d), rows + d * kH, t == 0, g, c);
  }
  // the small sums over the block's waves, the waves' loss and db4
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
  __threadfence_block();
  __syncthreads();
  const double* block = a.small_wave + (size_t)blockIdx.x * 8 * 11 * kH;
  double* out = a.small_part + (size_t)blockIdx.x * kSmallRow;
  for (int e = threadIdx.x; e < 11 * kH; e += kTrainThreads) {
    double s = 0.0;
#pragma unroll
    for (int w = 0; w < 8; ++w) s += block[(size_t)w * 11 * kH + e];
    out[e] = s;
  }
  if (threadIdx.x < 5) {
    double s = 0.0;
    for (int w = 0; w < 8; ++w) s += s_loss[w][threadIdx.x];
    out[threadIdx.x == 0 ? kNSmall : 11 * kH + threadIdx.x - 1] = s;
  }
}

// Gradients from the blocks' partial sums, each in a fixed order in float64.
// The first kDwBlocks blocks: 64 elements of dW1..dW3 each, four threads per
// element over a quarter of the tiles; the others: 16 small sums each, 16
// threads per sum over every 16th block.
constexpr int kDwBlocks = 3 * kH * kH / 64;
constexpr int kSmallBlocks = (kSmallRow + 15) / 16;
__global__ __launch_bounds__(256) void mlp_reduce_kernel(const float* __restrict__ dwpart,
                                                         const double* __restrict__ small_part,
                                                         int ntile, int nblk,
                                                         float* __restrict__ grads,
                                                         double* __restrict__ loss_out) {
  __shared__ double sh[256];
  const int t = threadIdx.x;
  if (blockIdx.x < kDwBlocks) {
    const int e = blockIdx.x * 64 + (t & 63);
    const int per = (ntile + 3) / 4, b0 = (t >> 6) * per, b1 = min(b0 + per, ntile);
    double s = 0.0;
#pragma unroll 8
    for (int b = b0; b < b1; ++b) s += (double)dwpart[(size_t)b * 3 * kH * kH + e];
    sh[t] = s;
    __syncthreads();
    if (t < 64)
      grads[kHidOff[e / (kH * kH)] + e % (kH * kH)] = (float)(((sh[t] + sh[64 + t]) + sh[128 + t]) + sh[192 + t]);
    return;
  }
  const int e = (blockIdx.x - kDwBlocks) * 16 + (t & 15), j = t >> 4;
  double s = 0.0;
  if (e < kSmallRow) {
#pragma unroll 4
    for (int b = j; b < nblk; b += 16) s += small_part[(size_t)b * kSmallRow + e];
  }
  sh[t] = s;
  __syncthreads();
  for (int w = 8; w > 0; w >>= 1) {
    if (j < w) sh[t] += sh[t + 16 * w];
    __syncthreads();
  }
  if (j != 0 || e >= kSmallRow) return;
  const double v = sh[t];
  if (e < 3 * kH) grads[kOffW0 + (e % kH) * kNIn + e / kH] = (float)v;
  else if (e < 7 * kH) {
    const int l = e / kH - 3;
    grads[(l == 0 ? kOffB0 : l == 1 ? kOffB1 : l == 2 ? kOffB2 : kOffB3) + e % kH] = (float)v;
  } else if (e < 11 * kH) grads[kOffW4 + e - 7 * kH] = (float)v;
  else if (e < kNSmall) grads[kOffB4 + e - 11 * kH] = (float)v;
  else if (loss_out) loss_out[0] = v;
}

// bf16 operand copies of W1..W3: Wp[l][o][k] = W[o][pi(k)], Wt[l][i][k] = W[pi(k)][i].
__global__ void mlp_sync_kernel(const float* __restrict__ params, __bf16* __restrict__ Wp,
                                __bf16* __restrict__ Wt) {
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  const int layer = blockIdx.y;
  if (e >= kH * kH) return;
  const int o = e / kH, i = e % kH;
  const __bf16 w = (__bf16)params[kHidOff[layer] + e];
  Wp[(size_t)layer * kH * kH + o * kH + pi_inverse(i)] = w;
  Wt[(size_t)layer * kH * kH + i * kH + pi_inverse(o)] = w;
}

struct AdamArgs {
  float lr, b1, b2, eps, c1, c2;  // c1 = 1 - b1^t, c2 = 1 - b2^t
};

__global__ void mlp_adam_kernel(float* __restrict__ params, const float* __restrict__ grads,
                                float* __restrict__ m, float* __restrict__ v, AdamArgs a) {
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= kNParams) return;
  const float gr = grads[e];
  const float mm = a.b1 * m[e] + (1.f - a.b1) * gr;
  const float vv = a.b2 * v[e] + (1.f - a.b2) * gr * gr;
  m[e] = mm;
  v[e] = vv;
  params[e] -= a.lr * (mm / a.c1) / (sqrtf(vv / a.c2) + a.eps);
}


// ---------------------------------------------------------------------------
// Orbit integration with the surrogate (integrate.py:129-143 update rule).
// ---------------------------------------------------------------------------
struct MLPOrbitAux {
  float ax, ay, az, maxerr;   // current acceleration, largest checked force error
  double e0, drift;           // initial energy (BFE potential), max |E - E0| / |E0|
  int nfallback, nchecked;    // BFE fallback evaluations, checked evaluations
};

struct MLPLeapArgs {
  float *x, *y, *z, *vx, *vy, *vz;
  int64_t n;
  double dt, t0, omega;
  int64_t k0, k1;             // steps (k0, k1] are taken
  int init;                   // 1: compute a0 and E0 at step k0 only
  int energy_check;           // 1: compare the energy at k1 with E0
  int check_period;           // every step 1 wave in check_period is checked against the BFE
  float rmax2, zmax;          // training domain R^2 < rmax2, |z| < zmax
  MLPOrbitAux* aux;
  double* partE;              // [checks][nblocks] block energy sums, or NULL
  int check_index, nblocks;
  const float* params;
  const __bf16* Wp;
  MLPCfg cfg;
  FieldTables T;
};

// The plain-BFE evaluation on the surrogate's rare paths (fallback, checks,
// energies) is an out-of-line call so that its float64 register demand does
// not add to the MLP loop's.
#ifndef BFE_MLP_INLINE_BFE
#define BFE_MLP_INLINE_BFE 0
#endif
#if BFE_MLP_INLINE_BFE
__device__ __forceinline__
#else
__device__ __noinline__
#endif
void bfe_point_call(const FieldTables& T, double x, double y, double z, double* cv) {
  field_eval_point(T, x, y, z, cv);
}

// Cartesian acceleration and potential of orbit (x, y, z) from the
// surrogate outputs, or from the BFE when the point is outside the domain.
// GRAD: yv holds (y0, dy0/df_0..2) of mlp_tile_grad, the forces are -grad.
template <bool GRAD>
__device__ __forceinline__ void surrogate_accel(const MLPLeapArgs& a, FieldTables& T, float x,
                                                float y, float z, const float (&yv)[4], float& fx,
                                                float& fy, float& fz, float& pot, bool& fb) {
  const float R2 = x * x + y * y;
  fb = !(R2 < a.rmax2 && fabsf(z) < a.zmax);
  if (fb) {
    double cv[8];
    bfe_point_call(T, x, y, z, cv);
    fx = (float)(cv[0] + cv[1]);
    fy = (float)(cv[2] + cv[3]);
    fz = (float)(cv[4] + cv[5]);
    pot = (float)(cv[6] + cv[7]);
    return;
  }
  if constexpr (GRAD) {
    const float dy[3] = {yv[1], yv[2], yv[3]};
    conservative_field(a.cfg, x, y, z, yv[0], dy, fx, fy, fz, pot);
    return;
  }
  const float R = sqrtf(R2);
  float bv[4];
  mlp_base_eval(a.cfg.base, R, z, bv);
  const float FR = a.cfg.os[1] * yv[1] + a.cfg.ob[1] + bv[1];
  const float Fp = a.cfg.os[2] * yv[2] + a.cfg.ob[2];
  const float cp = R > 0.f ? x / R : 1.f, sp = R > 0.f ? y / R : 0.f;
  fx = FR * cp - Fp * sp;
  fy = FR * sp + Fp * cp;
  fz = a.cfg.os[3] * yv[3] + a.cfg.ob[3] + bv[3];
  pot = a.cfg.os[0] * yv[0] + a.cfg.ob[0] + bv[0];
}

template <bool GRAD, int kBlock>
__global__ __launch_bounds__(kBlock) void mlp_leapfrog_kernel(MLPLeapArgs a) {
  // GRAD: conservative forces from mlp_tile_grad, 16-point tiles
  constexpr int NT = GRAD ? 1 : kNT;
  constexpr int kBlockPts = 16 * NT * (kBlock / 64);
  extern __shared__ __align__(16) unsigned char smem[];
  __bf16* sW = reinterpret_cast<__bf16*>(smem);
  float* sS = reinterpret_cast<float*>(smem + kLdsWBytes);
  __shared__ double s_e[kBlock / 64];
  load_small(a.params, sS);
  load_weights(a.Wp, sW);
  __syncthreads();
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int g = lane >> 4, c = lane & 15;
  const bool owner = g < NT;                       // lane (g, c) owns orbit 16 g + c of the wave
  const int64_t ntiles = (a.n + kBlockPts - 1) / kBlockPts;
  double esum = 0.0;
  FieldTables T = a.T;
  for (int64_t tile = blockIdx.x; tile < ntiles; tile += gridDim.x) {
    const int64_t base = tile * kBlockPts + wave * 16 * NT;
    const int64_t me = base + 16 * (owner ? g : 0) + c;
    const bool live = owner && me < a.n;
    float px = 0, py = 0, pz = 0, ux = 0, uy = 0, uz = 0;
    MLPOrbitAux o{};
    if (live) {
      px = a.x[me]; py = a.y[me]; pz = a.z[me];
      ux = a.vx[me]; uy = a.vy[me]; uz = a.vz[me];
      if (!a.init) o = a.aux[me];
    }
    const float dt = (float)a.dt, hdt = 0.5f * dt, hdt2 = 0.5f * dt * dt;
    const int64_t gwave = tile * (kBlock / 64) + wave;
    const int64_t kstart = a.init ? a.k0 : a.k0 + 1;
    for (int64_t k = kstart; k <= a.k1; ++k) {
      if (!a.init && live) {
        px = px + ux * dt + o.ax * hdt2;
        py = py + uy * dt + o.ay * hdt2;
        pz = pz + uz * dt + o.az * hdt2;
      }
      // surrogate forward for the wave's points (column c, tiles nt)
      float f[NT][3];
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) {
        const float qx = __shfl(px, 16 * nt + c), qy = __shfl(py, 16 * nt + c), qz = __shfl(pz, 16 * nt + c);
        mlp_features(a.cfg, qx, qy, qz, f[nt]);
      }
      float yk[NT][4];
      if constexpr (GRAD) {
        float y0[NT], dy[NT][3];
        mlp_tile_grad<NT>(sW, sS, f, y0, dy, g, c);
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
          yk[nt][0] = y0[nt];
          yk[nt][1] = dy[nt][0];
          yk[nt][2] = dy[nt][1];
          yk[nt][3] = dy[nt][2];
        }
      } else {
        mlp_tile_forward(sW, sS, f, yk, g, c);
      }
      if (live) {
        float yv[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          yv[q] = yk[0][q];
#pragma unroll
          for (int nt = 1; nt < NT; ++nt)
            if (g == nt) yv[q] = yk[nt][q];
        }
        if (a.omega != 0.0) {
          const double ang = a.omega * (a.t0 + (double)k * a.dt);
          T.crot = cos(ang);
          T.srot = sin(ang);
        }
        float nx, ny, nz, pot;
        bool fb;
        surrogate_accel<GRAD>(a, T, px, py, pz, yv, nx, ny, nz, pot, fb);
        if (fb) o.nfallback += 1;
        if (!fb && a.check_period > 0 && ((gwave + k) % a.check_period) == 0) {
          double cv[8];
          bfe_point_call(T, px, py, pz, cv);
          const double bx = cv[0] + cv[1], by = cv[2] + cv[3], bz = cv[4] + cv[5];
          const double err = sqrt((nx - bx) * (nx - bx) + (ny - by) * (ny - by) + (nz - bz) * (nz - bz)) /
                             sqrt(bx * bx + by * by + bz * bz);
          if (err > o.maxerr || !(err == err)) o.maxerr = (float)err;
          o.nchecked += 1;
        }
        if (a.init) {
          o.ax = nx; o.ay = ny; o.az = nz;
        } else {
          ux = ux + (o.ax + nx) * hdt;
          uy = uy + (o.ay + ny) * hdt;
          uz = uz + (o.az + nz) * hdt;
          o.ax = nx; o.ay = ny; o.az = nz;
        }
      }
    }
    if (live) {
      // energy with the BFE potential (the reference for measuring drift)
      if (a.init || a.energy_check) {
        if (a.omega != 0.0) {
          const double ang = a.omega * (a.t0 + (double)a.k1 * a.dt);
          T.crot = cos(ang);
          T.srot = sin(ang);
        }
        double cv[8];
        bfe_point_call(T, px, py, pz, cv);
        const double e = 0.5 * ((double)ux * ux + (double)uy * uy + (double)uz * uz) + (cv[6] + cv[7]);
        if (a.init) {
          o.e0 = e;
          o.drift = 0.0;
        } else {
          const double rel = fabs(e - o.e0) / fabs(o.e0);
          if (rel > o.drift || !(rel == rel)) o.drift = rel;
        }
        esum += e;
      }
      a.x[me] = px; a.y[me] = py; a.z[me] = pz;
      a.vx[me] = ux; a.vy[me] = uy; a.vz[me] = uz;
      a.aux[me] = o;
    }
  }
  if (a.partE) {
    for (int off = 32; off > 0; off >>= 1) esum += __shfl_xor(esum, off);
    if (lane == 0) s_e[wave] = esum;
    __syncthreads();
    if (threadIdx.x == 0) {
      double sum = 0.0;
      for (int w = 0; w < kBlock / 64; ++w) sum += s_e[w];
      a.partE[(size_t)a.check_index * a.nblocks + blockIdx.x] = sum;
    }
  }
}

__global__ void mlp_orbit_stats_kernel(const MLPOrbitAux* __restrict__ aux, int64_t n,
                                       double* __restrict__ drift, float* __restrict__ maxerr,
                                       int* __restrict__ counts) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  if (drift) drift[i] = aux[i].drift;
  if (maxerr) maxerr[i] = aux[i].maxerr;
  if (counts) {
    counts[2 * i] = aux[i].nfallback;
    counts[2 * i + 1] = aux[i].nchecked;
  }
}

__global__ void mlp_energy_reduce_kernel(const double* __restrict__ partE, int nchecks, int nblocks,
                                         double* __restrict__ log_out) {
  const int c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= nchecks) return;
  double s = 0.0;
  for (int b = 0; b < nblocks; ++b) s += partE[(size_t)c * nblocks + b];
  log_out[c] = s;
}

int field_tables(Context* c, double rotpos, FieldTables& T);

}  // namespace bfe

using namespace bfe;

namespace {

MLPCfg make_cfg(const MLPState& M) {
  const double* cfg = M.cfg;
  MLPCfg c;
  c.sxy = (float)cfg[0];
  c.hz = (float)cfg[1];
  c.wz = (float)cfg[2];
  for (int k = 0; k < 4; ++k) {
    c.os[k] = (float)cfg[3 + k];
    c.ob[k] = (float)cfg[7 + k];
  }
  // base layout: nmn, (M, a, b) x nmn, Mh, ah, phi0
  const double* b = M.base;
  c.base.nmn = (int)b[0];
  for (int k = 0; k < kMaxMN; ++k) {
    const bool on = k < c.base.nmn;
    c.base.M[k] = on ? b[1 + 3 * k] : 0.0;
    c.base.a[k] = on ? b[2 + 3 * k] : 0.0;
    c.base.b[k] = on ? b[3 + 3 * k] : 1.0;
  }
  const int o = 1 + 3 * c.base.nmn;
  c.base.mh = b[o];
  c.base.ah = b[o + 1];
  c.base.phi0 = b[o + 2];
  c.conservative = M.conservative;
  for (int k = 0; k < 4; ++k) c.lw[k] = (float)M.lw[k];
  return c;
}

int mlp_ready(Context* c) {
  if (!c->mlp.params) return set_error(c, BFE_ENOTABLE, "mlp: parameters not set (bfe_mlp_set_params)");
  return 0;
}

// 128-point tiles of a batch, and how many each block takes: as many as
// leave one block for each of the 256 CUs (a block fills a CU's LDS).
int64_t train_tiles(int64_t n) { return (n + kTrainPts - 1) / kTrainPts; }
int tiles_per_block(int64_t tiles) { return (int)((tiles + 255) / 256); }

int mlp_batch_buffers(Context* c, int64_t tiles, hipStream_t s) {
  MLPState& M = c->mlp;
  if (tiles <= M.bcap) return 0;
  BFE_HIP(c, hipStreamSynchronize(s));
  if (M.dwpart) (void)hipFree(M.dwpart);
  if (M.small_wave) (void)hipFree(M.small_wave);
  if (M.small_part) (void)hipFree(M.small_part);
  M.dwpart = nullptr;
  M.small_wave = nullptr;
  M.small_part = nullptr;
  M.bcap = 0;
  BFE_HIP(c, hipMalloc(&M.dwpart, sizeof(float) * 3 * kH * kH * (size_t)tiles));
  BFE_HIP(c, hipMalloc(&M.small_wave, sizeof(double) * 8 * 11 * kH * 256));
  BFE_HIP(c, hipMalloc(&M.small_part, sizeof(double) * kSmallRow * 256));
  M.bcap = tiles;
  return 0;
}

MLPKArgs base_args(Context* c) {
  MLPKArgs a{};
  a.params = c->mlp.params;
  a.Wp = c->mlp.Wp;
  a.cfg = make_cfg(c->mlp);
  return a;
}

// Gradient of the loss over n points.
int mlp_gradient(Context* c, const float* x, const float* y, const float* z, const float* target,
                 const float* weight, int64_t n, float* grads, double* loss_out, hipStream_t s) {
  const int64_t tiles = train_tiles(n);
  if (tiles > (int64_t)0x7fffffff) return set_error(c, BFE_ELIMIT, "mlp_gradient: n too large");
  int rc = mlp_batch_buffers(c, tiles, s);
  if (rc) return rc;
  MLPState& M = c->mlp;
  MLPTrainArgs a{};
  a.x = x; a.y = y; a.z = z; a.n = n;
  a.target = target;
  a.weight = weight;
  a.tiles = tiles_per_block(tiles);
  const int nblk = (int)((tiles + a.tiles - 1) / a.tiles);   // at most 256
  a.inv_n = 1.f / (float)n;
  a.params = M.params;
  a.Wp = M.Wp;
  a.Wt = M.Wt;
  a.dwpart = M.dwpart;
  a.small_wave = M.small_wave;
  a.small_part = M.small_part;
  a.cfg = make_cfg(M);
  hipLaunchKernelGGL(mlp_train_kernel, dim3((unsigned)nblk), dim3(kTrainThreads), kTrainLds, s, a);
  hipLaunchKernelGGL(mlp_reduce_kernel, dim3(kDwBlocks + kSmallBlocks), dim3(256), 0, s, M.dwpart,
                     M.small_part, (int)tiles, nblk, grads, loss_out);
  BFE_HIP(c, hipGetLastError());
  return 0;
}

int mlp_sync(Context* c, hipStream_t s) {
  hipLaunchKernelGGL(mlp_sync_kernel, dim3((kH * kH + 255) / 256, 3), dim3(256), 0, s,
                     c->mlp.params, c->mlp.Wp, c->mlp.Wt);
  BFE_HIP(c, hipGetLastError());
  return 0;
}

}  // namespace

namespace bfe {
void mlp_free(Context* c) {
  MLPState& M = c->mlp;
  for (float** p : {&M.params, &M.grads, &M.m, &M.v, &M.dwpart}) {
    if (*p) (void)hipFree(*p);
    *p = nullptr;
  }
  if (M.Wp) (void)hipFree(M.Wp);
  if (M.Wt) (void)hipFree(M.Wt);
  if (M.small_wave) (void)hipFree(M.small_wave);
  if (M.small_part) (void)hipFree(M.small_part);
  M = MLPState();
}
}  // namespace bfe

extern "C" int bfe_mlp_set_params(bfe_ctx* h, const float* params, int64_t count,
                                  const double* cfg) {
  if (!h) return BFE_EINVAL;
  Context* c = &h->c;
  if (count != kNParams) return set_error(c, BFE_EINVAL, "mlp: %lld params given, %d expected", (long long)count, kNParams);
  if (!params || !cfg) return set_error(c, BFE_EINVAL, "mlp: NULL params or cfg");
  if (!(cfg[0] > 0) || !(cfg[1] > 0) || !(cfg[2] > 0)) return set_error(c, BFE_EINVAL, "mlp: feature scales must be > 0");
  BFE_HIP(c, hipSetDevice(c->device));
  MLPState& M = c->mlp;
  if (!M.params) {
    BFE_HIP(c, hipMalloc(&M.params, sizeof(float) * kNParams));
    BFE_HIP(c, hipMalloc(&M.grads, sizeof(float) * kNParams));
    BFE_HIP(c, hipMalloc(&M.m, sizeof(float) * kNParams));
    BFE_HIP(c, hipMalloc(&M.v, sizeof(float) * kNParams));
    BFE_HIP(c, hipMalloc(&M.Wp, sizeof(__bf16) * 3 * kH * kH));
    BFE_HIP(c, hipMalloc(&M.Wt, sizeof(__bf16) * 3 * kH * kH));
    BFE_HIP(c, hipFuncSetAttribute((const void*)mlp_fwd_kernel,
                                   hipFuncAttributeMaxDynamicSharedMemorySize, (int)kLdsBytes));
    BFE_HIP(c, hipFuncSetAttribute((const void*)mlp_train_kernel,
                                   hipFuncAttributeMaxDynamicSharedMemorySize, (int)kTrainLds));
    BFE_HIP(c, hipFuncSetAttribute((const void*)mlp_leapfrog_kernel<false, kBlockInf>,
                                   hipFuncAttributeMaxDynamicSharedMemorySize, (int)kLdsBytes));
    BFE_HIP(c, hipFuncSetAttribute((const void*)mlp_leapfrog_kernel<true, kBlockGradSmall>,
                                   hipFuncAttributeMaxDynamicSharedMemorySize, (int)kLdsBytes));
    BFE_HIP(c, hipFuncSetAttribute((const void*)mlp_leapfrog_kernel<true, kBlockGrad>,
                                   hipFuncAttributeMaxDynamicSharedMemorySize, (int)kLdsBytes));
    BFE_HIP(c, hipFuncSetAttribute((const void*)mlp_fwd_grad_kernel,
                                   hipFuncAttributeMaxDynamicSharedMemorySize, (int)kLdsBytes));
  }
  BFE_HIP(c, hipMemcpy(M.params, params, sizeof(float) * kNParams, hipMemcpyHostToDevice));
  BFE_HIP(c, hipMemset(M.m, 0, sizeof(float) * kNParams));
  BFE_HIP(c, hipMemset(M.v, 0, sizeof(float) * kNParams));
  for (int k = 0; k < 11; ++k) M.cfg[k] = cfg[k];
  M.step = 0;
  int rc = mlp_sync(c, nullptr);
  if (rc) return rc;
  BFE_HIP(c, hipDeviceSynchronize());
  return 0;
}

extern "C" int bfe_mlp_set_base(bfe_ctx* h, const double* base, int count) {
  if (!h) return BFE_EINVAL;
  Context* c = &h->c;
  if (!base || count < 1) return set_error(c, BFE_EINVAL, "mlp_set_base: NULL or empty base");
  const int nmn = (int)base[0];
  if (base[0] != (double)nmn || nmn < 0 || nmn > kMaxMN)
    return set_error(c, BFE_EINVAL, "mlp_set_base: %g Miyamoto-Nagai components (0..%d)", base[0], kMaxMN);
  if (count != 4 + 3 * nmn)
    return set_error(c, BFE_EINVAL, "mlp_set_base: %d values given, %d expected", count, 4 + 3 * nmn);
  for (int k = 0; k < count; ++k)
    if (!std::isfinite(base[k])) return set_error(c, BFE_EINVAL, "mlp_set_base: non-finite value");
  for (int k = 0; k < nmn; ++k)
    if (!(base[3 + 3 * k] > 0.0)) return set_error(c, BFE_EINVAL, "mlp_set_base: b must be > 0");
  if (base[1 + 3 * nmn] != 0.0 && !(base[2 + 3 * nmn] > 0.0))
    return set_error(c, BFE_EINVAL, "mlp_set_base: Hernquist scale must be > 0");
  MLPState& M = c->mlp;
  for (int k = 0; k < kMLPBaseMax; ++k) M.base[k] = k < count ? base[k] : 0.0;
  return 0;
}

extern "C" int bfe_mlp_set_mode(bfe_ctx* h, int conservative, const double* loss_weights) {
  if (!h) return BFE_EINVAL;
  Context* c = &h->c;
  if (conservative != 0 && conservative != 1)
    return set_error(c, BFE_EINVAL, "mlp_set_mode: conservative must be 0 or 1");
  MLPState& M = c->mlp;
  for (int k = 0; k < 4; ++k) {
    const double w = loss_weights ? loss_weights[k] : 1.0;
    if (!(w >= 0.0) || !std::isfinite(w)) return set_error(c, BFE_EINVAL, "mlp_set_mode: loss weights must be >= 0");
    M.lw[k] = w;
  }
  M.conservative = conservative;
  return 0;
}

extern "C" int bfe_mlp_get_params(bfe_ctx* h, float* params, int64_t count) {
  if (!h) return BFE_EINVAL;
  Context* c = &h->c;
  if (int rc = mlp_ready(c)) return rc;
  if (count != kNParams || !params) return set_error(c, BFE_EINVAL, "mlp_get_params: bad buffer");
  BFE_HIP(c, hipSetDevice(c->device));
  BFE_HIP(c, hipDeviceSynchronize());
  BFE_HIP(c, hipMemcpy(params, c->mlp.params, sizeof(float) * kNParams, hipMemcpyDeviceToHost));
  return 0;
}

extern "C" int bfe_mlp_forward(bfe_ctx* h, const float* x, const float* y, const float* z,
                               int64_t n, float* out, void* stream) {
  if (!h) return BFE_EINVAL;
  Context* c = &h->c;
  if (int rc = mlp_ready(c)) return rc;
  if (n < 0) return set_error(c, BFE_EINVAL, "mlp_forward: n < 0");
  if (n == 0) return 0;
  if (!x || !y || !z || !out) return set_error(c, BFE_EINVAL, "mlp_forward: NULL pointer");
  BFE_HIP(c, hipSetDevice(c->device));
  hipStream_t s = (hipStream_t)stream;
  MLPKArgs a = base_args(c);
  a.x = x; a.y = y; a.z = z; a.n = n; a.out = out;
  if (c->mlp.conservative) {
    const GradLaunch g = mlp_grad_launch(n);
    hipLaunchKernelGGL(mlp_fwd_grad_kernel, dim3(g.blocks), dim3(kBlockGrad), kLdsBytes, s, a, g.waves, g.per);
    BFE_HIP(c, hipGetLastError());
    return 0;
  }
  const int64_t ntiles = (n + kInfPts - 1) / kInfPts;
  const int nb = (int)(ntiles < 1024 ? ntiles : 1024);
  hipLaunchKernelGGL(mlp_fwd_kernel, dim3(nb), dim3(kBlockInf), kLdsBytes, s, a);
  BFE_HIP(c, hipGetLastError());
  return 0;
}

extern "C" int bfe_mlp_gradient(bfe_ctx* h, const float* x, const float* y, const float* z,
                                const float* target, const float* weight, int64_t n,
                                float* grad_out, double* loss_out, void* stream) {
  if (!h) return BFE_EINVAL;
  Context* c = &h->c;
  if (int rc = mlp_ready(c)) return rc;
  if (n <= 0 || !x || !y || !z || !target || !grad_out)
    return set_error(c, BFE_EINVAL, "mlp_gradient: bad arguments");
  BFE_HIP(c, hipSetDevice(c->device));
  return mlp_gradient(c, x, y, z, target, weight, n, grad_out, loss_out, (hipStream_t)stream);
}

extern "C" int bfe_mlp_train_step(bfe_ctx* h, const float* x, const float* y, const float* z,
                                  const float* target, const float* weight, int64_t n, float lr,
                                  float beta1, float beta2, float eps, double* loss_out,
                                  void* stream) {
  if (!h) return BFE_EINVAL;
  Context* c = &h->c;
  if (int rc = mlp_ready(c)) return rc;
  if (n <= 0 || !x || !y || !z || !target) return set_error(c, BFE_EINVAL, "mlp_train_step: bad arguments");
  BFE_HIP(c, hipSetDevice(c->device));
  hipStream_t s = (hipStream_t)stream;
  MLPState& M = c->mlp;
  int rc = mlp_gradient(c, x, y, z, target, weight, n, M.grads, loss_out, s);
  if (rc) return rc;
  M.step += 1;
  AdamArgs a;
  a.lr = lr; a.b1 = beta1; a.b2 = beta2; a.eps = eps;
  a.c1 = (float)(1.0 - pow((double)beta1, (double)M.step));
  a.c2 = (float)(1.0 - pow((double)beta2, (double)M.step));
  hipLaunchKernelGGL(mlp_adam_kernel, dim3((kNParams + 255) / 256), dim3(256), 0, s, M.params, M.grads, M.m, M.v, a);
  BFE_HIP(c, hipGetLastError());
  return mlp_sync(c, s);
}

extern "C" int bfe_mlp_leapfrog(bfe_ctx* h, float* x, float* y, float* z, float* vx, float* vy,
                                float* vz, int64_t n, double dt, int64_t nsteps, double t0,
                                double rotfreq, int energy_every, float rmax, float zmax,
                                int check_period, double* drift_out, float* maxerr_out,
                                int* counts_out, double* energy_log, void* stream) {
  if (!h) return BFE_EINVAL;
  Context* c = &h->c;
  if (int rc = mlp_ready(c)) return rc;
  if (n < 0 || nsteps < 0 || energy_every < 0 || check_period < 0)
    return set_error(c, BFE_EINVAL, "mlp_leapfrog: negative size");
  if (n > 0 && (!x || !y || !z || !vx || !vy || !vz)) return set_error(c, BFE_EINVAL, "mlp_leapfrog: NULL state");
  if (energy_log && energy_every == 0) return set_error(c, BFE_EINVAL, "mlp_leapfrog: energy_log needs energy_every > 0");
  FieldTables T;
  int rc = field_tables(c, 0.0, T);
  if (rc) return rc;
  if (n == 0) return 0;
  BFE_HIP(c, hipSetDevice(c->device));
  hipStream_t s = (hipStream_t)stream;
  const LeapLaunch shape = mlp_leap_launch(n, c->mlp.conservative != 0);
  const int nb = shape.blocks;
  const int chunk = energy_every > 0 ? energy_every : (int)(nsteps < 100 ? (nsteps > 0 ? nsteps : 1) : 100);
  const int nchecks = energy_every > 0 ? (int)(nsteps / energy_every) + 1 : 1;
  const size_t aux_bytes = (size_t)n * sizeof(MLPOrbitAux);
  const size_t part_bytes = (size_t)nchecks * nb * sizeof(double);
  rc = ensure_scratch(c, ((aux_bytes + 255) & ~(size_t)255) + part_bytes);
  if (rc) return rc;
  MLPOrbitAux* aux = (MLPOrbitAux*)c->scratch;
  double* partE = (double*)((char*)c->scratch + ((aux_bytes + 255) & ~(size_t)255));
  MLPLeapArgs a{};
  a.x = x; a.y = y; a.z = z; a.vx = vx; a.vy = vy; a.vz = vz;
  a.n = n;
  a.dt = dt; a.t0 = t0; a.omega = 2.0 * kPi * rotfreq;
  a.check_period = check_period;
  a.rmax2 = rmax * rmax;
  a.zmax = zmax;
  a.aux = aux;
  a.nblocks = nb;
  a.params = c->mlp.params;
  a.Wp = c->mlp.Wp;
  a.cfg = make_cfg(c->mlp);
  a.T = T;
  // step 0: accelerations and initial energies
  a.init = 1;
  a.k0 = 0;
  a.k1 = 0;
  a.energy_check = 1;
  a.partE = energy_log ? partE : nullptr;
  a.check_index = 0;
  auto launch = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3(nb), dim3(64 * shape.waves), kLdsBytes, s, a);
  };
  auto go = [&]() {
    if (!a.cfg.conservative) launch(mlp_leapfrog_kernel<false, kBlockInf>);
    else if (shape.waves == kBlockGradSmall / 64) launch(mlp_leapfrog_kernel<true, kBlockGradSmall>);
    else launch(mlp_leapfrog_kernel<true, kBlockGrad>);
  };
  go();
  BFE_HIP(c, hipGetLastError());
  a.init = 0;
  for (int64_t k0 = 0, ci = 0; k0 < nsteps; k0 += chunk, ++ci) {
    a.k0 = k0;
    a.k1 = k0 + chunk < nsteps ? k0 + chunk : nsteps;
    a.energy_check = (energy_every > 0 && a.k1 - a.k0 == energy_every) ? 1 : 0;
    a.partE = (energy_log && a.energy_check) ? partE : nullptr;
    a.check_index = (int)ci + 1;
    go();
    BFE_HIP(c, hipGetLastError());
  }
  if (drift_out || maxerr_out || counts_out)
    hipLaunchKernelGGL(mlp_orbit_stats_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s,
                       aux, n, drift_out, maxerr_out, counts_out);
  if (energy_log)
    hipLaunchKernelGGL(mlp_energy_reduce_kernel, dim3((nchecks + 63) / 64), dim3(64), 0, s, partE,
                       nchecks, nb, energy_log);
  BFE_HIP(c, hipGetLastError());
  return 0;
}

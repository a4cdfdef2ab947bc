// fx_mlp.hpp -- the learned Newton seed of the exact Riemann solver: a
// 6 -> 64 -> 64 -> 1 tanh MLP evaluated and trained one wavefront (64
// interfaces) at a time on BF16 MFMA (v_mfma_f32_16x16x32_bf16) with FP32
// accumulation.  No counterpart in the reference.
//
// Features of an interface (Galilean and scale invariant): with
// P0 = sqrt(pL pR), R0 = sqrt(rhoL rhoR), C0 = sqrt(gamma P0 / R0),
//   x = (ln rhoL/R0, ln pL/P0, (uL - ubar)/C0, ln rhoR/R0, ln pR/P0, (uR - ubar)/C0)
// and the network predicts y = ln(p*/P0); the seed is P0 exp(y) (used where
// the interface is not weak, see fx_learned.hpp).
//
// Layout.  Layers compute H^T = W X^T (units as MFMA rows, interfaces as
// columns).  A 16x16 MFMA result tile sits in lane l as column l%16 and rows
// 4(l/16)+i, i<4, which is exactly the B-operand fragment of a K=16 slice;
// two result tiles form one K=32 operand when the K slots of lane group
// g = l/16 are taken as units {4g..4g+3} of the first tile then of the
// second.  The packed weight fragments use the same slot permutation, so
// layers chain in registers without shuffles.
#pragma once
#include <hip/hip_runtime.h>

namespace fx {

constexpr int MLP_IN = 6, MLP_H = 64;
constexpr int OFF_W1 = 0;                          // W1[64][6]
constexpr int OFF_B1 = OFF_W1 + MLP_H * MLP_IN;    // b1[64]
constexpr int OFF_W2 = OFF_B1 + MLP_H;             // W2[64 out][64 in]
constexpr int OFF_B2 = OFF_W2 + MLP_H * MLP_H;     // b2[64]
constexpr int OFF_W3 = OFF_B2 + MLP_H;             // w3[64]
constexpr int OFF_B3 = OFF_W3 + MLP_H;             // b3
constexpr int MLP_NPARAM = OFF_B3 + 1;             // 4673

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) float f32x4;

// round to nearest even (v_cvt_pk_bf16_f32)
__device__ __forceinline__ bf16x8 to_bf16x8(const float v[8]) {
  bf16x8 h;
#pragma unroll
  for (int j = 0; j < 8; ++j) h[j] = (__bf16)v[j];
  return h;
}

// tanh from the hardware exponential: 1 - 2 / (exp(2x) + 1), saturating to
// +-1 at both ends; a few ulp in FP32, ample for a Newton seed.  The powers of
// two are exact wherever they stand, so the first joins exp's log2(e) and the
// second an FMA; a reciprocal below 2^-25 leaves 1 whatever its value, so no
// operand needs scaling.  Inference is bound by these two quarter-rate
// operations (12 instructions a unit -> 6: 4M interfaces 311 -> 236 us,
// with v_cvt_pk_bf16_f32 for the operands).
__device__ __forceinline__ float act_tanh(float x) {
  const float e = __builtin_amdgcn_exp2f(x * (2.f * 1.4426950408889634f));
  return fmaf(-2.f, __builtin_amdgcn_rcpf(e + 1.f), 1.f);
}

__device__ __forceinline__ f32x4 mfma(bf16x8 a, bf16x8 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// unit held in K slot j of lane group g for K step ks (see the header note)
__device__ __forceinline__ int kslot_unit(int ks, int g, int j) {
  return 32 * ks + (j < 4 ? 4 * g + j : 16 + 4 * g + (j - 4));
}

// BF16 weight fragments in lane order plus FP32 biases.
struct MlpPacked {
  bf16x8 w1[4 * 64];     // [mt][lane]: rows 16mt + l%16, K slots = features 8g+j (< 6)
  bf16x8 w2[8 * 64];     // [mt][ks][lane]: W2[16mt + l%16][kslot_unit]
  bf16x8 w2t[8 * 64];    // [mt][ks][lane]: W2[kslot_unit][16mt + l%16]  (for W2^T)
  float b1[64], b2[64], w3[64], b3;
};

__global__ void k_mlp_pack(const float* __restrict__ prm, MlpPacked* out) {
  const int tid = blockIdx.x * blockDim.x + threadIdx.x;
  if (tid < 4 * 64) {
    const int mt = tid / 64, l = tid % 64, g = l / 16, c = l % 16;
    float v[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int f = 8 * g + j;
      v[j] = f < MLP_IN ? prm[OFF_W1 + (16 * mt + c) * MLP_IN + f] : 0.f;
    }
    out->w1[tid] = to_bf16x8(v);
  }
  if (tid < 8 * 64) {
    const int mt = tid / 128, ks = (tid / 64) % 2, l = tid % 64, g = l / 16, c = l % 16;
    float v[8], vt[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int u = kslot_unit(ks, g, j);
      v[j] = prm[OFF_W2 + (16 * mt + c) * MLP_H + u];
      vt[j] = prm[OFF_W2 + u * MLP_H + (16 * mt + c)];
    }
    out->w2[tid] = to_bf16x8(v);
    out->w2t[tid] = to_bf16x8(vt);
  }
  if (tid < 64) {
    out->b1[tid] = prm[OFF_B1 + tid];
    out->b2[tid] = prm[OFF_B2 + tid];
    out->w3[tid] = prm[OFF_W3 + tid];
  }
  if (tid == 0) out->b3 = prm[OFF_B3];
}

__device__ __forceinline__ void mlp_features(double g, double rl, double ul, double pl, double rr,
                                             double ur, double pr, float x[6], double& P0) {
  P0 = sqrt(pl * pr);
  const double R0 = sqrt(rl * rr);
  const double C0 = sqrt(g * P0 / R0);
  const float hr = 0.5f * logf((float)(rl / rr));
  const float hp = 0.5f * logf((float)(pl / pr));
  const float hu = (float)(0.5 * (ur - ul) / C0);
  x[0] = hr; x[1] = hp; x[2] = -hu;
  x[3] = -hr; x[4] = -hp; x[5] = hu;
}

// Activations of one wavefront (16 NT interfaces): result tile [mt][nt] of
// each layer, 4 floats per lane (column 16nt + l%16, rows 16mt + 4g + i).
template <int NT> struct MlpActs {
  f32x4 h1[4][NT];
  f32x4 h2[4][NT];
};

// xs: this wavefront's LDS block of 16 NT x 8 floats (features 0..5 used);
// yOut: interface lane's value in the first 16 NT lanes
template <int NT>
__device__ __forceinline__ void mlp_forward_wave(const MlpPacked& W, const float* xs, int lane,
                                                 MlpActs<NT>& A, float& yOut) {
  const int g = lane / 16, c = lane % 16;
  bf16x8 bx[NT];
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) {
    float v[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = (g == 0 && j < MLP_IN) ? xs[(16 * nt + c) * 8 + j] : 0.f;
    bx[nt] = to_bf16x8(v);
  }
#pragma unroll
  for (int mt = 0; mt < 4; ++mt) {
    const bf16x8 a = W.w1[mt * 64 + lane];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      f32x4 d = mfma(a, bx[nt], f32x4{0.f, 0.f, 0.f, 0.f});
#pragma unroll
      for (int i = 0; i < 4; ++i) d[i] = act_tanh(d[i] + W.b1[16 * mt + 4 * g + i]);
      A.h1[mt][nt] = d;
    }
  }
  // layer 2: K = 64 as two K=32 steps over result tiles (2ks, 2ks+1)
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) {
    bf16x8 b[2];
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      float v[8];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        v[j] = A.h1[2 * ks][nt][j];
        v[4 + j] = A.h1[2 * ks + 1][nt][j];
      }
      b[ks] = to_bf16x8(v);
    }
#pragma unroll
    for (int mt = 0; mt < 4; ++mt) {
      f32x4 d = mfma(W.w2[(mt * 2 + 0) * 64 + lane], b[0], f32x4{0.f, 0.f, 0.f, 0.f});
      d = mfma(W.w2[(mt * 2 + 1) * 64 + lane], b[1], d);
#pragma unroll
      for (int i = 0; i < 4; ++i) d[i] = act_tanh(d[i] + W.b2[16 * mt + 4 * g + i]);
      A.h2[mt][nt] = d;
    }
  }
  // layer 3 (64 -> 1) on the VALU: partial dot products, then across groups
  float part[NT];
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) {
    float s = 0.f;
#pragma unroll
    for (int mt = 0; mt < 4; ++mt)
#pragma unroll
      for (int i = 0; i < 4; ++i) s += W.w3[16 * mt + 4 * g + i] * A.h2[mt][nt][i];
    s += __shfl_xor(s, 16);
    s += __shfl_xor(s, 32);
    part[nt] = s;
  }
  // interface n = lane: its sum sits in part[n/16] of lane n%16
  float y = 0.f;
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) {
    const float v = __shfl(part[nt], c);
    if (g == nt) y = v;
  }
  yOut = y + W.b3;
}

// LDS ordering between lanes of one wavefront (no cross-wave barrier: the
// callers' loops are wavefront-uniform, not workgroup-uniform)
__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// sum over the 16 lanes of a lane group (same g), a DPP row: pairs, quads by
// permuting within four lanes, then eights and the row by mirroring
template <int CTRL> __device__ __forceinline__ float dpp_add(float v) {
  return v + __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(
                                           0, __builtin_bit_cast(int, v), CTRL, 0xF, 0xF, true));
}
__device__ __forceinline__ float group_sum(float v) {
  v = dpp_add<0xB1>(v);    // quad_perm [1,0,3,2]
  v = dpp_add<0x4E>(v);    // quad_perm [2,3,0,1]
  v = dpp_add<0x141>(v);   // row_half_mirror
  return dpp_add<0x140>(v);   // row_mirror
}

// Gradient of sum_n dy[n] * y[n] with respect to the parameters, one workgroup
// on kGradWaves * kGradCols interfaces at a time; every sum stays in registers
// from one set to the next.
constexpr int kGradNT = 2, kGradCols = 16 * kGradNT;   // interfaces of a wavefront
constexpr int kGradWaves = 4;                          // = the row tiles of W2
// rows of the bf16 operands of dW2, padded: 16-byte reads, and the four lane
// groups' writes fall into different banks
constexpr int kGradRow = kGradWaves * kGradCols + 8;
struct MlpGradAcc {
  f32x4 w2[4];      // dW2 rows 16 wave + 4g + i, columns 16ut + c, of all wavefronts' interfaces
  float unit[16];   // unit 16mt + 4g + i at [4mt + i], this wavefront's interfaces: lanes
                    // c = 0..5 dW1, 6 db1, 7 db2, 8 dw3
  float b3;         // each lane's own
};

// This wavefront's part; dZ2 and H1 go to sZ and sH (64 rows of kGradRow, this
// wavefront's columns) for mlp_grad_w2.  dy: this lane's interface (0 for lanes
// without one).
__device__ __forceinline__ void mlp_backward_wave(const MlpPacked& W, const float* xs, int lane,
                                                  const MlpActs<kGradNT>& A, float dy, __bf16* sZ,
                                                  __bf16* sH, MlpGradAcc& acc) {
  constexpr int NT = kGradNT;
  const int g = lane / 16, c = lane % 16;
  float dyc[NT], x[NT][MLP_IN];
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) {
    dyc[nt] = __shfl(dy, 16 * nt + c);
#pragma unroll
    for (int f = 0; f < MLP_IN; ++f) x[nt][f] = xs[(16 * nt + c) * 8 + f];
  }
  acc.b3 += dy;
  // output layer and layer-2 pre-activation gradient
  f32x4 dz2[4][NT];
#pragma unroll
  for (int mt = 0; mt < 4; ++mt)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int u = 16 * mt + 4 * g + i;
      float s3 = 0.f, s2 = 0.f;
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) {
        const float h = A.h2[mt][nt][i];
        const float z = W.w3[u] * dyc[nt] * (1.f - h * h);
        dz2[mt][nt][i] = z;
        s3 += dyc[nt] * h;
        s2 += z;
        sZ[u * kGradRow + 16 * nt + c] = (__bf16)z;
        sH[u * kGradRow + 16 * nt + c] = (__bf16)A.h1[mt][nt][i];
      }
      s2 = group_sum(s2);
      s3 = group_sum(s3);
      acc.unit[4 * mt + i] += c == 7 ? s2 : (c == 8 ? s3 : 0.f);
    }
  // dH1 = W2^T dZ2, chained from the dz2 tiles
  f32x4 dh1[4][NT];
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) {
    bf16x8 b[2];
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      float v[8];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        v[j] = dz2[2 * ks][nt][j];
        v[4 + j] = dz2[2 * ks + 1][nt][j];
      }
      b[ks] = to_bf16x8(v);
    }
#pragma unroll
    for (int mt = 0; mt < 4; ++mt) {
      f32x4 d = mfma(W.w2t[(mt * 2 + 0) * 64 + lane], b[0], f32x4{0.f, 0.f, 0.f, 0.f});
      dh1[mt][nt] = mfma(W.w2t[(mt * 2 + 1) * 64 + lane], b[1], d);
    }
  }
  // layer 1: dZ1, db1, dW1 (K = 6 features, on the VALU)
#pragma unroll
  for (int mt = 0; mt < 4; ++mt)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      float sum[MLP_IN + 1] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) {
        const float h = A.h1[mt][nt][i];
        const float z = dh1[mt][nt][i] * (1.f - h * h);
        sum[MLP_IN] += z;
#pragma unroll
        for (int f = 0; f < MLP_IN; ++f) sum[f] += z * x[nt][f];
      }
      float mine = 0.f;
#pragma unroll
      for (int f = 0; f <= MLP_IN; ++f) {
        const float v = group_sum(sum[f]);
        mine = c == f ? v : mine;
      }
      acc.unit[4 * mt + i] += mine;
    }
}

// dW2[o][in] += sum_n dZ2[o][n] H1[in][n] over the workgroup's interfaces:
// wavefront wv takes rows 16 wv .. 16 wv + 15.
__device__ __forceinline__ void mlp_grad_w2(int wv, int lane, const __bf16* sZ, const __bf16* sH,
                                            MlpGradAcc& acc) {
  const int g = lane / 16, c = lane % 16;
#pragma unroll
  for (int ks = 0; ks < kGradWaves * kGradCols / 32; ++ks) {
    const bf16x8 az =
        *reinterpret_cast<const bf16x8*>(&sZ[(16 * wv + c) * kGradRow + 32 * ks + 8 * g]);
#pragma unroll
    for (int ut = 0; ut < 4; ++ut)
      acc.w2[ut] = mfma(az,
                        *reinterpret_cast<const bf16x8*>(
                            &sH[(16 * ut + c) * kGradRow + 32 * ks + 8 * g]),
                        acc.w2[ut]);
  }
}

}  // namespace fx

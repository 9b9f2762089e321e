// Per-element gate math of the four cells, forward and adjoint, in fp32 registers.
// Shared by the fused kernels (a lane owns a few elements) and the alternating kernels
// (a thread owns one element).
//
// Forward definitions follow flashrnn/flashrnn/vanilla/{lstm,gru,elman,slstm}.py; adjoints
// follow flashrnn/flashrnn/alternating/{lstm,gru,slstm,elman}_pointwise.cu (backward kernels).
// Two deliberate differences from the reference's native kernels, both on the side of accuracy:
//  * all arithmetic is fp32 whatever the storage type (the reference computes in the storage
//    type, flashrnn/flashrnn/fused/lstm_fused_pointwise.cuh:48-87);
//  * the sLSTM cache holds the stabilised forget gate exp(logsig(f)+m-m') and sigmoid(-f)
//    instead of the raw f (slstm_fused_pointwise.cuh:75), so that the backward pass does not
//    rebuild them from storage-rounded f and m.
#pragma once
#include "frnn_common.h"

namespace frnn {

// Which product of a sum is contracted into a fused multiply-add is written out in the forward math, not left to the compiler
// (whose choice between f * c + (i * z) and (f * c) + i * z differs from kernel to kernel): a step then rounds the same way in every
// tiling, tile height and kernel, and single steps give the bits of a sequence whichever kernels run them.  The forms are those that
// it had chosen for nearly all of them: the product with the carried state is the one that is not rounded.
template <bool FAST> struct Math {
  static __device__ __forceinline__ float exp(float x) { return FAST ? __expf(x) : expf(x); }
  static __device__ __forceinline__ float rcp(float x) { return FAST ? __builtin_amdgcn_rcpf(x) : 1.0f / x; }
  static __device__ __forceinline__ float sigmoid(float x) { return rcp(1.0f + exp(-x)); }
  static __device__ __forceinline__ float tanh(float x) {
    if (FAST) return __builtin_fmaf(-2.0f, rcp(1.0f + __expf(2.0f * x)), 1.0f);
    return tanhf(x);
  }
  // log(sigmoid(x)) = min(x,0) - log1p(exp(-|x|))
  static __device__ __forceinline__ float logsigmoid(float x) {
#pragma clang fp contract(off)
    const float e = exp(-fabsf(x));
    return fminf(x, 0.0f) - (FAST ? __logf(1.0f + e) : log1pf(e));
  }
};

// a product that is rounded, whatever it is added to
__device__ __forceinline__ float mul(float a, float b) {
#pragma clang fp contract(off)
  return a * b;
}

// fwd:  ry[GR] recurrent pre-activations WITH the bias of their gate slot already added (the
//       fused kernels fold it into the MFMA accumulator), wx[GW], bx = biases of the gate slots
//       that have no recurrent input (gru: the n gate), s[S] in/out, cache[NC] out
//       ONCE: the state that is a sum of products a * b + c (or -1); mix[3] = {a, b, c} where the caller asks for them
// bwd:  cache[NC], sp[S] = s_{t-1}, sn[S] = s_t, dso[S] upstream cotangent of s_t,
//       ds[S] in: running cotangent arriving from step t+1; out: cotangent for s_{t-1}
//       WITHOUT the recurrent term R^T dgr (the caller adds it to ds[0]);
//       dgr[GR] / dgw[GW] / dgb[GT]: cotangents of the R-side, Wx-side and bias pre-activations.
// prepare, finish: bwd in two halves, for reverse kernels that do the first ahead of time: what does not depend on the running cotangent, into NP
//       values, and the rest, which needs only those and ds.  bwd stays beside them: composed of the two, or with the values computed where
//       finish uses them, the same instructions come in another order (reverse pass, Elman B64 N2 D192 T256 112.6 -> 117.4 us, D160 105.8 -> 111.2,
//       recompute mode, sLSTM B64 N2 D128 331 -> 336).
template <int F, bool FAST> struct CellMath;

// A state a * b + c as it is stored in fp16: rounded once, from the exact sum.  Through the fp32 state it would be rounded twice, and
// 4e-5 of the stored values would be the farther of their two neighbours.  Written out because the compiler does it by
// itself in most kernels but not in all, and every kernel has to store the same bits.
__device__ __forceinline__ float fma_f16(const float* mix) {
  half_t h;
  asm("v_fma_mixlo_f16 %0, %1, %2, %3" : "=v"(h) : "v"(mix[0]), "v"(mix[1]), "v"(mix[2]));
  return (float)h;
}

template <bool FAST> struct CellMath<FRNN_LSTM, FAST> {
  typedef Math<FAST> M;
  static constexpr int ONCE = 1;
  static __device__ __forceinline__ void fwd(const float* ry, const float* wx, const float* b, float* s, float* cache, float* mix = nullptr) {
    const float i = M::sigmoid(wx[0] + ry[0]);
    const float f = M::sigmoid(wx[1] + ry[1]);
    const float z = M::tanh(wx[2] + ry[2]);
    const float o = M::sigmoid(wx[3] + ry[3]);
    const float iz = mul(i, z), c = __builtin_fmaf(f, s[1], iz);
    if (mix) { mix[0] = f; mix[1] = s[1]; mix[2] = iz; }
    s[1] = c;
    s[0] = mul(o, M::tanh(c));
    cache[0] = i; cache[1] = f; cache[2] = z; cache[3] = o;
  }
  static __device__ __forceinline__ void bwd(const float* cache, const float* sp, const float* sn, const float* dso,
                                             float* ds, float* dgr, float* dgw, float* dgb) {
    const float i = cache[0], f = cache[1], z = cache[2], o = cache[3];
    const float dy = dso[0] + ds[0];
    const float tc = M::tanh(sn[1]);
    const float dc = dso[1] + ds[1] + (1.0f - tc * tc) * o * dy;
    dgr[0] = i * (1.0f - i) * z * dc;
    dgr[1] = f * (1.0f - f) * sp[1] * dc;
    dgr[2] = (1.0f - z * z) * i * dc;
    dgr[3] = o * (1.0f - o) * tc * dy;
#pragma unroll
    for (int g = 0; g < 4; ++g) { dgw[g] = dgr[g]; dgb[g] = dgr[g]; }
    ds[0] = 0.0f;
    ds[1] = f * dc;
  }
  static constexpr int NP = 8;
  static __device__ __forceinline__ void prepare(const float* cache, const float* sp, const float* sn, const float* dso, float* p) {
    const float i = cache[0], f = cache[1], z = cache[2], o = cache[3];
    const float tc = M::tanh(sn[1]);
    p[0] = (1.0f - tc * tc) * o;
    p[1] = i * (1.0f - i) * z;
    p[2] = f * (1.0f - f) * sp[1];
    p[3] = (1.0f - z * z) * i;
    p[4] = o * (1.0f - o) * tc;
    p[5] = f; p[6] = dso[0]; p[7] = dso[1];
  }
  static __device__ __forceinline__ void finish(const float* p, float* ds, float* dgr, float* dgw, float* dgb) {
    const float dy = p[6] + ds[0];
    const float dc = p[7] + ds[1] + p[0] * dy;
    dgr[0] = p[1] * dc;
    dgr[1] = p[2] * dc;
    dgr[2] = p[3] * dc;
    dgr[3] = p[4] * dy;
#pragma unroll
    for (int g = 0; g < 4; ++g) { dgw[g] = dgr[g]; dgb[g] = dgr[g]; }
    ds[0] = 0.0f;
    ds[1] = p[5] * dc;
  }
};

template <bool FAST> struct CellMath<FRNN_SLSTM, FAST> {
  typedef Math<FAST> M;
  static constexpr int ONCE = 1;
  static __device__ __forceinline__ void fwd(const float* ry, const float* wx, const float* b, float* s, float* cache, float* mix = nullptr) {
    const float ir = wx[0] + ry[0];
    const float fr = wx[1] + ry[1];
    const float z = M::tanh(wx[2] + ry[2]);
    const float o = M::sigmoid(wx[3] + ry[3]);
    const float lfm = M::logsigmoid(fr) + s[3];
    // first step of a fresh sequence: n == 0 (per element, as the native reference kernels,
    // flashrnn/flashrnn/fused/slstm_fused_pointwise.cuh:54-62)
    const float mn = (s[2] == 0.0f) ? ir : fmaxf(ir, lfm);
    const float ig = M::exp(ir - mn);
    const float fg = M::exp(lfm - mn);
    const float iz = mul(ig, z), c = __builtin_fmaf(fg, s[1], iz);
    if (mix) { mix[0] = fg; mix[1] = s[1]; mix[2] = iz; }
    const float n = fmaxf(__builtin_fmaf(fg, s[2], ig), 1.0f);
    s[0] = mul(mul(o, c), M::rcp(n));
    s[1] = c; s[2] = n; s[3] = mn;
    cache[0] = ig; cache[1] = fg; cache[2] = z; cache[3] = o; cache[4] = M::sigmoid(-fr);
  }
  static __device__ __forceinline__ void bwd(const float* cache, const float* sp, const float* sn, const float* dso,
                                             float* ds, float* dgr, float* dgw, float* dgb) {
    const float ig = cache[0], fg = cache[1], z = cache[2], o = cache[3], omf = cache[4];
    const float dy = dso[0] + ds[0];
    const float dyi = dy * M::rcp(sn[2]);
    const float dc = dso[1] + ds[1] + dyi * o;
    const float dn = dso[2] + ds[2] - dyi * sn[0];
    dgr[0] = ig * (z * dc + dn);
    dgr[1] = fg * (dc * sp[1] + dn * sp[2]) * omf;
    dgr[2] = dc * ig * (1.0f - z * z);
    dgr[3] = (1.0f - o) * sn[0] * dy;
#pragma unroll
    for (int g = 0; g < 4; ++g) { dgw[g] = dgr[g]; dgb[g] = dgr[g]; }
    // the stabiliser m is held constant (slstm_pointwise.cu:205): no cotangent flows into it
    ds[0] = 0.0f; ds[1] = fg * dc; ds[2] = fg * dn; ds[3] = 0.0f;
  }
  static constexpr int NP = 14;
  static __device__ __forceinline__ void prepare(const float* cache, const float* sp, const float* sn, const float* dso, float* p) {
    const float ig = cache[0], fg = cache[1], z = cache[2], o = cache[3], omf = cache[4];
    p[0] = M::rcp(sn[2]); p[1] = o; p[2] = sn[0];
    p[3] = ig; p[4] = z; p[5] = fg; p[6] = sp[1]; p[7] = sp[2]; p[8] = omf;
    p[9] = 1.0f - z * z;
    p[10] = (1.0f - o) * sn[0];
    p[11] = dso[0]; p[12] = dso[1]; p[13] = dso[2];
  }
  static __device__ __forceinline__ void finish(const float* p, float* ds, float* dgr, float* dgw, float* dgb) {
    const float dy = p[11] + ds[0];
    const float dyi = dy * p[0];
    const float dc = p[12] + ds[1] + dyi * p[1];
    const float dn = p[13] + ds[2] - dyi * p[2];
    dgr[0] = p[3] * (p[4] * dc + dn);
    dgr[1] = p[5] * (dc * p[6] + dn * p[7]) * p[8];
    dgr[2] = dc * p[3] * p[9];
    dgr[3] = p[10] * dy;
#pragma unroll
    for (int g = 0; g < 4; ++g) { dgw[g] = dgr[g]; dgb[g] = dgr[g]; }
    // the stabiliser m is held constant (slstm_pointwise.cu:205): no cotangent flows into it
    ds[0] = 0.0f; ds[1] = p[5] * dc; ds[2] = p[5] * dn; ds[3] = 0.0f;
  }
};

template <bool FAST> struct CellMath<FRNN_GRU, FAST> {
  typedef Math<FAST> M;
  static constexpr int ONCE = -1;
  // R gates [g, r, z]; Wx gates [r, z, n]; bias gates [g, r, z, n]
  static __device__ __forceinline__ void fwd(const float* ry, const float* wx, const float* b, float* s, float* cache, float* = nullptr) {
    const float g = ry[0];
    const float r = M::sigmoid(wx[0] + ry[1]);
    const float z = M::sigmoid(wx[1] + ry[2]);
    const float nv = M::tanh(__builtin_fmaf(r, g, wx[2] + b[0]));
    s[0] = __builtin_fmaf(z, s[0], mul(1.0f - z, nv));
    cache[0] = g; cache[1] = r; cache[2] = z; cache[3] = nv;  // the candidate itself: the adjoint needs no tanh
  }
  static __device__ __forceinline__ void bwd(const float* cache, const float* sp, const float* sn, const float* dso,
                                             float* ds, float* dgr, float* dgw, float* dgb) {
    const float g = cache[0], r = cache[1], z = cache[2], nv = cache[3];
    const float dy = dso[0] + ds[0];
    const float dz = z * (1.0f - z) * dy * (sp[0] - nv);
    const float dn = dy * (1.0f - z) * (1.0f - nv * nv);
    const float dr = dn * g * r * (1.0f - r);
    const float dg = dn * r;
    dgr[0] = dg; dgr[1] = dr; dgr[2] = dz;
    dgw[0] = dr; dgw[1] = dz; dgw[2] = dn;
    dgb[0] = dg; dgb[1] = dr; dgb[2] = dz; dgb[3] = dn;
    ds[0] = z * dy;
  }
  static constexpr int NP = 9;
  static __device__ __forceinline__ void prepare(const float* cache, const float* sp, const float* sn, const float* dso, float* p) {
    const float g = cache[0], r = cache[1], z = cache[2], nv = cache[3];
    p[0] = dso[0]; p[1] = z * (1.0f - z); p[2] = sp[0] - nv; p[3] = 1.0f - z; p[4] = 1.0f - nv * nv;
    p[5] = g; p[6] = r; p[7] = 1.0f - r; p[8] = z;
  }
  static __device__ __forceinline__ void finish(const float* p, float* ds, float* dgr, float* dgw, float* dgb) {
    const float dy = p[0] + ds[0];
    const float dz = p[1] * dy * p[2];
    const float dn = dy * p[3] * p[4];
    const float dr = dn * p[5] * p[6] * p[7];
    const float dg = dn * p[6];
    dgr[0] = dg; dgr[1] = dr; dgr[2] = dz;
    dgw[0] = dr; dgw[1] = dz; dgw[2] = dn;
    dgb[0] = dg; dgb[1] = dr; dgb[2] = dz; dgb[3] = dn;
    ds[0] = p[8] * dy;
  }
};

template <bool FAST> struct CellMath<FRNN_ELMAN, FAST> {
  typedef Math<FAST> M;
  static constexpr int ONCE = -1;
  static __device__ __forceinline__ void fwd(const float* ry, const float* wx, const float* b, float* s, float*, float* = nullptr) {
    s[0] = M::tanh(wx[0] + ry[0]);
  }
  static __device__ __forceinline__ void bwd(const float*, const float*, const float* sn, const float* dso,
                                             float* ds, float* dgr, float* dgw, float* dgb) {
    const float dy = dso[0] + ds[0];
    dgr[0] = (1.0f - sn[0] * sn[0]) * dy;
    dgw[0] = dgr[0]; dgb[0] = dgr[0];
    ds[0] = 0.0f;
  }
  static constexpr int NP = 1;  // (never split: one product would move)
};

// Elman under forward_clipval: cache[0] is the unclamped tanh (the caller clamps s[0] after fwd)
template <bool FAST> struct CellMath<FRNN_ELMAN_CLIP, FAST> {
  typedef Math<FAST> M;
  static constexpr int ONCE = -1;
  static __device__ __forceinline__ void fwd(const float* ry, const float* wx, const float* b, float* s, float* cache, float* = nullptr) {
    s[0] = M::tanh(wx[0] + ry[0]);
    cache[0] = s[0];
  }
  static __device__ __forceinline__ void bwd(const float* cache, const float*, const float*, const float* dso,
                                             float* ds, float* dgr, float* dgw, float* dgb) {
    const float dy = dso[0] + ds[0];
    dgr[0] = (1.0f - cache[0] * cache[0]) * dy;
    dgw[0] = dgr[0]; dgb[0] = dgr[0];
    ds[0] = 0.0f;
  }
  static constexpr int NP = 1;  // (never split: one product would move)
};

}  // namespace frnn

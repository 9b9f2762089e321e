// One time step with carried state, fused backend, 16-bit types (frnn_fused_step).
//
// The scan kernel can run a single step, but it first loads its whole slice of R into registers, D * G_r / 8 fragments per wave, and
// a head has few workgroups so that they exchange little: LSTM B8 N3 D256, 24 workgroups that read 128 KB each, 7.8 us.  A single
// step exchanges nothing, so here R is spread over as many waves as it has (unit tile, gate) rows of fragments.  Kernel time, scan
// kernel's step -> this one (4-row tiles unless noted): LSTM N12 D64 B1 4.0 -> 3.7 us, N6 D128 B16 7.1 -> 4.5, N3 D256 B8 7.8 -> 5.0, D512 B8
// 11.6 -> 7.3, D768 B8 22.3 -> 10.9, D1024 B4 18.9 -> 11.6, B64 (16 rows) 21.9 -> 13.8; GRU D1024 B4 22.4 -> 11.2; Elman D1024 B4 11.0 -> 4.4, N12
// D64 B1 3.1 -> 3.2.
//
// The step gives the bits of the sequence kernel (with the fp32 carry): every gate of a tile is one chain of MFMAs in the order of
// that kernel's, which is why the waves split the gates and not k.  What that order depends on comes from the host with the
// tiling of a sequence call of the same size; the gate math rounds the same way in every kernel (frnn_pointwise.h).  Bound by the trip of R from memory (nothing of it survives in L2 from launch to
// launch): all fragments of up to RND k-steps are requested at once.
#include "frnn_fused_fwd.h"  // load_frag
#include "frnn_pointwise.h"
#include "frnn_step.h"

namespace frnn {

template <int F, typename T, int RND>
__global__ void __launch_bounds__(256) fused_step_kernel(const StepArgs a) {
  typedef Cell<F> C;
  typedef ST<T> X;
  typedef typename X::Frag Frag;
  typedef CellMath<F, X::FAST> CM;
  constexpr int GR = C::GR, GW = C::GW, GT = C::GT, S = C::S, NC = C::NC;
  __shared__ __attribute__((aligned(16))) float red[4][256];
  const int B = a.B, BS = a.BS, N = a.N, D = a.D, tiles = D / 16, KS = D / X::KM;
  const int tile = blockIdx.x % tiles, n = (blockIdx.x / tiles) % N, bt = blockIdx.x / (tiles * N);
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r16 = lane & 15, q4 = lane >> 4, d0 = tile * 16;
  const size_t ND = (size_t)N * D;
  const T* const Wx = static_cast<const T*>(a.Wx);
  const T* const R = static_cast<const T*>(a.R);
  const T* const bias = static_cast<const T*>(a.b);
  const T* const s0 = static_cast<const T*>(a.s0);
  T* const states = static_cast<T*>(a.states);

  // thread -> unit d0 + tid % 16 of batch row bt * 16 + tid / 16 for the gate math; its operands travel behind the fragments
  const int bl = tid >> 4, b = bt * 16 + bl, d = d0 + (tid & 15);
  const bool evalid = b < B;
  const int be = evalid ? b : 0;
  const size_t idx = (size_t)n * D + d;

  // ---- wave w: gate w of the tile (one-gate cells: chain w of the gate) x batch rows bt * 16 .. + 15 ----
  const int stride = GR == 1 ? a.nacc : 1, first = GR == 1 ? w : 0;
  const bool active = GR == 1 ? w < a.nacc : w < GR;  // (uniform)
  const int bm = bt * 16 + r16;
  const bool bvalid = bm < B;
  const T* const vrow = s0 + (size_t)(bvalid ? bm : 0) * ND + (size_t)n * D;
  const T* const rrow = R + ((size_t)((GR == 1 || !active ? 0 : w) * N + n) * D + d0 + r16) * D;
  const int rot = a.own_ks ? (tile / a.ut_wg) * a.own_ks : 0, half = KS / a.ksp;
  const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
  f32x4 acc[2] = {zero, zero};
  Frag vf[RND], rf[RND];
  auto request = [&](int i0) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < RND; ++j) {
      const int i = i0 + j * stride;
      vf[j] = rf[j] = Frag{};
      if (active && i < KS) {  // (uniform)
        const int ks = i + rot < KS ? i + rot : i + rot - KS;
        rf[j] = load_frag<T>(rrow, ks, q4);
        vf[j] = load_frag<T>(vrow, ks, q4);
        if (!bvalid) vf[j] = Frag{};
      }
    }
  };
  request(first);
  if (a.bias_first && active && (GR > 1 || w == 0)) {
    float v[4];
    unpack4<T>(*reinterpret_cast<const typename X::Vec4*>(bias + (size_t)((GR == 1 ? 0 : w) * N + n) * D + d0 + q4 * 4), v);
    acc[0] = f32x4{v[0], v[1], v[2], v[3]};
  }
  float bo[GR], wx[GW], bx[GT - GR + 1], s[S], cc[NC > 0 ? NC : 1];
#pragma unroll
  for (int g = 0; g < GR; ++g) bo[g] = (float)bias[(size_t)(g * N + n) * D + d];
#pragma unroll
  for (int g = GR; g < GT; ++g) bx[g - GR] = (float)bias[(size_t)(g * N + n) * D + d];
#pragma unroll
  for (int g = 0; g < GW; ++g) wx[g] = (float)Wx[((size_t)be * GW + g) * ND + idx];
#pragma unroll
  for (int k = 0; k < S; ++k)
    s[k] = a.carry ? a.carry[((size_t)k * B + be) * ND + idx] : (float)s0[((size_t)k * BS + be) * ND + idx];

  for (int i0 = first; i0 < KS; i0 += RND * stride) {
    if (i0 != first) request(i0);
#pragma unroll
    for (int j = 0; j < RND; ++j) {
      const int i = i0 + j * stride;
      if (i < KS) {  // (uniform)
        if (GR == 1 || i < half) acc[0] = X::mfma(rf[j], vf[j], acc[0]);
        else acc[1] = X::mfma(rf[j], vf[j], acc[1]);
      }
    }
  }
  if (a.ksp > 1) acc[0] += acc[1];
  *reinterpret_cast<f32x4*>(&red[w][lane * 4]) = acc[0];
  __syncthreads();
  if (!evalid) return;

  // (result layout of the MFMA: lane l holds units 4 * (l / 16) + i of batch row l % 16)
  const int src = (((tid & 15) >> 2) * 16 + bl) * 4 + (tid & 3);
  float ry[GR];
  if constexpr (GR == 1) {
    ry[0] = red[0][src];
    for (int j = 1; j < a.nacc; ++j) ry[0] += red[j][src];
  } else {
#pragma unroll
    for (int g = 0; g < GR; ++g) ry[g] = red[g][src];
  }
  if (!a.bias_first) {
#pragma unroll
    for (int g = 0; g < GR; ++g) ry[g] += bo[g];
  }
  float mix[3];
  CM::fwd(ry, wx, bx, s, cc, mix);
  s[0] = clamp_if(s[0], a.h_clip);
#pragma unroll
  for (int k = 0; k < S; ++k) {
    const float so = X::ID == FRNN_F16 && k == CM::ONCE ? fma_f16(mix) : s[k];
    const Dw<1> v = pack<1>(&so, (T*)0);
    reinterpret_cast<unsigned short*>(states)[((size_t)k * BS + b) * ND + idx] = (unsigned short)v.v[0];
    if (a.carry) a.carry[((size_t)k * B + b) * ND + idx] = s[k];
  }
}

template <int F, typename T> static int step_t(const StepArgs& a, hipStream_t st) {
  const dim3 grid((unsigned)((size_t)(a.D / 16) * a.N * ((a.B + 15) / 16)));
  const int ks = a.D / 32 / (Cell<F>::GR == 1 ? a.nacc : 1);
  if (ks <= 8) hipLaunchKernelGGL((fused_step_kernel<F, T, 8>), grid, dim3(256), 0, st, a);
  else if (ks <= 16) hipLaunchKernelGGL((fused_step_kernel<F, T, 16>), grid, dim3(256), 0, st, a);
  else hipLaunchKernelGGL((fused_step_kernel<F, T, 32>), grid, dim3(256), 0, st, a);
  return (int)hipGetLastError();
}

int launch_fused_step(int function, int dtype, const Plan& p, int tile_rows, StepArgs a, hipStream_t st) {
  const int GR = cell_dims(function).GR, ks = a.D / 32;
  a.ksp = fwd_k_split(p.D, p.waves, p.utw, p.kw);
  a.own_ks = fwd_own_slice_first(GR, p.D, p.waves, p.utw, p.kw, tile_rows, 2) ? a.D / p.kw / 32 : 0;
  a.ut_wg = p.waves * p.utw / a.ksp;
  const int nacc = p.utw * GR >= 3 ? 1 : p.utw * GR == 2 ? 2 : 4;  // (as in the sequence kernel)
  a.nacc = nacc < ks ? nacc : ks;
  a.bias_first = tile_rows == 16;
#define FRNN_STEP(F) return dtype == FRNN_BF16 ? step_t<F, bf16_t>(a, st) : step_t<F, half_t>(a, st);
  switch (function) {
    case FRNN_LSTM:  FRNN_STEP(FRNN_LSTM)
    case FRNN_SLSTM: FRNN_STEP(FRNN_SLSTM)
    case FRNN_GRU:   FRNN_STEP(FRNN_GRU)
    case FRNN_ELMAN: FRNN_STEP(FRNN_ELMAN)
    default:         FRNN_STEP(FRNN_ELMAN_CLIP)
  }
#undef FRNN_STEP
}

}  // namespace frnn

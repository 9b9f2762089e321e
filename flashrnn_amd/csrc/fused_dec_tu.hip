// One translation unit per (function, storage type): instantiates the resident decode kernel, i.e. the fused
// forward kernel in mailbox mode (4-row batch tiles), for the forward tilings in the plan table that a session may have.
// Build with -DFRNN_F=<0..3> -DFRNN_DT=<0|1|2>.
#include "frnn_fused_fwd.h"
#include "frnn_launch.h"

namespace frnn {

template <int Dv, int VAR, int W, int U, int K> static void (*dec_kernel_for(int order))(const FwdArgs) {
  if constexpr (VAR == 0 && order_compiled(Dv, 2)) { if (order == 2) return fused_fwd_kernel<FRNN_F, FRNN_TU_T, Dv, W, U, K, 4, true, false, 2>; }
  if constexpr (VAR == 0 && order_compiled(Dv, 4)) { if (order == 4) return fused_fwd_kernel<FRNN_F, FRNN_TU_T, Dv, W, U, K, 4, true, false, 4>; }
  // (the dense tilings and those that spread a head by splitting its tiles are never a session's)
  if constexpr (VAR != 0 && (VAR == kDenseVariant || fwd_k_split(Dv, W, U, K) > 1)) return nullptr;
  else return order > 1 ? nullptr : fused_fwd_kernel<FRNN_F, FRNN_TU_T, Dv, W, U, K, 4, true>;
}

template <>
int fused_dec_launch<FRNN_F, FRNN_DT>(const Plan& p, const FwdArgs& a, hipStream_t st) {
  const dim3 grid(grid_for(a.groups, p.kw));
#define FRNN_CASE(Dv, VAR, W, U, K, MTR)                                                     \
  if (p.D == Dv && p.waves == W && p.utw == U && p.kw == K) {                                 \
    auto kern = dec_kernel_for<Dv, VAR, W, U, K>(p.order);                                           \
    if (!kern) return FRNN_E_UNSUPPORTED;                                                     \
    hipLaunchKernelGGL(kern, grid, dim3(W * 64), 0, st, a);                                   \
    return (int)hipGetLastError();                                                            \
  }
  FRNN_TU_PLANS(FRNN_CASE)
#undef FRNN_CASE
  return FRNN_E_UNSUPPORTED;
}

}  // namespace frnn

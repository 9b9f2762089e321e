// Declarations shared between the per-(function, dtype) kernel translation units and the API.
#pragma once
#include "frnn_common.h"
#include "frnn_plan.h"
#include <mutex>
#include <unordered_map>

namespace frnn {

struct FwdArgs;
struct BwdArgs;

// Each is defined in exactly one translation unit (fused_fwd_tu.hip / fused_bwd_tu.hip compiled
// with -DFRNN_F=<function> -DFRNN_DT=<dtype>).  Return: hipError_t, or FRNN_E_UNSUPPORTED if the
// plan is not compiled in.
template <int F, int DT> int fused_fwd_launch(const Plan& p, const FwdArgs& a, hipStream_t st);
template <int F, int DT> int fused_bwd_launch(const Plan& p, const BwdArgs& a, hipStream_t st);
// the forward kernel as a resident decode kernel (mailbox mode, 4-row tiles): fused_dec_tu.hip, functions 0..3
template <int F, int DT> int fused_dec_launch(const Plan& p, const FwdArgs& a, hipStream_t st);

// plan table lookup: function, dtype, D, variant -> plan; false if none.
// backward: 0 forward, 1 reverse scan with gate cache, 2 reverse scan in recompute mode
bool find_plan(int function, int dtype, int D, int variant, int backward, Plan* out);

// dynamic LDS with which two workgroups of a kernel do not fit one compute unit (its static LDS, a constant of the code object, is asked once:
// the question takes longer than the rest of a launch)
inline size_t alone_on_a_compute_unit(const void* kern) {
  static std::mutex lock;
  static std::unordered_map<const void*, size_t> known;
  size_t more;
  {
    std::lock_guard<std::mutex> g(lock);
    const auto it = known.find(kern);
    if (it != known.end()) more = it->second;
    else {
      hipFuncAttributes at;
      if (hipFuncGetAttributes(&at, kern) != hipSuccess) { (void)hipGetLastError(); return 0; }
      const size_t half = 80 * 1024 + 512;
      more = known[kern] = at.sharedSizeBytes < half ? half - at.sharedSizeBytes : 0;
    }
  }
  if (more > 65536 && hipFuncSetAttribute(kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)more) != hipSuccess) { (void)hipGetLastError(); return 0; }
  return more;
}

}  // namespace frnn

#if defined(FRNN_F) && defined(FRNN_DT)
#if FRNN_DT == 0
#define FRNN_TU_T frnn::bf16_t
#elif FRNN_DT == 2
#define FRNN_TU_T frnn::half_t
#else
#define FRNN_TU_T float
#endif
#if FRNN_F == 0 || FRNN_F == 1
#if FRNN_DT != 1 && FRNN_F == 1
#define FRNN_TU_BWD_RC_PLANS FRNN_BWD_RC_PLANS_SLSTM_BF16
#elif FRNN_DT != 1
#define FRNN_TU_BWD_RC_PLANS FRNN_BWD_RC_PLANS_GR4_BF16
#else
#define FRNN_TU_BWD_RC_PLANS FRNN_BWD_RC_PLANS_GR4_F32
#endif
#elif FRNN_F == 2
#if FRNN_DT != 1
#define FRNN_TU_BWD_RC_PLANS FRNN_BWD_RC_PLANS_GR3_BF16
#else
#define FRNN_TU_BWD_RC_PLANS FRNN_BWD_RC_PLANS_GR3_F32
#endif
#else
#define FRNN_TU_BWD_RC_PLANS FRNN_BWD_RC_PLANS_NONE
#endif
#if FRNN_F == 0 || FRNN_F == 1
#if FRNN_DT != 1 && FRNN_F == 1
#define FRNN_TU_PLANS FRNN_PLANS_SLSTM_BF16
#define FRNN_TU_BWD_PLANS FRNN_BWD_PLANS_SLSTM_BF16
#elif FRNN_DT != 1
#define FRNN_TU_PLANS FRNN_PLANS_GR4_BF16
#define FRNN_TU_BWD_PLANS FRNN_BWD_PLANS_GR4_BF16
#elif FRNN_F == 1
#define FRNN_TU_PLANS FRNN_PLANS_GR4_F32
#define FRNN_TU_BWD_PLANS FRNN_BWD_PLANS_SLSTM_F32
#else
#define FRNN_TU_PLANS FRNN_PLANS_GR4_F32
#define FRNN_TU_BWD_PLANS FRNN_BWD_PLANS_GR4_F32
#endif
#elif FRNN_F == 2
#if FRNN_DT != 1
#define FRNN_TU_PLANS FRNN_PLANS_GR3_BF16
#define FRNN_TU_BWD_PLANS FRNN_BWD_PLANS_GR3_BF16
#else
#define FRNN_TU_PLANS FRNN_PLANS_GR3_F32
#define FRNN_TU_BWD_PLANS FRNN_BWD_PLANS_GR3_F32
#endif
#else
#if FRNN_DT != 1
#define FRNN_TU_PLANS FRNN_PLANS_GR1_BF16
#define FRNN_TU_BWD_PLANS FRNN_BWD_PLANS_GR1_BF16
#else
#define FRNN_TU_PLANS FRNN_PLANS_GR1_F32
#define FRNN_TU_BWD_PLANS FRNN_BWD_PLANS_GR1_F32
#endif
#endif
#endif

#ifdef FRNN_TU_PLANS
namespace frnn {
// whether the tables of this cell and type have a forward tiling of D units whose waves sum k in `parts` parts (then the default tiling
// of D is compiled with that order as well)
constexpr bool order_compiled(int D, int parts) {
#define FRNN_HAS(Dv, VAR, W, U, K, MTR) if (D == Dv && (VAR == 2 || VAR == 3) && fwd_k_split(Dv, W, U, K) == parts) return true;
  FRNN_TU_PLANS(FRNN_HAS)
#undef FRNN_HAS
  return false;
}
}  // namespace frnn
#endif

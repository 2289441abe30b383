// vedic_gemm_f32_tn.hip -- fp32 kernels, TN: A stored [K x M].
#include "vedic_gemm_f32.hpp"
#include "vedic_gemm_f32s.hpp"

namespace vedic {

VEDIC_F32_KINDS(2, CfgF32Narrow);
VEDIC_F32_KINDS(2, CfgF32Small);
VEDIC_F32S_KINDS(2, CfgSLarge);
VEDIC_F32S_KINDS(2, CfgSMid);
VEDIC_F32S_KINDS(2, CfgSSmall);

hipError_t launch_gemm_f32_direct_tn(bool vec, const GemmArgs& a, hipStream_t s) {
    if (!f32_use_split(2, a.M, a.N, a.K, vec, a.head_cols > 0, device_cu_count())) return launch_gemm_f32_mfma_op<2>(a, s);
    return launch_gemm_f32s_op<2, true>(a, s);
}

}  // namespace vedic

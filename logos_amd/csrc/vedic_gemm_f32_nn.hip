// vedic_gemm_f32_nn.hip -- fp32 kernels, NN: A and B row-major.
#include "vedic_gemm_f32.hpp"
#include "vedic_gemm_f32s.hpp"

namespace vedic {

VEDIC_F32_KINDS(0, CfgF32Narrow);
VEDIC_F32_KINDS(0, CfgF32Small);
VEDIC_F32S_KINDS(0, CfgSLarge);
VEDIC_F32S_KINDS(0, CfgSMid);
VEDIC_F32S_KERNEL(0, false, CfgSMid, EK_GENERIC);
VEDIC_F32S_KERNEL(0, false, CfgSSmall, EK_GENERIC);

hipError_t launch_gemm_f32_direct_nn(bool vec, const GemmArgs& a, hipStream_t s) {
    if (!f32_use_split(0, a.M, a.N, a.K, vec, a.head_cols > 0, device_cu_count())) return launch_gemm_f32_mfma_op<0>(a, s);
    return vec ? launch_gemm_f32s_op<0, true>(a, s) : launch_gemm_f32s_op<0, false>(a, s);
}

}  // namespace vedic

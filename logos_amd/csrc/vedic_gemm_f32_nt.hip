// vedic_gemm_f32_nt.hip -- fp32 kernels, NT: B stored [N x K].
#include "vedic_gemm_f32.hpp"
#include "vedic_gemm_f32s.hpp"

namespace vedic {

VEDIC_F32_KINDS(1, CfgF32Narrow);
VEDIC_F32_KINDS(1, CfgF32Small);
VEDIC_F32_KINDS(1, CfgF32WaveK);
VEDIC_F32S_KINDS(1, CfgSLarge);
VEDIC_F32S_KINDS(1, CfgSMid);
VEDIC_F32S_KERNEL(1, false, CfgSMid, EK_GENERIC);
VEDIC_F32S_KERNEL(1, false, CfgSSmall, EK_GENERIC);

hipError_t launch_gemm_f32_direct_nt(bool vec, const GemmArgs& a, hipStream_t s) {
    if (!f32_use_split(1, a.M, a.N, a.K, vec, a.head_cols > 0, device_cu_count())) return launch_gemm_f32_mfma_op<1>(a, s);
    return vec ? launch_gemm_f32s_op<1, true>(a, s) : launch_gemm_f32s_op<1, false>(a, s);
}

}  // namespace vedic

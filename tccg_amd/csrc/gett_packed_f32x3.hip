// Packed-operand GETT, FP32 on the BF16 MFMAs: pack blocks whose values the
// three parts do not hold exactly keep their FP32 bits, and the k-steps that
// read them run on the FP32 MFMA (gett_pack.hpp split_holds(), gett_packed.hpp
// PackedFrags::mma_f32()).
#include "gett_launch.hpp"

extern "C" int tccg_gett_f32_split(const float* A, const float* B, float* C, float alpha, float beta,
                                   const tccg_gett_plan* plan, void* workspace, size_t workspace_bytes,
                                   int prepacked, void* stream) {
  return tccg_lib::run_gett_packed<tccg::F32X3>(A, B, C, alpha, beta, plan, workspace, workspace_bytes, stream,
                                                !prepacked);
}

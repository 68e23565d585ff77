// FPUOp on the FP32 / FP64 matrix instructions with multiplicands narrower than the accumulators (reference
// configs/configs.jl:489-497): converted exactly on their way into LDS, as Julia's promotion converts them in fma(a, b, c).
#include "fpu_mfma_instances.inc"

namespace gk {

int family_fpu_mfma_mixed(const InstanceKey& key, const GemmArgs& args, dim3 grid, hipStream_t stream, int mode, InstanceInfo* info,
                          hipError_t* err) {
  GK_CHAIN_T(64, 64, 32, 2, 2, 2, 2, 1, _Float16, float, "64x64x32_w2x2_f16")
  GK_CHAIN_T(64, 64, 32, 2, 2, 2, 2, 1, float, double, "64x64x32_w2x2_f32_f64")
  return 0;
}

}  // namespace gk

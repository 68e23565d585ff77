// FPUOp on the FP64 matrix instructions: Float64 operands.
#include "fpu_mfma_instances.inc"

namespace gk {

int family_fpu_mfma_f64(const InstanceKey& key, const GemmArgs& args, dim3 grid, hipStream_t stream, int mode, InstanceInfo* info,
                        hipError_t* err) {
  GK_CHAIN_T(64, 64, 32, 2, 2, 2, 2, 1, double, double, "64x64x32_w2x2_f64")
  GK_CHAIN_T(32, 32, 32, 2, 2, 2, 2, 2, double, double, "32x32x32_w2x2_f64")
  return 0;
}

}  // namespace gk

// FPUOp on the FP32 matrix instructions, Float32 operands: the tiles of products that do not fill the chip.
#include "fpu_mfma_instances.inc"

namespace gk {

int family_fpu_mfma_f32_small(const InstanceKey& key, const GemmArgs& args, dim3 grid, hipStream_t stream, int mode, InstanceInfo* info,
                              hipError_t* err) {
  GK_CHAIN_T(64, 64, 32, 2, 2, 2, 2, 1, float, float, "64x64x32_w2x2_f32")
  GK_CHAIN_T(32, 32, 32, 2, 2, 3, 8, 2, float, float, "32x32x32_w2x2_f32")
  GK_CHAIN_T(32, 32, 32, 1, 1, 2, 2, 1, float, float, "32x32x32_w1x1_f32")
  return 0;
}

}  // namespace gk

// FPUOp on the FP32 matrix instructions, Float32 operands: the tiles of products that fill the chip.
#include "fpu_mfma_instances.inc"

namespace gk {

int family_fpu_mfma_f32_large(const InstanceKey& key, const GemmArgs& args, dim3 grid, hipStream_t stream, int mode, InstanceInfo* info,
                              hipError_t* err) {
  GK_CHAIN_T(128, 128, 32, 2, 2, 3, 2, 1, float, float, "128x128x32_w2x2_f32")
  GK_CHAIN_T(128, 128, 16, 2, 2, 3, 2, 1, float, float, "128x128x16_w2x2_f32")
  return 0;
}

}  // namespace gk

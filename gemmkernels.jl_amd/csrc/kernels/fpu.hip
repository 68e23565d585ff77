// FPUOp and TropicalFPUOp: which kernel runs a launch, and the instances of the max-plus product.
//
// Floating-point FPUOp runs on the FP32 / FP64 matrix instructions (fpu_mfma.hpp: the same bits at two to six times the
// speed); the vector-ALU kernel (fpu_gemm.hpp) keeps what has no matrix instruction -- the max-plus product, the
// integers -- and the lane grids other than 8 x 8, which are a way of dealing outputs out to lanes of the vector ALUs.
#include "fpu_instances.inc"

// Whether a launch runs on the instances for one workgroup per CU (fpu_mfma_deep.hip; measured there): at most one tile per CU, and for
// 32 x 32 x 32, whose K tiles they fetch in pairs, a K of some length (256^3 4.8 us either way, 540 x 730 x 332 8.1, 8.7 in pairs).
static bool fpu_mfma_deep(const InstanceKey& key, const GemmArgs& args) {
  if (key.waves_m != 2 || key.waves_n != 2 || key.BK != 32 || key.BM != key.BN || (key.BM != 64 && key.BM != 32) || key.dtype != key.acc_dtype) return false;
  const long long tiles = (long long)((args.M + key.BM - 1) / key.BM) * ((args.N + key.BN - 1) / key.BN);
  return tiles <= kNumCUs && (key.BM == 64 || args.K >= 512);
}

int family_fpu(const InstanceKey& as_asked, const GemmArgs& args, dim3 grid, hipStream_t stream, int mode, InstanceInfo* info,
               hipError_t* err) {
  InstanceKey key = as_asked;
  key.variant &= ~kShallow;
  if ((key.variant >> 4) != 0) return family_fpu_lanes(key, args, grid, stream, mode, info, err);
  if ((key.variant & 1) == 0) {
    if ((as_asked.variant & kShallow) == 0 && fpu_mfma_deep(key, args) && family_fpu_mfma_deep(key, args, grid, stream, mode, info, err)) return 1;
    for (FamilyFn fn : {family_fpu_mfma_f32_large, family_fpu_mfma_f32_small, family_fpu_mfma_f64, family_fpu_mfma_mixed, family_fpu_integers})
      if (fn(key, args, grid, stream, mode, info, err)) return 1;
    return 0;
  }
  GK_FPU_T(64, 64, 32, 2, 2, float, 0, 1, "64x64x32_w2x2_f32_tropical")
  GK_FPU_T(64, 64, 32, 2, 2, float, 1, 1, "64x64x32_w2x2_f32_tropical_checked")
  return 0;
}

}  // namespace gk

// FPUOp on the FP32 / FP64 matrix instructions: the tiles of launches with at most one workgroup per CU.  Nothing else runs on the SIMD
// then, so a step that waits -- for the first fragments behind a barrier, for a tile on its way -- is time lost: three LDS
// stages with the first fragments read ahead of the barrier and the loads of two tiles in flight on 64 x 64 tiles, and K
// tiles of 64 (half the barriers) on 32 x 32 ones.  The same fma chains, same bits.  us, before -> after: Float64 1000^3 'T','N' 40.8 -> 36.7 (with
// factors on A and C 42.9 -> 41.4), 'N','N' 42.6 -> 41.4; Float32
// 1024^3 26.0 -> 24.0, 512^3 7.05 -> 6.7, 300 x 700 x 1500 17.8 -> 15.8, 64 x 64 x 8000 71 -> 56; Float64 107 x 16 x 7982 96 -> 89.  Where workgroups share a
// CU they cost more than they give: Float64 2048 x 2048 x 1024 136 -> 154, Float32 2048 x 1024 x 1024 on 32 x 32 46 -> 53.  More loads in
// flight (four, six) gain nothing.
#include "fpu_mfma_instances.inc"

namespace gk {

// (hook lists stay with the other instances: registers)
int family_fpu_mfma_deep(const InstanceKey& key, const GemmArgs& args, dim3 grid, hipStream_t stream, int mode, InstanceInfo* info,
                         hipError_t* err) {
  if (key.fused > 1) return 0;
#define GK_DEEP(bm_, bk_, STAGES, RING, DEPTH, T, akm_, bkm_, NAME)                                                                     \
  if (key.BM == bm_ && key.BN == bm_ && key.dtype == DtypeOf<T>::DT && key.a_kmajor == akm_ && key.b_kmajor == bkm_) {                 \
    if (key.fused == 0) {                                                                                                               \
      typedef FpuMfmaConfig<bm_, bm_, bk_, 2, 2, T, (akm_ != 0), (bkm_ != 0), T, 0, STAGES, RING, DEPTH> Plain;                         \
      return run_instance<Plain>(fpu_mfma_kernel<Plain>, NAME, args, grid, stream, mode, info, err, Plain::LDS_BYTES, Plain::THREADS);  \
    }                                                                                                                                   \
    typedef FpuMfmaConfig<bm_, bm_, bk_, 2, 2, T, (akm_ != 0), (bkm_ != 0), T, 1, STAGES, RING, DEPTH> Scale;                           \
    return run_instance<Scale>(fpu_mfma_kernel<Scale>, NAME "_fused", args, grid, stream, mode, info, err, Scale::LDS_BYTES, Scale::THREADS); \
  }
#define GK_DEEP_T(bm_, bk_, STAGES, RING, DEPTH, T, TAG)                                  \
  GK_DEEP(bm_, bk_, STAGES, RING, DEPTH, T, 0, 1, "fpu_mfma_nn_" TAG)                      \
  GK_DEEP(bm_, bk_, STAGES, RING, DEPTH, T, 0, 0, "fpu_mfma_nt_" TAG)                      \
  GK_DEEP(bm_, bk_, STAGES, RING, DEPTH, T, 1, 1, "fpu_mfma_tn_" TAG)                      \
  GK_DEEP(bm_, bk_, STAGES, RING, DEPTH, T, 1, 0, "fpu_mfma_tt_" TAG)
  GK_DEEP_T(64, 32, 3, 4, 2, float, "64x64x32_w2x2_s3_f32")
  GK_DEEP_T(32, 64, 3, 8, 2, float, "32x32x32_w2x2_pairs_f32")
  GK_DEEP_T(64, 32, 3, 2, 2, double, "64x64x32_w2x2_s3_f64")
  GK_DEEP_T(32, 64, 3, 4, 2, double, "32x32x32_w2x2_pairs_f64")
#undef GK_DEEP_T
#undef GK_DEEP
  return 0;
}

}  // namespace gk

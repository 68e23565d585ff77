// K-split instances of FPUOp on the FP32 / FP64 matrix instructions: Float32 and Float64 products with few output tiles and a long K, without hooks or
// with single factors.
//
// Such a launch waits for one fma chain per output, 8 (FP32) or 16 (FP64) clocks a k and more where a wave is alone on its SIMD, on a chip that
// is nearly idle.  Slices of K are as many shorter chains; the last workgroup to arrive at a tile adds them up in slice order (splitk_reduce), so the result is
// the same on every run.  Its error is that of the shorter chains and a few additions.  us on the device, one chain -> slices, 'N','N' on inputs that
// rotate: Float32 64 x 64 x 8000 57.0 -> 9.7 (16 slices), 448 x 31 x 7872 56.7 -> 12.3 (16), 320 x 24 x 1914 17.9 -> 7.4 (8), 64 x 833 x 2192 19.0 -> 9.4 (8),
// 392 x 36 x 730 9.4 -> 6.6 (6), 500 x 500 x 2000 19.3 -> 16.9 (4), 153 x 1808 x 7164 97.8 -> 60.3 (6), 1000 x 1000 x 4000 on 64 x 64 tiles 92.1 -> 79.0 (4); Float64 64 x 64 x 8000 90.8 ->
// 11.9 (16), 448 x 31 x 7872 89.6 -> 14.5 (16), 320 x 320 x 1000 15.6 -> 10.4 (6), 153 x 1808 x 7164 143.7 -> 92.2 (6), 500 x 500 x 2000 27.7 -> 24.4 (3).
// Tiles of 32 x 32 in K tiles of 32, of which a CU holds four or five: K tiles of 64 (one workgroup per CU in FP64) are up to 8 % faster where a CU has one
// workgroup and up to twice slower where it has four.  Float64 on 64 x 64 tiles gains nothing (1000^3 42.9 -> 42.6, 1000 x 1000 x 4000 142.1 -> 138.3).
#include "fpu_mfma.hpp"
#include "registry.hpp"

namespace gk {

int family_fpu_mfma_splitk(const InstanceKey& key, const GemmArgs& args, dim3 grid, hipStream_t stream, int mode, InstanceInfo* info,
                           hipError_t* err) {
  if (key.fused > 1 || key.BK != 32 || key.BM != key.BN || key.waves_m != 2 || key.waves_n != 2 || key.dtype != key.acc_dtype) return 0;
#define GK_SLICED(bm_, STAGES, RING, DEPTH, T, akm_, bkm_, NAME)                                                                             \
  if (key.BM == bm_ && key.dtype == DtypeOf<T>::DT && key.a_kmajor == akm_ && key.b_kmajor == bkm_) {                                       \
    if (key.fused == 0) {                                                                                                                    \
      typedef FpuMfmaConfig<bm_, bm_, 32, 2, 2, T, (akm_ != 0), (bkm_ != 0), T, 0, STAGES, RING, DEPTH, true> Plain;                         \
      return run_instance<Plain>(fpu_mfma_kernel<Plain>, NAME, args, grid, stream, mode, info, err, Plain::LDS_BYTES, Plain::THREADS);       \
    }                                                                                                                                        \
    typedef FpuMfmaConfig<bm_, bm_, 32, 2, 2, T, (akm_ != 0), (bkm_ != 0), T, 1, STAGES, RING, DEPTH, true> Scale;                           \
    return run_instance<Scale>(fpu_mfma_kernel<Scale>, NAME "_fused", args, grid, stream, mode, info, err, Scale::LDS_BYTES, Scale::THREADS); \
  }
#define GK_SLICED_T(bm_, STAGES, RING, DEPTH, T, TAG)                          \
  GK_SLICED(bm_, STAGES, RING, DEPTH, T, 0, 1, "fpu_mfma_splitk_nn_" TAG)      \
  GK_SLICED(bm_, STAGES, RING, DEPTH, T, 0, 0, "fpu_mfma_splitk_nt_" TAG)      \
  GK_SLICED(bm_, STAGES, RING, DEPTH, T, 1, 1, "fpu_mfma_splitk_tn_" TAG)      \
  GK_SLICED(bm_, STAGES, RING, DEPTH, T, 1, 0, "fpu_mfma_splitk_tt_" TAG)
  GK_SLICED_T(32, 3, 8, 2, float, "32x32x32_w2x2_f32")
  GK_SLICED_T(64, 2, 2, 1, float, "64x64x32_w2x2_f32")
  GK_SLICED_T(32, 2, 2, 2, double, "32x32x32_w2x2_f64")
#undef GK_SLICED_T
#undef GK_SLICED
  return 0;
}

}  // namespace gk

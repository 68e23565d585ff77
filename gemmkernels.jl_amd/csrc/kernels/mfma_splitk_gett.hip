// K-split instances of tensor contractions: the 64 x 64 x 64 tile on four LDS stages, without hooks or bias.
#include "mfma_gemm.hpp"
#include "registry.hpp"

namespace gk {

int family_mfma_splitk_gett(const InstanceKey& key, const GemmArgs& args, dim3 grid, hipStream_t stream, int mode, InstanceInfo* info,
                            hipError_t* err) {
  if (key.BM != 64 || key.BN != 64 || key.BK != 64 || key.waves_m != 2 || key.waves_n != 2 || key.dtype != DT_F16 || key.fused != 0) return 0;
#define GK_SKG(akm_, bkm_, NAME)                                                                                                         \
  if (key.a_kmajor == akm_ && key.b_kmajor == bkm_) {                                                                                    \
    typedef MfmaGemmConfig<64, 64, 64, 2, 2, 4, (akm_ ? OPK_KMAJOR : OPK_MMAJOR), (bkm_ ? OPK_KMAJOR : OPK_MMAJOR), _Float16, 0, true,   \
                           FIX_NONE, true, 16> Cfg;                                                                                      \
    return run_instance<Cfg>(mfma_gemm_kernel<Cfg>, NAME, args, grid, stream, mode, info, err, Cfg::LDS_BYTES, Cfg::THREADS);            \
  }
  GK_SKG(0, 1, "mfma_gemm_splitk_nn_64x64x64_w2x2_f16_gett")
  GK_SKG(0, 0, "mfma_gemm_splitk_nt_64x64x64_w2x2_f16_gett")
  GK_SKG(1, 1, "mfma_gemm_splitk_tn_64x64x64_w2x2_f16_gett")
  GK_SKG(1, 0, "mfma_gemm_splitk_tt_64x64x64_w2x2_f16_gett")
#undef GK_SKG
  return 0;
}

}  // namespace gk

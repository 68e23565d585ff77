// BF16 products with a factor on A, for the 'TT' transpose pair (A K-major, B M-major in memory).
#define GK_A_KMAJOR true
#define GK_B_KMAJOR false
#define GK_FAMILY_FN family_mfma_bf16_scaled_tt
#define GK_TAG "tt"
#include "mfma_bf16_scaled_instances.inc"

// BF16 products with a factor on A, for the 'NT' transpose pair (A M-major, B M-major in memory).
#define GK_A_KMAJOR false
#define GK_B_KMAJOR false
#define GK_FAMILY_FN family_mfma_bf16_scaled_nt
#define GK_TAG "nt"
#include "mfma_bf16_scaled_instances.inc"

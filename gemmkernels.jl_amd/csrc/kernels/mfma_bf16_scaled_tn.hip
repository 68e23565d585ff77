// BF16 products with a factor on A, for the 'TN' transpose pair (A K-major, B K-major in memory).
#define GK_A_KMAJOR true
#define GK_B_KMAJOR true
#define GK_FAMILY_FN family_mfma_bf16_scaled_tn
#define GK_TAG "tn"
#include "mfma_bf16_scaled_instances.inc"

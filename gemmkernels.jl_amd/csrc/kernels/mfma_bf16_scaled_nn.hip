// BF16 products with a factor on A, for the 'NN' transpose pair (A M-major, B K-major in memory).
#define GK_A_KMAJOR false
#define GK_B_KMAJOR true
#define GK_FAMILY_FN family_mfma_bf16_scaled_nn
#define GK_TAG "nn"
#include "mfma_bf16_scaled_instances.inc"

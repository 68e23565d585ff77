// The 128 x 128 and 64 x 64 tiles with four LDS stages, for the 'NN' transpose pair (A M-major, B K-major in memory).
#define GK_A_KMAJOR false
#define GK_B_KMAJOR true
#define GK_FAMILY_FN family_mfma_deep_nn
#define GK_TAG "nn"
#include "mfma_deep_instances.inc"

// The 128 x 128 and 64 x 64 tiles with four LDS stages, for the 'TT' transpose pair (A K-major, B M-major in memory).
#define GK_A_KMAJOR true
#define GK_B_KMAJOR false
#define GK_FAMILY_FN family_mfma_deep_tt
#define GK_TAG "tt"
#include "mfma_deep_instances.inc"

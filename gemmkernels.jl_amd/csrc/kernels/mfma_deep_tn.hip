// The 128 x 128 and 64 x 64 tiles with four LDS stages, for the 'TN' transpose pair (A K-major, B K-major in memory).
#define GK_A_KMAJOR true
#define GK_B_KMAJOR true
#define GK_FAMILY_FN family_mfma_deep_tn
#define GK_TAG "tn"
#include "mfma_deep_instances.inc"

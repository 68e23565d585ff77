// The 128 x 128 and 64 x 64 tiles with four LDS stages, for the 'NT' transpose pair (A M-major, B M-major in memory).
#define GK_A_KMAJOR false
#define GK_B_KMAJOR false
#define GK_FAMILY_FN family_mfma_deep_nt
#define GK_TAG "nt"
#include "mfma_deep_instances.inc"

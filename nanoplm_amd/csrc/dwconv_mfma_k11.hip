// Matrix-core kernels of 11 taps.
#define NPLM_K 11
#include "dwconv_mfma_inst.inc"

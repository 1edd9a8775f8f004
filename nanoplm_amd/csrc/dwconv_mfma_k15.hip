// Matrix-core kernels of 15 taps.
#define NPLM_K 15
#include "dwconv_mfma_inst.inc"

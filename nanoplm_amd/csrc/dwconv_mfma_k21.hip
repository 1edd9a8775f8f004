// Matrix-core kernels of 21 taps.
#define NPLM_K 21
#include "dwconv_mfma_inst.inc"

// Matrix-core kernels of 31 taps.
#define NPLM_K 31
#include "dwconv_mfma_inst.inc"

// Role-split kernels of 21 taps (K = 17, 19, 21).
#define NPLM_K 21
#include "dwconv_lds_inst.inc"

// LDS-staged forward, role-split backward and gated kernels of 11 taps (K = 11).
#define NPLM_K 11
#include "dwconv_lds_inst.inc"

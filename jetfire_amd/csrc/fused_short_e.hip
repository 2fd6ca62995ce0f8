// One-pass scan kernels of the fused decode step, INT4 keys with the bf16 scoring model
// in the form for short splits (SHORT in fused_scan_impl.h).
#define JF_SHORT_FORM
#include "fused_full_e.hip"

// One-pass scan kernels of the fused decode step, INT3 / INT4 keys with INT3 values
// in the form for short splits (SHORT in fused_scan_impl.h).
#define JF_SHORT_FORM
#include "fused_full_c.hip"

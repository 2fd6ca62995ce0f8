// One-pass scan kernels of the fused decode step, symmetric INT2 keys
// in the form for short splits (SHORT in fused_scan_impl.h).
#define JF_SHORT_FORM
#include "fused_full_b.hip"

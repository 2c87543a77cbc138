// Mixed-radix kernels, double.
#include "sgpe_mixed_inst.h"

template struct sgpe::MixKernels<double>;

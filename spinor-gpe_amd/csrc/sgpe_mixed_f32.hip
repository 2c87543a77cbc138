// Mixed-radix kernels, float.
#include "sgpe_mixed_inst.h"

template struct sgpe::MixKernels<float>;

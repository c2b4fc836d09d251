// k_reduce, lists of one-column tensors.

#include "tftq_reduce_kernels.h"

TFTQ_REDUCE_FLAVOUR(R_ONE)

// k_reduce, lists with rows of more than 16384 columns.

#include "tftq_reduce_kernels.h"

TFTQ_REDUCE_FLAVOUR(R_WIDE)

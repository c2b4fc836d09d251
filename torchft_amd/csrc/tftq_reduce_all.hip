// k_reduce, every kind of row.

#include "tftq_reduce_kernels.h"

TFTQ_REDUCE_FLAVOUR(R_ALL)

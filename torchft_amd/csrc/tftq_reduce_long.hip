// k_reduce, lists whose rows run in teams of 64 or 256 lanes.

#include "tftq_reduce_kernels.h"

TFTQ_REDUCE_FLAVOUR(R_LONG)

// FP64 matrix-core neighbour pass of ORDER 7.
#include "mfma64_kernels.h"

template struct sdg::mfma64::MfmaOrder64<7>;

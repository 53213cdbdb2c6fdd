// Matrix-core passes in the real type, ORDER 4.
#include "mx_local.h"
#include "mx_neighbor.h"

template struct sdg::mx::Order<4>;

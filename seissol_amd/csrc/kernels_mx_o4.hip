// Matrix-core passes in the real type, ORDER 4.
#include "mx_local.h"

template struct sdg::mx::Order<4>;

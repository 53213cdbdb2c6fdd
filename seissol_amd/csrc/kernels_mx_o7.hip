// Matrix-core passes in the real type, ORDER 7.
#include "mx_local.h"

template struct sdg::mx::Order<7>;

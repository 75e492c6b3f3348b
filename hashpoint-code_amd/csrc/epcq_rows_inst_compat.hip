// Row-run sampling kernels of neighbour mode compat (see epcq_rows_kernels.h).
#include "epcq_rows_kernels.h"

EPCQ_INSTANTIATE_ROWS(EPCQ_MODE_COMPAT, epcq::kCompatBuffer)

// Row-run sampling kernels of neighbour mode knn32 (see epcq_rows_kernels.h).
#include "epcq_rows_kernels.h"

EPCQ_INSTANTIATE_ROWS(EPCQ_MODE_KNN, 32)

// conv_rows_in.inc in FP64.
#include "conv_rows.hpp"

#define XATU_REAL double
#include "conv_rows_in.inc"

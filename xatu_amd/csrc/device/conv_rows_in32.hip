// conv_rows_in.inc in FP32.
#include "conv_rows.hpp"

#define XATU_REAL float
#include "conv_rows_in.inc"

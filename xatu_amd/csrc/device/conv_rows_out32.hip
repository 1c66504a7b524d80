// conv_rows_out.inc in FP32.
#include "conv_rows.hpp"

#define XATU_REAL float
#include "conv_rows_out.inc"

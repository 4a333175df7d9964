// Launchers of the int8 GEMM tiles with a zero point in the k loop or on ragged rows, epilogue DEQUANT_F32.
#include "qgemm_launch.h"

DQ8_INSTANTIATE_LAUNCH_ZP(DQ8_EPI_DEQUANT_F32)

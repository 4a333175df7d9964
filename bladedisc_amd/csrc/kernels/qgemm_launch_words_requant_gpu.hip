// Launchers of the int8 GEMM tiles on operand rows that begin on four bytes, epilogue REQUANT_GPU.
#include "qgemm_launch.h"

DQ8_INSTANTIATE_LAUNCH_WORDS(DQ8_EPI_REQUANT_GPU)

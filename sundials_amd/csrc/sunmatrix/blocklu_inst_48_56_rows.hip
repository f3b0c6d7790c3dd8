#include "blocklu_device.h"

LU_INSTANTIATE_ROW(48, double)
LU_INSTANTIATE_ROW(48, float)
LU_INSTANTIATE_ROW(56, double)
LU_INSTANTIATE_ROW(56, float)

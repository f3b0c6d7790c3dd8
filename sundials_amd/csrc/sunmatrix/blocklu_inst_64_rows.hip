#include "blocklu_device.h"

LU_INSTANTIATE_ROW(64, double)
LU_INSTANTIATE_ROW(64, float)

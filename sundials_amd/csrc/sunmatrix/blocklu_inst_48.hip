#include "blocklu_device.h"

LU_INSTANTIATE_SIZE(48, double)
LU_INSTANTIATE_SIZE(48, float)

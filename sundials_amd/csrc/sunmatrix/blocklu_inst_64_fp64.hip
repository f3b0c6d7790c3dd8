#include "blocklu_device.h"

LU_INSTANTIATE_SIZE(64, double)

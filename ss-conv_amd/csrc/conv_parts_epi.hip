// The bfloat16-parts form of the convolution kernel with the epilogue (conv_instances.h).
#include "conv_instances.h"

SSC_CONV_INSTANCE(1, 16, true, 4)
SSC_CONV_INSTANCE(2, 16, true, 4)
SSC_CONV_INSTANCE(1, 16, true, 5)
SSC_CONV_INSTANCE(2, 16, true, 5)

// The convolution kernel on float rows in its bfloat16-parts form (conv_instances.h).
#include "conv_instances.h"

SSC_CONV_INSTANCE(1, 16, false, 4)
SSC_CONV_INSTANCE(2, 16, false, 4)
SSC_CONV_INSTANCE(1, 16, false, 5)
SSC_CONV_INSTANCE(2, 16, false, 5)

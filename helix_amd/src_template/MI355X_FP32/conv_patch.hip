// FP32 convolution with the input under a block in LDS: see common/helix_conv_patch.h.
#define PATCH_F32 1
#include "helix_conv_patch.h"

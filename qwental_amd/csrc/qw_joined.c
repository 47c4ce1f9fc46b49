// The code object of the kernels that stand for several launches in one (kernels/qw_joined.hip.h), loaded beside the other one by qw_gpu_open.
#include "qw_internal.h"

QW_INTERNAL extern const unsigned char qw_joined_object[];
const unsigned char qw_joined_object[] = {
#embed <qw_joined_gfx950.hsaco>
};

// bridge_gen_0.hip -- fused generator kernels, part 0 of the step counts
// (bridge_gen.h).
#include "bridge_gen.h"

const void* koo::bridge_gen_kernel_0(int steps) { return gen_kernel<0>(steps); }

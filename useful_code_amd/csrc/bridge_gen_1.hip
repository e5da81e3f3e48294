// bridge_gen_1.hip -- fused generator kernels, part 1 of the step counts
// (bridge_gen.h).
#include "bridge_gen.h"

const void* koo::bridge_gen_kernel_1(int steps) { return gen_kernel<1>(steps); }

// bridge_gen_2.hip -- fused generator kernels, part 2 of the step counts
// (bridge_gen.h).
#include "bridge_gen.h"

const void* koo::bridge_gen_kernel_2(int steps) { return gen_kernel<2>(steps); }

// bridge_gen_3.hip -- fused generator kernels, part 3 of the step counts
// (bridge_gen.h).
#include "bridge_gen.h"

const void* koo::bridge_gen_kernel_3(int steps) { return gen_kernel<3>(steps); }

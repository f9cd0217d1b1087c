// mk_batch_one.hip — the batched decode kernel's one-layer instantiations as a
// translation unit of their own (the layer seam: a step of one layer per
// launch), so that the looping kernels' code does not change with them.
// Compiled with the thread index opaque (tid() in mk_common.h): with the plain
// one batch 20 took 64.1 us instead of 62.4, batch 3 37.5 instead of 36.9.
// mk_batch.hip's batch_kernel_for() hands these out.
#define MK_BATCH_ONE 1
#define MK_OPAQUE_TID 1
#include "mk_batch.hip"

// queue_1024.hip -- work-queue kernels, a 1024-thread workgroup per instance.
#include "queue_kernel.h"

namespace flock {
FLOCK_QUEUE_KERNELS(1024, 1024);
}  // namespace flock

// queue_256.hip -- work-queue kernels, a 256-thread workgroup per instance.
#include "queue_kernel.h"

namespace flock {
FLOCK_QUEUE_KERNELS(256, 256);
}  // namespace flock

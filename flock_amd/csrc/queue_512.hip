// queue_512.hip -- work-queue kernels, a 512-thread workgroup per instance.
#include "queue_kernel.h"

namespace flock {
FLOCK_QUEUE_KERNELS(512, 512);
}  // namespace flock

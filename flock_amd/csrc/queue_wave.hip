// queue_wave.hip -- work-queue kernels, a wavefront per instance.
#include "queue_kernel.h"

namespace flock {
FLOCK_QUEUE_KERNELS(256, 64);
FLOCK_QUEUE_KERNELS(128, 64);
FLOCK_QUEUE_KERNELS(64, 64);
}  // namespace flock

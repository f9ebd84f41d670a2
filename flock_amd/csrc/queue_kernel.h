// queue_kernel.h -- the persistent work-queue kernel (body: queue_worker in engine.h).
#pragma once
#include "kernels.h"

// The workgroup-per-
// instance configurations of up to 512 threads are held to 168 VGPRs, i.e. three waves
// per SIMD; the few values that spill are stored at kernel entry and reloaded once per
// instance, outside the pivot loop.
namespace flock {
template <int T, int G, int R>
struct QueueWaves { static constexpr int value = (G == T && T <= 512 && R != kRuleMulti) ? 3 : 1; };
template <int T, int G, int R>
__global__ __launch_bounds__(T) __attribute__((amdgpu_waves_per_eu(QueueWaves<T, G, R>::value))) void k_solve_queue(DevInstance* insts, const int32_t* order, int32_t count,
                                                   int32_t* head, EngineParams P) {
  extern __shared__ __align__(16) char smem[];
  queue_worker<T, G, R>(insts, order, count, head, P, smem);
}

#define FLOCK_QUEUE_KERNELS(T, G)                                                                                  \
  extern const void* const queue_kernels_##T##_##G[3] = {(const void*)k_solve_queue<T, G, kRuleDantzig>,           \
                                                         (const void*)k_solve_queue<T, G, kRuleCandidates>,        \
                                                         (const void*)k_solve_queue<T, G, kRuleMulti>}
}  // namespace flock

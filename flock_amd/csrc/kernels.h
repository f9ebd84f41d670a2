// kernels.h -- the compiled kernels by configuration.  Each workgroup size is a translation
// unit of its own, so they build in parallel.
#pragma once
#include "engine.h"

namespace flock {
// work-queue kernels k_solve_queue<threads, group, rule>, indexed by pricing rule
extern const void* const queue_kernels_256_64[3];
extern const void* const queue_kernels_128_64[3];
extern const void* const queue_kernels_64_64[3];
extern const void* const queue_kernels_256_256[3];
extern const void* const queue_kernels_512_512[3];
extern const void* const queue_kernels_1024_1024[3];
// large-instance path: set-up and rounds by workgroup size (and tree in global memory)
extern const void* const setup_kernel_512;
extern const void* const setup_kernel_1024;
extern const void* const round_kernels_512[3];
extern const void* const round_kernels_1024[3];
extern const void* const round_kernels_1024_global[3];
}  // namespace flock

__global__ void k_large_transpose(const flock::DevInstance* insts);
__global__ void k_large_books(const flock::DevInstance* insts, int16_t* books);
__global__ void k_large_sweep(flock::SweepArgs A);

// large.hip -- kernels of the large-instance path.
#include "kernels.h"

// Large-instance path (bodies in engine.h): setup and rounds run on one workgroup of
// T = 512 or 1024 threads, the sweep on a grid of 256-thread workgroups, one matrix tile
// each.
using namespace flock;

template <int T>
__global__ __launch_bounds__(T) void k_large_setup(DevInstance* insts, const int16_t* books, EngineParams P) {
  extern __shared__ __align__(16) char smem[];
  large_setup<T>(insts[0], smem, (size_t)P.lds_bytes, P, gl(books));
}
// Transpose of the cost matrix, one 64x64 tile per workgroup staged through LDS.
__global__ __launch_bounds__(256) void k_large_transpose(const DevInstance* insts) {
  __shared__ int32_t tile[64 * 65];
  const DevInstance& D = insts[0];
  const int m = D.m, n = D.n, ld = D.ld, ldT = D.ldT;
  const int32_t* cost = D.cost;
  int32_t* costT = D.costT;
  const int bi = (int)blockIdx.y * 64, bj = (int)blockIdx.x * 64;
  const int tx = (int)threadIdx.x % 64, ty = (int)threadIdx.x / 64;
  for (int r = ty; r < 64; r += 4) {
    const int i = bi + r, j = bj + tx;
    tile[r * 65 + tx] = (i < m && j < n) ? cost[(size_t)i * ld + j] : 0;
  }
  __syncthreads();
  for (int r = ty; r < 64; r += 4) {
    const int j = bj + r, i = bi + tx;
    if (j < n && i < m) costT[(size_t)j * ldT + i] = tile[tx * 65 + r];
  }
}
// Vogel books: one workgroup sorts one line (rows, then columns).
__global__ __launch_bounds__(256) void k_large_books(const DevInstance* insts, int16_t* books) {
  __shared__ uint32_t keys[16384];  // a line of up to 16384 entries (m+n <= 16383)
  const DevInstance& D = insts[0];
  Ctx C;
  C.cost = gl(uniform_ptr(D.cost)); C.costT = gl(uniform_ptr(D.costT));
  C.m = uniform(D.m); C.n = uniform(D.n); C.V = C.m + C.n; C.ld = uniform(D.ld); C.ldT = uniform(D.ldT);
  line_book<256>(C, (int)blockIdx.x, keys, gl(books));
}
template <int T, int R, bool TG>
__global__ __launch_bounds__(T) void k_large_round(DevInstance* insts, DevInstance geo, const uint64_t* keys,
                                                   const int32_t* cands, int32_t nblocks, EngineParams P) {
  extern __shared__ __align__(16) char smem[];
  large_round<T, R, TG>(insts[0], geo, smem, (size_t)P.lds_bytes, P, keys, cands, nblocks);
}
__global__ __launch_bounds__(256) void k_large_sweep(SweepArgs A) {
  __shared__ Shared S;
  sweep_tile<256>(A, blockIdx.x, S);
}

namespace flock {
extern const void* const setup_kernel_512 = (const void*)k_large_setup<512>;
extern const void* const setup_kernel_1024 = (const void*)k_large_setup<1024>;
#define FLOCK_ROUNDS(T, TG) \
  {(const void*)k_large_round<T, kRuleDantzig, TG>, (const void*)k_large_round<T, kRuleCandidates, TG>, (const void*)k_large_round<T, kRuleMulti, TG>}
extern const void* const round_kernels_512[3] = FLOCK_ROUNDS(512, false);
extern const void* const round_kernels_1024[3] = FLOCK_ROUNDS(1024, false);
extern const void* const round_kernels_1024_global[3] = FLOCK_ROUNDS(1024, true);
#undef FLOCK_ROUNDS
}  // namespace flock

// engine.h -- a group of threads solves one balanced transportation instance end to end:
//   transpose -> Vogel (or north-west corner) -> basis tree in LDS (level by level over
//   the basic cells, which also yields the duals) -> loop { reduced-cost sweep fused with
//   argmin -> stepping-stone pivot with parallel cycle discovery and parallel subtree
//   re-rooting } -> basis, duals, objective.
//
// A group is either one 64-lane wavefront (G = 64: several instances per workgroup,
// lockstep execution, no workgroup barriers) or the whole workgroup (G = blockDim).
//
// Exact integer arithmetic throughout (int32 costs, flows, duals; int64 objective).
// The rules follow the reference's sequential path so that, with Dantzig pricing, the
// pivot sequence is the reference's (see the per-function citations).
//
// Tree representation (rooted at vertex 0 = row 0, the reference's BFS root,
// DUAL_solver.cu:44-46).  Vertices: rows 0..m-1, columns m..m+n-1.  For every
// non-root vertex x the basic arc (x, parent[x]) is stored at x:
//   parent[x], depth[x], slot[x] (basis slot of the arc), flow[x]
// plus a preorder numbering pre[x] and subtree size size[x], so that
//   y is an ancestor-or-self of x  <=>  pre[y] <= pre[x] < pre[y] + size[y].
// That O(1) test is what makes cycle discovery and subtree identification
// embarrassingly parallel over vertices.
//
// Every device function here is forced inline: an outlined one takes generic pointers, so
// its LDS accesses become flat ones, and its caller keeps a stack (Vogel's register mode
// outlined in the set-up kernel, for one).
#pragma once
#include "device_common.h"

namespace flock {

// ---------------------------------------------------------------------------
// groups
// ---------------------------------------------------------------------------
// The rank is opaque to the compiler at each call: values derived from it are computed
// again in the phase that uses them, where the optimiser would otherwise hoist them to the
// kernel's entry and spill them (up to 40 registers in the work-queue kernels).
template <int G>
__device__ __forceinline__ int grank() {
  int r = (int)(threadIdx.x % G);
  asm volatile("" : "+v"(r));
  return r;
}

// One wavefront executes in lockstep; this orders its LDS/global accesses for the compiler
// and the memory model at wavefront scope.
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}
template <int G>
__device__ __forceinline__ void gsync() {
  if constexpr (G == kWave) wave_sync();
  else __syncthreads();
}

// Scalars shared by one group; they sit at the start of the group's LDS region.
struct Shared {
  uint64_t red[17];
  int64_t tk[6];      // phase tick counters (rank 0 updates them), as DevInstance::ticks
  int64_t reprice_ticks;  // samples of this call's candidate re-pricings
  int32_t cnt;
  int32_t pend_row, pend_col;  // Vogel: kinds of line the next step rescans
  int32_t status;
  int32_t level[3];   // tree build: vertices that a level reached, in turn
  int32_t idx;
  int32_t stop;       // deadline reached (rank 0 decides, the group follows)
  int32_t pad0_[1];
  int32_t cnt2;       // Vogel, register mode: list count of the odd steps (cnt: the even ones)
  int32_t dlo[2];     // pivot: least depth of a cycle vertex (atomicMin), by pivot parity
  int32_t pad_[5];
  uint64_t red1[3][16];  // one-barrier reductions (group_min1 / group_max1), by buffer
};

// Every reduction orders the group's memory accesses before it with those after it: a
// workgroup's by its barrier, a wavefront's by a sync point of its own (its lane moves only
// touch registers, so the compiler could otherwise move LDS accesses across them).
template <int G>
__device__ __forceinline__ void reduction_sync() {
  if constexpr (G == kWave) gsync<G>();
}
template <int G>
__device__ __forceinline__ uint64_t group_min_u64(uint64_t x, Shared& S) {
  reduction_sync<G>();
  if constexpr (G == kWave) return wave_min_u64(x);
  else return block_min_u64<G>(x, S.red);
}
// One-barrier variants for the solve loop.  Buffer use: 0 candidate re-pricing and
// Vogel's penalty argmax, 1 the pivot's leaving arc, 2 the full sweep; consecutive
// reductions on one buffer always have another barrier between them.
template <int G, int kBuf>
__device__ __forceinline__ uint64_t group_min1_u64(uint64_t x, Shared& S) {
  reduction_sync<G>();
  if constexpr (G == kWave) return wave_min_u64(x);
  else return block_min1_u64<G>(x, S.red1[kBuf]);
}
template <int G, int kBuf>
__device__ __forceinline__ uint64_t group_max1_u64(uint64_t x, Shared& S) {
  reduction_sync<G>();
  if constexpr (G == kWave) return wave_max_u64(x);
  else return block_max1_u64<G>(x, S.red1[kBuf]);
}
// The same max on buffer 0 or 2 in turn, for a loop with no other barrier.
template <int G>
__device__ __forceinline__ uint64_t group_max_alt(uint64_t x, Shared& S, int odd) {
  reduction_sync<G>();
  if constexpr (G == kWave) return wave_max_u64(x);
  else return block_max1_u64<G>(x, S.red1[2 * odd]);
}
template <int G>
__device__ __forceinline__ int64_t group_sum_i64(int64_t x, Shared& S) {
  reduction_sync<G>();
  if constexpr (G == kWave) return wave_sum_i64(x);
  else return block_sum_i64<G>(x, S.red);
}

// ---------------------------------------------------------------------------
// LDS layout of one group.
//   [Shared][tree: parent depth (int16) | pre,size interleaved (int16 pairs) | slot vat (int16)
//    | flow (int32) | du | dv]
//   (vat[p]: the vertex at pre-order position p)
//   [aux: tree-build scratch, later the pivot's path snapshot]
// The Vogel state aliases tree+aux (Vogel finishes before the tree is built).  When
// tree+aux does not fit, aux lives in the instance's global scratch instead.
// ---------------------------------------------------------------------------
struct TreeLds {
  int16_t *parent, *depth, *ps, *slot, *vat;  // ps: pre-order number and subtree size, interleaved
  int32_t *flow, *du, *dv;
  __device__ __forceinline__ int16_t& pre(int x) const { return ps[2 * x]; }
  __device__ __forceinline__ int16_t& size(int x) const { return ps[2 * x + 1]; }
  // both in one 32-bit load: pre | size << 16
  __device__ __forceinline__ int32_t pre_size(int x) const {
    int32_t v;
    __builtin_memcpy(&v, ps + 2 * x, 4);
    return v;
  }
};

__host__ __device__ inline size_t align16(size_t x) { return (x + 15) & ~(size_t)15; }

__host__ __device__ inline size_t shared_bytes() { return align16(sizeof(Shared)); }

__host__ __device__ inline size_t tree_lds_bytes(int m, int n) {
  const int V = m + n;
  return 4 * align16(2 * (size_t)V) + 2 * align16(4 * (size_t)V) + align16(4 * (size_t)((m + 3) & ~3)) +
         align16(4 * (size_t)((n + 3) & ~3));
}
// Vogel state without its tracked keys: cover flags, residuals, penalties, scan list,
// tracked count/flag, book position
__host__ __device__ inline size_t vogel_lds_bytes(int m, int n);
// the register mode keeps no per-line penalty array (the penalties live in the ranks'
// argmax keys), so its line state is one V-word array smaller
__host__ __device__ inline size_t vogel_reg_lds_bytes(int m, int n) {
  return vogel_lds_bytes(m, n) - align16(4 * (size_t)(m + n));
}
__host__ __device__ inline size_t vogel_lds_bytes(int m, int n) {
  const int V = m + n;
  return align16((size_t)((m + 3) & ~3)) + align16((size_t)((n + 3) & ~3)) + 2 * align16(4 * (size_t)V) +
         2 * align16(2 * (size_t)V) + align16((size_t)V);
}
// aux region in int32 units: max(tree-build scratch, path snapshot)
//   build: cell ends, cell costs, depths, sizes, next positions, V each, the vertices by
//   level and where each level starts (int16)
//   snapshot: for each side of the cycle, vertex, slot (int16), pre | size << 16 and flow (int32)
//   of its vertices by depth, V entries each
__host__ __device__ inline size_t aux_ints(int m, int n) {
  const size_t V = (size_t)(m + n);
  const size_t build = 5 * V + 2 * (V / 2 + 1);
  const size_t snap = 2 * (2 * ((V + 1) / 2 + 4) + 2 * (V + 4));
  return build > snap ? build : snap;
}
// bytes of one group's LDS region (aux in LDS if that fits `cap`, else in global)
__host__ __device__ inline size_t group_lds_bytes(int m, int n, size_t cap, bool* aux_in_lds) {
  const size_t base = shared_bytes();
  const size_t tree = tree_lds_bytes(m, n);
  const size_t vog = vogel_lds_bytes(m, n);
  const size_t tile = 64 * 65 * 4;
  size_t full = base + tree + 4 * aux_ints(m, n);
  full = full > base + vog ? full : base + vog;
  full = full > base + tile ? full : base + tile;
  if (full <= cap) { if (aux_in_lds) *aux_in_lds = true; return full; }
  if (aux_in_lds) *aux_in_lds = false;
  size_t part = base + tree;
  part = part > base + vog ? part : base + vog;
  part = part > base + tile ? part : base + tile;
  return part;
}

__device__ __forceinline__ TreeLds carve_tree(char* base, int m, int n) {
  const int V = m + n;
  TreeLds t;
  size_t off = 0;
  t.parent = (int16_t*)(base + off); off += align16(2 * (size_t)V);
  t.depth = (int16_t*)(base + off); off += align16(2 * (size_t)V);
  t.ps = (int16_t*)(base + off); off += align16(4 * (size_t)V);
  t.slot = (int16_t*)(base + off); off += align16(2 * (size_t)V);
  t.vat = (int16_t*)(base + off); off += align16(2 * (size_t)V);
  t.flow = (int32_t*)(base + off); off += align16(4 * (size_t)V);
  t.du = (int32_t*)(base + off); off += align16(4 * (size_t)((m + 3) & ~3));
  t.dv = (int32_t*)(base + off);
  return t;
}

// Cycle snapshot used by the pivot (generic pointers: LDS or global aux): side 0 holds
// the cycle vertices that are ancestors of the entering row, side 1 those of the
// entering column, each indexed by depth.
// Addresses are computed from the side (no runtime-indexed pointer arrays, which would
// live in scratch memory).
template <class I32, class I16>
struct SnapT {
  I32* base;
  int h;     // int32 words per int16 array
  int w;     // int32 words per int32 array
  int side;  // int32 words per side
  __device__ __forceinline__ I16* vert(int k) const { return (I16*)(base + k * side); }
  __device__ __forceinline__ I16* slot(int k) const { return (I16*)(base + k * side + h); }
  // pre-order number | subtree size << 16 (one load per interval)
  __device__ __forceinline__ I32* ps(int k) const { return base + k * side + 2 * h; }
  __device__ __forceinline__ I32* flow(int k) const { return base + k * side + 2 * h + w; }
};

__device__ __forceinline__ int32_t pack_ps(int pre, int size) { return (int32_t)((uint32_t)(uint16_t)pre | ((uint32_t)size << 16)); }
__device__ __forceinline__ int ps_pre(int32_t v) { return (int)((uint32_t)v & 0xffffu); }
__device__ __forceinline__ int ps_size(int32_t v) { return (int)((uint32_t)v >> 16); }
// generic pointers (aux in LDS or in global scratch) and LDS-typed pointers (aux known
// to be in LDS: ds_read/ds_write instead of flat accesses)
typedef SnapT<int32_t, int16_t> Snap;
typedef SnapT<FLOCK_LDS int32_t, FLOCK_LDS int16_t> SnapL;
template <class SN>
__device__ __forceinline__ SN carve_snap(int32_t* aux, int V) {
  SN s;
  s.base = (decltype(s.base))aux;
  s.h = (V + 1) / 2 + 4;
  s.w = V + 4;
  s.side = 2 * s.h + 2 * s.w;
  return s;
}

typedef const FLOCK_GLOBAL int32_t gcint;
typedef FLOCK_GLOBAL int32_t gint;

struct Ctx {
  gcint* cost;
  gint* costT;
  int32_t m, n, V, ld, ldT;
};

__device__ __forceinline__ int32_t cost_at(const Ctx& C, int i, int j) { return C.cost[(uint32_t)(i * C.ld + j)]; }

// ---------------------------------------------------------------------------
// transpose: costT[j*ldT + i] = cost[i*ld + j], 64x64 tiles staged through LDS
// (reads and writes both coalesced).  Uses 64*65*4 bytes at `tile`.  Each rank's loads
// of a tile are issued together (clamped addresses, unconditional), so a tile costs one
// global round trip instead of one per row.  The tiles are software-pipelined: the
// loads of tile k+1 are issued before the stores of tile k, so they are not queued
// behind those stores (the vector memory counter counts loads and stores in issue
// order) and their latency overlaps tile k's LDS reads and stores.
// ---------------------------------------------------------------------------
template <int G>
__device__ __forceinline__ void transpose(const Ctx& C, int32_t* tile) {
  const int rk = grank<G>();
  const int tx = rk % 64, ty = rk / 64;
  constexpr int R = G / 64;                // rows of a tile per pass of the group
  constexpr int PER = 64 / R;              // tile rows per rank
  constexpr int CH = PER < 16 ? PER : 16;  // loads in flight per rank (one chunk)
  constexpr int NCH = PER / CH;            // chunks per tile
  const int mLast = C.m - 1, nLast = C.n - 1;
  const int tilesJ = (C.n + 63) >> 6, units = ((C.m + 63) >> 6) * tilesJ * NCH;
  int32_t v[CH];
  auto load_chunk = [&](int q) {  // chunk q % NCH of tile q / NCH
    const int k = q / NCH, c = q % NCH;
    const int bi = (k / tilesJ) << 6, bj = (k % tilesJ) << 6;
    const int j = bj + tx < nLast ? bj + tx : nLast;
#pragma unroll
    for (int u = 0; u < CH; ++u) {
      const int i = bi + ty + (c * CH + u) * R;
      v[u] = C.cost[(uint32_t)((i < mLast ? i : mLast) * C.ld + j)];
    }
  };
  auto unit = [&](int q) {
    const int k = q / NCH, c = q % NCH;
#pragma unroll
    for (int u = 0; u < CH; ++u) tile[(ty + (c * CH + u) * R) * 65 + tx] = v[u];
    if (c < NCH - 1) {  // uniform: more rows of this tile to load first
      load_chunk(q + 1);
      return;
    }
    gsync<G>();
    load_chunk(q + 1 < units ? q + 1 : q);  // unconditional (the last one reloads), so the wait is exact
    const int bi = (k / tilesJ) << 6, bj = (k % tilesJ) << 6;
    // Ranks past the matrix's last row or column store the edge element (the value the
    // edge rank stores at the same address), so every store is unconditional and the
    // compiler can wait for the next chunk's loads without waiting for these stores.
    const int i = bi + tx < mLast ? bi + tx : mLast;
    for (int c2 = 0; c2 < NCH; ++c2) {
      int32_t w[CH];
      int32_t jc[CH];
#pragma unroll
      for (int u = 0; u < CH; ++u) {
        const int jj = bj + ty + (c2 * CH + u) * R;
        jc[u] = jj < nLast ? jj : nLast;
        w[u] = tile[(i - bi) * 65 + (jc[u] - bj)];
      }
#pragma unroll
      for (int u = 0; u < CH; ++u) C.costT[(uint32_t)(jc[u] * C.ldT + i)] = w[u];
    }
    gsync<G>();
  };
  // The first unit is peeled, so every entry to the loop has the same memory operations
  // in flight (next loads, then this unit's stores) and the wait for the loads is exact.
  load_chunk(0);
  unit(0);
  for (int q = 1; q < units; ++q) unit(q);
}

// Padding cells of every row (in the library's own copy of the matrix) price positive in
// the sweeps, see kPadCost.
template <int G>
__device__ __forceinline__ void write_padding(const Ctx& C) {
  const int padw = C.ld - C.n;
  FLOCK_GLOBAL int32_t* cw = (FLOCK_GLOBAL int32_t*)C.cost;
  if (padw > 0)
    for (int e = grank<G>(); e < C.m * padw; e += G) cw[(uint32_t)((e / padw) * C.ld + C.n + e % padw)] = kPadCost;
}

// ---------------------------------------------------------------------------
// Vogel's approximation (restates IBFS_vogel.cu:546-769, the host variant):
//  * penalty of a line = 2nd smallest - smallest uncovered cost (kBig sentinels,
//    :588-606); rows are refreshed only after a row was eliminated and columns only
//    after a column was eliminated (prev_row/prev_col, :588-642), so one kind can be
//    stale -- restated as is;
//  * argmax over [rows | columns] keeps the LAST maximum (>=, :654);
//  * the min-cost cell of the chosen line is the FIRST minimum (<, :673, :723);
//  * res_d > res_s eliminates the row, otherwise the column (:690-703), except that
//    the last uncovered column is never eliminated (the reference is undefined there).
// Parallel form.  Every line tracks its kTrack smallest uncovered keys (cost << b |
// cross index, b = index bits of the cross kind), ascending, found by one wavefront
// scanning the line (or reading its sorted book).  Covering a line only removes keys,
// so the uncovered tracked keys stay the smallest uncovered keys of the line: the two
// smallest (the penalty) and the smallest (the chosen cell) come from LDS alone until
// fewer than two tracked keys are left of a line that had more cells, which is then
// scanned again.  A step is one pass in which every rank refreshes the penalties of
// its own lines (pending kind) and forms their argmax keys -- (penalty + 1, line,
// first uncovered tracked cell) -- one group max, and rank 0 eliminating; lines that
// need a scan raise a flag bit in their key, and the step then scans them and takes
// the max again.
// ---------------------------------------------------------------------------
constexpr int kTrack = 4;
constexpr uint8_t kTrackFull = 0x80;  // nt flag: the tracked keys were all of the line's uncovered cells

__device__ __forceinline__ int index_bits(int len) {
  int b = 0;
  while ((1 << b) < len) ++b;
  return b;
}
// penalty from the two smallest keys (~0u: absent, worth kBig)
__device__ __forceinline__ int32_t key_penalty(uint32_t k1, uint32_t k2, int b) {
  const int64_t v1 = k1 == ~0u ? (int64_t)kBig : (int64_t)(k1 >> b);
  const int64_t v2 = k2 == ~0u ? (int64_t)kBig : (int64_t)(k2 >> b);
  return (int32_t)(v2 - v1);
}

__device__ __forceinline__ void track_insert(uint32_t k, uint32_t* l) {
  const bool c0 = k < l[0], c1 = k < l[1], c2 = k < l[2], c3 = k < l[3];
  l[3] = c2 ? l[2] : (c3 ? k : l[3]);
  l[2] = c1 ? l[1] : (c2 ? k : l[2]);
  l[1] = c0 ? l[0] : (c1 ? k : l[1]);
  l[0] = c0 ? k : l[0];
}

// Line scan by one wavefront: the kTrack smallest uncovered keys of the line in
// ascending order into out[0..kTrack) (lane 0 writes), their count and full flag into
// *nt; returns the two smallest in k1/k2 (~0u when absent), uniform over the wave.
// 16-byte loads (the line starts 16-byte aligned and is padded to a multiple of 4),
// four cover flags read as one word, U vectors in flight per lane.
template <class TRK>
__device__ __forceinline__ void wave_line_track(gcint* data, int len, const uint8_t* crossCov, int lane, int b,
                                                TRK* out, uint8_t* nt, uint32_t& k1, uint32_t& k2) {
  uint32_t l[kTrack] = {~0u, ~0u, ~0u, ~0u};
  constexpr int U = 4;
  if (len <= U * kWave) {  // short line: one scalar load per lane and slot
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int j = lane + u * kWave;
      const int32_t c = data[j < len ? j : 0];
      const bool live = j < len && !crossCov[j < len ? j : 0];
      track_insert(live ? (((uint32_t)c << b) | (uint32_t)j) : ~0u, l);  // ~0u inserts nothing
    }
  }
  const int nvec = len > U * kWave ? (len + 3) >> 2 : 0;
  for (int v0 = lane; v0 < nvec; v0 += U * kWave) {
    i32x4 c[U];
    uint32_t f[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int v = v0 + u * kWave;
      const int vv = v < nvec ? v : 0;
      c[u] = *(const FLOCK_GLOBAL i32x4*)(data + 4 * vv);
      f[u] = *(const uint32_t*)(crossCov + 4 * vv);
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int v = v0 + u * kWave;
      const int j0 = v < nvec ? 4 * v : len;  // out-of-range vectors never count
      const int32_t cc[4] = {c[u].x, c[u].y, c[u].z, c[u].w};
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int j = j0 + e;
        const bool live = j < len && ((f[u] >> (8 * e)) & 0xffu) == 0;
        track_insert(live ? (((uint32_t)cc[e] << b) | (uint32_t)j) : ~0u, l);
      }
    }
  }
  // the kTrack smallest of the wave: every lane holds its own kTrack smallest, so
  // kTrack rounds of (wave min, the owner pops it) find them in order (keys are unique)
  uint32_t got[kTrack];
#pragma unroll
  for (int e = 0; e < kTrack; ++e) {
    const uint32_t mn = wave_min_u32(l[0]);
    got[e] = mn;
    if (l[0] == mn && mn != ~0u) { l[0] = l[1]; l[1] = l[2]; l[2] = l[3]; l[3] = ~0u; }
  }
  const bool more = __ballot(l[0] != ~0u) != 0;  // a further uncovered cell in some lane
  if (lane == 0) {
    int found = 0;
#pragma unroll
    for (int e = 0; e < kTrack; ++e) { out[e] = got[e]; found += got[e] != ~0u ? 1 : 0; }
    *nt = (uint8_t)(found | (more ? 0 : kTrackFull));
  }
  k1 = got[0]; k2 = got[1];
}

// ---------------------------------------------------------------------------
// Sorted lines ("books") for Vogel on large instances: line L's cross indices in
// increasing (cost, index) order -- row L at books + L*n, column q at books + m*n + q*m
// (int16).  The smallest uncovered keys of a line are then its first uncovered book
// entries, and entries before the first one stay covered for good, so each line
// keeps a read position that only moves forward.  One workgroup sorts one line: keys
// cost << b | index (b = index bits; cost * 2^b < 2^31 by the range contract) in LDS,
// bitonic.
// ---------------------------------------------------------------------------
typedef const FLOCK_GLOBAL int16_t gcshort;

template <int G>
__device__ __forceinline__ void line_book(const Ctx& C, int L, uint32_t* keys, FLOCK_GLOBAL int16_t* books) {
  const int m = C.m, n = C.n, tid = grank<G>();
  const bool row = L < m;
  gcint* data = row ? C.cost + (uint32_t)(L * C.ld) : C.costT + (uint32_t)((L - m) * C.ldT);
  FLOCK_GLOBAL int16_t* book = books + (row ? (size_t)L * n : (size_t)m * n + (size_t)(L - m) * m);
  const int len = row ? n : m;
  const int b = index_bits(len);
  const int npow = 1 << b;
  for (int i = tid; i < npow; i += G) keys[i] = i < len ? ((uint32_t)data[i] << b) | (uint32_t)i : 0xffffffffu;
  gsync<G>();
  for (int k = 2; k <= npow; k <<= 1)
    for (int j = k >> 1; j > 0; j >>= 1) {
      for (int i = tid; i < npow; i += G) {
        const int p = i ^ j;
        if (p > i) {
          const uint32_t a = keys[i], c = keys[p];
          if ((a > c) == ((i & k) == 0)) { keys[i] = c; keys[p] = a; }
        }
      }
      gsync<G>();
    }
  const uint32_t mask = (1u << b) - 1u;
  for (int i = tid; i < len; i += G) book[i] = (int16_t)(keys[i] & mask);
}

// Book read by one wavefront: the first kTrack uncovered entries from the read position
// *pos on (64 entries per ballot), as keys, with count and full flag; *pos moves to the
// first uncovered entry.  k1/k2 as for wave_line_track.
template <class TRK>
__device__ __forceinline__ void wave_book_track(gcshort* book, gcint* data, int len, int16_t* pos,
                                                const uint8_t* crossCov, int lane, int b, TRK* out, uint8_t* nt,
                                                uint32_t& k1, uint32_t& k2) {
  int at = *pos, found = 0, first = -1;
  wave_sync();  // every lane has the position before lane 0 moves it
  uint32_t r0 = ~0u, r1 = ~0u;  // this lane's key if it holds rank 0 / rank 1
  while (at < len && found <= kTrack) {
    const int q = at + lane;
    const int idx = q < len ? book[q] : 0;
    // every lane loads its entry's cost with the entry's cover flag (one global round trip
    // after the book read, instead of a second one after the ballot)
    const int32_t cst = data[idx];
    const bool live = q < len && !crossCov[idx];
    const uint64_t mask = __ballot(live);
    if (first < 0 && mask) first = at + __ffsll((unsigned long long)mask) - 1;
    if (live) {
      const int rank = found + __popcll(mask & ((1ull << lane) - 1ull));
      const uint32_t key = ((uint32_t)cst << b) | (uint32_t)idx;
      if (rank < kTrack) out[rank] = key;
      if (rank == 0) r0 = key;
      if (rank == 1) r1 = key;
    }
    found += __popcll(mask);
    at += kWave;
  }
  if (lane == 0) {
    *pos = (int16_t)(first >= 0 ? first : len);
    *nt = (uint8_t)((found < kTrack ? found : kTrack) | (found <= kTrack ? kTrackFull : 0));
  }
  k1 = wave_min_u32(r0);
  k2 = wave_min_u32(r1);
}

// Minimum over the lanes of each 16-lane row, in the row's lane 15.
__device__ __forceinline__ uint32_t row_min_u32(uint32_t x) {
  MaxU32 op;
  x = ~x;
  x = op(x, dpp_u32<0x111, 0xf>(0u, x));
  x = op(x, dpp_u32<0x112, 0xf>(0u, x));
  x = op(x, dpp_u32<0x114, 0xf>(0u, x));
  x = op(x, dpp_u32<0x118, 0xf>(0u, x));
  return ~x;
}

// Book read of four lines by one wavefront, a 16-lane row each: as wave_book_track, 16
// entries per ballot.  line: the row's line (its row's lanes agree), active: whether the row
// has one.  k1/k2 are valid in the row's lane 15.
template <class TRK>
__device__ __forceinline__ void row_book_track(gcshort* book, gcint* data, int len, int16_t* pos, const uint8_t* crossCov,
                                               int lane, int b, bool active, TRK* out, uint8_t* nt, uint32_t& k1,
                                               uint32_t& k2) {
  const int shift = lane & ~15, sl = lane & 15;
  int at = *pos, found = 0, first = -1;
  wave_sync();  // every lane has the position before a row's first lane moves it
  uint32_t r0 = ~0u, r1 = ~0u;
  for (;;) {
    const bool on = active && at < len && found <= kTrack;
    if (__ballot(on) == 0) break;
    const int q = at + sl;
    const bool in = on && q < len;
    const int idx = in ? book[q] : 0;
    const int32_t cst = data[idx];
    const bool live = in && !crossCov[idx];
    const uint32_t mask = (uint32_t)(__ballot(live) >> shift) & 0xffffu;
    if (on && first < 0 && mask) first = at + __ffsll((unsigned long long)mask) - 1;
    if (live) {
      const int rank = found + __popcll((unsigned long long)(mask & ((1u << sl) - 1u)));
      const uint32_t key = ((uint32_t)cst << b) | (uint32_t)idx;
      if (rank < kTrack) out[rank] = key;
      if (rank == 0) r0 = key;
      if (rank == 1) r1 = key;
    }
    if (on) { found += __popcll((unsigned long long)mask); at += 16; }
  }
  if (active && sl == 0) {
    *pos = (int16_t)(first >= 0 ? first : len);
    *nt = (uint8_t)((found < kTrack ? found : kTrack) | (found <= kTrack ? kTrackFull : 0));
  }
  k1 = row_min_u32(r0);
  k2 = row_min_u32(r1);
}

// Vogel's LDS state (aliases the tree and aux regions): cover flags, residuals,
// penalties, the scan list, per-line tracked count/flag and book position; the tracked
// keys (kTrack per line, 16 bytes) follow in LDS when they fit, else they live in the
// instance's global scratch.
__host__ __device__ inline size_t vogel_trk_bytes(int m, int n) { return align16(16 * (size_t)(m + n)); }

// Vogel's line state in LDS (or global memory), carved from `base`.  kPen: the scan mode's
// penalties (the register mode's live in its ranks' registers).
struct VogelState {
  uint8_t *covR, *covC;  // cover flags
  int32_t* res;          // residual supplies, then demands
  int32_t* pen;
  int16_t* list;         // lines to scan
  uint8_t* nt;           // tracked count and full flag of a line
  int16_t* bpos;         // book read positions
};
template <bool kPen>
__device__ __forceinline__ VogelState vogel_state(const Ctx& C, char* base) {
  const int m = C.m, n = C.n, V = C.V;
  VogelState st;
  size_t off = 0;
  st.covR = (uint8_t*)(base + off); off += align16((size_t)((m + 3) & ~3));
  st.covC = (uint8_t*)(base + off); off += align16((size_t)((n + 3) & ~3));
  st.res = (int32_t*)(base + off); off += align16(4 * (size_t)V);
  st.pen = kPen ? (int32_t*)(base + off) : nullptr;
  if (kPen) off += align16(4 * (size_t)V);
  st.list = (int16_t*)(base + off); off += align16(2 * (size_t)V);
  st.nt = (uint8_t*)(base + off); off += align16((size_t)V);
  st.bpos = (int16_t*)(base + off);
  return st;
}

// First pass without books: the kTrack smallest keys of every line, one rank per line,
// read from the opposite-major copy (row L is column L of the transpose), so the lanes of
// a wavefront read consecutive addresses and each rank keeps its own top keys with no
// cross-lane reduction.  Every cell is uncovered at step 0.
template <int G, class TRK>
__device__ __forceinline__ void vogel_first_pass(const Ctx& C, TRK* trk, uint8_t* nt, int bRow, int bCol) {
  const int m = C.m, n = C.n, V = C.V, tid = grank<G>();
  constexpr int U = 16;  // loads in flight per rank
  for (int L = tid; L < V; L += G) {
    const bool row = L < m;
    gcint* lbase = row ? (gcint*)C.costT + L : C.cost + (L - m);
    const uint32_t stride = (uint32_t)(row ? C.ldT : C.ld);
    const int len = row ? n : m;
    const int b = row ? bRow : bCol;
    uint32_t l[kTrack] = {~0u, ~0u, ~0u, ~0u};
    for (int k0 = 0; k0 < len; k0 += U) {
      int32_t c[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int k = k0 + u < len ? k0 + u : len - 1;
        c[u] = lbase[(uint32_t)k * stride];
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int k = k0 + u;
        track_insert(k < len ? (((uint32_t)c[u] << b) | (uint32_t)k) : ~0u, l);  // ~0u inserts nothing
      }
    }
#pragma unroll
    for (int e = 0; e < kTrack; ++e) trk[4 * L + e] = l[e];
    nt[L] = (uint8_t)((len < kTrack ? len : kTrack) | (len <= kTrack ? kTrackFull : 0));
  }
}

// The first minimum uncovered cell of line Lc, by the whole group, as (cost, cross index);
// kNoKey when every cross line is covered.
template <int G>
__device__ __forceinline__ uint64_t vogel_search(const Ctx& C, int Lc, const VogelState& st, Shared& S, gcshort* books) {
  const int m = C.m, n = C.n, tid = grank<G>();
  const uint8_t* cross = Lc < m ? st.covC : st.covR;
  gcint* data = Lc < m ? C.cost + (uint32_t)(Lc * C.ld) : C.costT + (uint32_t)((Lc - m) * C.ldT);
  const int len = Lc < m ? n : m;
  uint64_t mk = kNoKey;
  if (books) {  // first uncovered book entry from the line's read position on
    gcshort* book = books + (Lc < m ? (size_t)Lc * n : (size_t)m * n + (size_t)(Lc - m) * m);
    for (int at = st.bpos[Lc]; at < len; at += G) {
      const int q = at + tid;
      uint64_t f = kNoKey;
      if (q < len) { const int j = book[q]; if (!cross[j]) f = (uint64_t)q; }
      f = group_min_u64<G>(f, S);
      if (f != kNoKey) { const int j = book[(int)f]; mk = pack_vi(data[j], (uint32_t)j); break; }
    }
  } else {
    for (int j = tid; j < len; j += G)
      if (!cross[j]) { const uint64_t k = pack_vi(data[j], (uint32_t)j); mk = k < mk ? k : mk; }
    mk = group_min_u64<G>(mk, S);
  }
  return mk;
}

// Scan mode: every step walks every line's state (instances with more lines than the
// register mode takes, and line state in global memory).
template <int G, class TRK>
__device__ __forceinline__ void vogel_scan(const Ctx& C, gcint* supply, gcint* demand, char* base, TRK* trk, Shared& S, gint* brow,
                          gint* bcol, gint* bflow, gcshort* books) {
  const int m = C.m, n = C.n, V = C.V, tid = grank<G>();
  const int lane = tid % kWave, wave = tid / kWave;
  constexpr int W = G / kWave;
  const VogelState st = vogel_state<true>(C, base);
  uint8_t *covR = st.covR, *covC = st.covC, *nt = st.nt;
  int32_t *res = st.res, *pen = st.pen;
  int16_t *list = st.list, *bpos = st.bpos;
  const int bRow = index_bits(n), bCol = index_bits(m);  // rows track column indices and vice versa

  for (int L = tid; L < V; L += G) {
    res[L] = L < m ? supply[L] : demand[L - m];
    pen[L] = 0;
    nt[L] = 0; bpos[L] = 0;  // with books nothing is tracked: every line is read at step 0
    if (L < m) covR[L] = 0; else covC[L - m] = 0;
  }
  if (!books) vogel_first_pass<G>(C, trk, nt, bRow, bCol);
  if (tid == 0) { S.pend_row = 1; S.pend_col = 1; S.cnt = 0; }
  int covCols = 0;  // columns covered so far (only rank 0 eliminates, so only its copy counts)
  gsync<G>();

  for (int step = 0; step < V - 1; ++step) {
    const bool pendR = S.pend_row != 0, pendC = S.pend_col != 0;
    uint64_t best = 0;
    {
      // kVB lines per rank at a time, every LDS load of a batch issued before first use
      constexpr int kVB = 4;
      for (int L0 = tid; L0 < V; L0 += kVB * G) {
        uint32_t key[kVB][4];
        uint8_t ntv[kVB], cov[kVB], fl[kVB][4];
        int32_t pv[kVB];
#pragma unroll
        for (int u = 0; u < kVB; ++u) {  // lines past V re-read this rank's first line L0
          const int L = L0 + u * G;
          const bool in = L < V;
          const int LL = in ? L : L0;
          ntv[u] = nt[LL];
          const u32x4 tk = *(const u32x4*)(trk + 4 * LL);
          key[u][0] = tk.x; key[u][1] = tk.y; key[u][2] = tk.z; key[u][3] = tk.w;
          const uint8_t cv = LL < m ? covR[LL] : covC[LL - m];
          cov[u] = in ? cv : 1;
          pv[u] = pen[LL];
        }
#pragma unroll
        for (int u = 0; u < kVB; ++u) {
          const int L = L0 + u * G;
          const bool row = L < m;
          const uint8_t* cross = row ? covC : covR;
          const uint32_t mask = (1u << (row ? bRow : bCol)) - 1u;
          const int cnt = ntv[u] & 0x7f;
#pragma unroll
          for (int e = 0; e < 4; ++e) fl[u][e] = cross[e < cnt ? (key[u][e] & mask) : 0];
        }
        // branch-free except the scan list append: the two smallest uncovered tracked
        // keys by selects, every in-range line's penalty rewritten
#pragma unroll
        for (int u = 0; u < kVB; ++u) {
          const int L = L0 + u * G;
          const bool row = L < m;
          const int b = row ? bRow : bCol;
          const uint32_t mask = (1u << b) - 1u;
          const int cnt = ntv[u] & 0x7f;
          bool unc[4];
#pragma unroll
          for (int e = 0; e < 4; ++e) unc[e] = (e < cnt) & (fl[u][e] == 0);
          const uint32_t* kk = key[u];
          const uint32_t k1 = unc[0] ? kk[0] : unc[1] ? kk[1] : unc[2] ? kk[2] : unc[3] ? kk[3] : ~0u;
          const uint32_t a3 = unc[3] ? kk[3] : ~0u;
          const uint32_t a2 = unc[2] ? kk[2] : a3;
          const uint32_t a1 = unc[1] ? kk[1] : a2;
          const uint32_t k2 = unc[0] ? a1 : unc[1] ? a2 : unc[2] ? a3 : ~0u;
          const bool refreshL = !cov[u] & (row ? pendR : pendC);
          const bool resolved = (k2 != ~0u) | ((ntv[u] & kTrackFull) != 0);
          const bool need = refreshL & !resolved;
          const int32_t p = refreshL ? (resolved ? key_penalty(k1, k2, b) : 0) : pv[u];
          if (L < V) pen[L] = p;
          if (need) list[atomicAdd(&S.cnt, 1)] = (int16_t)L;
          const bool jv = k1 != ~0u;
          const uint64_t k = ((uint64_t)(uint32_t)(p + 1) << 32) | ((uint64_t)(uint32_t)L << 18) |
                             (jv ? ((1u << 17) | (k1 & mask)) : 0u);
          best = (L < V && !need && k > best) ? k : best;
        }
      }
    }
    {
      best = group_max1_u64<G, 0>(best, S);
      // lines to scan (the count was published by the atomics before the max's barrier);
      // uniform: every rank reads the same count
      const int cnt = uniform(S.cnt);
      if (cnt == 0) goto decided;
      // one wavefront per listed line; each wavefront's max key of its lines is combined
      // with the max above through buffer 1 (idle outside pivots)
      uint64_t wbest = 0;
      for (int e = wave; e < cnt; e += W) {
        const int L = list[e];
        if (L < 0 || L >= V) continue;  // guard: list entries are lines
        const bool row = L < m;
        gcint* data = row ? C.cost + (uint32_t)(L * C.ld) : C.costT + (uint32_t)((L - m) * C.ldT);
        const int len = row ? n : m;
        const int b = row ? bRow : bCol;
        const uint8_t* cross = row ? covC : covR;
        uint32_t k1, k2;
        if (books)
          wave_book_track(books + (row ? (size_t)L * n : (size_t)m * n + (size_t)(L - m) * m), data, len, &bpos[L],
                          cross, lane, b, trk + 4 * L, &nt[L], k1, k2);
        else
          wave_line_track(data, len, cross, lane, b, trk + 4 * L, &nt[L], k1, k2);
        const int32_t p = key_penalty(k1, k2, b);
        if (lane == 0) pen[L] = p;
        const uint64_t k = ((uint64_t)(uint32_t)(p + 1) << 32) | ((uint64_t)(uint32_t)L << 18) |
                           (k1 != ~0u ? ((1u << 17) | (k1 & ((1u << b) - 1u))) : 0u);
        wbest = k > wbest ? k : wbest;
      }
      if (lane == 0) S.red1[1][wave] = wbest;
      gsync<G>();
#pragma unroll
      for (int w = 0; w < W; ++w) best = S.red1[1][w] > best ? S.red1[1][w] : best;
      if (tid == 0) S.cnt = 0;  // read above, before the barrier; next used after this step's last one
    }
  decided:
    const int Lc = (int)((best >> 18) & 0x3fffu);
    int jc;
    if ((best >> 17) & 1u) {
      jc = (int)(best & 0x1ffffu);  // the line's first uncovered tracked key: its first minimum
    } else {  // nothing uncovered is tracked: search the line itself
      const uint64_t mk = vogel_search<G>(C, Lc, st, S, books);
      if (mk == kNoKey) {  // no uncovered cross line: cannot happen for a balanced instance
        if (tid == 0) S.status = 4;
        gsync<G>();
        return;
      }
      jc = (int)key_idx(mk);
      // every rank has read the cover flags for the search before rank 0 changes them
      gsync<G>();
    }
    // rank 0 eliminates; nobody else reads the state it changes before the barrier
    if (tid == 0) {
      const int r = Lc < m ? Lc : jc, q = Lc < m ? jc : Lc - m;
      const int32_t rs = res[r], rd = res[m + q];
      bool coverRow = rd > rs;
      if (!coverRow && covCols == n - 1) coverRow = true;
      int32_t f;
      if (coverRow) {
        f = rs; res[m + q] = rd - rs; res[r] = 0; covR[r] = 1;
        pen[r] = -1;
      } else {
        f = rd; res[r] = rs - rd; res[m + q] = 0; covC[q] = 1;
        pen[m + q] = -1;
        ++covCols;
      }
      S.pend_row = coverRow ? 1 : 0;
      S.pend_col = coverRow ? 0 : 1;
      brow[step] = r; bcol[step] = q; bflow[step] = f;
    }
    gsync<G>();
  }
}

// Register mode: each rank keeps its (at most KL) lines' tracked keys, their cross lines
// and the lines' penalties in registers.  A step compares the line covered last with the
// tracked cross lines (packed 16-bit vertex numbers); a line that tracked it drops that
// key, so the first two keys left are always its smallest uncovered ones and no cover flag
// is read outside scans.  Its penalty is refreshed when its kind is pending (the stale
// rule) and, with fewer than two keys left of a longer line, the line is listed for a scan.
// Every rank follows the elimination itself from the two residuals, so a step has one
// barrier, the argmax's: rank 0 writes a step's residuals back in the next step, after
// that barrier, and meanwhile every rank takes those two from its registers; two buffers
// alternate under the argmax.
// Bound: the chain of a step (two wavefront minima, barrier, residuals) and its vector
// instructions, about 20 a line slot.  The former step (cover flags re-read for every
// touched line, rank 0 eliminating between two barriers, 320 vector instructions at four
// slots) took 2.0 us at 500x480 on 256 threads and 2.4 us at 1000x1000 on 512; this one
// takes 1.5 and 1.6 us, and 3.6 instead of 5.9 us at 4000x2000 on 1024.
constexpr int kRegLines = 4;       // lines per rank of the work-queue engines
constexpr int kRegLinesWide = 8;   // where m+n needs them, on 512 threads (and the set-up on 1024)
template <int G, class TRK, int KL>
__device__ __forceinline__ void vogel_reg(const Ctx& C, gcint* supply, gcint* demand, char* base, TRK* trk, Shared& S,
                                          gint* brow, gint* bcol, gint* bflow, gcshort* books) {
  const int m = C.m, n = C.n, V = C.V, tid = grank<G>();
  const int lane = tid % kWave, wave = tid / kWave;
  constexpr int W = G / kWave;
  const VogelState st = vogel_state<false>(C, base);
  const int bRow = index_bits(n), bCol = index_bits(m);  // rows track column indices and vice versa
  for (int L = tid; L < V; L += G) {
    st.res[L] = L < m ? supply[L] : demand[L - m];
    st.nt[L] = 0; st.bpos[L] = 0;  // with books nothing is tracked: every line is read at step 0
    if (L < m) st.covR[L] = 0; else st.covC[L - m] = 0;
  }
  if (!books) vogel_first_pass<G>(C, trk, st.nt, bRow, bCol);
  if (tid == 0) { S.cnt = 0; S.cnt2 = 0; }
  // per line L = tid + u*G: tracked keys (~0u: none), their cross vertices (0xffff: none),
  // penalty + 1 (0: covered, listed or past V), flags: dirty row / dirty column, all
  // uncovered cells tracked
  constexpr uint32_t fFull = 4;
  uint32_t l[KL][4], id01[KL], id23[KL], pen1[KL], fl[KL];
  auto penalty1 = [&](uint32_t k1, uint32_t k2, int b) { return (uint32_t)key_penalty(k1, k2, b) + 1u; };
  // a freshly tracked line (all keys uncovered, clean)
  auto load_line = [&](int u, int L) {
    const u32x4 tk = *(const u32x4*)(trk + 4 * L);
    const uint32_t ntl = st.nt[L];
    const int cnt = (int)(ntl & 0x7fu);
    const bool row = L < m;
    const int b = row ? bRow : bCol;
    const uint32_t mask = (1u << b) - 1u, base0 = row ? (uint32_t)m : 0u;  // first cross vertex
    l[u][0] = cnt > 0 ? tk.x : ~0u; l[u][1] = cnt > 1 ? tk.y : ~0u;
    l[u][2] = cnt > 2 ? tk.z : ~0u; l[u][3] = cnt > 3 ? tk.w : ~0u;
    uint32_t id[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) id[e] = e < cnt ? (l[u][e] & mask) + base0 : 0xffffu;
    id01[u] = id[0] | (id[1] << 16); id23[u] = id[2] | (id[3] << 16);
    fl[u] = (ntl & kTrackFull) ? fFull : 0u;
    pen1[u] = penalty1(l[u][0], l[u][1], b);
  };
#pragma unroll
  for (int u = 0; u < KL; ++u) {
    const int L = tid + u * G;
    l[u][0] = l[u][1] = l[u][2] = l[u][3] = ~0u;
    id01[u] = id23[u] = ~0u;
    pen1[u] = 0;
    fl[u] = L >= V ? 0u : L < m ? 1u : 2u;
    if (!books && L < V) load_line(u, L);
  }
  // the line covered last, the pending kinds (1 rows, 2 columns) and the last step's cell
  // with its new residuals: the same in every rank
  int X = 0xfffe, pr = -1, pq = -1, covCols = 0;
  uint32_t pend = 3;
  int32_t prs = 0, prd = 0;
  gsync<G>();

  for (int step = 0; step < V - 1; ++step) {
    // the rank index, opaque to the compiler here, so line numbers are recomputed each step
    // instead of being kept (spilled) across the whole loop
    int tidr = tid;
    asm volatile("" : "+v"(tidr));
    const int wave0 = uniform(tid & ~(kWave - 1));  // this wavefront's first rank
    const uint32_t xx = (uint32_t)X | ((uint32_t)X << 16);
    // a rank may list lines of the next step before another has read this step's count
    int32_t* listed = step & 1 ? &S.cnt2 : &S.cnt;
    uint32_t bpen = 0, bkey = ~0u;
    int bL = tidr;
#pragma unroll
    for (int u = 0; u < KL; ++u) {
      if (wave0 + u * G >= V) continue;  // uniform: the wavefront has no line in slot u
      const int L = tidr + u * G;
      const uint32_t d01 = id01[u] ^ xx, d23 = id23[u] ^ xx;
      const uint32_t d = min_u16x2(d01, d23);
      const bool hit = ((d - 0x00010001u) & ~d & 0x80008000u) != 0;  // a zero half: X is tracked
      if (hit | (L == X) | ((fl[u] & pend) != 0)) {  // few lines per step
        if (L == X) {
          pen1[u] = 0; id01[u] = id23[u] = ~0u; fl[u] = 0;
        } else {
          const bool row = L < m;
          if (hit) {  // drop that key
            const bool h0 = (d01 & 0xffffu) == 0, h1 = h0 | (d01 < 0x10000u), h2 = h1 | ((d23 & 0xffffu) == 0);
            l[u][0] = h0 ? l[u][1] : l[u][0];
            l[u][1] = h1 ? l[u][2] : l[u][1];
            l[u][2] = h2 ? l[u][3] : l[u][2];
            l[u][3] = ~0u;
            const uint32_t i1 = id01[u] >> 16, i2 = id23[u] & 0xffffu, i3 = id23[u] >> 16;
            const uint32_t j0 = h0 ? i1 : (id01[u] & 0xffffu);
            id01[u] = j0 | ((h1 ? i2 : i1) << 16);
            id23[u] = (h2 ? i3 : i2) | 0xffff0000u;
            fl[u] |= row ? 1u : 2u;
          }
          if (fl[u] & pend) {
            if ((l[u][1] != ~0u) | ((fl[u] & fFull) != 0)) {
              pen1[u] = penalty1(l[u][0], l[u][1], row ? bRow : bCol);
            } else {
              pen1[u] = 0;
              st.list[atomicAdd(listed, 1)] = (int16_t)L;
              fl[u] |= 8u;  // listed
            }
            fl[u] &= ~3u;
          }
        }
      }
      const bool better = pen1[u] >= bpen;  // the last maximum
      bpen = better ? pen1[u] : bpen;
      bkey = better ? l[u][0] : bkey;
      bL = better ? L : bL;
    }
    auto argmax_key = [&](uint32_t p1, int L, uint32_t k1) {
      const uint32_t mask = (1u << (L < m ? bRow : bCol)) - 1u;
      return ((uint64_t)p1 << 32) | ((uint64_t)(uint32_t)L << 18) | (k1 != ~0u ? ((1u << 17) | (k1 & mask)) : 0u);
    };
    uint64_t best = group_max_alt<G>(argmax_key(bpen, bL, bkey), S, step & 1);
    // lines to scan (the count was published by the atomics before the max's barrier);
    // uniform: every rank reads the same count
    const int cnt = uniform(*listed);
    if (cnt != 0) {
      // one wavefront per listed line; each wavefront's max key of its lines is combined
      // with the max above through buffer 1 (idle outside pivots)
      uint64_t wbest = 0;
      if (books && cnt > W) {
        // more lines than wavefronts: four at a time (equal costs let one covered column
        // list hundreds of rows; 4000x2000 with costs 1..8 scans 55 lines a step)
        for (int e0 = 4 * wave; e0 < cnt; e0 += 4 * W) {
          const int e = e0 + (lane >> 4);
          const bool active = e < cnt;
          const int L = st.list[active ? e : e0];
          const bool row = L < m;
          const int b = row ? bRow : bCol;
          uint32_t k1, k2;
          row_book_track(books + (row ? (size_t)L * n : (size_t)m * n + (size_t)(L - m) * m),
                         row ? C.cost + (uint32_t)(L * C.ld) : (gcint*)(C.costT + (uint32_t)((L - m) * C.ldT)),
                         row ? n : m, &st.bpos[L], row ? st.covC : st.covR, lane, b, active, trk + 4 * L, &st.nt[L],
                         k1, k2);
          const uint64_t k = argmax_key(penalty1(k1, k2, b), L, k1);
          if (active && (lane & 15) == 15) wbest = k > wbest ? k : wbest;
        }
        wbest = wave_max_u64(wbest);
      } else
      for (int e = wave; e < cnt; e += W) {
        const int L = st.list[e];
        if (L < 0 || L >= V) continue;  // guard: list entries are lines
        const bool row = L < m;
        gcint* data = row ? C.cost + (uint32_t)(L * C.ld) : C.costT + (uint32_t)((L - m) * C.ldT);
        const int len = row ? n : m;
        const int b = row ? bRow : bCol;
        const uint8_t* cross = row ? st.covC : st.covR;
        uint32_t k1, k2;
        if (books)
          wave_book_track(books + (row ? (size_t)L * n : (size_t)m * n + (size_t)(L - m) * m), data, len, &st.bpos[L],
                          cross, lane, b, trk + 4 * L, &st.nt[L], k1, k2);
        else
          wave_line_track(data, len, cross, lane, b, trk + 4 * L, &st.nt[L], k1, k2);
        const uint64_t k = argmax_key(penalty1(k1, k2, b), L, k1);
        wbest = k > wbest ? k : wbest;
      }
      if (lane == 0) S.red1[1][wave] = wbest;
      gsync<G>();
#pragma unroll
      for (int w = 0; w < W; ++w) best = S.red1[1][w] > best ? S.red1[1][w] : best;
      if (tid == 0) *listed = 0;  // read by every rank before the barrier
      int tids = tid;  // opaque, as above
      asm volatile("" : "+v"(tids));
#pragma unroll
      for (int u = 0; u < KL; ++u)
        if (fl[u] & 8u) load_line(u, tids + u * G);
      // no barrier closes the scan: the list, the tracked keys and buffer 1 are written
      // again only after the next step's argmax barrier, this count two steps on
    }
    const int Lc = (int)((best >> 18) & 0x3fffu);
    int jc;
    if ((best >> 17) & 1u) {
      jc = (int)(best & 0x1ffffu);  // the line's first uncovered tracked key: its first minimum
    } else {  // nothing uncovered is tracked: search the line itself
      const uint64_t mk = vogel_search<G>(C, Lc, st, S, books);
      if (mk == kNoKey) {  // no uncovered cross line: cannot happen for a balanced instance
        if (tid == 0) S.status = 4;
        gsync<G>();
        return;
      }
      jc = (int)key_idx(mk);
      // every rank has read the cover flags for the search before rank 0 changes them
      gsync<G>();
    }
    const int r = Lc < m ? Lc : jc, q = Lc < m ? jc : Lc - m;
    const int32_t lr = lds_load(&st.res[r]), lq = lds_load(&st.res[m + q]);
    const int32_t rs = r == pr ? prs : lr, rd = q == pq ? prd : lq;
    bool coverRow = rd > rs;
    coverRow = coverRow | (covCols == n - 1);
    if (tid == 0) {
      if (pr >= 0) { lds_store(&st.res[pr], prs); lds_store(&st.res[m + pq], prd); }
      if (coverRow) st.covR[r] = 1; else st.covC[q] = 1;  // next read by a scan, after a barrier
      brow[step] = r; bcol[step] = q; bflow[step] = coverRow ? rs : rd;
    }
    pr = r; pq = q;
    prs = coverRow ? 0 : rs - rd;
    prd = coverRow ? rd - rs : 0;
    X = coverRow ? r : m + q;
    pend = coverRow ? 1u : 2u;
    covCols += coverRow ? 0 : 1;
  }
}

// books: sorted lines (large instances) or null (scan lines).  scratch: the instance's
// global scratch (at least vogel_trk_bytes), used for the tracked keys when they do not
// fit in LDS after the rest of the state (`avail` bytes at `base`).
// gstate: global memory of at least vogel_lds_bytes for the line state when even that
// does not fit the `avail` LDS bytes at `base` (large-instance path with the tree in
// global memory); null otherwise.
// kWide: also instantiate the register mode with kRegLinesWide lines per rank, with the
// tracked keys in LDS or in global scratch.
template <int G, bool kWide = false>
__device__ __forceinline__ void vogel(const Ctx& C, gcint* supply, gcint* demand, char* base, size_t avail, Shared& S, gint* brow,
                      gint* bcol, gint* bflow, int32_t* scratch, gcshort* books = nullptr, char* gstate = nullptr) {
  const size_t need = vogel_lds_bytes(C.m, C.n);
  const size_t needR = vogel_reg_lds_bytes(C.m, C.n);
  const size_t trkBytes = vogel_trk_bytes(C.m, C.n);
  typedef FLOCK_LDS uint32_t LdsTrk;
  typedef FLOCK_GLOBAL uint32_t GlTrk;
  const bool regLines = C.V <= kRegLines * G;
  const bool regWide = kWide && C.V <= kRegLinesWide * G;
  if ((regLines || regWide) && needR + trkBytes <= avail) {  // register mode, tracked keys in LDS
    LdsTrk* trk = (LdsTrk*)(base + needR);
    if (regLines) {
      vogel_reg<G, LdsTrk, kRegLines>(C, supply, demand, base, trk, S, brow, bcol, bflow, books);
    } else {
      if constexpr (kWide) vogel_reg<G, LdsTrk, kRegLinesWide>(C, supply, demand, base, trk, S, brow, bcol, bflow, books);
    }
  } else if (!regLines && !regWide && need + trkBytes <= avail) {  // scan mode, tracked keys in LDS
    vogel_scan<G, LdsTrk>(C, supply, demand, base, (LdsTrk*)(base + need), S, brow, bcol, bflow, books);
  } else if (need <= avail) {
    GlTrk* trk = (GlTrk*)scratch;
    if (regWide) {
      if constexpr (kWide) vogel_reg<G, GlTrk, kRegLinesWide>(C, supply, demand, base, trk, S, brow, bcol, bflow, books);
    } else {
      vogel_scan<G, GlTrk>(C, supply, demand, base, trk, S, brow, bcol, bflow, books);
    }
  } else if (gstate) {
    vogel_scan<G, GlTrk>(C, supply, demand, gstate, (GlTrk*)scratch, S, brow, bcol, bflow, books);
  } else {  // the host sizes LDS so that this cannot happen; report instead of overrunning it
    if (grank<G>() == 0) S.status = 6;
    gsync<G>();
  }
}

// North-west corner rule (IBFS_nwc.cu:3-34; a tie moves to the next row, :17-23, except
// on the last row).  Sequential, m+n-1 steps.
template <int G>
__device__ __forceinline__ void nwc(const Ctx& C, gcint* supply, gcint* demand, gint* brow, gint* bcol, gint* bflow) {
  if (grank<G>() != 0) return;
  int i = 0, j = 0;
  int64_t rs = supply[0], rd = demand[0];
  for (int k = 0; k < C.V - 1; ++k) {
    brow[k] = i; bcol[k] = j;
    if ((rd >= rs && i < C.m - 1) || j == C.n - 1) {
      bflow[k] = (int32_t)rs; rd -= rs; ++i; rs = i < C.m ? supply[i] : 0;
    } else {
      bflow[k] = (int32_t)rd; rs -= rd; ++j; rd = j < C.n ? demand[j] : 0;
    }
  }
}

__device__ __forceinline__ int32_t dual_of(const TreeLds& t, int m, int x) { return x < m ? t.du[x] : t.dv[x - m]; }
__device__ __forceinline__ void set_dual(const TreeLds& t, int m, int x, int32_t v) {
  if (x < m) t.du[x] = v; else t.dv[x - m] = v;
}

// ---------------------------------------------------------------------------
// Basis tree from the m+n-1 basic cells, rooted at vertex 0: level by level, every cell
// not used yet whose one end has the level's depth hangs its other end below it (parent,
// depth, slot and dual, x_child = c(row,col) - x_parent, DUAL_solver.cu:52-62; the
// reference's CSR, parallel_kernels.cu:205-319, is not needed for that).  Then subtree
// sizes bottom-up and preorder numbers top-down, again level by level, over the level's own
// vertices (the first pass lists them): a vertex takes its interval from its parent's next
// free position (siblings in any order: preorder numbers only serve ancestor tests).
// Returns false if the cells do not form a spanning tree: of V - 1 cells that leave no
// vertex unreached none closes a cycle.
// Bound: three passes of one barrier and a few LDS round trips per level, and the first
// pass's look at every cell.  Levels are few in Vogel's trees (94 at 505x475), about 0.66 V
// in a square north-west corner one.  The cells' ends and costs are read from global memory
// once.  A BFS over a CSR, reading its cells from global memory level by level with two
// barriers each, took 146 us at 490x490 and 24.2 ms at 4500x4500 north-west corner (tree in
// global memory); size and preorder passes over every vertex 39 us and 32.0 ms; this 34 us
// and 19.0 ms (1000x1000 north-west corner: 3.4, 1.9 and 1.3 ms).
// scr: aux_ints.
// ---------------------------------------------------------------------------
template <int G>
__device__ __forceinline__ bool build_tree(const Ctx& C, gcint* brow, gcint* bcol, gcint* bflow, const TreeLds& t, int32_t* scr,
                           Shared& S) {
  const int m = C.m, V = C.V, tid = grank<G>();
  int32_t* arc = scr;        // V-1: row << 16 | column vertex (-1: used)
  int32_t* acost = arc + V;  // V-1
  int32_t* dep = acost + V;  // V: depth, -1 unreached
  int32_t* size = dep + V;   // V
  int32_t* next = size + V;  // V: next free preorder position below the vertex
  int16_t* order = (int16_t*)(next + V);  // V: the vertices but the root, level by level
  int16_t* start = order + 2 * (V / 2 + 1);  // V+1: where depth d's vertices start in it, d = 1 ..
  int badCell = 0;
  for (int k = tid; k < V - 1; k += G) {
    const int r = brow[k], c = bcol[k];
    const bool bad = r < 0 || r >= m || c < 0 || c >= C.n;  // guard
    badCell |= bad ? 1 : 0;
    arc[k] = bad ? -1 : (int32_t)(((uint32_t)r << 16) | (uint32_t)(m + c));
    acost[k] = bad ? 0 : cost_at(C, r, c);
  }
  for (int x = tid; x < V; x += G) { dep[x] = x == 0 ? 0 : -1; size[x] = 1; }
  if (badCell) atomicAdd(&S.status, 1);
  if (tid == 0) {
    t.parent[0] = -1; t.slot[0] = -1; t.flow[0] = 0; set_dual(t, m, 0, 0);
    S.level[0] = S.level[1] = S.level[2] = 0;
  }
  gsync<G>();
  if (S.status != 0) return false;
  constexpr int U = 4;  // cells a rank looks at together
  int d = 0, placed = 0;  // vertices placed so far, the same in every rank
  for (;; ++d) {
    // how many vertices this level reaches; the counter of the next level is cleared here:
    // it was last read two barriers ago
    int32_t* grown = &S.level[d % 3];
    if (tid == 0) { S.level[(d + 1) % 3] = 0; start[d + 1] = (int16_t)placed; }
    for (int k0 = tid; k0 < V - 1; k0 += U * G) {
      int32_t a[U], dr[U], dc[U];
#pragma unroll
      for (int u = 0; u < U; ++u) a[u] = k0 + u * G < V - 1 ? arc[k0 + u * G] : -1;
#pragma unroll
      for (int u = 0; u < U; ++u) {
        dr[u] = lds_load(&dep[a[u] < 0 ? 0 : a[u] >> 16]);
        dc[u] = lds_load(&dep[a[u] < 0 ? 0 : a[u] & 0xffff]);
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const bool down = dr[u] == d && dc[u] < 0, up = dc[u] == d && dr[u] < 0;
        if (a[u] >= 0 && (down | up)) {
          const int k = k0 + u * G, r = a[u] >> 16, c = a[u] & 0xffff;
          const int x = down ? r : c, y = down ? c : r;  // y hangs below x
          t.parent[y] = (int16_t)x; t.slot[y] = (int16_t)k;
          set_dual(t, m, y, acost[k] - dual_of(t, m, x));
          lds_store(&dep[y], d + 1);
          arc[k] = -1;
          order[placed + atomicAdd(grown, 1)] = (int16_t)y;  // (a cell once: at most V - 1)
        }
      }
    }
    gsync<G>();
    const int reached = uniform(lds_load(grown));  // written before the barrier
    if (reached == 0) break;
    placed += reached;
  }
  // depths 1 .. d are in use, and start[1 .. d + 1] set
  bool all = true;
  for (int x = tid; x < V; x += G) all = all & (dep[x] >= 0);
  if (!all) atomicAdd(&S.status, 1);
  gsync<G>();
  if (S.status != 0) {  // (the caller reports the forest; the status is its own)
    gsync<G>();
    if (tid == 0) S.status = 0;
    gsync<G>();
    return false;
  }
  for (int x = tid; x < V; x += G)
    if (x > 0) t.flow[x] = bflow[t.slot[x]];
  int at = d > 0 ? start[d] : 0, end = placed;
  for (int dd = d; dd >= 1; --dd) {  // subtree sizes, deepest level first
    const int before = dd > 1 ? start[dd - 1] : 0;
    for (int q = at + tid; q < end; q += G) {
      const int x = order[q];
      atomicAdd(&size[t.parent[x]], size[x]);
    }
    end = at; at = before;
    gsync<G>();
  }
  if (tid == 0) { t.pre(0) = 0; next[0] = 1; }
  gsync<G>();
  at = 0; end = d > 1 ? start[2] : placed;
  for (int dd = 1; dd <= d; ++dd) {
    const int after = dd + 1 < d ? start[dd + 2] : placed;
    for (int q = at + tid; q < end; q += G) {
      const int x = order[q];
      const int p = atomicAdd(&next[t.parent[x]], size[x]);
      t.pre(x) = (int16_t)p;
      next[x] = p + 1;
    }
    at = end; end = after;
    gsync<G>();
  }
  for (int x = tid; x < V; x += G) { t.size(x) = (int16_t)size[x]; t.depth[x] = (int16_t)dep[x]; }
  gsync<G>();
  return true;
}

// ---------------------------------------------------------------------------
// Reduced-cost sweep fused with the argmin (computeReducedCosts + thrust::min_element,
// parallel_kernels.cu:329-353 and uv_model_parallel.cu:169; host scan :184-194):
// r_ij = c_ij - u_i - v_j over all cells, minimum r, ties -> lowest row-major index.
// The padded matrix is walked in blocks of kSlots * G 16-byte vectors that are whole rows:
// slot s of rank t holds position p = t + s*G of the block, i.e. column vector p % w and
// row p / w of the block's h = kSlots*G / w rows (w vectors per row), and the next block
// is h rows further down.  A slot's columns never change, so their four duals stay in
// registers and its next address is one uniform step away: per vector one LDS read (u),
// the four subtractions and the running minimum remain, 11 vector-ALU instructions.
// (Vectors dealt to ranks by flat index took 23: a 40-bit multiply for the row, both
// addresses and an LDS read of the four duals each time.)  The load of a slot's next
// vector is issued as soon as its present one is consumed, so kSlots loads stay in flight
// across blocks.  Positions past the block or the matrix repeat the last one.
// A strict `<` keeps each slot's first minimum (rows only grow), so the least
// (r, row, column) key over the slots is the rank's, and the group min over ranks finishes
// the argmin.  With K = kSlots each slot's best cell is also a pricing candidate; with
// K = 1 (one pivot per sweep) the rank's single best cell is, and only its vector is read
// again to find the column inside it.
// Bound: one compute unit's cache bandwidth (about 64 bytes a clock, 150 GB/s) for large
// matrices, load latency and the closing minimum for small ones.  A sweep of 500x480 at
// 512 threads went from 15.1 to 8.2 us (64 -> 117 GB/s), one of 100x100 at 256 threads from
// 3.0 to 1.8 us; the 4096-instance batch from 10.2 to 9.43 ms (candidates) and from 58 to
// 38 ms (Dantzig).
// ---------------------------------------------------------------------------
// 16-byte loads in flight per rank: 8 for workgroup groups, 4 for wavefront groups
template <int G>
struct SweepSlots { static constexpr int value = G == kWave ? 4 : 8; };
// candidates per rank: 8 for workgroup groups (2048 at 256 threads, 8192 at 1024; more
// candidates measured fewer sweeps and pivots at every group size: at 1024 threads an
// 1800x1800 instance needs 1645 sweeps instead of 7692 with one per rank), 4 for
// wavefront groups
template <int G>
struct CandsPerRank { static constexpr int value = G == kWave ? 4 : 8; };

// Cell (row, col) as one word whose order is row-major order (m+n <= 16383); the halves are
// the byte offsets of the row's and the column's dual.
__device__ __forceinline__ uint32_t cell_id(uint32_t row, uint32_t col) { return (row << 18) | (col << 2); }
__device__ __forceinline__ int cell_row(uint64_t key) { return (int)((uint32_t)key >> 18); }
__device__ __forceinline__ int cell_col(uint64_t key) { return (int)(((uint32_t)key & 0xffffu) >> 2); }

struct Cand {
  int32_t row, col, cost;
};
// K candidate cells of one rank: cell id and cost (an empty slot is cell 0 at the padding
// cost, which never prices negative: u_0 = 0 and every dual is below 2^30)
template <int K>
struct CandSet {
  uint32_t id[K];
  int32_t cost[K];
  __device__ __forceinline__ void clear() {
#pragma unroll
    for (int k = 0; k < K; ++k) { id[k] = 0; cost[k] = kPadCost; }
  }
  __device__ __forceinline__ Cand get(int k) const {
    Cand c;
    c.row = cell_row(id[k]);
    c.col = cell_col(id[k]);
    c.cost = cost[k];
    return c;
  }
  __device__ __forceinline__ void set(int k, const Cand& c) {
    id[k] = cell_id((uint32_t)c.row, (uint32_t)c.col);
    cost[k] = c.cost;
  }
};

// Shape of a sweep over w column vectors: a block is h rows, the matrix `full` whole
// blocks and `rest` rows.  p / w is the high word of p * magic, exact while p * w < 2^32
// (both are at most kSlots * G <= 8192).
struct SweepShape {
  uint32_t w, magic, h, full, rest;
  __device__ __forceinline__ uint32_t div(uint32_t p) const {
    return w > 1 ? (uint32_t)(((uint64_t)p * magic) >> 32) : p;
  }
};
// w: at most a block, kSlots * G vectors
template <int G>
__device__ __forceinline__ SweepShape sweep_shape(int m, int w) {
  SweepShape s;
  s.w = (uint32_t)w;
  s.magic = w > 1 ? 0xffffffffu / (uint32_t)w + 1 : 0;
  s.h = s.div((uint32_t)(SweepSlots<G>::value * G));
  s.full = (uint32_t)m / s.h;
  s.rest = (uint32_t)m - s.full * s.h;
  return s;
}
// whether a row can be longer than one block (wavefront groups with n > 1024 only: a
// workgroup's block is at least 8192 columns, more than m+n of any instance in LDS)
template <int G>
struct SweepChunks { static constexpr bool value = SweepSlots<G>::value * G * 4 < 8000; };

// shape: sweep_shape<G> of the whole row (used unless SweepChunks)
template <int G, int K>
__device__ __forceinline__ uint64_t sweep_argmin(const Ctx& C, const TreeLds& t, Shared& S, const SweepShape& shape, CandSet<K>& mine) {
  constexpr int kSlots = SweepSlots<G>::value;
  static_assert(K == 1 || K == kSlots, "one candidate per rank or one per slot");
  constexpr bool kChunks = SweepChunks<G>::value;
  // the rank index, opaque to the compiler here: the slots' positions depend on nothing
  // else, and kept across the pivots between two sweeps they would spill
  int tidr = grank<G>();
  asm volatile("" : "+v"(tidr));
  const uint32_t tid = (uint32_t)tidr;
  const uint32_t m = (uint32_t)C.m, ld = (uint32_t)C.ld;
  const uint32_t vpr = ld >> 2;
  typedef const FLOCK_GLOBAL char gcbyte;
  int32_t bestR[kSlots];
  uint32_t bestRow[kSlots], col[kSlots];
#pragma unroll
  for (int s = 0; s < kSlots; ++s) { bestR[s] = kBig; bestRow[s] = 0; col[s] = 0; }
  uint32_t c0 = 0;
  do {
    const SweepShape sh =
        kChunks ? sweep_shape<G>((int)m, (int)(vpr - c0 < (uint32_t)(kSlots * G) ? vpr - c0 : (uint32_t)(kSlots * G)))
                : shape;
    const uint32_t rowBytes = 4 * ld, blockBytes = sh.h * rowBytes;
    // row and column of a slot's position in a block
    auto place = [&](uint32_t rank, int s, uint32_t* row, uint32_t* cc) {
      uint32_t p = rank + (uint32_t)(s * G);
      p = p < sh.h * sh.w ? p : sh.h * sh.w - 1;
      *row = sh.div(p);
      *cc = 4 * (c0 + p - *row * sh.w);
    };
    uint32_t row[kSlots], off[kSlots];  // off: byte offset of the slot's vector in the block at hand
    i32x4 dv[kSlots], cv[kSlots];
#pragma unroll
    for (int s = 0; s < kSlots; ++s) {
      uint32_t cc;
      place(tid, s, &row[s], &cc);
      off[s] = row[s] * rowBytes + 4 * cc;
      const uint32_t back = row[s] < m ? 0 : row[s] - (m - 1);  // rows past the matrix repeat the last
      cv[s] = *(const FLOCK_GLOBAL i32x4*)((gcbyte*)C.cost + (off[s] - back * rowBytes));
      dv[s] = *(const i32x4*)(t.dv + cc);
    }
    auto take = [&](int s, uint32_t r, const i32x4& c) {
      const int32_t u = t.du[r];
      const int32_t mn = imin(imin(c.x - dv[s].x, c.y - dv[s].y), imin(c.z - dv[s].z, c.w - dv[s].w)) - u;
      bool better = mn < bestR[s];
      if constexpr (kChunks) {
        uint32_t rr, cc;
        place(tid, s, &rr, &cc);
        better = better | ((mn == bestR[s]) & (cell_id(r, cc) < cell_id(bestRow[s], col[s])));
        col[s] = better ? cc : col[s];
      }
      bestR[s] = better ? mn : bestR[s];
      bestRow[s] = better ? r : bestRow[s];
    };
    const uint32_t blocks = sh.full + (sh.rest ? 1u : 0u);
    uint32_t b = 0;
    gcbyte* next = (gcbyte*)C.cost + blockBytes;
    for (; b + 1 < sh.full; ++b) {  // this block and the next are whole
#pragma unroll
      for (int s = 0; s < kSlots; ++s) {
        take(s, b * sh.h + row[s], cv[s]);
        cv[s] = *(const FLOCK_GLOBAL i32x4*)(next + off[s]);
        sched_fence();  // keep one vector per slot in registers, not two
      }
      next += blockBytes;
    }
    if (b + 1 < blocks) {  // the last whole block, then the partial one
      const uint32_t left = m - (b + 1) * sh.h;  // rows of the partial block
#pragma unroll
      for (int s = 0; s < kSlots; ++s) {
        take(s, b * sh.h + row[s], cv[s]);
        const uint32_t back = row[s] < left ? 0 : row[s] - (left - 1);
        cv[s] = *(const FLOCK_GLOBAL i32x4*)(next + (off[s] - back * rowBytes));
        sched_fence();
      }
      ++b;
    }
#pragma unroll
    for (int s = 0; s < kSlots; ++s) {
      const uint32_t r = b * sh.h + row[s];
      take(s, r < m ? r : m - 1, cv[s]);
    }
    if constexpr (!kChunks) {
      // the slots' columns, computed again rather than kept through the loop
      int tide = grank<G>();
      asm volatile("" : "+v"(tide));
#pragma unroll
      for (int s = 0; s < kSlots; ++s) {
        uint32_t rr;
        place((uint32_t)tide, s, &rr, &col[s]);
      }
    }
    c0 += (uint32_t)(kSlots * G);
  } while (kChunks && c0 < vpr);
  // A real cell's c - v is at most V * max cost < 2^30, so a padding cell (cost 2^30,
  // dual 0) is never its vector's minimum.
  uint64_t key = kNoKey;
  if constexpr (K == 1) {
    // the rank's least (r, row, first column of the vector), then the vector's first cell
    // at the minimum: the vectors are disjoint and ordered, so this is row-major order
    int32_t r = kBig;
    uint32_t id = ~0u;
#pragma unroll
    for (int s = 0; s < kSlots; ++s) {
      const uint32_t is = cell_id(bestRow[s], col[s]);
      const bool better = (bestR[s] < r) | ((bestR[s] == r) & (is < id));
      r = better ? bestR[s] : r;
      id = better ? is : id;
    }
    const uint32_t br = (uint32_t)cell_row(id), bc = (uint32_t)cell_col(id);
    const i32x4 c = *(const FLOCK_GLOBAL i32x4*)((gcbyte*)C.cost + 4 * (br * ld + bc));
    const int32_t u = t.du[br];
    const i32x4 vv = *(const i32x4*)(t.dv + bc);
    const int e = c.x - vv.x - u == r ? 0 : c.y - vv.y - u == r ? 1 : c.z - vv.z - u == r ? 2 : 3;
    mine.id[0] = id + 4 * (uint32_t)e;
    mine.cost[0] = e == 0 ? c.x : e == 1 ? c.y : e == 2 ? c.z : c.w;
    key = pack_vi(r, id + 4 * (uint32_t)e);
  } else {
    // each slot's first cell at its minimum (its vector reloaded; the K loads together)
    i32x4 cv[K];
#pragma unroll
    for (int k = 0; k < K; ++k) cv[k] = *(const FLOCK_GLOBAL i32x4*)((gcbyte*)C.cost + 4 * (bestRow[k] * ld + col[k]));
#pragma unroll
    for (int k = 0; k < K; ++k) {
      const int32_t u = t.du[bestRow[k]];
      const i32x4 vv = *(const i32x4*)(t.dv + col[k]);
      const i32x4 c = cv[k];
      const int e = c.x - vv.x - u == bestR[k] ? 0 : c.y - vv.y - u == bestR[k] ? 1 : c.z - vv.z - u == bestR[k] ? 2 : 3;
      const uint32_t id = cell_id(bestRow[k], col[k] + (uint32_t)e);
      mine.id[k] = id;
      mine.cost[k] = e == 0 ? c.x : e == 1 ? c.y : e == 2 ? c.z : c.w;
      const uint64_t kk = pack_vi(bestR[k], id);
      key = kk < key ? kk : key;
    }
  }
  return group_min1_u64<G, 2>(key, S);
}

// Re-price a rank's candidates with the current duals (costs kept in registers): the key of
// the least reduced cost (of equal ones the rank's first).
template <int K>
__device__ __forceinline__ uint64_t reprice_set(const TreeLds& t, const CandSet<K>& cs) {
  int32_t best = kBig;
  uint32_t id = 0;
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const int32_t u = *(const int32_t*)((const char*)t.du + (cs.id[k] >> 16));
    const int32_t v = *(const int32_t*)((const char*)t.dv + (cs.id[k] & 0xffffu));
    const int32_t r = cs.cost[k] - u - v;
    const bool better = r < best;
    best = better ? r : best;
    id = better ? cs.id[k] : id;
  }
  return pack_vi(best, id);
}

// Re-price a candidate with the current duals (cost kept in a register).
__device__ __forceinline__ uint64_t reprice(const Ctx& C, const TreeLds& t, const Cand& c) {
  if (c.row < 0) return kNoKey;
  const int32_t r = c.cost - t.du[c.row] - t.dv[c.col];
  return pack_vi(r, cell_id((uint32_t)c.row, (uint32_t)c.col));
}

// ---------------------------------------------------------------------------
// One tile of a full sweep (the large-instance path's sweep grid): vectors [tile*vpt,
// (tile+1)*vpt) of the padded matrix against the duals of the saved tree (global memory).
// Writes the tile's argmin key (r, cell) to keys[tile] and, per 16-lane row of its
// wavefronts, the best cell (row, col, cost) to cands (row -1: none).
// Everything comes from kernel arguments, so a rank issues its cost vectors, their row
// duals, their column duals (one aligned vector: the saved tree pads them like the rows)
// and the phase word together (one round trip); as in sweep_argmin, a vector is compared
// by its least reduced cost and the winning cell is recovered once at the end.  When the
// phase word is not 1 (instance done) nothing is written.
// ---------------------------------------------------------------------------
// candidates a 256-thread sweep tile writes: one per 16-lane row of each wavefront
constexpr int kTileCands = 16;
struct MinU64Row { __device__ __forceinline__ uint64_t operator()(uint64_t a, uint64_t b) const { return b < a ? b : a; } };
struct SweepArgs {
  const int32_t* cost;   // m x ld, padded rows
  const int32_t* du;     // the saved tree's duals
  const int32_t* dv;     // 16-byte aligned, padded to ld with zeros
  const int32_t* phase;  // instance phase word
  uint64_t* keys;
  int32_t* cands;
  int32_t m, n, ld;
  uint32_t vpt;
};

template <int G>
__device__ __forceinline__ void sweep_tile(const SweepArgs& A, uint32_t tile, Shared& S) {
  const int tid = grank<G>(), lane = tid % kWave, wave = tid / kWave;
  static_assert(G / kWave * 4 == kTileCands, "a tile's candidates: four rows per wavefront");
  constexpr int U = 4;  // vectors in flight per rank
  gcint* cost = gl(A.cost);
  gcint* du = gl(A.du);
  gcint* dv = gl(A.dv);
  const int m = A.m;
  const uint32_t vpr = (uint32_t)A.ld >> 2;
  const uint32_t nvec = (uint32_t)m * vpr;
  // q / vpr as (q * magic) >> 40 with magic = floor(2^40 / vpr) + 1: the error term is
  // below q / 2^40 < 2^-16 while the fractional part of q / vpr is at most
  // 1 - 1/vpr, so the quotient is exact for q < 2^24 and vpr <= 2^11 (m*n <= 2^26).
  const uint64_t magic = (0x10000000000ull / vpr) + 1;
  const uint32_t ld = (uint32_t)A.ld;
  const uint32_t v0 = tile * A.vpt;
  const uint32_t v1 = v0 + A.vpt < nvec ? v0 + A.vpt : nvec;
  const int32_t ph = *gl(A.phase);
  int32_t bestR = kBig;
  uint32_t bestQ = 0xffffffffu;
  for (uint32_t q0 = v0 + (uint32_t)tid; q0 < v1; q0 += U * G) {
    i32x4 cv[U], vv[U];
    int32_t uu[U];
#pragma unroll
    for (int k = 0; k < U; ++k) {
      const uint32_t q = q0 + (uint32_t)k * G;
      const uint32_t qq = q < v1 ? q : q0;  // slots past the tile repeat the rank's first vector
      const uint32_t r = (uint32_t)(((uint64_t)qq * magic) >> 40);
      const uint32_t c4 = 4 * (qq - r * vpr);
      cv[k] = *(const FLOCK_GLOBAL i32x4*)(cost + (r * ld + c4));
      uu[k] = du[r];
      vv[k] = *(const FLOCK_GLOBAL i32x4*)(dv + c4);
    }
#pragma unroll
    for (int k = 0; k < U; ++k) {
      const uint32_t q = q0 + (uint32_t)k * G;
      // padding cells price above every real cell of their vector (see sweep_argmin)
      const int32_t mn =
          imin(imin(cv[k].x - vv[k].x, cv[k].y - vv[k].y), imin(cv[k].z - vv[k].z, cv[k].w - vv[k].w)) - uu[k];
      const bool better = mn < bestR;  // a repeated vector never is
      bestR = better ? mn : bestR;
      bestQ = better ? q : bestQ;
    }
  }
  if (ph != 1) return;  // uniform over the grid
  // the rank's best cell: its vector reloaded, the first cell at the minimum
  const bool none = bestQ == 0xffffffffu;
  const uint32_t qb = none ? v0 : bestQ;
  const uint32_t rb = (uint32_t)(((uint64_t)qb * magic) >> 40);
  const uint32_t cb = 4 * (qb - rb * vpr);
  const i32x4 c = *(const FLOCK_GLOBAL i32x4*)(cost + (rb * ld + cb));
  const int32_t ub = du[rb];
  const i32x4 vb = *(const FLOCK_GLOBAL i32x4*)(dv + cb);
  const int e = c.x - vb.x - ub == bestR ? 0 : c.y - vb.y - ub == bestR ? 1 : c.z - vb.z - ub == bestR ? 2 : 3;
  const int32_t ce = e == 0 ? c.x : e == 1 ? c.y : e == 2 ? c.z : c.w;
  const uint32_t colb = cb + (uint32_t)e;
  const uint64_t key = none ? kNoKey : pack_vi(bestR, cell_id(rb, colb));
  // one candidate per 16-lane row of each wavefront (kTileCands per tile): the row's
  // least key by DPP row shifts lands in the row's lane 15
  uint64_t rk = key;
  rk = MinU64Row{}(rk, dpp_u64<0x111, 0xf>(kNoKey, rk));
  rk = MinU64Row{}(rk, dpp_u64<0x112, 0xf>(kNoKey, rk));
  rk = MinU64Row{}(rk, dpp_u64<0x114, 0xf>(kNoKey, rk));
  rk = MinU64Row{}(rk, dpp_u64<0x118, 0xf>(kNoKey, rk));
  const int row16 = lane >> 4;
  const uint64_t r0 = readlane_u64(rk, 15), r1 = readlane_u64(rk, 31), r2 = readlane_u64(rk, 47),
                 r3 = readlane_u64(rk, 63);
  const uint64_t rowMin = row16 == 0 ? r0 : row16 == 1 ? r1 : row16 == 2 ? r2 : r3;
  int32_t* cw = A.cands + 3 * ((size_t)tile * kTileCands + (size_t)wave * 4 + (size_t)row16);
  if (rowMin == kNoKey) {
    if ((lane & 15) == 0) cw[0] = -1;
  } else if (key == rowMin) {  // the one lane holding the row's best cell (keys are unique)
    cw[0] = (int32_t)rb; cw[1] = (int32_t)colb; cw[2] = ce;
  }
  const uint64_t wk = r0 < r1 ? (r0 < r2 ? (r0 < r3 ? r0 : r3) : (r2 < r3 ? r2 : r3))
                              : (r1 < r2 ? (r1 < r3 ? r1 : r3) : (r2 < r3 ? r2 : r3));
  const uint64_t bk = group_min_u64<G>(wk, S);
  if (tid == 0) A.keys[tile] = bk;
}

// ---------------------------------------------------------------------------
// One stepping-stone pivot on entering cell (ei, ej) with reduced cost r < 0
// (perform_a_sequencial_pivot / execute_pivot_on_host / do_flow_adjustment_on_host,
// PIVOT_uv.cu:156-308, 318-401):
//  A. cycle discovery, parallel over vertices: x is on the tree path between row I and
//     column J iff it is an ancestor-or-self of exactly one of them.  The arc (x,
//     parent x) carries -theta when x has the type of the path end it hangs from (rows
//     on I's side, columns on J's side).  Leaving arc = the FIRST minimum flow among
//     the -theta arcs in path order J -> apex -> I (PIVOT_uv.cu:280-296), found with
//     one group min over (flow, side, depth rank, vertex) keys.
//  B. flows +-theta on the path; the chain a = P[0] .. P[k] = q from the leaving arc's
//     lower vertex a down to the entering endpoint q inside subtree(a) is recorded with
//     a snapshot of its old preorder number, size, arc slot and (updated) arc flow.
//  C. subtree(a) is cut, re-rooted at q and hung below the other endpoint o, as o's
//     first child.  Every vertex's new preorder number, depth, size, parent, arc
//     slot/flow and dual follow from its own old values, the snapshot and a few scalars,
//     so all vertices update in place in parallel (the re-rooted subtree's preorder is
//     the concatenation of the old intervals of P[k], P[k-1] minus P[k], ..., P[0]
//     minus P[1]).  The entering arc takes the leaving arc's slot (PIVOT_uv.cu:248-261);
//     duals in the subtree shift by -/+ r so that the entering arc becomes tight.
// ---------------------------------------------------------------------------
template <int N>
struct IntC { static constexpr int value = N; };

// Phase timers: reading the clock takes 80 cycles and drains the LDS queue, and a pivot has
// four readings, so every eighth event of a kind is timed, the first one among them.  Events
// are counted over the whole solve (pivots, and sweeps but the candidate rule's few, which
// are all timed) or over one call (candidate re-pricings), and the samples' sum is scaled to
// all of them at the end.
constexpr int kTimedEvery = 8;
__device__ __forceinline__ bool timed_event(int count) { return count % kTimedEvery == 0; }
__device__ __forceinline__ int64_t scale_samples(int64_t sum, int64_t events) {
  const double samples = (double)((events + kTimedEvery - 1) / kTimedEvery);
  return events > 0 ? (int64_t)((double)sum * ((double)events / samples) + 0.5) : 0;
}

// kR: vertices each rank handles per pass, their LDS loads issued together.
// kWideWin: the re-root's windowed form takes twice the slots per rank where kR is below
// four (the graph path's round kernel and the work-queue kernels below 1024 threads; the
// 1024-thread work-queue kernel keeps kR, as it would spill more in its other phases).
template <int G, int kR, class SN, bool kWideWin = false>
__device__ __forceinline__ bool pivot_pass(const Ctx& C, const TreeLds& t, const SN& sn, Shared& S, int ei, int ej, int32_t r,
                                           int count) {
  const int m = C.m, V = C.V, tid = grank<G>();
  const bool timed = timed_event(count);
  uint64_t t0 = 0;
  if (timed) t0 = now_ticks();
  const int I = ei, J = m + ej;
  // every scalar the in-place pass needs is read here or taken from the snapshot: once
  // the group minimum is known, ranks go straight on to rewrite their own vertices
  const int preI = t.pre(I), preJ = t.pre(J), depI = t.depth[I], depJ = t.depth[J];
  const int sel = count & 1;
  // ---- A: leaving arc, and every cycle vertex snapshotted by side and depth (the least
  // cycle depth, one below the apex, goes to S.dlo[sel])
  uint64_t best = kNoKey;
  int dlo = 0x7fffffff;
  // with several vertices per rank, every LDS load of a pass is issued before the first
  // use (no per-vertex branch waits on a load), so one wait covers all kR vertices
  for (int x0 = tid; x0 < V; x0 += kR * G) {
    int px[kR], sx[kR], dx[kR], slx[kR];
    int32_t fx[kR];
#pragma unroll
    for (int u = 0; u < kR; ++u) {
      const int x = x0 + u * G;
      const int xx = x < V ? x : 0;
      const int32_t psv = t.pre_size(xx);
      px[u] = ps_pre(psv);
      const int sv = ps_size(psv);
      sx[u] = x < V ? sv : 0;  // size 0: never an ancestor
      if constexpr (kR > 1) { dx[u] = t.depth[xx]; fx[u] = t.flow[xx]; slx[u] = t.slot[xx]; }
    }
#pragma unroll
    for (int u = 0; u < kR; ++u) {
      const int x = x0 + u * G;
      const bool aI = (uint32_t)(preI - px[u]) < (uint32_t)sx[u];  // px <= preI < px + sx
      const bool aJ = (uint32_t)(preJ - px[u]) < (uint32_t)sx[u];
      if (aI != aJ) {
        // one vertex per rank: only cycle vertices load the rest (fewer LDS reads)
        if constexpr (kR == 1) { dx[u] = t.depth[x]; fx[u] = t.flow[x]; slx[u] = t.slot[x]; }
        const int d = dx[u];
        const int sd = aI ? 0 : 1;
        sn.vert(sd)[d] = (int16_t)x; sn.ps(sd)[d] = pack_ps(px[u], sx[u]);
        sn.slot(sd)[d] = (int16_t)slx[u]; sn.flow(sd)[d] = fx[u];
        dlo = d < dlo ? d : dlo;
        const uint32_t lowbits =
            aI ? ((1u << 31) | ((uint32_t)d << 16) | (uint32_t)x) : (((32767u - (uint32_t)d) << 16) | (uint32_t)x);
        const uint64_t k = aI == (x < m) ? (((uint64_t)(uint32_t)fx[u] << 32) | lowbits) : kNoKey;
        best = k < best ? k : best;
      }
    }
  }
  if (dlo != 0x7fffffff) {
    int z = 0;  // opaque: known to be uniform, the address would get a loop over the lanes
    asm volatile("" : "+v"(z));
    atomicMin(&S.dlo[sel + z], dlo);
  }
  best = group_min1_u64<G, 1>(best, S);  // its barrier also publishes the snapshot
  if (best == kNoKey) return false;  // no blocking arc: the tree is corrupt (the same in every rank)
  const int a = (int)(best & 0xffffu);
  const int32_t theta = (int32_t)(best >> 32);
  const bool sideI = (best >> 31) & 1u;
  const int dA = sideI ? (int)((best >> 16) & 0x7fffu) : 32767 - (int)((best >> 16) & 0x7fffu);
  const int o = sideI ? J : I;
  uint64_t t1 = 0;
  if (timed) {
    t1 = now_ticks();
    if (tid == 0) S.tk[4] += (int64_t)(t1 - t0);
  }
  // the chain P[0] = a .. P[k] = q on q's side: snapshot entries dA .. dA + k
  const int qs = sideI ? 0 : 1;
  const int32_t psA = sn.ps(qs)[dA];
  const int A = ps_pre(psA), s = ps_size(psA), slotA = sn.slot(qs)[dA];
  const int k = (sideI ? depI : depJ) - dA;
  const int B = sideI ? preJ : preI;
  const int dO = sideI ? depJ : depI;
  const auto cVert = sn.vert(qs) + dA;
  const auto cPS = sn.ps(qs) + dA;
  const auto cSlot = sn.slot(qs) + dA;
  const auto cFlow = sn.flow(qs) + dA;
  // ---- C (in place): flows +-theta on the cycle, subtree(a) re-rooted at q below o
  const int newStart = B < A ? B + 1 : B - s + 1;
  const int32_t dRow = sideI ? r : -r;   // q = I: u += r, v -= r ; q = J: u -= r, v += r
  const int32_t dCol = -dRow;
  // binary search for the deepest chain vertex P[tt] whose old interval holds a position:
  // the candidate range [lo, lo + len) shrinks by the same scalar half in every lane, so
  // a probe lo + half never passes k; "P[c] holds p" is true for c <= tt and false
  // after, and false for every c >= 1 outside subtree(a), where lo stays 0
  const int len0 = uniform(k + 1);
  // window: subtree(a) and the pre-order positions it moves across (the same in every
  // lane; readfirstlane makes the branch below, which holds a barrier, scalar).  The
  // windowed form keeps three values per window slot; with kWideWin it takes twice the
  // dense form's vertices per rank where those are fewer than four (one below 2G
  // vertices, two on 1024-thread groups): every window then fits one pass up to 2G
  // vertices, and up to 4G at 1024 threads
  const int wsize = uniform(B < A ? A + s - 1 - B : B - A + 1);
  constexpr int kRW = kWideWin && kR < 4 ? 2 * kR : kR;
  if (wsize <= kRW * G) {
    // Windowed form, whenever this pivot's window fits one pass (whatever m+n).  Only
    // the pre-order window [wlo, whi] (subtree(a) and the vertices it moves across)
    // changes pre-order number, depth or dual, and only cycle vertices change size,
    // flow, parent or slot.  Window positions are visited through vat; cycle vertices
    // through the snapshot (depths dLca+1 .. depI on I's side, .. depJ on J's side).
    const int dLca = S.dlo[sel] - 1;
    const int n0 = depI - dLca, nc = n0 + depJ - dLca;
    // window slot w = rank + u*G: the subtree's positions first (w < s: A + w), then the
    // positions it moves across (B < A: B+1 .. A-1; else A+s .. B, i.e. A + w again)
    const int outBase = B < A ? B + 1 - s : A;
    const int shift = B < A ? s : -s;  // every window position outside subtree(a) moves
    const int depBase = dO + 1 + k - dA;  // new depth of subtree vertices: depBase + old - 2 tt
    const int dvIdx = (int)(t.dv - t.du) - m;  // column x's dual at t.du[x + dvIdx]
    // the rank index, opaque here: slot numbers rank + u*G are recomputed (one add)
    // instead of being hoisted to the kernel start and kept in scratch
    int tidr = tid;
    asm volatile("" : "+v"(tidr));
    int xs[kRW], np[kRW];  // vertex (complemented: none) and new position of each slot
#pragma unroll
    for (int u = 0; u < kRW; ++u) { xs[u] = -1; np[u] = 0; }
    // NS slots of this wavefront: a wavefront takes only the slots that reach the window
    // (half of them on average; four slots' work for every window was a fifth of a pivot's
    // instructions)
    auto slots = [&](auto ns) {
      constexpr int NS = decltype(ns)::value;
      int lo[NS];
#pragma unroll
      for (int u = 0; u < NS; ++u) {
        const int w = tidr + u * G;
        const int p = (w < s ? A : outBase) + w;
        const bool valid = w < wsize;
        // slots past the window read position 0, the root, and keep it complemented: the
        // root is never in the window (it has no parent arc), so no rank rewrites its
        // depth or dual in this pass; vat itself is rewritten only after the barrier below
        const int x = t.vat[valid ? p : 0];
        xs[u] = valid ? x : ~x;
        lo[u] = 0;
      }
      // every slot searches (a slot outside the subtree keeps lo = 0)
      for (int len = len0; len > 1;) {
        const int half = len >> 1;
        int32_t v[NS];
#pragma unroll
        for (int u = 0; u < NS; ++u) v[u] = cPS[lo[u] + half];
#pragma unroll
        for (int u = 0; u < NS; ++u) {
          const int p = A + tidr + u * G;
          const bool anc = (uint16_t)(p - v[u]) < (uint16_t)((uint32_t)v[u] >> 16);  // p - pre < size
          lo[u] = anc ? lo[u] + half : lo[u];
        }
        len -= half;
      }
#pragma unroll
      for (int u = 0; u < NS; ++u) {
        const int w = tidr + u * G;
        const bool inSub = w < s;
        const int p = (inSub ? A : outBase) + w;
        const int tt = lo[u];
        const int x = xs[u] < 0 ? ~xs[u] : xs[u];
        const int dx = t.depth[x], di = x < m ? x : x + dvIdx;
        const int32_t du = t.du[di];
        // P[tt] \ P[tt+1] follows P[tt+1]'s interval; for tt = k (P[k] = q) entry t1 = k
        // gives p >= p1, so the same formula leaves q's interval in place
        const int t1 = tt < k ? tt + 1 : k;
        const int32_t v0 = cPS[tt], v1 = cPS[t1];
        const int p1 = ps_pre(v1), sz1 = ps_size(v1);
        const int nrel = p - ps_pre(v0) + (p < p1 ? sz1 : 0);
        np[u] = inSub ? newStart + nrel : p + shift;
        const int ndep = inSub ? depBase + dx - 2 * tt : dx;
        const int32_t ndual = du + (inSub ? (x < m ? dRow : dCol) : 0);
        if (xs[u] >= 0) {
          t.pre(x) = (int16_t)np[u]; t.depth[x] = (int16_t)ndep;
          t.du[di] = ndual;
        }
      }
    };
    const int reach = wsize - uniform(tid & ~(kWave - 1));  // window slots from this wavefront's first on
    if (kRW > 2 && reach > 2 * G) slots(IntC<(kRW > 2 ? kRW : 2)>{});
    else if (reach > G) slots(IntC<2>{});
    else if (reach > 0) slots(IntC<1>{});
    // cycle vertices: sizes on the paths to o and a, flows +-theta, the chain's arcs
    for (int i = tid; i < nc; i += G) {
      const int sd = i < n0 ? 0 : 1;
      const int d = dLca + 1 + (i < n0 ? i : i - n0);
      const int32_t psx = sn.ps(sd)[d];
      const int x = sn.vert(sd)[d], px = ps_pre(psx), sx = ps_size(psx);
      const int32_t fx = sn.flow(sd)[d];
      const bool chain = sd == qs && d >= dA;
      if (chain) {
        const int tt = d - dA;
        if (tt == k) {
          t.size(x) = (int16_t)s; t.parent[x] = (int16_t)o; t.flow[x] = theta; t.slot[x] = (int16_t)slotA;
        } else {
          const int up = cVert[tt + 1];
          const bool upMinus = sideI ? (up < m) : (up >= m);
          t.size(x) = (int16_t)(s - ps_size(cPS[tt + 1])); t.parent[x] = (int16_t)up;
          t.flow[x] = cFlow[tt + 1] + (upMinus ? -theta : theta); t.slot[x] = cSlot[tt + 1];
        }
      } else {
        const bool ancO = (uint32_t)(B - px) < (uint32_t)sx;
        const bool ancPa = px < A && A < px + sx;  // proper ancestor of a
        t.size(x) = (int16_t)(sx + ((int)ancO - (int)ancPa) * s);
        t.flow[x] = fx + (((sd == 0) == (x < m)) ? -theta : theta);
      }
    }
    gsync<G>();  // publishes every tree field; later readers need nothing below
    // vat and the depth-minimum slots are next read by the next pivot (after its phase
    // A barrier; every caller also has a re-pricing or sweep barrier between pivots), so
    // no barrier closes this pass
#pragma unroll
    for (int u = 0; u < kRW; ++u)
      if (xs[u] >= 0) t.vat[np[u]] = (int16_t)xs[u];
    if (tid == 0) S.dlo[sel ^ 1] = 0x7fffffff;
    if (timed && tid == 0) S.tk[5] += (int64_t)(now_ticks() - t1);
    return true;
  }
  for (int x0 = tid; x0 < V; x0 += kR * G) {
    int px[kR], sx[kR], dx[kR], lo[kR];
    int32_t fl[kR], du[kR];
#pragma unroll
    for (int u = 0; u < kR; ++u) {
      const int x = x0 + u * G;
      // ranks past the last vertex re-read their own first vertex (x0 < V): every other
      // vertex is being rewritten by its own rank in this pass
      const bool in = x < V;
      const int xx = in ? x : x0;
      const int32_t psv = t.pre_size(xx);
      const int pv = ps_pre(psv), sv = ps_size(psv);
      px[u] = in ? pv : -1;
      sx[u] = in ? sv : 0;
      dx[u] = t.depth[xx];
      fl[u] = t.flow[xx];
      du[u] = xx < m ? t.du[xx] : t.dv[xx - m];
    }
#pragma unroll
    for (int u = 0; u < kR; ++u) lo[u] = 0;
    // deepest chain vertex P[tt] that is an ancestor-or-self of x (nested intervals),
    // the kR searches' loads issued together each round; tail ranks (px = -1) hold no
    // interval, so their lo stays 0
    for (int len = len0; len > 1;) {
      const int half = len >> 1;
      int32_t v[kR];
#pragma unroll
      for (int u = 0; u < kR; ++u) v[u] = cPS[lo[u] + half];
#pragma unroll
      for (int u = 0; u < kR; ++u) {
        const bool anc = (uint32_t)(px[u] - ps_pre(v[u])) < (uint32_t)ps_size(v[u]);
        lo[u] = anc ? lo[u] + half : lo[u];
      }
      len -= half;
    }
    // chain entries tt and tt + 1 (clamped to k) for every vertex, loaded together (the
    // arc fields of entry tt + 1 only on the chain itself)
    int cp0[kR], cp1[kR], cs1[kR];
#pragma unroll
    for (int u = 0; u < kR; ++u) {
      const int tt = lo[u], t1 = tt < k ? tt + 1 : k;
      const int32_t v0 = cPS[tt], v1 = cPS[t1];
      cp0[u] = ps_pre(v0); cp1[u] = ps_pre(v1); cs1[u] = ps_size(v1);
    }
    // every field of the vertex is rewritten (unchanged ones with their old value), so
    // the only branches are the tail guard and the chain's arc update
#pragma unroll
    for (int u = 0; u < kR; ++u) {
      const int x = x0 + u * G;
      const bool inSub = A <= px[u] && px[u] < A + s;
      const int tt = lo[u];
      const int py = cp0[u];
      const bool last = tt == k;
      const int sz1 = cs1[u];
      const int rel = px[u] - py;  // position inside P[tt]'s old interval
      const int nrel = last ? rel : sz1 + rel - (px[u] < cp1[u] ? 0 : sz1);
      const bool chain = inSub & (px[u] == py);  // x is P[tt]: its arc becomes the old arc above P[tt+1]
      const int shifted = B < A ? ((B < px[u] && px[u] < A) ? px[u] + s : px[u])
                                : ((A + s <= px[u] && px[u] <= B) ? px[u] - s : px[u]);
      const int npre = inSub ? newStart + nrel : shifted;
      const int ndep = inSub ? dO + 1 + (k - tt) + (dx[u] - (dA + tt)) : dx[u];
      const bool ancO = (uint32_t)(B - px[u]) < (uint32_t)sx[u];
      const bool ancPa = px[u] < A && A < px[u] + sx[u];  // proper ancestor of a
      const int outDelta = ((int)ancO - (int)ancPa) * s;
      const int chainSize = s - (last ? 0 : sz1);
      const int otherSize = sx[u] + (inSub ? 0 : outDelta);
      const int nsize = chain ? chainSize : otherSize;
      const bool aI = (uint32_t)(preI - px[u]) < (uint32_t)sx[u];  // px <= preI < px + sx
      const bool aJ = (uint32_t)(preJ - px[u]) < (uint32_t)sx[u];
      const bool minus = aI == (x < m);  // the arc to the parent carries -theta
      int32_t nflow = fl[u] + (aI != aJ ? (minus ? -theta : theta) : 0);
      const int32_t ndual = du[u] + (inSub ? (x < m ? dRow : dCol) : 0);
      if (x < V) {
        if (chain) {
          int up, sl;
          if (last) {
            up = o; sl = slotA; nflow = theta;
          } else {
            up = cVert[tt + 1];
            const bool upMinus = sideI ? (up < m) : (up >= m);
            sl = cSlot[tt + 1];
            nflow = cFlow[tt + 1] + (upMinus ? -theta : theta);
          }
          t.parent[x] = (int16_t)up; t.slot[x] = (int16_t)sl;
        }
        t.pre(x) = (int16_t)npre; t.depth[x] = (int16_t)ndep; t.size(x) = (int16_t)nsize; t.flow[x] = nflow;
        *(x < m ? &t.du[x] : &t.dv[x - m]) = ndual;
        t.vat[npre] = (int16_t)x;  // nobody reads vat in this pass
      }
    }
  }
  if (tid == 0) S.dlo[sel ^ 1] = 0x7fffffff;
  gsync<G>();
  if (timed && tid == 0) S.tk[5] += (int64_t)(now_ticks() - t1);
  return true;
}

// count: the solve's pivots so far (modulo kTimedEvery, or counted on from there): one pivot
// to the next it grows by one, so its parity alternates.  Returns false, in every rank, when
// the tree is corrupt.
template <int G, bool kWideWin = false, class SN>
__device__ __forceinline__ bool pivot(const Ctx& C, const TreeLds& t, const SN& sn, Shared& S, int ei, int ej,
                                      int32_t r, int count) {
  // 1024-thread groups take two vertices per rank and pass at most (their registers are
  // capped at 128)
  constexpr int kRBig = G >= 1024 ? 2 : 4;
  if (C.V > 2 * G) return pivot_pass<G, kRBig, SN, kWideWin>(C, t, sn, S, ei, ej, r, count);
  return pivot_pass<G, 1, SN, kWideWin>(C, t, sn, S, ei, ej, r, count);
}

// ---------------------------------------------------------------------------
// Multi-pivot rounds (the reference's parallel stepping stone, SS_METHOD::
// perform_a_parallel_pivot, PIVOT_ss.cu:294-580, and its conflict check
// check_pivot_feasibility, parallel_kernels.cu:620-660).  Every rank holds one candidate
// entering cell from the last full sweep.  In a round, ranks whose candidate prices
// negative with the current duals walk its cycle (the tree path row -> apex <- column,
// by parent pointers and depths) and claim each arc on it (an arc is named by its child
// vertex) with an atomicMin of a priority key (more negative reduced cost first, then
// rank); a candidate whose second walk finds every claim still its own is accepted.
// Accepted cycles share no arc, so pivoting them one after another leaves every other
// accepted cycle, its reduced cost and its theta unchanged; they pivot best first.  The
// best candidate always wins.  Rounds repeat on the same candidates (re-priced) up to
// minor_limit times or until none prices negative; then the caller sweeps again.  iter: the
// pivots made before, maxIt: the budget, count: the pivot count at iter = 0.
// `claim` needs V words (the pivot's snapshot region, free between pivots).  Returns
// the pivots made (-1: the tree is corrupt); stops at the iteration budget.
// ---------------------------------------------------------------------------
template <int G, class SN>
__device__ __forceinline__ int multi_pivot(const Ctx& C, const TreeLds& t, const SN& sn, uint32_t* claim,
                                           Shared& S, const Cand& cand, int iter, int maxIt, int rounds, int count) {
  const int m = C.m, V = C.V, tid = grank<G>();
  constexpr uint32_t kRange = (1u << 22) - 1;
  const int I = cand.row, J = m + cand.col;
  const uint32_t mine = cell_id((uint32_t)cand.row, (uint32_t)cand.col);
  bool spent = cand.row < 0;  // this rank's candidate has entered the basis
  int done = 0;
  for (int round = 0; round < rounds && iter + done < maxIt; ++round) {
    int32_t r = 0;
    if (!spent) r = cand.cost - t.du[cand.row] - t.dv[cand.col];
    const bool active = !spent && r < 0;
    const uint32_t mag = (uint32_t)(-(int64_t)r) < kRange ? (uint32_t)(-(int64_t)r) : kRange;
    const uint32_t key = active ? ((kRange - mag) << 10) | ((uint32_t)tid & 1023u) : 0xffffffffu;
    for (int x = tid; x < V; x += G) claim[x] = 0xffffffffu;
    gsync<G>();
    if (active) {
      int x = I, y = J;
      while (t.depth[x] > t.depth[y]) { atomicMin(&claim[x], key); x = t.parent[x]; }
      while (t.depth[y] > t.depth[x]) { atomicMin(&claim[y], key); y = t.parent[y]; }
      while (x != y) { atomicMin(&claim[x], key); atomicMin(&claim[y], key); x = t.parent[x]; y = t.parent[y]; }
    }
    gsync<G>();
    bool accepted = false;
    if (active) {
      bool own = true;
      int x = I, y = J;
      while (own && t.depth[x] > t.depth[y]) { own = claim[x] == key; x = t.parent[x]; }
      while (own && t.depth[y] > t.depth[x]) { own = claim[y] == key; y = t.parent[y]; }
      while (own && x != y) { own = claim[x] == key && claim[y] == key; x = t.parent[x]; y = t.parent[y]; }
      accepted = own;
    }
    gsync<G>();  // the claim words are the pivot's snapshot region from here on
    int inRound = 0;
    while (iter + done < maxIt) {
      const uint64_t k = group_min_u64<G>(accepted ? reprice(C, t, cand) : kNoKey, S);
      if (k == kNoKey || key_val(k) >= 0) break;
      if (accepted && key_idx(k) == mine) { accepted = false; spent = true; }
      if (!pivot<G>(C, t, sn, S, cell_row(k), cell_col(k), key_val(k), count + iter + done)) return -1;
      ++done; ++inRound;
    }
    if (inRound == 0) break;  // nothing prices negative any more (uniform)
  }
  return done;
}

// ---------------------------------------------------------------------------
// Pivot set-up after the tree is built or loaded: the cycle-depth minima, and (tree_index)
// vat, the vertex at each pre-order position.
template <int G>
__device__ __forceinline__ void pivot_init(Shared& S) {
  if (grank<G>() == 0) { S.dlo[0] = 0x7fffffff; S.dlo[1] = 0x7fffffff; }
}
template <int G>
__device__ __forceinline__ void tree_index(const Ctx& C, const TreeLds& t, Shared& S) {
  for (int x = grank<G>(); x < C.V; x += G) t.vat[t.pre(x)] = (int16_t)x;
  pivot_init<G>(S);
  gsync<G>();
}

// The saved tree (server slices, graph-path rounds) is the LDS tree region as it is,
// copied in 16-byte vectors: 20 bytes per vertex and no conversion.  (Seven int32 arrays
// took 28 bytes, a scalar load and a 16-bit store per field and vertex, and a pass to
// rebuild vat.)  A state buffer also holds Vogel's line state when that does not fit LDS.
__host__ __device__ inline size_t state_bytes(int m, int n) {
  const size_t a = tree_lds_bytes(m, n), b = vogel_lds_bytes(m, n);
  return a > b ? a : b;
}
template <int G>
__device__ __forceinline__ void save_state(const char* tree, size_t bytes, gint* st) {
  const int nv = (int)(bytes / 16);
  FLOCK_GLOBAL i32x4* o = (FLOCK_GLOBAL i32x4*)st;
  for (int k = grank<G>(); k < nv; k += G) o[k] = ((const FLOCK_LDS i32x4*)tree)[k];
}
// (the caller's next barrier publishes the tree)
template <int G>
__device__ __forceinline__ void load_state(char* tree, size_t bytes, gcint* st) {
  const int nv = (int)(bytes / 16), tid = grank<G>();
  const FLOCK_GLOBAL i32x4* in = (const FLOCK_GLOBAL i32x4*)st;
  constexpr int U = 4;  // loads in flight
  for (int k0 = tid; k0 < nv; k0 += U * G) {
    i32x4 v[U];
#pragma unroll
    for (int u = 0; u < U; ++u) v[u] = in[k0 + u * G < nv ? k0 + u * G : k0];
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (k0 + u * G < nv) ((FLOCK_LDS i32x4*)tree)[k0 + u * G] = v[u];
  }
}

// Final outputs: basis by slot, duals, objective, count of positive flows.
template <int G>
__device__ __forceinline__ void write_outputs(const Ctx& C, const TreeLds& t, DevInstance& D, Shared& S) {
  const int m = C.m, V = C.V;
  gint* dual = gl(uniform_ptr(D.dual));
  gint* brow = gl(uniform_ptr(D.basis_row));
  gint* bcol = gl(uniform_ptr(D.basis_col));
  gint* bflow = gl(uniform_ptr(D.basis_flow));
  int64_t obj = 0, nz = 0;
  for (int x = grank<G>(); x < V; x += G) {
    dual[x] = dual_of(t, m, x);
    if (x == 0) continue;
    const int p = t.parent[x];
    const int r = x < m ? x : p, c = (x < m ? p : x) - m;
    const int k = t.slot[x];
    if (k < 0 || k >= V - 1 || r < 0 || r >= m || c < 0 || c >= C.n) continue;  // corrupt tree guard
    brow[k] = r; bcol[k] = c; bflow[k] = t.flow[x];
    obj += (int64_t)t.flow[x] * (int64_t)cost_at(C, r, c);
    nz += t.flow[x] != 0;
  }
  obj = group_sum_i64<G>(obj, S);
  nz = group_sum_i64<G>(nz, S);
  if (grank<G>() == 0) { D.objective = obj; D.n_flows = (int32_t)nz; }
}

// ---------------------------------------------------------------------------
// Solve (or advance) one instance with one group.  `region` is the group's LDS region
// of `region_bytes` bytes, starting with its Shared block.
// ---------------------------------------------------------------------------
// kRule: the pricing rule this instantiation carries (kernels are launched for one rule, so
// each keeps only its own state in registers: one kernel for Dantzig and candidates kept
// the candidate set alive through Dantzig's sweeps).
enum { kRuleDantzig = 0, kRuleCandidates = 1, kRuleMulti = 2 };
template <int G, int kRule>
__device__ __forceinline__ void solve_instance(DevInstance& D, char* region, size_t region_bytes, const EngineParams& P) {
  if (D.phase == 2) return;
  Shared& S = *(Shared*)region;
  char* smem = region + shared_bytes();
  const size_t avail = region_bytes - shared_bytes();
  Ctx C;
  C.cost = gl(uniform_ptr(D.cost)); C.costT = gl(uniform_ptr(D.costT));
  C.m = uniform(D.m); C.n = uniform(D.n); C.V = C.m + C.n; C.ld = uniform(D.ld); C.ldT = uniform(D.ldT);
  gcint* supply = gl(uniform_ptr(D.supply));
  gcint* demand = gl(uniform_ptr(D.demand));
  gint* brow = gl(uniform_ptr(D.basis_row));
  gint* bcol = gl(uniform_ptr(D.basis_col));
  gint* bflow = gl(uniform_ptr(D.basis_flow));
  const int m = C.m, n = C.n, V = C.V;
  const TreeLds t = carve_tree(smem, m, n);
  const size_t treeBytes = tree_lds_bytes(m, n);
  const bool auxLds = treeBytes + 4 * aux_ints(m, n) <= avail;
  // 256- and 512-thread engines keep the pivot's snapshot in LDS only (one pivot code
  // path, fewer live registers); the host gives them only instances whose tree and
  // snapshot fit their LDS
  constexpr bool kMulti = kRule == kRuleMulti, kCands = kRule == kRuleCandidates;
  constexpr bool kSnapLdsOnly = G == 256 || G == 512;
  if constexpr (kSnapLdsOnly) {
    if (!auxLds) {
      if (grank<G>() == 0) { D.status = 6; D.phase = 2; D.iterations = 0; }
      return;
    }
  }
  int32_t* aux = kSnapLdsOnly || auxLds ? (int32_t*)(smem + treeBytes) : uniform_ptr(D.scratch);
  const Snap sn = carve_snap<Snap>(aux, V);
  const SnapL snL = carve_snap<SnapL>(aux, V);
  const bool fresh = D.phase == 0;
  int32_t mode = fresh ? 0 : uniform(D.mode);  // switch rule: 1 once multi-pivoting stopped
  const bool lead = grank<G>() == 0;
  if (lead) {
    S.status = 0;
    if (kCands) S.reprice_ticks = 0;
    for (int k = 0; k < 6; ++k) S.tk[k] = fresh ? 0 : D.ticks[k];
    if (fresh) D.t_start = now_ticks();
  }
  uint64_t tp = now_ticks();
  gsync<G>();
  if (fresh) {
    // Vogel and the tree build cannot stop at a slice deadline: count this group as busy
    // meanwhile (relaxed device-scope counter; it only decides when pivoting groups stop)
    if (P.busy && lead) __hip_atomic_fetch_add(P.busy, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    write_padding<G>(C);
    if (P.initial == 1) {
      nwc<G>(C, supply, demand, brow, bcol, bflow);
    } else {
      transpose<G>(C, (int32_t*)smem);
      __threadfence_block();
      gsync<G>();
      vogel<G, G == 512>(C, supply, demand, smem, avail, S, brow, bcol, bflow, uniform_ptr(D.scratch));
    }
    __threadfence_block();
    gsync<G>();
    if (S.status != 0) {
      if (grank<G>() == 0) { D.status = S.status; D.phase = 2; D.iterations = 0; }
      if (P.busy && lead) __hip_atomic_fetch_add(P.busy, -1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      return;
    }
    { const uint64_t t2 = now_ticks(); if (lead) S.tk[0] += (int64_t)(t2 - tp); tp = t2; }
    const bool ok = build_tree<G>(C, brow, bcol, bflow, t, aux, S);
    { const uint64_t t2 = now_ticks(); if (lead) S.tk[1] += (int64_t)(t2 - tp); tp = t2; }
    if (P.busy && lead) __hip_atomic_fetch_add(P.busy, -1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (!ok) {
      if (grank<G>() == 0) { D.status = 2; D.phase = 2; D.iterations = 0; }
      return;
    }
  } else {
    load_state<G>(smem, treeBytes, gl(uniform_ptr(D.state)));
  }
  // padding duals, 0 in a saved tree already (published below)
  if (fresh) {
    for (int j = n + grank<G>(); j < C.ld; j += G) t.dv[j] = 0;
    tree_index<G>(C, t, S);
  } else {
    pivot_init<G>(S);
    gsync<G>();
  }
  // pivots still allowed (this call counts in 32 bits; D.iterations holds the earlier ones)
  const int64_t iter0 = fresh ? 0 : D.iterations;
  const int64_t maxIt = P.max_iterations > 0 ? P.max_iterations : 50LL * V + 100000;
  const int32_t budget = uniform((int32_t)(maxIt - iter0 < 0x7fffffff ? maxIt - iter0 : 0x7fffffff));
  int32_t status = 0;
  bool finished = false;
  int32_t done = 0, sweeps = 0;  // pivots and full sweeps of this call
  int32_t priced = 0;            // candidate re-pricings of this call's earlier lists
  // the earlier calls' pivots and sweeps, modulo kTimedEvery
  const int32_t count0 = uniform((int32_t)iter0 & (kTimedEvery - 1));
  const int32_t scount0 = fresh ? 0 : uniform((int32_t)D.sweeps & (kTimedEvery - 1));
  constexpr int K = kCands ? CandsPerRank<G>::value : 1;
  CandSet<K> cands;
  cands.clear();
  SweepShape shape{};
  if constexpr (!SweepChunks<G>::value) shape = sweep_shape<G>(m, C.ld >> 2);
  int minor = 0;
  bool haveList = false;
  for (;;) {
    uint64_t key;
    if (kCands && haveList && minor < P.minor_limit) {
      const bool timed = timed_event(priced + minor);
      if (timed) tp = now_ticks();
      key = group_min1_u64<G, 0>(reprice_set(t, cands), S);
      if (timed && lead) S.reprice_ticks += (int64_t)(now_ticks() - tp);
      ++minor;
      if (key_val(key) >= 0) { haveList = false; continue; }
    } else {
      priced += minor;
      const bool timed = kCands || timed_event(scount0 + sweeps);
      if (timed) tp = now_ticks();
      key = sweep_argmin<G, K>(C, t, S, shape, cands);
      if (timed && lead) S.tk[2] += (int64_t)(now_ticks() - tp);
      ++sweeps;
      haveList = kCands;
      minor = 0;
      if (key == kNoKey || key_val(key) >= 0) { finished = true; break; }
    }
    if (done >= budget) { status = 1; finished = true; break; }
    if (P.step_pivots > 0 && done >= P.step_pivots) break;
    // one decision for the whole group, >= 1 pivot per call: after every sweep (where it
    // costs little beside it), and on every fourth pivot of a candidate list (the clock, a
    // barrier and, past the deadline, a read of the launch's counter)
    if (P.deadline && (kCands ? done % 4 == 1 : done > 0)) {
      if (lead)
        S.stop = now_ticks() >= P.deadline &&
                 (!P.busy || __hip_atomic_load(P.busy, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == 0);
      gsync<G>();
      if (S.stop) break;
    }
    if constexpr (kMulti) {  // multi-pivot: every accepted disjoint cycle of this sweep
      if (mode == 0) {
        // the switch rule makes one claim round per sweep and leaves multi-pivoting for
        // good once a round pivots fewer than 10 times (switch_model_parallel.cu:182-184)
        const bool sw = P.pricing == 4;
        int made;
        if constexpr (kSnapLdsOnly)
          made = multi_pivot<G>(C, t, snL, (uint32_t*)aux, S, cands.get(0), done, budget, sw ? 1 : P.minor_limit, count0);
        else
          made = multi_pivot<G>(C, t, sn, (uint32_t*)aux, S, cands.get(0), done, budget, sw ? 1 : P.minor_limit, count0);
        if (made < 0) { status = 2; finished = true; break; }
        done = uniform(done + made);
        if (sw && made < 10) mode = 1;
        continue;
      }
    }
    const int ei = cell_row(key), ej = cell_col(key);
    bool ok;
    if (kSnapLdsOnly || auxLds) ok = pivot<G, (G < 1024)>(C, t, snL, S, ei, ej, key_val(key), count0 + done);
    else ok = pivot<G, (G < 1024)>(C, t, sn, S, ei, ej, key_val(key), count0 + done);
    if (!ok) { status = 2; finished = true; break; }
    ++done;
  }
  if (finished) {
    write_outputs<G>(C, t, D, S);
  } else {
    save_state<G>(smem, treeBytes, gl(uniform_ptr(D.state)));
  }
  if (lead) {
    // a fresh instance's counters start at zero (the launch's reset cleared them)
    if (finished) D.status = status;
    D.phase = finished ? 2 : 1;
    const int64_t allPivots = (fresh ? 0 : D.iterations) + done, allSweeps = (fresh ? 0 : D.sweeps) + sweeps;
    D.iterations = allPivots;
    D.sweeps = allSweeps;
    D.mode = mode;
    for (int k = 0; k < 6; ++k) D.ticks[k] = S.tk[k];
    if (kCands) D.ticks[3] = S.tk[3] + scale_samples(S.reprice_ticks, priced + minor);
    if (finished) {
      if (!kCands) D.ticks[2] = scale_samples(S.tk[2], allSweeps);
      for (int k = 4; k < 6; ++k) D.ticks[k] = scale_samples(S.tk[k], allPivots);
      D.t_done = now_ticks();
    }
  }
  gsync<G>();
}

// ---------------------------------------------------------------------------
// Large-instance path: the solve loop split into kernels that communicate only through
// global memory between launches (the host captures them in a graph):
//   setup  (one workgroup): transpose, initial basis, tree; tree and duals -> state
//   sweep  (a grid, one tile of the matrix per workgroup; sweep_tile): tile argmin key
//          and per-wavefront best cells, duals read from the saved state
//   round  (one workgroup): state -> LDS; argmin over the tile keys; one pivot (Dantzig)
//          or a pivot plus re-priced candidate pivots (candidate list); state <- LDS,
//          or the outputs when no reduced cost is negative.
// D.phase is 1 while the loop runs and 2 when done; later kernels return at once.
// ---------------------------------------------------------------------------
template <int G>
__device__ __forceinline__ void large_setup(DevInstance& D, char* region, size_t region_bytes, const EngineParams& P,
                            gcshort* books) {
  Shared& S = *(Shared*)region;
  char* smem = region + shared_bytes();
  const size_t avail = region_bytes - shared_bytes();
  Ctx C;
  C.cost = gl(uniform_ptr(D.cost)); C.costT = gl(uniform_ptr(D.costT));
  C.m = uniform(D.m); C.n = uniform(D.n); C.V = C.m + C.n; C.ld = uniform(D.ld); C.ldT = uniform(D.ldT);
  gint* brow = gl(uniform_ptr(D.basis_row));
  gint* bcol = gl(uniform_ptr(D.basis_col));
  gint* bflow = gl(uniform_ptr(D.basis_flow));
  // tree_global: the tree lives in the instance's state buffer for the whole solve
  // (instances whose tree does not fit LDS); otherwise in LDS, saved to state per round
  const bool treeGlobal = P.tree_global != 0;
  char* gtree = (char*)uniform_ptr(D.state);
  const size_t treeBytes = tree_lds_bytes(C.m, C.n);
  const bool auxLds = !treeGlobal && treeBytes + 4 * aux_ints(C.m, C.n) <= avail;
  const bool lead = grank<G>() == 0;
  if (lead) {
    S.status = 0;
    for (int k = 0; k < 6; ++k) S.tk[k] = 0;
    D.t_start = now_ticks();
  }
  uint64_t tp = now_ticks();
  gsync<G>();
  if (P.initial == 1) {
    nwc<G>(C, gl(uniform_ptr(D.supply)), gl(uniform_ptr(D.demand)), brow, bcol, bflow);
  } else {
    if (!books) {  // with books the grid kernels have transposed the matrix already
      transpose<G>(C, (int32_t*)smem);
      __threadfence_block();
      gsync<G>();
    }
    vogel<G, true>(C, gl(uniform_ptr(D.supply)), gl(uniform_ptr(D.demand)), smem, avail, S, brow, bcol, bflow,
             uniform_ptr(D.scratch), books, treeGlobal ? gtree : nullptr);
  }
  __threadfence_block();
  gsync<G>();
  bool ok = S.status == 0;
  { const uint64_t t2 = now_ticks(); if (lead) S.tk[0] += (int64_t)(t2 - tp); tp = t2; }
  // one call for a tree and scratch in LDS, so that its accesses are LDS ones
  auto finish = [&](const TreeLds& t, int32_t* aux) {
    ok = build_tree<G>(C, brow, bcol, bflow, t, aux, S);
    if (!ok) return;
    write_padding<G>(C);
    for (int j = C.n + grank<G>(); j < C.ld; j += G) t.dv[j] = 0;  // padding duals
    tree_index<G>(C, t, S);
  };
  if (ok) {
    if (auxLds) finish(carve_tree(smem, C.m, C.n), (int32_t*)(smem + treeBytes));
    else finish(carve_tree(treeGlobal ? gtree : smem, C.m, C.n), uniform_ptr(D.scratch));
  }
  { const uint64_t t2 = now_ticks(); if (lead) S.tk[1] += (int64_t)(t2 - tp); tp = t2; }
  // a tree in global memory stays where it is; the sweep grid reads its duals there
  if (ok && !treeGlobal) save_state<G>(smem, treeBytes, gl(uniform_ptr(D.state)));
  if (lead) {
    for (int k = 0; k < 6; ++k) D.ticks[k] = S.tk[k];
    D.iterations = 0; D.sweeps = 0; D.mode = 0;
    if (ok) { D.status = 0; D.phase = 1; }
    else { D.status = S.status != 0 ? S.status : 2; D.phase = 2; D.t_done = now_ticks(); }
  }
}

// geo: the instance's sizes and buffers (a copy in the kernel's arguments, so that its first
// loads do not wait for the descriptor's); D: the descriptor in memory.
// kTreeGlobal: the tree lives in the state buffer (see large_setup).  With the choice made
// at run time every access to the tree was a flat one: at 1000x1000 a pivot's cycle pass
// took 1.9 us instead of 1.2.
template <int G, int kRule, bool kTreeGlobal>
__device__ __forceinline__ void large_round(DevInstance& D, const DevInstance& geo, char* region, size_t region_bytes,
                            const EngineParams& P, const uint64_t* keys, const int32_t* cands, int nblocks) {
  constexpr bool kMulti = kRule == kRuleMulti, kCands = kRule == kRuleCandidates;
  Shared& S = *(Shared*)region;
  char* smem = region + shared_bytes();
  const size_t avail = region_bytes - shared_bytes();
  Ctx C;
  C.cost = gl(geo.cost); C.costT = gl(geo.costT);
  C.m = geo.m; C.n = geo.n; C.V = C.m + C.n; C.ld = geo.ld; C.ldT = geo.ldT;
  const int tid = grank<G>();
  const TreeLds t = carve_tree(kTreeGlobal ? (char*)geo.state : smem, C.m, C.n);
  const size_t treeBytes = tree_lds_bytes(C.m, C.n);
  const bool auxLds = !kTreeGlobal && treeBytes + 4 * aux_ints(C.m, C.n) <= avail;
  int32_t* aux = auxLds ? (int32_t*)(smem + treeBytes) : geo.scratch;
  const Snap sn = carve_snap<Snap>(aux, C.V);
  const SnapL snL = carve_snap<SnapL>(aux, C.V);
  const bool lead = tid == 0;
  // the phase is tested after the tree's loads are under way: a finished instance's rounds
  // load it for nothing, the others save a memory round trip
  const int32_t phase = D.phase;
  if constexpr (!kTreeGlobal) load_state<G>(smem, treeBytes, gl((const int32_t*)geo.state));
  if (phase != 1) return;
  if (lead) {
    S.status = 0;
    if (kCands) S.reprice_ticks = 0;
    for (int k = 0; k < 6; ++k) S.tk[k] = D.ticks[k];
  }
  pivot_init<G>(S);
  gsync<G>();
  uint64_t key = kNoKey;
  for (int b = tid; b < nblocks; b += G) { const uint64_t k = keys[b]; key = k < key ? k : key; }
  key = group_min_u64<G>(key, S);
  // candidate list: the tiles' candidates dealt round-robin to the ranks; the i-th one a
  // rank is dealt goes to its slot i % K, and each slot keeps the one that prices lowest
  // with the current duals (the candidate rule re-prices the whole set in its minor
  // iterations; the multi-pivot rules take the rank's best)
  constexpr int K = CandsPerRank<G>::value;
  CandSet<K> cs;
  cs.clear();
  Cand cand;
  cand.row = -1; cand.col = 0; cand.cost = 0;
  if constexpr (kRule != kRuleDantzig) {
    uint64_t bestk[K];
#pragma unroll
    for (int k = 0; k < K; ++k) bestk[k] = kNoKey;
    uint64_t bestc = kNoKey;
    int slot = 0;
    for (int q = tid; q < nblocks * kTileCands; q += G) {
      const int32_t* c = cands + 3 * q;
      Cand x;
      x.row = c[0];
      x.col = x.row < 0 ? 0 : c[1];
      x.cost = x.row < 0 ? 0 : c[2];
      const uint64_t k = x.row < 0 ? kNoKey : reprice(C, t, x);
#pragma unroll
      for (int e = 0; e < K; ++e)
        if (e == slot && k < bestk[e]) { bestk[e] = k; cs.set(e, x); }
      if (k < bestc) { bestc = k; cand = x; }
      slot = slot + 1 < K ? slot + 1 : 0;
    }
  }
  // multi-pivot rules: rank 0 holds the sweep's argmin cell, so every round pivots at
  // least once whatever tiles the ranks' candidates came from (the grid can have more
  // tiles than a rank per wavefront candidate)
  if (kMulti && tid == 0 && key != kNoKey && key_val(key) < 0) {
    cand.row = cell_row(key);
    cand.col = cell_col(key);
    cand.cost = cost_at(C, cand.row, cand.col);
  }
  int64_t iter = D.iterations;
  const int64_t maxIt = P.max_iterations > 0 ? P.max_iterations : 50LL * C.V + 100000;
  int32_t status = 0;
  bool finished = key == kNoKey || key_val(key) >= 0;
  bool multiDone = false;
  int32_t mode = D.mode;  // switch rule: 1 once multi-pivoting stopped
  if constexpr (kMulti) {  // multi-pivot rounds on the tiles' candidates
    if (!finished && mode == 0) {
      multiDone = true;
      if (iter >= maxIt) { status = 1; finished = true; }
      else {
        const bool sw = P.pricing == 4;
        const int made = multi_pivot<G>(C, t, sn, (uint32_t*)aux, S, cand, 0,
                                        maxIt - iter < 0x7fffffff ? (int)(maxIt - iter) : 0x7fffffff,
                                        sw ? 1 : P.minor_limit, (int)iter);
        if (made < 0) { status = 2; finished = true; }
        else iter += made;
        if (sw && made < 10) mode = 1;
      }
    }
  }
  int priced = 0;  // candidate re-pricings of this round
  if (!finished && !multiDone) {
    int minor = 0;
    for (;;) {
      if (iter >= maxIt) { status = 1; finished = true; break; }
      const int ei = cell_row(key), ej = cell_col(key);
      bool ok;
      if (auxLds) ok = pivot<G, true>(C, t, snL, S, ei, ej, key_val(key), (int)iter);
      else ok = pivot<G, true>(C, t, sn, S, ei, ej, key_val(key), (int)iter);
      if (!ok) { status = 2; finished = true; break; }
      ++iter;
      if (!kCands || ++minor >= P.minor_limit) break;  // Dantzig: one pivot per sweep
      const bool timed = timed_event(minor - 1);
      uint64_t tp = 0;
      if (timed) tp = now_ticks();
      key = group_min1_u64<G, 0>(reprice_set(t, cs), S);
      if (timed && lead) S.reprice_ticks += (int64_t)(now_ticks() - tp);
      priced = minor;
      if (key_val(key) >= 0) break;  // list exhausted: next full sweep
    }
  }
  if (finished) {
    write_outputs<G>(C, t, D, S);
  } else if constexpr (!kTreeGlobal) {
    gsync<G>();  // the last pivot's vat writes
    save_state<G>(smem, treeBytes, gl(geo.state));
  }
  if (lead) {
    for (int k = 0; k < 6; ++k) D.ticks[k] = S.tk[k];
    if (kCands) D.ticks[3] = S.tk[3] + scale_samples(S.reprice_ticks, priced);
    D.iterations = iter;
    D.mode = mode;
    D.sweeps = D.sweeps + 1;
    if (finished) {
      for (int k = 4; k < 6; ++k) D.ticks[k] = scale_samples(S.tk[k], iter);
      D.status = status; D.phase = 2; D.t_done = now_ticks();
    }
  }
}

// Arguments of the sweep grid for instance D (duals of the tree in its state buffer).
__host__ __device__ inline SweepArgs sweep_args(const DevInstance& D, uint64_t* keys, int32_t* cands, uint32_t vpt,
                                                const int32_t* phase) {
  SweepArgs A;
  const size_t rows = align16(4 * (size_t)((D.m + 3) & ~3)), cols = align16(4 * (size_t)((D.n + 3) & ~3));
  const char* end = (const char*)D.state + tree_lds_bytes(D.m, D.n);  // u and v are the last arrays
  A.cost = D.cost; A.du = (const int32_t*)(end - cols - rows); A.dv = (const int32_t*)(end - cols);
  A.phase = phase; A.keys = keys; A.cands = cands;
  A.m = D.m; A.n = D.n; A.ld = D.ld; A.vpt = vpt;
  return A;
}

// ---------------------------------------------------------------------------
// Persistent work-queue worker (the body of k_solve_queue for workgroup `block` of
// `grid`): every group of G threads (one wavefront or the whole workgroup) pops
// instance indices from `head` and solves them one after another.  With a slice
// deadline no instance is started after it.
// ---------------------------------------------------------------------------
template <int T, int G, int kRule>
__device__ __forceinline__ void queue_worker(DevInstance* insts, const int32_t* order, int32_t count, int32_t* head,
                             const EngineParams& P, char* smem) {
  const size_t region_bytes = (size_t)P.lds_bytes;
  char* region = smem + (size_t)(threadIdx.x / G) * region_bytes;
  Shared& S = *(Shared*)region;
  EngineParams Q = P;
  Q.deadline = P.slice_ticks > 0 ? uniform64(*P.clock0 + P.slice_ticks) : 0;
  for (;;) {
    int idx;
    if constexpr (G == kWave) {
      int v = 0;
      if (grank<G>() == 0) v = (Q.deadline && now_ticks() >= Q.deadline) ? count : atomicAdd(head, 1);
      idx = __shfl(v, 0, kWave);
    } else {
      if (threadIdx.x == 0) S.idx = (Q.deadline && now_ticks() >= Q.deadline) ? count : atomicAdd(head, 1);
      __syncthreads();
      idx = S.idx;
      __syncthreads();
    }
    idx = uniform(idx);
    if (idx >= count) break;
    // the largest instances set the launch's makespan: their waves get issue priority
    // over co-resident workgroups' (uniform per group)
    if (idx < Q.prio_count) __builtin_amdgcn_s_setprio(3);
    else __builtin_amdgcn_s_setprio(0);
    solve_instance<G, kRule>(*uniform_ptr(insts + order[idx]), region, region_bytes, Q);
  }
}

}  // namespace flock

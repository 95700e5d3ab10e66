// Token dispatch for calls too large for the fused router kernel: a stable
// counting sort of assignments by expert (definition in dispatch_dev.h).
//
// Three kernels per batch of calls, all integer work:
//   k_dispatch_count   per 1024-assignment tile: LDS histogram
//   k_dispatch_scan    one block per call: offsets, M-tile offsets, active
//                      list, per-tile bases; marks unused perm slots −1
//   k_dispatch_scatter per tile: stable rank via wavefront ballots (one per id
//                      bit), then place
#include "dispatch_dev.h"

namespace {

using namespace moe_dev;
constexpr int DBLOCK = 256;

__global__ __launch_bounds__(DBLOCK) void k_dispatch_count(const float *__restrict__ route,
                                                           int64_t route_cs, int A, int k,
                                                           DispatchBufs db) {
  __shared__ int32_t hist[DISPATCH_MAX_E];
  const int call = blockIdx.y;
  const int E = db.E;
  route += call * route_cs;
  for (int e = threadIdx.x; e < E; e += DBLOCK) hist[e] = 0;
  __syncthreads();
  const int64_t a0 = (int64_t)blockIdx.x * DISPATCH_TILE;
  for (int i = threadIdx.x; i < DISPATCH_TILE; i += DBLOCK) {
    int64_t a = a0 + i;
    if (a >= A) break;
    int e = route_expert(route, a, k, E);
    if (e >= 0) atomicAdd(&hist[e], 1);
  }
  __syncthreads();
  int32_t *cnt = db.blk_counts + call * db.cnt_cs() + (int64_t)blockIdx.x * E;
  for (int e = threadIdx.x; e < E; e += DBLOCK) cnt[e] = hist[e];
}

// Block counts staged in LDS when they fit: every load is then out at once
// (summing them straight from memory waits one latency per few blocks).
constexpr int SCAN_LDS_COUNTS = 8192;

__global__ __launch_bounds__(1024) void k_dispatch_scan(DispatchBufs db, int tile_m) {
  __shared__ int32_t tot[DISPATCH_MAX_E];
  __shared__ int32_t off[DISPATCH_MAX_E + 1];
  __shared__ int32_t cl[SCAN_LDS_COUNTS];
  const int call = blockIdx.x;
  const int E = db.E, nblk = db.nblk;
  const int32_t *cnt = db.blk_counts + call * db.cnt_cs();
  const bool staged = nblk * E <= SCAN_LDS_COUNTS;
  if (staged) {
    // Up to eight counts a thread, all loaded before the first store (an
    // index past the end reloads the last count, which is not stored).
    const int n = nblk * E;
    for (int i0 = threadIdx.x; i0 < n; i0 += 8 * blockDim.x) {
      int32_t v[8];
#pragma unroll
      for (int u = 0; u < 8; u++) v[u] = cnt[min(i0 + u * (int)blockDim.x, n - 1)];
#pragma unroll
      for (int u = 0; u < 8; u++)
        if (i0 + u * (int)blockDim.x < n) cl[i0 + u * blockDim.x] = v[u];
    }
    __syncthreads();
    cnt = cl;
  }
  for (int e = threadIdx.x; e < E; e += blockDim.x) {
    int32_t c = 0;
    for (int b = 0; b < nblk; b++) c += cnt[(int64_t)b * E + e];
    tot[e] = c;
  }
  __syncthreads();
  if (threadIdx.x < WAVE)
    wave_scan_experts(tot, E, tile_m, threadIdx.x, db.offsets + call * db.off_cs(),
                      db.tile_off + call * db.off_cs(), db.active + call * db.act_cs(),
                      db.meta + call * db.meta_cs(), off);
  __syncthreads();
  int32_t *base = db.blk_base + call * db.cnt_cs();
  for (int e = threadIdx.x; e < E; e += blockDim.x) {
    int32_t run = off[e];
    for (int b = 0; b < nblk; b++) {
      base[(int64_t)b * E + e] = run;
      run += cnt[(int64_t)b * E + e];
    }
  }
  int32_t *perm = db.perm + call * db.perm_cs();
  for (int i = off[E] + threadIdx.x; i < db.A; i += blockDim.x) perm[i] = -1;
}

__global__ __launch_bounds__(DBLOCK) void k_dispatch_scatter(const float *__restrict__ route,
                                                             int64_t route_cs, int A, int k,
                                                             DispatchBufs db) {
  __shared__ int32_t cursor[DISPATCH_MAX_E];
  __shared__ int32_t wc[4 * DISPATCH_MAX_E];
  const int call = blockIdx.y;
  const int E = db.E;
  route += call * route_cs;
  const int32_t *base = db.blk_base + call * db.cnt_cs() + (int64_t)blockIdx.x * E;
  for (int e = threadIdx.x; e < E; e += DBLOCK) cursor[e] = base[e];
  int32_t *perm = db.perm + call * db.perm_cs();
  const int64_t a0 = (int64_t)blockIdx.x * DISPATCH_TILE;
  for (int pass = 0; pass < DISPATCH_TILE / DBLOCK; pass++) {
    int64_t a = a0 + pass * DBLOCK + threadIdx.x;
    int e = (a < A) ? route_expert(route, a, k, E) : -1;
    block_place(e, a, E, cursor, wc, perm);
  }
}

// The whole sort of a call in one block of 16 wavefronts, for calls of up to
// 16 · 64 · NC assignments: each wavefront takes a contiguous run of 64-wide
// chunks, whose ids stay in registers from the count to the placement.
// Bound by latency: one read of the ids, four barriers, one scan, where the
// three kernels above read the ids twice and wait for each other's launches.
// Measured: 308 assignments (E 128) 11.8 → 4.2 µs, 2400 (E 64) 16.8 → 6.4,
// 6000 (E 128) 16.3 → 10.0; 16384 (E 32, 16 chunks a wavefront) 18.0 → 18.2,
// so from 8193 on the three kernels stay.
constexpr int ONE_WAVES = 16;
constexpr int ONE_MAX_A = ONE_WAVES * WAVE * 8;
constexpr int ONE_MAX_E = 512;  // (16 + 2)·E counts in LDS: 37 KB

// Orders the wavefront's LDS accesses before and after it (no instruction:
// the LDS serves a wavefront in order).
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

template <int NC>
__global__ __launch_bounds__(ONE_WAVES *WAVE) void k_dispatch_one(const float *__restrict__ route,
                                                                  int64_t route_cs, int A, int k,
                                                                  DispatchBufs db, int tile_m) {
  extern __shared__ int32_t one_lds[];
  const int call = blockIdx.x;
  const int E = db.E;
  int32_t *wc = one_lds;                // [16][E] counts, then bases, per wavefront
  int32_t *tot = wc + ONE_WAVES * E;    // [E]
  int32_t *off = tot + E;               // [E + 1]
  route += call * route_cs;
  const int lane = threadIdx.x & (WAVE - 1);
  const int wave = threadIdx.x / WAVE;
  const int nc = ((A + WAVE - 1) / WAVE + ONE_WAVES - 1) / ONE_WAVES;  // ≤ NC
  const int a0 = wave * nc * WAVE + lane;
  int id[NC];
#pragma unroll
  for (int i = 0; i < NC; i++) {
    // in bounds: past the run or A, assignment A − 1, not counted
    const int a = a0 + i * WAVE;
    const uint32_t c = (uint32_t)min(a, A - 1), t = c / (uint32_t)k;  // 32-bit: A is small
    const float f = route[(int64_t)t * 2 * k + (c - t * k)];
    const int v = f >= 0.f && f < (float)E ? (int)f : -1;
    id[i] = i < nc && a < A && v >= 0 && (float)v == f ? v : -1;
  }
  for (int i = threadIdx.x; i < ONE_WAVES * E; i += ONE_WAVES * WAVE) wc[i] = 0;
  __syncthreads();
  int32_t *mine = wc + wave * E;
#pragma unroll
  for (int i = 0; i < NC; i++)
    if (id[i] >= 0) atomicAdd(&mine[id[i]], 1);
  __syncthreads();
  for (int e = threadIdx.x; e < E; e += ONE_WAVES * WAVE) {
    int32_t c = 0;
#pragma unroll
    for (int w = 0; w < ONE_WAVES; w++) {
      const int32_t v = wc[w * E + e];
      wc[w * E + e] = c;
      c += v;
    }
    tot[e] = c;
  }
  __syncthreads();
  if (wave == 0)
    wave_scan_experts(tot, E, tile_m, lane, db.offsets + call * db.off_cs(),
                      db.tile_off + call * db.off_cs(), db.active + call * db.act_cs(),
                      db.meta + call * db.meta_cs(), off);
  __syncthreads();
  int32_t *perm = db.perm + call * db.perm_cs();
#pragma unroll
  for (int i = 0; i < NC; i++) {
    if (i >= nc) break;
    const int e = id[i];
    // Lanes with the same expert: one ballot per bit of the id.
    uint64_t same = __ballot(e >= 0);
    for (int bit = 0; (1 << bit) < E; bit++) {
      const uint64_t ones = __ballot(e >= 0 && ((e >> bit) & 1));
      same &= ((e >> bit) & 1) ? ones : ~ones;
    }
    const int rank = __popcll(same & ((1ull << lane) - 1ull));
    const int32_t base = e >= 0 ? mine[e] : 0;
    wave_sync();  // every lane has read before the first one of an expert adds
    if (e >= 0) {
      perm[off[e] + base + rank] = a0 + i * WAVE;
      if (rank == 0) mine[e] = base + __popcll(same);
    }
    wave_sync();  // and the next chunk reads what this one wrote
  }
  for (int i = off[E] + threadIdx.x; i < A; i += ONE_WAVES * WAVE) perm[i] = -1;
}

}  // namespace

int launch_dispatch(const float *route, int64_t route_cs, int T, int E, int k, int calls,
                    int tile_m, const DispatchBufs &db, hipStream_t s) {
  MOE_NONNULL(route);
  MOE_NONNULL(db.blk_counts);
  MOE_NONNULL(db.blk_base);
  MOE_NONNULL(db.offsets);
  MOE_NONNULL(db.tile_off);
  MOE_NONNULL(db.active);
  MOE_NONNULL(db.meta);
  MOE_NONNULL(db.perm);
  if (E > DISPATCH_MAX_E) return moe_fail(MOE_INVALID_ARGUMENT, "dispatch: more than 1024 experts");
  const int A = T * k;
  if (db.E != E || db.A != A || db.nblk != (A + DISPATCH_TILE - 1) / DISPATCH_TILE)
    return moe_fail(MOE_EXECUTION_FAILED, "dispatch: workspace sized for another shape");
  if (A <= ONE_MAX_A && E <= ONE_MAX_E) {
    const size_t lds = sizeof(int32_t) * ((ONE_WAVES + 2) * (size_t)E + 1);
    const dim3 g(calls), b(ONE_WAVES * WAVE);
    if (A <= ONE_WAVES * WAVE)
      hipLaunchKernelGGL(k_dispatch_one<1>, g, b, lds, s, route, route_cs, A, k, db, tile_m);
    else if (A <= 2 * ONE_WAVES * WAVE)
      hipLaunchKernelGGL(k_dispatch_one<2>, g, b, lds, s, route, route_cs, A, k, db, tile_m);
    else if (A <= 4 * ONE_WAVES * WAVE)
      hipLaunchKernelGGL(k_dispatch_one<4>, g, b, lds, s, route, route_cs, A, k, db, tile_m);
    else
      hipLaunchKernelGGL(k_dispatch_one<8>, g, b, lds, s, route, route_cs, A, k, db, tile_m);
    return 0;
  }
  hipLaunchKernelGGL(k_dispatch_count, dim3(db.nblk, calls), dim3(DBLOCK), 0, s, route, route_cs,
                     A, k, db);
  hipLaunchKernelGGL(k_dispatch_scan, dim3(calls), dim3(1024), 0, s, db, tile_m);
  hipLaunchKernelGGL(k_dispatch_scatter, dim3(db.nblk, calls), dim3(DBLOCK), 0, s, route,
                     route_cs, A, k, db);
  return 0;
}

// Float-weight expert products (f32 or f16 weights) for gfx950: the
// privacy filter's float branch.
//
// Reference: src/core/kernels/matmul/matmulGather.ts:38-103 (out[i] =
// a[i]·W[e_i] + bias[e_i], W = rows [e·K, (e+1)·K) of w [E·K, N]),
// src/core/graph/ops/matmul.ts:180-210 (the op), src/zoo/privacy-filter/
// moeMlp.ts:85-100 (the float forward: glu and lin gathers, clamped
// SwiGLU, the out gather, gate-weighted sum over the slots, + x).
//
// Rows arrive grouped by expert (dispatch.hip), so each expert's weight
// rows stream once per 16·RT of its rows, where the reference reads them
// once per (row, slot). A block is one row tile × 64 columns; its 8
// wavefronts split K (up: four parts of glu and four of lin), and their sums
// meet in LDS, added in part order, before the bias and the SwiGLU. The
// products are v_mfma_f32_16x16x4_f32: the weights are row-major [K, N], so
// per 16 k a lane loads four consecutive columns of four weight rows (whole
// 256-byte runs per 16 lanes, read once: nontemporal) and four consecutive k
// of its row, and MFMA step j takes weight row j and element j, with no LDS
// or conversion between (f16 values widen to f32 first). FPD steps are in
// flight per wavefront. A step's sums start from zero and join the total, so
// no chain of additions is longer than 16 or K / 64 terms.
//
// Bound by the weight stream. Measured (E 128, top-4, 640 × 640, 77 tokens,
// f32 weights) against 4-row chunks on the VALU with x in LDS: up 112 → 63 µs,
// down 66 → 34 (6.1 and 5.6 TB/s); 500 tokens, whole block, 649 → 171, f16
// 505 → 126. More steps in flight cost wavefronts that fit (77 tokens, one to
// four steps: 123, 133, 151, 167 µs a block).
#include "moe_internal.h"

namespace {

constexpr int WAVE = 64;
constexpr int FWAVES = 8;
constexpr int FSTEP = 16;  // k per step
constexpr int FCOLS = 64;  // columns per block
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef _Float16 half4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ float swiglu(float glu, float lin) {
  // activations.ts:127-133, exp via the hardware 2^x and the quotient via
  // the hardware reciprocal (each within 1 ulp), as the int8 path does.
  const float g = fminf(glu, 7.0f);
  const float l = fminf(fmaxf(lin, -7.0f), 7.0f);
  const float e = __builtin_amdgcn_exp2f(g * (-1.702f * 1.4426950408889634f));
  return g * __builtin_amdgcn_rcpf(1.0f + e) * (l + 1.0f);
}

// Weights are read once: nontemporal buffer loads. A step's 16 weight rows get
// a descriptor of their own (scalar arithmetic), so the lanes' offsets are
// loop constants and a row past K or a column past N reads zeros. (64-bit row
// addresses per lane cost more VALU time than the products.)
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
constexpr uint32_t F_OOB = 0x80000000u;
__device__ __forceinline__ __amdgpu_buffer_rsrc_t rows_rsrc(const void *base, int bytes) {
  return __builtin_amdgcn_make_buffer_rsrc((void *)base, 0, bytes, 0x00020000 /* raw, 32-bit */);
}
__device__ __forceinline__ void stream4(floatx4 &d, __amdgpu_buffer_rsrc_t r, uint32_t off) {
  d = __builtin_bit_cast(floatx4, __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 2 /* nt */));
}
__device__ __forceinline__ void stream4(half4 &d, __amdgpu_buffer_rsrc_t r, uint32_t off) {
  d = __builtin_bit_cast(half4, __builtin_amdgcn_raw_buffer_load_b64(r, off, 0, 2 /* nt */));
}
__device__ __forceinline__ floatx4 load4(const float *p) { return *(const floatx4 *)p; }
__device__ __forceinline__ half4 load4(const _Float16 *p) { return *(const half4 *)p; }
__device__ __forceinline__ floatx4 wide(floatx4 v) { return v; }
__device__ __forceinline__ floatx4 wide(half4 v) {
  return floatx4{(float)v[0], (float)v[1], (float)v[2], (float)v[3]};
}
__device__ __forceinline__ void store4(float *p, floatx4 v) { *(floatx4 *)p = v; }
__device__ __forceinline__ void store4(_Float16 *p, floatx4 v) {
  *(half4 *)p = half4{(_Float16)v[0], (_Float16)v[1], (_Float16)v[2], (_Float16)v[3]};
}
template <typename T> struct Vec4;
template <> struct Vec4<float> { typedef floatx4 type; };
template <> struct Vec4<_Float16> { typedef half4 type; };

// MODE_UP: act[a] = swiglu(x·glu[e] + bias_glu[e], x·lin[e] + bias_lin[e]).
// MODE_DOWN (and the plain gather): out[a] = x·w[e] + bias[e].
// AT: activation type, WT: weight and bias type, OT: output type.
// K % 16 == 0, % 4 == 0 (rows of a aligned), any; any with weight rows so wide
// that 16 of them pass the buffer offsets (64-bit addresses)
enum KForm { K_STEPS = 0, K_QUADS = 1, K_ANY = 2, K_WIDE = 3 };
constexpr int F_MAX_N = 1 << 24;
// FPD: steps loaded (the one multiplied and those ahead of it).
template <int MODE, typename AT, typename WT, typename OT, int RT, int KF, int FPD>
__global__ __launch_bounds__(FWAVES *WAVE) __attribute__((amdgpu_waves_per_eu(4))) void k_float_tile(FloatArgs p, int gx, int blk0) {
  constexpr int NS = MODE == MODE_UP ? 2 : 1;
  constexpr int KW = FWAVES / NS;           // wavefronts per weight array
  constexpr int ROWS = 16 * RT;
  typedef typename Vec4<AT>::type av4;
  typedef typename Vec4<WT>::type wv4;
  __shared__ floatx4 red[FWAVES][4 * RT][WAVE];

  const int lane = threadIdx.x & (WAVE - 1);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
  const int call = blockIdx.y;
  // This block's row tile and column block, one contiguous range of the
  // call's tiles per XCD (blocks go round-robin over the 8 XCDs).
  const int32_t *meta = p.db.meta + call * p.db.meta_cs();
  const int4 *active = (const int4 *)(p.db.active + call * p.db.act_cs());
  const int E = p.db.E;
  int4 ad = active[min(lane, E - 1)];
  const int na = meta[META_ACTIVE];
  const int total = meta[META_TILES] * gx;
  const int per = (total + 7) / 8;
  const int blk = blk0 + (int)blockIdx.x;  // blk0 a multiple of 8
  const int slot = blk >> 3;
  const int o = (blk & 7) * per + slot;
  if (slot >= per || o >= total) return;
  const int mt = o / gx, xb = o - mt * gx;
  int hit = __popcll(__ballot(lane < na && ad.w <= mt)) - 1;
  for (int b = WAVE; hit == WAVE - 1 && b < na; b += WAVE) {
    const int4 nx = active[min(b + lane, na - 1)];
    const int h = __popcll(__ballot(b + lane < na && nx.w <= mt)) - 1;
    if (h < 0) break;
    ad = nx;
    hit = h;
  }
  const int e = __builtin_amdgcn_readlane(ad.x, hit);
  const int r0 = (mt - __builtin_amdgcn_readlane(ad.w, hit)) * ROWS;
  const int rows = min(ROWS, __builtin_amdgcn_readlane(ad.z, hit) - r0);
  const int p0 = __builtin_amdgcn_readlane(ad.y, hit) + r0;
  const int32_t *perm = p.db.perm + call * p.db.perm_cs() + p0;

  const int arr = wave / KW, part = wave % KW;
  const int m = lane & 15, kq = lane >> 4;
  const int col = xb * FCOLS + 4 * m;  // N is a multiple of 4
  const bool col_ok = col < p.N;
  const int64_t wcall = call * (arr ? p.w1_cs : p.w0_cs);
  const WT *w = (const WT *)(arr ? p.w1 : p.w0) + wcall + (int64_t)e * p.K * p.N;
  uint32_t woff[4];
#pragma unroll
  for (int j = 0; j < 4; j++)
    woff[j] = col_ok ? ((uint32_t)(4 * kq + j) * (uint32_t)p.N + col) * (uint32_t)sizeof(WT) : F_OOB;
  // Rows past the tile read its first one; their sums are not stored.
  const AT *xr[RT];
#pragma unroll
  for (int t = 0; t < RT; t++) {
    const int r = 16 * t + m;
    xr[t] = (const AT *)p.a + call * p.a_cs +
            (int64_t)(perm[r < rows ? r : 0] / p.a_row_div) * p.K;
  }
  const int steps = (p.K + FSTEP - 1) / FSTEP;
  const int sp = (steps + KW - 1) / KW;
  const int s0 = part * sp, s1 = min(steps, s0 + sp);

  struct Step {
    av4 a[RT];
    wv4 b[4];
  };
  // Addresses of a stay inside its rows: a step past the last reads that one
  // (not used), a k past K reads k = 0. Of W, a step past the wavefront's share
  // reads nothing: with five steps a share, two of seven were read for no use
  // (block of 8 tokens, f32 54.5 → 51.0 µs, f16 44.3 → 43.6; 68.5 and 51.6 with
  // the VALU gathers; the same tokens again and again, weights in cache, 53.9 →
  // 50.3 and 44.5 → 43.9, 48.7 and 42.0 with the gathers). Two steps ahead: 52.2
  // and 45.1, three 54.0 and 47.6.
  auto load = [&](int s, Step &d) {
    const bool past = s >= s1;
    s = min(s, steps - 1);
    const int k = s * FSTEP + 4 * kq;
    if constexpr (KF == K_WIDE) {
#pragma unroll
      for (int j = 0; j < 4; j++) {
        const bool ok = k + j < p.K && col_ok;
        const wv4 v = load4(w + (ok ? (int64_t)(k + j) * p.N + col : 0));
#pragma unroll
        for (int c = 0; c < 4; c++) d.b[j][c] = ok ? v[c] : (WT)0;
      }
    } else {
      const int left = past ? 0 : KF == K_STEPS ? FSTEP : min(FSTEP, p.K - s * FSTEP);
      const __amdgpu_buffer_rsrc_t wr =
          rows_rsrc(w + (int64_t)s * FSTEP * p.N, left * p.N * (int)sizeof(WT));
#pragma unroll
      for (int j = 0; j < 4; j++) stream4(d.b[j], wr, woff[j]);
    }
#pragma unroll
    for (int t = 0; t < RT; t++) {
      if constexpr (KF == K_STEPS || KF == K_QUADS) {
        d.a[t] = load4(xr[t] + (KF == K_STEPS || k < p.K ? k : 0));
      } else {
#pragma unroll
        for (int j = 0; j < 4; j++) d.a[t][j] = xr[t][k + j < p.K ? k + j : 0];
      }
    }
  };
  floatx4 tot[RT][4];
#pragma unroll
  for (int t = 0; t < RT; t++)
#pragma unroll
    for (int c = 0; c < 4; c++) tot[t][c] = floatx4{0.f, 0.f, 0.f, 0.f};
  auto compute = [&](int s, const Step &d) {
    floatx4 a[RT], b[4];
#pragma unroll
    for (int t = 0; t < RT; t++) a[t] = wide(d.a[t]);
#pragma unroll
    for (int j = 0; j < 4; j++) b[j] = wide(d.b[j]);
    if (KF != K_STEPS) {  // k past K count as zeros (their weights read as zeros)
#pragma unroll
      for (int j = 0; j < 4; j++)
#pragma unroll
        for (int t = 0; t < RT; t++) a[t][j] = s * FSTEP + 4 * kq + j < p.K ? a[t][j] : 0.f;
    }
#pragma unroll
    for (int c = 0; c < 4; c++)
#pragma unroll
      for (int t = 0; t < RT; t++) {
        floatx4 v = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int j = 0; j < 4; j++)
          v = __builtin_amdgcn_mfma_f32_16x16x4f32(a[t][j], b[j][c], v, 0, 0, 0);
        tot[t][c] = tot[t][c] + v;
      }
  };
  Step ring[FPD];
#pragma unroll
  for (int j = 0; j < FPD - 1; j++) load(s0 + j, ring[j]);
  for (int s = s0; s < s1; s += FPD) {
#pragma unroll
    for (int j = 0; j < FPD; j++) {
      load(s + j + FPD - 1, ring[(j + FPD - 1) % FPD]);
      __builtin_amdgcn_sched_barrier(0);  // the loads go out before this step's products
      if (j == 0 || s + j < s1) compute(s + j, ring[j]);
    }
  }
  // tot[t][c][q]: row 16t + 4kq + q, column col + c.
#pragma unroll
  for (int t = 0; t < RT; t++)
#pragma unroll
    for (int q = 0; q < 4; q++)
      red[wave][4 * t + q][lane] = floatx4{tot[t][0][q], tot[t][1][q], tot[t][2][q], tot[t][3][q]};
  __syncthreads();
  if (!col_ok) return;
  OT *out = (OT *)p.out + call * p.out_cs;
  for (int i = wave; i < 4 * RT; i += FWAVES) {
    const int r = 16 * (i >> 2) + 4 * kq + (i & 3);
    if (r >= rows) continue;
    floatx4 v[NS];
#pragma unroll
    for (int s = 0; s < NS; s++) {
      v[s] = red[s * KW][i][lane];
#pragma unroll
      for (int g = 1; g < KW; g++) v[s] = v[s] + red[s * KW + g][i][lane];
      const WT *b = (const WT *)(s ? p.b1 : p.b0);
      if (b) v[s] = v[s] + wide(load4(b + call * (s ? p.b1_cs : p.b0_cs) + (int64_t)e * p.N + col));
    }
    floatx4 u = v[0];
    if constexpr (MODE == MODE_UP) {
#pragma unroll
      for (int c = 0; c < 4; c++) u[c] = swiglu(v[0][c], v[1][c]);
    }
    store4(out + (int64_t)perm[r] * p.N + col, u);
  }
}

__global__ void k_idx_route(const float *__restrict__ idx, int M, float *__restrict__ route) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < M) {
    route[2 * i] = idx[i];
    route[2 * i + 1] = 1.0f;
  }
}

}  // namespace

int launch_idx_route(const float *idx, int M, float *route, hipStream_t s) {
  MOE_NONNULL(idx);
  MOE_NONNULL(route);
  hipLaunchKernelGGL(k_idx_route, dim3((M + 255) / 256), dim3(256), 0, s, idx, M, route);
  return 0;
}

// Rows per tile, from the rows an expert has on average (block of 640 × 640, E
// 128, top-4, µs, 16- and 32-row tiles: f32 150 tokens 143, 147, 300 tokens
// 156, 155, 500 tokens 192, 171; f16, whose tiles cost half the bytes, 500
// tokens 134, 142).
int float_tile_rows(int A, int max_active, moe_dtype w_dt) {
  return A / max_active <= (w_dt == MOE_F16 ? 16 : 6) ? 16 : 32;
}

template <int MODE, typename AT, typename WT, typename OT>
static void launch_float_tile(const FloatArgs &p, int rows, int max_active, int calls, hipStream_t s) {
  const int gx = (int)(((int64_t)p.N + FCOLS - 1) / FCOLS);
  const int64_t tiles = (int64_t)(p.db.A - max_active) / rows + max_active;
  // A grid holds fewer than 2^32 threads: larger outputs in several launches.
  const int64_t nblk = (tiles * gx + 7) / 8 * 8;
  constexpr int64_t GRID = 1 << 22;
  const dim3 block(FWAVES * WAVE);
  const bool vx = p.K % 4 == 0 && (uintptr_t)p.a % (4 * sizeof(AT)) == 0 && p.a_cs % 4 == 0;
  const int kf = !vx ? K_ANY : p.K % FSTEP ? K_QUADS : K_STEPS;
  // 16-row tiles that fill the CUs twice: no step ahead, the registers for
  // more wavefronts instead (77 tokens f32 133 → 123 µs a block, 150 tokens 143
  // → 129, f16 99 → 95); fewer blocks: one ahead (4 tokens 44 → 41).
  const bool full = tiles * gx >= 512;
#define FLT_KF(RT_, KF_)                                                                            \
  do {                                                                                              \
    if (RT_ == 1 && full)                                                                           \
      hipLaunchKernelGGL((k_float_tile<MODE, AT, WT, OT, RT_, KF_, 1>), grid, block, 0, s, p, gx, (int)b);  \
    else                                                                                            \
      hipLaunchKernelGGL((k_float_tile<MODE, AT, WT, OT, RT_, KF_, 2>), grid, block, 0, s, p, gx, (int)b);  \
  } while (0)
#define FLT_RT(RT_)                                \
  do {                                             \
    if (kf == K_STEPS) FLT_KF(RT_, K_STEPS);       \
    else if (kf == K_QUADS) FLT_KF(RT_, K_QUADS);  \
    else FLT_KF(RT_, K_ANY);                       \
  } while (0)
  for (int64_t b = 0; b < nblk; b += GRID) {
    const dim3 grid((unsigned)(nblk - b < GRID ? nblk - b : GRID), calls);
    if (p.N > F_MAX_N && rows == 16)
      hipLaunchKernelGGL((k_float_tile<MODE, AT, WT, OT, 1, K_WIDE, 2>), grid, block, 0, s, p, gx,
                         (int)b);
    else if (p.N > F_MAX_N)
      hipLaunchKernelGGL((k_float_tile<MODE, AT, WT, OT, 2, K_WIDE, 2>), grid, block, 0, s, p, gx,
                         (int)b);
    else if (rows == 16) FLT_RT(1);
    else FLT_RT(2);
  }
#undef FLT_RT
#undef FLT_KF
}

int launch_float_expert(const FloatArgs &p, int mode, moe_dtype a_dt, moe_dtype w_dt,
                        moe_dtype o_dt, int max_active, int calls, hipStream_t s) {
  MOE_NONNULL(p.a);
  MOE_NONNULL(p.w0);
  MOE_NONNULL(p.out);
  MOE_NONNULL(p.db.perm);
  MOE_NONNULL(p.db.active);
  MOE_NONNULL(p.db.meta);
  if (mode == MODE_UP) MOE_NONNULL(p.w1);
  const int rows = float_tile_rows(p.db.A, max_active, w_dt);
  if (((int64_t)p.db.A + max_active) * (((int64_t)p.N + FCOLS - 1) / FCOLS) > 0x7ffffff0)
    return moe_fail(MOE_INVALID_ARGUMENT, "float expert: too many rows");
#define FLT(M_, A_, W_, O_) launch_float_tile<M_, A_, W_, O_>(p, rows, max_active, calls, s)
  const bool af = a_dt == MOE_F16, wf = w_dt == MOE_F16, of = o_dt == MOE_F16;
  if (mode == MODE_UP) {
    // act is f32 (the layer keeps its intermediates in f32)
    if (af && wf) FLT(MODE_UP, _Float16, _Float16, float);
    else if (!af && !wf) FLT(MODE_UP, float, float, float);
    else return moe_fail(MOE_INVALID_ARGUMENT, "float expert: x and weights need one dtype");
  } else {
    if (wf) {
      if (af && of) FLT(MODE_DOWN, _Float16, _Float16, _Float16);
      else if (!af && !of) FLT(MODE_DOWN, float, _Float16, float);
      else if (!af && of) FLT(MODE_DOWN, float, _Float16, _Float16);
      else FLT(MODE_DOWN, _Float16, _Float16, float);
    } else {
      if (!af && !of) FLT(MODE_DOWN, float, float, float);
      else return moe_fail(MOE_INVALID_ARGUMENT, "float expert: f32 weights need f32 rows");
    }
  }
#undef FLT
  return 0;
}

// Dense Linear for the privacy filter's attention projections and head:
// y [T, N] = x [T, K] · W [K, N] + bias (+ addend), f32, W row-major.
//
// Reference: src/core/nn/layers.ts:166-263 (Linear: y = x·W + bias +
// addend, W stored [in, out]), src/core/graph/compose.ts:45-53. A quantized
// checkpoint weight is dequantized once at load (q · scale per group of
// inputs, the values the reference's kernel multiplies by), so float and
// quantized Linears share this kernel.
//
// One launch: a block is 16·RT rows × 16·CT columns, its KW wavefronts take a
// contiguous part of K each, and their sums meet in LDS, added in wavefront
// order, before the bias and the addend. The products are
// v_mfma_f32_16x16x4_f32 (f32 operands and sums). Per 16 k a lane loads four
// consecutive k of its row in each of the RT row tiles and CT consecutive
// columns of four rows of W: MFMA step j takes element j of the row (k =
// 4·(lane / 16) + j) and row j of W, column tile c the columns
// CT·(lane mod 16) + c, so operands go from memory to the matrix cores
// without LDS and a lane ends with CT consecutive outputs of a row. Loads run
// PD steps ahead; nothing but the last sums passes a barrier. Every 32 k the
// sums join the total and start from zero, so no chain of additions is
// longer than 32 or K / 32 terms (one chain over a wavefront's K: 2.1e-7 of
// the attention block's result instead of 1.5e-7).
//
// Bound by latency at a text's tens of rows, by the f32 matrix rate at a
// document's. Measured against K slices of 32 whose partial sums went
// through memory to a second kernel, 640 → 1152 and 896 → 640 together:
// 1500 rows 133 → 58 µs (66 TFLOP/s), 64 rows 24.3 → 15.0.
#include "moe_internal.h"

namespace {

typedef float floatx4 __attribute__((ext_vector_type(4)));

constexpr int WAVE = 64;
constexpr int LSTEP = 16;  // k per step

// A step's 16 weight rows get a buffer descriptor of their own (scalar
// arithmetic), so the lanes' offsets are loop constants and a row past K or a
// column past N reads zeros. (64-bit row addresses per lane cost as much VALU
// time as the products take.)
constexpr uint32_t L_OOB = 0x80000000u;
__device__ __forceinline__ __amdgpu_buffer_rsrc_t rows_rsrc(const float *base, int bytes) {
  return __builtin_amdgcn_make_buffer_rsrc((void *)base, 0, bytes, 0x00020000 /* raw, 32-bit */);
}

template <int CT> struct Cols {
  typedef float type __attribute__((ext_vector_type(CT)));
};
template <> struct Cols<1> {
  struct type {
    float v;
    __device__ __forceinline__ float &operator[](int) { return v; }
    __device__ __forceinline__ float operator[](int) const { return v; }
  };
};

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
template <int CT>
__device__ __forceinline__ typename Cols<CT>::type load_cols(__amdgpu_buffer_rsrc_t r, uint32_t off) {
  typedef typename Cols<CT>::type colv;
  if constexpr (CT == 4)
    return __builtin_bit_cast(colv, __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0));
  else if constexpr (CT == 2)
    return __builtin_bit_cast(colv, __builtin_amdgcn_raw_buffer_load_b64(r, off, 0, 0));
  else
    return __builtin_bit_cast(colv, __builtin_amdgcn_raw_buffer_load_b32(r, off, 0, 0));
}

// CT > 1 needs N a multiple of CT and the pointers other than x aligned to CT
// floats.
// K % 16 == 0, % 4 == 0 (x aligned), any; any with rows of W so wide that 16 of
// them pass the buffer offsets (64-bit addresses, CT = 1)
enum KForm { K_STEPS = 0, K_QUADS = 1, K_ANY = 2, K_WIDE = 3 };
constexpr int L_MAX_N = 1 << 24;
template <int RT, int CT, int KW, int KF>
__global__ __launch_bounds__(64 * KW) void k_linear(const float *__restrict__ x,
                                                    const float *__restrict__ w,
                                                    const float *__restrict__ bias,
                                                    const float *__restrict__ addend,
                                                    float *__restrict__ y, int T, int K, int N,
                                                    int ncb, int blk0) {
  typedef typename Cols<CT>::type colv;
  constexpr int PD = RT == 1 ? 4 : 2;  // steps loaded (this one and those ahead)
  __shared__ colv red[KW][RT * 4][WAVE];
  const int lane = threadIdx.x & (WAVE - 1);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
  const int blk = blk0 + (int)blockIdx.x;
  const int rb = blk / ncb, cb = blk - rb * ncb;
  const int row0 = rb * 16 * RT, col0 = cb * 16 * CT;
  const int m = lane & 15, kq = lane >> 4;
  const int steps = (K + LSTEP - 1) / LSTEP;
  const int per = (steps + KW - 1) / KW;
  const int s0 = wave * per, s1 = min(steps, s0 + per);
  // Rows past T and columns past N read valid ones; their sums are not stored.
  const float *xr[RT];
#pragma unroll
  for (int t = 0; t < RT; t++) xr[t] = x + (int64_t)min(row0 + 16 * t + m, T - 1) * K;
  const int col = col0 + CT * m;
  uint32_t woff[4];
#pragma unroll
  for (int j = 0; j < 4; j++)
    woff[j] = col < N ? ((uint32_t)(4 * kq + j) * (uint32_t)N + col) * 4u : L_OOB;

  struct Step {
    floatx4 a[RT];
    colv b[4];
  };
  // Addresses of x stay inside its rows: a step past the last reads that one
  // (not used), a k past K reads k = 0.
  auto load = [&](int s, Step &d) {
    s = min(s, steps - 1);
    const int k = s * LSTEP + 4 * kq;
#pragma unroll
    for (int t = 0; t < RT; t++) {
      if constexpr (KF == K_STEPS || KF == K_QUADS) {
        d.a[t] = *(const floatx4 *)(xr[t] + (KF == K_STEPS || k < K ? k : 0));
      } else {
#pragma unroll
        for (int j = 0; j < 4; j++) d.a[t][j] = xr[t][k + j < K ? k + j : 0];
      }
    }
    if constexpr (KF == K_WIDE) {
#pragma unroll
      for (int j = 0; j < 4; j++) {
        const bool ok = k + j < K && col < N;
        const float v = w[ok ? (int64_t)(k + j) * N + col : 0];
        d.b[j][0] = ok ? v : 0.f;
      }
    } else {
      const int left = KF == K_STEPS ? LSTEP : min(LSTEP, K - s * LSTEP);
      const __amdgpu_buffer_rsrc_t wr = rows_rsrc(w + (int64_t)s * LSTEP * N, left * N * 4);
#pragma unroll
      for (int j = 0; j < 4; j++) d.b[j] = load_cols<CT>(wr, woff[j]);
    }
  };
  floatx4 acc[RT][CT], tot[RT][CT];
#pragma unroll
  for (int t = 0; t < RT; t++)
#pragma unroll
    for (int c = 0; c < CT; c++) acc[t][c] = tot[t][c] = floatx4{0.f, 0.f, 0.f, 0.f};
  auto compute = [&](int s, Step &d) {
    if (KF != K_STEPS) {  // k past K count as zeros (their weights read as zeros)
#pragma unroll
      for (int j = 0; j < 4; j++)
#pragma unroll
        for (int t = 0; t < RT; t++) d.a[t][j] = s * LSTEP + 4 * kq + j < K ? d.a[t][j] : 0.f;
    }
#pragma unroll
    for (int j = 0; j < 4; j++)
#pragma unroll
      for (int c = 0; c < CT; c++)
#pragma unroll
        for (int t = 0; t < RT; t++)
          acc[t][c] = __builtin_amdgcn_mfma_f32_16x16x4f32(d.a[t][j], d.b[j][c], acc[t][c], 0, 0, 0);
  };
  auto fold = [&]() {
#pragma unroll
    for (int t = 0; t < RT; t++)
#pragma unroll
      for (int c = 0; c < CT; c++) {
        tot[t][c] = tot[t][c] + acc[t][c];
        acc[t][c] = floatx4{0.f, 0.f, 0.f, 0.f};
      }
  };
  Step ring[PD];
#pragma unroll
  for (int j = 0; j < PD - 1; j++) load(s0 + j, ring[j]);
  for (int s = s0; s < s1; s += PD) {
#pragma unroll
    for (int j = 0; j < PD; j++) {
      load(s + j + PD - 1, ring[(j + PD - 1) % PD]);
      __builtin_amdgcn_sched_barrier(0);  // the loads go out before this step's products
      if (j == 0 || s + j < s1) compute(s + j, ring[j]);
      if (j % 2 == 1) fold();
    }
  }
  // tot[t][c][q]: row 16t + 4kq + q, column col + c.
#pragma unroll
  for (int t = 0; t < RT; t++)
#pragma unroll
    for (int q = 0; q < 4; q++) {
      colv v;
#pragma unroll
      for (int c = 0; c < CT; c++) v[c] = tot[t][c][q];
      red[wave][4 * t + q][lane] = v;
    }
  __syncthreads();
  for (int i = wave; i < RT * 4; i += KW) {
    const int row = row0 + 16 * (i >> 2) + 4 * kq + (i & 3);
    if (row >= T || col >= N) continue;
    colv v = red[0][i][lane];
#pragma unroll
    for (int g = 1; g < KW; g++) {
      const colv u = red[g][i][lane];
#pragma unroll
      for (int c = 0; c < CT; c++) v[c] = v[c] + u[c];
    }
    const int64_t o = (int64_t)row * N + col;
    if (bias) {
      const colv u = *(const colv *)(bias + col);
#pragma unroll
      for (int c = 0; c < CT; c++) v[c] = v[c] + u[c];
    }
    if (addend) {
      const colv u = *(const colv *)(addend + o);
#pragma unroll
      for (int c = 0; c < CT; c++) v[c] = v[c] + u[c];
    }
    *(colv *)(y + o) = v;
  }
}

__global__ void k_copy(const float *__restrict__ from, float *__restrict__ to, size_t n) {
  const size_t stride = (size_t)gridDim.x * blockDim.x;
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) to[i] = from[i];
}

}  // namespace

int launch_copy(const float *from, float *to, size_t n, hipStream_t s) {
  const size_t blocks = (n + 255) / 256;
  hipLaunchKernelGGL(k_copy, dim3((unsigned)(blocks < 4096 ? blocks : 4096)), dim3(256), 0, s, from,
                     to, n);
  return 0;
}

int launch_linear(const float *x, const float *w, const float *bias, const float *addend, float *y,
                  int T, int K, int N, hipStream_t s) {
  MOE_NONNULL(x);
  MOE_NONNULL(w);
  MOE_NONNULL(y);
  auto aligned = [](const void *p, int bytes) { return (uintptr_t)p % bytes == 0; };
  const bool vx = K % 4 == 0 && aligned(x, 16);
  auto cols_ok = [&](int ct) {
    return N % ct == 0 && aligned(w, 4 * ct) && aligned(y, 4 * ct) && aligned(bias, 4 * ct) &&
           aligned(addend, 4 * ct);
  };
  auto blocks = [&](int rt, int ct) {
    return (((int64_t)T + 16 * rt - 1) / (16 * rt)) * (((int64_t)N + 16 * ct - 1) / (16 * ct));
  };
  // 32 × 64 outputs a block (four wavefronts over K) from 100 blocks on, else
  // 16 × 32 from 130, else 16 × 16 (eight wavefronts each): the attention
  // block, µs, at 1500 rows 180, 238, 266; 300 rows 77, 85, 89; 150 rows 66,
  // 63, 65; the network at 110 rows 894, 837, 858; at 32 rows 715, 661, 639.
  int rt = 1, ct = 1;
  const bool wide = N > L_MAX_N;
  if (!wide && vx && cols_ok(4) && blocks(2, 4) >= 100) rt = 2, ct = 4;
  else if (!wide && vx && cols_ok(2) && blocks(1, 2) >= 130) ct = 2;
  const int64_t n = blocks(rt, ct);
  if (n > 0x7fffffff) return moe_fail(MOE_INVALID_ARGUMENT, "linear: output too large");
  const int ncb = (int)(((int64_t)N + 16 * ct - 1) / (16 * ct));
  // A grid holds fewer than 2^32 threads: larger outputs in several launches.
  if (T > 0x7fffffc0) return moe_fail(MOE_INVALID_ARGUMENT, "linear: output too large");
  constexpr int64_t GRID = 1 << 22;
#define LIN_KF(RT_, CT_, KW_, KF_)                                                                \
  for (int64_t b = 0; b < n; b += GRID)                                                           \
  hipLaunchKernelGGL((k_linear<RT_, CT_, KW_, KF_>), dim3((unsigned)(n - b < GRID ? n - b : GRID)), \
                     dim3(64 * KW_), 0, s, x, w, bias, addend, y, T, K, N, ncb, (int)b)
#define LIN(RT_, CT_, KW_)                                   \
  do {                                                       \
    if (K % LSTEP == 0) LIN_KF(RT_, CT_, KW_, K_STEPS);      \
    else LIN_KF(RT_, CT_, KW_, K_QUADS);                     \
  } while (0)
  if (wide) LIN_KF(1, 1, 8, K_WIDE);
  else if (rt == 2) LIN(2, 4, 4);
  else if (ct == 2) LIN(1, 2, 8);
  else if (vx) LIN(1, 1, 8);
  else LIN_KF(1, 1, 8, K_ANY);
#undef LIN
#undef LIN_KF
  return 0;
}

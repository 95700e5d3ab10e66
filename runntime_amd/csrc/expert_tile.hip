// Expert products for a few dozen rows per expert, and for every int4 or
// group-scaled weight, on gfx950.
//
// Reference: src/core/kernels/matmul/moeQuantW.ts:122-175 (moeUp) and
// :188-237 (moeDown), src/core/kernels/activations.ts:120-133 (SwiGLU),
// src/core/kernels/quantCommon.ts:8-31 (quantW layout).
//
// k_expert_tile: one block = one row tile (16·RT rows of one expert) × four
// streams of 64 output columns (16 quantW units), one wavefront each; up
// pairs a glu and a lin stream. The weights go straight from memory into
// registers as in k_expert_skinny (whole 128-byte lines, nontemporal, SK
// load steps ahead), and each converted weight feeds RT row tiles, so an
// expert's weights are read and converted once for up to 64 rows. The
// block's A rows come through LDS KC columns at a time, double-buffered:
// the next piece is loaded into registers while this one is multiplied, so
// LDS holds 2·KC columns instead of whole rows and three blocks fit a CU.
//
// A in LDS, 16-byte fragments of 8 consecutive k per row:
//   f16 x                 one f16 plane, exact
//   f32 x, int8 weights   f16 hi + lo (~2^-22 of the value), as in the
//                         other int8 kernels
//   f32 x, int4 weights   three bf16 planes of 8 bits each: x exactly, over
//                         f32's whole range
// int4 weights are taken 64 k at a time (128 bytes of a unit): of the two
// load instructions' lines the lanes trade halves so that MFMA step h of the
// two has k 32h .. 32h + 31, a whole scale group when the group is 32.
//
// Group scales (GROUPED: g a multiple of 32, below K) travel in the ring
// with the weights they scale; every MFMA step's sums start from zero and
// join the total times their scale, so no load waits inside the loop.
//
// Bound by the weight stream while an expert has up to ~32 rows, by the
// int8 → f16 conversions and MFMAs above. Measured (2048 × 1408, E 64, 300
// tokens, top-8, f16 x): layer 611 → 168 µs against the skinny kernel (up 397,
// down 208), which takes 16 rows at a time and streams (and converts) the
// weights once for each.
// Ring of 4 load steps: 8 is no faster with plain scales and spills with
// group scales (56 tokens int4 g 32: 76 → 130 µs a layer).
#include "gemm_dev.h"

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

constexpr int TW = 4;    // wavefronts (streams) per block
constexpr int TPD = 4;   // load steps in the weight ring
constexpr uint32_t T_OOB = 0x80000000u;

struct TileArgs {
  const void *a;
  int64_t a_cs;
  int a_row_div;
  const uint32_t *w0, *w1;
  const float *s0, *s1, *b0, *b1;
  int64_t w0_cs, s0_cs, b0_cs, w1_cs, s1_cs, b1_cs;
  int K, N, g;
  float *out;
  int64_t out_cs;
  int sorted;   // act in dispatch order (up writes, down reads it there)
  int nsub;     // row tiles per M-tile of the dispatch
  int tile_m;   // rows of the dispatch's M-tiles
  int gx;       // column blocks
  DispatchBufs db;
};

__device__ __forceinline__ u32x4 t_load(__amdgpu_buffer_rsrc_t r, uint32_t off) {
  return __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 2 /* nt */));
}
__device__ __forceinline__ floatx4 t_loadf(__amdgpu_buffer_rsrc_t r, uint32_t off) {
  return __builtin_bit_cast(floatx4, __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0));
}
// Lane L of a 16-lane row receives the value of lane L ^ 8 (DPP row_ror:8).
__device__ __forceinline__ uint32_t t_swap8(uint32_t v) {
  return (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0x128, 0xf, 0xf, false);
}

// Eight int4 values of a column (k 0-3 in the low half of x, 4-7 in the high
// half) as f16, in the order 0 4 1 5 2 6 3 7: u = q + 8 under the exponent
// byte 0x64 is 1024 + u, minus 1032 is q.
__device__ __forceinline__ u32x4 i4x8_f16(uint32_t x) {
  const half2v bias = {(_Float16)1032.0f, (_Float16)1032.0f};
  x ^= 0x88888888u;
  u32x4 r;
#pragma unroll
  for (int j = 0; j < 4; j++)
    r[j] = __builtin_bit_cast(
        uint32_t,
        __builtin_bit_cast(half2v, ((x >> (4 * j)) & 0x000f000fu) | 0x64006400u) - bias);
  return r;
}
// The same as bf16 of q / 16 (v_cvt_off_f32_i4, exact; the scales carry the 16).
__device__ __forceinline__ u32x4 i4x8_bf16(uint32_t x) {
  u32x4 r;
#pragma unroll
  for (int j = 0; j < 4; j++) {
    const uint32_t lo = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_off_f32_i4(x >> (4 * j)));
    const uint32_t hi = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_off_f32_i4(x >> (4 * j + 16)));
    r[j] = __builtin_amdgcn_perm(hi, lo, 0x07060302u);
  }
  return r;
}

// How A is held: planes, and whether they are bf16.
template <typename AT, int BITS>
struct APlanes {
  static constexpr bool F32 = sizeof(AT) == 4;
  static constexpr bool BF = F32 && BITS == 4;
  static constexpr int N = !F32 ? 1 : BF ? 3 : 2;
};

// Columns of A per LDS piece: 64 keeps two buffers of 64 f32 rows near 36 KB
// (three blocks a CU); 16 f32 rows need 128 for one 8-value load per thread.
template <typename AT, int RT>
constexpr int tile_kc() { return sizeof(AT) == 4 && RT > 1 ? 64 : 128; }

// Wavefronts per SIMD the registers are kept to: what fits with at most a few
// registers spilled. 64-row tiles of f32 rows under int8: three (two more
// spilled values, but the block of d 640, E 128, top-4, I 640 at 1500 tokens
// was 1.5% faster at three than at two). 16-row tiles of three planes: three,
// since they spill at four (int4 layer of 64 tokens 62.8 us instead of 65).
template <typename AT, int BITS, bool GROUPED, int RT>
constexpr int tile_waves() {
  if (RT == 4) return BITS == 8 && !GROUPED && sizeof(AT) == 4 ? 3 : 2;
  return RT == 2 || APlanes<AT, BITS>::BF ? 3 : 4;
}

template <int MODE, typename AT, int BITS, bool GROUPED, int RT>
__global__ __launch_bounds__(64 * TW) __attribute__((
    amdgpu_waves_per_eu(tile_waves<AT, BITS, GROUPED, RT>())))
void k_expert_tile(TileArgs p) {
  typedef APlanes<AT, BITS> AP;
  constexpr int ROWS = 16 * RT;
  constexpr int KC = tile_kc<AT, RT>();
  constexpr int LK = BITS == 8 ? 32 : 64;   // k per load step
  constexpr int SUB = LK / 32;              // MFMA steps per load step
  constexpr int CS = KC / LK;               // load steps per piece
  static_assert(TPD % CS == 0, "whole pieces per ring turn");
  constexpr int RS = KC + 8;                // LDS row stride (halves): rows shift by 4 banks
  constexpr int PLANE = ROWS * RS;
  constexpr int BUF = AP::N * PLANE;
  constexpr int PER = ROWS * KC / 8 / (64 * TW);  // 8-value pieces per thread
  static_assert(PER >= 1, "at least one load per thread");
  constexpr int PPR = KC / 8;               // such pieces per row
  // No chain of additions runs over all of K: it would be longer, and its
  // error larger, than that of the K-split streams this kernel stands in for
  // (1536 x 1000, E 32, top-4, 500 tokens on few experts: 3.8e-7 of the
  // result there, 4.3e-7 in one chain, 2.2e-7 so). FOLD: the sums of a piece
  // start from zero and join the total. Larger tiles of several planes have
  // no registers for that: every MFMA step's planes start from zero and join
  // the total. It costs 64-row tiles some time (2048 x 1408, E 64, top-8, 300
  // tokens of f16: layer 150 -> 174 us for 5.2e-7 -> 3.1e-7; d 640 at 1500
  // tokens of f32: block 100 -> 112 us for 4.4e-7 -> 3.1e-7), 16-row tiles none.
  constexpr bool FOLD = !GROUPED && (RT == 1 || (AP::N == 1 && BITS == 8));
  extern __shared__ __align__(16) unsigned char smem[];
  uint16_t *abuf = (uint16_t *)smem;
  __shared__ int s_row[ROWS];  // rows of the dispatch's assignments

  const int lane = threadIdx.x & (WAVE - 1);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
  const int call = blockIdx.y;
  // This block's row tile and column block: the call's actual tiles in
  // order, in one contiguous range per XCD (blocks go round-robin over the 8
  // XCDs), so the row tiles of an expert meet its weights in one L2.
  // Its expert is the last active one whose first M-tile is not past it.
  const int32_t *meta = p.db.meta + call * p.db.meta_cs();
  const int4 *active = (const int4 *)(p.db.active + call * p.db.act_cs());
  const int E = p.db.E;
  int4 ad = active[min(lane, E - 1)];  // read with meta: one latency for both
  const int na = meta[META_ACTIVE];
  const int total = meta[META_TILES] * p.nsub * p.gx;
  const int per = (total + 7) / 8;
  const int slot = blockIdx.x >> 3;
  const int o = (blockIdx.x & 7) * per + slot;
  if (slot >= per || o >= total) return;
  const int y = o / p.gx, xb = o - y * p.gx;
  const int mt = y / p.nsub, sub = y - mt * p.nsub;
  int hit = __popcll(__ballot(lane < na && ad.w <= mt)) - 1;
  for (int b = WAVE; hit == WAVE - 1 && b < na; b += WAVE) {
    const int4 nx = active[min(b + lane, na - 1)];
    const int h = __popcll(__ballot(b + lane < na && nx.w <= mt)) - 1;
    if (h < 0) break;
    ad = nx;
    hit = h;
  }
  const int e = __builtin_amdgcn_readlane(ad.x, hit);
  const int r0 = (mt - __builtin_amdgcn_readlane(ad.w, hit)) * p.tile_m + sub * ROWS;
  const int rows = min(min(ROWS, p.tile_m - sub * ROWS), __builtin_amdgcn_readlane(ad.z, hit) - r0);
  if (rows <= 0) return;
  const int p0 = __builtin_amdgcn_readlane(ad.y, hit) + r0;

  const AT *abase = (const AT *)p.a + call * p.a_cs;
  float *out = p.out + call * p.out_cs;
  const int N4 = p.N / 4;
  const int arr = MODE == MODE_UP ? (wave & 1) : 0;
  const int cg = MODE == MODE_UP ? xb * (TW / 2) + (wave >> 1) : xb * TW + wave;
  const int unit = cg * 16 + (lane & 15);
  const bool uok = unit < N4;
  const int kq = lane >> 4, m = lane & 15;
  const bool odd = (lane & 8) != 0;
  const int lsteps = (p.K + LK - 1) / LK;
  const int kg = GROUPED ? p.K / p.g : 1;

  const uint32_t *w = arr ? p.w1 + call * p.w1_cs : p.w0 + call * p.w0_cs;
  const float *sc = (arr ? p.s1 + call * p.s1_cs : p.s0 + call * p.s0_cs) + (int64_t)e * kg * p.N;
  const float *bi = arr ? (p.b1 ? p.b1 + call * p.b1_cs : nullptr)
                        : (p.b0 ? p.b0 + call * p.b0_cs : nullptr);
  const int64_t slab = quantw_bytes(p.K, p.N, BITS);  // < 2^31 (expert_tile_eligible)
  const __amdgpu_buffer_rsrc_t wr = __builtin_amdgcn_make_buffer_rsrc(
      (void *)((const char *)w + e * slab), 0, (int)slab, BUF_DWORD3);
  const __amdgpu_buffer_rsrc_t sr = __builtin_amdgcn_make_buffer_rsrc(
      (void *)sc, 0, (int)((uint32_t)kg * (uint32_t)p.N * 4u), BUF_DWORD3);
  // Loaded units and 16-byte chunks (a chunk: one int8 tile, 4 k, or two int4
  // tiles, 8 k). Instruction 0 reads unit 16·cg + (lane & 7), instruction 1
  // unit 8 further; 8 lanes cover the 8 chunks of one unit's step. int8: chunk
  // lane >> 3 (^ 1 for instruction 1), so that a lane's own chunk is 2kq and
  // its partner (lane ^ 8) holds 2kq + 1. int4: chunk kq + 4·(lane bit 3) (^
  // 4), own chunk kq (MFMA step 0), the partner's kq + 4 (step 1).
  const int unit_chunks = p.K * BITS / 32;
  const int c0 = BITS == 8 ? (lane >> 3) : kq + (odd ? 4 : 0);
  const int c1 = BITS == 8 ? ((lane >> 3) ^ 1) : (c0 ^ 4);
  const int u0 = cg * 16 + (lane & 7), u1 = u0 + 8;
  const uint32_t wl0 = u0 < N4 ? (uint32_t)u0 * (uint32_t)unit_chunks * 16u : T_OOB;
  const uint32_t wl1 = u1 < N4 ? (uint32_t)u1 * (uint32_t)unit_chunks * 16u : T_OOB;
  const uint32_t sl = uok ? (uint32_t)unit * 16u : T_OOB;

  struct Step {
    u32x4 t0, t1;
    floatx4 s[GROUPED ? SUB : 1];
  };
  auto issue = [&](int s, Step &d) {
    const int ca = s * 8 + c0, cb = s * 8 + c1;
    d.t0 = t_load(wr, ca < unit_chunks ? wl0 + (uint32_t)ca * 16u : T_OOB);
    d.t1 = t_load(wr, cb < unit_chunks ? wl1 + (uint32_t)cb * 16u : T_OOB);
    if constexpr (GROUPED) {
#pragma unroll
      for (int h = 0; h < SUB; h++) {
        const int grp = (s * LK + 32 * h) / p.g;
        d.s[h] = t_loadf(sr, grp < kg ? sl + (uint32_t)grp * (uint32_t)p.N * 4u : T_OOB);
      }
    }
  };

  Step ring[TPD];
#pragma unroll
  for (int j = 0; j < TPD - 1; j++) issue(j, ring[j]);

  // The tile's rows: assignment (or sorted position) of each.
  if (threadIdx.x < ROWS) {
    const int r = threadIdx.x;
    s_row[r] = r < rows ? p.db.perm[call * p.db.perm_cs() + p0 + r] : -1;
  }
  __syncthreads();
  // This thread's pieces: 8 values at column ac of row ar[u]; rows past the
  // tile read row 0 and are zeroed.
  const int ac = (threadIdx.x % PPR) * 8;
  const AT *arow[PER];
  bool aok[PER];
#pragma unroll
  for (int u = 0; u < PER; u++) {
    const int r = threadIdx.x / PPR + u * (64 * TW / PPR);
    aok[u] = r < rows;
    const int rr = aok[u] ? r : 0;
    const int64_t src = (MODE == MODE_DOWN && p.sorted) ? p0 + rr : s_row[rr] / p.a_row_div;
    arow[u] = abase + src * p.K;
  }
  constexpr int AV = sizeof(AT) == 4 ? 2 : 1;  // 16-byte loads per piece
  u32x4 av[PER][AV];
  auto load_a = [&](int kc0) {
#pragma unroll
    for (int u = 0; u < PER; u++)
#pragma unroll
      for (int v = 0; v < AV; v++) {
        const int k = kc0 + ac + 4 * v;
        // past K: the row's start, zeroed in store_a
        av[u][v] = *(const u32x4 *)(arow[u] + (k < p.K ? k : 0));
      }
  };
  auto store_a = [&](int kc0, uint16_t *dst) {
#pragma unroll
    for (int u = 0; u < PER; u++) {
      const int r = threadIdx.x / PPR + u * (64 * TW / PPR);
      const int left = aok[u] ? p.K - kc0 - ac : 0;  // columns of the piece in K
      uint16_t *d = dst + r * RS + ac;
      // Slot i of the 16 bytes holds k = order(i): int4 fragments come out of
      // their words as 0 4 1 5 2 6 3 7.
      constexpr int O[8] = {0, BITS == 4 ? 4 : 1, BITS == 4 ? 1 : 2, BITS == 4 ? 5 : 3,
                            BITS == 4 ? 2 : 4, BITS == 4 ? 6 : 5, BITS == 4 ? 3 : 6, 7};
      if constexpr (!AP::F32) {
        typedef uint16_t u16x8 __attribute__((ext_vector_type(8)));
        const u16x8 x = __builtin_bit_cast(u16x8, left > 0 ? av[u][0] : u32x4{0, 0, 0, 0});
        u16x8 y;
#pragma unroll
        for (int i = 0; i < 8; i++) y[i] = x[O[i]];
        *(u16x8 *)d = y;
      } else {
        float x[8];
#pragma unroll
        for (int i = 0; i < 8; i++) {
          const uint32_t b = av[u][i >> 2][i & 3];
          x[i] = left > (i & 4) ? __uint_as_float(b) : 0.f;
        }
        if constexpr (AP::BF) {
          u32x4 h, md, lo;
#pragma unroll
          for (int q = 0; q < 4; q++) {
            uint32_t ph[2], pm[2], pl[2];
#pragma unroll
            for (int z = 0; z < 2; z++) {
              // Truncated to 8 bits three times: nothing is left over. An
              // infinity is its own first part.
              const float v = x[O[2 * q + z]];
              ph[z] = __builtin_bit_cast(uint32_t, v) & 0xffff0000u;
              const float hf = __builtin_bit_cast(float, ph[z]);
              const float r1 = hf == v ? 0.f : v - hf;
              pm[z] = __builtin_bit_cast(uint32_t, r1) & 0xffff0000u;
              pl[z] = __builtin_bit_cast(uint32_t, r1 - __builtin_bit_cast(float, pm[z]));
            }
            h[q] = __builtin_amdgcn_perm(ph[1], ph[0], 0x07060302u);
            md[q] = __builtin_amdgcn_perm(pm[1], pm[0], 0x07060302u);
            lo[q] = __builtin_amdgcn_perm(pl[1], pl[0], 0x07060302u);
          }
          *(u32x4 *)d = h;
          *(u32x4 *)(d + PLANE) = md;
          *(u32x4 *)(d + 2 * PLANE) = lo;
        } else {
          half8 h, lo;
#pragma unroll
          for (int i = 0; i < 8; i++) {
            const float v = x[O[i]];
            const _Float16 hv = (_Float16)v;
            h[i] = hv;
            lo[i] = (_Float16)(v - (float)hv);
          }
          *(half8 *)d = h;
          *(half8 *)(d + PLANE) = lo;
        }
      }
    }
  };

  floatx4 tot[RT][4], acc[FOLD ? RT : 1][4];
#pragma unroll
  for (int t = 0; t < RT; t++)
#pragma unroll
    for (int i = 0; i < 4; i++) {
      tot[t][i] = floatx4{0.f, 0.f, 0.f, 0.f};
      if (FOLD) acc[FOLD ? t : 0][i] = floatx4{0.f, 0.f, 0.f, 0.f};
    }
  auto fold = [&]() {
    if constexpr (FOLD) {
#pragma unroll
      for (int t = 0; t < RT; t++)
#pragma unroll
        for (int i = 0; i < 4; i++) {
          tot[t][i] += acc[FOLD ? t : 0][i];
          acc[FOLD ? t : 0][i] = floatx4{0.f, 0.f, 0.f, 0.f};
        }
    }
  };

  auto mfma = [&](u32x4 a, u32x4 b, floatx4 c) -> floatx4 {
    if constexpr (AP::BF)
      return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a),
                                                     __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
    else
      return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8, a),
                                                    __builtin_bit_cast(half8, b), c, 0, 0, 0);
  };
  // MFMA steps of load step d; its first column in the piece is `col`.
  auto compute = [&](const Step &d, const uint16_t *buf, int col) {
#pragma unroll
    for (int h = 0; h < SUB; h++) {
      u32x4 a[AP::N][RT];
#pragma unroll
      for (int q = 0; q < AP::N; q++)
#pragma unroll
        for (int t = 0; t < RT; t++)
          a[q][t] = *(const u32x4 *)(buf + q * PLANE + (16 * t + m) * RS + col + 32 * h + 8 * kq);
      // int4: this step's chunk of the lane's unit (own for h = 0, else the
      // partner's): dwords {c0 c1}, {c2 c3} of the two tiles.
      u32x4 ch;
      if constexpr (BITS == 4) {
#pragma unroll
        for (int i = 0; i < 4; i++)
          ch[i] = h == 0 ? (odd ? d.t1[i] : d.t0[i]) : t_swap8(odd ? d.t0[i] : d.t1[i]);
      }
#pragma unroll
      for (int i = 0; i < 4; i++) {
        u32x4 b;
        if constexpr (BITS == 8) {
          const uint32_t own = odd ? d.t1[i] : d.t0[i];
          const uint32_t other = t_swap8(odd ? d.t0[i] : d.t1[i]);
          b = __builtin_bit_cast(u32x4, cvt_i8x8(own, other));
        } else {
          const uint32_t x = __builtin_amdgcn_perm(ch[2 + (i >> 1)], ch[i >> 1],
                                                   (i & 1) ? 0x07060302u : 0x05040100u);
          b = AP::BF ? i4x8_bf16(x) : i4x8_f16(x);
        }
#pragma unroll
        for (int t = 0; t < RT; t++) {
          if constexpr (GROUPED) {
            floatx4 v = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int q = AP::N - 1; q >= 0; q--) v = mfma(a[q][t], b, v);
            tot[t][i] += v * d.s[h][i];
          } else {
            floatx4 one = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int q = AP::N - 1; q >= 0; q--) {
              floatx4 &c = FOLD ? acc[FOLD ? t : 0][i] : one;
              c = mfma(a[q][t], b, c);
            }
            if (!FOLD) tot[t][i] += one;
          }
        }
      }
    }
  };

  load_a(0);
  store_a(0, abuf);
  __syncthreads();
  int cur = 0;
  for (int s = 0; s < lsteps; s += TPD) {
#pragma unroll
    for (int j = 0; j < TPD; j++) {
      // Loads (and the barriers) are unconditional: past K they read nothing
      // or are not used. Only the products are guarded.
      if (j % CS == 0) load_a((s + j + CS) * LK);
      issue(s + j + TPD - 1, ring[(j + TPD - 1) % TPD]);
      if (j == 0 || s + j < lsteps) compute(ring[j], abuf + cur * BUF, (j % CS) * LK);
      if (j % CS == CS - 1) {
        fold();
        cur ^= 1;
        store_a((s + j + 1) * LK, abuf + cur * BUF);
        __syncthreads();
      }
    }
  }

  // Scales (one per column) and biases, then the SwiGLU (up: the lin
  // wavefront hands its sums over in LDS) and the rows.
  const float unscale = AP::BF ? 16.f : 1.f;
  floatx4 s1 = floatx4{unscale, unscale, unscale, unscale};
  if (!GROUPED) s1 = s1 * t_loadf(sr, sl);
  const floatx4 bias = (bi && uok) ? *(const floatx4 *)(bi + (int64_t)e * p.N + 4 * unit)
                                   : floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int t = 0; t < RT; t++)
#pragma unroll
    for (int i = 0; i < 4; i++) tot[t][i] = tot[t][i] * s1[i] + bias[i];
  floatx4 *park = (floatx4 *)smem + (wave >> 1) * RT * 4 * WAVE;
  if constexpr (MODE == MODE_UP) {
    __syncthreads();  // every wavefront is done with the A pieces
    if (arr == 1) {
#pragma unroll
      for (int t = 0; t < RT; t++)
#pragma unroll
        for (int i = 0; i < 4; i++) park[(t * 4 + i) * WAVE + lane] = tot[t][i];
    }
    __syncthreads();
    if (arr == 1) return;
  }
  if (!uok) return;
#pragma unroll
  for (int t = 0; t < RT; t++)
#pragma unroll
    for (int q = 0; q < 4; q++) {
      const int r = 16 * t + 4 * kq + q;
      if (r >= rows) continue;
      const int64_t orow = (MODE == MODE_UP && p.sorted) ? p0 + r : s_row[r];
      floatx4 v;
#pragma unroll
      for (int i = 0; i < 4; i++)
        v[i] = MODE == MODE_UP ? swiglu(tot[t][i][q], park[(t * 4 + i) * WAVE + lane][q])
                               : tot[t][i][q];
      *(floatx4 *)(out + orow * p.N + 4 * unit) = v;
    }
}

template <int MODE, typename AT, int BITS, bool GROUPED, int RT>
int launch_rt(const TileArgs &p, int blocks, int calls, hipStream_t s) {
  typedef APlanes<AT, BITS> AP;
  constexpr int KC = tile_kc<AT, RT>();
  constexpr size_t abytes = (size_t)2 * AP::N * 16 * RT * (KC + 8) * 2;
  constexpr size_t park = MODE == MODE_UP ? (size_t)(TW / 2) * RT * 4 * WAVE * 16 : 0;
  constexpr size_t lds = abytes > park ? abytes : park;
  static_assert(lds <= 64 * 1024, "within the default dynamic LDS");
  hipLaunchKernelGGL((k_expert_tile<MODE, AT, BITS, GROUPED, RT>), dim3(blocks, calls), dim3(64 * TW),
                     lds, s, p);
  return 0;
}

template <int MODE, typename AT, int BITS, bool GROUPED>
int launch_g(const TileArgs &p, int rows, int blocks, int calls, hipStream_t s) {
  if (rows == 16) return launch_rt<MODE, AT, BITS, GROUPED, 1>(p, blocks, calls, s);
  if (rows == 32) return launch_rt<MODE, AT, BITS, GROUPED, 2>(p, blocks, calls, s);
  return launch_rt<MODE, AT, BITS, GROUPED, 4>(p, blocks, calls, s);
}

template <int MODE, typename AT>
int launch_bits(const TileArgs &p, int bits, bool grouped, int rows, int blocks, int calls,
                hipStream_t s) {
  if (bits == 8)
    return grouped ? launch_g<MODE, AT, 8, true>(p, rows, blocks, calls, s)
                   : launch_g<MODE, AT, 8, false>(p, rows, blocks, calls, s);
  return grouped ? launch_g<MODE, AT, 4, true>(p, rows, blocks, calls, s)
                 : launch_g<MODE, AT, 4, false>(p, rows, blocks, calls, s);
}

}  // namespace

bool expert_tile_eligible(const ExpertArgs &ea) {
  // 16-byte loads of A stay inside its rows: K in whole loads. Scale groups
  // fill whole MFMA steps; int4 tiles come in pairs of 8 k.
  const bool kok = ea.g != ea.K ? ea.g % 32 == 0
                   : ea.bits == 4 || ea.a_dtype == MOE_F16 ? ea.K % 8 == 0 : ea.K % 4 == 0;
  return kok && (uintptr_t)ea.a % 16 == 0 && ea.a_cs * (ea.a_dtype == MOE_F16 ? 2 : 4) % 16 == 0 &&
         (ea.mode == MODE_UP || ea.a_dtype == MOE_F32) &&
         quantw_bytes(ea.K, ea.N, ea.bits) < (1ll << 31) &&
         (int64_t)(ea.K / ea.g) * ea.N * 4 < (1ll << 31);
}

// Rows per tile for these arguments, 0 if another kernel takes them. Where
// the lines lie (whole layer, d × I, E experts, top-k, µs on one MI355X):
//   int4, group scales: always here. Before, one VALU thread per output
//     column: 56 tokens of 640 × 640, E 128, top-4, int4 g 32: 364 → 76;
//     1500 tokens: 7030 → 146. int8 g 32 on the skinny kernel: 102 → 74.
//   int8, one scale per column: one row per expert and few wavefronts stay on
//     the skinny kernel, which splits K over wavefronts (one token: 33 there,
//     36 here; 2048 × 1408 two tokens 57, 60), from three rows an expert or
//     1000 wavefronts on it is this one (640 × 640 32 tokens 60 → 54;
//     2048 × 1408 f16 64 tokens 232 → 121, 300 tokens 611 → 168).
//   Row tile: as the rows an expert has on average, with room for their
//     spread (2048 × 1408, E 64, f16 x, 10 rows each: 121 with 16-row tiles, 116
//     with 32; 12: 124, 117; 24: 201, 143, 158 with 64; 48: 316, 234, 186),
//     halved while the launch has under two blocks a CU (512 × 1024, E 8, 48
//     rows each: 37, 41, 57).
int expert_tile_rows(const ExpertArgs &ea) {
  if (!expert_tile_eligible(ea) || expert_uses_gemm(ea)) return 0;
  const int max_active = ea.E < ea.A ? ea.E : ea.A;
  const int avg = ea.A / max_active;
  const int64_t waves = (int64_t)ea.calls * max_active * ((ea.N + 63) / 64 + (ea.K + 63) / 64);
  if (ea.bits == 8 && ea.g == ea.K && (ea.A == ea.k || (avg < 3 && waves < 1000))) return 0;
  const int ncg = (ea.N / 4 + 15) / 16;
  int rows = avg <= 10 ? 16 : avg <= 24 ? 32 : 64;
  auto blocks = [&](int r) {
    return (int64_t)ea.calls * ((ea.A - max_active) / r + max_active) * ((ncg + 1) / 2);
  };
  while (rows > 16 && blocks(rows) < 512) rows /= 2;
  return rows;
}

int launch_expert_tile(const ExpertArgs &ea, const DispatchBufs &db, hipStream_t s) {
  const int rows = ea.tile_rows;
  TileArgs p;
  p.a = ea.a;
  p.a_cs = ea.a_cs;
  p.a_row_div = ea.a_row_div;
  p.w0 = ea.w0.w;
  p.w1 = ea.w1.w;
  p.s0 = ea.w0.scales;
  p.s1 = ea.w1.scales;
  p.b0 = ea.w0.bias;
  p.b1 = ea.w1.bias;
  p.w0_cs = ea.w0_cs;
  p.s0_cs = ea.s0_cs;
  p.b0_cs = ea.b0_cs;
  p.w1_cs = ea.w1_cs;
  p.s1_cs = ea.s1_cs;
  p.b1_cs = ea.b1_cs;
  p.K = ea.K;
  p.N = ea.N;
  p.g = ea.g;
  p.out = ea.out;
  p.out_cs = ea.out_cs;
  p.sorted = ea.dispatch_order;
  p.tile_m = ea.tile_m;
  p.nsub = ea.tile_m / rows;
  p.db = db;
  const int ncg = (ea.N / 4 + 15) / 16;
  p.gx = ea.mode == MODE_UP ? (ncg + TW / 2 - 1) / (TW / 2) : (ncg + TW - 1) / TW;
  // Each active expert adds at most one partial M-tile.
  const int max_active = ea.E < ea.A ? ea.E : ea.A;
  const int64_t tiles = ((int64_t)(ea.A - max_active) / ea.tile_m + max_active) * p.nsub;
  const int64_t blocks = (tiles * p.gx + 7) / 8 * 8;
  if (ea.tile_m % rows || blocks > 0x7fffffff)
    return moe_fail(MOE_EXECUTION_FAILED, "expert tile: bad launch shape");
  if (ea.mode == MODE_UP) {
    if (ea.a_dtype == MOE_F16)
      return launch_bits<MODE_UP, _Float16>(p, ea.bits, ea.g != ea.K, rows, (int)blocks, ea.calls, s);
    return launch_bits<MODE_UP, float>(p, ea.bits, ea.g != ea.K, rows, (int)blocks, ea.calls, s);
  }
  if (ea.a_dtype != MOE_F32)
    return moe_fail(MOE_EXECUTION_FAILED, "expert tile: down takes f32 act");
  return launch_bits<MODE_DOWN, float>(p, ea.bits, ea.g != ea.K, rows, (int)blocks, ea.calls, s);
}

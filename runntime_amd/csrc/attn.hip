// Attention ops of the privacy-filter block for gfx950: the rotary
// embedding and banded GQA attention with sinks.
//
// Reference: src/core/graph/ops/attention.ts:28-145 (sdpa: band mask
// qPos − windowLeft ≤ j ≤ qPos + windowRight, qPos = qPosOffset + i, GQA,
// sinks, segments, key bias), :146-214 (sdpaPacked: q, k, v as column
// blocks of one tensor), :220-262 (rope); kernels src/core/kernels/
// attention/rope.ts:14-68 and attn.ts; the semantics pinned by the
// reference's f64 check test/core/kernels/attention/checkSdpa.ts:55-103:
// q and k arrive pre-scaled, a sink adds exp(sink · ln 2) to the softmax
// denominator alone, a row that sees no key (and has no sink) is 0.
//
// sdpa: one block of 8 wavefronts per (group of query rows, kv head). The
// block's items are (row, query head of this kv head), at most 8 per
// wavefront; the keys its rows can see are staged 64 at a time into LDS as
// f32 (K and V rows padded to a 16-byte bank shift). Per chunk a wavefront
// holds 64 keys' K rows in registers (lane = key) to score each of its
// items, updates the item's online softmax (running max m, sum l), and
// accumulates P·V with lane = output column, the weights read from the
// scoring lanes with readlane. Sums are f32; exp is expf.
#include "moe_internal.h"

#include <math.h>

#include <algorithm>
#include <initializer_list>
#include <type_traits>

namespace {

constexpr int WAVE = 64;
constexpr int AW = 8;        // wavefronts per block
constexpr int AI = 8;        // items per wavefront
constexpr int AKC = 64;      // keys per chunk
constexpr float LN2 = 0.69314718055994530942f;

__device__ __forceinline__ float ld(const float *p, int64_t i) { return p[i]; }
__device__ __forceinline__ float ld(const _Float16 *p, int64_t i) { return (float)p[i]; }
__device__ __forceinline__ void st(float *p, int64_t i, float v) { p[i] = v; }
__device__ __forceinline__ void st(_Float16 *p, int64_t i, float v) { p[i] = (_Float16)v; }

// Element x of a head row after rope (rope.ts:55-66): pair (x0, x1) =
// (x & ~1, x | 1), out[2p] = x0·c − x1·s, out[2p+1] = x1·c + x0·s; c and s
// are the pair-duplicated table entries of the element's row.
template <typename T>
__device__ __forceinline__ float roped(const T *p, int64_t i, int x, float c, float s) {
  const int64_t pair = i - (x & 1);
  const float x0 = ld(p, pair), x1 = ld(p, pair + 1);
  return (x & 1) ? x1 * c + x0 * s : x0 * c - x1 * s;
}

__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
  for (int m = 1; m < WAVE; m <<= 1) v = fmaxf(v, __shfl_xor(v, m));
  return v;
}
__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
  for (int m = 1; m < WAVE; m <<= 1) v += __shfl_xor(v, m);
  return v;
}
__device__ __forceinline__ float lane_f(float v, int l) {
  return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), l));
}

// rope.ts:14-68: one thread per (row, pair) of the output window.
template <typename T>
__global__ void k_rope(const T *__restrict__ x, const float *__restrict__ cs,
                       const float *__restrict__ sn, T *__restrict__ out, int rows, int cols,
                       int hd, int src_start, int width) {
  const int64_t pairs = width / 2;
  const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= (int64_t)rows * pairs) return;
  const int64_t row = idx / pairs;
  const int col0 = (int)(idx - row * pairs) * 2;
  const int dcol = col0 % hd;
  const float c = cs[row * hd + dcol], s = sn[row * hd + dcol];
  const int64_t src = row * cols + src_start + col0;
  const float x0 = ld(x, src), x1 = ld(x, src + 1);
  st(out, row * width + col0, x0 * c - x1 * s);
  st(out, row * width + col0 + 1, x1 * c + x0 * s);
}

// NS 64-column slabs of the head (head_dim ≤ 64·NS).
template <typename T, int NS>
__global__ __launch_bounds__(AW *WAVE) void k_sdpa(AttnArgs a) {
  constexpr int HP = 64 * NS;   // padded head width
  constexpr int KST = HP + 4;   // LDS row stride of K and V (floats)
  extern __shared__ __align__(16) float smem[];
  float *qs = smem;                    // [AW·AI][HP]
  float *ks = qs + AW * AI * HP;       // [AKC][KST]
  float *vs = ks + AKC * KST;          // [AKC][KST]

  const int lane = threadIdx.x & (WAVE - 1);
  const int wave = threadIdx.x / WAVE;
  const int G = a.q_heads / a.kv_heads;
  const int R = a.rows_per_block;
  const int row0 = blockIdx.x * R;
  const int kvh = blockIdx.y;
  const int hd = a.head_dim;
  const T *q = (const T *)a.q;
  const T *k = (const T *)a.k;
  const T *v = (const T *)a.v;
  T *out = (T *)a.out;

  // Items: it = wave + AW·i → row it / G, head kvh·G + it % G.
  const int nitems = min(R, a.q_len - row0) * G;
  // Staging (q here, K and V per chunk below): 8 elements per thread at a
  // time, their loads issued before the LDS stores, from indices clamped
  // into the tensors (values past them zeroed), so no load sits under a
  // branch; rope or not is one uniform choice around the whole loop. (A
  // load and store per strided iteration waited out each load in turn.)
  constexpr int NT = AW * WAVE;    // threads per block
  constexpr int PER = AKC * HP / NT;  // = AW·AI·HP / NT: elements per thread
  static_assert(AKC == AW * AI && PER % 8 == 0, "staging shape");
  auto stage_q = [&](auto rope) {
#pragma unroll
    for (int b0 = 0; b0 < PER; b0 += 8) {
      float qv[8];
#pragma unroll
      for (int u = 0; u < 8; u++) {
        const int e = threadIdx.x + NT * (b0 + u), it = e / HP, x = e % HP;
        const int itc = min(it, nitems - 1), xc = min(x, hd - 1);
        const int r = row0 + itc / G, h = kvh * G + itc % G;
        const int64_t qi = (int64_t)r * a.q_rs + (int64_t)h * hd + xc;
        float val;
        if constexpr (decltype(rope)::value)
          val = roped(q, qi, xc, a.rope_cos[(int64_t)r * hd + xc], a.rope_sin[(int64_t)r * hd + xc]);
        else
          val = ld(q, qi);
        qv[u] = (it < nitems && x < hd) ? val : 0.f;
      }
#pragma unroll
      for (int u = 0; u < 8; u++) qs[threadIdx.x + NT * (b0 + u)] = qv[u];
    }
  };
  if (a.rope_cos) stage_q(std::true_type{});
  else stage_q(std::false_type{});

  // The rows' key ranges.
  auto range = [&](int r, int &lo, int &hi) {
    const long long qpos = (long long)a.q_pos_offset + r;
    long long l = a.window_left < 0 ? 0 : qpos - a.window_left;
    long long hgh = a.window_right < 0 ? (long long)a.kv_len - 1 : qpos + a.window_right;
    if (l < 0) l = 0;
    if (hgh > a.kv_len - 1) hgh = a.kv_len - 1;
    if (a.segs) {
      const long long s0 = (long long)a.segs[2 * r], s1 = (long long)a.segs[2 * r + 1] - 1;
      if (s0 > l) l = s0;
      if (s1 < hgh) hgh = s1;
    }
    lo = (int)l;
    hi = (int)(hgh < l - 1 ? l - 1 : hgh);  // empty: hi < lo
  };
  int lo_i[AI], hi_i[AI];
  bool ok_i[AI];
  float m_i[AI], l_i[AI], acc[AI][NS];
#pragma unroll
  for (int i = 0; i < AI; i++) {
    const int it = wave + AW * i;
    ok_i[i] = it < nitems;
    lo_i[i] = 0;
    hi_i[i] = -1;
    if (ok_i[i]) range(row0 + it / G, lo_i[i], hi_i[i]);
    m_i[i] = -INFINITY;
    l_i[i] = 0.f;
#pragma unroll
    for (int sl = 0; sl < NS; sl++) acc[i][sl] = 0.f;
  }
  // The block's key span: the union of its rows' ranges.
  int blo = 0x7fffffff, bhi = -1;
  for (int r = row0; r < min(a.q_len, row0 + R); r++) {
    int l, h;
    range(r, l, h);
    if (h >= l) {
      blo = min(blo, l);
      bhi = max(bhi, h);
    }
  }

  for (int c0 = blo; c0 <= bhi; c0 += AKC) {
    __syncthreads();  // the previous chunk's reads are done (and qs is written)
    auto stage_kv = [&](auto rope) {
#pragma unroll
      for (int b0 = 0; b0 < PER; b0 += 8) {
        float kv[8], vv[8];
#pragma unroll
        for (int u = 0; u < 8; u++) {
          const int e = threadIdx.x + NT * (b0 + u), j = e / HP, x = e % HP;
          const int key = c0 + j;
          const int kc = min(key, bhi), xc = min(x, hd - 1);  // c0 ≤ kc ≤ bhi < kv_len
          const int64_t ki = (int64_t)kc * a.k_rs + (int64_t)kvh * hd + xc;
          float kval;
          if constexpr (decltype(rope)::value)
            kval = roped(k, ki, xc, a.rope_cos[(int64_t)kc * hd + xc],
                         a.rope_sin[(int64_t)kc * hd + xc]);
          else
            kval = ld(k, ki);
          const float vval = ld(v, (int64_t)kc * a.v_rs + (int64_t)kvh * hd + xc);
          const bool in = key <= bhi && x < hd;
          kv[u] = in ? kval : 0.f;
          vv[u] = in ? vval : 0.f;
        }
#pragma unroll
        for (int u = 0; u < 8; u++) {
          const int e = threadIdx.x + NT * (b0 + u), j = e / HP, x = e % HP;
          ks[j * KST + x] = kv[u];
          vs[j * KST + x] = vv[u];
        }
      }
    };
    if (a.rope_cos) stage_kv(std::true_type{});
    else stage_kv(std::false_type{});
    __syncthreads();
    const int key = c0 + lane;
    float s[AI];
#pragma unroll
    for (int i = 0; i < AI; i++) s[i] = 0.f;
    bool live[AI];
#pragma unroll
    for (int i = 0; i < AI; i++) live[i] = ok_i[i] && lo_i[i] <= c0 + AKC - 1 && hi_i[i] >= c0;
    // Scores: lane = key, the key's K row in registers, q broadcast from LDS.
#pragma unroll
    for (int sl = 0; sl < NS; sl++) {
      float kr[64];
#pragma unroll
      for (int x = 0; x < 64; x += 4) {
        const float4 t = *(const float4 *)&ks[lane * KST + sl * 64 + x];
        kr[x] = t.x;
        kr[x + 1] = t.y;
        kr[x + 2] = t.z;
        kr[x + 3] = t.w;
      }
#pragma unroll
      for (int i = 0; i < AI; i++) {
        if (!live[i]) continue;
        const float *qr = qs + (wave + AW * i) * HP + sl * 64;
        // Two chains (even and odd columns) halve the dependent FMA latency.
        float d0 = 0.f, d1 = 0.f;
#pragma unroll
        for (int x = 0; x < 64; x += 4) {
          const float4 t = *(const float4 *)&qr[x];
          d0 = fmaf(t.x, kr[x], d0);
          d1 = fmaf(t.y, kr[x + 1], d1);
          d0 = fmaf(t.z, kr[x + 2], d0);
          d1 = fmaf(t.w, kr[x + 3], d1);
        }
        s[i] += d0 + d1;
      }
    }
    // Online softmax per item.
    float p[AI];
#pragma unroll
    for (int i = 0; i < AI; i++) {
      p[i] = 0.f;
      if (!live[i]) continue;
      const bool vis = key >= lo_i[i] && key <= hi_i[i];
      float sc = s[i];
      if (a.has_kb && key >= a.kb_start && key < a.kb_end) sc += a.kb_value;
      sc = vis ? sc : -INFINITY;
      const float mc = wave_max(sc);
      const float mn = fmaxf(m_i[i], mc);
      if (mn == -INFINITY) continue;
      const float scale = m_i[i] == -INFINITY ? 0.f : expf(m_i[i] - mn);
      p[i] = vis ? expf(sc - mn) : 0.f;
      l_i[i] = l_i[i] * scale + wave_sum(p[i]);
#pragma unroll
      for (int sl = 0; sl < NS; sl++) acc[i][sl] *= scale;
      m_i[i] = mn;
    }
    // P·V: lane = output column, V column in registers.
#pragma unroll
    for (int sl = 0; sl < NS; sl++) {
      float vr[AKC];
#pragma unroll
      for (int j = 0; j < AKC; j++) vr[j] = vs[j * KST + sl * 64 + lane];
#pragma unroll
      for (int i = 0; i < AI; i++) {
        if (!live[i]) continue;
        float o0 = 0.f, o1 = 0.f;
#pragma unroll
        for (int j = 0; j < AKC; j += 2) {
          o0 = fmaf(lane_f(p[i], j), vr[j], o0);
          o1 = fmaf(lane_f(p[i], j + 1), vr[j + 1], o1);
        }
        acc[i][sl] += o0 + o1;
      }
    }
  }

  // Sinks join the denominator; store.
#pragma unroll
  for (int i = 0; i < AI; i++) {
    if (!ok_i[i]) continue;
    const int it = wave + AW * i;
    const int r = row0 + it / G, h = kvh * G + it % G;
    const float sg = a.sinks ? a.sinks[h] * LN2 : -INFINITY;
    const float mf = fmaxf(m_i[i], sg);
    float scale = 0.f, inv = 0.f;
    if (mf != -INFINITY) {
      scale = m_i[i] == -INFINITY ? 0.f : expf(m_i[i] - mf);
      const float l = l_i[i] * scale + (a.sinks ? expf(sg - mf) : 0.f);
      inv = 1.0f / l;
    }
#pragma unroll
    for (int sl = 0; sl < NS; sl++) {
      const int x = sl * 64 + lane;
      if (x < hd) st(out, (int64_t)r * a.o_rs + (int64_t)h * hd + x, acc[i][sl] * scale * inv);
    }
  }
}

// ------------------------------------------------ on the f32 matrix cores
//
// k_sdpa_mfma (head_dim 64 or 128): a wavefront takes 16 query rows of one
// head and walks its keys 16·NT at a time with v_mfma_f32_16x16x4_f32 (f32
// operands and sums):
//   Sᵀ = K·Qᵀ  keys × rows: lane (r = lane mod 16, g = lane / 16) gets row r's
//              scores of keys 4g .. 4g + 3 of each 16,
//   Oᵀ = Vᵀ·Pᵀ head columns × rows: its B operand is exactly those values, so P
//              never leaves the lane's registers.
// A lane keeps one row's running max and sum (its four lanes hold equal
// copies; two exchanges across them per step). Operands come from memory in
// 16-byte loads, four consecutive head columns a lane: step (s, j) of Sᵀ uses
// element j of columns 16s + 4g .. + 3 of K and Q; step j of Oᵀ key 4g + j, its
// column tile c of slab b the columns 64b + 4·(lane mod 16) + c. Nothing is
// staged in LDS; the wavefronts of a block (HW heads of one kv head) walk the
// same keys together, so K, V and the rope tables come out of L1.
// KS > 1 splits the keys of a head over KS wavefronts, whose sums meet in LDS
// in order (short sequences, few heads).
// Bound by latency and L1 (each wavefront reads K, V and the rope tables of
// its keys, 32 KB a step). Against k_sdpa below (f32 VALU, K and V through
// LDS), 14 heads over 2 kv heads of 64, rope, window ±128: 64 rows 9.8 → 7.4
// µs, 1500 rows 123 → 50 (27 TFLOP/s), 4096 rows 308 → 108.
template <typename T> struct Ld4;
template <> struct Ld4<float> {
  static __device__ __forceinline__ float4 at(const float *p) { return *(const float4 *)p; }
};
template <> struct Ld4<_Float16> {
  static __device__ __forceinline__ float4 at(const _Float16 *p) {
    typedef _Float16 h4 __attribute__((ext_vector_type(4)));
    const h4 v = *(const h4 *)p;
    return make_float4((float)v[0], (float)v[1], (float)v[2], (float)v[3]);
  }
};
typedef float floatx4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ void st4(float *p, float x, float y, float z, float w) {
  *(float4 *)p = make_float4(x, y, z, w);
}
__device__ __forceinline__ void st4(_Float16 *p, float x, float y, float z, float w) {
  typedef _Float16 h4 __attribute__((ext_vector_type(4)));
  *(h4 *)p = h4{(_Float16)x, (_Float16)y, (_Float16)z, (_Float16)w};
}

// Four head columns after rope: two interleaved pairs (the expression of
// `roped`).
__device__ __forceinline__ floatx4 rope4(float4 x, float4 c, float4 s) {
  return floatx4{x.x * c.x - x.y * s.x, x.y * c.y + x.x * s.y, x.z * c.z - x.w * s.z,
                 x.w * c.w + x.z * s.w};
}

// What a wavefront of k_sdpa_mfma leaves for its keys.
template <int NB> struct SdpaSums {
  float mx, sum;
  floatx4 acc[NB][4];
};

// The V operand of P·V is shared by the tile's rows, and 0 times an infinity
// or a NaN of a key that a row does not see is NaN. Such a NaN stays in the sums,
// so k_sdpa_mfma's loop needs no test: a wavefront that ends with one walks its
// keys again here, P·V for one row after the other with the V it does not see
// zeroed. Nothing is kept for it: it reads the kernel's arguments again and loads
// where it multiplies, so that the loop keeps its registers and its schedule.
// (Written with the loop's own parts it cost every call 3 to 10%, 77 rows 9.0 →
// 9.8 µs; so 64 rows 6.6, 6.6; 300 rows 18.3, 18.4; 4096 rows 105, 105.)
template <typename T, int NB, int NT, bool ROPE>
__device__ __forceinline__ SdpaSums<NB> sdpa_by_rows(int h, int lo, int hi, int blo, int bhi,
                                                     int c_first, int c_last) {
  constexpr int HD = 64 * NB, NS = HD / 16, KC = 16 * NT;
  // AttnArgs is k_sdpa_mfma's first argument.
  typedef const __attribute__((address_space(4))) AttnArgs *KernArgs;
  uint64_t kp0 = (uint64_t)__builtin_amdgcn_kernarg_segment_ptr();
  int lane = threadIdx.x & (WAVE - 1);
  asm("" : "+s"(kp0), "+v"(lane));
  const KernArgs a = (KernArgs)kp0;
  const int row0 = blockIdx.x * 16, kvh = h / (a->q_heads / a->kv_heads);
  const int m = lane & 15, g = lane >> 4;
  const int row = min(row0 + m, a->q_len - 1);
  const T *qp = (const T *)a->q + (int64_t)row * a->q_rs + (int64_t)h * HD;
  const T *kp = (const T *)a->k + (int64_t)kvh * HD;
  const T *vp = (const T *)a->v + (int64_t)kvh * HD;
  auto roped = [&](const T *p, int64_t r, int x) {
    const float4 v = Ld4<T>::at(p + x);
    if constexpr (ROPE)
      return rope4(v, *(const float4 *)(a->rope_cos + r * HD + x),
                   *(const float4 *)(a->rope_sin + r * HD + x));
    else
      return floatx4{v.x, v.y, v.z, v.w};
  };
  SdpaSums<NB> o;
  o.mx = -INFINITY;
  o.sum = 0.f;
#pragma unroll
  for (int b = 0; b < NB; b++)
#pragma unroll
    for (int c = 0; c < 4; c++) o.acc[b][c] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
  for (int st = c_first; st < c_last; st++) {
    const int k0 = blo + st * KC;
    floatx4 sc[NT];
#pragma unroll
    for (int n = 0; n < NT; n++) {
      const int64_t key = min(k0 + 16 * n + m, bhi);
      sc[n] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
      for (int s = 0; s < NS; s++) {
        const int x = 16 * s + 4 * g;
        const floatx4 k4 = roped(kp + key * a->k_rs, key, x), q4 = roped(qp, row, x);
#pragma unroll
        for (int j = 0; j < 4; j++)
          sc[n] = __builtin_amdgcn_mfma_f32_16x16x4f32(k4[j], q4[j], sc[n], 0, 0, 0);
      }
    }
    auto key_of = [&](int n, int j) { return k0 + 16 * n + 4 * g + j; };
    float top = -INFINITY;
#pragma unroll
    for (int n = 0; n < NT; n++)
#pragma unroll
      for (int j = 0; j < 4; j++) {
        const int key = key_of(n, j);
        if (a->has_kb && key >= a->kb_start && key < a->kb_end) sc[n][j] += a->kb_value;
        sc[n][j] = key >= lo && key <= hi ? sc[n][j] : -INFINITY;
        top = fmaxf(top, sc[n][j]);
      }
    top = fmaxf(top, __shfl_xor(top, 16));
    top = fmaxf(top, __shfl_xor(top, 32));
    const float mn = fmaxf(o.mx, top);
    const float base = mn == -INFINITY ? 0.f : mn;
    const float scale = o.mx == -INFINITY ? 0.f : expf(o.mx - base);
    float add = 0.f;
#pragma unroll
    for (int n = 0; n < NT; n++)
#pragma unroll
      for (int j = 0; j < 4; j++) {
        const int key = key_of(n, j);
        sc[n][j] = key >= lo && key <= hi ? expf(sc[n][j] - base) : 0.f;
        add += sc[n][j];
      }
    add += __shfl_xor(add, 16);
    add += __shfl_xor(add, 32);
    o.sum = o.sum * scale + add;
    o.mx = mn;
#pragma unroll 1
    for (int r = 0; r < 16; r++) {
      const int rlo = __builtin_amdgcn_readlane(lo, r), rhi = __builtin_amdgcn_readlane(hi, r);
#pragma unroll
      for (int b = 0; b < NB; b++) {
        floatx4 pv[4];
#pragma unroll
        for (int c = 0; c < 4; c++) pv[c] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int n = 0; n < NT; n++)
#pragma unroll
          for (int j = 0; j < 4; j++) {
            const int key = key_of(n, j);
            const float4 v = Ld4<T>::at(vp + (int64_t)min(key, bhi) * a->v_rs + 64 * b + 4 * m);
            const bool in = key >= rlo && key <= rhi;
            pv[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(in ? v.x : 0.f, sc[n][j], pv[0], 0, 0, 0);
            pv[1] = __builtin_amdgcn_mfma_f32_16x16x4f32(in ? v.y : 0.f, sc[n][j], pv[1], 0, 0, 0);
            pv[2] = __builtin_amdgcn_mfma_f32_16x16x4f32(in ? v.z : 0.f, sc[n][j], pv[2], 0, 0, 0);
            pv[3] = __builtin_amdgcn_mfma_f32_16x16x4f32(in ? v.w : 0.f, sc[n][j], pv[3], 0, 0, 0);
          }
#pragma unroll
        for (int c = 0; c < 4; c++)
          if (m == r) o.acc[b][c] = o.acc[b][c] * scale + pv[c];
      }
    }
  }
  return o;
}

template <typename T, int NB, int NT, bool ROPE>  // head_dim 64·NB, 16·NT keys a step
__global__ __launch_bounds__(512) void k_sdpa_mfma(AttnArgs a, int hw, int ksplit) {
  constexpr int HD = 64 * NB, NS = HD / 16;
  constexpr int KC = 16 * NT;
  extern __shared__ __align__(16) float mlds[];
  const int lane = threadIdx.x & (WAVE - 1);
  const int wave = threadIdx.x / WAVE;
  const int part = wave / hw;
  const int G = a.q_heads / a.kv_heads;
  const int hgroups = (G + hw - 1) / hw;
  const int kvh = blockIdx.y / hgroups;
  const int hg = (blockIdx.y - kvh * hgroups) * hw + wave % hw;
  const bool head_ok = hg < G;
  const int h = kvh * G + (head_ok ? hg : 0);
  const int m = lane & 15, g = lane >> 4;
  const int row0 = blockIdx.x * 16;
  const int row = min(row0 + m, a.q_len - 1);
  const T *kp = (const T *)a.k + (int64_t)kvh * HD;
  const T *vp = (const T *)a.v + (int64_t)kvh * HD;

  // The row's keys, and the tile's.
  int lo, hi;
  {
    const long long qpos = (long long)a.q_pos_offset + row;
    long long l = a.window_left < 0 ? 0 : qpos - a.window_left;
    long long u = a.window_right < 0 ? (long long)a.kv_len - 1 : qpos + a.window_right;
    if (l < 0) l = 0;
    if (u > a.kv_len - 1) u = a.kv_len - 1;
    if (a.segs) {
      const long long s0 = (long long)a.segs[2 * row], s1 = (long long)a.segs[2 * row + 1] - 1;
      if (s0 > l) l = s0;
      if (s1 < u) u = s1;
    }
    lo = (int)l;
    hi = (int)(u < l - 1 ? l - 1 : u);  // empty: hi < lo
  }
  int blo = hi >= lo ? lo : 0x7fffffff, bhi = hi >= lo ? hi : -1;
#pragma unroll
  for (int x = 1; x < 16; x <<= 1) {
    blo = min(blo, __shfl_xor(blo, x));
    bhi = max(bhi, __shfl_xor(bhi, x));
  }
  blo = __builtin_amdgcn_readfirstlane(blo);
  bhi = __builtin_amdgcn_readfirstlane(bhi);
  // This wavefront's steps of KC keys: an equal run of them per part.
  const int nstep = bhi >= blo ? (bhi - blo) / KC + 1 : 0;
  const int per = (nstep + ksplit - 1) / ksplit;
  const int c_first = part * per, c_last = min(nstep, c_first + per);

  floatx4 q[NS];
#pragma unroll
  for (int s = 0; s < NS; s++) {
    const int x = 16 * s + 4 * g;
    const float4 v = Ld4<T>::at((const T *)a.q + (int64_t)row * a.q_rs + (int64_t)h * HD + x);
    if constexpr (ROPE)
      q[s] = rope4(v, *(const float4 *)(a.rope_cos + (int64_t)row * HD + x),
                   *(const float4 *)(a.rope_sin + (int64_t)row * HD + x));
    else
      q[s] = floatx4{v.x, v.y, v.z, v.w};
  }
  struct KTile {
    float4 k[NT][NS], c[ROPE ? NT : 1][ROPE ? NS : 1], s[ROPE ? NT : 1][ROPE ? NS : 1];
  };
  // Keys past the tile's last read that one (their probability is 0).
  auto load_k = [&](int step, KTile &t) {
#pragma unroll
    for (int n = 0; n < NT; n++) {
      const int64_t key = min(blo + step * KC + 16 * n + m, bhi);
#pragma unroll
      for (int s = 0; s < NS; s++) {
        const int x = 16 * s + 4 * g;
        t.k[n][s] = Ld4<T>::at(kp + key * a.k_rs + x);
        if constexpr (ROPE) {
          t.c[n][s] = *(const float4 *)(a.rope_cos + key * HD + x);
          t.s[n][s] = *(const float4 *)(a.rope_sin + key * HD + x);
        }
      }
    }
  };
  float4 v[NT][4][NB];
  auto load_v = [&](int step) {
#pragma unroll
    for (int n = 0; n < NT; n++)
#pragma unroll
      for (int j = 0; j < 4; j++) {
        const int64_t key = min(blo + step * KC + 16 * n + 4 * g + j, bhi);
#pragma unroll
        for (int b = 0; b < NB; b++) v[n][j][b] = Ld4<T>::at(vp + key * a.v_rs + 64 * b + 4 * m);
      }
  };
  float mx = -INFINITY, sum = 0.f;
  floatx4 acc[NB][4];
#pragma unroll
  for (int b = 0; b < NB; b++)
#pragma unroll
    for (int c = 0; c < 4; c++) acc[b][c] = floatx4{0.f, 0.f, 0.f, 0.f};
  if (c_first < c_last) {  // then blo ≤ bhi: every address is a key's
    KTile kt;
    load_k(c_first, kt);
    load_v(c_first);
    for (int st = c_first; st < c_last; st++) {
      floatx4 sc[NT];
#pragma unroll
      for (int n = 0; n < NT; n++) {
        // two chains: halves the dependent MFMA latency
        floatx4 s0 = floatx4{0.f, 0.f, 0.f, 0.f}, s1 = s0;
#pragma unroll
        for (int s = 0; s < NS; s++) {
          floatx4 k4;
          if constexpr (ROPE)
            k4 = rope4(kt.k[n][s], kt.c[n][s], kt.s[n][s]);
          else
            k4 = floatx4{kt.k[n][s].x, kt.k[n][s].y, kt.k[n][s].z, kt.k[n][s].w};
          s0 = __builtin_amdgcn_mfma_f32_16x16x4f32(k4[0], q[s][0], s0, 0, 0, 0);
          s1 = __builtin_amdgcn_mfma_f32_16x16x4f32(k4[1], q[s][1], s1, 0, 0, 0);
          s0 = __builtin_amdgcn_mfma_f32_16x16x4f32(k4[2], q[s][2], s0, 0, 0, 0);
          s1 = __builtin_amdgcn_mfma_f32_16x16x4f32(k4[3], q[s][3], s1, 0, 0, 0);
        }
        sc[n] = s0 + s1;
      }
      load_k(min(st + 1, c_last - 1), kt);  // lands under the softmax and P·V
      const int key0 = blo + st * KC + 4 * g;
      float top = -INFINITY;
#pragma unroll
      for (int n = 0; n < NT; n++)
#pragma unroll
        for (int j = 0; j < 4; j++) {
          const int key = key0 + 16 * n + j;
          float x = sc[n][j];
          if (a.has_kb && key >= a.kb_start && key < a.kb_end) x += a.kb_value;
          x = key >= lo && key <= hi ? x : -INFINITY;
          sc[n][j] = x;
          top = fmaxf(top, x);
        }
      top = fmaxf(top, __shfl_xor(top, 16));
      top = fmaxf(top, __shfl_xor(top, 32));
      const float mn = fmaxf(mx, top);
      const float base = mn == -INFINITY ? 0.f : mn;  // nothing seen yet
      const float scale = mx == -INFINITY ? 0.f : expf(mx - base);
      float add = 0.f;
#pragma unroll
      for (int n = 0; n < NT; n++)
#pragma unroll
        for (int j = 0; j < 4; j++) {
          const int key = key0 + 16 * n + j;
          const float p = key >= lo && key <= hi ? expf(sc[n][j] - base) : 0.f;
          sc[n][j] = p;
          add += p;
        }
      add += __shfl_xor(add, 16);
      add += __shfl_xor(add, 32);
      sum = sum * scale + add;
      mx = mn;
#pragma unroll
      for (int b = 0; b < NB; b++)
#pragma unroll
        for (int c = 0; c < 4; c++) {
          floatx4 o = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int n = 0; n < NT; n++)
#pragma unroll
            for (int j = 0; j < 4; j++) {
              const float4 &vv = v[n][j][b];
              const float ve = c == 0 ? vv.x : c == 1 ? vv.y : c == 2 ? vv.z : vv.w;
              o = __builtin_amdgcn_mfma_f32_16x16x4f32(ve, sc[n][j], o, 0, 0, 0);
            }
          acc[b][c] = acc[b][c] * scale + o;
        }
      load_v(min(st + 1, c_last - 1));
    }
  }
  bool nan = false;
#pragma unroll
  for (int b = 0; b < NB; b++)
#pragma unroll
    for (int c = 0; c < 4; c++)
#pragma unroll
      for (int i = 0; i < 4; i++) nan |= acc[b][c][i] != acc[b][c][i];
  if (__builtin_expect(__any(nan), 0)) {
    const SdpaSums<NB> o =
        sdpa_by_rows<T, NB, NT, ROPE>(h, lo, hi, blo, bhi, c_first, c_last);
    mx = o.mx;
    sum = o.sum;
#pragma unroll
    for (int b = 0; b < NB; b++)
#pragma unroll
      for (int c = 0; c < 4; c++) acc[b][c] = o.acc[b][c];
  }
  // acc[b][c][i]: row `row`, head column 64b + 16g + 4i + c.
  if (ksplit > 1) {
    // The later parts leave (max, sum, acc); the first folds them in, in order.
    constexpr int SLOT = (2 + 16 * NB) * WAVE;
    if (part > 0) {
      float *d = mlds + ((part - 1) * hw + wave % hw) * SLOT + lane;
      d[0] = mx;
      d[WAVE] = sum;
#pragma unroll
      for (int b = 0; b < NB; b++)
#pragma unroll
        for (int c = 0; c < 4; c++)
#pragma unroll
          for (int i = 0; i < 4; i++) d[(2 + 16 * b + 4 * c + i) * WAVE] = acc[b][c][i];
    }
    __syncthreads();
    if (part > 0) return;
    for (int p = 1; p < ksplit; p++) {
      const float *d = mlds + ((p - 1) * hw + wave % hw) * SLOT + lane;
      const float m2 = d[0];
      const float mn = fmaxf(mx, m2);
      const float base = mn == -INFINITY ? 0.f : mn;
      const float f1 = mx == -INFINITY ? 0.f : expf(mx - base);
      const float f2 = m2 == -INFINITY ? 0.f : expf(m2 - base);
      sum = sum * f1 + d[WAVE] * f2;
      mx = mn;
#pragma unroll
      for (int b = 0; b < NB; b++)
#pragma unroll
        for (int c = 0; c < 4; c++)
#pragma unroll
          for (int i = 0; i < 4; i++)
            acc[b][c][i] = acc[b][c][i] * f1 + d[(2 + 16 * b + 4 * c + i) * WAVE] * f2;
    }
  }
  if (!head_ok || row0 + m >= a.q_len) return;
  // Sinks join the denominator; store.
  const float sg = a.sinks ? a.sinks[h] * LN2 : -INFINITY;
  const float mf = fmaxf(mx, sg);
  float f = 0.f;
  if (mf != -INFINITY) {
    const float scale = mx == -INFINITY ? 0.f : expf(mx - mf);
    f = scale * (1.0f / (sum * scale + (a.sinks ? expf(sg - mf) : 0.f)));
  }
  T *out = (T *)a.out + (int64_t)row * a.o_rs + (int64_t)h * HD + 16 * g;
#pragma unroll
  for (int b = 0; b < NB; b++)
#pragma unroll
    for (int i = 0; i < 4; i++)
      st4(out + 64 * b + 4 * i, acc[b][0][i] * f, acc[b][1][i] * f, acc[b][2][i] * f,
          acc[b][3][i] * f);
}

}  // namespace

int launch_rope(const void *x, moe_dtype dt, int rows, int cols, int hd, int src_start, int width,
                const float *cs, const float *sn, void *out, hipStream_t s) {
  MOE_NONNULL(x);
  MOE_NONNULL(cs);
  MOE_NONNULL(sn);
  MOE_NONNULL(out);
  const int64_t n = (int64_t)rows * (width / 2);
  const int64_t blocks = (n + 255) / 256;
  if (blocks > 0x7fffffff) return moe_fail(MOE_INVALID_ARGUMENT, "rope: input too large");
  if (dt == MOE_F16)
    hipLaunchKernelGGL(k_rope<_Float16>, dim3((unsigned)blocks), dim3(256), 0, s,
                       (const _Float16 *)x, cs, sn, (_Float16 *)out, rows, cols, hd, src_start,
                       width);
  else
    hipLaunchKernelGGL(k_rope<float>, dim3((unsigned)blocks), dim3(256), 0, s, (const float *)x, cs,
                       sn, (float *)out, rows, cols, hd, src_start, width);
  return 0;
}

// k_sdpa_mfma: head_dim 64 or 128, every row's four-column groups aligned.
static bool sdpa_mfma_ok(const AttnArgs &a) {
  if (a.head_dim != 64 && a.head_dim != 128) return false;
  const uintptr_t al = a.dtype == MOE_F16 ? 8 : 16;
  for (const void *p : {a.q, a.k, a.v, (const void *)a.out})
    if ((uintptr_t)p % al) return false;
  if (a.q_rs % 4 || a.k_rs % 4 || a.v_rs % 4 || a.o_rs % 4) return false;
  return (uintptr_t)a.rope_cos % 16 == 0 && (uintptr_t)a.rope_sin % 16 == 0 &&
         (int64_t)a.kv_heads * (a.q_heads / a.kv_heads) <= 65535;
}

int launch_sdpa(AttnArgs a, hipStream_t s) {
  MOE_NONNULL(a.q);
  MOE_NONNULL(a.k);
  MOE_NONNULL(a.v);
  MOE_NONNULL(a.out);
  const int G = a.q_heads / a.kv_heads;
  if (G > AW * AI)
    return moe_fail(MOE_INVALID_ARGUMENT, "sdpa: more than " + std::to_string(AW * AI) +
                                              " query heads per kv head");
  if (sdpa_mfma_ok(a)) {
    // Keys of a row tile: the window and 15 more rows, at most kv_len.
    const int64_t span = a.window_left < 0 || a.window_right < 0
                             ? a.kv_len
                             : std::min<int64_t>(a.kv_len, a.window_left + a.window_right + 16);
    const int kc = a.head_dim == 64 ? 32 : 16;
    const int64_t nstep = (span + kc - 1) / kc;
    const int64_t tiles = ((int64_t)a.q_len + 15) / 16;
    // Heads of a kv head together (K, V and rope tables from one L1) once that
    // gives two blocks a CU, else a block per head; up to 4 wavefronts over its
    // keys while heads × row tiles × parts stay near 2500 (attention block,
    // µs, one head and 1, 2, 4, 8 parts, seven heads: 300 rows 58, 50, 46, 51,
    // 81; 1500 rows 109, 109, 113, 131, 115; 4096 rows 259, 244, 250, 298, 236).
    const int64_t heads = tiles * a.q_heads;
    int hw = std::min(G, 8);
    if (tiles * a.kv_heads * ((G + hw - 1) / hw) < 512) hw = 1;
    int ks = 1;
    while (hw == 1 && ks < 4 && ks * 2 <= nstep && heads * ks * 2 <= 2700) ks *= 2;
    const dim3 grid((unsigned)tiles, a.kv_heads * ((G + hw - 1) / hw)), block(WAVE * hw * ks);
    const size_t lds = (size_t)(ks - 1) * hw * (2 + 16 * (a.head_dim / 64)) * WAVE * 4;
#define SDPA_M(T_, NB_, NT_)                                                                     \
  do {                                                                                           \
    if (a.rope_cos) hipLaunchKernelGGL((k_sdpa_mfma<T_, NB_, NT_, true>), grid, block, lds, s, a, hw, ks); \
    else hipLaunchKernelGGL((k_sdpa_mfma<T_, NB_, NT_, false>), grid, block, lds, s, a, hw, ks); \
  } while (0)
    if (a.dtype == MOE_F16) {
      if (a.head_dim == 64) SDPA_M(_Float16, 1, 2);
      else SDPA_M(_Float16, 2, 1);
    } else {
      if (a.head_dim == 64) SDPA_M(float, 1, 2);
      else SDPA_M(float, 2, 1);
    }
#undef SDPA_M
    return 0;
  }
  // Rows per block: up to the 64 items a block holds, fewer for short
  // sequences so that the grid still has ~512 blocks (each block stages its
  // keys once; more rows per block share more of them).
  const int max_rows = (AW * AI) / G;
  const long want = ((long)a.q_len * a.kv_heads + 511) / 512;
  a.rows_per_block = (int)std::max(1L, std::min((long)max_rows, want));
  const int ns = a.head_dim <= 64 ? 1 : 2;
  const size_t lds = (size_t)(AW * AI * 64 * ns + 2 * AKC * (64 * ns + 4)) * 4;
  dim3 grid((a.q_len + a.rows_per_block - 1) / a.rows_per_block, a.kv_heads), block(AW * WAVE);
  // Dynamic LDS past 64 KB (the two-slab kernels) needs the kernel's limit raised.
  static bool raised = false;
  if (!raised) {
    const int big = (AW * AI * 128 + 2 * AKC * 132) * 4;
    if (hipFuncSetAttribute((const void *)k_sdpa<_Float16, 2>,
                            hipFuncAttributeMaxDynamicSharedMemorySize, big) != hipSuccess ||
        hipFuncSetAttribute((const void *)k_sdpa<float, 2>,
                            hipFuncAttributeMaxDynamicSharedMemorySize, big) != hipSuccess)
      return moe_fail(MOE_EXECUTION_FAILED, "sdpa: cannot raise the LDS limit of the kernel");
    raised = true;
  }
  if (a.dtype == MOE_F16) {
    if (ns == 1) hipLaunchKernelGGL((k_sdpa<_Float16, 1>), grid, block, lds, s, a);
    else hipLaunchKernelGGL((k_sdpa<_Float16, 2>), grid, block, lds, s, a);
  } else {
    if (ns == 1) hipLaunchKernelGGL((k_sdpa<float, 1>), grid, block, lds, s, a);
    else hipLaunchKernelGGL((k_sdpa<float, 2>), grid, block, lds, s, a);
  }
  return 0;
}

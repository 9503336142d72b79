// Decode attention over a codebook cache (the GPU TurboQuant caches' fused
// attention, turboquant.rs:763-923, for one query position): keys and values
// are stored rotated (y = R x) as u8 codes + f32 sigma, so the query is
// rotated the same way, attention runs in the rotated basis over
// centroid[c] * sigma, and the output goes back through R^T.
//
// Four launches: the query's rotation (and, with QJL, its projection by Phi),
// the attention over splits of the tokens, the merge of the splits, and the
// rotation back.
//
// Bound: HBM (2 (D + 4) bytes a token of a KV head), if looking a code up
// and multiplying it costs less. The products run on the matrix cores in f16
// split in two: a centroid, a query value and a weight are each hi + lo, two
// f16 values of a power-of-two multiple that puts the largest near 2^15, so
// hi + lo holds 22 bits and products are exact in f32. The rows of a product
// are 16 tokens (scores) or 16 channels (values), its columns the query heads:
// up to 8 heads take one column for their hi and one for their lo part, so
// two products (centroid hi, centroid lo) give all four partial products; 16
// heads take three products. A code is looked up once for all heads (one
// 4-byte LDS read: hi | lo << 16), where f32 multiply-adds a head repeated
// the lookups for every two heads at D = 512 and cost a vector operation a
// code and head. Against 64 bits the merged rows (before the rotation back and
// the bf16 rounding) are 0.36 to 0.80 times as far off as that kernel's over 81
// shapes of every head dim, width and head count (D = 512, 16 heads: 2.8e-6 ->
// 1.2e-6; D = 64: 1.2e-6 -> 1.0e-6): the f32 chain over D channels had lost
// more than the operands' last bits.
// Measured a call: Gemma 4's global layers (B = 1, 32 / 2 heads, D = 512,
// 32,768 tokens, 4-bit) 227 -> 43 us; B = 32, 16 / 8 heads, D = 256, 32,768
// tokens, 3-bit 850 -> 795 us (5.5 TB/s; vector issue 63% of its cycles, LDS
// 43%); B = 26, 8 heads, D = 128, 7,677 tokens 158 -> 109 us; B = 22, 32 / 8
// heads, D = 64, 31,445 tokens 293 -> 204 us. Wavefronts a SIMD (registers
// against spills outside the loop): 4 at D = 256 (3: 860 us for the 3-bit
// shape), 3 at D = 64 and 128 (4: 167 us for the D = 128 one), 2 at D = 512.
#include <cmath>

#include "common.hpp"

namespace tqkv {
namespace cb {
namespace {

constexpr int kWave = 64;
constexpr int kMaxQjl = 1024;  // most QJL rows (m = 32 * qjl_words)

typedef _Float16 h8_t __attribute__((ext_vector_type(8)));
typedef float f4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u4_t __attribute__((ext_vector_type(4)));

// ---------------------------------------------------------------- rotations
// y[r][i] = sum_j x[r][j] M[i][j] (kRows: rows of M are the outputs: the
// query's rotation R q and its projection Phi q) or sum_j x[r][j] M[j][i]
// (!kRows: R^T o), r < rows, i < n, j < D, in f32 on
// v_mfma_f32_16x16x4_f32. A workgroup takes 16 rows and 16 outputs, its four
// wavefronts a quarter of j each (summed in wavefront order): latency bound
// (M is at most 1 MB, in L2), so many small workgroups and short chains.
// Measured at Gemma 4's global shape (32 rows, D = 512, kernel trace): 15 ->
// 5 us for the query, 38 -> 5 + 5 us for the merge and the rotation back.
// x: bf16 or f32 rows. y: f32 (and ys = y * scale, if given) or bf16.
template <int D, bool kRows, typename X>
__global__ __launch_bounds__(256) void cb_matmul_kernel(const X* __restrict__ x,
                                                        const float* __restrict__ M, int n,
                                                        int64_t rows, float scale,
                                                        float* __restrict__ y,
                                                        float* __restrict__ ys,
                                                        uint16_t* __restrict__ yb) {
  __shared__ f4_t s_acc[3][kWave];
  const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
  const int lr = lane % 16, lg = lane / 16;
  const int64_t r0 = int64_t(blockIdx.x) * 16;
  const int i0 = int(blockIdx.y) * 16;
  const int64_t r = r0 + lr < rows ? r0 + lr : rows - 1;  // past the end: repeated, not written
  const int i = i0 + lr < n ? i0 + lr : n - 1;
  f4_t acc = {0.0f, 0.0f, 0.0f, 0.0f};
  const int j0 = wave * (D / 4);
#pragma unroll
  for (int j = 0; j < D / 4; j += 16) {
    const int jj = j0 + j + 4 * lg;  // this lane's four steps
    float a[4], b[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      if constexpr (sizeof(X) == 2)
        a[e] = bf16_to_f32(x[r * D + jj + e]);
      else
        a[e] = x[r * D + jj + e];
      b[e] = kRows ? M[int64_t(i) * D + jj + e] : M[int64_t(jj + e) * n + i];
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a[e], b[e], acc, 0, 0, 0);
  }
  if (wave) s_acc[wave - 1][lane] = acc;
  __syncthreads();
  if (wave) return;
#pragma unroll
  for (int w = 0; w < 3; ++w) acc += s_acc[w][lane];
  if (i0 + lr >= n) return;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int64_t ro = r0 + 4 * lg + e;
    if (ro >= rows) break;
    if (yb) {
      yb[ro * n + i] = f32_to_bf16(acc[e]);
    } else {
      y[ro * n + i] = acc[e];
      if (ys) ys[ro * n + i] = acc[e] * scale;
    }
  }
}

// ---------------------------------------------------------------- attention
struct Args {
  const float* qs;      // [B, H, D]: R q, scaled to log2 units
  const float* pq;      // QJL: [B, H, m] Phi q
  const uint8_t* kc;
  const float* ks;
  const uint8_t* vc;
  const float* vs;
  const float* cent_k;
  const float* cent_v;
  const uint32_t* ksg;  // QJL signs and residual norms
  const float* krn;
  float* part_o;
  float* part_m;
  float* part_l;
  int64_t cap, n, split_len;
  int H, H_kv, G, n_k, n_v, n_splits, qm;
  float qscale;
};

// The power of two that puts values of magnitude up to the one with bits
// `mx` into [2^14, 2^15), as its exponent (at most 90, so that sums of scaled
// weights stay finite; 0 for zero, infinity and NaN).
__device__ __forceinline__ int norm_exp(uint32_t mx) {
  const int e = int(mx >> 23) - 127;
  if (mx == 0 || e == 128) return 0;
  return 14 - e < 90 ? 14 - e : 90;
}
// The same for a whole operand (a table, a head's query): kWide where its
// largest is an infinity, NaN or outside [2^-64, 2^64), which hi + lo does not
// hold as f32 does. The decode then marks the head's partials (a sum of
// kWideSum, which no sum of weights is) and the merge attends in f32.
constexpr int kWide = 1 << 10;
constexpr float kWideSum = -1.0f;
__device__ __forceinline__ int operand_exp(uint32_t mx) {
  const int e = int(mx >> 23) - 127;
  return mx != 0 && (e < -64 || e > 63) ? kWide : norm_exp(mx);
}
__device__ __forceinline__ float pow2(int e) { return __uint_as_float(uint32_t(127 + e) << 23); }
__device__ __forceinline__ uint32_t mag(float x) { return __float_as_uint(x) & 0x7fffffffu; }

// x (|x| < 2^15) as hi | lo << 16, f16 each: hi + lo = x to 22 bits.
__device__ __forceinline__ uint32_t split_h16(float x) {
  const _Float16 hi = _Float16(x);
  const _Float16 lo = _Float16(x - float(hi));
  return uint32_t(__builtin_bit_cast(uint16_t, hi)) |
         (uint32_t(__builtin_bit_cast(uint16_t, lo)) << 16);
}

// The hi and lo operands of eight table entries.
__device__ __forceinline__ void pair_up(const uint32_t (&e)[8], h8_t& hi, h8_t& lo) {
  u4_t h, l;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    h[k] = __builtin_amdgcn_perm(e[2 * k + 1], e[2 * k], 0x05040100u);
    l[k] = __builtin_amdgcn_perm(e[2 * k + 1], e[2 * k], 0x07060302u);
  }
  hi = __builtin_bit_cast(h8_t, h);
  lo = __builtin_bit_cast(h8_t, l);
}

__device__ __forceinline__ f4_t mma(h8_t a, h8_t b, f4_t c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
}

// The launch shape: D / 64 wavefronts, each scoring kSub blocks of 16 tokens
// of a tile and then accumulating its 64 channels over the whole tile (so an
// accumulator is 16 registers a wavefront at any D, and four wavefronts a
// SIMD keep the loads in flight).
template <int D>
struct Shape {
  static constexpr int kWaves = D / 64;
  static constexpr int kSub = D == 64 ? 4 : D == 128 ? 2 : 1;
  static constexpr int kTokens = 16 * kWaves * kSub;  // a tile: 64, or 128 at D = 512
};

// One workgroup per (split, KV head, batch row): softmax state and
// unnormalized output over the split's tokens for the G = H / H_kv heads.
// G16: 16 heads; otherwise 1, 2, 4 or 8 (column c: head c's hi part for c <
// G, head c - G's lo part for G <= c < 2 G, unused beyond).
// PAIR: codes of at most 4 bits, looked up two at a time: entry c | c' << bits
// of a 256-entry table holds the operands' words for codes c and c' (their hi
// parts, their lo parts), so a code costs about one vector operation and half
// an LDS read where single lookups take two and one. V's two words are read
// together and used as they land, hi and lo in one operand (k slots 4 p + {0,
// 1}: hi of tokens 2 p, 2 p + 1 of a group of four; {2, 3}: lo) against
// weights held twice; assembling separate hi and lo operands took 1.5 moves a
// pair.
// QJL: each key's score gains the estimate of q . r from its residual signs
// (qjl.rs:86-118, the two-stage scores of compressor.rs:122-159), as a
// product of the signs (+-1 in f16) with Phi q.
template <int D, bool G16, bool QJL, bool PAIR>
__global__ __launch_bounds__(D) __attribute__((amdgpu_waves_per_eu(D == 256 ? 4 : D == 512 ? 2 : 3)))
void cb_decode_kernel(const Args a) {
  constexpr int kSub = Shape<D>::kSub, T = Shape<D>::kTokens;
  constexpr int NU = D / 64, NP = T / 32;
  constexpr int kParts = G16 ? 2 : 1;  // operand sets of the query: hi and lo, or both in one
  extern __shared__ __attribute__((aligned(16))) uint16_t s_q[];  // [parts][k step][lane][8]
  __shared__ __attribute__((aligned(16))) uint32_t s_ck[256], s_cv[256];  // hi | lo << 16
  __shared__ uint2 s_pk[PAIR ? 256 : 1], s_pv[PAIR ? 256 : 1];            // pairs of codes
  __shared__ __attribute__((aligned(16))) float s_s[2][16][T + 4];  // the tile's scores
  __shared__ __attribute__((aligned(16))) float s_sv[2][T];         // and value sigmas
  __shared__ int s_e[34];  // scale exponents: heads' q, heads' Phi q, centroids of K and V
  const int tid = threadIdx.x, lane = tid % kWave;
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int lr = lane % 16, lg = lane / 16;
  const int split = blockIdx.x, kvh = blockIdx.y, b = blockIdx.z;
  const int G = G16 ? 16 : a.G;
  const int mk = QJL ? (a.qm + 31) / 32 : 0;  // k steps of the signs
  const int steps = D / 32 + mk;
  const int64_t slab = (int64_t(b) * a.H_kv + kvh) * a.cap;
  const int64_t t0 = int64_t(split) * a.split_len;
  const int64_t t1 = t0 + a.split_len < a.n ? t0 + a.split_len : a.n;
  const int64_t qrow = int64_t(b) * a.H + int64_t(kvh) * G;

  // Loads of the tile at `base` (a multiple of T past t0, before t1): tokens
  // past the range re-read its last one, masked in the scores.
  // Scores: token 16 (kSub wave + q) + lr, channels 64 u + 16 lg + [0, 16).
  u4_t kr[kSub][NU];
  float skr[kSub][4];
  auto load_k = [&](int64_t base) __attribute__((always_inline)) {
    const uint32_t last = uint32_t(t1 - base < T ? t1 - base : T) - 1;
    const uint8_t* src = a.kc + (slab + base) * D;
    const float* sg = a.ks + slab + base;
#pragma unroll
    for (int q = 0; q < kSub; ++q) {
      const uint32_t tok = 16 * (kSub * wave + q);
      const uint32_t off = min(tok + lr, last) * D + 16 * lg;
#pragma unroll
      for (int u = 0; u < NU; ++u) kr[q][u] = *reinterpret_cast<const u4_t*>(src + (off + 64 * u));
#pragma unroll
      for (int r = 0; r < 4; ++r) skr[q][r] = sg[min(tok + 4 * lg + r, last)];
    }
  };
  // Values: tokens 32 u + 4 lg + i and 32 u + 16 + 4 lg + i (the order of the
  // weight operand's k slots), channels 64 wave + 4 lr + [0, 4).
  uint32_t vr[8 * NP];
  float svr = 0.0f;
  auto load_v = [&](int64_t base) __attribute__((always_inline)) {
    const uint32_t last = uint32_t(t1 - base < T ? t1 - base : T) - 1;
    const uint8_t* src = a.vc + (slab + base) * D + 64 * wave;
    // (Value codes need no alignment below D = 256: a plain 4-byte copy.)
    if (last == T - 1) {
      const uint32_t off = 4 * lg * D + 4 * lr;
#pragma unroll
      for (int i = 0; i < 8 * NP; ++i)
        __builtin_memcpy(&vr[i], src + (off + (32 * (i / 8) + 16 * (i / 4 % 2)) * D) + i % 4 * D, 4);
    } else {
#pragma unroll
      for (int i = 0; i < 8 * NP; ++i) {
        const uint32_t tok = 32 * (i / 8) + 16 * (i / 4 % 2) + 4 * lg + i % 4;
        __builtin_memcpy(&vr[i], src + (min(tok, last) * D + 4 * lr), 4);
      }
    }
    svr = tid < T ? a.vs[slab + base + min(uint32_t(tid), last)] : 0.0f;
  };
  load_k(t0);
  load_v(t0);

  // Tables and query operands, no wavefront needing another's part before
  // the one barrier. The largest magnitude among `width` lanes:
  auto largest = [&](uint32_t mx, int width) __attribute__((always_inline)) {
    for (int off = 1; off < width; off <<= 1) mx = max(mx, uint32_t(__shfl_xor(int(mx), off, kWave)));
    return mx;
  };
  auto table = [&](const float* cent, int n, uint32_t* tab, int* exp) __attribute__((always_inline)) {
    float c[4];
    uint32_t mx = 0;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      c[k] = 4 * lane + k < n ? cent[4 * lane + k] : 0.0f;
      mx = max(mx, mag(c[k]));
    }
    const int e = operand_exp(largest(mx, kWave));
    u4_t t;
#pragma unroll
    for (int k = 0; k < 4; ++k) t[k] = split_h16(c[k] * pow2(e));
    *reinterpret_cast<u4_t*>(tab + 4 * lane) = t;
    if (lane == 0) *exp = e;
  };
  constexpr int kWaves = Shape<D>::kWaves;
  if (wave == 0) table(a.cent_k, a.n_k, s_ck, &s_e[32]);
  if (wave == kWaves - 1) table(a.cent_v, a.n_v, s_cv, &s_e[33]);
  // Eight values of head h at k step `step`, lane group g, their scale 2^e.
  auto put_q = [&](int h, int step, int g, const float (&v)[8], int e) __attribute__((always_inline)) {
    uint32_t w[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) w[k] = split_h16(v[k] * pow2(e));
    h8_t hi, lo;
    pair_up(w, hi, lo);
    h8_t* at = reinterpret_cast<h8_t*>(s_q) + step * kWave + 16 * g;
    at[h] = hi;
    at[G16 ? steps * kWave + h : h + G] = lo;
  };
  // D / 8 lanes a head, eight channels each. The scores' k order: channels
  // 8 i + [0, 8) sit in step 2 (i / 8) + i % 2 at lane group i / 2 % 4 (a
  // lane's 16-byte load is two steps).
  constexpr int kLph = D / 8, kHpw = kWave / kLph;
  for (int h0 = wave * kHpw; h0 < G; h0 += kWaves * kHpw) {
    const int h = h0 + lane / kLph, i = lane % kLph;
    const float* src = a.qs + (qrow + (h < G ? h : G - 1)) * D + 8 * i;
    float v[8];
    uint32_t mx = 0;
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      v[k] = src[k];
      mx = max(mx, mag(v[k]));
    }
    const int e = operand_exp(largest(mx, kLph));
    if (h < G) {
      put_q(h, 2 * (i / 8) + i % 2, i / 2 % 4, v, e);
      if (i == 0) s_e[h] = e;
    }
  }
  if constexpr (QJL) {  // a wavefront a head, sign rows 8 i + [0, 8) a lane
    for (int h = wave; h < G; h += kWaves) {
      const float* src = a.pq + (qrow + h) * a.qm;
      uint32_t mx = 0;
      for (int i = lane; i < a.qm; i += kWave) mx = max(mx, mag(src[i]));
      const int e = operand_exp(largest(mx, kWave));
      for (int i = lane; i < 4 * mk; i += kWave) {
        float v[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) v[k] = 8 * i + k < a.qm ? src[8 * i + k] : 0.0f;
        put_q(h, D / 32 + i / 4, i % 4, v, e);
      }
      if (lane == 0) s_e[16 + h] = e;
    }
  }
  if (!G16 && G < 8)  // the unused columns
    for (int i = tid; i < steps * kWave; i += D)
      if (i % 16 >= 2 * G) reinterpret_cast<u4_t*>(s_q)[i] = u4_t{0, 0, 0, 0};
  __syncthreads();
  if constexpr (PAIR) {
    for (int i = tid; i < 256; i += D) {
      const uint32_t ck = s_ck[i & (a.n_k - 1)], dk = s_ck[i / a.n_k];  // (zeros past n - 1)
      s_pk[i] = uint2{__builtin_amdgcn_perm(dk, ck, 0x05040100u), __builtin_amdgcn_perm(dk, ck, 0x07060302u)};
      const uint32_t cv = s_cv[i & (a.n_v - 1)], dv = s_cv[i / a.n_v];
      s_pv[i] = uint2{__builtin_amdgcn_perm(dv, cv, 0x05040100u), __builtin_amdgcn_perm(dv, cv, 0x07060302u)};
    }
    __syncthreads();
  }
  const int bits_k = 31 - __builtin_clz(a.n_k), bits_v = 31 - __builtin_clz(a.n_v);
  const int hd = lr & (G - 1);  // this lane's head
  const float fq = pow2(-s_e[hd]), fk = pow2(-s_e[32]);
  // sqrt(pi/2) / sqrt(m), and the scores' log2 units.
  const float fj = QJL ? 1.2533141373155001f / sqrtf(float(a.qm)) * a.qscale * pow2(-s_e[16 + hd]) : 0.0f;
  const bool lo_col = !G16 && lr >= G;
  auto q_op = [&](int part, int step) __attribute__((always_inline)) {
    return *reinterpret_cast<const h8_t*>(s_q + ((part * steps + step) * kWave + lane) * 8);
  };

  float m = -INFINITY, l = 0.0f;
  f4_t o[4];  // channels 64 wave + 4 (4 lg + r) + j of this lane's column
#pragma unroll
  for (int j = 0; j < 4; ++j) o[j] = f4_t{0.0f, 0.0f, 0.0f, 0.0f};
  // The weights' exponentials p are held times 2^sv_exp, which puts p * sigma
  // below 2^15 for sigma < sv_lim; l sums them so scaled. The scale follows
  // the tiles' largest sigmas, down as they pass sv_lim and up as a whole tile
  // stays below sv_low, so that a weight keeps its 22 bits after a tile of
  // zeros or of far larger sigmas. (In one tile with sigmas 2^15 times larger
  // its last bits are below theirs.) Up it stays within 2^64 of the lowest
  // scale so far, where the older sums (below 2^61) cannot overflow.
  int sv_exp = 0, sv_top = 90;
  float sv_lim = 0.0f, sv_low = 0.0f;

  int buf = 0;
  for (int64_t base = t0; base < t1; base += T, buf ^= 1) {
    const int64_t next = base + T < t1 ? base + T : base;  // (the last tile re-loads itself)
    if (tid < T) s_sv[buf][tid] = svr;
    // Scores of this wavefront's tokens.
#pragma unroll
    for (int q = 0; q < kSub; ++q) {
      // (hi and lo parts apart: two chains of products)
      f4_t sc = {0.0f, 0.0f, 0.0f, 0.0f}, sl = sc, sj = sc;
#pragma unroll
      for (int u = 0; u < NU; ++u)
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          h8_t hi, lo;
          if constexpr (PAIR) {
            u4_t hw, lw;
#pragma unroll
            for (int k = 0; k < 2; ++k) {
              const uint32_t w = kr[q][u][2 * h + k];
              const uint32_t t = w | (w >> (8 - bits_k));  // pairs in bytes 0 and 2
              const uint2 e0 = s_pk[t & 0xffu], e1 = s_pk[(t >> 16) & 0xffu];
              hw[2 * k] = e0.x, hw[2 * k + 1] = e1.x;
              lw[2 * k] = e0.y, lw[2 * k + 1] = e1.y;
            }
            hi = __builtin_bit_cast(h8_t, hw);
            lo = __builtin_bit_cast(h8_t, lw);
          } else {
            uint32_t e[8];
#pragma unroll
            for (int k = 0; k < 8; ++k) e[k] = s_ck[(kr[q][u][2 * h + k / 4] >> (8 * (k % 4))) & 0xffu];
            pair_up(e, hi, lo);
          }
          const h8_t qh = q_op(0, 2 * u + h);
          sc = mma(hi, qh, sc);
          sl = mma(lo, qh, sl);
          if constexpr (G16) sl = mma(hi, q_op(1, 2 * u + h), sl);
        }
      const int64_t tok = base + 16 * (kSub * wave + q);  // of the block's first row
      float rn[4];
      if constexpr (QJL) {
        const int64_t row = slab + (tok + lr < t1 ? tok + lr : t1 - 1);
        for (int s = 0; s < mk; ++s) {
          const uint32_t bits = a.ksg[row * mk + s] >> (8 * lg);
          u4_t sg;  // bit set: +1, clear: -1
#pragma unroll
          for (int k = 0; k < 4; ++k) {
            const uint32_t neg = ~(bits >> (2 * k));
            sg[k] = 0x3c003c00u | ((neg & 1u) << 15) | ((neg & 2u) << 30);
          }
          const h8_t sv = __builtin_bit_cast(h8_t, sg);
          sj = mma(sv, q_op(0, D / 32 + s), sj);
          if constexpr (G16) sj = mma(sv, q_op(1, D / 32 + s), sj);
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int64_t at = tok + 4 * lg + r;
          rn[r] = a.krn[slab + (at < t1 ? at : t1 - 1)];
        }
      }
      f4_t out;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        float x = sc[r] + sl[r];
        if constexpr (!G16) x += __shfl_xor(x, G, kWave);
        x = x * fk * fq * skr[q][r];
        if constexpr (QJL) {
          float c = sj[r];
          if constexpr (!G16) c += __shfl_xor(c, G, kWave);
          if (rn[r] >= 1e-10f) x = fmaf(c * rn[r], fj, x);
        }
        out[r] = tok + 4 * lg + r < t1 ? x : -INFINITY;
      }
      if (lr < G)
        *reinterpret_cast<f4_t*>(&s_s[buf][lr][16 * (kSub * wave + q) + 4 * lg]) = out;
    }
    load_k(next);
    // One barrier a tile: a buffer is written again two tiles on, after the
    // next tile's barrier, which every wavefront reaches past its reads here.
    __syncthreads();
    f4_t s[2 * NP], sv[2 * NP];
    float mx = -INFINITY, smx = 0.0f;
#pragma unroll
    for (int i = 0; i < 2 * NP; ++i) {
      s[i] = *reinterpret_cast<const f4_t*>(&s_s[buf][hd][16 * i + 4 * lg]);
      sv[i] = *reinterpret_cast<const f4_t*>(&s_sv[buf][16 * i + 4 * lg]);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        mx = fmaxf(mx, s[i][r]);
        smx = fmaxf(smx, fabsf(sv[i][r]));
      }
    }
    mx = fmaxf(mx, __shfl_xor(mx, 16, kWave));
    mx = fmaxf(mx, __shfl_xor(mx, 32, kWave));
    const float mn = fmaxf(m, mx);
    float f = m == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(m - mn);
    m = mn;
    if (__any(smx >= sv_lim) || !__any(smx >= sv_low)) {
      smx = fmaxf(smx, __shfl_xor(smx, 16, kWave));
      smx = fmaxf(smx, __shfl_xor(smx, 32, kWave));
      // (The same in all lanes: the scale stays in scalar registers.)
      const uint32_t top = __builtin_amdgcn_readfirstlane(__float_as_uint(smx));
      if (top != 0) {  // (a tile of zeros weighs nothing at any scale)
        const int e = min(norm_exp(top), sv_top);
        f *= ldexpf(1.0f, e - sv_exp);
        sv_exp = e;
        sv_top = min(sv_top, e + 64);
        sv_lim = pow2(15 - e);
        sv_low = pow2(15 - 8 - e);
      }
    }
    l *= f;
#pragma unroll
    for (int j = 0; j < 4; ++j) o[j] *= f;
    // (No key scored above -infinity yet: exponents of -infinity, not NaN.)
    const float off = (mn == -INFINITY ? 0.0f : mn) - float(sv_exp);
    // Weight operands (PAIR: of tokens i = 0, 1, 0, 1, 2, 3, 2, 3 and 4, 5, 4,
    // 5, 6, 7, 6, 7 of the lane's eight; else of 0 .. 7).
    h8_t w[kParts][NP][PAIR ? 2 : 1];
#pragma unroll
    for (int u = 0; u < NP; ++u)
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const float p = __builtin_amdgcn_exp2f(s[2 * u + i / 4][i % 4] - off);
        l += p;
        const float x = p * sv[2 * u + i / 4][i % 4];
        const _Float16 hi = _Float16(x);
        const _Float16 lo = _Float16(x - float(hi));
        auto put = [&](int part, _Float16 v) __attribute__((always_inline)) {
          if constexpr (PAIR) {
            w[part][u][i / 4][i / 2 % 2 * 4 + i % 2] = v;
            w[part][u][i / 4][i / 2 % 2 * 4 + 2 + i % 2] = v;
          } else {
            w[part][u][0][i] = v;
          }
        };
        if constexpr (G16) {
          put(0, hi);
          put(kParts - 1, lo);
        } else {
          put(0, lo_col ? lo : hi);
        }
      }
    // O^T += V^T W^T, 16 channels by 32 tokens, hi and lo: two products.
#pragma unroll
    for (int u = 0; u < NP; ++u) {
      if constexpr (PAIR) {
        uint32_t t[4];  // byte j: the pair of tokens 2 k and 2 k + 1 at channel j
#pragma unroll
        for (int k = 0; k < 4; ++k) t[k] = vr[8 * u + 2 * k] | (vr[8 * u + 2 * k + 1] << bits_v);
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            const uint2 e0 = s_pv[(t[2 * h] >> (8 * j)) & 0xffu];
            const uint2 e1 = s_pv[(t[2 * h + 1] >> (8 * j)) & 0xffu];
            const h8_t x = __builtin_bit_cast(h8_t, u4_t{e0.x, e0.y, e1.x, e1.y});
            o[j] = mma(x, w[0][u][h], o[j]);
            // (16 heads: the lo weights take the lo parts too.)
            if constexpr (G16) o[j] = mma(x, w[kParts - 1][u][h], o[j]);
          }
      } else {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          uint32_t e[8];
#pragma unroll
          for (int k = 0; k < 8; ++k) e[k] = s_cv[(vr[8 * u + k] >> (8 * j)) & 0xffu];
          h8_t hi, lo;
          pair_up(e, hi, lo);
          o[j] = mma(hi, w[0][u][0], o[j]);
          o[j] = mma(lo, w[0][u][0], o[j]);
          if constexpr (G16) o[j] = mma(hi, w[kParts - 1][u][0], o[j]);
        }
      }
    }
    load_v(next);
  }
  l += __shfl_xor(l, 16, kWave);
  l += __shfl_xor(l, 32, kWave);
  const float fo = pow2(-s_e[33]);
#pragma unroll
  for (int j = 0; j < 4; ++j)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      float x = o[j][r];
      if constexpr (!G16) x += __shfl_xor(x, G, kWave);
      o[j][r] = ldexpf(x * fo, -sv_exp);
    }
  if (lr >= G) return;
  const int64_t row = (qrow + lr) * a.n_splits + split;
  float* po = a.part_o + row * D + 64 * wave + 16 * lg;
#pragma unroll
  for (int r = 0; r < 4; ++r)
    *reinterpret_cast<f4_t*>(po + 4 * r) = f4_t{o[0][r], o[1][r], o[2][r], o[3][r]};
  if (wave == 0 && lg == 0) {
    a.part_m[row] = m;
    const bool wide = s_e[hd] == kWide || (QJL && s_e[16 + hd] == kWide) || s_e[32] == kWide ||
                      s_e[33] == kWide;
    a.part_l[row] = wide ? kWideSum : ldexpf(l, -sv_exp);
  }
}

// Channel d of one (batch row, head)'s attention over all tokens, in f32 on
// the vector units: for operands marked kWide, which no cache's own are
// (Lloyd-Max centroids of a unit normal, bf16 queries of common sizes). A
// wavefront: a lane a token for the scores, then a channel.
__device__ float attend_f32(const Args& a, int64_t bh, int D, int d) {
  const int lane = threadIdx.x;
  const int64_t slab = bh / a.H * a.H_kv * a.cap + bh % a.H / a.G * a.cap;
  const float *q = a.qs + bh * D, *pq = a.pq + bh * a.qm;
  float m = -INFINITY, l = 0.0f, o = 0.0f;
  for (int64_t base = 0; base < a.n; base += kWave) {
    const int cnt = a.n - base < kWave ? int(a.n - base) : kWave;
    const int64_t row = slab + base + lane;
    float x = -INFINITY;
    if (lane < cnt) {
      x = 0.0f;
      for (int i = 0; i < D; ++i) {
        const int c = a.kc[row * D + i];
        x = fmaf(q[i], c < a.n_k ? a.cent_k[c] : 0.0f, x);
      }
      x *= a.ks[row];
      if (a.ksg && a.krn[row] >= 1e-10f) {
        float c = 0.0f;
        for (int i = 0; i < a.qm; ++i)
          c += (a.ksg[row * ((a.qm + 31) / 32) + i / 32] >> (i % 32)) & 1u ? pq[i] : -pq[i];
        x = fmaf(c * (a.krn[row] * (1.2533141373155001f / sqrtf(float(a.qm)))), a.qscale, x);
      }
    }
    float mx = x;
    for (int off = 1; off < kWave; off <<= 1) mx = fmaxf(mx, __shfl_xor(mx, off, kWave));
    const float mn = fmaxf(m, mx);
    const float f = m == -INFINITY ? 0.0f : exp2f(m - mn);
    m = mn;
    const float p = lane < cnt ? exp2f(x - (mn == -INFINITY ? 0.0f : mn)) : 0.0f;
    const float w = lane < cnt ? p * a.vs[row] : 0.0f;
    float ps = p;
    for (int off = 1; off < kWave; off <<= 1) ps += __shfl_xor(ps, off, kWave);
    l = l * f + ps;
    o *= f;
    for (int t = 0; t < cnt; ++t) {
      const int c = a.vc[(slab + base + t) * D + d];
      o = fmaf(__shfl(w, t, kWave), c < a.n_v ? a.cent_v[c] : 0.0f, o);
    }
  }
  return l > 0.0f ? o / l : 0.0f;
}

// The splits of one (batch row, head) merged in the rotated basis: a thread a
// channel, every split's partial loaded with no test between (an empty
// weight is 0), so the loads issue together.
__global__ __launch_bounds__(64) void cb_merge_kernel(const Args a, int D, float* __restrict__ o) {
  __shared__ float s_w[64];
  const int64_t bh = blockIdx.x;
  const int n_splits = a.n_splits;
  const int lane = threadIdx.x;  // n_splits <= 64: a lane a split, then a channel
  const int d = int(blockIdx.y) * kWave + lane;
  const float pm = lane < n_splits ? a.part_m[bh * n_splits + lane] : -INFINITY;
  const float pl = lane < n_splits ? a.part_l[bh * n_splits + lane] : 0.0f;
  if (__any(pl == kWideSum)) {
    o[bh * D + d] = attend_f32(a, bh, D, d);
    return;
  }
  float mx = pm;
#pragma unroll
  for (int off = 1; off < kWave; off <<= 1) mx = fmaxf(mx, __shfl_xor(mx, off, kWave));
  const float w = pm != -INFINITY ? exp2f(pm - mx) : 0.0f;
  s_w[lane] = w;
  float ls = pl * w;
#pragma unroll
  for (int off = 1; off < kWave; off <<= 1) ls += __shfl_xor(ls, off, kWave);
  __syncthreads();
  float os = 0.0f;
#pragma unroll 16
  for (int s = 0; s < n_splits; ++s) os += a.part_o[(bh * n_splits + s) * D + d] * s_w[s];
  o[bh * D + d] = ls > 0.0f ? os / ls : 0.0f;
}

template <bool kRows, typename X>
void launch_matmul(const X* x, const float* M, int D, int n, int64_t rows, float scale, float* y,
                   float* ys, uint16_t* yb, hipStream_t st) {
  const dim3 grid{unsigned((rows + 15) / 16), unsigned((n + 15) / 16)};
#define TQKV_MM(DD)                                                                              \
  case DD:                                                                                       \
    hipLaunchKernelGGL((cb_matmul_kernel<DD, kRows, X>), grid, dim3(256), 0, st, x, M, n, rows,  \
                       scale, y, ys, yb);                                                        \
    break;
  switch (D) { TQKV_MM(64) TQKV_MM(128) TQKV_MM(256) TQKV_MM(512) }
#undef TQKV_MM
}

template <int D>
void launch_decode(const Args& a, dim3 grid, hipStream_t st) {
  const bool g16 = a.G == 16, qjl = a.ksg != nullptr;
  const size_t lds = size_t(g16 ? 2 : 1) * (D / 32 + (qjl ? (a.qm + 31) / 32 : 0)) * 1024;
  const bool pair = a.n_k <= 16 && a.n_v <= 16;
#define TQKV_CB(G16, QJL, PAIR)                                                                 \
  if (g16 == G16 && qjl == QJL && pair == PAIR)                                                 \
    hipLaunchKernelGGL((cb_decode_kernel<D, G16, QJL, PAIR>), grid, dim3(D), lds, st, a)
  TQKV_CB(false, false, false);
  TQKV_CB(false, false, true);
  TQKV_CB(false, true, false);
  TQKV_CB(false, true, true);
  TQKV_CB(true, false, false);
  TQKV_CB(true, false, true);
  TQKV_CB(true, true, false);
  TQKV_CB(true, true, true);
#undef TQKV_CB
}

}  // namespace
}  // namespace cb
}  // namespace tqkv

using namespace tqkv;

extern "C" size_t tqkv_decode_codebook_workspace_size(int32_t B, int32_t H, int32_t D,
                                                       int64_t total_tokens) {
  if (B <= 0 || H <= 0 || D <= 0 || total_tokens <= 0) return 0;
  // The most splits decode_codebook plans for any context up to total_tokens.
  const int64_t splits = (total_tokens + 255) / 256 < 64 ? (total_tokens + 255) / 256 : 64;
  return size_t(B) * H *
         (2 * size_t(D) + size_t(cb::kMaxQjl) + size_t(splits) * (size_t(D) + 2)) * sizeof(float);
}

namespace {
int32_t decode_codebook(const uint16_t* q, int32_t B, int32_t H, int32_t H_kv, int32_t D,
                        float scale, const float* rotation, const float* centroids_k,
                        int32_t bits_k, const float* centroids_v, int32_t bits_v,
                        const uint8_t* k_codes, const float* k_sigma, const uint32_t* k_signs,
                        const float* k_rnorm, const float* qjl, int32_t qjl_m,
                        const uint8_t* v_codes, const float* v_sigma, int64_t cap, int64_t n,
                        uint16_t* out, void* workspace, size_t workspace_bytes,
                        tqkv_stream stream, bool qjl_rotated = false) {
  if (!q || !rotation || !centroids_k || !centroids_v || !k_codes || !k_sigma || !v_codes ||
      !v_sigma || !out)
    return fail(TQKV_EINVAL_ARG, "null pointer");
  if (qjl_m != 0 && (!k_signs || !k_rnorm || !qjl || qjl_m < 0 || qjl_m > cb::kMaxQjl))
    return fail(TQKV_EINVAL_ARG, "qjl_m=%d needs signs, residual norms and the QJL matrix "
                "(m <= %d)", qjl_m, cb::kMaxQjl);
  if (B <= 0 || H <= 0 || H_kv <= 0 || H % H_kv != 0 || n <= 0 || n > cap)
    return fail(TQKV_EINVAL_SHAPE, "B=%d H=%d H_kv=%d n=%lld cap=%lld", B, H, H_kv, (long long)n,
                (long long)cap);
  if (bits_k < 1 || bits_k > 8 || bits_v < 1 || bits_v > 8)
    return fail(TQKV_EUNSUPPORTED, "bits %d/%d", bits_k, bits_v);
  // Value codes are copied 4 bytes at a time, at any alignment: what is asked
  // of their pointer is the entry's stated contract, refused as ever. Key rows
  // are read 16 bytes a load (rows of D >= 64 bytes keep that alignment).
  const int v_align = D >= 256 ? 4 : D >= 128 ? 2 : 1;
  if (reinterpret_cast<uintptr_t>(v_codes) % v_align != 0)
    return fail(TQKV_EINVAL_ARG, "v_codes must be %d-byte aligned", v_align);
  if (reinterpret_cast<uintptr_t>(k_codes) % 16 != 0)
    return fail(TQKV_EINVAL_ARG, "k_codes must be 16-byte aligned");
  const int G = H / H_kv;
  if (G > 16 || (G & (G - 1)) != 0)
    return fail(TQKV_EUNSUPPORTED, "codebook decode with %d query heads per KV head (1, 2, 4, "
                "8 or 16)", G);
  if (D != 64 && D != 128 && D != 256 && D != 512)
    return fail(TQKV_EUNSUPPORTED, "codebook decode D=%d not in {64,128,256,512}", D);
  // Splits: enough for ~4,096 wavefronts (four a SIMD; a workgroup is D / 64
  // wavefronts), never under 256 tokens a split, at most 64 (the workspace
  // size assumes no more), each a whole number of tiles.
  const int tile = D == 512 ? 128 : 64;
  const int64_t units = int64_t(B) * H_kv, waves = D / 64;
  int64_t n_splits64 = (4096 + units * waves - 1) / (units * waves);
  if (n_splits64 > (n + 255) / 256) n_splits64 = (n + 255) / 256;
  if (n_splits64 > 64) n_splits64 = 64;
  const int64_t split_len = ((n + n_splits64 - 1) / n_splits64 + tile - 1) / tile * tile;
  const int n_splits = int((n + split_len - 1) / split_len);
  const size_t need = tqkv_decode_codebook_workspace_size(B, H, D, n);
  void* ws = workspace;
  if (!ws) {
    if (int32_t rc = scratch_for_current_device(need, &ws)) return rc;
  } else if (workspace_bytes < need) {
    return fail(TQKV_EINVAL_ARG, "workspace of %zu bytes, need %zu", workspace_bytes, need);
  }
  float* qr = static_cast<float*>(ws);
  float* qsc = qr + size_t(B) * H * D;
  float* pq = qsc + size_t(B) * H * D;
  float* po = pq + size_t(B) * H * cb::kMaxQjl;
  float* pm = po + size_t(B) * H * n_splits * D;
  float* pl = pm + size_t(B) * H * n_splits;
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  const float qscale = scale * 1.4426950408889634f;
  const int64_t qrows = int64_t(B) * H;
  if (H_kv > 65535 || B > 65535)
    return fail(TQKV_EINVAL_SHAPE, "B=%d H_kv=%d: grid too large", B, H_kv);
  cb::launch_matmul<true>(q, rotation, D, D, qrows, qscale, qr, qsc, nullptr, st);
  TQKV_LAUNCHED();
  if (qjl_m > 0) {
    // Signs of the rotated residual take the rotated query, others q itself.
    if (qjl_rotated)
      cb::launch_matmul<true>(static_cast<const float*>(qr), qjl, D, qjl_m, qrows, 1.0f, pq,
                              nullptr, nullptr, st);
    else
      cb::launch_matmul<true>(q, qjl, D, qjl_m, qrows, 1.0f, pq, nullptr, nullptr, st);
    TQKV_LAUNCHED();
  }
  cb::Args a{};
  a.qs = qsc;
  a.pq = pq;
  a.kc = k_codes;
  a.ks = k_sigma;
  a.vc = v_codes;
  a.vs = v_sigma;
  a.cent_k = centroids_k;
  a.cent_v = centroids_v;
  a.ksg = qjl_m > 0 ? k_signs : nullptr;
  a.krn = k_rnorm;
  a.part_o = po;
  a.part_m = pm;
  a.part_l = pl;
  a.cap = cap;
  a.n = n;
  a.split_len = split_len;
  a.H = H;
  a.H_kv = H_kv;
  a.G = G;
  a.n_k = 1 << bits_k;
  a.n_v = 1 << bits_v;
  a.n_splits = n_splits;
  a.qm = qjl_m;
  a.qscale = qscale;
  const dim3 grid{unsigned(n_splits), unsigned(H_kv), unsigned(B)};
  switch (D) {
    case 64: cb::launch_decode<64>(a, grid, st); break;
    case 128: cb::launch_decode<128>(a, grid, st); break;
    case 256: cb::launch_decode<256>(a, grid, st); break;
    default: cb::launch_decode<512>(a, grid, st); break;
  }
  TQKV_LAUNCHED();
  // The merged rows take the rotated query's place (its last reader has run).
  hipLaunchKernelGGL(cb::cb_merge_kernel, dim3(unsigned(qrows), unsigned(D / 64)), dim3(64), 0, st,
                     a, D, qr);
  TQKV_LAUNCHED();
  cb::launch_matmul<false>(static_cast<const float*>(qr), rotation, D, D, qrows, 1.0f, nullptr,
                           nullptr, out, st);
  TQKV_LAUNCHED();
  return ok();
}
}  // namespace

extern "C" int32_t tqkv_decode_attend_codebook(
    const uint16_t* q, int32_t B, int32_t H, int32_t H_kv, int32_t D, float scale,
    const float* rotation, const float* centroids_k, int32_t bits_k, const float* centroids_v,
    int32_t bits_v, const uint8_t* k_codes, const float* k_sigma, const uint8_t* v_codes,
    const float* v_sigma, int64_t cap, int64_t n, uint16_t* out, void* workspace,
    size_t workspace_bytes, tqkv_stream stream) {
  return decode_codebook(q, B, H, H_kv, D, scale, rotation, centroids_k, bits_k, centroids_v,
                         bits_v, k_codes, k_sigma, nullptr, nullptr, nullptr, 0, v_codes, v_sigma,
                         cap, n, out, workspace, workspace_bytes, stream);
}

namespace tqkv {
// Codebook decode with QJL signs of the rotated-basis residual (a GPU-path
// cache): the score correction projects the rotated query.
int32_t decode_codebook_qjl_rotated(
    const uint16_t* q, int32_t B, int32_t H, int32_t H_kv, int32_t D, float scale,
    const float* rotation, const float* centroids_k, int32_t bits_k, const float* centroids_v,
    int32_t bits_v, const uint8_t* k_codes, const float* k_sigma, const uint32_t* k_signs,
    const float* k_rnorm, const float* qjl, int32_t qjl_m, const uint8_t* v_codes,
    const float* v_sigma, int64_t cap, int64_t n, uint16_t* out, void* workspace,
    size_t workspace_bytes, tqkv_stream stream) {
  if (qjl_m <= 0) return fail(TQKV_EINVAL_ARG, "qjl_m=%d", qjl_m);
  return decode_codebook(q, B, H, H_kv, D, scale, rotation, centroids_k, bits_k, centroids_v,
                         bits_v, k_codes, k_sigma, k_signs, k_rnorm, qjl, qjl_m, v_codes, v_sigma,
                         cap, n, out, workspace, workspace_bytes, stream, true);
}
}  // namespace tqkv

extern "C" int32_t tqkv_decode_attend_codebook_qjl(
    const uint16_t* q, int32_t B, int32_t H, int32_t H_kv, int32_t D, float scale,
    const float* rotation, const float* centroids_k, int32_t bits_k, const float* centroids_v,
    int32_t bits_v, const uint8_t* k_codes, const float* k_sigma, const uint32_t* k_signs,
    const float* k_rnorm, const float* qjl, int32_t qjl_m, const uint8_t* v_codes,
    const float* v_sigma, int64_t cap, int64_t n, uint16_t* out, void* workspace,
    size_t workspace_bytes, tqkv_stream stream) {
  if (qjl_m <= 0) return fail(TQKV_EINVAL_ARG, "qjl_m=%d", qjl_m);
  return decode_codebook(q, B, H, H_kv, D, scale, rotation, centroids_k, bits_k, centroids_v,
                         bits_v, k_codes, k_sigma, k_signs, k_rnorm, qjl, qjl_m, v_codes, v_sigma,
                         cap, n, out, workspace, workspace_bytes, stream);
}

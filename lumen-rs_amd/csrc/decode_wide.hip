// Decode attention at head dim 512 (Gemma 4's full-attention layers) over 4-
// and 8-bit affine caches: up to 16 query heads of a KV head as the columns
// of the matrix products, f16 operands as prefill_affine_kernel's f16 variant
// has them (packed f16 dequantization, one rounding), which serves the other
// widths (it stages K and V through one LDS tile at one wavefront a SIMD and
// three barriers a 64-key tile).
//
// Bound: latency at these sizes (B = 4, 32 / 2 heads, 8,179 keys of 4 bits
// are 38 MB over 256 workgroups, two tiles each), then vector issue (about
// three operations a code). So nothing is staged but what wavefronts share,
// and a tile costs one barrier: of a 128-key tile each of the eight wavefronts
// scores 16 keys over all 512 channels from registers (lane lr's key, its 32-
// code runs dequantized straight into the A operand), the scores meet in LDS,
// and each wavefront accumulates 64 output channels over the 128 keys: two
// keys' codes of a channel pair up in one packed f16 dequantization, which is
// the V^T operand, with the keys' scales and biases from LDS. A wavefront's
// accumulator is 16 registers. A tile's loads are issued a tile ahead; that
// they stay in flight over the work between takes `loaded` and `moved` below
// (without: 29.8 us at the shape above, with: 28.0).
//
// Measured, the tile kernel -> this one, a step (append, decode, merge): the
// shape above 36.9 -> 28.0 us, with 8-bit codes 43.2 -> 31.2; B = 16, 16,000
// keys 174 -> 97; one sequence of 120,000 keys (8 bits) 131 -> 74, of 257 keys
// 27.0 -> 16.4 (three splits of 128), of 21 keys 14.2 -> 13.5.
// Against 64 bits the merged rows (before the bf16 rounding) are 0.60 to 1.05
// times as far off as the tile kernel's over 48 shapes (median 0.89; 4-bit,
// 32 / 2 heads, 8,179 keys 1.97e-4 -> 1.42e-4): small weights keep their bits.
#include "prefill_affine.hpp"

namespace tqkv {
namespace prefill {
namespace {

constexpr int kD = 512, kT = 128;
constexpr int kPShift = 14;  // weights are held times 2^14 (f16 keeps 2^-24)

__device__ __forceinline__ h2_t h2(uint32_t x) { return __builtin_bit_cast(h2_t, x); }

// Keeps the compiler from moving operations on a prefetched value up to its
// load, where they would wait for it.
__device__ __forceinline__ void loaded(uint32_t& x) { asm volatile("" : "+v"(x)); }

// A pointer to device memory (the kept pointers below would otherwise be
// generic, and their loads flat).
template <typename T>
using dev = const __attribute__((address_space(1))) T*;

// p + n elements, kept in a register.
template <typename T>
__device__ __forceinline__ dev<T> moved(const T* p, int64_t n) {
  dev<T> r = (dev<T>)p + n;
  asm volatile("" : "+s"(r));
  return r;
}

// The packed f16 value pair of codes (bits of 1024 + c each) with the pairs'
// scales and biases.
__device__ __forceinline__ uint32_t dequant_pair(uint32_t x, h2_t s, h2_t b) {
  const h2_t c = h2(x) + h2_t{_Float16(-1024.0f), _Float16(-1024.0f)};  // exact
  return __builtin_bit_cast(uint32_t, __builtin_elementwise_fma(c, s, b));
}

template <int BK, int BV>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2)))
void decode_wide_kernel(const Args a) {
  static_assert((BK == 4 || BK == 8) && (BV == 4 || BV == 8), "packed f16 dequantization");
  __shared__ __attribute__((aligned(16))) uint16_t s_q[16 * 64 * 8];    // [k step][lane][8]
  __shared__ __attribute__((aligned(16))) float s_s[2][16][kT + 4];     // the tile's scores
  __shared__ __attribute__((aligned(16))) uint16_t s_vs[2][16][kT + 8]; // V scales, [group][key]
  __shared__ __attribute__((aligned(16))) uint16_t s_vb[2][16][kT + 8]; // and biases, f16
  const int tid = threadIdx.x, lane = tid % kWave, lr = lane % 16, lg = lane / 16;
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int n_hb = a.n_blocks;  // blocks of 16 heads a KV head
  const int hb = int(blockIdx.x) % n_hb, split = int(blockIdx.x) / n_hb % a.n_splits;
  const int kvh = int(blockIdx.x) / (n_hb * a.n_splits) % a.H_kv;
  const int b = int(blockIdx.x) / (n_hb * a.n_splits * a.H_kv);
  const int h0 = kvh * a.G + 16 * hb;  // first query head
  const int nh = a.G - 16 * hb < 16 ? a.G - 16 * hb : 16;
  // (The host keeps total + 128 within 31 bits.)
  const int total = int(a.total), n0 = int(a.n0);
  const int t0 = int(split * a.split_len);
  const int t1 = t0 + a.split_len < total ? t0 + int(a.split_len) : total;
  const int groups = kD / a.gs, run_shift = __builtin_ctz(a.gs / 32);  // 16, 8 or 4 groups
  // The two segments' buffers in registers: a lane's choice between them is
  // then no load from the arguments.
  // Segment 1's start n0 rows early, so that a key's index serves both
  // (formed only, never read below n0).
  const int64_t r0 = int64_t(b) * a.seg[0].b_stride + int64_t(kvh) * a.seg[0].cap;
  const int64_t r1 = int64_t(b) * a.seg[1].b_stride + int64_t(kvh) * a.seg[1].cap - n0;
  constexpr int kKw = kD * BK / 32, kVw = kD * BV / 32;
  const dev<uint32_t> kw0 = moved(a.seg[0].kw, r0 * kKw), kw1 = moved(a.seg[1].kw, r1 * kKw);
  const dev<uint32_t> vw0 = moved(a.seg[0].vw, r0 * kVw), vw1 = moved(a.seg[1].vw, r1 * kVw);
  const dev<uint16_t> ks0 = moved(a.seg[0].ks, r0 * groups), ks1 = moved(a.seg[1].ks, r1 * groups);
  const dev<uint16_t> kb0 = moved(a.seg[0].kb, r0 * groups), kb1 = moved(a.seg[1].kb, r1 * groups);
  const dev<uint16_t> vs0 = moved(a.seg[0].vs, r0 * groups), vs1 = moved(a.seg[1].vs, r1 * groups);
  const dev<uint16_t> vb0 = moved(a.seg[0].vb, r0 * groups), vb1 = moved(a.seg[1].vb, r1 * groups);

  // Loads of the tile at `base`; keys past the range re-read its last one
  // (masked in the scores).
  uint32_t kw[4][BK];  // runs 4 u + lg of key 16 wave + lr
  uint32_t ks[4], kb[4];
  auto load_k = [&](int base) __attribute__((always_inline)) {
    const int k = base + 16 * wave + lr, kk = k < t1 ? k : t1 - 1;
    const bool first = kk < n0;
    const dev<uint32_t> w = (first ? kw0 : kw1) + int64_t(kk) * kKw + lg * BK;
    const dev<uint16_t> sc = (first ? ks0 : ks1) + int64_t(kk) * groups;
    const dev<uint16_t> bi = (first ? kb0 : kb1) + int64_t(kk) * groups;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
#pragma unroll
      for (int i = 0; i < BK; i += 4) {
        const u32x4_t x = *(dev<u32x4_t>)(w + 4 * u * BK + i);
        kw[u][i] = x.x, kw[u][i + 1] = x.y, kw[u][i + 2] = x.z, kw[u][i + 3] = x.w;
      }
      const int g = (4 * u + lg) >> run_shift;
      ks[u] = sc[g];
      kb[u] = bi[g];
    }
  };
  // Keys 32 u + 4 lg + i and 32 u + 16 + 4 lg + i (the weight operand's k
  // slots), channels 64 wave + 4 lr + [0, 4): BV / 2 bytes a key.
  using chunk_t = std::conditional_t<BV == 4, uint16_t, uint32_t>;
  uint32_t vw[32];
  auto load_v = [&](int base) __attribute__((always_inline)) {
    constexpr int kRow = kD * BV / 8;  // bytes a key
    const int lane_off = 8 * BV * wave + lr * (BV / 2);
    const bool in0 = base + kT <= n0;
    if (__builtin_amdgcn_readfirstlane(base + kT <= t1 && (in0 || base >= n0))) {
      const dev<char> w = (dev<char>)(in0 ? vw0 : vw1) + int64_t(base) * kRow;
      const uint32_t lane_row = 4 * lg * kRow + lane_off;
#pragma unroll
      for (int i = 0; i < 8; ++i)  // a uniform base, one lane offset, a constant
#pragma unroll
        for (int r = 0; r < 4; ++r)
          vw[4 * i + r] = *(dev<chunk_t>)(w + 16 * i * kRow + lane_row + r * kRow);
    } else {
      int k = base + 4 * lg;
#pragma unroll
      for (int i = 0; i < 32; ++i) {
        const int kk = k < t1 ? k : t1 - 1;
        vw[i] = *(dev<chunk_t>)((dev<char>)(kk < n0 ? vw0 : vw1) + int64_t(kk) * kRow + lane_off);
        k += i % 4 == 3 ? 13 : 1;
        if (i % 4 == 3) __builtin_amdgcn_sched_barrier(0);  // few addresses live at a time
      }
    }
  };
  // The tile's V scales and biases: four groups of key tid / 4 a thread, the
  // same again where a key has fewer than 16.
  uint32_t vs[4], vb[4];
  const int gmask = groups - 1, g0 = 4 * (tid % 4);
  auto load_scales = [&](int base) __attribute__((always_inline)) {
    const int k = base + tid / 4, kk = k < t1 ? k : t1 - 1;
    const bool first = kk < n0;
    const dev<uint16_t> sc = (first ? vs0 : vs1) + int64_t(kk) * groups;
    const dev<uint16_t> bi = (first ? vb0 : vb1) + int64_t(kk) * groups;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      vs[j] = sc[(g0 + j) & gmask];
      vb[j] = bi[(g0 + j) & gmask];
    }
  };
  load_scales(t0);
  load_k(t0);
  load_v(t0);
  // The query: block i = 4 rho + e of 8 channels sits in k step 4 (rho / 4) +
  // e at lane group rho % 4. Columns past the heads are zeros.
  for (int i = tid; i < 16 * 64; i += 512) {
    const int h = i / 64, blk = i % 64, rho = blk / 4, e = blk % 4;
    h8_t v = {0, 0, 0, 0, 0, 0, 0, 0};
    if (h < nh) {
      const uint16_t* src = a.q + int64_t(b) * a.qs_b + int64_t(h0 + h) * a.qs_h + 8 * blk;
#pragma unroll
      for (int k = 0; k < 8; ++k) v[k] = _Float16(bf16_to_f32(src[k]));
    }
    reinterpret_cast<h8_t*>(s_q)[(4 * (rho / 4) + e) * kWave + 16 * (rho % 4) + h] = v;
  }
  __syncthreads();

  float m = -INFINITY, l = 0.0f;
  f4_t o[4];  // channels 64 wave + 4 (4 lg + r) + j of head lr
#pragma unroll
  for (int j = 0; j < 4; ++j) o[j] = f4_t{0.0f, 0.0f, 0.0f, 0.0f};
  const int vg = (64 * wave + 4 * lr) / a.gs;  // this lane's V group
  int buf = 0;
  for (int base = t0; base < t1; base += kT, buf ^= 1) {
    const int next = base + kT < t1 ? base + kT : base;  // (the last tile re-loads itself)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      loaded(vs[j]);
      loaded(vb[j]);
      const int g = (g0 + j) & gmask;
      s_vs[buf][g][tid / 4] = __builtin_bit_cast(uint16_t, _Float16(__uint_as_float(vs[j] << 16)));
      s_vb[buf][g][tid / 4] = __builtin_bit_cast(uint16_t, _Float16(__uint_as_float(vb[j] << 16)));
    }
    f4_t sc0 = {0.0f, 0.0f, 0.0f, 0.0f}, sc1 = sc0;  // two chains of products
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      loaded(ks[u]);
      loaded(kb[u]);
      uint32_t w[16];
      dequant_run<BK, true>(kw[u], ks[u] | kb[u] << 16, w);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const h8_t ka = __builtin_bit_cast(h8_t, u32x4_t{w[4 * e], w[4 * e + 1], w[4 * e + 2], w[4 * e + 3]});
        const h8_t qb = reinterpret_cast<const h8_t*>(s_q)[(4 * u + e) * kWave + lane];
        if (e % 2)
          sc1 = mma<true>(ka, qb, sc1);
        else
          sc0 = mma<true>(ka, qb, sc0);
      }
    }
    f4_t x = (sc0 + sc1) * a.qscale;
#pragma unroll
    for (int r = 0; r < 4; ++r)
      if (base + 16 * wave + 4 * lg + r >= t1) x[r] = -INFINITY;
    *reinterpret_cast<f4_t*>(&s_s[buf][lr][16 * wave + 4 * lg]) = x;
    load_scales(next);
    load_k(next);
    // One barrier a tile: a buffer is written again two tiles on, after the
    // next tile's barrier, which every wavefront reaches past its reads here.
    __syncthreads();
    f4_t s[8];
    float mx = -INFINITY;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      s[i] = *reinterpret_cast<const f4_t*>(&s_s[buf][lr][16 * i + 4 * lg]);
#pragma unroll
      for (int r = 0; r < 4; ++r) mx = fmaxf(mx, s[i][r]);
    }
    mx = xor32_max(xor16_max(mx));
    const float mn = fmaxf(m, mx);
    const float f = m == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(m - mn);
    m = mn;
    l *= f;
#pragma unroll
    for (int j = 0; j < 4; ++j) o[j] *= f;
    const float off = (mn == -INFINITY ? 0.0f : mn) - float(kPShift);
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      float p[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) p[i] = __builtin_amdgcn_exp2f(s[2 * u + i / 4][i % 4] - off);
      const u32x4_t w = {pack_h16(p[0], p[1]), pack_h16(p[2], p[3]), pack_h16(p[4], p[5]),
                         pack_h16(p[6], p[7])};
#pragma unroll
      for (int i = 0; i < 8; ++i) loaded(vw[8 * u + i]);
      const h8_t pw = __builtin_bit_cast(h8_t, w);
      // The sum counts the weights as rounded for the matrix cores.
#pragma unroll
      for (int e = 0; e < 4; ++e) l = sum2<true>(w[e], l);
      u32x2_t sp[2], bp[2];  // scales and biases of the lane's eight keys
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        sp[h] = *reinterpret_cast<const u32x2_t*>(&s_vs[buf][vg][32 * u + 16 * h + 4 * lg]);
        bp[h] = *reinterpret_cast<const u32x2_t*>(&s_vb[buf][vg][32 * u + 16 * h + 4 * lg]);
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        u32x4_t v;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          const uint32_t w0 = vw[8 * u + 2 * k], w1 = vw[8 * u + 2 * k + 1];
          uint32_t c;
          if constexpr (BV == 4)
            c = ((w0 | w1 << 16) >> (4 * j)) & 0x000f000fu;
          else
            c = __builtin_amdgcn_perm(w1, w0, 0x0c040c00u + uint32_t(j) * 0x00010001u);
          v[k] = dequant_pair(c | 0x64006400u, h2(sp[k / 2][k % 2]), h2(bp[k / 2][k % 2]));
        }
        o[j] = mma<true>(__builtin_bit_cast(h8_t, v), pw, o[j]);
      }
    }
    load_v(next);
  }
  l = xor32_sum(xor16_sum(l));
  if (lr >= nh) return;
  const int c0 = 64 * wave + 16 * lg;
  if (a.part_o) {
    constexpr float kDown = 1.0f / float(1 << kPShift);
    const int64_t slot = (int64_t(b) * a.H + h0 + lr) * a.n_part + a.split_base + split;
#pragma unroll
    for (int r = 0; r < 4; ++r)
      *reinterpret_cast<f4_t*>(a.part_o + slot * kD + c0 + 4 * r) =
          f4_t{o[0][r], o[1][r], o[2][r], o[3][r]} * kDown;
    if (wave == 0 && lg == 0) {
      a.part_m[slot] = m;
      a.part_l[slot] = l * kDown;
    }
  } else {
    const float inv = l > 0.0f ? 1.0f / l : 0.0f;
    uint16_t* dst = a.out + int64_t(b) * a.qs_b + int64_t(h0 + lr) * a.qs_h + c0;
#pragma unroll
    for (int r = 0; r < 4; ++r)
      *reinterpret_cast<u32x2_t*>(dst + 4 * r) =
          u32x2_t{pack_bf16(o[0][r] * inv, o[1][r] * inv), pack_bf16(o[2][r] * inv, o[3][r] * inv)};
  }
}

}  // namespace

KernelFn pick_decode_wide(int bk, int bv) {
  if (bk == 4 && bv == 4) return decode_wide_kernel<4, 4>;
  if (bk == 4 && bv == 8) return decode_wide_kernel<4, 8>;
  if (bk == 8 && bv == 4) return decode_wide_kernel<8, 4>;
  if (bk == 8 && bv == 8) return decode_wide_kernel<8, 8>;
  return nullptr;
}

}  // namespace prefill
}  // namespace tqkv

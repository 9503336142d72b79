// Prefill-chunk attention at head dims 256 and 512 over keys dequantized
// beforehand: K as bf16 rows, V as transposed tiles of f16 operands (width
// kPreF16T). The results are prefill_affine_kernel's bit for bit
// (prefill_affine.hpp: the same products in the same order, the same 64-key
// steps of the running maximum); this is its shape for wide heads.
//
// Bound: no unit is full. Each wavefront holds 16 query rows (Q, O and a
// tile's scores then fit 256 registers at D = 512), so a K or V operand read
// (1 KB, 4 LDS cycles) feeds one product (16 cycles on one of four SIMDs): the
// matrix cores and the LDS are each busy 60% of the kernel's cycles at D = 512
// and 39% at D = 256 (counters), the vector units 30 and 34%. The rest is the
// two wavefronts of a SIMD in the same phase (products, then softmax, then the
// tile's barrier), and the clock, which the card holds at 1.84 GHz (D = 512)
// and 2.07 (D = 256) of 2.4 under this load. So nothing else may stall:
// the tiles go from HBM (mostly L2: the blocks of a KV head share an XCD)
// straight into LDS, 16-byte chunks permuted within their rows so that every
// operand read is free of bank conflicts (counter: 0), with no staging
// registers; and no register spills (what depends on the lane alone is
// recomputed a tile, see lane_now). The kernel before it staged tiles through
// registers: at D = 512 that took one wavefront a SIMD and 110 spilled registers.
// 32 rows a wavefront (half the LDS reads) measured 193 against 197 us at D
// = 256 (sliding chunk, 2 x 32 heads, 3,071 keys) and needs twice the chunk
// to fill the chip; at D = 512 it spills.
// Measured: 32 / 2 heads, D = 512, 2,048 rows over 8,192 keys 4.30 -> 0.84
// ms (1.14 PFLOP/s); 16 / 8 heads, D = 256, 2,048 rows over 16,384 keys 0.61
// -> 0.53 ms; the sliding chunk above 229 -> 197 us.
#include "prefill_affine.hpp"

namespace tqkv {
namespace prefill {
namespace {

// lds_dma16 from a uniform base plus a 32-bit lane offset.
__device__ __forceinline__ void lds_dma16_at(const char* base, uint32_t off, uint32_t lds) {
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(off), "s"(base),
               "s"(lds)
               : "memory", "m0");
#pragma clang diagnostic pop
}

// The lane's index, computed anew at each use: what depends on it (operand
// and load addresses) is then recomputed a tile instead of held in registers
// across the tile loop, which has none to spare (at D = 512 holding them
// measured 1.19 against 0.85 ms).
__device__ __forceinline__ uint32_t lane_now() {
  uint32_t l;
  asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=v"(l));
  return l;
}

template <int D, int kWaves>
__global__ __launch_bounds__(64 * kWaves) __attribute__((amdgpu_waves_per_eu(kWaves / 4)))
void prefill_wide_kernel(const Args a) {
  constexpr int ND = D / 32, NT = D / 16;
  constexpr int kRows = 16 * kWaves;
  constexpr int kAhead = 6;                            // operand reads in flight
  constexpr int kTileBytes = kTile * D * 2;            // of K, and of V
  constexpr int kPieces = kTileBytes / 1024 / kWaves;  // 1 KB loads a wavefront, K and V each
  // Two buffers of each at D = 256. One at D = 512 (two would pass the 160 KB
  // of LDS): the next K loads while P V runs, the next V while the scores do.
  constexpr int kNB = D == 256 ? 2 : 1;
  __shared__ __attribute__((aligned(1024))) unsigned char s_mem[2 * kNB * kTileBytes];
  __shared__ int s_ql[kRows];  // each row's position in the chunk

  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int lane = tid % kWave, lr = lane % 16, lg = lane / 16;
  const int n_wg = int(gridDim.x);
  int lin = int(blockIdx.x);
  if (n_wg % kXcds == 0) lin = (lin % kXcds) * (n_wg / kXcds) + lin / kXcds;
  const int per_unit = a.n_blocks * a.n_splits;
  const int blk = a.n_blocks - 1 - lin % a.n_blocks;
  const int split = (lin % per_unit) / a.n_blocks;
  const int kvh = (lin / per_unit) % a.H_kv, b = lin / (per_unit * a.H_kv);
  const int64_t rows = int64_t(a.L) * a.G;
  const int64_t row0 = int64_t(blk) * kRows;
  const int64_t row_end = row0 + kRows < rows ? row0 + kRows : rows;
  const int64_t qa_lo = a.q_start + row0 / a.G, qa_hi = a.q_start + (row_end - 1) / a.G;
  int64_t kk_lo = a.split_lo + int64_t(split) * a.split_len, kk_hi = a.total - 1;
  if (kk_lo + a.split_len - 1 < kk_hi) kk_hi = kk_lo + a.split_len - 1;
  if (a.causal) {
    if (qa_hi - a.k_start < kk_hi) kk_hi = qa_hi - a.k_start;
    if (a.window >= 0 && qa_lo - a.window + 1 - a.k_start > kk_lo)
      kk_lo = qa_lo - a.window + 1 - a.k_start;
  }

  // This lane's row: row0 + 16 wave + lr of the flattened (position, head)
  // rows (past the end: the last row, not written).
  auto orow_of = [&](int64_t r) __attribute__((always_inline)) {
    const int64_t rr = r < rows ? r : rows - 1;
    const int64_t l = rr / a.G, g = rr % a.G;
    return int64_t(b) * a.qs_b + (int64_t(kvh) * a.G + g) * a.qs_h + l * a.qs_l;
  };
  bf8_t qf[ND];
  {
    const int64_t r = row0 + 16 * wave + lr;
    if (lg == 0) s_ql[16 * wave + lr] = int((r < rows ? r : rows - 1) / a.G);
    const uint16_t* src = a.q + orow_of(r) + 8 * lg;
#pragma unroll
    for (int s = 0; s < ND; ++s) qf[s] = *reinterpret_cast<const bf8_t*>(src + 32 * s);
  }
  float m = -INFINITY, nm = 0.0f, thr = -INFINITY, lsum = 0.0f;
  f4_t o[NT];
  const float iqs = 1.0f / a.qscale;
#pragma unroll
  for (int t = 0; t < NT; ++t) o[t] = f4_t{0.0f, 0.0f, 0.0f, 0.0f};

  if (kk_lo <= kk_hi) {
    const int t_lo = int(kk_lo / kTile), t_hi = int(kk_hi / kTile);
    const int64_t slab = (int64_t(b) * a.H_kv + kvh) * a.seg[0].cap;
    const char* kg = reinterpret_cast<const char*>(a.seg[0].kw) + slab * (D * 2);
    const char* vg = reinterpret_cast<const char*>(a.seg[0].vw) + slab * (D * 2);
    // LDS: K buffers, then V buffers. A K row keeps its 16-byte chunk c at
    // position c ^ 2 (row mod 16) (rows of 512 or 1,024 bytes: 16 rows x 2
    // chunks, a half-wavefront's read, then fall in distinct banks); V^T row
    // R (64 bytes) its chunk c at vt_chunk_pos(R, c).
    const uint32_t lds = lds_addr(s_mem);
    // This wavefront's pieces of a tile: its 1 KB pieces p = kPieces wave + i.
    // A lane's source offset within K's piece p is (its chunk at permutation
    // 0) ^ (p's share of the permutation); V^T's is the same for every piece.
    // Rows of the last tile past the last key are whatever the slab's padding
    // holds: their scores are masked, and V^T is zero there.
    constexpr int kPieceRows = 512 / D;  // K rows a piece
    auto dma_k = [&](int t, int buf) __attribute__((always_inline)) {
      const uint32_t base = __builtin_amdgcn_readfirstlane(lds + uint32_t(buf) * kTileBytes);
      const char* src = kg + size_t(t < t_hi ? t : t_hi) * kTileBytes;
      const uint32_t l = lane_now(), row = l / (D / 8);
      const uint32_t koff = row * (D * 2) + 16 * ((l % (D / 8)) ^ (2 * row));
#pragma unroll
      for (int i = 0; i < kPieces; ++i) {
        const uint32_t p = uint32_t(kPieces * wave + i);
        const uint32_t perm = 32 * (kPieceRows * p % 16);
        lds_dma16_at(src + p * 1024, koff ^ perm, base + p * 1024);
      }
    };
    auto dma_v = [&](int t, int buf) __attribute__((always_inline)) {
      const uint32_t base = __builtin_amdgcn_readfirstlane(lds + uint32_t(kNB + buf) * kTileBytes);
      const char* src = vg + size_t(t < t_hi ? t : t_hi) * kTileBytes;
      const uint32_t l = lane_now();
      const uint32_t voff = l / 4 * 64 + 16 * vt_chunk_pos(l / 4, l % 4);
#pragma unroll
      for (int i = 0; i < kPieces; ++i) {
        const uint32_t p = uint32_t(kPieces * wave + i);
        lds_dma16_at(src + p * 1024, voff, base + p * 1024);
      }
    };

    __builtin_amdgcn_s_waitcnt(0x0F70);  // the Q fragments have landed
    dma_k(t_lo, 0);
    dma_v(t_lo, 0);
    __builtin_amdgcn_s_waitcnt(0x0F70);
    __syncthreads();
    int cur = 0;
    for (int t = t_lo; t <= t_hi; ++t, cur ^= kNB - 1) {
      if constexpr (kNB == 2) {  // over tile t - 1's, read before the barrier that ended it
        dma_k(t + 1, cur ^ 1);
        dma_v(t + 1, cur ^ 1);
      }
      // S^T of the tile: K chunk 4 s + lg of row 16 i + lr at kc ^ 64 s for
      // s < 8 (+ 512 bytes beyond).
      f4_t sc[4];
      {
        const unsigned char* kb = s_mem + cur * kTileBytes;
        const uint32_t l = lane_now();
        const uint32_t kc = l % 16 * (D * 2) + 16 * ((l / 16) ^ (2 * (l % 16)));
#pragma unroll
        for (int i = 0; i < 4; ++i) sc[i] = f4_t{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int s = 0; s < ND; ++s)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const bf8_t ka = *reinterpret_cast<const bf8_t*>(kb + (kc ^ (64 * (s % 8))) +
                                                             (s / 8) * 512 + i * 16 * D * 2);
            sc[i] = mma<false>(ka, qf[s], sc[i]);
          }
        // The order for the scheduler: kAhead operand reads first, then one
        // after every product.
        __builtin_amdgcn_sched_group_barrier(0x100, kAhead, 0);
#pragma unroll
        for (int k = 0; k < 4 * ND - kAhead; ++k) {
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
          __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        }
        __builtin_amdgcn_sched_group_barrier(0x008, kAhead, 0);
        __builtin_amdgcn_sched_barrier(0);
      }
      if constexpr (kNB == 1) {
        __builtin_amdgcn_s_waitcnt(0x0F70);  // this wavefront's part of V t is in LDS
        __syncthreads();                     // K t has been read
        dma_k(t + 1, 0);
      }
      // Mask: only where some row of the block sees the tile in part.
      const int64_t kbase = a.k_start + int64_t(t) * kTile;
      const int rem = a.total - int64_t(t) * kTile < kTile ? int(a.total - int64_t(t) * kTile) : kTile;
      const bool full = rem == kTile &&
                        (!a.causal || (kbase + kTile - 1 <= qa_lo &&
                                       (a.window < 0 || qa_hi < kbase + a.window)));
      if (!full) {
        keep_branch();
        const int l = int(lane_now());
        int hi = rem - 1, lo = 0;
        if (a.causal) {
          const int64_t dq = a.q_start + s_ql[16 * wave + l % 16] - kbase;
          if (dq < hi) hi = dq < -1 ? -1 : int(dq);
          if (a.window >= 0) {
            const int64_t first = dq - a.window + 1;
            lo = first < 0 ? 0 : (first > kTile ? kTile : int(first));
          }
        }
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int off = 16 * i + 4 * (l / 16) + r;
            if (off < lo || off > hi) sc[i][r] = -INFINITY;
          }
      }
      // The running maximum may lag by up to kTau (see prefill_affine.hpp).
      float mx = -INFINITY;
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) mx = fmaxf(mx, sc[i][r]);
      if (__any(mx > thr)) {
        keep_branch();
        mx = xor32_max(xor16_max(mx));
        const bool up = mx > thr;
        const float mn = up ? mx * a.qscale : m;
        const float alpha = up ? __builtin_amdgcn_exp2f(m - mn) : 1.0f;
        lsum *= alpha;
#pragma unroll
        for (int t2 = 0; t2 < NT; ++t2) o[t2] *= alpha;
        m = mn;
        nm = mn == -INFINITY ? 0.0f : -mn;
        thr = (mn + kTau) * iqs;
      }
      // The weights, 32 keys at a time, and their P V.
      {
        const unsigned char* vb = s_mem + (kNB + cur) * kTileBytes;
        const uint32_t l = lane_now();  // V^T chunk lg of row 16 t2 + lr
        const uint32_t vco = l % 16 * 64 + 16 * vt_chunk_pos(l % 16, l / 16);
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          float p[8];
#pragma unroll
          for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int r = 0; r < 4; ++r)
              p[4 * i + r] = __builtin_amdgcn_exp2f(__builtin_fmaf(sc[2 * u + i][r], a.qscale, nm));
          const u32x4_t w = {pack_h16(p[0], p[1]), pack_h16(p[2], p[3]), pack_h16(p[4], p[5]),
                             pack_h16(p[6], p[7])};
          const h8_t pp = __builtin_bit_cast(h8_t, w);
          // The row sum counts the weights as rounded for the matrix cores.
#pragma unroll
          for (int e = 0; e < 4; ++e) lsum = sum2<true>(w[e], lsum);
#pragma unroll
          for (int t2 = 0; t2 < NT; ++t2) {
            const h8_t va = *reinterpret_cast<const h8_t*>(vb + vco + u * (D * 64) + t2 * 1024);
            o[t2] = mma<true>(va, pp, o[t2]);
          }
          __builtin_amdgcn_sched_group_barrier(0x100, kAhead, 0);
#pragma unroll
          for (int k = 0; k < NT - kAhead; ++k) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
          }
          __builtin_amdgcn_sched_group_barrier(0x008, kAhead, 0);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
      __builtin_amdgcn_s_waitcnt(0x0F70);  // this wavefront's part of the next tile is in LDS
      __syncthreads();
      if constexpr (kNB == 1) dma_v(t + 1, 0);  // V t has been read
    }
    __builtin_amdgcn_s_waitcnt(0x0F70);  // the last re-loads land before the LDS is released
  }
  const int le = int(lane_now());
  const float tot = xor32_sum(xor16_sum(lsum));
  const int64_t r = row0 + 16 * wave + le % 16;
  if (r >= rows) return;
  const int c0 = 4 * (le / 16);
  if (a.part_o) {  // (V was scaled by 2^-kVShift)
    const int64_t l = r / a.G, h = int64_t(kvh) * a.G + r % a.G;
    const int64_t slot = ((int64_t(b) * a.L + l) * a.H + h) * a.n_part + a.split_base + split;
    float* po = a.part_o + slot * D + c0;
#pragma unroll
    for (int t2 = 0; t2 < NT; ++t2) *reinterpret_cast<f4_t*>(po + 16 * t2) = o[t2] * kVUp;
    if (le < 16) {
      a.part_m[slot] = m;
      a.part_l[slot] = tot;
    }
  } else {
    const float inv = tot > 0.0f ? kVUp / tot : 0.0f;
    uint16_t* dst = a.out + orow_of(r) + c0;
#pragma unroll
    for (int t2 = 0; t2 < NT; ++t2) {
      const f4_t v = o[t2] * inv;
      *reinterpret_cast<u32x2_t*>(dst + 16 * t2) =
          u32x2_t{pack_bf16(v[0], v[1]), pack_bf16(v[2], v[3])};
    }
  }
}

}  // namespace

// 128 rows a workgroup, or 64 (a block's tiles take half the LDS time).
KernelFn pick_wide(int D, int rows) {
  if (D == 256) return rows == 128 ? prefill_wide_kernel<256, 8> : prefill_wide_kernel<256, 4>;
  if (D == 512) return rows == 128 ? prefill_wide_kernel<512, 8> : prefill_wide_kernel<512, 4>;
  return nullptr;
}

}  // namespace prefill
}  // namespace tqkv

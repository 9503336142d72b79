// Host side of the affine prefill-chunk attention: argument checks, the
// kernel choice and the launch. The kernel and its design notes are in
// prefill_affine.hpp.
#include <cmath>
#include <cstdlib>
#include <cstring>

#include "prefill_affine.hpp"
#include "prefill_plan.hpp"

namespace tqkv {
namespace prefill {
namespace {

static_assert(kTile == prefillplan::kTileKeys, "whole tiles a split");

bool valid_bits(int bits) {
  return bits == 2 || bits == 3 || bits == 4 || bits == 5 || bits == 6 || bits == 8;
}

KernelFn pick(int D, int bk, int bv, bool h16 = false) {
  switch (D) {
    case 64: return pick_d64(bk, bv, h16);
    case 128: return pick_d128(bk, bv, h16);
    case 256: return pick_d256(bk, bv, h16);
    case 512: return pick_d512(bk, bv, h16);
  }
  return nullptr;
}

// Dequantize-once: keys [0, total) of every (batch row, KV head) (of segments
// that start at the first visible tile, see keys_from), K into kd
// as bf16 rows [B * H_kv, slab_rows, D] with mlx::dequantize's arithmetic
// (bf16(fma(scale, code, bias)), one rounding), V into vd as the prefill
// kernel's V operands (those bf16 values times 2^-kVShift, in f16; see
// v_operand_run): rows like K, or with vt (D >= 128) transposed key tiles
// (width kPreF16T; slab_rows a multiple of 64, zeros past the last key).
// Grid: (row-run chunks, slab, K and/or V); a thread takes one run of 32
// values of one row: its BITS words in one or two wide loads, its group's
// scale and bias (a run never straddles a group: gs is a multiple of 32).
// A wavefront's 64 runs are 4 KB of consecutive rows; they pass through LDS
// so that each of the wavefront's four 16-byte store instructions writes 1
// KB contiguously (measured on MI355X: 64-byte strided 16-byte stores reach
// 3.5 TB/s, contiguous ones 7.0). A V^T tile is a workgroup's 256 runs (64
// keys at D = 128), transposed through LDS with the transposing read, its
// 16 KB written 1 KB a store instruction. kinds: 1 = K, 2 = V, 3 = both
// (blockIdx.z picks). Keys [0, n0) come from segment 0, the rest from
// segment 1.
template <int D, int BITS>
__global__ __launch_bounds__(256) void dequantize_rows_kernel(const Args a, int kinds,
                                                              int64_t slab_rows, int vt,
                                                              uint16_t* kd, uint16_t* vd) {
  constexpr int kRuns = D / 32;
  static_assert(64 % kRuns == 0, "a wavefront covers whole rows");
  constexpr int kChunkRows = D / 8;  // 16-byte chunks a row
  // A V^T workgroup's channels and keys, and its row stride in LDS.
  constexpr int kVtCh = D == 128 ? 128 : 256, kVtKeys = 8192 / kVtCh;
  constexpr int KSTR = kKStride<kVtCh>;
  // A wavefront's 64 runs x 4 chunks each (rows), or the workgroup's keys
  // row-major (V^T).
  constexpr int kLds = D >= 128 ? kVtKeys * KSTR / 8 : 1024;
  __shared__ uint4 s_buf[kLds];
  const int wv = threadIdx.x / 64, l = threadIdx.x % 64;
  const uint32_t j = blockIdx.x * 256u + threadIdx.x;
  const uint32_t total = uint32_t(a.total);
  if (total == 0) return;  // (uniform: no wavefront reaches the exchange)
  const int slab = int(blockIdx.y), bb = slab / a.H_kv, kv = slab % a.H_kv;
  const bool isv = kinds == 3 ? blockIdx.z != 0 : kinds == 2;
  uint32_t row = j / kRuns;
  int run = int(j % kRuns);
  constexpr int kVtRuns = kVtCh / 32;           // runs of a key a V^T workgroup takes
  constexpr int kVtParts = D >= 128 ? D / kVtCh : 1;  // V^T workgroups a key block
  if (D > kVtCh && isv && vt) {  // channel part blockIdx.x % kVtParts of its keys
    row = blockIdx.x / kVtParts * kVtKeys + threadIdx.x / kVtRuns;
    run = int(blockIdx.x % kVtParts) * kVtRuns + int(threadIdx.x % kVtRuns);
  }
  const uint32_t lrow = row < total ? row : total - 1;  // past the end: load a live row
  const bool first = lrow < uint32_t(a.n0);
  const Seg& s = a.seg[first ? 0 : 1];
  const int64_t src = int64_t(bb) * s.b_stride + int64_t(kv) * s.cap +
                      (first ? lrow : lrow - uint32_t(a.n0));
  const uint32_t* pw = (isv ? s.vw : s.kw) + src * (D * BITS / 32) + run * BITS;
  const int64_t g = src * (D / a.gs) + (run * 32) / a.gs;
  const uint32_t sb = uint32_t((isv ? s.vs : s.ks)[g]) | (uint32_t((isv ? s.vb : s.kb)[g]) << 16);
  uint32_t w[BITS], out[16];
  load_words<BITS>(w, pw);
  if (isv)
    v_operand_run<BITS>(w, sb, out);
  else
    dequant_run<BITS, false>(w, sb, out);
  if constexpr (D >= 128) {
    if (isv && vt) {  // (block-uniform)
      // Keys past the end are zeros: their weights are exactly 0, and 0
      // times a zero operand stays 0.
      const int key = int(threadIdx.x) / kVtRuns, ch = int(threadIdx.x) % kVtRuns * 32;
      uint4* d = reinterpret_cast<uint4*>(reinterpret_cast<uint16_t*>(s_buf) + key * KSTR + ch);
#pragma unroll
      for (int i = 0; i < 4; ++i)
        d[i] = row < total ? uint4{out[4 * i], out[4 * i + 1], out[4 * i + 2], out[4 * i + 3]}
                           : uint4{0u, 0u, 0u, 0u};
      __syncthreads();
      // Store pass (u, tt) of wavefront wv: lane (grp, lr) takes channel
      // 16 tt + lr of keys 32 u + 4 grp + [0, 4) and 32 u + 16 + 4 grp +
      // [0, 4) (two transposing reads), the 16 bytes at slot 8 grp of that
      // channel's row in 32-key block u; the wavefront's 64 chunks are 16
      // whole rows.
      const int grp = l / 16, lr = l % 16;
      const int c0 = int(blockIdx.x % kVtParts) * kVtCh;
      uint4* tile = reinterpret_cast<uint4*>(
          vd + (int64_t(slab) * slab_rows + int64_t(blockIdx.x / kVtParts) * kVtKeys) * D);
      const uint16_t* sv = reinterpret_cast<const uint16_t*>(s_buf);
      constexpr int kTt = kVtCh / 16;
#pragma unroll
      for (int it = 0; it < 4; ++it) {
        const int pass = 4 * wv + it, u = pass / kTt, tt = pass % kTt;
        const uint16_t* vrow = sv + (32 * u + 4 * grp + lr / 4) * KSTR + 16 * tt + 4 * (lr % 4);
        const u32x2_t lo = tr_read(vrow);
        const u32x2_t hi = tr_read(vrow + 16 * KSTR);
        tile[(u * D + c0 + 16 * tt + lr) * 4 + grp] = uint4{lo.x, lo.y, hi.x, hi.y};
      }
      return;
    }
  }
  // Lane l's run is chunks 4 l .. 4 l + 3 of the wavefront's block; store i
  // of lane l writes chunk 64 i + l. The exchange stays inside one
  // wavefront, so a wavefront-scope fence orders it (no workgroup barrier).
  uint4* s_t = s_buf + 256 * wv;
#pragma unroll
  for (int i = 0; i < 4; ++i)
    s_t[4 * l + i] = uint4{out[4 * i], out[4 * i + 1], out[4 * i + 2], out[4 * i + 3]};
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  const uint32_t row0 = (blockIdx.x * 256u + wv * 64u) / kRuns;
  uint4* d = reinterpret_cast<uint4*>((isv ? vd : kd) + (int64_t(slab) * slab_rows + row0) * D);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int c = 64 * i + l;
    if (row0 + uint32_t(c / kChunkRows) < total) d[c] = s_t[c];
  }
}

template <int D>
void launch_dequantize_rows(const Args& a, int bits, int kinds, int64_t slab_rows, int vt,
                            dim3 grid, hipStream_t st, uint16_t* kd, uint16_t* vd) {
#define TQKV_DQ(B)                                                                            \
  hipLaunchKernelGGL((dequantize_rows_kernel<D, B>), grid, dim3(256), 0, st, a, kinds, slab_rows, \
                     vt, kd, vd)
  switch (bits) {
    case 2: TQKV_DQ(2); break;
    case 3: TQKV_DQ(3); break;
    case 4: TQKV_DQ(4); break;
    case 5: TQKV_DQ(5); break;
    case 6: TQKV_DQ(6); break;
    default: TQKV_DQ(8); break;
  }
#undef TQKV_DQ
}

// a's keys [lo, lo + keys) alone: its segments start at key lo.
Args keys_from(const Args& a, int D, int bk, int bv, int64_t lo, int64_t keys) {
  Args k = a;
  const int i = lo < a.n0 ? 0 : 1;
  const int64_t skip = i ? lo - a.n0 : lo;
  Seg& s = k.seg[i];
  s.kw += skip * (int64_t(D) * bk / 32);
  s.vw += skip * (int64_t(D) * bv / 32);
  s.ks += skip * (D / a.gs);
  s.kb += skip * (D / a.gs);
  s.vs += skip * (D / a.gs);
  s.vb += skip * (D / a.gs);
  k.n0 = i ? 0 : a.n0 - lo;
  k.total = keys;
  return k;
}

// Both halves of the dequantize-once pass: one launch when K and V share a
// width, else one each.
template <int D>
void dequantize_rows(const Args& a, int bk, int bv, int64_t slabs, bool tiled, hipStream_t st,
                     uint16_t* kd, uint16_t* vd) {
  const int64_t sr = prefillplan::once_slab_rows(tiled, a.total);
  // (Tiled V: whole 64-key blocks, so that every tile is written.)
  const unsigned chunks = unsigned((sr * (D / 32) + 255) / 256);
  const int vt = tiled ? 1 : 0;
  if (bk == bv) {
    launch_dequantize_rows<D>(a, bk, 3, sr, vt, dim3(chunks, unsigned(slabs), 2), st, kd, vd);
  } else {
    launch_dequantize_rows<D>(a, bk, 1, sr, vt, dim3(chunks, unsigned(slabs), 1), st, kd, vd);
    launch_dequantize_rows<D>(a, bv, 2, sr, vt, dim3(chunks, unsigned(slabs), 1), st, kd, vd);
  }
}

// The splits' partials of each row (slots (row, split), row = (b L + l) H +
// h) combined and written as bf16: four channels a thread.
__global__ __launch_bounds__(256) void merge_splits_kernel(const Args a, int D, int64_t rows) {
  const int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x;
  const int64_t r = i / (D / 4);
  const int c = int(i % (D / 4)) * 4;
  if (r >= rows) return;
  const float* pm = a.part_m + r * a.n_part;
  const float* pl = a.part_l + r * a.n_part;
  float mx = -INFINITY;
  for (int s = 0; s < a.n_part; ++s) mx = fmaxf(mx, pm[s]);
  float l = 0.0f;
  f4_t o = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll 4
  for (int s = 0; s < a.n_part; ++s) {
    const float f = pm[s] == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(pm[s] - mx);
    l += f * pl[s];
    o += *reinterpret_cast<const f4_t*>(a.part_o + (r * a.n_part + s) * D + c) * f;
  }
  const float inv = l > 0.0f ? 1.0f / l : 0.0f;
  const int64_t h = r % a.H, bl = r / a.H;
  uint16_t* dst = a.out + bl / a.L * a.qs_b + h * a.qs_h + bl % a.L * a.qs_l + c;
  *reinterpret_cast<u32x2_t*>(dst) =
      u32x2_t{pack_bf16(o[0] * inv, o[1] * inv), pack_bf16(o[2] * inv, o[3] * inv)};
}

}  // namespace
}  // namespace prefill
}  // namespace tqkv

using namespace tqkv;
using namespace tqkv::prefill;

namespace tqkv {
namespace prefill {

// The shared-prefix half of a decode step: the queries of all B sequences
// (one position each) against a prefix every sequence shares, read once per
// KV head. The B sequences act as B query positions of one batch row
// (rows (b, g) of a KV head), the prefix's keys are split over the grid,
// and each split's (o, m, l) go to slots [0, n_splits) of the decode's
// partials [B, H, n_part]. Rows b * H + h line up with the decode kernel's.
bool tile_decode_supported(int D, int bk, int bv) {
  return D == 512 && (pick_decode_wide(bk, bv) || pick(D, bk, bv, true));
}
int tile_decode_rows() { return Shape<512, true>::kRows; }
bool tile_decode_wide(int bk, int bv) { return pick_decode_wide(bk, bv) != nullptr; }

// Decode through the tile kernel (f16 operands): each sequence's G query
// heads of a KV head are the rows of one block (one position, L = 1), the
// keys of up to two segments split over the grid; with n_splits > 1 each
// split's (o, m, l) go to slots [0, n_splits) of the decode's partials
// [B, H, n_part] (the decode's merge finishes), else the block writes out.
// Serves head_dim 512, which no decode kernel takes on the matrix cores.
int32_t tile_decode(const uint16_t* q, int B, int H, int H_kv, int D, int gs, int bk, int bv,
                    float scale, const tqkv_affine_seg* segs, int n_segs, int n_splits,
                    int split_len, int n_part, float* part_o, float* part_m, float* part_l,
                    uint16_t* out, hipStream_t st) {
  const KernelFn wide = pick_decode_wide(bk, bv), fn = wide ? wide : pick(D, bk, bv, true);
  if (!fn || D != 512) return fail(TQKV_EUNSUPPORTED, "tile decode D=%d bits %d/%d", D, bk, bv);
  Args a{};
  a.q = q;
  a.out = out;
  a.qs_b = int64_t(H) * D;
  a.qs_h = D;
  a.qs_l = int64_t(H) * D;
  a.H = H;
  a.H_kv = H_kv;
  a.G = H / H_kv;
  a.L = 1;
  a.gs = gs;
  a.causal = 0;
  a.qscale = scale * kLog2e;
  for (int i = 0; i < n_segs; ++i) {
    const tqkv_affine_seg& sg = segs[i];
    // Rows of a slab are addressed with 32-bit word offsets.
    if (sg.cap > 0 && sg.cap * int64_t(D) * (bk > bv ? bk : bv) / 32 >= (int64_t(1) << 32))
      return fail(TQKV_EINVAL_SHAPE, "segment %d: cap=%lld rows too large", i, (long long)sg.cap);
    a.seg[i] = Seg{sg.k_packed, sg.k_scales, sg.k_biases, sg.v_packed, sg.v_scales, sg.v_biases,
                   sg.cap, sg.shared ? 0 : int64_t(H_kv) * sg.cap};
  }
  if (n_segs == 1) a.seg[1] = a.seg[0];
  a.n0 = segs[0].n;
  a.total = segs[0].n + (n_segs == 2 ? segs[1].n : 0);
  if (a.total > (int64_t(1) << 31) - 2 * kTile)
    return fail(TQKV_EINVAL_SHAPE, "%lld keys exceed the kernel's 32-bit key index",
                (long long)a.total);
  a.n_splits = n_splits;
  a.split_len = split_len;
  a.split_base = 0;
  a.n_part = n_part;
  a.part_o = n_splits > 1 ? part_o : nullptr;
  a.part_m = n_splits > 1 ? part_m : nullptr;
  a.part_l = n_splits > 1 ? part_l : nullptr;
  using S = Shape<512, true>;
  const int64_t blocks = (a.G + S::kRows - 1) / S::kRows;
  a.n_blocks = int(blocks);
  const int64_t grid = blocks * n_splits * H_kv * int64_t(B);
  if (grid > 0x7fffffff) return fail(TQKV_EINVAL_SHAPE, "grid too large");
  static_assert(S::kRows == 16, "16 heads a block in both kernels");
  hipLaunchKernelGGL(fn, dim3(unsigned(grid)), dim3(wide ? 512 : S::kThreads), 0, st, a);
  TQKV_LAUNCHED();
  return TQKV_OK;
}

int shared_prefix_block_rows(int D) {
  switch (D) {
    case 64: return Shape<64, true>::kRows;
    case 128: return Shape<128, true>::kRows;
    default: return Shape<256, true>::kRows;
  }
}

int32_t shared_prefix_partials(const uint16_t* q, int B, int H, int H_kv, int D, int gs, int bk,
                               int bv, float scale, const tqkv_affine_seg& prefix, int n_splits,
                               int split_len, int n_part, float* part_o, float* part_m,
                               float* part_l, hipStream_t st) {
  // f16 operands: decode's bar is the exact dequantization, and f16's
  // three more significand bits keep the shared-prefix path within it.
  KernelFn fn = pick(D, bk, bv, true);
  if (!fn) return fail(TQKV_EUNSUPPORTED, "shared-prefix decode D=%d bits %d/%d", D, bk, bv);
  Args a{};
  a.q = q;
  a.out = nullptr;
  a.qs_b = 0;
  a.qs_h = D;
  a.qs_l = int64_t(H) * D;  // position l of the one batch row = sequence l
  a.H = H;
  a.H_kv = H_kv;
  a.G = H / H_kv;
  a.L = B;
  a.gs = gs;
  a.causal = 0;
  a.qscale = scale * kLog2e;
  a.seg[0] = Seg{prefix.k_packed, prefix.k_scales, prefix.k_biases, prefix.v_packed,
                 prefix.v_scales, prefix.v_biases, prefix.cap, 0};
  a.seg[1] = a.seg[0];
  a.n0 = prefix.n;
  a.total = prefix.n;
  a.n_splits = n_splits;
  a.split_len = split_len;
  a.split_base = 0;
  a.n_part = n_part;
  a.part_o = part_o;
  a.part_m = part_m;
  a.part_l = part_l;
  int rows_per_block = 0, threads = 0;
  switch (D) {
    case 64: rows_per_block = Shape<64, true>::kRows, threads = Shape<64, true>::kThreads; break;
    case 128: rows_per_block = Shape<128, true>::kRows, threads = Shape<128, true>::kThreads; break;
    default: rows_per_block = Shape<256, true>::kRows, threads = Shape<256, true>::kThreads; break;
  }
  const int64_t blocks = (int64_t(B) * a.G + rows_per_block - 1) / rows_per_block;
  a.n_blocks = int(blocks);
  const int64_t grid = blocks * n_splits * H_kv;
  if (grid > 0x7fffffff) return fail(TQKV_EINVAL_SHAPE, "grid too large");
  hipLaunchKernelGGL(fn, dim3(unsigned(grid)), dim3(threads), 0, st, a);
  TQKV_LAUNCHED();
  return TQKV_OK;
}

}  // namespace prefill
}  // namespace tqkv

namespace {

// The prefill launch over affine segments, or (bf16_rows) over one segment
// whose "packed" arrays are bf16 rows of D values (K and V already
// dequantized or stored in bf16; scales and biases unused).
int32_t prefill_launch(const uint16_t* q, int32_t B, int32_t H, int32_t H_kv, int32_t L,
                       int32_t D, int32_t group_size, int32_t bits_k, int32_t bits_v, float scale,
                       const tqkv_affine_seg* segs, int32_t n_segs, int64_t q_start,
                       int64_t k_start, int32_t causal, int64_t window, uint16_t* out,
                       tqkv_stream stream, bool bf16_rows, bool library_scratch = true,
                       void* workspace = nullptr, size_t workspace_bytes = 0) {
  if (!q || !out || !segs) return fail(TQKV_EINVAL_ARG, "null pointer");
  if (B <= 0 || H <= 0 || H_kv <= 0 || H % H_kv != 0 || L <= 0)
    return fail(TQKV_EINVAL_SHAPE, "B=%d H=%d H_kv=%d L=%d", B, H, H_kv, L);
  if (n_segs < 1 || n_segs > 2 || (bf16_rows && n_segs != 1))
    return fail(TQKV_EINVAL_ARG, "n_segs=%d", n_segs);
  if (bf16_rows) {
    bits_k = bits_v = kPreBits;
  } else if (!valid_bits(bits_k) || !valid_bits(bits_v)) {
    return fail(TQKV_EUNSUPPORTED, "affine bits_k=%d bits_v=%d not in {2,3,4,5,6,8}", bits_k,
                bits_v);
  }
  if (!(group_size == 32 || group_size == 64 || group_size == 128) || D % group_size != 0)
    return fail(TQKV_EUNSUPPORTED, "group_size=%d with D=%d", group_size, D);
  KernelFn fn = pick(D, bits_k, bits_v);
  if (!fn) return fail(TQKV_EUNSUPPORTED, "prefill head dim D=%d (64, 128, 256 or 512)", D);
  if (causal && window == 0) return fail(TQKV_EINVAL_ARG, "window=0 hides every key");
  if (!(scale > 0.0f) || !std::isfinite(scale))
    return fail(TQKV_EINVAL_ARG, "softmax scale %g must be positive and finite", double(scale));
  if (int64_t(B) * H * L * D >= (int64_t(1) << 40))
    return fail(TQKV_EINVAL_SHAPE, "query tensor too large");

  Args a{};
  a.q = q;
  a.out = out;
  a.qs_l = D;
  a.qs_h = int64_t(L) * D;
  a.qs_b = int64_t(H) * L * D;
  a.H = H;
  a.H_kv = H_kv;
  a.G = H / H_kv;
  a.L = L;
  a.gs = group_size;
  a.causal = causal ? 1 : 0;
  a.qscale = scale * kLog2e;
  for (int i = 0; i < n_segs; ++i) {
    const tqkv_affine_seg& s = segs[i];
    if (s.n < 0 || s.n > s.cap)
      return fail(TQKV_EINVAL_SHAPE, "segment %d: n=%lld cap=%lld", i, (long long)s.n,
                  (long long)s.cap);
    if (s.n > 0 && (!s.k_packed || !s.k_scales || !s.k_biases || !s.v_packed || !s.v_scales ||
                    !s.v_biases))
      return fail(TQKV_EINVAL_ARG, "segment %d has a null buffer", i);
    // Rows of a slab are addressed with 32-bit word offsets.
    if (s.cap > 0 && s.cap * int64_t(D) * (bits_k > bits_v ? bits_k : bits_v) / 32 >= (int64_t(1) << 32))
      return fail(TQKV_EINVAL_SHAPE, "segment %d: cap=%lld rows too large", i, (long long)s.cap);
    a.seg[i] = Seg{s.k_packed, s.k_scales, s.k_biases, s.v_packed, s.v_scales, s.v_biases,
                   s.cap, s.shared ? 0 : int64_t(H_kv) * s.cap};
  }
  if (n_segs == 1) a.seg[1] = a.seg[0];
  a.n0 = segs[0].n;
  a.total = segs[0].n + (n_segs == 2 ? segs[1].n : 0);
  if (a.total <= 0) return fail(TQKV_EINVAL_SHAPE, "no keys to attend");
  if (a.total > (int64_t(1) << 31) - 2 * kTile)
    return fail(TQKV_EINVAL_SHAPE, "%lld keys exceed the kernel's 32-bit key index",
                (long long)a.total);
  a.q_start = q_start;
  a.k_start = k_start;
  a.window = window < 0 ? -1 : window;
  a.split_base = 0;

  int rows_per_block = 0, threads = 0;
  switch (D) {
    case 64: rows_per_block = Shape<64, false>::kRows, threads = Shape<64, false>::kThreads; break;
    case 128: rows_per_block = Shape<128, false>::kRows, threads = Shape<128, false>::kThreads; break;
    case 256: rows_per_block = Shape<256, false>::kRows, threads = Shape<256, false>::kThreads; break;
    default: rows_per_block = Shape<512, false>::kRows, threads = Shape<512, false>::kThreads; break;
  }
  const int64_t blocks = (int64_t(L) * a.G + rows_per_block - 1) / rows_per_block;
  if (blocks * H_kv * B > 0x7fffffff) return fail(TQKV_EINVAL_SHAPE, "grid too large");
  const int64_t units = blocks * H_kv * B, q_rows = int64_t(B) * H * L;
  const size_t ws_bytes = workspace ? workspace_bytes : 0;
  const prefillplan::Chunk chunk{B, H, H_kv, L, D, a.total, q_start, k_start, a.causal != 0,
                                 a.window, rows_per_block, blocks, bf16_rows, library_scratch,
                                 ws_bytes};
  size_t part_bytes = 0;
  const auto use_splits = [&](const prefillplan::Splits& sp) {
    a.n_splits = a.n_part = int(sp.n);
    a.split_len = int(sp.len);
    a.split_lo = sp.lo;
    part_bytes = sp.bytes;
  };
  use_splits(prefillplan::key_splits(chunk));
  a.n_blocks = int(blocks);
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  // The partials at p (16-byte aligned), and the merge after the kernel.
  const auto use_parts = [&](Args& args, void* p) {
    args.part_o = static_cast<float*>(p);
    args.part_m = args.part_o + size_t(q_rows) * a.n_splits * D;
    args.part_l = args.part_m + size_t(q_rows) * a.n_splits;
  };
  const auto merge = [&](const Args& args) {
    const int64_t threads = q_rows * (D / 4);
    hipLaunchKernelGGL(merge_splits_kernel, dim3(unsigned((threads + 255) / 256)), dim3(256), 0, st,
                       args, D, q_rows);
  };
  // TQKV_PREFILL_DEQUANT_ONCE=0 / 1 forces the choice (tests compare them).
  const char* once_env = getenv("TQKV_PREFILL_DEQUANT_ONCE");
  const int64_t slabs = int64_t(B) * H_kv;
  const prefillplan::Once rows =
      prefillplan::dequantize_once(chunk, once_env ? strcmp(once_env, "0") != 0 : -1);
  bool once = rows.on;
  if (once && slabs > prefillplan::kOnceMaxSlabs)
    return fail(TQKV_EINVAL_SHAPE, "B * H_kv = %lld slabs", (long long)slabs);
  // Scratch that the call could do without (the partials; the rows of few
  // blocks) is left out where the library's cannot grow.
  void* ws = workspace;
  if (library_scratch && (once || part_bytes)) {
    bool held = part_bytes && scratch_optional((once ? rows.bytes : 0) + part_bytes, st, &ws);
    if (!held) use_splits(prefillplan::no_splits(chunk));
    if (once && !held) {
      if (blocks >= prefillplan::kOnceBlocks || once_env) {
        if (int32_t rc = scratch_for_current_device(rows.bytes, &ws)) return rc;
      } else {
        once = scratch_optional(rows.bytes, st, &ws);
      }
    }
  }
  const int64_t grid = units * a.n_splits;
  if (once) {
    uint16_t* kd = static_cast<uint16_t*>(ws);
    uint16_t* vd = kd + size_t(slabs) * size_t(rows.slab_rows) * size_t(D);
    const Args d = keys_from(a, D, bits_k, bits_v, rows.lo, rows.keys);
    switch (D) {
      case 64: dequantize_rows<64>(d, bits_k, bits_v, slabs, rows.tiled, st, kd, vd); break;
      case 128: dequantize_rows<128>(d, bits_k, bits_v, slabs, rows.tiled, st, kd, vd); break;
      case 256: dequantize_rows<256>(d, bits_k, bits_v, slabs, rows.tiled, st, kd, vd); break;
      default: dequantize_rows<512>(d, bits_k, bits_v, slabs, rows.tiled, st, kd, vd); break;
    }
    TQKV_LAUNCHED();
    Args p = a;
    const uint16_t* none = kd;  // scales and biases: never read at this width
    p.seg[0] = Seg{reinterpret_cast<const uint32_t*>(kd), none, none,
                   reinterpret_cast<const uint32_t*>(vd), none, none, rows.slab_rows,
                   int64_t(H_kv) * rows.slab_rows};
    p.seg[1] = p.seg[0];
    // (The splits start at the first visible tile too.)
    p.n0 = p.total = rows.keys;
    p.k_start = a.k_start + rows.lo;
    p.split_lo = 0;
    if (part_bytes) use_parts(p, static_cast<char*>(ws) + rows.bytes);
    if (D >= 256 && rows.tiled) {
      // Rows a block by rounds of workgroups over the CUs (one a CU), a 64-row
      // block's taking 0.87 of a 128-row one's time (32 / 2 heads, D = 512,
      // 512 rows over 8,192 keys, one round each: 331 and 380 us).
      const int64_t unit_rows = int64_t(L) * a.G, per_block = int64_t(H_kv) * B * a.n_splits;
      const auto rounds = [&](int64_t rows) {
        return ((unit_rows + rows - 1) / rows * per_block + 255) / 256;
      };
      const int wide_rows = 100 * rounds(128) <= 87 * rounds(64) ? 128 : 64;
      p.n_blocks = int((unit_rows + wide_rows - 1) / wide_rows);
      hipLaunchKernelGGL(pick_wide(D, wide_rows), dim3(unsigned(p.n_blocks * per_block)),
                         dim3(4 * wide_rows), 0, st, p);
    } else {
      hipLaunchKernelGGL(pick(D, kPreBits, rows.tiled ? kPreF16T : kPreF16), dim3(unsigned(grid)),
                         dim3(threads), 0, st, p);
    }
    TQKV_LAUNCHED();
    if (part_bytes) {
      merge(p);
      TQKV_LAUNCHED();
    }
    return ok();
  }
  if (part_bytes) use_parts(a, ws);
  hipLaunchKernelGGL(fn, dim3(unsigned(grid)), dim3(threads), 0, st, a);
  TQKV_LAUNCHED();
  if (part_bytes) {
    merge(a);
    TQKV_LAUNCHED();
  }
  return ok();
}

}  // namespace

extern "C" int32_t tqkv_prefill_attend_affine(const uint16_t* q, int32_t B, int32_t H,
                                              int32_t H_kv, int32_t L, int32_t D,
                                              int32_t group_size, int32_t bits_k, int32_t bits_v,
                                              float scale, const tqkv_affine_seg* segs,
                                              int32_t n_segs, int64_t q_start, int64_t k_start,
                                              int32_t causal, int64_t window, uint16_t* out,
                                              tqkv_stream stream) {
  return prefill_launch(q, B, H, H_kv, L, D, group_size, bits_k, bits_v, scale, segs, n_segs,
                        q_start, k_start, causal, window, out, stream, false);
}

extern "C" size_t tqkv_prefill_workspace_size(int32_t B, int32_t H_kv, int32_t D,
                                              int64_t total_keys) {
  if (B <= 0 || H_kv <= 0 || D <= 0 || total_keys <= 0) return 0;
  return prefillplan::once_bytes(int64_t(B) * H_kv,
                                 prefillplan::once_slab_rows(D == 128, total_keys), D);
}

extern "C" int32_t tqkv_prefill_attend_affine_ws(
    const uint16_t* q, int32_t B, int32_t H, int32_t H_kv, int32_t L, int32_t D,
    int32_t group_size, int32_t bits_k, int32_t bits_v, float scale, const tqkv_affine_seg* segs,
    int32_t n_segs, int64_t q_start, int64_t k_start, int32_t causal, int64_t window,
    uint16_t* out, void* workspace, size_t workspace_bytes, tqkv_stream stream) {
  return prefill_launch(q, B, H, H_kv, L, D, group_size, bits_k, bits_v, scale, segs, n_segs,
                        q_start, k_start, causal, window, out, stream, false, false, workspace,
                        workspace_bytes);
}

namespace tqkv {
// Prefill-chunk attention over bf16 K and V rows ([B, H_kv, cap, D], keys
// [0, n) of each slab): the same MFMA kernel with the dequantization left
// out (codebook caches after tqkv_codebook_dequantize, bf16 caches).
int32_t prefill_bf16_rows(const uint16_t* q, int B, int H, int H_kv, int L, int D,
                          const uint16_t* k, const uint16_t* v, int64_t cap, int64_t n,
                          int64_t q_start, int64_t k_start, int64_t window, float scale,
                          uint16_t* out, hipStream_t stream) {
  tqkv_affine_seg s{};
  s.k_packed = reinterpret_cast<const uint32_t*>(k);
  s.v_packed = reinterpret_cast<const uint32_t*>(v);
  s.k_scales = s.k_biases = k;  // never read at this width
  s.v_scales = s.v_biases = v;
  s.cap = cap;
  s.n = n;
  return prefill_launch(q, B, H, H_kv, L, D, 64, 0, 0, scale, &s, 1, q_start, k_start, 1, window,
                        out, reinterpret_cast<tqkv_stream>(stream), true);
}
}  // namespace tqkv

// The reference GPU cache's TurboQuant encode (turboquant.rs:398-423,
// 720-745): y = x (mode 0), bf16(x M) (mode 1) or x M (mode 2), M = R or R^T,
// then sigma = sqrt(sum y^2 / D) and code = the number of inner boundaries b
// (ascending, f32) with b <= bf16(y / sigma).
//
// Bit for bit (the oracle restates this order): the rotation is one fmaf
// chain per output over j = 0 .. D - 1 from 0.0; the sum of squares runs over
// channels l, l + 64, l + 128, .. for each l in 0 .. 63, then over l by an
// xor butterfly 32, 16, .., 1; division and square root correctly rounded.
//
// Bound: the rotation's 2 D^2 f32 operations a row. It runs on
// v_mfma_f32_16x16x4_f32: checked on gfx950 over normal, wide-exponent,
// subnormal, infinite and NaN operands, a chain of those products gives the
// bits of the fmaf chain over k (each product's four steps in k order, one
// rounding each), at twice the rate of the vector FMAs. A workgroup takes
// 16 MR whole rows (sigma needs the row) and its 2 D threads are D / 32
// wavefronts of 32 columns each; M goes through LDS 16 rows a step, two
// steps' buffers, read coalesced for R and R^T alike (the wavefront-per-
// four-rows kernel this replaces read R^T with a stride of a row a lane).
// Measured a call of 16,384 rows of 256 channels, R^T: 457 -> 34 us (63
// TFLOP/s of the ~157 the f32 matrix rate gives; the rest is the divides and
// the passes over y); 24,792 rows of 64: 37 -> 9.8 us; 36 rows of 512: 131 ->
// 37 us (one workgroup a 16-row block: 14 us of products on one CU).
#include "common.hpp"

namespace tqkv {
namespace tq {
namespace {

typedef float f4_t __attribute__((ext_vector_type(4)));

// MR = 1 (few rows): 64 rows of M a step through one buffer, so the loads of
// a step, and not a wait a 16-row step, set the time (MR = 4's two 16-row
// buffers took 38 us a call at 48 rows of 512 channels).
template <int D, int MR>
struct EncShape {
  static constexpr int kRows = 16 * MR;
  static constexpr int kThreads = 2 * D;
  static constexpr int kStep = MR == 1 ? 64 : 16;  // rows of M a step
  static constexpr int kBufs = MR == 1 ? 1 : 2;
  static constexpr int kXs = D + 8;   // bf16 row stride of x in LDS: 16 rows x 4 k in distinct banks
  static constexpr int kMs = D + 16;  // f32 row stride of M: 4 k x 16 columns in distinct banks
  static constexpr int kYs = D + 4;   // f32 row stride of y: 16 rows x 4 lanes in distinct banks
  static constexpr int kXBytes = kRows * kXs * 2;
  static constexpr int kMBytes = kStep * kMs * 4;
  // y takes the same memory once the products are done.
  static constexpr int kYBytes = kRows * kYs * 4;
  static constexpr int kBytes =
      kXBytes + kBufs * kMBytes > kYBytes ? kXBytes + kBufs * kMBytes : kYBytes;
};

// wide: x and rotation 16-byte aligned. words: codes 4-byte aligned.
template <int D, int MR>
__global__ __launch_bounds__((EncShape<D, MR>::kThreads)) void tq_encode_gpu_kernel(
    const uint16_t* __restrict__ x, int64_t s, int64_t rows, const float* __restrict__ R, int mode,
    int transpose, const float* __restrict__ inner, int bits, uint8_t* __restrict__ codes,
    float* __restrict__ sigma, int64_t dst_cap, int64_t dst_start, int wide, int words) {
  using S = EncShape<D, MR>;
  constexpr int kThreads = S::kThreads, kRows = S::kRows, kYs = S::kYs;
  constexpr int kStep = S::kStep, kBufs = S::kBufs;
  __shared__ __attribute__((aligned(16))) unsigned char s_mem[S::kBytes];
  __shared__ float s_sg[kRows];
  __shared__ float s_bnd[256];
  const int tid = threadIdx.x, lane = tid % 64, wave = tid / 64;
  const int64_t r0 = int64_t(blockIdx.x) * kRows;
  const int nr = rows - r0 < kRows ? int(rows - r0) : kRows;
  const int n_inner = (1 << bits) - 1;
  for (int i = tid; i < n_inner; i += kThreads) s_bnd[i] = inner[i];
  float* y = reinterpret_cast<float*>(s_mem);
  if (mode == 0) {
    for (int i = tid; i < nr * D; i += kThreads)
      y[i / D * kYs + i % D] = bf16_to_f32(x[r0 * D + i]);
  } else {
    uint16_t* xs = reinterpret_cast<uint16_t*>(s_mem);
    // x rows (rows past the end are zeros, their results unused).
    if (wide) {
      for (int i = tid; i < kRows * (D / 8); i += kThreads) {
        const int r = i / (D / 8), c = i % (D / 8);
        uint4 v{0u, 0u, 0u, 0u};
        if (r < nr) v = *reinterpret_cast<const uint4*>(x + (r0 + r) * D + 8 * c);
        *reinterpret_cast<uint4*>(xs + r * S::kXs + 8 * c) = v;
      }
    } else {
      for (int i = tid; i < kRows * D; i += kThreads) {
        const int r = i / D, c = i % D;
        xs[r * S::kXs + c] = r < nr ? x[(r0 + r) * D + c] : uint16_t(0);
      }
    }
    // A thread's values of a step of M (rows k0 .. of D columns): column
    // tid % D, kPer consecutive k (of a row of R for R^T).
    constexpr int kPer = kStep / 2;
    const int col = tid % D, kh = kPer * (tid / D);
    float mv[kPer];
    auto load_m = [&](int k0) __attribute__((always_inline)) {
      if (transpose) {
        const float* p = R + int64_t(col) * D + k0 + kh;
        if (wide) {
#pragma unroll
          for (int e = 0; e < kPer; e += 4) {
            const f4_t a = *reinterpret_cast<const f4_t*>(p + e);
#pragma unroll
            for (int i = 0; i < 4; ++i) mv[e + i] = a[i];
          }
        } else {
#pragma unroll
          for (int e = 0; e < kPer; ++e) mv[e] = p[e];
        }
      } else {
#pragma unroll
        for (int e = 0; e < kPer; ++e) mv[e] = R[int64_t(k0 + kh + e) * D + col];
      }
    };
    auto store_m = [&](int buf) __attribute__((always_inline)) {
      float* ms = reinterpret_cast<float*>(s_mem + S::kXBytes + buf * S::kMBytes);
#pragma unroll
      for (int e = 0; e < kPer; ++e) ms[(kh + e) * S::kMs + col] = mv[e];
    };
    const int lr = lane % 16, lg = lane / 16;
    f4_t acc[MR][2];
#pragma unroll
    for (int a = 0; a < MR; ++a)
#pragma unroll
      for (int b = 0; b < 2; ++b) acc[a][b] = f4_t{0.0f, 0.0f, 0.0f, 0.0f};
    load_m(0);
    store_m(0);
    __syncthreads();
    for (int k0 = 0, buf = 0; k0 < D; k0 += kStep, buf ^= kBufs - 1) {
      const bool more = k0 + kStep < D;
      if (more) load_m(k0 + kStep);
      const float* ms = reinterpret_cast<const float*>(s_mem + S::kXBytes + buf * S::kMBytes);
#pragma unroll
      for (int k = 0; k < kStep; k += 4) {
        float bv[2];
#pragma unroll
        for (int b = 0; b < 2; ++b) bv[b] = ms[(k + lg) * S::kMs + 32 * wave + 16 * b + lr];
#pragma unroll
        for (int a = 0; a < MR; ++a) {
          const float av = bf16_to_f32(xs[(16 * a + lr) * S::kXs + k0 + k + lg]);
#pragma unroll
          for (int b = 0; b < 2; ++b)
            acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x4f32(av, bv[b], acc[a][b], 0, 0, 0);
        }
      }
      // Two buffers: the other one's last readers passed the barrier that
      // ended the step before. One: this step's readers pass one here.
      if constexpr (kBufs == 1) __syncthreads();
      if (more) store_m(buf ^ (kBufs - 1));
      __syncthreads();
    }
    // Lane (lr, lg) holds rows 4 lg + i, column lr of each 16 x 16 tile.
#pragma unroll
    for (int a = 0; a < MR; ++a)
#pragma unroll
      for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float v = acc[a][b][i];
          y[(16 * a + 4 * lg + i) * kYs + 32 * wave + 16 * b + lr] =
              mode == 1 ? bf16_to_f32(f32_to_bf16(v)) : v;
        }
  }
  __syncthreads();
  // sigma: four lanes a row, lane q channels 4 i + q + 64 k: the partial of
  // channel l = 4 i + q over k, the butterfly's 32, 16, 8 and 4 inside the
  // lane (i ^ 8, 4, 2, 1), its 2 and 1 across the four lanes. (A wavefront a
  // row, a lane an l, put 32 six-exchange chains in series at D = 64.)
  for (int r4 = tid / 4; r4 < kRows; r4 += kThreads / 4) {
    const int q = tid % 4;
    const int r = r4 < nr ? r4 : nr - 1;
    float p[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      p[i] = 0.0f;
#pragma unroll
      for (int k = 0; k < D / 64; ++k) {
        const float v = y[r * kYs + 4 * i + q + 64 * k];
        p[i] = __fadd_rn(p[i], __fmul_rn(v, v));
      }
    }
#pragma unroll
    for (int off = 8; off >= 1; off >>= 1)
#pragma unroll
      for (int i = 0; i < off; ++i) p[i] = __fadd_rn(p[i], p[i + off]);
    float t = p[0];
    t = __fadd_rn(t, __shfl_xor(t, 2, 64));
    t = __fadd_rn(t, __shfl_xor(t, 1, 64));
    const float sg = __builtin_sqrtf(t / float(D));
    if (q == 0 && r4 < nr) {
      s_sg[r4] = sg;
      const int64_t rr = r0 + r4;
      sigma[(rr / s) * dst_cap + dst_start + rr % s] = sg;
    }
  }
  __syncthreads();
  // Codes: four consecutive channels a thread, one 4-byte store (a byte at a
  // time where the code rows are not 4-byte aligned). The boundaries are
  // 2^bits - 1, so the search takes `bits` halvings.
  for (int i = tid; i < nr * (D / 4); i += kThreads) {
    const int r = i / (D / 4), c = 4 * (i % (D / 4));
    const f4_t v = *reinterpret_cast<const f4_t*>(y + r * kYs + c);
    const float sg = s_sg[r];
    float xn[4];
    int lo[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      xn[e] = bf16_to_f32(f32_to_bf16(v[e] / sg));
      lo[e] = 0;
    }
    for (int half = 1 << (bits - 1); half >= 1; half >>= 1)
#pragma unroll
      for (int e = 0; e < 4; ++e) lo[e] += s_bnd[lo[e] + half - 1] <= xn[e] ? half : 0;
    const int64_t rr = r0 + r;
    uint8_t* dst = codes + ((rr / s) * dst_cap + dst_start + rr % s) * D + c;
    if (words) {
      *reinterpret_cast<uint32_t*>(dst) =
          uint32_t(lo[0]) | uint32_t(lo[1]) << 8 | uint32_t(lo[2]) << 16 | uint32_t(lo[3]) << 24;
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) dst[e] = uint8_t(lo[e]);
    }
  }
}

template <int D>
void launch_encode(const uint16_t* x, int64_t s, int64_t rows, const float* R, int mode,
                   int transpose, const float* inner, int bits, uint8_t* codes, float* sigma,
                   int64_t dst_cap, int64_t dst_start, hipStream_t st) {
  const int wide = (reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(R)) % 16 == 0;
  const int words = reinterpret_cast<uintptr_t>(codes) % 4 == 0;
#define TQKV_ENC(MR)                                                                         \
  hipLaunchKernelGGL((tq_encode_gpu_kernel<D, MR>),                                          \
                     dim3(unsigned((rows + 16 * MR - 1) / (16 * MR))), dim3(2 * D), 0, st, x, s, \
                     rows, R, mode, transpose, inner, bits, codes, sigma, dst_cap, dst_start, \
                     wide, words)
  // 64 rows a workgroup read M a quarter as often, but up to 16,384 rows (a
  // workgroup a CU) they take the time of one workgroup: 17, 33 and 92 us at D =
  // 128, 256 and 512, where 16 rows grow in rounds of 12,288, 8,192 and 4,096
  // rows (what the CUs' LDS holds). R^T, 16 against 64 rows: D = 128, 16,384
  // rows 18.1 and 17.1 us, 20,000 rows 20.3 and 21.7, 24,577 rows 23.3 and 21.9
  // (R: 21.4 and 22.0, 32,768 rows 26.0 and 22.7); D = 256, 8,193 rows 32.5 and
  // 33.2, 10,000 rows 35.2 and 33.7 (R, whose loads are coalesced as they are:
  // 12,000 rows 31.3 and 33.7, 12,289 rows 36.4 and 34.2); D = 512, 8,192 rows
  // 87 and 92, 8,193 rows 124 and 92. Mode 0 (no products): D = 256, 24,577 rows
  // 19.9 and 22.6, 49,152 rows 36.4 and 35.1; D = 512, 12,289 rows 23.9 and
  // 23.2. At D = 64 (M is 16 KB) more wavefronts win.
  const int64_t most = D == 128 || (D == 256 && mode == 0) ? 24576
                       : D == 256 && !transpose            ? 12288
                                                           : 8192;
  if (D > 64 && rows > most)
    TQKV_ENC(4);
  else
    TQKV_ENC(1);
#undef TQKV_ENC
}

}  // namespace
}  // namespace tq
}  // namespace tqkv

using namespace tqkv;

extern "C" int32_t tqkv_tq_encode_gpu_path(const uint16_t* x, int64_t n_slabs, int64_t s,
                                           int32_t dim, const float* rotation, int32_t mode,
                                           int32_t transpose, const float* boundaries_inner,
                                           int32_t bits, uint8_t* codes, float* sigma,
                                           int64_t dst_cap, int64_t dst_start,
                                           tqkv_stream stream) {
  if (bits < 1 || bits > 8) return fail(TQKV_EUNSUPPORTED, "codebook bits=%d", bits);
  if (!(dim == 64 || dim == 128 || dim == 256 || dim == 512))
    return fail(TQKV_EUNSUPPORTED, "encode dim=%d not in {64,128,256,512}", dim);
  if (mode < 0 || mode > 2) return fail(TQKV_EINVAL_ARG, "mode=%d not in {0, 1, 2}", mode);
  if (n_slabs < 0 || s < 0 || dst_start < 0 || dst_start + s > dst_cap)
    return fail(TQKV_EINVAL_SHAPE, "rows [%lld, %lld) do not fit a buffer of %lld",
                (long long)dst_start, (long long)(dst_start + s), (long long)dst_cap);
  if (n_slabs == 0 || s == 0) return ok();
  if (!x || !boundaries_inner || !codes || !sigma || (mode != 0 && !rotation))
    return fail(TQKV_EINVAL_ARG, "null pointer");
  const int64_t rows = n_slabs * s;
  if (rows > 0x7fffffffLL) return fail(TQKV_EINVAL_SHAPE, "too many rows");
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  switch (dim) {
    case 64: tq::launch_encode<64>(x, s, rows, rotation, mode, transpose ? 1 : 0, boundaries_inner, bits, codes, sigma, dst_cap, dst_start, st); break;
    case 128: tq::launch_encode<128>(x, s, rows, rotation, mode, transpose ? 1 : 0, boundaries_inner, bits, codes, sigma, dst_cap, dst_start, st); break;
    case 256: tq::launch_encode<256>(x, s, rows, rotation, mode, transpose ? 1 : 0, boundaries_inner, bits, codes, sigma, dst_cap, dst_start, st); break;
    default: tq::launch_encode<512>(x, s, rows, rotation, mode, transpose ? 1 : 0, boundaries_inner, bits, codes, sigma, dst_cap, dst_start, st); break;
  }
  TQKV_LAUNCHED();
  return ok();
}

// TEST HARNESS (not product code). The prefill's plan (lumen-rs_amd/csrc/
// prefill_plan.hpp) behind plain C entries, for the CPU tests.
#include "prefill_plan.hpp"

using namespace tqkv::prefillplan;

// c: B, H, H_kv, L, D, total, q_start, k_start, causal, window,
// block_rows, blocks, bf16_rows, library_scratch, ws_bytes.
static Chunk chunk(const int64_t* c) {
  return Chunk{c[0], c[1],      c[2], c[3],  c[4],  c[5],       c[6],       c[7],
               c[8] != 0, c[9], c[10], c[11], c[12] != 0, c[13] != 0, size_t(c[14])};
}

extern "C" {
// out: lo, hi.
void planhost_visible(const int64_t* c, int64_t* out) {
  const Visible v = visible_keys(chunk(c));
  out[0] = v.lo;
  out[1] = v.hi;
}
// out: n, len, lo, bytes.
void planhost_splits(const int64_t* c, int64_t* out) {
  const Splits s = key_splits(chunk(c));
  out[0] = s.n;
  out[1] = s.len;
  out[2] = s.lo;
  out[3] = int64_t(s.bytes);
}
// out: on, lo, keys, slab_rows, tiled, bytes.
void planhost_once(const int64_t* c, int64_t force, int64_t* out) {
  const Once o = dequantize_once(chunk(c), int(force));
  out[0] = o.on;
  out[1] = o.lo;
  out[2] = o.keys;
  out[3] = o.slab_rows;
  out[4] = o.tiled;
  out[5] = int64_t(o.bytes);
}
}

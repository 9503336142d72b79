// How a prefill call splits its work and what scratch that takes, as plain
// C++ (no HIP): prefill_affine.hip launches by it, the tests check it on the
// CPU over all forms of a call.
#pragma once

#include <cstddef>
#include <cstdint>

namespace tqkv {
namespace prefillplan {

constexpr int64_t kTileKeys = 64;  // keys a step of every prefill kernel

struct Chunk {
  int64_t B, H, H_kv, L, D;
  int64_t total;  // keys of both segments
  int64_t q_start, k_start;
  bool causal;
  int64_t window;        // < 0: none
  int64_t block_rows;    // (position, head) rows a block of the in-block kernel
  int64_t blocks;        // row blocks a KV head in it
  bool bf16_rows;        // K and V are bf16 rows, not packed codes
  bool library_scratch;  // else a caller's workspace, which holds rows only
  size_t ws_bytes;       // of that workspace
};

// The keys [lo, hi] that some row of the chunk sees, lo down to a whole tile;
// hi < lo where no row sees any.
struct Visible {
  int64_t lo, hi;
};
inline Visible visible_keys(const Chunk& c) {
  int64_t lo = 0, hi = c.total - 1;
  if (c.causal) {
    if (c.q_start + c.L - 1 - c.k_start < hi) hi = c.q_start + c.L - 1 - c.k_start;
    if (c.window >= 0 && c.q_start - c.window + 1 - c.k_start > lo)
      lo = c.q_start - c.window + 1 - c.k_start;
  }
  return Visible{lo / kTileKeys * kTileKeys, hi};
}

// Bytes of the dequantized K and V rows of every (batch row, KV head).
inline size_t once_bytes(int64_t slabs, int64_t slab_rows, int64_t D) {
  return 2 * size_t(slabs) * size_t(slab_rows) * size_t(D) * 2;
}
// Rows a slab of them holds: the keys, up to whole tiles where V is tiled (K
// shares the stride).
inline int64_t once_slab_rows(bool tiled, int64_t keys) {
  return tiled ? (keys + kTileKeys - 1) / kTileKeys * kTileKeys : keys;
}

// Row blocks sharing one (batch row, KV head) from which its visible keys are
// dequantized once into scratch instead of in every block: the blocks would
// otherwise repeat the same dequantization, the kernel's VALU-bound part.
// The wide kernel takes fewer: at D = 512 any (the in-block kernel spills;
// 16 / 4 heads, 94 rows over 1,117 keys: 131 us in block, 44 once; 32 / 2
// heads, 4 rows over 64 keys: 21.1 and 16.5), at D = 256
// half as many over 2,048 keys or more (B = 4, 16 / 8 heads, 300 rows over
// 3,000 keys: 132 us in block, 107 once; 298 rows over 809: 35 and 42).
// Only the keys that the chunk sees are dequantized and counted: of 65,536
// keys under a window of 1,024, 300 rows take 47 us at D = 256 (16 / 8 heads)
// and 67 at D = 512 (32 / 2); with all keys 154 and 121.
constexpr int64_t kOnceBlocks = 8;
inline int64_t once_blocks(int64_t D, int64_t keys) {
  return D == 512 ? 1 : D == 256 && keys >= 2048 ? 4 : kOnceBlocks;
}
// The scratch that path may take; more keys dequantize in every block instead.
constexpr size_t kOnceMaxBytes = size_t(4) << 30;
// Slabs its launch takes. With more, fewer than kOnceBlocks row blocks stay in
// block; a call of more blocks is refused.
constexpr int64_t kOnceMaxSlabs = 65535;

// Dequantize once: keys [lo, lo + keys) as slabs of slab_rows rows, V as
// transposed tiles where `tiled`.
struct Once {
  bool on = false;
  int64_t lo = 0, keys = 0, slab_rows = 0;
  bool tiled = false;
  size_t bytes = 0;
};
// force: 0 or 1 (tests compare the two ways), -1 for the rule.
inline Once dequantize_once(const Chunk& c, int force) {
  Once o;
  const Visible v = visible_keys(c);
  o.lo = v.lo;
  o.keys = v.hi - v.lo + 1;
  if (c.bf16_rows || force == 0 || o.keys <= 0) return o;
  // V as transposed tiles: always at D = 128; at D = 256 and 512 (the wide
  // kernel) wherever there is room for whole tiles, which a caller's workspace
  // sized for rows alone may not have.
  const int64_t slabs = c.B * c.H_kv;
  o.tiled = c.D == 128 ||
            (c.D > 128 && (c.library_scratch ||
                           c.ws_bytes >= once_bytes(slabs, once_slab_rows(true, o.keys), c.D)));
  o.slab_rows = once_slab_rows(o.tiled, o.keys);
  o.bytes = once_bytes(slabs, o.slab_rows, c.D);
  if (!c.library_scratch && c.ws_bytes < o.bytes) return o;
  const int64_t few = slabs <= kOnceMaxSlabs ? once_blocks(c.D, o.keys) : kOnceBlocks;
  o.on = force == 1 || (c.blocks >= few &&
                        once_bytes(slabs, o.keys, c.D) <= kOnceMaxBytes);
  return o;
}

// Key splits of a chunk whose row blocks would leave CUs idle (a short chunk
// over a long context): workgroups wanted, keys a split holds at least (a
// split pays its partials' write and read), bytes of partials at most.
// Measured (4-bit, without and with): 16 / 8 heads, D = 128, 64 rows over
// 24,000 keys 569 and 42 us, 147 rows over 16,384 565 and 55; D = 256, 256
// rows over 16,384 661 and 104; 32 / 2 heads, D = 512, 64 rows over 20,000
// 2,700 and 134 (with the wide kernel).
// The keys a split holds are counted of what one row block sees: under a window
// a block sees no more than the window and its own positions, and splits of
// the chunk's whole range cost it their partials for nothing (D = 256, 8 heads,
// 700 rows under a window of 512: 38 us unsplit, 47 in two splits of the range;
// 300 rows under a window of 1,024: 44 us in two, 36 in three, even ones).
// Not over bf16 rows: a codebook cache's dequantized rows and rotated queries
// sit in the library scratch that the partials would take, and a bf16 cache's
// chunk uses no scratch, so that caches on different streams stay independent.
constexpr int64_t kSplitWorkgroups = 256, kSplitMinKeys = 512;
constexpr size_t kSplitMaxBytes = size_t(1) << 30;

struct Splits {
  int64_t n = 1, len = 0, lo = 0;  // split s: keys lo + [s * len, (s + 1) * len)
  size_t bytes = 0;                // of partials (0: the keys are not split)
};
inline Splits no_splits(const Chunk& c) {
  Splits s;
  s.len = (c.total + kTileKeys - 1) / kTileKeys * kTileKeys;
  return s;
}
inline Splits key_splits(const Chunk& c) {
  Splits s = no_splits(c);
  const int64_t units = c.blocks * c.H_kv * c.B, rows = c.B * c.H * c.L;
  if (c.bf16_rows || !c.library_scratch || units * 2 > kSplitWorkgroups) return s;
  const Visible v = visible_keys(c);
  const int64_t keys = v.hi + 1 - v.lo;
  int64_t most = keys;  // that a row block sees
  if (c.causal && c.window >= 0) {
    const int64_t at = c.block_rows * c.H_kv / c.H + 1;  // positions it spans at most
    const int64_t own = (at < c.L ? at : c.L) - 1;
    if (most > c.window && most - c.window > own) most = c.window + own;
  }
  const int64_t room = kSplitWorkgroups / units;
  int64_t n = room;
  if (n > (most - 1) / kSplitMinKeys) n = (most - 1) / kSplitMinKeys;
  if (n < 2) return s;
  const auto whole = [](int64_t len) { return (len + kTileKeys - 1) / kTileKeys * kTileKeys; };
  int64_t len = whole((most + n - 1) / n);
  n = (keys + len - 1) / len;
  if (most < keys) {  // the same number of splits, even over the whole range
    if (n > room) n = room;
    len = whole((keys + n - 1) / n);
    n = (keys + len - 1) / len;
  }
  const size_t slot = size_t(c.D + 2) * sizeof(float);
  if (n < 2 || size_t(rows) * size_t(n) * slot > kSplitMaxBytes) return s;
  s.n = n;
  s.len = len;
  s.lo = v.lo;
  s.bytes = size_t(rows) * size_t(n) * slot;
  return s;
}

}  // namespace prefillplan
}  // namespace tqkv

"""The prefill's plan (lumen-rs_amd/csrc/prefill_plan.hpp) over all forms of a
call, on the CPU: which keys a chunk sees, and how they are split."""
import ctypes
import os
import random
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
BUILD = os.path.join(ROOT, "tests", "_build")
LIB = os.path.join(BUILD, "libprefillplanhost.so")
FIELDS = ("B", "H", "Hkv", "L", "D", "total", "q_start", "k_start", "causal", "window",
          "block_rows", "blocks", "bf16_rows", "library_scratch", "ws_bytes")
ROWS = {64: 128, 128: 256, 256: 128, 512: 64}  # rows a block of the in-block kernel


@pytest.fixture(scope="module")
def host():
    os.makedirs(BUILD, exist_ok=True)
    subprocess.run(["g++", "-O2", "-std=c++17", "-Wall", "-Werror", "-shared", "-fPIC",
                    "-I", os.path.join(ROOT, "lumen-rs_amd", "csrc"),
                    os.path.join(ROOT, "tests", "prefill_plan_host.cpp"), "-o", LIB], check=True)
    return ctypes.CDLL(LIB)


def ask(fn, c, n, *more):
    out = (ctypes.c_int64 * n)()
    fn((ctypes.c_int64 * len(FIELDS))(*(int(c[f]) for f in FIELDS)), *map(ctypes.c_int64, more), out)
    return list(out)


def once(host, c, force=-1):
    return dict(zip(("on", "lo", "keys", "slab_rows", "tiled", "bytes"),
                    ask(host.planhost_once, c, 6, force)))


def blocked(c):
    c["block_rows"] = ROWS[c["D"]]
    c["blocks"] = -(-c["L"] * (c["H"] // c["Hkv"]) // ROWS[c["D"]])
    return c


def chunk(rng, **fixed):
    D = rng.choice((64, 128, 256, 512))
    Hkv = rng.choice((1, 2, 4, 8))
    G = rng.choice((1, 2, 3, 4, 8, 16))
    L = int(2 ** rng.uniform(0, 12))
    total = int(2 ** rng.uniform(0, 17))
    c = dict(B=rng.choice((1, 1, 2, 5)), H=Hkv * G, Hkv=Hkv, L=L, D=D, total=total,
             k_start=rng.choice((0, 0, 40, 100000)), causal=rng.random() < 0.8,
             window=rng.choice((-1, -1, 1, 100, 1500, 1 << 40)), bf16_rows=False,
             library_scratch=rng.random() < 0.8, ws_bytes=0)
    c["q_start"] = rng.choice((c["k_start"] + total - L, 0, c["k_start"] + total // 2))
    c.update(fixed)
    return blocked(c)


def seen(c):
    """The keys that some row sees, by the mask's own rule."""
    if not c["causal"]:
        return 0, c["total"] - 1
    first = max(c["q_start"] - c["k_start"], 0)  # the rows that see a key
    last = c["q_start"] + c["L"] - 1 - c["k_start"]
    if c["window"] >= 0:
        last = min(last, c["total"] + c["window"] - 2)
    if first > last:
        return 0, -1
    return max(0, first - c["window"] + 1) if c["window"] >= 0 else 0, min(c["total"] - 1, last)


def test_visible_keys_cover_what_rows_see(host):
    rng = random.Random(1)
    for _ in range(3000):
        c = chunk(rng)
        lo, hi = ask(host.planhost_visible, c, 2)
        a, b = seen(c)
        if a <= b:
            assert lo % 64 == 0 and lo <= a and hi >= b and hi < c["total"], (c, lo, hi)


def test_splits_cover_the_visible_keys(host):
    rng = random.Random(2)
    split = 0
    for _ in range(3000):
        c = chunk(rng)
        n, ln, lo, size = ask(host.planhost_splits, c, 4)
        a, b = seen(c)
        assert n >= 1 and ln % 64 == 0 and lo % 64 == 0
        if a <= b:
            assert lo <= a and lo + n * ln > b, (c, n, ln, lo)
        assert (size > 0) == (n > 1)
        if n > 1:
            split += 1
            assert c["library_scratch"] and lo + (n - 1) * ln <= b, c  # none is empty
            assert n * c["blocks"] * c["Hkv"] * c["B"] <= 256
            assert size == c["B"] * c["H"] * c["L"] * n * (c["D"] + 2) * 4 <= 1 << 30
    assert split > 100


def test_bf16_rows_are_never_split(host):
    # A codebook cache's chunk attends dequantized rows and rotated queries
    # that sit in the library scratch, where partials would overwrite them; a
    # bf16 cache's uses no scratch, so that two caches on two streams do not
    # meet there.
    rng = random.Random(3)
    c = chunk(rng, B=1, H=32, Hkv=8, L=64, D=128, total=8192, q_start=8128, k_start=0, causal=True,
              window=-1, library_scratch=True)
    assert ask(host.planhost_splits, c, 4)[0] > 1  # packed codes at this shape are
    for D in (64, 128, 256, 512):
        for _ in range(500):
            n, _, lo, size = ask(host.planhost_splits, chunk(rng, D=D, bf16_rows=True), 4)
            assert (n, lo, size) == (1, 0, 0)


def test_dequantize_once_takes_the_visible_keys_alone(host):
    rng = random.Random(4)
    seen_once = 0
    for _ in range(4000):
        c = chunk(rng)
        if not c["library_scratch"]:
            c["ws_bytes"] = rng.choice((0, 1 << 20, 1 << 33))
        o = once(host, c)
        a, b = seen(c)
        if a > b:
            assert not o["on"], c
            continue
        assert o["lo"] == a // 64 * 64 and o["lo"] + o["keys"] == b + 1, (c, o)
        if not o["on"]:
            continue
        seen_once += 1
        assert o["slab_rows"] == (-(-o["keys"] // 64) * 64 if o["tiled"] else o["keys"])
        assert o["bytes"] == 4 * c["B"] * c["Hkv"] * o["slab_rows"] * c["D"]
        assert c["library_scratch"] or o["bytes"] <= c["ws_bytes"]
        assert o["tiled"] == (c["D"] >= 128) or not c["library_scratch"]
    assert seen_once > 500


@pytest.mark.parametrize("D", [256, 512])
def test_a_window_over_a_long_cache_is_priced_by_its_own_keys(host, D):
    # A few row blocks that see 1,000 of 60,000 keys.
    c = dict(B=1, H=16, Hkv=8, L=300, D=D, total=60000, q_start=59700, k_start=0, causal=True,
             window=700, bf16_rows=False, library_scratch=True, ws_bytes=0)
    o = once(host, blocked(c))
    assert o["on"] == (D == 512)  # at D = 256 the rule for few blocks asks for 2,048 keys
    assert o["keys"] < 1064 and o["lo"] + o["keys"] == 60000
    if o["on"]:
        assert o["bytes"] < 4 * 8 * 1100 * D


def test_dequantize_once_never_takes_bf16_rows(host):
    rng = random.Random(5)
    for force in (-1, 1):
        for _ in range(500):
            assert not once(host, chunk(rng, bf16_rows=True), force)["on"]


def test_more_slabs_than_the_pass_takes_stay_in_block(host):
    # Fewer than 8 row blocks over more than 65,535 slabs are attended in
    # block; 8 or more are the pass's, whose launch refuses them.
    c = dict(B=8192, H=8, Hkv=8, L=1, D=512, total=3, q_start=2, k_start=0, causal=True, window=-1,
             block_rows=64, blocks=1, bf16_rows=False, library_scratch=True, ws_bytes=0)
    assert not once(host, c)["on"] and once(host, dict(c, B=8191))["on"]
    assert not once(host, dict(c, blocks=7))["on"] and once(host, dict(c, blocks=8))["on"]


def test_a_window_splits_by_what_a_row_block_sees(host):
    # A row block under a window sees the window and its own positions, however
    # many keys the whole chunk sees: it takes two splits' keys or none is made.
    base = dict(B=1, H=8, Hkv=8, L=700, D=256, total=1211, q_start=511, k_start=0, causal=True,
                window=512, bf16_rows=False, library_scratch=True, ws_bytes=0)
    assert ask(host.planhost_splits, blocked(dict(base)), 4)[0] == 1
    assert ask(host.planhost_splits, blocked(dict(base, window=-1)), 4)[0] == 2
    rng = random.Random(6)
    split = 0
    for _ in range(3000):
        c = chunk(rng, causal=True, window=rng.choice((100, 600, 1024, 1500, 4000)))
        n, ln = ask(host.planhost_splits, c, 4)[:2]
        if n == 1:
            continue
        split += 1
        sees = 0  # the most that a row block does
        G, q0 = c["H"] // c["Hkv"], c["q_start"] - c["k_start"]
        for r in range(0, c["L"] * G, c["block_rows"]):
            first, last = r // G, (min(r + c["block_rows"], c["L"] * G) - 1) // G
            a, b = max(0, q0 + first - c["window"] + 1), min(c["total"] - 1, q0 + last)
            sees = max(sees, b - a + 1)
        assert sees + 64 > 1024 and ln >= 256, (c, n, ln, sees)
    assert split > 50


def test_splits_without_a_window_are_even(host):
    # At least 512 keys a split, at most 256 workgroups, whole tiles.
    rng = random.Random(7)
    for _ in range(3000):
        c = chunk(rng, window=-1, library_scratch=True, k_start=0)
        n, ln = ask(host.planhost_splits, c, 4)[:2]
        a, b = seen(c)
        keys, units = b + 1 - a, c["blocks"] * c["Hkv"] * c["B"]
        want = min(256 // units, (keys - 1) // 512) if units <= 128 else 1
        cut = -(-keys // (want * 64)) * 64 if want > 1 else 0
        want = -(-keys // cut) if cut else 1
        if want < 2 or c["B"] * c["H"] * c["L"] * want * (c["D"] + 2) * 4 > 1 << 30:
            assert n == 1
        else:
            assert (n, ln) == (want, cut), c

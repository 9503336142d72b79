"""Performance cases of the compressed KV cache, through its public entry points.

A case is a dict of plain values; `kind` names the call a serving program makes:

  decode    one decode step over an affine cache: quantize the new token, attend
  stack     one decode step of a whole model through the cache objects
  prefix    one decode step of sequences that share a prompt prefix
  prefill   chunk attention over an affine cache (causal, with or without a window)
  append    quantize a chunk's keys and values into the cache
  codebook  one decode step's attention over a TurboQuant codebook cache
  encode    compress a chunk's keys and values into a codebook cache

listed() gives the fixed cases, draw() more of the same ranges, prepare() the
inputs of one, run() one pass, work() what a pass cannot do without,
tolerance() how far two correct implementations may be apart, exact() the
outputs in 64 bits by plain torch.
"""
import math
import os
import sys

import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(_ROOT, "lumen-rs_amd"))
import tqkv as T  # noqa: E402

# One HIP runtime a process: the buffers here are torch's, so the library is
# given the runtime that torch has loaded.
_TORCH_HIP = os.path.join(os.path.dirname(torch.__file__), "lib", "libamdhip64.so")
if os.path.exists(_TORCH_HIP):
    T.HIP_PATH = _TORCH_HIP

_CHUNK = 1 << 25  # elements handled at a time while inputs are made


def listed():
    return [
        # A single user's decode step at a medium context (32 query / 8 KV heads): latency.
        dict(name="decode_single", kind="decode", B=1, H=32, Hkv=8, D=128, n=8192, bk=4, bv=4, gs=64),
        # The headline: a serving batch at 32K context, 3-bit cache: HBM bandwidth.
        dict(name="decode_batch_32k", kind="decode", B=32, H=16, Hkv=8, D=256, n=32768, bk=3, bv=3, gs=64),
        # Gemma 4's full-attention layers: 32 heads over 2 KV heads, head dim 512, ragged context.
        dict(name="decode_gemma_global", kind="decode", B=4, H=32, Hkv=2, D=512, n=8179, bk=4, bv=4, gs=64),
        # A decode step of all 30 layers (5 global, 25 sliding rings of 1,024) through the caches.
        dict(name="decode_stack_30", kind="stack", B=4, H=32, Hkv=8, D=128, n=16450, bits=4, layers=30, window=1024),
        # Eight sequences over one shared 64K prompt, each with its own suffix; 8-bit K, 4-bit V.
        dict(name="decode_shared_prefix", kind="prefix", B=8, H=32, Hkv=8, D=128, n=65536, own=4096, bk=8, bv=4),
        # The last 2,048-token chunk of a 16K prompt on a global layer: matrix cores.
        dict(name="prefill_global_128", kind="prefill", B=4, H=32, Hkv=8, D=128, L=2048, n=16384, bk=4, bv=4, gs=64, window=-1),
        # A Gemma sliding layer's chunk: head dim 256, groups of 32, a ring's 1,023 older keys.
        dict(name="prefill_gemma_sliding", kind="prefill", B=2, H=32, Hkv=16, D=256, L=2048, n=3071, bk=4, bv=4, gs=32, window=1024),
        # A Gemma 4 full-attention chunk: head dim 512, 16 query heads a KV head.
        dict(name="prefill_gemma_global", kind="prefill", B=1, H=32, Hkv=2, D=512, L=2048, n=8192, bk=4, bv=4, gs=64, window=-1),
        # Quantize-on-append of a prompt chunk: 8 KV heads x 4,096 tokens, K and V.
        dict(name="append_chunk", kind="append", slabs=8, s=4096, D=128, bk=4, bv=4, gs=64, rotated=False),
        # The headline shape over a 3-bit TurboQuant codebook cache.
        dict(name="codebook_batch_32k", kind="codebook", B=32, H=16, Hkv=8, D=256, n=32768, bits=3, m=0),
        # Gemma 4's full-attention layers over a 4-bit codebook cache, one sequence.
        dict(name="codebook_gemma_global", kind="codebook", B=1, H=32, Hkv=2, D=512, n=32768, bits=4, m=0),
        # A prompt chunk into a codebook cache: rotate and encode K and V, as the cache object calls it.
        dict(name="codebook_append", kind="encode", slabs=8, s=2048, D=256, bits=4, path="gpu", transpose=True, m=0),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("decode", "decode", "stack", "prefix", "prefill", "prefill", "prefill", "append", "codebook", "codebook", "encode"))
    if kind == "decode":
        D = rng.choice((64, 128, 256, 512))
        H, Hkv = rng.choice(((8, 8), (16, 8), (32, 8), (32, 16), (24, 8))) if D < 512 else rng.choice(((32, 2), (16, 2), (16, 4)))
        bk, bv = rng.choice(((3, 3), (4, 4), (4, 4), (6, 6), (8, 8), (8, 4)))
        c = dict(kind=kind, B=_log(rng, 1, 32), H=H, Hkv=Hkv, D=D, n=_log(rng, 16, 65536), bk=bk, bv=bv, gs=rng.choice((32, 64, 64)))
        while work(c)["bytes"] > 1.8e9:
            c["n"] = c["n"] // 2 + 1
        return c
    if kind == "stack":
        return dict(kind=kind, B=_log(rng, 1, 8), H=rng.choice((16, 32)), Hkv=8, D=rng.choice((64, 128)), n=_log(rng, 500, 16000),
                    bits=rng.choice((4, 8)), layers=rng.choice((12, 18, 24, 30)), window=rng.choice((512, 1024)))
    if kind == "prefix":
        return dict(kind=kind, B=rng.randint(2, 16), H=rng.choice((16, 32)), Hkv=8, D=rng.choice((64, 128, 256)), n=_log(rng, 2048, 131072),
                    own=_log(rng, 16, 8192), bk=8, bv=rng.choice((4, 8)))
    if kind == "prefill":
        D = rng.choice((64, 128, 256, 512))
        H, Hkv = rng.choice(((16, 8), (32, 8), (32, 16))) if D < 512 else rng.choice(((32, 2), (16, 2), (16, 4)))
        L = _log(rng, 64, 4096)
        window = rng.choice((-1, -1, 512, 1024))
        n = L + (_log(rng, 16, 24576) if window < 0 else window - 1)
        c = dict(kind=kind, B=rng.choice((1, 2, 4)), H=H, Hkv=Hkv, D=D, L=L, n=n, bk=rng.choice((3, 4, 4, 8)), gs=rng.choice((32, 64, 64)), window=window)
        c["bv"] = 4 if c["bk"] == 8 and rng.random() < 0.5 else c["bk"]
        while work(c)["flops"] > (0.85e12 if D == 512 else 1.9e12 if D == 128 else 1.2e12):
            if c["B"] > 1:
                c["B"] //= 2
            else:
                cut = c["n"] - c["L"] - (c["n"] - c["L"]) // 2 if window < 0 else 0
                c["n"], c["L"] = (c["n"] - cut, c["L"]) if cut > 64 else (c["n"] - c["L"] // 2, c["L"] - c["L"] // 2)
        return c
    if kind == "append":
        c = dict(kind=kind, slabs=rng.choice((2, 8, 16, 32)), s=_log(rng, 1, 8192), D=rng.choice((64, 128, 256, 512)), gs=rng.choice((32, 64, 64)), rotated=False)
        c["bk"], c["bv"] = rng.choice(((3, 3), (4, 4), (6, 6), (8, 8), (8, 4)))
        c["rotated"] = c["D"] in (128, 256) and rng.random() < 0.3
        return c
    if kind == "codebook":
        D = rng.choice((64, 128, 256, 512))
        H, Hkv = rng.choice(((8, 8), (16, 8), (32, 8))) if D < 512 else rng.choice(((32, 2), (16, 2), (16, 4)))
        c = dict(kind=kind, B=_log(rng, 1, 32), H=H, Hkv=Hkv, D=D, n=_log(rng, 64, 65536), bits=rng.choice((2, 3, 4, 4, 6)), m=rng.choice((0, 0, 0, 64)))
        while work(c)["bytes"] > (1e9 if c["m"] or D != 256 else 4e9):
            c["n"] = c["n"] // 2 + 1
        return c
    c = dict(kind=kind, slabs=rng.choice((2, 4, 8, 16)), s=_log(rng, 1, 8192), D=rng.choice((64, 128, 256, 512)), bits=rng.choice((2, 3, 4, 4)),
             path=rng.choice(("gpu", "gpu", "cpu")), transpose=rng.random() < 0.7, m=0)
    c["m"] = 64 if c["path"] == "cpu" and rng.random() < 0.5 else 0
    while c["slabs"] * c["s"] * c["D"] ** 2 > 1.1e9:
        c["s"] = c["s"] // 2 + 1
    return c


# ------------------------------------------------------------------ sizes
def _row_bytes(D, bits, gs):
    return D * bits // 8 + 4 * (D // gs)


def _visible(L, n, window):
    """(query, key) pairs of a causal chunk of L queries ending at key n."""
    pairs = L * n - L * (L - 1) // 2
    if window > 0:  # query i (of L) sees keys (n - L + i - window, n - L + i]
        first = n - L + 1
        over = max(0, n - window) - max(0, first - window - 1)
        a, b = max(1, first - window), n - window
        pairs -= (a + b) * over // 2 if over else 0
    return pairs


def work(case):
    c, k = case, case["kind"]
    if k == "decode":
        row = _row_bytes(c["D"], c["bk"], c["gs"]) + _row_bytes(c["D"], c["bv"], c["gs"])
        kv = c["B"] * c["Hkv"] * (c["n"] + 1) * row
        return {"bytes": kv + 4 * c["B"] * (c["H"] + c["Hkv"]) * c["D"], "flops": 4 * c["B"] * c["H"] * c["D"] * (c["n"] + 1)}
    if k == "stack":
        keys = sum(c["n"] + 1 if g else min(c["n"] + 1, c["window"]) for g in _stack_global(c))
        return {"bytes": c["B"] * c["Hkv"] * keys * 2 * _row_bytes(c["D"], c["bits"], 64) + c["layers"] * 4 * c["B"] * c["H"] * c["D"],
                "flops": 4 * c["B"] * c["H"] * c["D"] * keys}
    if k == "prefix":
        row = _row_bytes(c["D"], c["bk"], 64) + _row_bytes(c["D"], c["bv"], 64)
        return {"bytes": c["Hkv"] * (c["n"] + c["B"] * (c["own"] + 1)) * row + 4 * c["B"] * (c["H"] + c["Hkv"]) * c["D"],
                "flops": 4 * c["B"] * c["H"] * c["D"] * (c["n"] + c["own"] + 1)}
    if k == "prefill":
        row = _row_bytes(c["D"], c["bk"], c["gs"]) + _row_bytes(c["D"], c["bv"], c["gs"])
        return {"bytes": c["B"] * c["Hkv"] * c["n"] * row + 4 * c["B"] * c["H"] * c["L"] * c["D"],
                "flops": 4 * c["B"] * c["H"] * c["D"] * _visible(c["L"], c["n"], c["window"])}
    if k == "append":
        rows = c["slabs"] * c["s"]
        return {"bytes": rows * (4 * c["D"] + _row_bytes(c["D"], c["bk"], c["gs"]) + _row_bytes(c["D"], c["bv"], c["gs"])),
                "flops": 2 * rows * c["D"] ** 2 if c["rotated"] else 0}
    if k == "codebook":
        row = 2 * (c["D"] + 4) + (c["m"] // 8 + 4 if c["m"] else 0)
        return {"bytes": c["B"] * c["Hkv"] * c["n"] * row + 4 * c["B"] * c["H"] * c["D"] + 4 * c["D"] ** 2,
                "flops": 4 * c["B"] * c["H"] * c["D"] * c["n"] + 4 * c["B"] * c["H"] * c["D"] ** 2}
    rows = 2 * c["slabs"] * c["s"]  # K and V
    m = 2 * c["m"] * c["D"] if c["path"] == "cpu" else 0
    back = 2 * c["D"] ** 2 if c["m"] else 0  # the residual's reconstruction
    return {"bytes": rows * (3 * c["D"] + 4 + (c["m"] // 8 + 4 if c["m"] else 0)) + 4 * c["D"] ** 2, "flops": rows * (2 * c["D"] ** 2 + back + m)}


def tolerance(case):
    k = case["kind"]
    if k == "append":
        # Packed codes and bf16 scales are whole results (the quantizer is bit-exact); a
        # rotated key's f32 sum may round to the other bf16 neighbour in another order.
        return {"rel": 4e-3, "max": 0.3, "differ": 0.002} if case["rotated"] else "exact"
    if k == "encode":
        return {"rel": 2e-5, "max": 1e-3, "differ": 0.0}  # codes and signs are whole results
    # bf16 outputs of f32 sums (half a step is up to 2^-9 of a value) with the new token's
    # and the cache's bytes bit-exact.
    return {"rel": 1e-2, "max": 0.2, "differ": 0.0}


# ------------------------------------------------------------------ inputs
class _Rand:
    """Seeded draws on the device."""

    def __init__(self, case, seed):
        self.g = torch.Generator(device="cuda")
        salt = sum((i + 1) * ord(ch) for i, ch in enumerate(repr(sorted((k, v) for k, v in case.items() if k != "name")))) % 100003
        self.g.manual_seed(int(seed) * 100003 + salt)

    def normal(self, *shape):
        return torch.randn(shape, generator=self.g, device="cuda")

    def uniform(self, lo, hi, *shape):
        return torch.rand(shape, generator=self.g, device="cuda") * (hi - lo) + lo

    def words(self, *shape):
        return torch.randint(-2 ** 31, 2 ** 31, shape, generator=self.g, device="cuda").to(torch.int32)

    def rows(self, *shape):
        """bf16 K or V rows: N(0, 1) with 2% of the channels eight times larger."""
        x = self.normal(*shape)
        big = torch.rand(shape[-1], generator=self.g, device="cuda") < 0.02
        return (x * torch.where(big, 8.0, 1.0)).to(torch.bfloat16)

    def query(self, *shape):
        return self.normal(*shape).to(torch.bfloat16)


def _round_away(x):
    t = torch.trunc(x)
    return t + torch.where((x - t).abs() >= 0.5, torch.sign(x), torch.zeros_like(x))


def _quantize(x, bits, gs):
    """The affine triple (packed int32, scales bf16, biases bf16) of bf16 rows [..., D], by plain torch."""
    D = x.shape[-1]
    v = x.float().reshape(-1, D // gs, gs)
    bins = torch.tensor(float(2 ** bits - 1), device=x.device)  # a tensor: a divide by a plain number is a multiply
    lo, hi = v.amin(-1), v.amax(-1).clamp_min(0.0)
    scale = torch.clamp_min((hi - lo) / bins, 1e-7)
    side = lo.abs() > hi.abs()
    scale = torch.where(side, scale, -scale)
    edge = torch.where(side, lo, hi)
    q0 = _round_away(edge / scale)
    zero = q0 == 0
    scale = torch.where(zero, scale, edge / torch.where(zero, torch.ones_like(q0), q0))
    bias = torch.where(zero, torch.zeros_like(edge), edge)
    code = _round_away((v - bias[..., None]) / scale[..., None]).clamp(0.0, float(2 ** bits - 1))
    code = code.to(torch.int64).reshape(-1, D // 32, 32)
    words = torch.zeros(code.shape[:-1] + (bits,), dtype=torch.int64, device=x.device)
    for i in range(32):  # 32 codes are `bits` words, least significant bit first
        w, off = divmod(i * bits, 32)
        words[..., w] |= code[..., i] << off
        if off + bits > 32:
            words[..., w + 1] |= code[..., i] >> (32 - off)
    words &= 0xffffffff
    words = torch.where(words >= 2 ** 31, words - 2 ** 32, words).to(torch.int32)
    lead = x.shape[:-1]
    return words.reshape(*lead, D * bits // 32), scale.to(torch.bfloat16).reshape(*lead, D // gs), bias.to(torch.bfloat16).reshape(*lead, D // gs)


def _dequantize(t, bits, gs, dtype=torch.float64):
    """scale * code + bias of a triple's rows."""
    words, scales, biases = t
    lead, D = words.shape[:-1], words.shape[-1] * 32 // bits
    w = (words.to(torch.int64) & 0xffffffff).reshape(-1, D // 32, bits)
    code = torch.empty(w.shape[:-1] + (32,), dtype=dtype, device=words.device)
    for i in range(32):
        j, off = divmod(i * bits, 32)
        c = w[..., j] >> off
        if off + bits > 32:
            c = c | (w[..., j + 1] << (32 - off))
        code[..., i] = (c & (2 ** bits - 1)).to(dtype)
    code = code.reshape(-1, D // gs, gs)
    s, b = (z.to(dtype).reshape(-1, D // gs, 1) for z in (scales, biases))
    return (code * s + b).reshape(*lead, D)


def _affine_cache(r, slabs, n, cap, D, bits, gs):
    """A cache's triple [slabs, cap, .] with rows [0, n) quantized from seeded values."""
    out = (torch.zeros(slabs, cap, D * bits // 32, dtype=torch.int32, device="cuda"),
           torch.zeros(slabs, cap, D // gs, dtype=torch.bfloat16, device="cuda"),
           torch.zeros(slabs, cap, D // gs, dtype=torch.bfloat16, device="cuda"))
    step = max(1, _CHUNK // (n * D))
    rows = max(1, min(n, _CHUNK // D))
    for a in range(0, slabs, step):
        b = min(slabs, a + step)
        for t in range(0, n, rows):
            e = min(n, t + rows)
            for dst, src in zip(out, _quantize(r.rows(b - a, e - t, D), bits, gs)):
                dst[a:b, t:e] = src
    return out


def _ptrs(ts):
    return tuple(t.data_ptr() for t in ts)


def _bytes(n):
    return torch.zeros(max(int(n), 16), dtype=torch.uint8, device="cuda")


def _decode_inputs(c, seed):
    r = _Rand(c, seed)
    slabs, cap = c["B"] * c["Hkv"], (c["n"] + 1 + 255) // 256 * 256
    kt = _affine_cache(r, slabs, c["n"], cap, c["D"], c["bk"], c["gs"])
    vt = _affine_cache(r, slabs, c["n"], cap, c["D"], c["bv"], c["gs"])
    return kt, vt, r.query(c["B"], c["H"], 1, c["D"]), r.rows(slabs, 1, c["D"]), r.rows(slabs, 1, c["D"]), cap


def _prepare_decode(c, seed):
    B, H, Hkv, D, n, gs, bk, bv = (c[x] for x in ("B", "H", "Hkv", "D", "n", "gs", "bk", "bv"))
    kt, vt, q, nk, nv, cap = _decode_inputs(c, seed)
    out = torch.zeros(B, H, 1, D, dtype=torch.bfloat16, device="cuda")
    ws = _bytes(T.decode_workspace_size(B, H, Hkv, D, cap))
    kp, vp, scale = _ptrs(kt), _ptrs(vt), D ** -0.5
    qp, nkp, nvp, op, wp, wb = *_ptrs((q, nk, nv, out, ws)), ws.numel()
    if T.decode_kernel_for_rows(H, Hkv, D, gs, bk, bv, n) == "mfma":  # the fused step's layouts
        segs = [T.affine_seg(kp, vp, cap, n)]

        def call():
            T.decode_attend_affine_append(qp, B, H, Hkv, D, gs, bk, bv, scale, segs, nkp, nvp, kp + vp, cap, n, op, wp, wb)
    else:
        segs = [T.affine_seg(kp, vp, cap, n + 1)]

        def call():
            T.affine_quantize_kv(nkp, nvp, B * Hkv, 1, D, gs, bk, bv, kp, vp, cap, n)
            T.decode_attend_affine(qp, B, H, Hkv, D, gs, bk, bv, scale, segs, op, wp, wb)
    # The attention and the rows the step writes into the cache.
    return call, [out] + [t[:, n] for t in kt + vt], (kt, vt, q, nk, nv, ws)


def _stack_global(c):
    """Which layers attend globally: every sixth, as Gemma's 5:1 pattern."""
    return [i % 6 == 5 for i in range(c["layers"])]


def _stack_inputs(c, seed):
    r = _Rand(c, seed)
    slabs = c["B"] * c["Hkv"]
    for g in _stack_global(c):
        n = c["n"] if g else min(c["n"], c["window"])
        yield g, n, r.rows(slabs, n, c["D"]), r.rows(slabs, n, c["D"]), r.rows(slabs, 1, c["D"]), r.rows(slabs, 1, c["D"]), r.query(c["B"], c["H"], 1, c["D"])


def _prepare_stack(c, seed):
    B, H, Hkv, D, bits = (c[x] for x in ("B", "H", "Hkv", "D", "bits"))
    layers, keep = [], []
    ws = _bytes(T.decode_workspace_size(B, H, Hkv, D, c["n"] + 256))
    for g, n, k, v, nk, nv, q in _stack_inputs(c, seed):
        cache = T.Cache(T.CACHE_AFFINE, B, Hkv, D, D, 64, bits, bits, prealloc=True, max_size=0 if g else c["window"])
        cache.append(k.data_ptr(), v.data_ptr(), n)
        out = torch.zeros(B, H, 1, D, dtype=torch.bfloat16, device="cuda")
        layers.append((cache, n if g else 0) + _ptrs((nk, nv, q, out)))
        keep.append((nk, nv, q, out))
        torch.cuda.synchronize()  # k and v are read before they go
    wp, wb = ws.data_ptr(), ws.numel()

    def call():
        for cache, n, nk, nv, q, out in layers:
            if n:
                cache.truncate(n)  # the step before is taken back, so that every pass is this one
            cache.append_decode(nk, nv, q, H, 1.0 / math.sqrt(D), out, wp, wb)
    return call, [x[3] for x in keep], (layers, keep, ws)


def _prefix_inputs(c, seed):
    r = _Rand(c, seed)
    B, Hkv, D, cap = c["B"], c["Hkv"], c["D"], (c["own"] + 256) // 256 * 256
    pk, pv = (_affine_cache(r, Hkv, c["n"], c["n"], D, c[b], 64) for b in ("bk", "bv"))
    sk, sv = (_affine_cache(r, B * Hkv, c["own"], cap, D, c[b], 64) for b in ("bk", "bv"))
    return pk, pv, sk, sv, r.query(B, c["H"], 1, D), r.rows(B * Hkv, 1, D), r.rows(B * Hkv, 1, D), cap


def _prepare_prefix(c, seed):
    B, H, Hkv, D, n, own, bk, bv = (c[x] for x in ("B", "H", "Hkv", "D", "n", "own", "bk", "bv"))
    pk, pv, sk, sv, q, nk, nv, cap = _prefix_inputs(c, seed)
    out = torch.zeros(B, H, 1, D, dtype=torch.bfloat16, device="cuda")
    ws = _bytes(T.decode_workspace_size(B, H, Hkv, D, n + cap))
    kp, vp, scale = _ptrs(sk), _ptrs(sv), D ** -0.5
    qp, nkp, nvp, op, wp, wb = *_ptrs((q, nk, nv, out, ws)), ws.numel()
    shared = T.affine_seg(_ptrs(pk), _ptrs(pv), n, n, True)
    if T.decode_kernel_for_rows(H, Hkv, D, 64, bk, bv, max(n, own)) == "mfma":
        segs = [shared, T.affine_seg(kp, vp, cap, own)]

        def call():
            T.decode_attend_affine_append(qp, B, H, Hkv, D, 64, bk, bv, scale, segs, nkp, nvp, kp + vp, cap, own, op, wp, wb)
    else:
        segs = [shared, T.affine_seg(kp, vp, cap, own + 1)]

        def call():
            T.affine_quantize_kv(nkp, nvp, B * Hkv, 1, D, 64, bk, bv, kp, vp, cap, own)
            T.decode_attend_affine(qp, B, H, Hkv, D, 64, bk, bv, scale, segs, op, wp, wb)
    return call, [out] + [t[:, own] for t in sk + sv], (pk, pv, sk, sv, q, nk, nv, ws)


def _prefill_inputs(c, seed):
    r = _Rand(c, seed)
    slabs = c["B"] * c["Hkv"]
    kt, vt = (_affine_cache(r, slabs, c["n"], c["n"], c["D"], c[b], c["gs"]) for b in ("bk", "bv"))
    return kt, vt, r.query(c["B"], c["H"], c["L"], c["D"])


def _prepare_prefill(c, seed):
    B, H, Hkv, D, L, n, gs, bk, bv, window = (c[x] for x in ("B", "H", "Hkv", "D", "L", "n", "gs", "bk", "bv", "window"))
    kt, vt, q = _prefill_inputs(c, seed)
    out = torch.zeros(B, H, L, D, dtype=torch.bfloat16, device="cuda")
    segs, scale = [T.affine_seg(_ptrs(kt), _ptrs(vt), n, n)], D ** -0.5
    qp, op = _ptrs((q, out))

    def call():
        T.prefill_attend_affine(qp, B, H, Hkv, L, D, gs, bk, bv, scale, segs, op, q_start=n - L, k_start=0, causal=True, window=window)
    return call, [out], (kt, vt, q)


def _rotation(r, D):
    return torch.linalg.qr(r.normal(D, D).double().cpu())[0].float().contiguous().cuda()


def _append_inputs(c, seed):
    r = _Rand(c, seed)
    k, v = (r.rows(c["slabs"], c["s"], c["D"]) for _ in range(2))
    return k, v, _rotation(r, c["D"]) if c["rotated"] else None


def _prepare_append(c, seed):
    slabs, s, D, gs, bk, bv = (c[x] for x in ("slabs", "s", "D", "gs", "bk", "bv"))
    k, v, R = _append_inputs(c, seed)
    kt, vt = (tuple(torch.zeros(slabs, s, w, dtype=d, device="cuda") for w, d in
                    ((D * b // 32, torch.int32), (D // gs, torch.bfloat16), (D // gs, torch.bfloat16))) for b in (bk, bv))
    kx, vx, kp, vp = k.data_ptr(), v.data_ptr(), _ptrs(kt), _ptrs(vt)
    if c["rotated"]:
        rp = R.data_ptr()

        def call():
            T.affine_quantize_kv_rotated(kx, vx, slabs, s, D, gs, bk, bv, rp, kp, vp)
    else:
        def call():
            T.affine_quantize_kv(kx, vx, slabs, s, D, gs, bk, bv, kp, vp)
    return call, list(kt + vt), (k, v, R)


def _levels(bits):
    """(boundaries, centroids) of a Lloyd-Max quantizer of N(0, 1): 2^bits + 1 and 2^bits values."""
    n = 1 << bits
    c = math.sqrt(2) * torch.erfinv(2 * (torch.arange(n, dtype=torch.float64) + 0.5) / n - 1)
    for _ in range(200):
        b = torch.cat((torch.tensor([-math.inf], dtype=torch.float64), (c[1:] + c[:-1]) / 2, torch.tensor([math.inf], dtype=torch.float64)))
        pdf, cdf = torch.exp(-b * b / 2) / math.sqrt(2 * math.pi), 0.5 * (1 + torch.erf(b / math.sqrt(2)))
        c = (pdf[:-1] - pdf[1:]) / (cdf[1:] - cdf[:-1])
    return b, c


def _codes(r, slabs, n, D, inner):
    out = torch.empty(slabs, n, D, dtype=torch.uint8, device="cuda")
    flat = out.view(-1, D)
    step = max(1, _CHUNK // D)
    for a in range(0, flat.shape[0], step):
        rows = flat[a:a + step]
        rows.copy_(torch.bucketize(r.normal(*rows.shape), inner, out_int32=True))
    return out


def _codebook_inputs(c, seed):
    r = _Rand(c, seed)
    B, H, Hkv, D, n, m = (c[x] for x in ("B", "H", "Hkv", "D", "n", "m"))
    b, cent = _levels(c["bits"])
    inner, cent = b[1:-1].float().cuda(), cent.float().cuda()
    s = dict(cent=cent, R=_rotation(r, D), q=r.query(B, H, 1, D) * 2)
    for x in "kv":
        s[x] = _codes(r, B * Hkv, n, D, inner)
        s[x + "s"] = r.uniform(0.5, 2.0, B * Hkv, n)
    if m:
        s["signs"], s["rn"] = r.words(B * Hkv, n, m // 32), r.uniform(0.5, 2.0, B * Hkv, n)
        s["phi"] = r.normal(m, D) / math.sqrt(m)
    return s


def _prepare_codebook(c, seed):
    B, H, Hkv, D, n, bits, m = (c[x] for x in ("B", "H", "Hkv", "D", "n", "bits", "m"))
    s = _codebook_inputs(c, seed)
    out = torch.zeros(B, H, 1, D, dtype=torch.bfloat16, device="cuda")
    ws = _bytes(T.decode_codebook_workspace_size(B, H, D, n))
    q, R, cent, kc, ks, vc, vs, op, wp, wb = *_ptrs([s[x] for x in ("q", "R", "cent", "k", "ks", "v", "vs")] + [out, ws]), ws.numel()
    scale = D ** -0.5
    if m:
        sg, rn, phi = _ptrs((s["signs"], s["rn"], s["phi"]))

        def call():
            T.check(T.lib().tqkv_decode_attend_codebook_qjl(q, B, H, Hkv, D, scale, R, cent, bits, cent, bits, kc, ks, sg, rn, phi, m,
                                                            vc, vs, n, n, op, wp, wb, None))
    else:
        def call():
            T.decode_attend_codebook(q, B, H, Hkv, D, scale, R, cent, bits, cent, bits, kc, ks, vc, vs, n, n, op, wp, wb)
    return call, [out], (s, ws)


def _encode_inputs(c, seed):
    r = _Rand(c, seed)
    b, cent = _levels(c["bits"])
    R = _rotation(r, c["D"])
    phi = r.normal(c["m"], c["D"]) / math.sqrt(c["m"]) if c["m"] else None
    return [r.rows(c["slabs"], c["s"], c["D"]) for _ in range(2)], R, b.cuda(), cent.float().cuda(), phi


def _prepare_encode(c, seed):
    slabs, s, D, bits, m = (c[x] for x in ("slabs", "s", "D", "bits", "m"))
    xs, R, bnd, cent, phi = _encode_inputs(c, seed)
    inner = bnd[1:-1].float()
    outs, calls = [], []
    for x in xs:
        o = [torch.zeros(slabs, s, D, dtype=torch.uint8, device="cuda"), torch.zeros(slabs, s, device="cuda")]
        if m:
            o += [torch.zeros(slabs, s, (m + 31) // 32, dtype=torch.int32, device="cuda"), torch.zeros(slabs, s, device="cuda")]
        outs.append(o)
        calls.append((x.data_ptr(),) + _ptrs(o) + ((None, None) if not m else ()))
    rp, bp, ip, cp, pp, tr = R.data_ptr(), bnd.data_ptr(), inner.data_ptr(), cent.data_ptr(), phi.data_ptr() if m else None, c["transpose"]
    if c["path"] == "gpu":
        def call():
            for x, codes, sigma, _, _ in calls:
                T.tq_encode_gpu_path(x, slabs, s, D, rp, 1, tr, ip, bits, codes, sigma)
    else:
        def call():
            for x, codes, sigma, signs, rn in calls:
                T.tq_encode(x, 1, slabs, s, D, rp, bp, cp, bits, pp, m, codes, sigma, signs, rn)
    return call, outs, (xs, R, bnd, inner, cent, phi)


_PREPARE = {"decode": _prepare_decode, "stack": _prepare_stack, "prefix": _prepare_prefix, "prefill": _prepare_prefill,
            "append": _prepare_append, "codebook": _prepare_codebook, "encode": _prepare_encode}


def prepare(case, seed):
    call, outs, held = _PREPARE[case["kind"]](case, seed)
    return {"call": call, "outs": outs, "held": held}


def run(state):
    state["call"]()
    return state["outs"]


# ------------------------------------------------------------------ 64-bit results
def _attend(q, k, v, scale, first_key=None, window=-1):
    """softmax(scale q k^T) v in 64 bits; q [G, L, D] of one KV head. first_key: position of q's row 0 (causal)."""
    G, L, D = q.shape
    n, out = k.shape[0], torch.empty(G, L, v.shape[1], dtype=torch.float64, device=q.device)
    step = max(1, (1 << 26) // (n * G))
    for a in range(0, L, step):
        b = min(L, a + step)
        s = (q[:, a:b].reshape(-1, D) @ k.T).reshape(G, b - a, n) * scale
        if first_key is not None:
            at = torch.arange(first_key + a, first_key + b, device=q.device)[:, None]
            key = torch.arange(n, device=q.device)[None]
            hide = key > at
            if window > 0:
                hide = hide | (key <= at - window)
            s.masked_fill_(hide, -math.inf)
        out[:, a:b] = (torch.softmax(s, -1).reshape(-1, n) @ v).reshape(G, b - a, -1)
    return out


def _by_heads(q, Hkv, kv, scale, **more):
    """q [B, H, L, D]; kv(slab) gives that KV head's (k, v) in 64 bits."""
    B, H, L, D = q.shape
    G, out = H // Hkv, torch.empty(q.shape, dtype=torch.float64, device=q.device)
    for b in range(B):
        for h in range(Hkv):
            k, v = kv(b * Hkv + h)
            out[b, h * G:(h + 1) * G] = _attend(q[b, h * G:(h + 1) * G].double(), k, v, scale, **more)
    return out


def _new_rows(nk, nv, bk, bv, gs):
    """The new token's triples: codes have no value in 64 bits, scales and biases are as stored."""
    k, v = _quantize(nk, bk, gs), _quantize(nv, bv, gs)
    return (k, v), [None, k[1][:, 0].double(), k[2][:, 0].double(), None, v[1][:, 0].double(), v[2][:, 0].double()]


def exact(case, seed):
    c, kind = case, case["kind"]
    if kind == "decode":
        kt, vt, q, nk, nv, _ = _decode_inputs(c, seed)
        new, said = _new_rows(nk, nv, c["bk"], c["bv"], c["gs"])

        def kv(i):
            return [torch.cat((_dequantize([x[i, :c["n"]] for x in t], b, c["gs"]), _dequantize([x[i] for x in w], b, c["gs"])))
                    for t, w, b in ((kt, new[0], c["bk"]), (vt, new[1], c["bv"]))]
        return [_by_heads(q, c["Hkv"], kv, c["D"] ** -0.5)] + said
    if kind == "stack":
        outs = []
        for g, n, k, v, nk, nv, q in _stack_inputs(c, seed):
            if not g and n == c["window"]:
                k, v = k[:, 1:], v[:, 1:]  # the ring's oldest token makes room
            both = [_quantize(torch.cat(x, 1), c["bits"], 64) for x in ((k, nk), (v, nv))]
            outs.append(_by_heads(q, c["Hkv"], lambda i: [_dequantize([x[i] for x in t], c["bits"], 64) for t in both], 1.0 / math.sqrt(c["D"])))
        return outs
    if kind == "prefix":
        pk, pv, sk, sv, q, nk, nv, _ = _prefix_inputs(c, seed)
        new, said = _new_rows(nk, nv, c["bk"], c["bv"], 64)

        def kv(i):
            return [torch.cat([_dequantize([x[i % c["Hkv"]] for x in p], b, 64), _dequantize([x[i, :c["own"]] for x in t], b, 64),
                               _dequantize([x[i] for x in w], b, 64)]) for p, t, w, b in ((pk, sk, new[0], c["bk"]), (pv, sv, new[1], c["bv"]))]
        return [_by_heads(q, c["Hkv"], kv, c["D"] ** -0.5)] + said
    if kind == "prefill":
        kt, vt, q = _prefill_inputs(c, seed)

        def kv(i):  # a prefill reads the cache as bf16 rows
            return [_dequantize([x[i] for x in t], b, c["gs"], torch.float32).to(torch.bfloat16).double() for t, b in ((kt, c["bk"]), (vt, c["bv"]))]
        return [_by_heads(q, c["Hkv"], kv, c["D"] ** -0.5, first_key=c["n"] - c["L"], window=c["window"])]
    if kind == "append":
        k, v, R = _append_inputs(c, seed)
        if R is not None:
            k = (k.double() @ R.double()).to(torch.bfloat16)
        (_, a, b), (_, d, e) = _quantize(k, c["bk"], c["gs"]), _quantize(v, c["bv"], c["gs"])
        return [None, a.double(), b.double(), None, d.double(), e.double()]
    if kind == "codebook":
        s = _codebook_inputs(c, seed)
        B, H, Hkv, D, m = (c[x] for x in ("B", "H", "Hkv", "D", "m"))
        R, cent, G = s["R"].double(), s["cent"].double(), H // Hkv
        out = torch.empty(B, H, 1, D, dtype=torch.float64, device="cuda")
        for i in range(B * Hkv):
            q = s["q"][i // Hkv, i % Hkv * G:(i % Hkv + 1) * G, 0].double()
            k, v = (cent[s[x][i].long()] * s[x + "s"][i].double()[:, None] for x in "kv")
            sc = (q @ R.T) @ k.T
            if m:
                w = s["signs"][i].long() & 0xffffffff
                sign = ((w[:, :, None] >> torch.arange(32, device="cuda")) & 1).reshape(-1, m).double() * 2 - 1
                sc += (q @ s["phi"].double().T) @ sign.T * (s["rn"][i].double() * math.sqrt(math.pi / 2) / math.sqrt(m))
            out[i // Hkv, i % Hkv * G:(i % Hkv + 1) * G, 0] = torch.softmax(sc * D ** -0.5, -1) @ v @ R
        return [out]
    xs, R, bnd, cent, phi = _encode_inputs(c, seed)
    R, outs = R.double(), []
    for x in xs:
        if c["path"] == "gpu":
            y = (x.double() @ (R.T if c["transpose"] else R)).to(torch.bfloat16).double()
            outs.append([None, y.square().mean(-1).sqrt()])
            continue
        y = x.double() @ R.T
        sigma = y.square().mean(-1).sqrt()
        o = [None, sigma]
        if c["m"]:
            code = torch.bucketize(y / sigma[..., None], bnd[1:-1], right=True)
            back = (cent.double()[code] * sigma[..., None]) @ R
            o += [None, (x.double() - back).square().sum(-1).sqrt()]
        outs.append(o)
    return outs

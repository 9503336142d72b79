"""Calls under a stream capture whose library scratch cannot grow: they take
the path that needs none (prefill: no key splits, no dequantized rows; head dim
512 decode: the splits that fit), the capture lives, and every replay gives
that path's bits, eager calls and synchronizations between."""
import contextlib
import ctypes

import numpy as np
import pytest

from inputs import kv_bf16
from test_gpu_affine import _cache

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def T():
    import tqkv
    assert tqkv.hip().device_count() > 0, "no GPU visible"
    return tqkv


@contextlib.contextmanager
def captured(T, call):
    """A launcher of the graph of call(stream), captured on a stream of its own."""
    hip = T.hip()
    h, P = hip.h, ctypes.c_void_p
    stream, graph, run = P(hip.stream()), P(), P()
    hip._ok(h.hipStreamBeginCapture(stream, ctypes.c_int(1)), "hipStreamBeginCapture")  # this thread's
    call(stream.value)
    hip._ok(h.hipStreamEndCapture(stream, ctypes.byref(graph)), "hipStreamEndCapture")
    hip._ok(h.hipGraphInstantiate(ctypes.byref(run), graph, None, None, ctypes.c_size_t(0)),
            "hipGraphInstantiate")

    def launch():
        hip._ok(h.hipGraphLaunch(run, stream), "hipGraphLaunch")
        hip.sync()
    try:
        yield launch
    finally:
        hip.sync()
        h.hipGraphExecDestroy(run)
        h.hipGraphDestroy(graph)
        h.hipStreamDestroy(stream)


def replays(T, call, eager, out, want):
    """call(stream) captured and replayed three times, eager() between."""
    hip = T.hip()
    with captured(T, call) as launch:
        for i in range(3):
            hip.copy_in(out.ptr, np.full(out.shape, 0x7FC0, np.uint16))
            launch()
            assert np.array_equal(out.numpy(), want), f"replay {i}"
            eager()
            hip.sync()


@pytest.mark.parametrize("D,H,Hkv,L,N", [(128, 16, 8, 20, 3000), (512, 16, 2, 40, 700),
                                         (256, 8, 2, 130, 2300)])
def test_captured_prefill_without_scratch(T, D, H, Hkv, L, N):
    print(f"[capture] prefill D={D} L={L} N={N}", flush=True)
    B = 1
    q = kv_bf16((B, H, L, D), N)
    (_, kd), (_, vd) = (_cache(kv_bf16((B, Hkv, N, D), i), 64, 4) for i in (1, 2))
    dq = T.DeviceArray.of(q)
    seg = T.affine_seg(tuple(a.ptr for a in kd), tuple(a.ptr for a in vd), N, N)
    args = (B, H, Hkv, L, D, 64, 4, 4, D ** -0.5, [seg])
    out, other, plain = (T.DeviceArray((B, H, L, D), np.uint16) for _ in range(3))
    # Every block dequantizes for itself, the keys whole.
    T.prefill_attend_affine_ws(dq.ptr, *args, plain.ptr, None, 0, N - L, 0, True, -1)
    T.hip().sync()
    T.scratch_release()

    def call(stream):
        T.prefill_attend_affine(dq.ptr, *args, out.ptr, N - L, 0, True, -1, stream)

    with captured(T, call) as launch:
        assert T.scratch_bytes() == 0
        for i in range(3):
            T.hip().copy_in(out.ptr, np.full(out.shape, 0x7FC0, np.uint16))
            launch()
            assert np.array_equal(out.numpy(), plain.numpy()), f"replay {i}"
            T.prefill_attend_affine(dq.ptr, *args, other.ptr, N - L, 0, True, -1)  # grows it
            T.hip().sync()
    assert T.scratch_bytes() > 0


def test_captured_wide_head_decode_takes_the_splits_that_fit(T):
    B, H, Hkv, D = 1, 32, 2, 512
    small, N = 2000, 4096
    q = kv_bf16((B, H, 1, D), 3)
    (_, kd), (_, vd) = (_cache(kv_bf16((B, Hkv, N, D), i), 64, 4) for i in (1, 2))
    dq = T.DeviceArray.of(q)

    def seg(n):
        return T.affine_seg(tuple(a.ptr for a in kd), tuple(a.ptr for a in vd), N, n)

    def decode(n, o, stream=None, ws=None, wsb=0):
        T.decode_attend_affine(dq.ptr, B, H, Hkv, D, 64, 4, 4, D ** -0.5, [seg(n)], o.ptr, ws, wsb,
                               stream)

    out, other, plain = (T.DeviceArray((B, H, 1, D), np.uint16) for _ in range(3))
    coarse = 16 * B * H * (D + 2) * 4  # 16 splits of 256 keys; 32 of 128 do not fit
    ws = T.DeviceArray((coarse,), np.uint8)
    decode(N, plain, None, ws.ptr, coarse)
    T.hip().sync()
    T.scratch_release()
    decode(small, other)  # 16 splits of 128 keys: the scratch holds as much
    T.hip().sync()
    held = T.scratch_bytes()
    assert coarse <= held < 2 * coarse
    with captured(T, lambda stream: decode(N, out, stream)) as launch:
        assert T.scratch_bytes() == held
        for i in range(3):
            T.hip().copy_in(out.ptr, np.full(out.shape, 0x7FC0, np.uint16))
            launch()
            assert np.array_equal(out.numpy(), plain.numpy()), f"replay {i}"
            decode(small, other)
            T.hip().sync()


def test_captured_codebook_decode(T):
    # Four launches over the caller's workspace.
    B, Hkv, G, D, N, bits = 2, 2, 4, 256, 1000, 4
    H, rng = Hkv * G, np.random.default_rng(1)
    R, cent = T.rotation_matrix(D, 42), T.lloyd_max(bits, 100)[1].astype(np.float32)
    x = [T.DeviceArray.of(a) for a in
         [kv_bf16((B, H, 1, D), 5), R, cent] +
         [rng.integers(0, 1 << bits, (B, Hkv, N, D), dtype=np.uint8) for _ in "kv"] +
         [rng.uniform(0.5, 2, (B, Hkv, N)).astype(np.float32) for _ in "kv"]]
    wsb = T.decode_codebook_workspace_size(B, H, D, N)
    out, plain = (T.DeviceArray((B, H, 1, D), np.uint16) for _ in range(2))
    ws = [T.DeviceArray((wsb,), np.uint8) for _ in range(2)]

    def decode(o, w, stream=None):
        T.decode_attend_codebook(x[0].ptr, B, H, Hkv, D, D ** -0.5, x[1].ptr, x[2].ptr, bits,
                                 x[2].ptr, bits, x[3].ptr, x[5].ptr, x[4].ptr, x[6].ptr, N, N,
                                 o.ptr, w.ptr, wsb, stream)

    decode(plain, ws[1])
    T.hip().sync()
    want = plain.numpy()
    replays(T, lambda stream: decode(out, ws[0], stream), lambda: decode(plain, ws[1]), out, want)


def test_captured_bf16_cache_prefill(T):
    B, H, Hkv, D, N, L = 1, 16, 4, 128, 2500, 20
    c = T.Cache(T.CACHE_BF16, B, Hkv, D, D)
    k, v, q = (T.DeviceArray.of(kv_bf16(s, i)) for i, s in
               enumerate(((B, Hkv, N, D),) * 2 + ((B, H, L, D),)))
    c.append(k.ptr, v.ptr, N)
    out, plain = (T.DeviceArray((B, H, L, D), np.uint16) for _ in range(2))
    c.prefill_attend(q.ptr, H, L, D ** -0.5, plain.ptr)
    T.hip().sync()
    T.scratch_release()
    replays(T, lambda stream: c.prefill_attend(q.ptr, H, L, D ** -0.5, out.ptr, stream=stream),
            lambda: c.prefill_attend(q.ptr, H, L, D ** -0.5, plain.ptr), out, plain.numpy())
    assert T.scratch_bytes() == 0

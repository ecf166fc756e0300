"""The split-K decode over f16 caches of 128-channel heads and over f32 caches of 64 and 128 channels
(moearc_attn_decode_{f16d128,f32d64,f32d128}_*), against the float64 oracle at the sizes where tiles,
chunks and splits end, over page sizes below and above a tile, groups of 1 to 16 heads, f32 and f16
outputs, the single, batched and allocation-free entry points, under capture, and with buffers that
only the general kernel takes.

Tolerance: a score is a sum of D products in f32, off by at most (D + 8) 2^-24 sum|q_d k_d| scale; a
weight by that share of itself, twice counting the denominator; an output by that share of max|V|.
f16 outputs add half an ulp."""
from __future__ import annotations

import ctypes

import numpy as np
import pytest

import fixtures as fx
from moearc_amd import Context, DeviceView, KvType, OUT_F16, OUT_F32
from oracle import oracle

pytestmark = pytest.mark.gpu

KINDS = [("f16", 128), ("f32", 64), ("f32", 128)]


class Batch:
    """Sequences of the given lengths over one scattered page pool."""

    def __init__(self, seed, kv, D, lens, pt, G, group, windows=None):
        self.kv, self.D, self.lens, self.pt, self.G, self.H = kv, D, lens, pt, G, G * group
        n, row = sum(lens), G * D
        counts = [-(-x // pt) for x in lens]
        bt = fx.synth.random_block_table(seed, sum(counts))
        self.stride = max(counts)
        self.table = np.zeros((len(lens), self.stride), np.uint32)
        k = np.zeros((sum(counts) * pt, row), np.float32)
        v = np.zeros_like(k)
        kv_rows, vv_rows = (fx.synth.normal(seed + i, n * row).reshape(n, row) for i in (1, 2))
        at = key = 0
        for b, (x, c) in enumerate(zip(lens, counts)):
            self.table[b, :c] = bt[at:at + c]
            j = np.arange(x)
            phys = self.table[b, j // pt].astype(np.int64) * pt + j % pt
            k[phys], v[phys] = kv_rows[key:key + x], vv_rows[key:key + x]
            at, key = at + c, key + x
        if kv == "f16":
            k, v = fx.synth.f16_bits(k.ravel()), fx.synth.f16_bits(v.ravel())
        self.k, self.v = np.ascontiguousarray(k), np.ascontiguousarray(v)
        self.q = fx.synth.normal(seed + 3, len(lens) * self.H * D)
        self.sinks = fx.synth.normal(seed + 4, self.H)
        self.begin = [max(0, x - w) if w else 0 for x, w in zip(lens, windows or [0] * len(lens))]
        self.scale = float(np.float32(1.0 / np.sqrt(D)))
        self.type = KvType.F16 if kv == "f16" else KvType.F32

    def upload(self, cx):
        return [cx.upload(x) for x in (self.q, self.k, self.v, self.table, self.sinks)]

    def want(self, b, sinks=True):
        w = self.H * self.D
        return oracle.attn_decode(self.q[b * w:(b + 1) * w], self.k, self.v, self.table[b], self.H, self.G, self.D,
                                  self.begin[b], self.lens[b], self.pt, self.scale, kv_type=int(self.type),
                                  sinks=self.sinks if sinks else None)

    def tol(self):
        kf = self.k.view(np.float16).astype(np.float32) if self.kv == "f16" else self.k
        vf = self.v.view(np.float16).astype(np.float32) if self.kv == "f16" else self.v
        kf = np.abs(kf.reshape(-1, self.G, self.D))
        qf = np.abs(self.q.reshape(len(self.lens), self.G, -1, self.D)).max(axis=(0, 2))
        dots = float((kf * qf[None]).sum(-1).max())
        return 2.0 * (self.D + 8) * 2.0 ** -24 * dots * self.scale * float(np.abs(vf).max())

    def check(self, got, b, sinks=True, half=False):
        want = self.want(b, sinks)
        err = np.abs(got.astype(np.float64) - want)
        tol = self.tol() + (2.0 ** -11 * np.abs(want) + 2.0 ** -25 if half else 0.0)
        print(f"{self.kv} d{self.D} lens={self.lens} pt={self.pt} H={self.H} G={self.G}: max err {err.max():.2e} "
              f"(bound {np.max(tol):.2e})", flush=True)
        assert np.all(err <= tol)


def _batched(cx, B, bufs, out_type, fn=None, out=None):
    q, k, v, bt, s = bufs
    n, half = len(B.lens), out_type == OUT_F16
    out = out if out is not None else cx.alloc(n * B.H * B.D * (2 if half else 4))
    if fn is None:
        cx.attn_decode_batched(out, q, k, v, bt, B.stride, B.begin, B.lens, s, B.H, B.G, B.D, B.pt, B.scale, B.type,
                               out_type=out_type)
    else:
        kb, nk = np.array(B.begin, np.uint32), np.array(B.lens, np.uint32)
        assert fn(cx.raw, out.ptr, out_type, q.ptr, k.ptr, v.ptr, bt.ptr, B.stride, kb.ctypes.data, nk.ctypes.data,
                  s.ptr, n, B.H, B.G, B.D, B.pt, B.scale, int(B.type)) == 0
    cx.sync()
    return cx.download(out, np.float16 if half else np.float32, (n, B.H * B.D))


@pytest.mark.parametrize("kv,D", KINDS)
@pytest.mark.parametrize("n,pt,G,group,window", [
    (1, 16, 4, 8, 0), (31, 1, 1, 16, 0), (33, 4, 4, 8, 32), (127, 16, 5, 3, 0), (128, 256, 16, 1, 0),
    (129, 16, 2, 7, 100), (511, 64, 4, 8, 0), (2085, 256, 4, 8, 128), (6000, 256, 4, 8, 0), (20003, 256, 3, 8, 0)])
def test_single_sequence(kv, D, n, pt, G, group, window):
    B = Batch(100 + n, kv, D, [n], pt, G, group, [window])
    with Context() as cx:
        q, k, v, bt, s = B.upload(cx)
        out = cx.alloc(B.H * D * 4)
        for sinks in (True, False):
            cx.attn_decode_ext(out, q, k, v, bt, s if sinks else None, B.H, G, D, B.begin[0], n, pt, B.scale, B.type)
            B.check(cx.download(out, np.float32, B.H * D), 0, sinks)


@pytest.mark.parametrize("variant", [None, "4x2x4", "1x4x1"])
@pytest.mark.parametrize("kv,D", KINDS)
def test_ragged_batch_and_entry_points(kv, D, variant, monkeypatch):
    if variant:  # the kind's long- or short-span shape, in splits that need the merge
        monkeypatch.setenv("MOEARC_DECODE_VARIANT", variant)
        monkeypatch.setenv("MOEARC_DECODE_SPLIT", "512")
    B = Batch(7, kv, D, [1, 700, 3000, 64, 5001], 16, 4, 8, [0, 0, 128, 0, 0])
    with Context() as cx:
        bufs = B.upload(cx)
        full = _batched(cx, B, bufs, OUT_F32)
        for b in range(len(B.lens)):
            B.check(full[b], b)
        half = _batched(cx, B, bufs, OUT_F16)
        assert np.array_equal(half, full.astype(np.float16))
        fixed = _batched(cx, B, bufs, OUT_F32, cx._lib.moearc_attn_decode_batched_noalloc)
        assert np.array_equal(fixed, full)


def test_records_past_the_fixed_array_widen_the_splits(monkeypatch):
    # 128-key splits of 20000 keys would keep 64 x 157 records of 130 floats, more than half the array;
    # of four such sequences more than it holds: the call is taken all the same
    monkeypatch.setenv("MOEARC_DECODE_VARIANT", "1x4x1")
    monkeypatch.setenv("MOEARC_DECODE_SPLIT", "128")
    B = Batch(9, "f16", 128, [20000, 19000, 18000, 20000], 256, 8, 8)
    with Context() as cx:
        got = _batched(cx, B, B.upload(cx), OUT_F32, cx._lib.moearc_attn_decode_batched_noalloc)
        for b in (0, 3):
            B.check(got[b], b)


@pytest.mark.parametrize("kv,D", KINDS)
def test_capture_needs_no_memory(kv, D):
    # the first call on a context is a captured one; the graph then replays beside the context's own
    # eager calls, whose larger batch makes the workspace grow; it is one launch without records, so
    # graphs on several streams share nothing
    hip = ctypes.CDLL("libamdhip64.so")
    B, big = Batch(11, kv, D, [3000], 256, 4, 8), Batch(12, kv, D, [9000, 9000, 9000], 256, 4, 8)
    with Context() as cx:
        q, k, v, bt, s = B.upload(cx)
        out, stream = cx.alloc(B.H * D * 4), ctypes.c_void_p(cx.stream)
        graph, exe = ctypes.c_void_p(), ctypes.c_void_p()
        assert hip.hipStreamBeginCapture(stream, 1) == 0
        cx.attn_decode_ext(out, q, k, v, bt, s, B.H, B.G, D, 0, 3000, 256, B.scale, B.type)
        assert hip.hipStreamEndCapture(stream, ctypes.byref(graph)) == 0
        nodes = ctypes.c_size_t()
        assert hip.hipGraphGetNodes(graph, None, ctypes.byref(nodes)) == 0 and nodes.value == 1
        assert hip.hipGraphInstantiate(ctypes.byref(exe), graph, None, None, ctypes.c_size_t(0)) == 0
        bigger = big.upload(cx)
        for _ in range(3):
            cx.zero(out, B.H * D)
            assert hip.hipGraphLaunch(exe, stream) == 0
            B.check(cx.download(out, np.float32, B.H * D), 0)
            big.check(_batched(cx, big, bigger, OUT_F32)[2], 2)
        hip.hipGraphExecDestroy(exe)
        hip.hipGraphDestroy(graph)


@pytest.mark.parametrize("kv,D", KINDS)
def test_unaligned_buffers(kv, D):
    # element-aligned only: the general kernel's calls
    B = Batch(13, kv, D, [300], 16, 2, 4)
    e = 2 if kv == "f16" else 4
    with Context() as cx:
        _, _, _, bt, s = B.upload(cx)

        def shifted(x, by):
            raw = np.frombuffer(b"\0" * by + np.ascontiguousarray(x).tobytes(), np.uint8)
            return DeviceView(cx.upload(raw), by)
        out = cx.alloc(B.H * D * 4 + 16)
        args = [(shifted(B.q, 4), cx.upload(B.k), cx.upload(B.v), out),
                (cx.upload(B.q), shifted(B.k, e), cx.upload(B.v), out),
                (cx.upload(B.q), cx.upload(B.k), shifted(B.v, e), out),
                (cx.upload(B.q), cx.upload(B.k), cx.upload(B.v), DeviceView(out, 4))]
        for q, k, v, o in args:
            cx.attn_decode_ext(o, q, k, v, bt, s, B.H, B.G, D, 0, 300, 16, B.scale, B.type)
            B.check(cx.download(o, np.float32, B.H * D), 0)


@pytest.mark.parametrize("octaves", [10, 18, 26])
@pytest.mark.parametrize("kv,D,group", [(*k, 8) for k in KINDS] + [("f16", 128, 1), ("f16", 128, 12)])
def test_one_channel_far_above_the_others(kv, D, group, octaves):
    # one channel of q some 2^octaves above the rest, its keys as far below: every channel has its share of
    # the scores, so the small ones must keep their f32 precision beside the large one
    B = Batch(19, kv, D, [300], 16, 4, group)
    dt = np.float16 if kv == "f16" else np.float32
    k = B.k.view(dt).reshape(-1, D).astype(np.float32) * np.float32(2.0 ** 12)
    k[:, 0] *= np.float32(2.0 ** -octaves)
    B.k = np.ascontiguousarray(fx.synth.f16_bits(k.ravel()) if kv == "f16" else k)
    B.q = (B.q.reshape(-1, D) * np.where(np.arange(D) == 0, 1.0, 2.0 ** -octaves)).astype(np.float32).ravel()
    B.scale = float(np.float32(2.0 ** (octaves - 12) / np.sqrt(D)))
    with Context() as cx:
        q, dk, dv, bt, s = B.upload(cx)
        out = cx.alloc(B.H * D * 4)
        cx.attn_decode_ext(out, q, dk, dv, bt, s, B.H, B.G, D, 0, 300, 16, B.scale, B.type)
        B.check(cx.download(out, np.float32, B.H * D), 0)


@pytest.mark.parametrize("kv,D", KINDS)
def test_infinities(kv, D):
    # a key of -inf in a whole first tile weighs nothing; an infinite value shows in its channel alone;
    # the span's last, partial tile does not multiply the repeated last row by its zero weights
    B = Batch(15, kv, D, [45], 16, 1, 8)
    dt = np.float16 if kv == "f16" else np.float32
    k, v = B.k.view(dt).reshape(-1, D).copy(), B.v.view(dt).reshape(-1, D).copy()
    phys = B.table[0, np.arange(45) // 16].astype(np.int64) * 16 + np.arange(45) % 16
    B.q[:] = np.abs(B.q) + np.float32(0.5)
    k[phys[:32], 0] = -np.inf
    v[phys[44], 3] = np.inf
    B.k, B.v = k.view(np.uint16 if kv == "f16" else np.float32), v.view(np.uint16 if kv == "f16" else np.float32)
    with Context() as cx:
        q, dk, dv, bt, s = B.upload(cx)
        out = cx.alloc(B.H * D * 4)
        cx.attn_decode_ext(out, q, dk, dv, bt, s, B.H, 1, D, 0, 45, 16, B.scale, B.type)
        got = cx.download(out, np.float32, (B.H, D))
    q64, j = B.q.reshape(B.H, D).astype(np.float64), np.arange(32, 45)
    sc = q64 @ k[phys[j]].astype(np.float64).T * B.scale
    w = np.exp(sc)
    want = w @ v[phys[j]].astype(np.float64) / (w.sum(-1) + np.exp(B.sinks))[:, None]
    assert np.all(np.isposinf(got[:, 3]))
    ch = [c for c in range(D) if c != 3]
    assert np.max(np.abs(got[:, ch] - want[:, ch])) < 1e-4

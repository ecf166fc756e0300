"""Prefill split along the keys (moearc_attn_prefill_split_g* and the merge of its pieces): short
chunks deep in a context, against the oracle at the suite's 2e-3 bar, over every group, windows longer
than a piece, pages below and above a tile, pieces that some rows see nothing of, both outputs, under
capture, and through the attention block. Each case checks that its launch was split (or not)."""
from __future__ import annotations

import ctypes

import numpy as np
import pytest

import fixtures as fx
from moearc_amd import AttnBlockDesc, Context, KvType, OUT_F16, OUT_F32
from oracle import oracle

pytestmark = pytest.mark.gpu

TOL = 2e-3


def _prefill(cx, pc, n_swa, out_type=OUT_F32):
    dk, dv, dbt = cx.upload(pc.k_raw), cx.upload(pc.v_raw), cx.upload(pc.bt)
    dq, ds = cx.upload(np.ascontiguousarray(pc.qp).view(np.uint16)), cx.upload(pc.sinks)
    half = out_type == OUT_F16
    out = cx.alloc(pc.n_q * pc.H * pc.D * (2 if half else 4))
    cx.attn_prefill(out, dq, dk, dv, dbt, ds, pc.n_q, pc.pos0, n_swa, pc.H, pc.G, pc.D, pc.pt, float(pc.scale),
                    KvType.F16, out_type=out_type)
    return cx.download(out, np.float16 if half else np.float32, (pc.n_q, pc.H, pc.D))


def _want(pc, n_swa):
    return oracle.attn_prefill(pc.qp.astype(np.float32), pc.k_raw, pc.v_raw, pc.bt, pc.n_q, pc.pos0, n_swa, pc.H,
                               pc.G, pc.D, pc.pt, float(pc.scale), sinks=pc.sinks, n_threads=8)


@pytest.mark.parametrize("group,G,n_q,pos0,pt,n_swa,split", [
    (8, 8, 33, 3000, 256, 0, True),     # two tiles, the second of one token
    (8, 2, 16, 6001, 16, 0, True),      # half a tile, pages below a tile, many pieces
    (8, 2, 300, 0, 64, 0, False),       # too short to gain
    (8, 4, 513, 1500, 256, 0, True),    # tiles of different lengths
    (8, 2, 64, 9000, 256, 4000, True),  # a window of many pieces
    (8, 8, 64, 9000, 256, 128, False),  # a window of five chunks
    (4, 4, 70, 5000, 32, 0, True),
    (2, 3, 129, 4095, 256, 0, True),
    (1, 16, 257, 3333, 256, 0, True),
    (1, 5, 1, 5000, 256, 0, True),      # one token
])
def test_split_prefill_against_oracle(group, G, n_q, pos0, pt, n_swa, split, monkeypatch):
    monkeypatch.setenv("MOEARC_PROFILE_KERNELS", "1")
    pc = fx.prefill_case(0x5B1 + n_q + pos0, n_q=n_q, pos0=pos0, pt=pt, H=G * group, G=G)
    want = _want(pc, n_swa)
    with Context() as cx:
        f32 = _prefill(cx, pc, n_swa)
        keys = cx.profile_events_report()
        assert any("merge" in k for k in keys) == split, keys
        f16 = _prefill(cx, pc, n_swa, OUT_F16)
    for label, got in (("f32", f32), ("f16", f16)):
        err = float(np.max(np.abs(got.astype(np.float64) - want)))
        print(f"split prefill {label} group={group} n_q={n_q} pos0={pos0}: {err:.2e}", flush=True)
        assert err <= TOL
    assert np.array_equal(f16, f32.astype(np.float16))


def test_score_jumps_across_pieces():
    # keys that outscore all before them, in several pieces, and a piece of the largest by far
    pc = fx.prefill_case(0x5B9, n_q=40, pos0=5000, pt=256, H=32, G=4,
                         boost=[(1000, 1010, 6.0), (2500, 2600, 8.0), (4990, 5010, 5.0)])
    with Context() as cx:
        got = _prefill(cx, pc, 0)
    assert np.max(np.abs(got.astype(np.float64) - _want(pc, 0))) <= TOL


def test_profile_counts_a_split_prefill_once(monkeypatch):
    monkeypatch.setenv("MOEARC_PROFILE_EVENTS", "1")
    pc = fx.prefill_case(0x5BA, n_q=33, pos0=3000, pt=256, H=16, G=2)
    with Context() as cx:
        _prefill(cx, pc, 0)
        keys = cx.profile_events_report()
    assert list(keys) == ["attn_prefill r16 m64"] and keys["attn_prefill r16 m64"][1] == 1


def test_capture_needs_no_memory():
    # a captured call on a fresh context, replayed beside eager calls that grow the workspace; it is
    # one launch without records, so graphs on several streams share nothing
    hip = ctypes.CDLL("libamdhip64.so")
    pc, big = (fx.prefill_case(s, n_q=n, pos0=4000, pt=256, H=16, G=2) for s, n in ((0x5BB, 40), (0x5BC, 200)))
    with Context() as cx:
        bufs = [cx.upload(np.ascontiguousarray(x)) for x in (pc.qp.view(np.uint16), pc.k_raw, pc.v_raw, pc.bt, pc.sinks)]
        out, stream = cx.alloc(pc.n_q * pc.H * 64 * 4), ctypes.c_void_p(cx.stream)
        graph, exe = ctypes.c_void_p(), ctypes.c_void_p()
        assert hip.hipStreamBeginCapture(stream, 1) == 0
        cx.attn_prefill(out, *bufs, pc.n_q, pc.pos0, 0, 16, 2, 64, 256, 0.125, KvType.F16)
        assert hip.hipStreamEndCapture(stream, ctypes.byref(graph)) == 0
        nodes = ctypes.c_size_t()
        assert hip.hipGraphGetNodes(graph, None, ctypes.byref(nodes)) == 0 and nodes.value == 1
        assert hip.hipGraphInstantiate(ctypes.byref(exe), graph, None, None, ctypes.c_size_t(0)) == 0
        want, want_big = _want(pc, 0), _want(big, 0)
        for _ in range(3):
            cx.zero(out, pc.n_q * pc.H * 64)
            assert hip.hipGraphLaunch(exe, stream) == 0
            got = cx.download(out, np.float32, (pc.n_q, 16, 64))
            assert np.max(np.abs(got - want)) <= TOL
            assert np.max(np.abs(_prefill(cx, big, 0) - want_big)) <= TOL
        hip.hipGraphExecDestroy(exe)
        hip.hipGraphDestroy(graph)


def test_workspace_grows_beside_another_contexts_capture():
    # the eager call's allocation neither fails nor breaks the capture (mode 0: global)
    hip = ctypes.CDLL("libamdhip64.so")
    pc = fx.prefill_case(0x5BE, n_q=40, pos0=4000, pt=256, H=16, G=2)
    with Context() as other, Context() as cx:
        x, stream, graph = other.upload(np.ones(64, np.float32)), ctypes.c_void_p(other.stream), ctypes.c_void_p()
        bufs = [cx.upload(np.ascontiguousarray(a)) for a in (pc.qp.view(np.uint16), pc.k_raw, pc.v_raw, pc.bt, pc.sinks)]
        out = cx.alloc(pc.n_q * pc.H * 64 * 4)
        assert hip.hipStreamBeginCapture(stream, 0) == 0
        other.zero(x, 64)
        cx.attn_prefill(out, *bufs, pc.n_q, pc.pos0, 0, 16, 2, 64, 256, 0.125, KvType.F16)
        assert hip.hipStreamEndCapture(stream, ctypes.byref(graph)) == 0
        hip.hipGraphDestroy(graph)
        got = cx.download(out, np.float32, (pc.n_q, 16, 64))
        assert np.max(np.abs(got - _want(pc, 0))) <= TOL


def test_block_deep_in_a_context(monkeypatch):
    # the merge writes the output projection's activation split: as the separate launches do
    E, H, G, D, pt, n, pos0 = 512, 16, 2, 64, 256, 100, 4000
    rng = np.random.default_rng(0x5BD)
    total = pos0 + n
    pages = -(-total // pt)
    shapes = [(H * D, E), (G * D, E), (G * D, E), (E, H * D)]
    ws = [(rng.standard_normal(s) * 0.05).astype(np.float16) for s in shapes]
    kv = [rng.standard_normal(pages * pt * G * D).astype(np.float16) for _ in range(2)]
    x, h0 = (rng.standard_normal((n, E)).astype(np.float32) for _ in range(2))
    pos = np.arange(pos0, total, dtype=np.int32)
    res = []
    for fused in ("1", "0"):
        monkeypatch.setenv("MOEARC_BLOCK_FUSED", fused)
        with Context() as cx:
            k, v = (cx.upload(a) for a in kv)
            desc = AttnBlockDesc.make([1] * 4, [cx.upload(w) for w in ws], [None] * 4, cx.upload(np.zeros(H, np.float32)),
                                      k, v, cx.upload(np.arange(pages, dtype=np.uint32)), E, H, G, D, pt, 0, 0.125, D,
                                      10000.0)
            h = cx.upload(h0)
            cx.attn_block_chunk(desc, h, cx.upload(x), n, pos0, cx.upload(pos),
                                cx.upload((pos // pt).astype(np.uint32)), cx.upload((pos % pt).astype(np.uint32)))
            res.append(cx.download(h, np.float32, (n, E)))
    assert np.array_equal(res[0], res[1]) and np.any(res[0] != h0)

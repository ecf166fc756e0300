"""How a work-group of the split decode finds its sequence in a batch: batches in which every sequence has
as many splits (windows, equal lengths) and ragged ones, past the 64 sequences of one launch, for both
head sizes. Each sequence must come out as it does alone, to the rounding of a sum over other splits:
2^-20 of the largest output."""
from __future__ import annotations

import numpy as np
import pytest

from moearc_amd import KvType

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_seqs,lens", [(5, "window"), (64, "window"), (66, "window"), (16, "ragged"), (17, "ragged"),
                                         (24, "ragged"), (25, "ragged"),
                                         (64, "ragged"), (70, "ragged"), (24, "equal"), (3, "equal")])
@pytest.mark.parametrize("heads,kv_heads,dim", [(16, 2, 64), (8, 1, 128)])
def test_each_sequence_as_alone(ctx, heads, kv_heads, dim, n_seqs, lens):
    pt, stride = 16, 48
    rng = np.random.default_rng(0xDB + n_seqs)
    n_kv = np.full(n_seqs, 700) if lens == "equal" else rng.integers(1, pt * stride + 1, n_seqs)
    begin = np.maximum(0, n_kv - 128) if lens == "window" else np.zeros(n_seqs, int)
    pool = 96
    row = kv_heads * dim
    k, v = (rng.standard_normal((pool, pt, row)).astype(np.float16) for _ in range(2))
    q = rng.standard_normal((n_seqs, heads, dim)).astype(np.float32)
    bt = rng.integers(0, pool, (n_seqs, stride)).astype(np.uint32)
    sinks = rng.standard_normal(heads).astype(np.float32)
    dk, dv, dq, dbt, ds = (ctx.upload(t.view(np.uint8).reshape(-1)) for t in (k, v, q, bt, sinks))
    out, one = ctx.alloc(q.nbytes), ctx.alloc(heads * dim * 4)
    ctx.attn_decode_batched(out, dq, dk, dv, dbt, stride, [int(b) for b in begin], [int(n) for n in n_kv], ds, heads,
                            kv_heads, dim, pt, dim ** -0.5, KvType.F16)
    got = ctx.download(out, np.float32, q.shape)
    for s in range(n_seqs):
        ctx.attn_decode_ext(one, ctx.upload(q[s]), dk, dv, ctx.upload(bt[s]), ds, heads, kv_heads, dim, int(begin[s]),
                            int(n_kv[s]), pt, dim ** -0.5, KvType.F16)
        want = ctx.download(one, np.float32, q.shape[1:])
        assert np.max(np.abs(got[s] - want)) <= 2.0 ** -20 * np.max(np.abs(want)), s

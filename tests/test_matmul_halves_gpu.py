"""The chunk product whose work-groups halve their reduction between two groups of four waves
(moearc_matmul2x_*: grids of three quarters of a tile per CU up to one): every format, reductions that
the halves share evenly and not (an odd block, three super-blocks), ragged last row and token tiles,
and bias. Oracle bound: the matvec's, the matrix core's block sums (64
wide at most, 2 * 64 u sum|w x|; one more f32 addition of the halves is half an ulp) and the bias add's
half an ulp."""
from __future__ import annotations

import numpy as np
import pytest

import fixtures as fx
from moearc_amd import QuantType
from oracle import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [6017, 8192])  # 48 and 64 row tiles x 4 token tiles
@pytest.mark.parametrize("ty,cols", [(QuantType.F16, 544), (QuantType.Q8_0, 576), (QuantType.MXFP4, 320),
                                     (QuantType.Q4_K, 768), (QuantType.Q5_K, 512), (QuantType.Q6_K, 768)], ids=str)
def test_halved_reduction(ctx, ty, cols, rows):
    n_tok = 400
    w, _ = fx.synth_blocks(int(ty), rows * cols // ty.block_elems, 0x3E1 + rows)
    x = fx.synth.unit(0x3E2 + cols, n_tok * cols).reshape(n_tok, cols)
    b = fx.synth.unit(0x3E3, rows)
    y = ctx.alloc(n_tok * rows * 4)
    ctx.matmul_q(ty, y, ctx.upload(w), ctx.upload(x), ctx.upload(b), n_tok, rows, cols)
    got = ctx.download(y, np.float32, (n_tok, rows)).astype(np.float64)
    worst = 0.0
    for t in (0, 33, 127, 128, 300, 383, 384, 399):
        want, absum = oracle.matvec_q(int(ty), w, x[t], rows, cols, n_threads=8)
        want = want.astype(np.float64) + b
        tol = fx.matvec_tolerance(cols, absum) + 2.0 * 64 * 2.0 ** -24 * absum + 2.0 ** -22 * np.abs(want)
        worst = max(worst, float(np.max(np.abs(got[t] - want) / tol)))
    print(f"{ty.name} {n_tok} x {rows} x {cols}: worst / bound = {worst:.3f}", flush=True)
    assert worst <= 1.0

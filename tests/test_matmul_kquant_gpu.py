"""The chunk product of Q4_K and Q5_K weights on 128 x 128 tiles (moearc_matmul2_{q4_k,q5_k}_k): one and
several super-blocks, whole and split reductions, ragged token and row tiles, and activations aligned
to four bytes (moearc_split_sums_k's element loads), against the oracle's matvec. The bound is the
matvec's, plus the matrix core's running sums of a pair of sub-blocks (2 * 64 u sum|w x|, the mins' eight
terms among them) and half an ulp for the bias add."""
from __future__ import annotations

import numpy as np
import pytest

import fixtures as fx
from moearc_amd import DeviceView, QuantType
from oracle import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_tok,rows,cols,x_off", [
    (65, 1, 256, 0), (70, 129, 512, 4), (128, 128, 2304, 0), (129, 300, 768, 8), (300, 257, 2048, 0)])
@pytest.mark.parametrize("ty", [QuantType.Q4_K, QuantType.Q5_K], ids=lambda t: t.name)
def test_super_blocks(ctx, ty, n_tok, rows, cols, x_off):
    w, _ = fx.synth_blocks(int(ty), rows * cols // 256, 0x3D1 + rows)
    x = 3.0 * fx.synth.unit(0x3D2 + cols, n_tok * cols).reshape(n_tok, cols).astype(np.float32) + np.float32(0.5)
    b = fx.synth.unit(0x3D3, rows)
    y = ctx.alloc(n_tok * rows * 4)
    raw = ctx.upload(np.concatenate([np.zeros(x_off // 4, np.float32), x.reshape(-1)]))
    ctx.matmul_q(ty, y, ctx.upload(w), DeviceView(raw, x_off), ctx.upload(b), n_tok, rows, cols)
    got = ctx.download(y, np.float32, (n_tok, rows)).astype(np.float64)
    worst = 0.0
    for t in sorted({0, 1, 31, 63, 64, n_tok // 2, n_tok - 2, n_tok - 1}):
        want, absum = oracle.matvec_q(int(ty), w, x[t], rows, cols, n_threads=8)
        want = want.astype(np.float64) + b
        tol = fx.matvec_tolerance(cols, absum) + 2.0 * 64 * 2.0 ** -24 * absum + 2.0 ** -23 * np.abs(want)
        worst = max(worst, float(np.max(np.abs(got[t] - want) / tol)))
    print(f"{ty.name} {n_tok} x {rows} x {cols}: worst / bound = {worst:.3f}", flush=True)
    assert worst <= 1.0


@pytest.mark.parametrize("n_tok,rows,cols", [(5, 40, 512), (24, 33, 256), (64, 50, 768),  # matmul_small.hip
                                             (70, 129, 512), (130, 40, 2304), (400, 6017, 512)])
@pytest.mark.parametrize("size", [1.0, 2.0 ** -20])
@pytest.mark.parametrize("ty", [QuantType.Q4_K, QuantType.Q5_K], ids=lambda t: t.name)
def test_mins_take_f32_sums(ctx, ty, size, n_tok, rows, cols):
    # payloads of zero leave -dmin * m * (sum of x): sums of f32 activations, not of the f16 pieces that the
    # payloads' product takes (at 2^-20 those keep 5 bits)
    w, _ = fx.synth_blocks(int(ty), rows * cols // 256, 0x3D4 + rows)
    w = w.reshape(-1, 144 if ty == QuantType.Q4_K else 176).copy()
    w[:, 16:] = 0
    x = (size * (fx.synth.unit(0x3D5 + cols, n_tok * cols).reshape(n_tok, cols) + 0.25)).astype(np.float32)
    y = ctx.alloc(n_tok * rows * 4)
    ctx.matmul_q(ty, y, ctx.upload(w), ctx.upload(x), None, n_tok, rows, cols)
    got = ctx.download(y, np.float32, (n_tok, rows)).astype(np.float64)
    worst = 0.0
    for t in sorted({0, 1, n_tok // 2, n_tok - 1}):
        want, absum = oracle.matvec_q(int(ty), w, x[t], rows, cols, n_threads=8)
        # the sums' 32 terms, then one multiply-add per sub-block
        tol = (32 + cols // 32 + 5) * 2.0 ** -24 * absum
        worst = max(worst, float(np.max(np.abs(got[t] - want) / tol)))
    print(f"{ty.name} {n_tok} x {rows} x {cols}: worst / bound = {worst:.3f}", flush=True)
    assert worst <= 1.0

"""The chunk product of a few tokens (moearc_matmul_small_*): every format against the oracle's matvec at
the token counts where its tiles end, at row counts around a tile and at reductions around its windows
(the shortest row, waves without work, a last window that starts early), with weights aligned to two
bytes and activations to four. The bound is the chunk product's: the matvec's, the matrix core's 32-wide
block sums (2 * 32 u sum|w x|) and half an ulp for the bias add."""
from __future__ import annotations

import numpy as np
import pytest

import fixtures as fx
from moearc_amd import Context, DeviceView, QuantType
from oracle import oracle

pytestmark = pytest.mark.gpu

BLOCKS = [QuantType.F16, QuantType.Q8_0, QuantType.MXFP4]
SUPER = [QuantType.Q4_K, QuantType.Q5_K, QuantType.Q6_K]


def _check(ctx, ty, n_tok, rows, cols, bias=True, w_off=0, x_off=0, run=32):
    w, _ = fx.synth_blocks(int(ty), rows * cols // ty.block_elems, 0x3C3 + rows)
    x = fx.synth.unit(0x3C4 + cols, n_tok * cols).reshape(n_tok, cols)
    b = fx.synth.unit(0x3C5, rows)
    y = ctx.alloc(n_tok * rows * 4)
    at = lambda raw, off: DeviceView(ctx.upload(np.concatenate([np.zeros(off, np.uint8), raw.reshape(-1).view(np.uint8)])), off)
    ctx.matmul_q(ty, y, at(w, w_off), at(x, x_off), ctx.upload(b) if bias else None, n_tok, rows, cols)
    got = ctx.download(y, np.float32, (n_tok, rows)).astype(np.float64)
    worst = 0.0
    for t in range(n_tok):
        want, absum = oracle.matvec_q(int(ty), w, x[t], rows, cols, n_threads=8)
        want = want.astype(np.float64) + (b if bias else 0.0)
        tol = fx.matvec_tolerance(cols, absum) + 2.0 * run * 2.0 ** -24 * absum + 2.0 ** -23 * np.abs(want)
        worst = max(worst, float(np.max(np.abs(got[t] - want) / tol)))
    print(f"{ty.name} {n_tok} x {rows} x {cols}: worst / bound = {worst:.3f}", flush=True)
    assert worst <= 1.0


@pytest.mark.parametrize("n_tok", [2, 16, 17, 32, 33, 48, 49, 64])
@pytest.mark.parametrize("ty", BLOCKS + SUPER, ids=lambda t: t.name)
def test_token_tiles(ctx, ty, n_tok):
    _check(ctx, ty, n_tok, 33, 512)


@pytest.mark.parametrize("rows", [1, 16, 300])
@pytest.mark.parametrize("cols", [256, 288, 2016, 2880])
@pytest.mark.parametrize("ty", BLOCKS, ids=lambda t: t.name)
def test_windows_of_blocks(ctx, ty, cols, rows):
    _check(ctx, ty, 5, rows, cols, bias=rows != 16)
    _check(ctx, ty, 40, rows, cols)


@pytest.mark.parametrize("cols", [256, 2048, 4352])
@pytest.mark.parametrize("ty", SUPER, ids=lambda t: t.name)
def test_windows_of_super_blocks(ctx, ty, cols):
    _check(ctx, ty, 5, 50, cols)
    _check(ctx, ty, 20, 50, cols)


@pytest.mark.parametrize("ty", BLOCKS + SUPER, ids=lambda t: t.name)
def test_unaligned_buffers(ctx, ty):
    _check(ctx, ty, 18, 40, 768, w_off=2, x_off=4)


@pytest.mark.parametrize("n_tok,shift", [(2, 0), (17, 0), (32, 512), (64, -1024)])
@pytest.mark.parametrize("ty", BLOCKS + SUPER, ids=lambda t: t.name)
def test_over_its_own_input(ctx, ty, n_tok, shift):
    # y on x, and y starting a row after x or two rows before it (shift floats)
    n = 512
    w, _ = fx.synth_blocks(int(ty), n * n // ty.block_elems, 0x3C8)
    x = fx.synth.unit(0x3C9, n_tok * n).reshape(n_tok, n)
    at_x, at_y = max(0, -shift), max(0, shift)
    raw = ctx.upload(np.concatenate([np.zeros(at_x, np.float32), x.reshape(-1), np.zeros(at_y, np.float32)]))
    ctx.matmul_q(ty, DeviceView(raw, 4 * at_y), ctx.upload(w), DeviceView(raw, 4 * at_x), None, n_tok, n, n)
    got = ctx.download(raw, np.float32, n_tok * n + abs(shift))[at_y:at_y + n_tok * n].reshape(n_tok, n)
    for t in range(n_tok):
        want, absum = oracle.matvec_q(int(ty), w, x[t], n, n, n_threads=8)
        tol = fx.matvec_tolerance(n, absum) + 2.0 * 64 * 2.0 ** -24 * absum
        assert np.all(np.abs(got[t] - want) <= tol)


@pytest.mark.parametrize("n_tok,rows,cols", [(5, 8200, 256), (20, 8200, 768), (40, 4112, 768),  # matmul.hip
                                             (40, 4112, 2048), (63, 4100, 1024), (66, 130, 256)])  # 128 x 128 tiles
@pytest.mark.parametrize("ty", BLOCKS + SUPER, ids=lambda t: t.name)
def test_where_the_form_ends(ctx, ty, n_tok, rows, cols):
    # more rows or tokens than it takes (tests/test_dispatch.py has the rule): the other kernels of few tokens.
    # The tiles' K-quants add up pairs of blocks in the matrix cores (run)
    _check(ctx, ty, n_tok, rows, cols, run=64)


def test_same_product_in_any_chunk_of_a_tile(ctx):
    # a token's result does not depend on its neighbours: rows of a 32-token product equal those of a
    # 7-token one (one or two token tiles, the same reduction)
    ty, rows, cols = QuantType.Q8_0, 100, 1024
    w, _ = fx.synth_blocks(int(ty), rows * cols // 32, 0x3C6)
    x = fx.synth.unit(0x3C7, 32 * cols).reshape(32, cols)
    dw, out = ctx.upload(w), []
    for n in (7, 32):
        y = ctx.alloc(n * rows * 4)
        ctx.matmul_q(ty, y, dw, ctx.upload(x[:n]), None, n, rows, cols)
        out.append(ctx.download(y, np.float32, (n, rows)))
    assert np.array_equal(out[0], out[1][:7])

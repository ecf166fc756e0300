"""Which kernels the entry points launch, and what memory they take for it, on the host alone (host_hip.py)."""
from __future__ import annotations

import pytest

import host_hip
from host_hip import at, names
from moearc_amd import Context, KvType, QuantType, native
from moearc_amd.context import Failed

MM = [QuantType.F16, QuantType.Q8_0, QuantType.MXFP4, QuantType.Q4_K, QuantType.Q5_K, QuantType.Q6_K]


@pytest.fixture(scope="module")
def built(tmp_path_factory):
    return host_hip.build(tmp_path_factory.mktemp("host"))


@pytest.fixture
def lib(built, monkeypatch):
    monkeypatch.setattr(native, "_lib", built)
    built.host_hip_reset()
    yield built
    built.host_hip_reset()


@pytest.mark.parametrize("n_tok", [1, 2, 17, 32, 33, 64])
@pytest.mark.parametrize("ty", MM, ids=lambda t: t.name)
def test_a_product_over_its_own_input_reads_it_first(lib, ty, n_tok):
    # y may overlap x: the activations are then split into the workspace before any row is written; the
    # one-launch form, whose work-groups read x while others write y, is for buffers apart
    n, size = 512, 64 * 512 * 4
    with Context() as cx:
        def call(y, x):
            lib.host_hip_reset()
            cx.matmul_q(ty, at(cx, y, size), at(cx, 1 << 33, ty.row_bytes(n) * n), at(cx, x, size), None, n_tok, n, n)
            return names(lib)
        x = 1 << 32
        used = n_tok * n * 4
        for y in (x - used, x + used):
            assert [k.rsplit("_t", 1)[0] for k in call(y, x)] == [f"moearc_matmul_small_{ty.name.lower()}"]
        for y in (x, x + 4, x - 4, x + used - 4, x - used + 4):
            got = call(y, x)
            assert any(k.startswith("moearc_split") for k in got) and not any("small" in k for k in got), got


def _product(cx, lib, ty, n_tok, rows, cols):
    lib.host_hip_reset()
    size = 1 << 40
    cx.matmul_q(ty, at(cx, 1 << 41, size), at(cx, 1 << 42, size), at(cx, 1 << 43, size), None, n_tok, rows, cols)
    got = [k for k in names(lib) if "split" not in k and "sums" not in k and "reduce" not in k]
    assert len(got) == 1
    return got[0]


Q = QuantType


@pytest.mark.parametrize("ty,n_tok,rows,cols,form", [
    # up to 32 tokens: the one launch while the rows are few, or long enough; F16 not past its row counts
    (Q.Q8_0, 32, 8192, 256, "small"), (Q.Q8_0, 1, 8193, 256, "16"), (Q.Q8_0, 16, 8193, 1024, "small"),
    (Q.Q8_0, 17, 8193, 1024, "16"), (Q.Q8_0, 17, 151936, 2048, "small"), (Q.MXFP4, 32, 8193, 1024, "small"),
    (Q.MXFP4, 2, 8193, 992, "16"), (Q.Q4_K, 32, 262144, 1024, "small"), (Q.Q4_K, 32, 8193, 768, "16"),
    (Q.Q5_K, 3, 8193, 768, "16"), (Q.Q6_K, 3, 8193, 768, "16"), (Q.F16, 32, 40960, 2880, "small"),
    (Q.F16, 17, 40961, 2880, "16"), (Q.F16, 16, 49152, 2880, "small"), (Q.F16, 9, 49153, 2880, "16"),
    (Q.F16, 8, 65536, 2880, "small"), (Q.F16, 8, 65537, 2880, "16"), (Q.F16, 8, 8193, 1000 - 1000 % 32, "16"),
    (Q.Q8_0, 32, 64, 224, "16"),
    # 33 to 64: in one round of work-groups the one launch, else the tiles, over short rows the 16 x 16 kernels
    (Q.Q8_0, 64, 4096, 2880, "small"), (Q.Q8_0, 63, 4097, 2880, "tiles"), (Q.Q8_0, 63, 4097, 960, "16"),
    (Q.Q4_K, 33, 4097, 1024, "tiles"), (Q.Q4_K, 63, 4097, 768, "16"), (Q.Q6_K, 33, 4097, 512, "16"),
    (Q.F16, 33, 4097, 2048, "tiles"), (Q.F16, 63, 4097, 2016, "16"), (Q.F16, 64, 4097, 256, "tiles"),
    # 65 and more: the tiles, but for rows of an odd number of Q8_0 or MXFP4 blocks
    (Q.Q6_K, 65, 16, 256, "tiles"), (Q.Q8_0, 65, 16, 288, "16"), (Q.MXFP4, 500, 16, 96, "16"),
    # a grid of about one tile per CU halves its reduction inside the work-group; F16, Q8_0 and MXFP4 go wide
    (Q.Q4_K, 1000, 4096, 2048, "halves"), (Q.Q4_K, 1000, 2944, 2048, "tiles"), (Q.Q8_0, 400, 6017, 576, "halves"),
    (Q.Q6_K, 2048, 4096, 2048, "tiles"), (Q.Q8_0, 2048, 4096, 2880, "wide"),
], ids=str)
def test_product_forms(lib, ty, n_tok, rows, cols, form):
    name = ty.name.lower()
    want = {"small": f"moearc_matmul_small_{name}_t{-(-n_tok // 16)}_k", "tiles": f"moearc_matmul2_{name}_k",
            "halves": f"moearc_matmul2x_{name}_k", "wide": f"moearc_matmul2w_{name}_k", "16": f"moearc_matmul_{name}_r"}
    with Context() as cx:
        got = _product(cx, lib, ty, n_tok, rows, cols)
        assert got.startswith(want[form]), got


def test_forms_that_the_gpu_tests_mean(lib):
    # the shapes of test_matmul_halves_gpu.py and test_matmul_kquant_gpu.py run the kernels that those are about
    with Context() as cx:
        for ty, cols in [(Q.F16, 544), (Q.Q8_0, 576), (Q.MXFP4, 320), (Q.Q4_K, 768), (Q.Q5_K, 512), (Q.Q6_K, 768)]:
            for rows in (6017, 8192):
                assert _product(cx, lib, ty, 400, rows, cols) == f"moearc_matmul2x_{ty.name.lower()}_k"
        for n_tok, rows, cols in [(65, 1, 256), (70, 129, 512), (128, 128, 2304), (129, 300, 768), (300, 257, 2048)]:
            for ty in (Q.Q4_K, Q.Q5_K):
                assert _product(cx, lib, ty, n_tok, rows, cols) == f"moearc_matmul2_{ty.name.lower()}_k"


def test_without_the_small_form(lib, monkeypatch):
    # MOEARC_MM_SMALL=0: the kernels that it replaced
    monkeypatch.setenv("MOEARC_MM_SMALL", "0")
    with Context() as cx:
        for ty in MM:
            assert _product(cx, lib, ty, 8, 4096, 2048).startswith(f"moearc_matmul_{ty.name.lower()}_r")
            assert _product(cx, lib, ty, 40, 4096, 2048) == f"moearc_matmul2_{ty.name.lower()}_k"


BIG = 1 << 44


def _decode(cx, kv, dim, n_kv, heads=32, kv_heads=4, page=256, base=1 << 33, scale=0.125):
    cx.attn_decode_ext(*(at(cx, base + i * BIG, BIG) for i in range(6)), heads, kv_heads, dim, 0, n_kv, page, scale,
                       KvType.F16 if kv == "f16" else KvType.F32)


def _prefill(cx, n_q=200, pos0=16301):
    cx.attn_prefill(*(at(cx, (1 << 33) + i * BIG, BIG) for i in range(6)), n_q, pos0, 0, 64, 8, 64, 256, 0.125)


KINDS = [("f16", 128), ("f32", 64), ("f32", 128)]


@pytest.mark.parametrize("kv,dim", KINDS)
def test_decode_without_memory_for_records_is_not_split(lib, kv, dim):
    # the general kernel, which took these caches before, needed no memory: neither may they
    with Context() as cx:
        lib.host_hip_largest(1 << 16)
        _decode(cx, kv, dim, 20000)
        one = names(lib)
        assert len(one) == 1 and f"{kv}d{dim}" in one[0] and lib.host_hip_last_error() == 0
        lib.host_hip_reset()
        _decode(cx, kv, dim, 20000)
        assert len(names(lib)) == 2 and "merge" in names(lib)[1]
        lib.host_hip_reset()
        lib.host_hip_largest(1 << 16)  # a workspace that cannot grow
        _decode(cx, kv, dim, 20000, heads=64)
        assert len(names(lib)) == 1


@pytest.mark.parametrize("kv,dim", KINDS)
def test_scales_past_the_log2_domain_take_the_general_kernel(lib, kv, dim):
    # the split kernels multiply scores by scale * log2(e), which must be finite
    with Context() as cx:
        for scale, general in ((2.0e38, False), (2.4e38, True), (0.0, True), (-1.0, True), (1.0e-40, False)):
            lib.host_hip_reset()
            _decode(cx, kv, dim, 100, scale=scale)
            assert (names(lib) == ["moearc_attn_decode_general_k"]) == general


def test_prefill_without_memory_for_records_is_not_split(lib):
    with Context() as cx:
        lib.host_hip_largest(1 << 16)
        _prefill(cx)
        assert names(lib) == ["moearc_attn_prefill_g8"] and lib.host_hip_last_error() == 0
        lib.host_hip_reset()
        _prefill(cx)
        assert names(lib) == ["moearc_attn_prefill_split_g8", "moearc_attn_prefill_merge_k"]


@pytest.mark.parametrize("kv,dim", KINDS)
def test_a_span_too_long_for_one_split_takes_the_general_kernel(lib, kv, dim):
    # a split holds at most 2^30 keys; where records are not to be had, longer spans stay with the general kernel
    n_kv = 3 << 30
    with Context() as cx:
        _decode(cx, kv, dim, n_kv, page=1 << 20)
        assert len(names(lib)) == 2
        for prepare in (lambda: lib.host_hip_capture(1, 0), lambda: lib.host_hip_largest(1 << 10)):
            lib.host_hip_reset()
            prepare()
            _decode(cx, kv, dim, n_kv, heads=64, page=1 << 20)
            assert names(lib) == ["moearc_attn_decode_general_k"]


def test_growing_a_workspace_leaves_another_capture_alone(lib):
    # a program may capture one stream while a context calls eagerly on its own: allocations then need a relaxed
    # thread, or they fail and break the capture
    with Context() as cx:
        lib.host_hip_capture(0, 1)
        _prefill(cx)
        assert names(lib) == ["moearc_attn_prefill_split_g8", "moearc_attn_prefill_merge_k"]
        for kv, dim in KINDS:
            _decode(cx, kv, dim, 20000)
        _prefill(cx, 200, 30000)
        assert lib.host_hip_broken_captures() == 0
        assert lib.hipMalloc(None, 16) != 0 and lib.host_hip_broken_captures() == 1  # the mode is the thread's own again
        lib.host_hip_capture(0, 0)


def test_a_captured_call_that_needs_a_workspace_is_refused(lib):
    # 64-channel f16 heads keep their records in the workspace: growing it under capture fails, as ever
    with Context() as cx:
        lib.host_hip_capture(1, 0)
        with pytest.raises(Failed):
            _decode(cx, "f16", 64, 20000)
        assert names(lib) == []
        lib.host_hip_capture(0, 0)
        _decode(cx, "f16", 64, 20000)
        lib.host_hip_capture(1, 0)
        _decode(cx, "f16", 64, 20000)
        lib.host_hip_capture(0, 0)

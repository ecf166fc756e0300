"""What the attention hot path is asked to do in use, case by case, through `moearc_amd.Context`.

Five kinds of call, in the sizes a program that serves a model makes them:

* ``step``    one decode step's attention of a 36-block model at batch 1: 18 windowed and 18 full
              calls of ``attn_decode_ext``, each block with its own cache (the reference's headline).
* ``decode``  one layer's decode attention: ``attn_decode_ext`` for a single sequence with f32
              output, ``attn_decode_batched`` for a ragged batch or f16 output.
* ``prefill`` one layer's chunked prefill attention, ``attn_prefill``.
* ``block``   the attention half of one block, ``attn_block_chunk``: projections, RoPE, the cache
              append, attention, the output projection and the residual; one token is a decode step.
* ``matmul``  one projection over a prompt chunk, ``matmul_q``.

Inputs are made on the GPU from a seed: N(0,1) queries, keys and values, normed activations of
N(0,1), weights of a trained projection's size in each GGUF format, caches in pages scattered by a
random permutation. Every buffer is a torch tensor that the library sees through a ``DeviceView``,
as a program that holds its model in torch would pass it.
"""
from __future__ import annotations

import math
import random
from types import SimpleNamespace

import torch

from moearc_amd import OUT_F16, OUT_F32, AttnBlockDesc, Context, DeviceView, KvType, QuantType, RopeScaling

YARN = dict(n_ctx_orig=4096, freq_base=150000.0, factor=32.0)  # the rotary scaling of the blocks


# ---- the cases -----------------------------------------------------------------------------------

def _decode(name, batch, keys_min, keys_max, window=0, heads=64, kv_heads=8, dim=64, kv="f16", page=256,
            out="f32", lens_seed=1):
    c = dict(kind="decode", batch=batch, keys_min=keys_min, keys_max=keys_max, window=window, heads=heads,
             kv_heads=kv_heads, dim=dim, kv=kv, page=page, out=out, lens_seed=lens_seed)
    return dict(name=name, **c) if name else c


def _prefill(name, tokens, pos0, window=0, heads=64, kv_heads=8, page=256, out="f16"):
    c = dict(kind="prefill", tokens=tokens, pos0=pos0, window=window, heads=heads, kv_heads=kv_heads, page=page,
             out=out)
    return dict(name=name, **c) if name else c


def _block(name, tokens, pos0, type="Q8_0", window=0, embd=2880, heads=64, kv_heads=8, page=256):
    c = dict(kind="block", tokens=tokens, pos0=pos0, type=type, window=window, embd=embd, heads=heads,
             kv_heads=kv_heads, page=page)
    return dict(name=name, **c) if name else c


def _matmul(name, type, tokens, rows, cols, bias=True):
    c = dict(kind="matmul", type=type, tokens=tokens, rows=rows, cols=cols, bias=bias)
    return dict(name=name, **c) if name else c


def listed():
    return [
        # The reference's own headline: the attention of one decode step at a chat-sized context.
        # 36 small calls, so launches and the host's share of each call count.
        dict(name="step_2k", kind="step", depth=2048, window=128, heads=64, kv_heads=8, page=256),
        # A single user at a long context: one full-causal layer over 32K keys.
        _decode("decode_b1_32k", 1, 32768, 32768, out="f16"),
        # A serving batch of 32 sequences of mixed lengths, a full-causal layer and a windowed one.
        _decode("decode_b32_ragged", 32, 1024, 32768, out="f16"),
        _decode("decode_b32_window", 32, 1024, 32768, window=128, out="f16"),
        # The largest call: eight sequences of 128K keys (documents, agents), 2 GiB of cache.
        _decode("decode_b8_128k", 8, 131072, 131072, out="f16"),
        # The other head size that the supported models have (Qwen3-30B-A3B: 32 heads over 4 KV
        # heads of 128 channels): four chats of mixed lengths.
        _decode("decode_d128_b4", 4, 2048, 8192, heads=32, kv_heads=4, dim=128),
        # A long prompt's 2048-token chunk behind 2048 cached tokens, both layer types.
        _prefill("prefill_2k", 2048, 2048),
        _prefill("prefill_2k_window", 2048, 2048, window=128),
        # A follow-up message of a few hundred tokens deep in a long conversation.
        _prefill("prefill_200_at_16k", 200, 16301),
        # One decode step of a whole attention block, and a short prompt through it.
        _block("block_step", 1, 3000),
        _block("block_prompt_128", 128, 0),
        # A K-quant projection (Qwen3-30B-A3B's q) over a ragged prompt.
        _matmul("matmul_q4k_1k", "Q4_K", 1000, 4096, 2048),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "prefill", "block", "matmul"])
    if kind == "decode":
        # 64-channel heads as gpt-oss groups them or otherwise, 128-channel heads, now and then an
        # f32 cache; up to 32 sequences and 512K keys in all
        heads, kv_heads, dim, kv = rng.choice([(64, 8, 64, "f16"), (64, 8, 64, "f16"), (32, 8, 64, "f16"),
                                               (32, 4, 128, "f16"), (32, 4, 128, "f16"), (16, 16, 128, "f16"),
                                               (64, 8, 64, "f32"), (32, 4, 128, "f32")])
        batch = rng.choice([1, 1, 2, 5, 8, 17, 32])
        top = _log_int(rng, 100, min(65536, 524288 // batch))
        return _decode(None, batch, max(1, top // rng.choice([1, 2, 16])), top, rng.choice([0, 0, 0, 128]), heads,
                       kv_heads, dim, kv, rng.choice([16, 256, 256]), rng.choice(["f32", "f16"]),
                       rng.randrange(1 << 20))
    if kind == "prefill":
        heads, kv_heads = rng.choice([(64, 8), (64, 8), (64, 8), (32, 8), (16, 16)])
        return _prefill(None, _log_int(rng, 16, 2048), rng.choice([0, _log_int(rng, 1, 24000)]),
                        rng.choice([0, 0, 128]), heads, kv_heads, rng.choice([16, 256, 256]),
                        rng.choice(["f16", "f32"]))
    if kind == "block":
        embd, heads, kv_heads, types = rng.choice([(2880, 64, 8, ["Q8_0", "Q8_0", "MXFP4", "F16"]),
                                                   (2880, 64, 8, ["Q8_0", "Q8_0", "MXFP4", "F16"]),
                                                   (2048, 32, 4, ["Q4_K", "Q5_K", "Q6_K", "Q8_0"])])
        return _block(None, rng.choice([1, _log_int(rng, 1, 1024)]), rng.choice([0, _log_int(rng, 1, 8000)]),
                      rng.choice(types), rng.choice([0, 128]), embd, heads, kv_heads)
    rows, cols, types = rng.choice([(4096, 2880, ["Q8_0", "MXFP4", "F16"]), (2880, 4096, ["Q8_0", "MXFP4", "F16"]),
                                    (512, 2880, ["Q8_0", "F16"]),
                                    (4096, 2048, ["Q4_K", "Q5_K", "Q6_K", "Q8_0", "MXFP4"]),
                                    (2048, 4096, ["Q4_K", "Q5_K", "Q6_K", "Q8_0"])])
    return _matmul(None, rng.choice(types), _log_int(rng, 2, 2048), rows, cols, rng.choice([True, False]))


# ---- inputs --------------------------------------------------------------------------------------

_kept = {}


def _context():
    """The program's one context."""
    if "ctx" not in _kept:
        _kept["ctx"] = Context()
    return _kept["ctx"]


def _view(t):
    """A torch tensor as the library's buffer; the view keeps the tensor alive."""
    owner = SimpleNamespace(ctx=_context(), ptr=t.data_ptr(), len=t.numel() * t.element_size(), tensor=t)
    return DeviceView(owner, 0)


def _rng(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _normal(g, *shape, dtype=torch.float32):
    return torch.randn(*shape, generator=g, device="cuda", dtype=dtype)


def _spans(case):
    """[(first key, end)] of a decode case's sequences."""
    r = random.Random(case["lens_seed"])
    lens = [r.randint(case["keys_min"], case["keys_max"]) for _ in range(case["batch"])]
    return [(max(0, n - case["window"]) if case["window"] else 0, n) for n in lens]


def _cache(g, tokens, kv_heads, dim, page, dtype=torch.float16):
    """K and V pools of enough pages for each sequence's tokens, and their block tables: every
    sequence's pages are its own, scattered over the pool."""
    counts = [-(-n // page) for n in tokens]
    total, stride = sum(counts), max(counts)
    perm = torch.randperm(total, generator=g, device="cuda").to(torch.int32)
    tables = torch.zeros(len(tokens), stride, device="cuda", dtype=torch.int32)
    at = 0
    for b, n in enumerate(counts):
        tables[b, :n] = perm[at:at + n]
        at += n
    k = _normal(g, total, page, kv_heads, dim, dtype=dtype)
    v = _normal(g, total, page, kv_heads, dim, dtype=dtype)
    return k, v, tables


def _bytes_of(x):
    return x.contiguous().view(torch.uint8)


def _weights(g, type, rows, cols, dense=False):
    """A weight matrix in a GGUF format, as uint8 [rows, row bytes], of N(0, 0.02)-like values; with
    `dense` its float64 value instead, from the same draws."""
    def ints(lo, hi, *shape):
        return torch.randint(lo, hi, shape, generator=g, device="cuda", dtype=torch.int32)

    def scales(size, *shape):
        return (torch.rand(*shape, generator=g, device="cuda") * 0.6 + 0.7).mul(size).half()

    u8 = torch.uint8
    if type == "F16":
        w = (_normal(g, rows, cols) * 0.02).half()
        return w.double() if dense else _bytes_of(w).view(rows, -1)
    if type == "Q8_0":
        n = cols // 32
        w = _normal(g, rows, n, 32) * 0.02
        d = (w.abs().amax(-1, keepdim=True) / 127).half()
        q = (w / d.float()).round().clamp(-127, 127).to(torch.int8)
        if dense:
            return (d.double() * q.double()).view(rows, cols)
        return torch.cat([_bytes_of(d), _bytes_of(q)], -1).view(rows, -1)
    if type == "MXFP4":
        n = cols // 32
        e, q = ints(119, 122, rows, n, 1), ints(0, 16, rows, n, 32)
        if dense:
            code = torch.tensor([0, 0.5, 1, 1.5, 2, 3, 4, 6], device="cuda", dtype=torch.float64)
            v = code[(q & 7).long()] * torch.where(q >= 8, -1.0, 1.0)
            return (v * torch.exp2((e - 127).double())).view(rows, cols)
        return torch.cat([e.to(u8), (q[..., :16] | q[..., 16:] << 4).to(u8)], -1).view(rows, -1)
    n = cols // 256
    if type in ("Q4_K", "Q5_K"):
        top = 16 if type == "Q4_K" else 32
        d, q = scales(0.02 / 45 / (top * 0.29), rows, n, 1), ints(0, top, rows, n, 8, 32)
        sc, m = ints(20, 64, rows, n, 8), ints(20, 64, rows, n, 8)
        dmin = (d.float() * (top - 1) / 2).half()
        if dense:
            w = d.double().unsqueeze(-1) * (sc.unsqueeze(-1) * q).double() - (dmin.double() * m.double()).unsqueeze(-1)
            return w.view(rows, cols)
        packed = torch.cat([sc[..., :4] | (sc[..., 4:] >> 4) << 6, m[..., :4] | (m[..., 4:] >> 4) << 6,
                            (sc[..., 4:] & 15) | (m[..., 4:] & 15) << 4], -1).to(u8)
        low = q & 15
        qs = (low[..., 0::2, :] | low[..., 1::2, :] << 4).to(u8).reshape(rows, n, 128)
        parts = [_bytes_of(d), _bytes_of(dmin), packed, qs]
        if type == "Q5_K":
            bit = torch.arange(8, device="cuda", dtype=torch.int32).view(8, 1)
            parts.insert(3, ((q >> 4) << bit).sum(-2).to(u8))
        return torch.cat(parts, -1).view(rows, -1)
    assert type == "Q6_K"
    d, q = scales(0.02 / 80 / 18.5, rows, n, 1), ints(0, 64, rows, n, 2, 4, 32)
    sc = ints(40, 120, rows, n, 16) * (ints(0, 2, rows, n, 16) * 2 - 1)
    if dense:
        w = d.double().unsqueeze(-1) * sc.double().unsqueeze(-1) * (q.view(rows, n, 16, 16) - 32).double()
        return w.view(rows, cols)
    low, high = q & 15, q >> 4
    ql = torch.cat([low[..., 0, :] | low[..., 2, :] << 4, low[..., 1, :] | low[..., 3, :] << 4], -1)
    qh = high[..., 0, :] | high[..., 1, :] << 2 | high[..., 2, :] << 4 | high[..., 3, :] << 6
    return torch.cat([ql.to(u8).view(rows, n, 128), qh.to(u8).view(rows, n, 64), _bytes_of(sc.to(torch.int8)),
                      _bytes_of(d)], -1).view(rows, -1)


def _block_shapes(case):
    q, kv = case["heads"] * 64, case["kv_heads"] * 64
    return [(q, case["embd"]), (kv, case["embd"]), (kv, case["embd"]), (case["embd"], q)]


def _block_inputs(case, seed, dense=False):
    g = _rng(seed)
    s = SimpleNamespace()
    n, total = case["tokens"], case["pos0"] + case["tokens"]
    s.k, s.v, s.table = _cache(g, [total], case["kv_heads"], 64, case["page"])
    s.x, s.h = _normal(g, n, case["embd"]), _normal(g, n, case["embd"])
    s.sinks = _normal(g, case["heads"])
    shapes = _block_shapes(case)
    s.bias = [_normal(g, r) * 0.1 for r, _ in shapes]
    s.w = [_weights(g, case["type"], r, c, dense) for r, c in shapes]
    t = torch.arange(case["pos0"], total, device="cuda", dtype=torch.int32)
    s.pos, s.pages, s.slots = t, s.table[0][(t // case["page"]).long()].contiguous(), t % case["page"]
    return s


def _decode_inputs(case, seed):
    g = _rng(seed)
    s = SimpleNamespace(spans=_spans(case))
    s.k, s.v, s.table = _cache(g, [n for _, n in s.spans], case["kv_heads"], case["dim"], case["page"],
                               torch.float16 if case["kv"] == "f16" else torch.float32)
    s.q, s.sinks = _normal(g, case["batch"], case["heads"], case["dim"]), _normal(g, case["heads"])
    return s


def _prefill_inputs(case, seed):
    g = _rng(seed)
    s = SimpleNamespace()
    s.k, s.v, s.table = _cache(g, [case["pos0"] + case["tokens"]], case["kv_heads"], 64, case["page"])
    s.q, s.sinks = _normal(g, case["tokens"], case["heads"], 64, dtype=torch.float16), _normal(g, case["heads"])
    return s


def _matmul_inputs(case, seed, dense=False):
    g = _rng(seed)
    s = SimpleNamespace(x=_normal(g, case["tokens"], case["cols"]))
    s.bias = _normal(g, case["rows"]) * 0.1 if case["bias"] else None
    s.w = _weights(g, case["type"], case["rows"], case["cols"], dense)
    return s


def _step_inputs(case, seed):
    """Per block (k, v, table, sinks, q): even blocks windowed, in a ring of two pages through the
    cyclic table, odd ones full causal in scattered pages."""
    g = _rng(seed)
    n = case["depth"]
    blocks = []
    for i in range(36):
        if i % 2 == 0:
            k, v, _ = _cache(g, [2 * case["page"]], case["kv_heads"], 64, case["page"])
            table = (torch.arange(-(-n // case["page"]), device="cuda", dtype=torch.int32) % 2).view(1, -1)
        else:
            k, v, table = _cache(g, [n], case["kv_heads"], 64, case["page"])
        blocks.append((k, v, table, _normal(g, case["heads"]), _normal(g, 1, case["heads"], 64)))
    return blocks


def prepare(case, seed):
    kind = case["kind"]
    out_dtype = torch.float16 if case.get("out") == "f16" else torch.float32
    st = SimpleNamespace(case=case, ctx=_context())
    if kind == "step":
        st.out = torch.empty(36, case["heads"], 64, device="cuda")
        st.calls = []
        for i, (k, v, table, sinks, q) in enumerate(_step_inputs(case, seed)):
            begin = max(0, case["depth"] - case["window"]) if i % 2 == 0 else 0
            st.calls.append((_view(st.out[i]), _view(q), _view(k), _view(v), _view(table), _view(sinks), begin))
    elif kind == "decode":
        s = _decode_inputs(case, seed)
        st.out = torch.empty(case["batch"], case["heads"], case["dim"], device="cuda", dtype=out_dtype)
        st.begin, st.end = [b for b, _ in s.spans], [e for _, e in s.spans]
        st.stride = s.table.shape[1]
        st.o, st.q, st.k, st.v = _view(st.out), _view(s.q), _view(s.k), _view(s.v)
        st.table, st.sinks = _view(s.table), _view(s.sinks)
    elif kind == "prefill":
        s = _prefill_inputs(case, seed)
        st.out = torch.empty(case["tokens"], case["heads"], 64, device="cuda", dtype=out_dtype)
        st.o, st.q, st.k, st.v = _view(st.out), _view(s.q), _view(s.k), _view(s.v)
        st.table, st.sinks = _view(s.table), _view(s.sinks)
    elif kind == "block":
        s = _block_inputs(case, seed)
        st.h, st.k, st.v = s.h, s.k, s.v
        rope = RopeScaling.yarn(64, YARN["n_ctx_orig"], YARN["freq_base"], YARN["factor"])
        st.desc = AttnBlockDesc.make([QuantType[case["type"]]] * 4, [_view(w) for w in s.w], [_view(b) for b in s.bias],
                                     _view(s.sinks), _view(s.k), _view(s.v), _view(s.table), case["embd"],
                                     case["heads"], case["kv_heads"], 64, case["page"], case["window"], 0.125, 64,
                                     YARN["freq_base"], rope)
        st.vh, st.x, st.pos, st.pages, st.slots = (_view(t) for t in (s.h, s.x, s.pos, s.pages, s.slots))
    else:
        s = _matmul_inputs(case, seed)
        st.out = torch.empty(case["tokens"], case["rows"], device="cuda")
        st.o, st.w, st.x = _view(st.out), _view(s.w), _view(s.x)
        st.bias = _view(s.bias) if s.bias is not None else None
    torch.cuda.synchronize()  # the context's stream is its own
    return st


# ---- one pass --------------------------------------------------------------------------------------

def run(st):
    c, ctx = st.case, st.ctx
    kind = c["kind"]
    if kind == "step":
        for o, q, k, v, table, sinks, begin in st.calls:
            ctx.attn_decode_ext(o, q, k, v, table, sinks, c["heads"], c["kv_heads"], 64, begin, c["depth"], c["page"],
                                0.125, KvType.F16)
        return st.out
    if kind == "decode":
        kv, scale = (KvType.F16 if c["kv"] == "f16" else KvType.F32), 1.0 / math.sqrt(c["dim"])
        if c["batch"] == 1 and c["out"] == "f32":
            ctx.attn_decode_ext(st.o, st.q, st.k, st.v, st.table, st.sinks, c["heads"], c["kv_heads"], c["dim"],
                                st.begin[0], st.end[0], c["page"], scale, kv)
        else:
            ctx.attn_decode_batched(st.o, st.q, st.k, st.v, st.table, st.stride, st.begin, st.end, st.sinks,
                                    c["heads"], c["kv_heads"], c["dim"], c["page"], scale, kv,
                                    OUT_F16 if c["out"] == "f16" else OUT_F32)
        return st.out
    if kind == "prefill":
        ctx.attn_prefill(st.o, st.q, st.k, st.v, st.table, st.sinks, c["tokens"], c["pos0"], c["window"], c["heads"],
                         c["kv_heads"], 64, c["page"], 0.125, KvType.F16, OUT_F16 if c["out"] == "f16" else OUT_F32)
        return st.out
    if kind == "block":  # h is updated in place, as the residual stream is
        ctx.attn_block_chunk(st.desc, st.vh, st.x, c["tokens"], c["pos0"], st.pos, st.pages, st.slots)
        return {"h": st.h, "k": st.k, "v": st.v}
    ctx.matmul_q(QuantType[c["type"]], st.o, st.w, st.x, st.bias, c["tokens"], c["rows"], c["cols"])
    return st.out


# ---- what a pass cannot do without -----------------------------------------------------------------

def _pairs(tokens, pos0, window):
    """(query, key) pairs of a chunk of tokens."""
    return sum(min(p + 1, window) if window else p + 1 for p in range(pos0, pos0 + tokens))


def _keys(tokens, pos0, window):
    """Keys that some query of the chunk attends."""
    return pos0 + tokens - (max(0, pos0 + 1 - window) if window else 0)


def work(case):
    kind = case["kind"]
    if kind == "matmul":
        t, r, c = case["tokens"], case["rows"], case["cols"]
        return {"bytes": r * QuantType[case["type"]].row_bytes(c) + 4 * (t * c + t * r + r * case["bias"]),
                "flops": 2 * t * r * c}
    heads, kv_heads = case["heads"], case["kv_heads"]
    if kind == "step":
        n, w = case["depth"], min(case["depth"], case["window"])
        keys = 18 * (n + w)
        return {"bytes": keys * kv_heads * 64 * 4 + 36 * heads * (64 * 8 + 4), "flops": keys * heads * 64 * 4}
    if kind == "decode":
        keys, d = sum(e - b for b, e in _spans(case)), case["dim"]
        elem, o = (2 if case["kv"] == "f16" else 4), (2 if case["out"] == "f16" else 4)
        return {"bytes": keys * kv_heads * d * 2 * elem + case["batch"] * heads * d * (4 + o) + heads * 4,
                "flops": keys * heads * d * 4}
    t, pos0, window = case["tokens"], case["pos0"], case["window"]
    flops = _pairs(t, pos0, window) * heads * 64 * 4
    keys = _keys(t, pos0, window)
    if kind == "prefill":
        o = 2 if case["out"] == "f16" else 4
        return {"bytes": keys * kv_heads * 64 * 4 + t * heads * 64 * (2 + o) + heads * 4, "flops": flops}
    shapes = _block_shapes(case)
    qt = QuantType[case["type"]]
    nbytes = sum(r * (qt.row_bytes(c) + 4) for r, c in shapes) + t * case["embd"] * 12 + \
        keys * kv_heads * 64 * 4 + heads * 4  # the chunk's own K and V are written, the earlier ones read
    return {"bytes": nbytes, "flops": flops + sum(2 * t * r * c for r, c in shapes)}


# ---- how far another correct implementation may be -------------------------------------------------

def tolerance(case):
    """About four times what the outputs were measured to be off from exact()."""
    kind = case["kind"]
    if kind == "step" or kind == "decode" and case["out"] == "f32":
        return {"rel": 5e-6}  # 2e-7 to 1.1e-6: f32 sums over thousands of keys
    if kind == "decode":
        return {"rel": 1e-3}  # 2.1e-4: the f16 output's rounding
    if kind == "matmul":
        return {"rel": 2e-6}  # 2.4e-7: f32 sums
    if kind == "prefill":
        return {"rel": 1.2e-3}  # 2.9e-4: softmax weights in f16
    # a decode step in 32 bits, 2.2e-6; a chunk's queries and softmax weights in f16, 1.6e-4; single
    # cache entries may round the other way
    return {"rel": 2e-5, "max": 2e-3} if case["tokens"] == 1 else {"rel": 1e-3, "max": 2e-2}


def _attend(q, k, v, begin, end, sinks, scale):
    """Attention of q [tokens, heads, dim] over keys [begin_t, end_t) of k, v [keys, kv_heads, dim]
    (float64), with the sinks in the denominator."""
    out = torch.empty_like(q)
    group = q.shape[1] // k.shape[1]
    j = torch.arange(k.shape[0], device=q.device)
    masked = None
    if q.shape[0] > 1:
        masked = (j[None, :] < begin[:, None]) | (j[None, :] >= end[:, None])
    for h in range(q.shape[1]):
        kh, vh = k[:, h // group].contiguous(), v[:, h // group].contiguous()
        s = (q[:, h].contiguous() @ kh.t().contiguous()) * scale
        if masked is not None:
            s.masked_fill_(masked, -math.inf)
        m = torch.maximum(s.amax(-1, keepdim=True), sinks[h])
        p = torch.exp(s - m)
        out[:, h] = (p @ vh) / (p.sum(-1, keepdim=True) + torch.exp(sinks[h] - m))
    return out


def _gather(pool, table, begin, end):
    """Keys [begin, end) of one sequence, in float64."""
    j = torch.arange(begin, end, device=pool.device)
    rows = table[(j // pool.shape[1])].long() * pool.shape[1] + j % pool.shape[1]
    return pool.view(-1, *pool.shape[2:])[rows].double()


def _rope(x, pos):
    """NeoX rotation of [tokens, heads, 64] with YaRN scaling, float64."""
    s = RopeScaling.yarn(64, YARN["n_ctx_orig"], YARN["freq_base"], YARN["factor"])
    p = torch.arange(32, device=x.device, dtype=torch.float64)
    extra = pos.double()[:, None] * YARN["freq_base"] ** (-p / 32)
    mix = (1 - ((p - s.corr_lo) / max(0.001, s.corr_hi - s.corr_lo)).clamp(0, 1)) * s.ext_factor
    theta = extra * s.freq_scale * (1 - mix) + extra * mix
    size = s.attn_factor * (1 + 0.1 * math.log(1 / s.freq_scale))
    c, n = (torch.cos(theta) * size)[:, None], (torch.sin(theta) * size)[:, None]
    a, b = x[..., :32], x[..., 32:]
    return torch.cat([a * c - b * n, a * n + b * c], -1)


def exact(case, seed):
    kind = case["kind"]
    if kind == "matmul":
        s = _matmul_inputs(case, seed, dense=True)
        y = s.x.double() @ s.w.t().contiguous()
        return y if s.bias is None else y + s.bias.double()
    if kind == "step":
        out = torch.empty(36, case["heads"], 64, device="cuda", dtype=torch.float64)
        for i, (k, v, table, sinks, q) in enumerate(_step_inputs(case, seed)):
            begin = max(0, case["depth"] - case["window"]) if i % 2 == 0 else 0
            kk, vv = (_gather(x, table[0], begin, case["depth"]) for x in (k, v))
            out[i] = _attend(q.double(), kk, vv, None, None, sinks.double(), 0.125)[0]
        return out
    if kind == "decode":
        s = _decode_inputs(case, seed)
        out = torch.empty(s.q.shape, device="cuda", dtype=torch.float64)
        for b, (begin, end) in enumerate(s.spans):
            k, v = (_gather(x, s.table[b], begin, end) for x in (s.k, s.v))
            out[b] = _attend(s.q[b:b + 1].double(), k, v, None, None, s.sinks.double(), 1.0 / math.sqrt(case["dim"]))[0]
        return out
    t, pos0, window = case["tokens"], case["pos0"], case["window"]
    total = pos0 + t
    end = torch.arange(pos0 + 1, total + 1, device="cuda")
    first = max(0, pos0 + 1 - window) if window else 0  # the first key that any of the tokens attends
    begin = (end - window).clamp(min=0) if window else torch.zeros_like(end)
    if kind == "prefill":
        s = _prefill_inputs(case, seed)
        k, v = (_gather(x, s.table[0], first, total) for x in (s.k, s.v))
        return _attend(s.q.double(), k, v, begin - first, end - first, s.sinks.double(), 0.125)
    s = _block_inputs(case, seed, dense=True)
    x = s.x.double()
    q, k, v = ((x @ s.w[i].t().contiguous() + s.bias[i].double()).view(t, -1, 64) for i in range(3))
    rows = s.pages.long() * case["page"] + s.slots.long()
    # the cache holds f16
    s.k.view(-1, case["kv_heads"], 64)[rows] = _rope(k, s.pos).half()
    s.v.view(-1, case["kv_heads"], 64)[rows] = v.half()
    kk, vv = (_gather(p, s.table[0], first, total) for p in (s.k, s.v))
    a = _attend(_rope(q, s.pos), kk, vv, begin - first, end - first, s.sinks.double(), 0.125)
    h = s.h.double() + a.reshape(t, -1) @ s.w[3].t().contiguous() + s.bias[3].double()
    return {"h": h, "k": s.k.double(), "v": s.v.double()}

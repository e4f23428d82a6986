"""What a user of this library has it do, as cases that can be timed.

Each case is one pass through the entry points of `blitz_scale_amd.kernel` with the state a serving program keeps (KV
pool, page table, plan, workspaces) made beforehand.  Kinds:

  decode   one layer's decode-time attention: append of the new K/V rows and paged attention over the cache
  layer    the same between the norms and the gated activation of its layer
  model    the attention part of all layers of one decode step, with the page-table upload and the plan in front of it
  prefill  one layer's prompt attention: K/V written into their pages (K rotated), then ragged causal attention; with
           `hidden` also the norms, the activation and the residual of the layer; with `prefix` a chunk of new tokens
           attends to the K/V rows of its whole prompt
  ends     both ends of the layer loop: embedding, last-token gather, greedy sampling
  migrate  KV pages of a batch packed for the wire and unpacked into another pool

Sequence and prompt lengths belong to the case, values and page placement to the seed.
"""
import math

import numpy as np
import torch

from blitz_scale_amd import kernel as K
from blitz_scale_amd import workloads as wl
from blitz_scale_amd._lib import BZ_E4M3, BZ_LAYOUT_HND, BZ_LAYOUT_NHD, BZ_ROPE_FULL, BZ_ROPE_Q_ONLY

DTYPES = {"f16": torch.float16, "bf16": torch.bfloat16, "e4m3": torch.uint8}
LAYOUTS = {"hnd": BZ_LAYOUT_HND, "nhd": BZ_LAYOUT_NHD}
FLOAT_WORKSPACE, INT_WORKSPACE = 128 << 20, 8 << 20  # what the worker reserves per model
E4M3_SCALE = 5.5 / 448  # amax of a large normal sample over the largest e4m3 value


# ---- the cases -----------------------------------------------------------------------------------------------------
def _decode(name, batch, q_heads, kv_heads, lens, lo, hi, *, mean=0, head_dim=128, page=16, dtype="bf16", kv="", layout="hnd",
            raw=False, theta=5e5, kind="decode", **more):
    case = dict(kind=kind, batch=batch, q_heads=q_heads, kv_heads=kv_heads, head_dim=head_dim, page=page, dtype=dtype,
                kv=kv or dtype, layout=layout, raw=raw, theta=theta, lens=lens, lo=lo, hi=hi, mean=mean, **more)
    return dict(case, name=name) if name else case


def _prefill(name, batch, q_heads, kv_heads, lo, hi, *, prefix_lo=0, prefix_hi=0, page=16, dtype="bf16", layout="hnd", theta=5e5,
             hidden=0, inter=0):
    case = dict(kind="prefill", batch=batch, q_heads=q_heads, kv_heads=kv_heads, head_dim=128, page=page, dtype=dtype,
                layout=layout, theta=theta, lens="uniform", lo=lo, hi=hi, mean=0, prefix_lo=prefix_lo, prefix_hi=prefix_hi,
                hidden=hidden, inter=inter)
    return dict(case, name=name) if name else case


def listed():
    return [
        # a small batch's trip through both ends of the model: four sequences, one row each (launch-bound)
        dict(name="ends_b4", kind="ends", tokens=4, batch=4, hidden=4096, vocab=128256, dtype="bf16"),
        # a lightly loaded instance: every token of eight conversations goes through all layers of an 8B model
        _decode("model_8b_b8", 8, 32, 8, "uniform", 700, 1350, kind="model", layers=32),
        # decode layer of a 7B model without grouped heads, with its norm and activation
        _decode("layer_7b_b64", 64, 32, 32, "uniform", 512, 2048, dtype="f16", theta=1e4, kind="layer", hidden=4096, inter=11008),
        # the headline: a well-filled decode batch of an 8B model with a long-tailed mix of conversations
        _decode("decode_8b_b128", 128, 32, 8, "lognormal", 64, 8192, mean=1024),
        # a large batch of long contexts over an fp8 cache, 70B head counts
        _decode("decode_70b_e4m3_b256", 256, 64, 8, "const", 4096, 4096, kv="e4m3"),
        # two whole books in context on one GPU: the split over the chip has to come from the sequences' length
        _decode("decode_long_b2", 2, 64, 8, "uniform", 40001, 90001, page=64),
        # small heads (64): the general decode kernel, the reference's in-page order
        _decode("decode_d64_b96", 96, 32, 8, "uniform", 17, 2048, head_dim=64, dtype="f16", layout="nhd", theta=1e4),
        # a cache that holds K as projected, rotated inside every call (the reference's own convention)
        _decode("decode_raw_k_b48", 48, 32, 8, "uniform", 200, 2048, raw=True),
        # a full prompt batch of a 13B model: long prompts, no grouped heads
        _prefill("prefill_13b", 16, 40, 40, 128, 4096, dtype="f16", theta=1e4),
        # many short questions at once
        _prefill("prefill_short_b61", 61, 32, 8, 16, 400),
        # chunked prefill: the next few hundred tokens of three long prompts, one whole layer of an 8B model
        _prefill("prefill_chunk_b3", 3, 32, 8, 200, 700, prefix_lo=3000, prefix_hi=16000, hidden=4096, inter=14336),
        # five prompts' pages leave for another instance: 32 layers, 16-bit wire
        dict(name="migrate_8b", kind="migrate", prompts=5, lo=400, hi=1500, layers=32, kv_heads=8, head_dim=128, page=16,
             dtype="bf16", wire="bf16"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


_HEADS = [(32, 32), (32, 8), (64, 8), (40, 40), (40, 8), (16, 4), (4, 1)]


def draw(rng):
    biggest = max(_cost(c) for c in listed())
    while True:
        case = _draw(rng)
        if _cost(case) <= biggest:
            return case


def _draw(rng):
    kind = rng.choice(["decode", "decode", "decode", "layer", "model", "prefill", "prefill", "chunk", "ends", "migrate"])
    hq, hkv = rng.choice(_HEADS)
    page, layout = rng.choice([16, 16, 32, 64]), rng.choice(["hnd", "hnd", "nhd"])
    dtype = rng.choice(["f16", "bf16", "bf16"])
    theta = rng.choice([1e4, 5e5])
    if kind in ("decode", "layer"):
        batch = _log_int(rng, 1, 256)
        # tokens in all: from a sequence or two to 2 GiB of K and V
        most = max(batch * 64, min(batch * 90000, (2 << 30) // (2 * hkv * 128 * 2)))
        mean = _log_int(rng, 64, max(65, most // batch))
        lens = rng.choice(["uniform", "lognormal"])
        lo, hi = (max(1, mean // 4), 2 * mean) if lens == "uniform" else (17, 8 * mean)
        if kind == "layer":
            return _decode("", batch, hq, hkv, lens, lo, hi, mean=mean, page=page, dtype=dtype, layout=layout, theta=theta,
                           kind="layer", hidden=rng.choice([4096, 5120, 8192]), inter=rng.choice([11008, 13824, 14336]))
        flavour = rng.choice(["plain", "plain", "plain", "e4m3", "e4m3", "d64", "raw"])
        return _decode("", batch, hq, hkv, lens, lo, hi, mean=mean, page=page, dtype=dtype, layout=layout, theta=theta,
                       head_dim=64 if flavour == "d64" else 128, kv="e4m3" if flavour == "e4m3" else "", raw=flavour == "raw")
    if kind == "model":
        mean = _log_int(rng, 64, 4096)
        return _decode("", _log_int(rng, 1, 24), hq, hkv, "uniform", max(1, mean // 2), mean * 3 // 2, page=page, dtype=dtype,
                       layout=layout, theta=theta, kind="model", layers=32)
    if kind == "prefill":
        mean = _log_int(rng, 30, 6000)
        batch = _log_int(rng, 1, max(1, min(256, 32768 // mean)))
        return _prefill("", batch, hq, hkv, max(1, mean // 4), mean * 7 // 4, page=page, dtype=dtype, layout=layout, theta=theta)
    if kind == "chunk":
        mean, prefix = _log_int(rng, 60, 2000), _log_int(rng, 500, 24000)
        norms = rng.random() < 0.5
        return _prefill("", _log_int(rng, 1, 6), hq, hkv, mean // 2, mean * 3 // 2, prefix_lo=prefix // 2, prefix_hi=prefix * 3 // 2,
                        page=page, dtype=dtype, layout=layout, theta=theta, hidden=rng.choice([4096, 5120, 8192]) if norms else 0,
                        inter=14336 if norms else 0)
    if kind == "ends":
        batch = _log_int(rng, 1, 256)
        return dict(kind="ends", tokens=max(batch, _log_int(rng, 1, 8192)), batch=batch, hidden=rng.choice([4096, 5120, 8192]),
                    vocab=rng.choice([32000, 128256]), dtype=dtype)
    mean = _log_int(rng, 60, 2000)
    return dict(kind="migrate", prompts=_log_int(rng, 1, 12), lo=mean // 2, hi=mean * 3 // 2, layers=rng.choice([16, 32]),
                kv_heads=hkv, head_dim=128, page=page, dtype=dtype, wire=rng.choice([dtype, "e4m3"]))


def _lengths(case, lo="lo", hi="hi", salt=0):
    """Sequence or prompt lengths of a case: the same for every seed."""
    rng = np.random.default_rng(wl.DEFAULT_SEED + salt)
    n = case["prompts"] if case["kind"] == "migrate" else case["batch"]
    if case.get("lens") == "lognormal":
        return wl.lognormal_ctx(rng, n, case["mean"], 1.0, case[lo], case[hi])
    return rng.integers(case[lo], case[hi] + 1, size=n).astype(np.int64)


# ---- the work a case cannot do without ---------------------------------------------------------------------------------
def work(case):
    es = 1 if case.get("kv") == "e4m3" else 2
    if case["kind"] == "ends":
        rows, b, h, v = case["tokens"], case["batch"], case["hidden"], case["vocab"]
        return {"bytes": 4 * rows * h + 4 * rows + 4 * b * h + 4 * (b + 1) + 2 * b * v + 4 * b, "flops": b * v}
    D, Hkv, P = case["head_dim"], case["kv_heads"], case["page"]
    lens = _lengths(case)
    if case["kind"] == "migrate":
        payload = int(((lens + P - 1) // P).sum()) * case["layers"] * 2 * Hkv * P * D * 2
        on_wire = payload // 2 if case["wire"] == "e4m3" else payload
        return {"bytes": 2 * (payload + on_wire), "flops": 0}
    Hq, B = case["q_heads"], case["batch"]
    if case["kind"] == "prefill":
        prefix = _prefixes(case)
        q, kv = int(lens.sum()), int((lens + prefix).sum())
        seen = int((lens * prefix + lens * (lens + 1) // 2).sum())  # (q row, K row) couples under the causal mask
        nbytes = 2 * D * (2 * q * Hq + 2 * kv * Hkv)
        if not case["prefix_hi"]:
            nbytes += 2 * D * Hkv * 3 * kv  # the rows in their pages, and the rotated K rows
        if case["hidden"]:
            nbytes += _layer_bytes(q, case["hidden"], case["inter"]) + 3 * q * case["hidden"] * 2
        return {"bytes": nbytes, "flops": 4 * D * Hq * seen}
    nbytes = wl.decode_algorithmic_bytes(lens, Hq, Hkv, D, es, 2, P)
    flops = 4 * D * Hq * int(lens.sum())
    if case["kind"] == "layer":
        nbytes += _layer_bytes(B, case["hidden"], case["inter"])
    layers = case.get("layers", 1)
    return {"bytes": nbytes * layers, "flops": flops * layers}


def _layer_bytes(rows, hidden, inter):
    """rms_norm, add_rms_norm and silu_and_mul over `rows` tokens."""
    return 2 * rows * hidden * 2 + 2 * hidden + 4 * rows * hidden * 2 + 2 * hidden + 3 * rows * inter * 2


def _cost(case):
    w = work(case)
    return max(w["bytes"], w["flops"] / 50)


def tolerance(case):
    """Gathers, page moves and argmax are exact.  For the rest four times what the results differ by from the same
    computation in float64 (2-norm / largest difference over the rms): decode 2.1e-4 / 0.003 in f16 and 1.7e-3 / 0.024 in
    bf16, which is the rounding of the stored rows; prompts, whose probabilities are 16-bit operands as well, 3.6e-4 / 0.009
    and 2.4e-3 / 0.045.  One cached fp8 byte in a thousand may round the other way."""
    if case["kind"] in ("ends", "migrate"):
        return "exact"
    f16 = case["dtype"] == "f16"
    return {"rel": 1.5e-3 if f16 else 9e-3, "max": 0.04 if f16 else 0.15, "differ": 1e-3}


# ---- state and one pass ------------------------------------------------------------------------------------------------
def _prefixes(case):
    if not case["prefix_hi"]:
        return np.zeros(case["batch"], np.int64)
    return _lengths(case, "prefix_lo", "prefix_hi", salt=1)


def _randn(shape, dtype, gen):
    return torch.randn(shape, dtype=dtype, device="cuda", generator=gen)


def _pool(elements, kv, gen):
    if kv != "e4m3":
        return _randn(elements, DTYPES[kv], gen)
    pool = torch.empty(elements, dtype=torch.uint8, device="cuda")
    for part in pool.split(1 << 28):
        part.copy_((_randn(part.numel(), torch.float32, gen) / E4M3_SCALE).clamp_(-448, 448).to(torch.float8_e4m3fn).view(torch.uint8))
    return pool


def _page_table(case, lens, kv, layers, gen, seed):
    """A pool of `layers` planes and the table of sequences of these lengths at a random placement in it."""
    P, Hkv, D = case["page"], case["kv_heads"], case["head_dim"]
    pages = int(((lens + P - 1) // P).sum())
    max_pages = pages + pages // 4 + 1
    pool = _pool(layers * max_pages * 2 * Hkv * P * D, kv, gen)
    pt = K.PageTable(len(lens), P, Hkv, D, pool, layout=LAYOUTS[case.get("layout", "hnd")])
    pt.indices, pt.indptr, pt.last_page_len = wl.page_table_for(lens, P, max_pages, np.random.default_rng(seed))
    pt.upload()
    return pt, max_pages


def _workspaces():
    return (torch.empty(FLOAT_WORKSPACE, dtype=torch.uint8, device="cuda"), torch.empty(INT_WORKSPACE, dtype=torch.uint8, device="cuda"))


def _norm_state(rows, hidden, inter, dtype, gen):
    return dict(rows=rows, hidden=hidden, inter=inter, x=_randn((rows, hidden), dtype, gen), residual=_randn((rows, hidden), dtype, gen),
                w_in=1 + 0.02 * _randn((hidden,), dtype, gen), w_post=1 + 0.02 * _randn((hidden,), dtype, gen),
                o_proj=_randn((rows, hidden), dtype, gen), gate_up=_randn((rows, 2 * inter), dtype, gen),
                act=torch.empty((rows, inter), dtype=dtype, device="cuda"))


def prepare(case, seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    s = dict(case=case)
    if case["kind"] == "ends":
        rng = np.random.default_rng(seed)
        n, b, h, v = case["tokens"], case["batch"], case["hidden"], case["vocab"]
        dtype = DTYPES[case["dtype"]]
        s.update(weight=_randn((v, h), dtype, gen), logits=_randn((b, v), dtype, gen),
                 ids=torch.from_numpy(rng.integers(0, v, size=n).astype(np.int32)).cuda(),
                 indptr=torch.from_numpy(np.linspace(0, n, b + 1).astype(np.int32)).cuda(),
                 rows=torch.empty((n, h), dtype=dtype, device="cuda"), last=torch.empty((b, h), dtype=dtype, device="cuda"),
                 token=torch.empty(b, dtype=torch.int32, device="cuda"))
        return s
    lens = _lengths(case)
    if case["kind"] == "migrate":
        src, max_pages = _page_table(case, lens, case["dtype"], case["layers"], gen, seed)
        dst = K.PageTable(len(lens), case["page"], case["kv_heads"], case["head_dim"], torch.zeros_like(src.base))
        wire_dtype = BZ_E4M3 if case["wire"] == "e4m3" else None
        there = np.random.default_rng(seed + 1).permutation(max_pages)[: len(src.indices)].astype(np.int32)
        scale = torch.full((case["layers"], case["kv_heads"]), E4M3_SCALE, dtype=torch.float32, device="cuda")
        s.update(src=src, dst=dst, max_pages=max_pages, src_ids=src.indices_d, dst_ids=torch.from_numpy(there).cuda(), wire_dtype=wire_dtype,
                 wire=torch.empty(K.kv_wire_bytes(src, len(src.indices), case["layers"], wire_dtype), dtype=torch.uint8, device="cuda"),
                 scale=scale if wire_dtype is not None else None)
        return s
    B, Hq, Hkv, D, P = (case[k] for k in ("batch", "q_heads", "kv_heads", "head_dim", "page"))
    dtype = DTYPES[case["dtype"]]
    s["float_ws"], s["int_ws"] = _workspaces()
    sizes = (s["float_ws"], FLOAT_WORKSPACE, s["int_ws"], INT_WORKSPACE)
    if case["kind"] == "prefill":
        prefix = _prefixes(case)
        qo = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
        kv = np.concatenate([[0], np.cumsum(lens + prefix)]).astype(np.int32)
        s["handler"] = K.BatchPrefillRaggedHandler()
        s["handler"].plan(*sizes, qo, kv, B, Hq, Hkv, D, P)
        if not case["prefix_hi"]:
            s["table"], _ = _page_table(case, lens, case["dtype"], 1, gen, seed)
        s.update(q=_randn((int(qo[-1]), Hq, D), dtype, gen), k=_randn((int(kv[-1]), Hkv, D), dtype, gen),
                 v=_randn((int(kv[-1]), Hkv, D), dtype, gen), out=torch.empty((int(qo[-1]), Hq, D), dtype=dtype, device="cuda"),
                 qo=torch.from_numpy(qo).cuda(), kv=torch.from_numpy(kv).cuda())
        if case["hidden"]:
            s["norm"] = _norm_state(int(qo[-1]), case["hidden"], case["inter"], dtype, gen)
        return s
    layers = case.get("layers", 1)
    s["table"], s["max_pages"] = _page_table(case, lens, case["kv"], layers, gen, seed)
    s["handler"] = K.BlitzBatchDecodeHandler()
    s["plan"] = lambda: s["handler"].plan(*sizes, s["table"].indptr, s["table"].last_page_len, B, Hq, Hkv, D, P)
    s["plan"]()
    s.update(q=_randn((layers, B, Hq, D), dtype, gen), k=_randn((layers, B, Hkv, D), dtype, gen),
             v=_randn((layers, B, Hkv, D), dtype, gen), out=torch.empty((layers, B, Hq, D), dtype=dtype, device="cuda"))
    scale = torch.full((Hkv,), E4M3_SCALE, dtype=torch.float32, device="cuda") if case["kv"] == "e4m3" else None
    s["scales"] = dict(k_scale=scale, v_scale=scale)
    # (the rows of each layer as the worker has them: buffers of their own)
    s["rows"] = [tuple(t[l] for t in (s["q"], s["k"], s["v"], s["out"])) for l in range(layers)]
    if case["kind"] == "layer":
        s["norm"] = _norm_state(B, case["hidden"], case["inter"], dtype, gen)
    return s


def _norms_before(n):
    K.rms_norm(n["residual"], n["w_in"], n["x"], n["rows"], n["hidden"])


def _norms_after(n):
    K.add_rms_norm(n["o_proj"], n["residual"], n["w_post"], n["rows"], n["hidden"])
    K.silu_and_mul(n["gate_up"], n["act"], n["rows"], n["inter"])


def _norm_outputs(n):
    return [n["x"], n["o_proj"], n["residual"], n["act"]]


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "ends":
        K.embedding(s["rows"], s["ids"], s["weight"], case["tokens"], case["hidden"])
        K.gather_last_token(s["last"], s["rows"], s["indptr"], case["tokens"], case["batch"], case["hidden"])
        K.batch_find_max(s["token"], s["logits"], case["batch"], case["vocab"])
        return [s["rows"], s["last"], s["token"]]
    if kind == "migrate":
        scales = dict(wire_dtype=s["wire_dtype"], k_scale=s["scale"], v_scale=s["scale"])
        K.pack_kv_pages(s["src"], s["max_pages"], s["src_ids"], 0, case["layers"], s["wire"], **scales)
        K.unpack_kv_pages(s["dst"], s["max_pages"], s["dst_ids"], 0, case["layers"], s["wire"], **scales)
        return [s["wire"], s["dst"].base]
    Hq, Hkv, D, theta = case["q_heads"], case["kv_heads"], case["head_dim"], case["theta"]
    norm = s.get("norm")
    if kind == "prefill":
        if norm:
            _norms_before(norm)
        if not case["prefix_hi"]:
            K.store_prefill_kv_cache(s["table"], s["k"], s["v"], s["qo"], rope=2, rope_theta=theta)
        K.batch_prefill_attention(s["handler"], s["q"], s["qo"], s["k"], s["v"], s["kv"], s["out"], case["batch"], Hq, Hkv, D,
                                  rope_mode=BZ_ROPE_Q_ONLY, rope_theta=theta)
        if norm:
            _norms_after(norm)
            K.add_residual(norm["o_proj"], norm["residual"], norm["rows"], norm["hidden"])
            return [s["out"], *_norm_outputs(norm)]
        return [s["out"], s["k"], s["table"].base]
    table, handler = s["table"], s["handler"]
    if kind == "model":
        table.upload()
        s["plan"]()
        for layer, (q, k, v, out) in enumerate(s["rows"]):
            table.set_layer(layer, s["max_pages"])
            K.decode_step(handler, q, k, v, table, out, Hq, rope_theta=theta)
        return [s["out"], table.base]
    q, k, v, out = s["rows"][0]
    if norm:
        _norms_before(norm)
    if case["raw"]:
        K.append_decode_kv_cache(table, k, v)
        K.batch_decode_attention(handler, q, table, out, Hq, rope_mode=BZ_ROPE_FULL, rope_theta=theta)
    else:
        K.decode_step(handler, q, k, v, table, out, Hq, rope_theta=theta, **s["scales"])
    if norm:
        _norms_after(norm)
        return [s["out"], table.base, *_norm_outputs(norm)]
    return [s["out"], table.base]

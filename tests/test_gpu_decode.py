"""GPU parity: paged batch decode through the C ABI against the CPU checker on identical bits.

Tolerances (stated by the task): max-abs <= 2e-3 for f16/bf16 results, <= 3e-2 with an e4m3 KV pool.
The fp32-output instantiation is held to 2e-5 to show the arithmetic itself agrees; where the result
is stored in bf16 the bound is widened to half a bf16 step for |o| >= 0.5 (the storage grid is then
coarser than 2e-3).
"""
import os

import numpy as np
import pytest
import torch

import oracle
from blitz_scale_amd import kernel as K
from blitz_scale_amd import workloads as wl
from blitz_scale_amd._lib import (BZ_BF16, BZ_E4M3, BZ_F16, BZ_F32, BZ_LAYOUT_HND, BZ_LAYOUT_NHD, BZ_ROPE_FULL,
                                  BZ_ROPE_NONE, BZ_ROPE_Q_ONLY)

from _gpu import DeviceDecode, to_dev, to_host_bits
from _util import DecodeProblem, dense_attention_f64, rope_f64, ulp_tol

pytestmark = pytest.mark.gpu


def check(p, split_tokens=0, rope_mode=BZ_ROPE_NONE, theta=1e4, f32_tol=2e-5, parallel=False):
    """Both kernels are held to the same bar: the MFMA kernel where it applies (library default) and
    the general kernel (BZ_DECODE_PATH=general at plan time)."""
    ref, ref_lse = oracle.batch_decode(p.q, p.dtype, p.oracle_kv(), p.Hq, rope_mode=rope_mode, rope_theta=theta,
                                       k_scale=p.k_scale, v_scale=p.v_scale, want_lse=True, parallel=parallel)
    os.environ["BZ_DECODE_PATH"] = "general"
    try:
        _check_one(p, split_tokens, rope_mode, theta, f32_tol, ref, ref_lse)
    finally:
        del os.environ["BZ_DECODE_PATH"]
    return _check_one(p, split_tokens, rope_mode, theta, f32_tol, ref, ref_lse)


def _check_one(p, split_tokens, rope_mode, theta, f32_tol, ref, ref_lse):
    dev = DeviceDecode(p)
    info = dev.plan(split_tokens)
    got32, lse = dev.decode(BZ_F32, rope_mode, theta, want_lse=True)
    err32 = np.abs(got32 - ref).max()
    assert err32 <= f32_tol, f"fp32-out max abs err {err32}"
    live = p.ctx > 0
    assert np.abs(lse[live] - ref_lse[live]).max() < 1e-3
    got = dev.decode(None, rope_mode, theta)
    base = 3e-2 if p.kv_dtype == BZ_E4M3 else 2e-3
    assert (np.abs(got - ref) <= ulp_tol(ref, p.dtype, base)).all(), f"max abs err {np.abs(got - ref).max()}"
    return info, got32, ref


def test_c1_plumbing_config():
    """benchmark configuration 1: fp16, batch 4, 4/4 heads, D 64, P 16, ctx {17,64,130,255}, 64-page pool, no RoPE."""
    cfg = wl.CONFIGS["C1"]
    p = DecodeProblem(wl.DEFAULT_SEED, cfg["ctx"], cfg["Hq"], cfg["Hkv"], cfg["D"], cfg["P"], cfg["dtype"],
                      pool_pages=cfg["pool_pages"])
    assert int(p.indptr[-1]) == 31
    info, got, ref = check(p)
    assert np.abs(got - ref).max() < 2e-5


@pytest.mark.parametrize("layout", [BZ_LAYOUT_NHD, BZ_LAYOUT_HND])
@pytest.mark.parametrize("dtype", [BZ_F16, BZ_BF16])
@pytest.mark.parametrize("Hq,Hkv,D,P", [(4, 4, 64, 16), (8, 4, 128, 16), (32, 8, 128, 16), (16, 2, 128, 64),
                                         (8, 8, 128, 1), (8, 1, 64, 8)])
def test_shapes_layouts_dtypes(layout, dtype, Hq, Hkv, D, P):
    ctx = [1, 2, 15, 16, 17, 63, 64, 65, 255, 300, 1000]
    check(DecodeProblem(100 + Hq + D + P, ctx, Hq, Hkv, D, P, dtype, layout=layout))


def test_empty_and_single_token_sequences():
    p = DecodeProblem(7, [0, 1, 0, 33, 1], 8, 2, 128, 16, BZ_F16)
    info, got, ref = check(p)
    assert np.array_equal(got[0], np.zeros_like(got[0])) and np.array_equal(got[2], np.zeros_like(got[2]))
    K, V = p.gather_kv(1)
    assert np.array_equal(got[1], np.repeat(V[0], 4, axis=0))  # ctx = 1: o == v0 exactly


@pytest.mark.parametrize("split_tokens", [16, 64, 256, 2048])
def test_split_k_equals_unsplit(split_tokens):
    p = DecodeProblem(8, [5000, 17, 2049, 640, 8192], 32, 8, 128, 16, BZ_BF16)
    dev = DeviceDecode(p)
    dev.plan(0xFFFFFFFF)
    whole = dev.decode(BZ_F32)
    info = dev.plan(split_tokens)
    assert info["split_seqs"] >= 3
    split = dev.decode(BZ_F32)
    assert np.abs(split - whole).max() < 2e-6
    ref = oracle.batch_decode(p.q, p.dtype, p.oracle_kv(), p.Hq, parallel=True)
    assert np.abs(split - ref).max() < 2e-5


def test_contexts_above_2048_are_split_by_default():
    p = DecodeProblem(9, [2048, 2049, 100], 8, 2, 128, 16, BZ_F16)
    dev = DeviceDecode(p)
    info = dev.plan(0)
    assert info["split_seqs"] >= 1


@pytest.mark.parametrize("rope_mode", [BZ_ROPE_Q_ONLY, BZ_ROPE_FULL])
@pytest.mark.parametrize("theta", [1e4, 5e5])
def test_rope_modes(rope_mode, theta):
    p = DecodeProblem(10, [3, 77, 500, 2100], 8, 2, 128, 16, BZ_F16)
    check(p, rope_mode=rope_mode, theta=theta, f32_tol=1e-4)


def test_page_permutation_is_bit_invariant():
    p = DecodeProblem(11, [700, 64, 3000], 32, 8, 128, 16, BZ_BF16)
    dev = DeviceDecode(p)
    dev.plan()
    a = dev.decode(BZ_F32)
    perm = np.random.default_rng(1).permutation(p.pool_pages)
    pool2 = np.empty_like(p.pool).reshape(p.pool_pages, -1)
    pool2[perm] = p.pool.reshape(p.pool_pages, -1)
    p.pool, p.indices = pool2.reshape(-1), perm[p.indices].astype(np.int32)
    dev2 = DeviceDecode(p)
    dev2.plan()
    assert np.array_equal(dev2.decode(BZ_F32), a)


def test_e4m3_kv_pool():
    """Q bf16, K/V e4m3 with per-kv-head fp32 scales amax/448, dequantised inside the kernel."""
    p = DecodeProblem(12, [100, 1024, 4096, 31], 64, 8, 128, 16, BZ_BF16, kv_dtype=BZ_E4M3)
    check(p, f32_tol=2e-5, parallel=True)


@pytest.mark.parametrize("batch", [12, 24])
@pytest.mark.parametrize("dtype,kv_dtype,rope_mode", [(BZ_F16, None, BZ_ROPE_NONE), (BZ_BF16, None, BZ_ROPE_Q_ONLY),
                                                       (BZ_F16, BZ_E4M3, BZ_ROPE_NONE), (BZ_BF16, BZ_E4M3, BZ_ROPE_Q_ONLY)])
def test_both_sides_of_the_streaming_threshold(batch, dtype, kv_dtype, rope_mode):
    """The planner picks the kernel instantiation whose K/V loads carry the non-temporal hint once every
    wave slot has two tiles or more.  12 and 24 sequences of 512 tokens on 8 kv heads are 1 536 and 3 072
    tiles, i.e. one tile per slot (plain loads) and two (hinted loads) on 256 compute units."""
    ctx = [512] * (batch - 1) + [497]
    p = DecodeProblem(40 + batch, ctx, 16, 8, 128, 16, dtype, kv_dtype=kv_dtype)
    check(p, rope_mode=rope_mode, theta=5e5, f32_tol=1e-4, parallel=True)


def test_c2_shape_reduced_batch():
    """Llama-2-7B MHA decode shape (32/32 heads, D 128, fp16, ctx U[512,2048]) at batch 8, q rotated in-kernel."""
    rng = np.random.default_rng(wl.DEFAULT_SEED)
    ctx = rng.integers(512, 2049, size=8)
    check(DecodeProblem(13, ctx, 32, 32, 128, 16, BZ_F16), rope_mode=BZ_ROPE_Q_ONLY, theta=1e4, f32_tol=1e-4,
          parallel=True)


def test_c3_headline_config_full_size():
    """Llama-3-8B GQA decode at full size: bf16, batch 128, 32/8 heads, log-normal contexts, 2x pool."""
    cfg = wl.CONFIGS["C3"]
    rng = np.random.default_rng(wl.DEFAULT_SEED)
    ctx = wl.ctx_lens_for(cfg, rng)
    p = DecodeProblem(wl.DEFAULT_SEED, ctx, cfg["Hq"], cfg["Hkv"], cfg["D"], cfg["P"], cfg["dtype"], oversub=2.0)
    info, got, ref = check(p, split_tokens=2048, rope_mode=BZ_ROPE_Q_ONLY, theta=5e5, f32_tol=1e-4, parallel=True)
    assert info["split_seqs"] == int((ctx > 2048).sum()) or info["split_seqs"] >= int((ctx > 2048).sum())


def test_c5_shape_reduced_batch():
    """Llama-3-70B GQA decode, e4m3 KV, uniform context 4096, at batch 8."""
    p = DecodeProblem(14, [4096] * 8, 64, 8, 128, 16, BZ_BF16, kv_dtype=BZ_E4M3)
    check(p, parallel=True)


def test_error_codes():
    from blitz_scale_amd import kernel as K
    p = DecodeProblem(15, [5], 4, 2, 64, 16, BZ_F16)
    dev = DeviceDecode(p)
    out = torch.empty((1, 4, 64), dtype=torch.float16, device="cuda")
    with pytest.raises(K.BzError, match="batchDecodeAttention error"):
        K.batch_decode_attention(dev.handler, dev.q, dev.pt, out, 4)  # plan() not called
    dev.plan()
    with pytest.raises(K.BzError):
        K.batch_decode_attention(dev.handler, dev.q, dev.pt, out, 8)  # head count differs from the plan
    with pytest.raises(K.BzError, match="Handler plan"):
        dev.handler.plan(dev.float_ws, dev.float_ws.numel(), dev.int_ws, 16, p.indptr, p.last_page_len, p.B, p.Hq,
                         p.Hkv, p.D, p.P)  # int workspace too small


def test_plan_fits_the_workspace_it_reports():
    """bz_decode_plan_workspace names the bytes plan() needs for the matrix-core kernel and the one-call step:
    buffers of exactly that size are enough; without room for the last section (the unit list of the one-call
    step) the matrix-core schedule is still taken; one more section less and the plan falls back to the general
    kernel (same results every time)."""
    from blitz_scale_amd import kernel as K
    p = DecodeProblem(77, [3000, 40, 900, 2100, 64, 1], 32, 8, 128, 16, BZ_BF16)
    ref = oracle.batch_decode(p.q, p.dtype, p.oracle_kv(), p.Hq)
    h = K.BlitzBatchDecodeHandler()
    fb, ib = h.workspace(p.indptr, p.last_page_len, p.B, p.Hq, p.Hkv, p.D, p.P, split_tokens=1024)
    slots = len(h.host_schedule(4)) - 1
    unit_bytes = (len(h.host_schedule(7)) * 32 + 255) // 256 * 256
    assert fb > 0 and ib > 0 and slots > 0 and unit_bytes > 0
    infos = []
    for int_bytes in (ib, ib - 256, ib - unit_bytes - 256):
        dev = DeviceDecode(p, float_ws_bytes=fb, int_ws_bytes=int_bytes)
        info = dev.plan(1024)
        got = dev.decode(None, BZ_ROPE_NONE)
        assert (np.abs(got - ref) <= ulp_tol(ref, p.dtype)).all()
        infos.append(info)
    assert infos[0]["workgroups"] == slots          # the matrix-core schedule was taken
    assert infos[1]["workgroups"] == slots          # still: only the one-call step's unit list is missing
    assert infos[2]["workgroups"] != slots          # no room for it: page-aligned segments x kv heads


@pytest.mark.parametrize("ctx,expect_min_partials", [
    ([20000], 65),            # one long sequence over the whole chip: hundreds of partials per kv head
    ([1024] * 8, 17),         # small batch: every (sequence, kv head) cut into ~32 one-tile pieces
    ([3000, 5], 17),
])
def test_splits_with_many_partials(ctx, expect_min_partials):
    """The split-K combine takes its sliced form (4 or 8 slices merged through LDS) when a (sequence, kv
    head) has more than 16 partials; results as for any other decode."""
    from blitz_scale_amd import kernel as K
    p = DecodeProblem(4242, ctx, 32, 8, 128, 16, BZ_BF16)
    ref, ref_lse = oracle.batch_decode(p.q, p.dtype, p.oracle_kv(), p.Hq, want_lse=True, parallel=True)
    dev = DeviceDecode(p)
    dev.plan(2048)
    counts = dev.handler.host_schedule(6)[:, 3]
    assert counts.max() >= expect_min_partials
    got32, lse = dev.decode(BZ_F32, BZ_ROPE_NONE, want_lse=True)
    assert np.abs(got32 - ref).max() <= 2e-5
    assert np.abs(lse - ref_lse).max() < 1e-3
    got = dev.decode(None, BZ_ROPE_NONE)
    assert (np.abs(got - ref) <= ulp_tol(ref, p.dtype)).all()


@pytest.mark.parametrize("Hq,Hkv,kv_dtype", [(32, 1, None), (48, 2, None), (128, 2, None), (64, 2, BZ_E4M3)])
def test_more_than_sixteen_q_heads_per_kv_head(Hq, Hkv, kv_dtype):
    """Groups of 24, 32 and 64 q heads run on the matrix-core kernel as equal parts of at most 16 (each part
    reads its kv head's K/V; with an e4m3 pool the scales are those of the kv head, not of the part)."""
    p = DecodeProblem(515, [70, 1500, 16, 333, 2600], Hq, Hkv, 128, 16, BZ_BF16, kv_dtype=kv_dtype)
    ref = oracle.batch_decode(p.q, p.dtype, p.oracle_kv(), Hq, k_scale=p.k_scale, v_scale=p.v_scale, parallel=True)
    dev = DeviceDecode(p)
    info = dev.plan(1024)
    G = Hq // Hkv
    parts = next(q for q in range((G + 15) // 16, G + 1) if G % q == 0)
    pieces = dev.handler.host_schedule(5)
    assert len(pieces) > 0 and pieces[:, 1].max() == Hkv * parts - 1   # the matrix-core schedule was built
    got = dev.decode(None, BZ_ROPE_NONE)
    base = 3e-2 if kv_dtype == BZ_E4M3 else 2e-3
    assert (np.abs(got - ref) <= ulp_tol(ref, p.dtype, base)).all(), float(np.abs(got - ref).max())
    if kv_dtype is None:
        got32 = dev.decode(BZ_F32, BZ_ROPE_NONE)
        assert np.abs(got32 - ref).max() <= 2e-5


@pytest.mark.parametrize("case", ["short_pieces", "chunk_crossing"])
@pytest.mark.parametrize("rope_mode", [BZ_ROPE_NONE, BZ_ROPE_Q_ONLY])
def test_e4m3_pool_with_several_tiles_per_wave_slot(case, rope_mode):
    """The one-byte-pool kernel keeps two tiles in flight per wave (two register sets taking turns).  Regimes of
    that pipeline on 256 compute units (2 048 wave slots):
      short_pieces    700 sequences of 1..200 tokens on 4 kv heads: ~4 or 5 tiles per slot (odd and even counts),
                      pieces of one to seven tiles, so consecutive tiles open new pieces and the q rows of a
                      piece are fetched one tile ahead several times in a row;
      chunk_crossing  150 sequences of 100..3 000 tokens on 8 kv heads: ~29 tiles per slot, i.e. the tile
                      descriptions come in more than one batch of 16 and ragged last tiles sit anywhere."""
    rng = np.random.default_rng(77 if case == "short_pieces" else 78)
    if case == "short_pieces":
        ctx, Hq, Hkv = rng.integers(1, 201, size=700).tolist(), 16, 4
    else:
        ctx, Hq, Hkv = rng.integers(100, 3001, size=150).tolist(), 32, 8
    p = DecodeProblem(500 + len(ctx), ctx, Hq, Hkv, 128, 16, BZ_BF16, kv_dtype=BZ_E4M3)
    ref = oracle.batch_decode(p.q, p.dtype, p.oracle_kv(), p.Hq, rope_mode=rope_mode, rope_theta=5e5, k_scale=p.k_scale,
                              v_scale=p.v_scale, parallel=True)
    dev = DeviceDecode(p)
    info = dev.plan(0)
    tiles = sum((c + 31) // 32 for c in ctx) * Hkv
    assert info["workgroups"] >= 2000 and tiles / info["workgroups"] > (3 if case == "short_pieces" else 20)
    got32 = dev.decode(BZ_F32, rope_mode, 5e5)
    assert np.abs(got32 - ref).max() <= (2e-5 if rope_mode == BZ_ROPE_NONE else 1e-4)
    got = dev.decode(None, rope_mode, 5e5)
    assert (np.abs(got - ref) <= ulp_tol(ref, p.dtype, 3e-2)).all()


@pytest.mark.parametrize("Hq,Hkv,kv_dtype", [(8, 8, None), (16, 8, None), (64, 4, None), (8, 8, BZ_E4M3)])
def test_many_finished_pieces_per_wave_slot(Hq, Hkv, kv_dtype):
    """Thousands of sequences of one or two tiles: a wave slot finishes ten and more (sequence, kv head)s, whose
    normalised rows wait in LDS until the slot is done.  The space holds 8 pieces or 16 rows, so it is emptied in
    the middle of a slot: by the piece count with one or two q heads per kv head, by the row count with sixteen.
    Final rows (16-bit and fp32) and log-sum-exps are checked for every sequence."""
    rng = np.random.default_rng(81)
    B = 2600 if Hkv == 8 else 5200
    ctx = rng.integers(1, 41, size=B).tolist()
    p = DecodeProblem(700 + Hq, ctx, Hq, Hkv, 128, 16, BZ_BF16, kv_dtype=kv_dtype)
    ref, ref_lse = oracle.batch_decode(p.q, p.dtype, p.oracle_kv(), p.Hq, k_scale=p.k_scale, v_scale=p.v_scale, want_lse=True,
                                       parallel=True)
    dev = DeviceDecode(p, float_ws_bytes=128 << 20)
    info = dev.plan(0)
    assert info["segments"] >= 9 * info["workgroups"]  # pieces per wave slot
    got32, lse = dev.decode(BZ_F32, BZ_ROPE_NONE, 1e4, want_lse=True)
    assert np.abs(got32 - ref).max() <= (3e-2 if kv_dtype == BZ_E4M3 else 2e-5)
    assert np.abs(lse - ref_lse).max() < 1e-3
    got = dev.decode(None, BZ_ROPE_NONE, 1e4)
    assert (np.abs(got - ref) <= ulp_tol(ref, p.dtype, 3e-2 if kv_dtype == BZ_E4M3 else 2e-3)).all()


@pytest.mark.parametrize("dtype,kv_dtype", [(BZ_F16, None), (BZ_BF16, None), (BZ_BF16, BZ_E4M3)])
def test_logits_with_a_large_dynamic_range(dtype, kv_dtype):
    """q rows eight times the usual size: logits of +-40 base-2 units, rows that attend to one or two tokens, and
    split-K partials whose log-sum-exps differ by tens of units (two-call path with the combine kernel, and the
    one-call step with its finishing kernel)."""
    from test_gpu_decode_step import run_step
    p = DecodeProblem(60, [3000, 40, 700, 1, 5000, 129], 32, 8, 128, 16, dtype, kv_dtype=kv_dtype)
    p.q = wl.to_bits(wl.to_f32(p.q, dtype) * np.float32(8.0), dtype)
    check(p, split_tokens=512, f32_tol=2e-5, parallel=True)  # matrix-core kernel and general kernel
    run_step(p, split_tokens=512, rope=False)


@pytest.mark.parametrize("Hq,Hkv,D", [(8, 2, 128), (4, 4, 64), (16, 2, 128)])
def test_rope_full_with_and_without_the_angle_table(Hq, Hkv, D):
    """kRoPELlama on a raw-K cache takes the angles of the cached rows from a table in the plan's float workspace
    when there is room behind the partials (groups of one, two and four q heads per workgroup), and evaluates
    them on the fly otherwise (no room; groups of eight).  Same results either way, also after a call in another
    mode has used the workspace in between."""
    p = DecodeProblem(70 + Hq, [3, 77, 500, 2100, 64], Hq, Hkv, D, 16, BZ_F16)
    ref = oracle.batch_decode(p.q, p.dtype, p.oracle_kv(), p.Hq, rope_mode=BZ_ROPE_FULL, rope_theta=5e5, parallel=True)
    roomy = DeviceDecode(p)                       # 32 MiB: partials + 2100 positions x D/2 x 8 bytes fit
    roomy.plan(256)
    a = roomy.decode(BZ_F32, BZ_ROPE_FULL, 5e5)
    assert np.abs(a - ref).max() <= 1e-4
    roomy.decode(BZ_F32, BZ_ROPE_Q_ONLY, 5e5)     # matrix-core path where it applies: its partials overwrite the table
    b = roomy.decode(BZ_F32, BZ_ROPE_FULL, 5e5)   # rebuilt
    assert np.array_equal(a, b)
    c = roomy.decode(BZ_F32, BZ_ROPE_FULL, 1e4)   # another base: rebuilt as well
    ref2 = oracle.batch_decode(p.q, p.dtype, p.oracle_kv(), p.Hq, rope_mode=BZ_ROPE_FULL, rope_theta=1e4, parallel=True)
    assert np.abs(c - ref2).max() <= 1e-4
    need = K.BlitzBatchDecodeHandler().workspace(p.indptr, p.last_page_len, p.B, Hq, Hkv, D, 16, split_tokens=256)[0]
    tight = DeviceDecode(p, float_ws_bytes=max(int(need), 4096))  # room for the partials only
    tight.plan(256)
    d = tight.decode(BZ_F32, BZ_ROPE_FULL, 5e5)
    assert np.abs(d - ref).max() <= 1e-4 and np.abs(d - a).max() <= 2e-6


@pytest.mark.parametrize("dtype", [BZ_F16, BZ_BF16])
@pytest.mark.parametrize("Hq,Hkv,P,layout", [(4, 4, 16, BZ_LAYOUT_HND), (8, 2, 64, BZ_LAYOUT_NHD), (12, 2, 48, BZ_LAYOUT_NHD),
                                             (32, 1, 16, BZ_LAYOUT_HND)])
def test_heads_of_64_on_the_matrix_core_kernel(dtype, Hq, Hkv, P, layout):
    """16-bit pools with heads of 64: two tiles in flight, slots of one, two and an odd number of tiles, whole and split
    sequences, ends inside and at a tile; rows of 16 bits against the checker, as a call and as the one-call step (groups
    of 1, 4, 6 and, in two parts, 32).  Rows and log-sum-exps in fp32 are the general kernel's, bit for bit."""
    from test_gpu_decode_step import run_step
    ctx = [1, 31, 32, 33, 64, 65, 1000, 0, 2049, 4096 + 17]
    p = DecodeProblem(640 + Hq, ctx, Hq, Hkv, 64, P, dtype, layout=layout)
    dev = DeviceDecode(p)
    outs = {}
    for path in ("", "general"):
        if path:
            os.environ["BZ_DECODE_PATH"] = path
        try:
            dev.plan(1024)
        finally:
            os.environ.pop("BZ_DECODE_PATH", None)
        assert len(dev.handler.host_schedule(5)) > 0  # pieces: the schedule is there
        outs[path] = [dev.decode(BZ_F32, mode, 1e4, want_lse=True) for mode in (BZ_ROPE_NONE, BZ_ROPE_Q_ONLY)]
        outs[path + "16"] = [dev.decode(None, mode, 1e4) for mode in (BZ_ROPE_NONE, BZ_ROPE_Q_ONLY)]
        outs[path + "16 lse"] = [dev.decode(None, mode, 1e4, want_lse=True) for mode in (BZ_ROPE_NONE, BZ_ROPE_Q_ONLY)]
    live = p.ctx > 0
    for i, mode in enumerate((oracle.ROPE_NONE, oracle.ROPE_Q_ONLY)):
        ref, ref_lse = oracle.batch_decode(p.q, dtype, p.oracle_kv(), Hq, rope_mode=mode, rope_theta=1e4, want_lse=True)
        for got, lse in (outs[""][i], outs["general"][i]):
            assert np.abs(got - ref).max() <= 2e-5 and np.abs(lse[live] - ref_lse[live]).max() < 1e-3
            assert not got[~live].any()
        for a, b in ((outs[""][i], outs["general"][i]), (outs["16 lse"][i], outs["general16 lse"][i])):
            assert np.array_equal(a[0], b[0]) and np.array_equal(a[1][live], b[1][live])
        # (head + tail operands hold 16 bits in bf16: scores of up to 8 to 2^-17 of themselves, 6e-5 of a probability)
        for got in (outs["16"][i], outs["general16"][i]):
            assert (np.abs(got - ref) <= ulp_tol(ref, dtype, 0.0, before_rounding=6e-5)).all()
            assert not got[~live].any()
    for split in (0, 1024):
        dev2, _, _ = run_step(p, split_tokens=split, theta=1e4, expect_units=False, want_lse=False)
        assert dev2.form == "one_call"


def test_heads_of_64_keep_the_range_of_fp32_operands():
    """f16 with heads of 64.  q near the largest f16, which leaves the type's range when it is rotated; and 4 000 tokens
    in one piece whose probabilities lie 2^-26 below the largest one's and carry the whole result."""
    p = DecodeProblem(645, [1, 33, 300, 1000], 8, 2, 64, 16, BZ_F16, kv_std=2.0 ** -12)
    half = p.stride_page // 2
    rng = np.random.default_rng(645)
    p.pool.reshape(-1, 2, half)[:, 1] = wl.randn_bits(rng, (len(p.pool) // p.stride_page, half), BZ_F16)
    p.q = wl.to_bits(np.where(rng.random((p.B, p.Hq, p.D)) < 0.5, -6e4, 6e4).astype(np.float32), BZ_F16)
    ref = oracle.batch_decode(p.q, BZ_F16, p.oracle_kv(), p.Hq, rope_mode=oracle.ROPE_Q_ONLY, rope_theta=1e4)
    dev = DeviceDecode(p)
    dev.plan()
    got = dev.decode(None, BZ_ROPE_Q_ONLY, 1e4)
    # (scores of up to 80, rotated with angles good to 2^-23: 1e-4 of a probability)
    assert (np.abs(got - ref) <= ulp_tol(ref, BZ_F16, 0.0, before_rounding=1e-4)).all()

    p = DecodeProblem(646, [4000], 4, 2, 64, 16, BZ_F16, oversub=1.0)
    planes = p.pool.reshape(-1, 2, 2, 16, 64)  # [page][K | V][kv head][token][dim]
    planes[:, 0] = 0
    planes[:, 1] = wl.to_bits(np.ones(1, np.float32), BZ_F16)
    page, slot = p.indices[3], 5
    planes[page, 0, :, slot] = wl.to_bits(np.full(1, 26 * np.log(2) / 8, np.float32), BZ_F16)
    planes[page, 1, :, slot] = 0
    p.q = wl.to_bits(np.ones((1, 4, 64), np.float32), BZ_F16)
    ref = oracle.batch_decode(p.q, BZ_F16, p.oracle_kv(), p.Hq)
    assert 5e-5 < ref.min() and ref.max() < 7e-5
    dev = DeviceDecode(p)
    dev.plan(0xFFFFFFFF)
    assert np.abs(dev.decode() / ref - 1).max() < 2e-3  # (a step of the stored f16 there is 1e-3)


def test_heads_of_64_with_buffers_of_the_reported_size():
    p = DecodeProblem(647, [700, 64, 3000], 8, 2, 64, 16, BZ_BF16)
    fb, ib = K.BlitzBatchDecodeHandler().workspace(p.indptr, p.last_page_len, p.B, p.Hq, p.Hkv, p.D, p.P, split_tokens=256)[:2]
    dev = DeviceDecode(p, float_ws_bytes=int(fb), int_ws_bytes=int(ib))
    dev.plan(256)
    ref = oracle.batch_decode(p.q, p.dtype, p.oracle_kv(), p.Hq)
    assert np.abs(dev.decode(BZ_F32) - ref).max() <= 2e-5
    assert (np.abs(dev.decode() - ref) <= ulp_tol(ref, p.dtype)).all()


@pytest.mark.parametrize("D,P,Hq,Hkv", [(128, 16, 4, 4), (128, 2, 4, 2), (128, 4, 8, 2), (128, 3, 16, 2), (128, 64, 10, 2), (64, 8, 8, 1),
                                        (64, 4, 4, 1), (64, 16, 3, 3)])
@pytest.mark.parametrize("dtype", [BZ_F16, BZ_BF16])
def test_raw_k_cache_with_angles_from_the_table(dtype, D, P, Hq, Hkv):
    """BZ_ROPE_FULL in groups of 1, 2, 4, 5 and 8 heads over pages that a wave's rows of one pass share (and smaller ones,
    that they do not), sequences that end inside a pass, split and whole, from one token on."""
    p = DecodeProblem(660 + D + P, [1, 2, 3, 15, 16, 17, 63, 64, 65, 0, 500, 1031], Hq, Hkv, D, P, dtype)
    check(p, split_tokens=256, rope_mode=BZ_ROPE_FULL)


@pytest.mark.parametrize("kv_dtype", [BZ_BF16, BZ_E4M3])
@pytest.mark.parametrize("Hq,Hkv,D,P", [(2, 2, 64, 8), (4, 2, 64, 16), (8, 2, 64, 8), (16, 2, 64, 16), (2, 2, 128, 8), (8, 2, 128, 4),
                                         (16, 2, 128, 8), (4, 2, 128, 2)])
def test_general_kernel_with_page_ids_of_a_set_ahead(kv_dtype, Hq, Hkv, D, P):
    """Segments of one set of tokens (64 of heads of 128, 128 of heads of 64) and more, ends at and beside the sets, in
    groups that take their page ids with the rows, a set ahead, or either by the segment's length."""
    p = DecodeProblem(680 + Hq + D + P, [1, 63, 64, 65, 127, 128, 129, 0, 191, 193, 256, 257, 385], Hq, Hkv, D, P, BZ_BF16, kv_dtype=kv_dtype)
    check(p)


@pytest.mark.parametrize("dtype", [BZ_F16, BZ_BF16])
@pytest.mark.parametrize("Hq,Hkv,P,layout", [(1, 1, 16, BZ_LAYOUT_HND), (8, 2, 32, BZ_LAYOUT_NHD), (5, 1, 16, BZ_LAYOUT_HND),
                                             (12, 2, 48, BZ_LAYOUT_NHD), (32, 2, 64, BZ_LAYOUT_HND), (20, 1, 16, BZ_LAYOUT_NHD)])
@pytest.mark.parametrize("split_tokens", [0, 96, 0xFFFFFFFF])
def test_raw_k_rows_of_16_bits(dtype, Hq, Hkv, P, layout, split_tokens):
    """16-bit rows over a raw-K cache of heads of 128: sequences that end on either side of 16, 32 and 64 tokens, whole and in
    pieces, groups of 1 to 20, no sequence at all."""
    p = DecodeProblem(700 + Hq + P, [1, 15, 16, 17, 31, 32, 33, 0, 47, 48, 49, 95, 97, 700, 2100], Hq, Hkv, 128, P, dtype, layout=layout)
    dev = DeviceDecode(p)
    dev.plan(split_tokens)
    for theta in (1e4, 5e5):
        ref = oracle.batch_decode(p.q, dtype, p.oracle_kv(), Hq, rope_mode=BZ_ROPE_FULL, rope_theta=theta, parallel=True)
        got = dev.decode(None, BZ_ROPE_FULL, theta)
        assert (np.abs(got - ref) <= ulp_tol(ref, dtype)).all(), np.abs(got - ref).max()


@pytest.mark.parametrize("dtype", [BZ_F16, BZ_BF16])
def test_raw_k_rows_under_a_table_that_runs_ahead(dtype):
    """The table lists five tokens more than there are: q and every K row are rotated at their present positions."""
    ctx, ahead = [22, 43, 166, 1030], 5  # (the last page keeps a token without them)
    p = DecodeProblem(730, ctx, 8, 2, 128, 16, dtype)
    assert (p.last_page_len > ahead).all()
    dev = DeviceDecode(p)
    dev.plan(256)
    dev.pt.steps_ahead_d = torch.tensor([ahead], dtype=torch.int32, device="cuda")
    got = dev.decode(None, BZ_ROPE_FULL, 1e4)
    p.last_page_len = p.last_page_len - ahead
    ref = oracle.batch_decode(p.q, dtype, p.oracle_kv(), 8, rope_mode=BZ_ROPE_FULL, rope_theta=1e4, parallel=True)
    assert (np.abs(got - ref) <= ulp_tol(ref, dtype)).all(), np.abs(got - ref).max()


def raw_k_rows_f64(p, theta):
    """The rows of a raw-K call in float64, from the stored bits."""
    out = np.zeros((p.B, p.Hq, p.D))
    for b in range(p.B):
        L = int(p.ctx[b])
        k, v = p.gather_kv(b)
        k = rope_f64(k, np.arange(L)[:, None, None], theta)
        out[b] = dense_attention_f64(rope_f64(wl.to_f32(p.q[b], p.dtype), L - 1, theta), k, v, p.D ** -0.5)
    return out


def with_values_of_one(p, seed):
    """V of standard normal values beside whatever K holds."""
    half = p.stride_page // 2
    planes = p.pool.reshape(-1, 2, half)
    planes[:, 1] = wl.randn_bits(np.random.default_rng(seed), (len(planes), half), p.dtype)
    return p


# The rounding of the stored rows alone is 2.1e-4 (f16) and 1.66e-3 (bf16) of their 2-norm.
ROWS_2NORM = {BZ_F16: 2.4e-4, BZ_BF16: 1.9e-3}


@pytest.mark.parametrize("dtype", [BZ_F16, BZ_BF16])
@pytest.mark.parametrize("split_tokens", [0, 0xFFFFFFFF])
def test_raw_k_rows_are_as_good_as_their_rounding(dtype, split_tokens):
    """Scores of a standard deviation of 4, so that what K, q and the probabilities lose in front of the softmax shows in the rows."""
    p = DecodeProblem(731, [300, 700, 1025, 2047], 8, 2, 128, 16, dtype)
    p.q = wl.to_bits(4 * wl.to_f32(p.q, dtype), dtype)
    dev, ref = DeviceDecode(p), raw_k_rows_f64(p, 1e4)
    dev.plan(split_tokens)
    got = dev.decode(None, BZ_ROPE_FULL, 1e4)
    assert np.linalg.norm(got - ref) <= ROWS_2NORM[dtype] * np.linalg.norm(ref)


@pytest.mark.parametrize("dtype", [BZ_F16, BZ_BF16])
def test_raw_k_rows_of_a_long_sequence(dtype):
    """30 000 tokens, theta 5e5.  The frequency and position * frequency in fp32 are each off by up to half a unit in the last
    place: over the 64 pairs 1.2e-4 rad rms for a K row (mean over the positions) and 2.1e-4 for q, at the end.  Scores of 1 are
    off by as much, together 2.4e-4, and the rows by that beside their rounding."""
    p = DecodeProblem(732, [30000], 4, 2, 128, 16, dtype)
    dev, ref = DeviceDecode(p), raw_k_rows_f64(p, 5e5)
    dev.plan()
    got = dev.decode(None, BZ_ROPE_FULL, 5e5)
    assert np.linalg.norm(got - ref) <= np.hypot(ROWS_2NORM[dtype], 2.4e-4) * np.linalg.norm(ref)


def test_raw_k_rows_of_small_values_keep_their_bits():
    """K of 1e-5, all of it below f16's normal range: a rotated value in fp32 has its 24 bits there, an f16 operand and what it
    leaves behind would have seven.  q of +-6e4 makes scores of 0.6 of it (and leaves f16's range itself when it is rotated)."""
    p = with_values_of_one(DecodeProblem(733, [1, 33, 300, 1000], 8, 2, 128, 16, BZ_F16, kv_std=1e-5), 733)
    p.q = wl.to_bits(np.where(np.random.default_rng(7).random((p.B, p.Hq, p.D)) < 0.5, -6e4, 6e4).astype(np.float32), BZ_F16)
    dev, ref = DeviceDecode(p), raw_k_rows_f64(p, 1e4)
    dev.plan()
    got = dev.decode(None, BZ_ROPE_FULL, 1e4)
    assert np.linalg.norm(got - ref) <= ROWS_2NORM[BZ_F16] * np.linalg.norm(ref)


def test_raw_k_rows_in_f16_keep_the_range_of_fp32():
    """K rows whose two largest values meet in one pair rotate to as much as 92 600: q picks them out, and V differs from token to
    token, so that the weights show."""
    p = with_values_of_one(DecodeProblem(734, [4000], 1, 1, 128, 16, BZ_F16), 734)
    k = np.zeros((len(p.pool) // p.stride_page, 16, 128), np.float32)
    k[..., 0] = k[..., 64] = 65504.0  # pair 0 turns by a radian a token
    p.pool.reshape(-1, 2, 16, 128)[:, 0] = wl.to_bits(k, BZ_F16)
    q = np.zeros((1, 1, 128), np.float32)
    q[0, 0, 0], q[0, 0, 64] = 2e-4, 1e-4
    p.q = wl.to_bits(q, BZ_F16)
    dev, ref = DeviceDecode(p), raw_k_rows_f64(p, 1e4)
    dev.plan()
    got = dev.decode(None, BZ_ROPE_FULL, 1e4)
    # (128 values, whose rounding comes to a fifth more or less than many do)
    assert np.linalg.norm(got - ref) <= 1.2 * ROWS_2NORM[BZ_F16] * np.linalg.norm(ref)


def test_raw_k_rows_of_a_long_tail_of_small_probabilities():
    """4 000 tokens in one piece whose probabilities lie 2^-26 below the largest one's and carry the whole result."""
    p = DecodeProblem(735, [4000], 4, 2, 128, 16, BZ_F16, oversub=1.0)
    planes = p.pool.reshape(-1, 2, 2, 16, 128)  # [page][K | V][kv head][token][dim]
    planes[:, 0] = 0
    planes[:, 1] = wl.to_bits(np.ones(1, np.float32), BZ_F16)
    page, slot = p.indices[-1], (4000 - 1) % 16  # the newest token: q and K turned by the same angles
    planes[page, 0, :, slot] = wl.to_bits(np.full(1, 26 * np.log(2) / 128 ** 0.5, np.float32), BZ_F16)
    planes[page, 1, :, slot] = 0
    p.q = wl.to_bits(np.ones((1, 4, 128), np.float32), BZ_F16)
    ref = raw_k_rows_f64(p, 1e4)
    assert 5e-5 < ref.min() and ref.max() < 7e-5
    dev = DeviceDecode(p)
    dev.plan(0xFFFFFFFF)
    assert np.abs(dev.decode(None, BZ_ROPE_FULL, 1e4) / ref - 1).max() < 2e-3  # (a step of the stored f16 there is 1e-3)


@pytest.mark.parametrize("offset", [0, 16, 4])
def test_tables_reach_a_workspace_that_begins_anywhere(offset):
    """The schedule goes up by a kernel where the workspace begins on a vector, by a copy where it does not; planned twice, so that
    the second schedule meets the first one's staging buffer."""
    p = DecodeProblem(760, [700, 64, 3000, 17], 8, 2, 128, 16, BZ_F16)
    dev = DeviceDecode(p)
    dev.int_ws = torch.full((8 << 20,), 255, dtype=torch.uint8, device="cuda")[offset:]
    ref = oracle.batch_decode(p.q, p.dtype, p.oracle_kv(), p.Hq, parallel=True)
    for split_tokens in (256, 0):
        dev.plan(split_tokens)
        assert (np.abs(dev.decode() - ref) <= ulp_tol(ref, p.dtype)).all()


def test_tables_above_half_a_megabyte_take_the_copy_engine():
    """800 sequences of a tile, eight kv heads each: 0.9 MB of tables, then few again from the same handle, then many."""
    many, few = DecodeProblem(761, [20] * 800, 8, 8, 128, 16, BZ_F16), DecodeProblem(762, [90, 1, 700], 8, 8, 128, 16, BZ_F16)
    handler = None
    for p in (many, few, many):
        dev = DeviceDecode(p)
        dev.handler = handler = handler or dev.handler
        dev.plan(0)
        ref = oracle.batch_decode(p.q, p.dtype, p.oracle_kv(), p.Hq, parallel=True)
        got = dev.decode()
        assert (np.abs(got - ref) <= ulp_tol(ref, p.dtype)).all()

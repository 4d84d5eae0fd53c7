"""Prefill attention on the matrix cores (gh_attention_prefill with several rows, every GQA group)
against the oracle, and against the reference's own prefill-attention test vectors.

Bars:
  * oracle (attention/mod.rs:582-725 restated): |got - want| <= 1e-3·|want| + 1e-5 — outputs
    are convex combinations of V rows; P·V runs with FP16 hi + lo probabilities, so the only
    FP16 rounding left is the output's (2^-11 relative);
  * the reference's Vulkan prefill test (vulkan/mod.rs:935-1110): its q/k/v generators, shapes
    (q_heads 4, kv_heads 1, head_dim 128; contexts 2048 / 8192 / 28000, n = 64 / 32 / 16 at the
    end of the context) and its bar |got - want| <= 2e-2 + 2e-2·|want| (vulkan/mod.rs:1245-1258),
    against both the per-row decode path and the CPU softmax.
"""
import numpy as np
import pytest

import oracle as O
from graph_horizon_amd import _ffi as F

pytestmark = pytest.mark.gpu


def _kv(hip, layers, ctx, kvh, kc, vc):
    return F.GhKv(hip.from_host(kc), hip.from_host(vc), F.KV_F16, layers, ctx, kvh, 128, 128)


def _free(hip, *bufs):
    for b in bufs:
        hip.free_buffer(b)


def _close(got, want, what, rel=1e-3, floor=1e-5):
    got, want = np.asarray(got, np.float64), np.asarray(want, np.float64)
    tol = rel * np.abs(want) + floor
    bad = np.abs(got - want) > tol
    assert not bad.any(), f"{what}: {bad.sum()} of {bad.size} outside, worst " \
        f"{np.max(np.abs(got - want) / tol):.3f}x tol"


@pytest.mark.parametrize("ctx,base,n,layer", [
    (512, 0, 32, 0),      # one query block, first tile only
    (512, 0, 100, 1),     # ragged rows
    (1024, 300, 200, 1),  # base inside a key tile, query blocks straddling tiles
    (2048, 0, 512, 0),    # the model's prefill chunk
    (4096, 4000, 96, 1),  # late chunk of a long context
])
def test_prefill_attention_matches_oracle(hip, ctx, base, n, layer):
    rng = np.random.default_rng(ctx + base + n)
    layers, qh, kvh = 2, 32, 8
    kc = O.f16(rng.standard_normal(layers * ctx * kvh * 128).astype(np.float32))
    vc = O.f16(rng.standard_normal(layers * ctx * kvh * 128).astype(np.float32))
    q = O.f16(rng.standard_normal(n * qh * 128).astype(np.float32))
    kv = _kv(hip, layers, ctx, kvh, kc, vc)
    qb, ob = hip.from_host(q), hip.alloc_buffer(n * qh * 128 * 2)
    hip.attention_prefill(ob, qb, kv, qh, base, n, layer)
    got = O.f32(hip.download(ob, np.uint16, n * qh * 128))
    want = O.f32(O.attention_prefill(q, kc, vc, 128, kvh, qh, base, n, layer, ctx))
    assert np.isfinite(got).all()
    _close(got, want, f"ctx {ctx} base {base} n {n}")
    _free(hip, qb, ob, kv.k, kv.v)


def test_prefill_attention_c4_2048(hip):
    """BASELINE config 4 prefill: 2048 causal rows, 32 q / 8 kv heads, head_dim 128; 48 rows
    (first, last and spread) checked against the oracle's decode of that row (prefill row r ==
    decode at base + r, attention/mod.rs:920-1024)."""
    n, ctx, qh, kvh = 2048, 2048, 32, 8
    rng = np.random.default_rng(2048)
    kc = O.f16(rng.standard_normal(ctx * kvh * 128).astype(np.float32))
    vc = O.f16(rng.standard_normal(ctx * kvh * 128).astype(np.float32))
    q = O.f16(rng.standard_normal(n * qh * 128).astype(np.float32))
    kv = _kv(hip, 1, ctx, kvh, kc, vc)
    qb, ob = hip.from_host(q), hip.alloc_buffer(n * qh * 128 * 2)
    hip.attention_prefill(ob, qb, kv, qh, 0, n, 0)
    got = O.f32(hip.download(ob, np.uint16, n * qh * 128)).reshape(n, qh * 128)
    assert np.isfinite(got).all()
    rows = sorted(set([0, 1, 31, 32, 63, 64, 1023, 2046, 2047] + list(rng.integers(0, n, 39))))
    for r in rows:
        want = O.f32(O.attention_decode(q[r * qh * 128:(r + 1) * qh * 128], kc, vc, 128, kvh, qh,
                                        r, 0, ctx))
        _close(got[r], want, f"row {r}")
    _free(hip, qb, ob, kv.k, kv.v)


@pytest.mark.parametrize("qh,kvh", [(8, 8), (16, 8), (32, 8), (64, 8), (12, 3), (24, 3)],
                         ids=["g1", "g2", "g4", "g8", "g4-kv3", "g8-kv3"])
@pytest.mark.parametrize("base,n", [(0, 2), (0, 17), (63, 16), (64, 65), (1000, 5), (700, 33), (1, 130),
                                    (40, 600)])
def test_prefill_attention_groups_rows_and_key_splits(hip, qh, kvh, base, n):
    """Every GQA group, at the edges of the 16- and 32-row query blocks and of the 64-key tiles,
    with the backend's key splits and forced ones: later splits start past some rows' last key
    (their partials weigh 0), or hold no tile of the block at all."""
    if n == 600 and qh == 8:
        n = 2050  # 32-row query tiles for the groups that fill the CUs with them
    rng = np.random.default_rng(qh * 1000 + kvh + base + n)
    ctx = base + n + 3
    kc = O.f16(rng.standard_normal(2 * ctx * kvh * 128).astype(np.float32))
    vc = O.f16(rng.standard_normal(2 * ctx * kvh * 128).astype(np.float32))
    q = O.f16(rng.standard_normal(n * qh * 128).astype(np.float32))
    kv = _kv(hip, 2, ctx, kvh, kc, vc)
    qb, ob = hip.from_host(q), hip.alloc_buffer(n * qh * 128 * 2)
    want = O.f32(O.attention_prefill(q, kc, vc, 128, kvh, qh, base, n, 1, ctx))
    try:
        for splits in (0, 1, 3, 32):
            hip.set_attention_splits(splits)
            hip.attention_prefill(ob, qb, kv, qh, base, n, 1)
            got = O.f32(hip.download(ob, np.uint16, n * qh * 128))
            assert np.isfinite(got).all()
            _close(got, want, f"splits {splits}")
    finally:
        hip.set_attention_splits(0)
    _free(hip, qb, ob, kv.k, kv.v)


@pytest.mark.parametrize("qh,kvh", [(8, 8), (16, 8), (32, 8), (64, 8)], ids=["g1", "g2", "g4", "g8"])
@pytest.mark.parametrize("base,n", [(1000, 5), (100, 40), (40, 600)])
def test_prefill_attention_non_finite_cache_rows(hip, qh, kvh, base, n):
    """An infinity or a NaN in the cache reaches the rows that see its position and no others: not the
    earlier rows of the same chunk, whose key tile holds it too, and not from slots past the chunk. 16-
    and 32-row query blocks, with and without key splits."""
    if n == 600 and qh == 8:
        n = 2050
    rng = np.random.default_rng(qh + base + n)
    ctx, at, last = base + n + 3, base + n // 2, base + n - 1
    kc = rng.standard_normal((ctx, kvh, 128)).astype(np.float32)
    vc = rng.standard_normal((ctx, kvh, 128)).astype(np.float32)
    vc[at, :, 0], vc[at, :, 1], vc[at, 0, 2] = np.inf, np.nan, -np.inf
    kc[last, 1, 5] = np.nan
    kc[base + n:], vc[base + n:] = np.nan, np.nan
    kc, vc = O.f16(kc.reshape(-1)), O.f16(vc.reshape(-1))
    q = O.f16(rng.standard_normal(n * qh * 128).astype(np.float32))
    kv = _kv(hip, 1, ctx, kvh, kc, vc)
    qb, ob = hip.from_host(q), hip.alloc_buffer(n * qh * 128 * 2)
    want = O.f32(O.attention_prefill(q, kc, vc, 128, kvh, qh, base, n, 0, ctx))
    finite = np.isfinite(want)
    seen = finite.reshape(n, -1).all(axis=1)
    assert seen[:at - base].all() and not seen[at - base:].any()
    try:
        for splits in (0, 1, 3):
            hip.set_attention_splits(splits)
            hip.attention_prefill(ob, qb, kv, qh, base, n, 0)
            got = O.f32(hip.download(ob, np.uint16, n * qh * 128))
            assert np.array_equal(np.isnan(got), np.isnan(want)), splits
            assert np.array_equal(got[np.isinf(want)], want[np.isinf(want)]), splits
            _close(got[finite], want[finite], f"splits {splits}")
    finally:
        hip.set_attention_splits(0)
    _free(hip, qb, ob, kv.k, kv.v)


@pytest.mark.parametrize("qh,kvh,n,splits", [(3, 3, 5, 3), (1, 1, 33, 5), (5, 5, 7, 1), (4, 1, 9, 31)])
def test_prefill_attention_odd_partial_counts(hip, qh, kvh, n, splits):
    """Key-split partials whose count (rows x heads x splits) is odd, and one that is not a multiple of
    four: the unnormalized sums start on 16 bytes all the same."""
    rng = np.random.default_rng(qh + n)
    base = 2000
    ctx = base + n
    kc, vc = (O.f16(rng.standard_normal(ctx * kvh * 128).astype(np.float32)) for _ in range(2))
    q = O.f16(rng.standard_normal(n * qh * 128).astype(np.float32))
    kv = _kv(hip, 1, ctx, kvh, kc, vc)
    qb, ob = hip.from_host(q), hip.alloc_buffer(n * qh * 128 * 2)
    want = O.f32(O.attention_prefill(q, kc, vc, 128, kvh, qh, base, n, 0, ctx))
    try:
        hip.set_attention_splits(splits)
        hip.attention_prefill(ob, qb, kv, qh, base, n, 0)
    finally:
        hip.set_attention_splits(0)
    _close(O.f32(hip.download(ob, np.uint16, n * qh * 128)), want, "odd")
    _free(hip, qb, ob, kv.k, kv.v)


@pytest.mark.parametrize("qh,kvh", [(8, 8), (16, 8)], ids=["g1", "g2"])
@pytest.mark.parametrize("gap", [26, 34])
def test_prefill_attention_long_flat_tail(hip, qh, kvh, gap):
    """One key far above 32768 others, whose weights are 2^-gap of its: together 2^-11 of the sum (or
    2^-19), all of the numerator where the large key's V is 0. Against fp64, with and without key splits
    and as the decode kernel gives each row. Bar: the output's FP16 rounding (2^-11 relative; 2^-25 where it
    is subnormal), and 2^-40 of the largest weight lost per key, both parts' ends: 2^(gap - 40) of each."""
    n, base = 24, 32768
    ctx = base + n
    # q is ones, so a key's score is the sum of its values / sqrt(128)
    step = gap * np.log(2.0) * np.sqrt(128.0) / 128
    kc = np.full((ctx, kvh, 128), -step, np.float32)
    kc[7] = 0.0
    vc = np.full((ctx, kvh, 128), 48.0, np.float32)
    vc[7] = 0.0
    q = np.ones(n * qh * 128, np.float32)
    k16, v16, q16 = O.f16(kc.reshape(-1)), O.f16(vc.reshape(-1)), O.f16(q)
    kv = _kv(hip, 1, ctx, kvh, k16, v16)
    qb, ob = hip.from_host(q16), hip.alloc_buffer(n * qh * 128 * 2)
    s = O.f32(k16[:128]).astype(np.float64).sum() / np.sqrt(128.0)  # the others' score
    tail = np.exp(s) * (base + np.arange(n))  # of base + r keys beside key 7
    want = np.repeat(48.0 * tail / (1.0 + tail), qh * 128)
    tol = want * (2.0 ** -11 + 2.0 ** (gap - 40) + 1e-5) + 2.0 ** -25
    try:
        for splits in (0, 1):
            hip.set_attention_splits(splits)
            hip.attention_prefill(ob, qb, kv, qh, base, n, 0)
            got = O.f32(hip.download(ob, np.uint16, n * qh * 128)).astype(np.float64)
            worst = np.max(np.abs(got - want) / tol)
            assert worst <= 1, (splits, worst)
    finally:
        hip.set_attention_splits(0)
    hip.attention_decode(ob, qb, kv, qh, base, 0)
    got = O.f32(hip.download(ob, np.uint16, qh * 128)).astype(np.float64)
    assert np.max(np.abs(got - want[:qh * 128]) / tol[:qh * 128]) <= 1
    _free(hip, qb, ob, kv.k, kv.v)


def _reference_case(ctx_total):
    """attention_prefill_decode_for_scheme inputs (vulkan/mod.rs:955-1000), one layer."""
    qh, hd = 4, 128
    pos = np.arange(ctx_total)[:, None]
    i = np.arange(hd)[None, :]
    k = (((pos * 7 + i) % 13).astype(np.float32) * np.float32(0.025) - np.float32(0.12))
    v = (((pos * 11 + i) % 19).astype(np.float32) * np.float32(0.02) - np.float32(0.15))
    return qh, O.f16(k.reshape(-1)), O.f16(v.reshape(-1))


@pytest.mark.parametrize("context", [2048, 8192, 28000])
def test_reference_prefill_attention_vectors(hip, context):
    qh, kc, vc = _reference_case(context)
    kv = _kv(hip, 1, context, 1, kc, vc)
    for n in (64, 32, 16):  # one key-split launch each
        base = context - n
        idx = np.arange(n * qh * 128)
        q = O.f16(((idx % 17).astype(np.float32) * np.float32(0.03) - np.float32(0.22)))
        qb, pb, db = hip.from_host(q), hip.alloc_buffer(q.nbytes), hip.alloc_buffer(q.nbytes)
        hip.attention_prefill(pb, qb, kv, qh, base, n, 0)
        for r in range(n):
            qr = hip.view(qb, r * qh * 256, qh * 256)
            dr = hip.view(db, r * qh * 256, qh * 256)
            hip.attention_decode(dr, qr, kv, qh, base + r, 0)
        got_p = O.f32(hip.download(pb, np.uint16, q.size)).astype(np.float64)
        got_d = O.f32(hip.download(db, np.uint16, q.size)).astype(np.float64)
        # CPU softmax in fp64 over the FP16 inputs (the reference test's own CPU oracle)
        kf = O.f32(kc).astype(np.float64).reshape(context, 128)
        vf = O.f32(vc).astype(np.float64).reshape(context, 128)
        qf = O.f32(q).astype(np.float64).reshape(n, qh, 128)
        cpu = np.empty((n, qh, 128))
        for r in range(n):
            s = qf[r] @ kf[:base + r + 1].T / np.sqrt(128.0)
            p = np.exp(s - s.max(axis=1, keepdims=True))
            cpu[r] = (p / p.sum(axis=1, keepdims=True)) @ vf[:base + r + 1]
        cpu = cpu.reshape(-1)
        for what, a, b in (("prefill vs decode", got_p, got_d), ("prefill vs cpu", got_p, cpu),
                           ("decode vs cpu", got_d, cpu)):
            err = np.abs(a - b)
            ok = err <= 2e-2 + 2e-2 * np.abs(b)
            assert ok.all(), f"ctx {context} n {n} {what}: {(~ok).sum()} outside"
            # and the repository's own bar on the same data
            _close(a, b, f"ctx {context} n {n} {what}", rel=1e-3, floor=1e-5)
        _free(hip, qb, pb, db)
    _free(hip, kv.k, kv.v)


@pytest.mark.parametrize("qh,kvh", [(32, 8), (8, 8), (16, 8), (64, 8)], ids=["g4", "g1", "g2", "g8"])
def test_decode_every_forced_split_count(hip, qh, kvh):
    """Decode attention with each split count 1..32 forced (gh_set_attention_splits), for each
    GQA group size: the split partials cross workgroups through agent-scope atomics and the
    last workgroup of each (row, kv head) merges them. Positions below, at and across chunk
    boundaries, and counts above the row's chunk count. Same bar as the oracle decode test."""
    rng = np.random.default_rng(321 + qh)
    ctx, layers = 2048, 2
    kc = O.f16(rng.standard_normal(layers * ctx * kvh * 128).astype(np.float32))
    vc = O.f16(rng.standard_normal(layers * ctx * kvh * 128).astype(np.float32))
    kv = _kv(hip, layers, ctx, kvh, kc, vc)
    q = O.f16(rng.standard_normal(qh * 128).astype(np.float32))
    qb, ob = hip.from_host(q), hip.alloc_buffer(qh * 128 * 2)
    cases = [(0, 0), (63, 1), (64, 0), (700, 1), (2047, 1)]
    want = {c: O.f32(O.attention_decode(q, kc, vc, 128, kvh, qh, c[0], c[1], ctx)) for c in cases}
    modes = [False, True] if hip.xcd_count else [False]
    try:
        for splits in range(1, 33):
            hip.set_attention_splits(splits)
            for pos, layer in cases:
                bits = []
                for xcd in modes:  # the split merge through device memory, then one XCD's L2
                    hip.set_attention_xcd_merge(xcd)
                    hip.attention_decode(ob, qb, kv, qh, pos, layer)
                    bits.append(hip.download(ob, np.uint16, qh * 128))
                    _close(O.f32(bits[-1]), want[(pos, layer)], f"splits {splits} pos {pos} xcd {xcd}")
                assert all(np.array_equal(b, bits[0]) for b in bits), f"merge forms differ: {splits} {pos}"
    finally:
        hip.set_attention_splits(0)
        hip.set_attention_xcd_merge(bool(hip.xcd_count))
    _free(hip, qb, ob, kv.k, kv.v)


def test_xcd_probe_confirms_the_mi355x_dispatch():
    """The start-up probe sees the eight XCDs of an MI355X (256 CUs) in one partition and
    workgroup i of each probed launch on XCD i mod 8, so decode attention merges its splits
    through one XCD's L2 by default."""
    from graph_horizon_amd import HipBackend

    with HipBackend() as b:
        print(f"xcd_count {b.xcd_count}")
        assert b.xcd_count == 8


@pytest.mark.parametrize("qh,kvh,n,base", [(12, 3, 7, 600), (64, 8, 5, 600), (32, 8, 20, 600), (16, 16, 3, 600),
                                           (8, 1, 6, 600), (4, 1, 20, 600), (16, 16, 3, 300), (6, 3, 8, 600)],
                         ids=["g4-kv3", "g8", "g4-rows20", "g1-kv16", "g8-kv1", "g4-kv1-rows20", "g1-kv16-near", "g2-kv3"])
def test_multi_row_decode_kernels_xcd_grid(hip, qh, kvh, n, base):
    """A few rows over little cache (rows x positions x kv heads up to 16384, 4096 with eight query
    heads per kv head: the first case and the last four) run the decode kernels with several query
    rows, the others the prefill kernels, which the merge form does not touch. In the XCD-local grid the (row, kv head) pairs fill
    z-groups of xcds, the last one partly (kv_heads 3: 21 pairs): both merge forms give the
    same bits, within the oracle bar, at every split count the row lengths allow."""
    if not hip.xcd_count:
        pytest.skip("dispatch placement not confirmed on this device")
    rng = np.random.default_rng(qh * 7 + kvh + n)
    ctx = 1024
    kc = O.f16(rng.standard_normal(ctx * kvh * 128).astype(np.float32))
    vc = O.f16(rng.standard_normal(ctx * kvh * 128).astype(np.float32))
    q = O.f16(rng.standard_normal(n * qh * 128).astype(np.float32))
    kv = _kv(hip, 1, ctx, kvh, kc, vc)
    qb, ob = hip.from_host(q), hip.alloc_buffer(n * qh * 128 * 2)
    want = O.f32(O.attention_prefill(q, kc, vc, 128, kvh, qh, base, n, 0, ctx))
    try:
        for splits in (0, 1, 5, 11):
            hip.set_attention_splits(splits)
            bits = []
            for xcd in (False, True):
                hip.set_attention_xcd_merge(xcd)
                hip.attention_prefill(ob, qb, kv, qh, base, n, 0)
                bits.append(hip.download(ob, np.uint16, n * qh * 128))
                _close(O.f32(bits[-1]), want, f"splits {splits} xcd {xcd}")
            assert np.array_equal(bits[0], bits[1]), f"merge forms differ at {splits} splits"
    finally:
        hip.set_attention_splits(0)
        hip.set_attention_xcd_merge(True)
    _free(hip, qb, ob, kv.k, kv.v)


def test_greedy_graph_with_forced_splits_matches_stream(hip):
    """A replayed decode graph whose attention grid is fixed at 32 splits (most of them idle at
    short positions) gives the tokens of the same steps launched on the stream."""
    from graph_horizon_amd import HipModel, synth

    shape = synth.SHAPES["tiny"]
    outs = []
    hip.set_attention_splits(32)
    try:
        for flags in (0, F.MODEL_NO_GRAPH):
            gm = HipModel(hip, synth.model_config(shape, 2304, 16, flags=flags))
            for layer, tid, fmt, data in synth.model_tensors(shape, 36):
                gm.load_tensor(layer, tid, fmt, data)
            gm.prefill(list(range(1, 60)), 0)
            outs.append(gm.decode_greedy(9, 59, 40))
            gm.close()
    finally:
        hip.set_attention_splits(0)
    assert np.array_equal(outs[0], outs[1])


@pytest.mark.parametrize("kept", [True, False], ids=["old-size-kept", "nothing-kept"])
def test_failed_scratch_growth_re_records_decode_graphs(kept):
    """A prefill attention launch whose partials do not fit runs unsplit. The failed growth may have
    moved or given up the workspace that recorded decode graphs write, so they are recorded again (or,
    without any workspace, the decode reports it) instead of replayed over freed memory."""
    from graph_horizon_amd import GhError, HipBackend, HipModel, synth

    shape, rng = synth.SHAPES["tiny"], np.random.default_rng(6)
    n, base, qh, kvh = 100, 4000, 32, 8  # six key splits: 10 MB of partials
    ctx = base + n
    kc, vc = (O.f16(rng.standard_normal(ctx * kvh * 128).astype(np.float32)) for _ in range(2))
    q = O.f16(rng.standard_normal(n * qh * 128).astype(np.float32))
    want = O.f32(O.attention_prefill(q, kc, vc, 128, kvh, qh, base, n, 0, ctx))
    with HipBackend(0) as b:
        kv = _kv(b, 1, ctx, kvh, kc, vc)
        qb, ob = b.from_host(q), b.alloc_buffer(n * qh * 128 * 2)
        gm = HipModel(b, synth.model_config(shape, 256, 64))
        for layer, tid, fmt, data in synth.model_tensors(shape, 33):
            gm.load_tensor(layer, tid, fmt, data)
        prompt = [3, 99, 1500, 42]
        gm.prefill(prompt, 0)
        first = gm.read_argmax()
        tokens = gm.decode_greedy(first, 4, 70)
        size, slots, gen = b.scratch_info()
        b.set_scratch_limit(size if kept else 64)
        b.attention_prefill(ob, qb, kv, qh, base, n, 0)
        _close(O.f32(b.download(ob, np.uint16, n * qh * 128)), want, "unsplit")
        now = b.scratch_info()
        assert now[0] == (size if kept else 0) and now[1] == slots and now[2] > gen
        if not kept:
            with pytest.raises(GhError) as e:
                gm.decode_greedy(first, 4, 70)
            assert e.value.code == -4  # GH_E_OOM
        b.set_scratch_limit(0)
        gm.prefill(prompt, 0)
        assert np.array_equal(gm.decode_greedy(first, 4, 70), tokens)
        b.attention_prefill(ob, qb, kv, qh, base, n, 0)
        _close(O.f32(b.download(ob, np.uint16, n * qh * 128)), want, "split")
        assert b.scratch_info()[0] > size
        gm.close()
        _free(b, qb, ob, kv.k, kv.v)


def test_graph_replay_ignores_partials_of_earlier_steps(hip):
    """A replayed decode graph whose attention grid is fixed at 4 splits (forced: one step
    graph over the whole 256-position context), while the splits in use follow the position.
    A run that crosses position 64 (two splits in use) leaves real partials and merge state
    behind; replaying the first steps again (one split in use) must give the first run's
    tokens."""
    from graph_horizon_amd import HipModel, synth

    shape = synth.SHAPES["tiny"]
    hip.set_attention_splits(4)
    try:
        gm = HipModel(hip, synth.model_config(shape, 256, 64))
        for layer, tid, fmt, data in synth.model_tensors(shape, 33):
            gm.load_tensor(layer, tid, fmt, data)
        prompt = [3, 99, 1500, 42]
        gm.prefill(prompt, 0)
        first = gm.read_argmax()
        short = gm.decode_greedy(first, 4, 8)
        gm.prefill(prompt, 0)
        long = gm.decode_greedy(first, 4, 70)
        gm.prefill(prompt, 0)
        again = gm.decode_greedy(first, 4, 8)
        gm.close()
    finally:
        hip.set_attention_splits(0)
    assert np.array_equal(long[:8], short) and np.array_equal(again, short)

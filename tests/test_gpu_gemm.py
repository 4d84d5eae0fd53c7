"""Matrix-core prefill GEMM (gh_matmul_batched with several tokens) against the oracle.

Bars:
  * kernel arithmetic: against an fp64 product of the FP16-rounded reference-dequantized
    weights (the GEMM's stated operands), |got - want| <= 1e-3·|want| + 2e-6·Σ|terms| — FP32
    accumulation plus the FP16 rounding of the output (2^-11 relative at most);
  * reference CPU kernel (q4k.rs:218-325 / q6k.rs:157-235 restated in the oracle) on the same
    seeded inputs: the bar above widened by + 2^-12·Σ|terms| for the FP16 rounding of the
    weights. Each rounded weight is within 2^-11 of its FP32 value (the worst-case envelope
    2^-11·Σ|terms|); the errors of thousands of independently rounded weights cancel, and
    the measured deviation (printed, run with -s) stays far below half that envelope;
  * the reference's own prefill parity tests (vulkan/kernels/matmul/prefill/mod.rs:160-300,
    330-450): their weight/activation generators and shapes, their bar
    |got - want| <= 5e-2 or <= 5e-3·max(|want|, 1) (mod.rs:275,440).
"""
import numpy as np
import pytest

import oracle as O
from graph_horizon_amd import synth
from graph_horizon_amd import _ffi as F

pytestmark = pytest.mark.gpu


def _f16_weights(fmt, w, rows, in_dim):
    deq = O.dequant(fmt, w, rows, in_dim)  # bit-exact reference dequantization (FP32)
    return deq.astype(np.float16).astype(np.float64)  # round-to-nearest-even to FP16


def _run(hip, fmt, rows, in_dim, n, seed, d_std=0.02):
    rng = np.random.default_rng(seed)
    w = synth.quant_blocks(rng, fmt, rows, in_dim, d_std)
    a16 = O.f16(rng.standard_normal(n * in_dim).astype(np.float32))
    wb = hip.load_weight(fmt, w, in_dim, rows)
    ab = hip.from_host(a16)
    ob = hip.alloc_buffer(n * rows * 2)
    hip.matmul_batched(ob, ab, wb, in_dim, rows, n)
    got = O.f32(hip.download(ob, np.uint16, n * rows)).reshape(n, rows).astype(np.float64)
    for b in (wb, ab, ob):
        hip.free_buffer(b)
    return w, a16, got


def _check_fp64(fmt, w, a16, got, rows, in_dim, n, what, f16_weights=True):
    w16 = (_f16_weights(fmt, w, rows, in_dim) if f16_weights
           else O.dequant(fmt, w, rows, in_dim).astype(np.float64))
    a = O.f32(a16).astype(np.float64).reshape(n, in_dim)
    want = a @ w16.T
    scale = np.abs(a) @ np.abs(w16).T
    tol = 1e-3 * np.abs(want) + 2e-6 * scale
    bad = np.abs(got - want) > tol
    assert not bad.any(), f"{what}: {bad.sum()} of {bad.size} outside, worst " \
        f"{np.max(np.abs(got - want) / tol):.3f}x tol"


def _check_reference(fmt, w, a16, got, rows, in_dim, n, what, tokens=None):
    tokens = range(n) if tokens is None else tokens
    deq = O.dequant(fmt, w, rows, in_dim).astype(np.float64)
    worst = 0.0
    for t in tokens:
        x = a16[t * in_dim:(t + 1) * in_dim]
        want = O.f32(O.matmul_batched(fmt, x, w, in_dim, rows, 1)).astype(np.float64)
        terms = np.abs(deq) @ np.abs(O.f32(x).astype(np.float64))
        tol = 1e-3 * np.abs(want) + (2e-6 + 2.0 ** -12) * terms
        dev = np.abs(got[t] - want)
        worst = max(worst, float(np.max(np.maximum(dev - 1e-3 * np.abs(want), 0.0) / terms)))
        bad = dev > tol
        assert not bad.any(), f"{what} token {t}: {bad.sum()} outside the FP16-weight envelope"
    print(f"{what}: worst deviation from the reference kernel beyond the output rounding "
          f"= {worst:.3e}·Σ|terms| (envelope 2^-11 = {2.0 ** -11:.3e}, bar 2^-12 + 2e-6)")


def _reference_bar(got, want, what):
    err = np.abs(got - want)
    ok = (err <= 5e-2) | (err <= 5e-3 * np.maximum(np.abs(want), 1.0))
    assert ok.all(), f"{what}: {(~ok).sum()} of {ok.size} outside the reference prefill bar"


@pytest.mark.parametrize("fmt,rows,in_dim,n", [
    (F.FMT_Q4_K, 128, 256, 8),      # smallest: one tile, four units, no split
    (F.FMT_Q4_K, 300, 1024, 37),    # ragged rows and tokens
    (F.FMT_Q6_K, 300, 1024, 130),   # ragged, two token tiles
    (F.FMT_Q4_K, 200, 4096, 129),   # split-K
    (F.FMT_Q6_K, 130, 12288, 64),   # down-projection depth, 16 splits
    (F.FMT_Q6_K, 1024, 5120, 200),  # 14B-shaped V projection
    # 256 tokens and more: the warp-specialized kernels
    (F.FMT_Q4_K, 96, 256, 257),     # smallest: one row tile, a one-token second token tile
    (F.FMT_Q4_K, 1000, 2048, 300),  # narrow output, 96-row tiles, split-K, ragged rows/tokens
    (F.FMT_Q6_K, 2000, 3072, 256),  # one token tile, ragged rows
    (F.FMT_Q6_K, 640, 8448, 700),   # 132 units: 16 splits shrunk to 15 (none empty)
    (F.FMT_Q4_K, 4096, 4096, 384),  # 128-row tiles with split-K
])
def test_gemm_parity(hip, fmt, rows, in_dim, n):
    w, a16, got = _run(hip, fmt, rows, in_dim, n, 7 + rows + n)
    assert np.isfinite(got).all()
    _check_fp64(fmt, w, a16, got, rows, in_dim, n, f"{fmt} {rows}x{in_dim} n={n}")
    _check_reference(fmt, w, a16, got, rows, in_dim, n, f"{fmt} {rows}x{in_dim}",
                     tokens=range(0, n, max(1, n // 8)))


@pytest.mark.parametrize("fmt,rows,in_dim", [(F.FMT_Q4_K, 12288, 4096), (F.FMT_Q6_K, 4096, 12288)])
def test_gemm_c3_full_size(hip, fmt, rows, in_dim):
    """The 512-token prefill GEMMs at full size (gate/up and down of the 8B-shaped block)."""
    n = 512
    w, a16, got = _run(hip, fmt, rows, in_dim, n, 4242 + fmt)
    assert np.isfinite(got).all()
    _check_fp64(fmt, w, a16, got, rows, in_dim, n, f"C3 {fmt} {rows}x{in_dim}")
    _check_reference(fmt, w, a16, got, rows, in_dim, n, f"C3 {fmt}", tokens=[0, 1, 255, 511])


def test_gemm_equals_gemv_within_tolerance_at_threshold(hip):
    """n = 7 of a matrix this small runs the GEMV (exact quant arithmetic), n = 8 the GEMM (FP16-rounded weights): each
    meets the fp64 bar of its own operands on the same data."""
    fmt, rows, in_dim = F.FMT_Q4_K, 256, 2048
    rng = np.random.default_rng(99)
    w = synth.quant_blocks(rng, fmt, rows, in_dim, 0.02)
    a16 = O.f16(rng.standard_normal(8 * in_dim).astype(np.float32))
    wb, ab = hip.load_weight(fmt, w, in_dim, rows), hip.from_host(a16)
    ob = hip.alloc_buffer(8 * rows * 2)
    for n in (7, 8):
        hip.matmul_batched(ob, ab, wb, in_dim, rows, n)
        got = O.f32(hip.download(ob, np.uint16, n * rows)).reshape(n, rows).astype(np.float64)
        _check_fp64(fmt, w, a16[:n * in_dim], got, rows, in_dim, n, f"n={n}", f16_weights=n >= 8)
    for b in (wb, ab, ob):
        hip.free_buffer(b)


@pytest.mark.parametrize("fmt", [F.FMT_Q4_K, F.FMT_Q6_K], ids=["q4k", "q6k"])
@pytest.mark.parametrize("rows,in_dim,n", [
    (13000, 4096, 2), (13000, 4096, 5), (16001, 3072, 7),  # exact weights; an odd block count
    (128, 256, 8), (1, 512, 9), (129, 768, 16), (300, 4096, 17), (1000, 1280, 32), (257, 2048, 33),
    (96, 16640, 40),  # 65 blocks: three per split, the last split shorter
    (640, 5120, 48), (640, 5120, 49),
])
def test_gemm_few_tokens(hip, fmt, rows, in_dim, n):
    """The few-token kernels at the edges of their token tiles, row tiles and K splits: below 8
    tokens against the unrounded weights, from 8 against the FP16-rounded ones."""
    w, a16, got = _run(hip, fmt, rows, in_dim, n, 31 + rows + n)
    assert np.isfinite(got).all()
    _check_fp64(fmt, w, a16, got, rows, in_dim, n, f"{fmt} {rows}x{in_dim} n={n}", f16_weights=n >= 8)


@pytest.mark.parametrize("in_dim,n,most", [
    (65536, 16, 32),  # the most blocks per split (eight, 70 KB of LDS)
    (65536, 48, 16), (16640, 48, 16),  # two blocks per split would be 128 and 33 splits: the tiles instead
])
def test_gemm_few_tokens_bounds_its_splits(in_dim, n, most):
    """The partials of deep matrices stay within 32 splits (16 in the tiles), and the sums right."""
    from graph_horizon_amd import HipBackend

    fmt, rows = F.FMT_Q4_K, 768 if in_dim == 65536 else 3000
    with HipBackend(0) as b:
        w, a16, got = _run(b, fmt, rows, in_dim, n, in_dim + n)
        assert b.scratch_info()[0] <= max(4 << 20, most * n * rows * 4 + 4096)
    _check_fp64(fmt, w, a16, got, rows, in_dim, n, f"{rows}x{in_dim} n={n}")


@pytest.mark.parametrize("fmt", [F.FMT_Q4_K, F.FMT_Q6_K], ids=["q4k", "q6k"])
@pytest.mark.parametrize("x_scale", [2.0 ** -20, 2.0 ** -10, 400.0])
def test_gemm_few_tokens_exact_extremes(hip, fmt, x_scale):
    """Exact weights at the ends of their formats (scales -128 and 127 and quants 0 and 63 in Q6_K,
    whose products exceed FP16's integers; scales and minima 63 in Q4_K, where the minima almost
    cancel the quants) over activations from FP16's subnormals to 1600, against fp64."""
    rows, in_dim, n = 16384, 4096, 3
    rng = np.random.default_rng(5)
    w = synth.quant_blocks(rng, fmt, rows, in_dim, 0.002).reshape(-1, 144 if fmt == F.FMT_Q4_K else 210).copy()
    if fmt == F.FMT_Q4_K:
        w[::3, 4:16] = 255
        w[1::3, 2:4] = (w[1::3, 0:2].view(np.float16) * np.float16(7.5)).view(np.uint8)
    else:
        w[::3, 192:208] = 128  # -128
        w[1::3, 192:208] = 127
        w[::2, :192] = rng.integers(0, 2, (len(w[::2]), 192)).astype(np.uint8) * 255
    w = w.reshape(-1)
    a16 = O.f16((rng.standard_normal(n * in_dim) * x_scale).astype(np.float32))
    wb, ab, ob = hip.load_weight(fmt, w, in_dim, rows), hip.from_host(a16), hip.alloc_buffer(n * rows * 2)
    hip.matmul_batched(ob, ab, wb, in_dim, rows, n)
    got = O.f32(hip.download(ob, np.uint16, n * rows)).reshape(n, rows).astype(np.float64)
    a = O.f32(a16).astype(np.float64).reshape(n, in_dim)
    for r0 in range(0, rows, 4096):
        deq = O.dequant(fmt, w, rows, in_dim)[r0:r0 + 4096].astype(np.float64)
        want, terms = a @ deq.T, np.abs(a) @ np.abs(deq).T
        # FP16 output (2^-11 relative, 2^-25 where it is subnormal) and FP32 sums
        tol = 1e-3 * np.abs(want) + 2e-6 * terms + 2.0 ** -24
        over = np.abs(want) > 65000
        assert (np.abs(got[:, r0:r0 + 4096] - want) <= tol)[~over].all(), (fmt, x_scale)
    for b in (wb, ab, ob):
        hip.free_buffer(b)


@pytest.mark.parametrize("scale", [1.0, 2.0 ** -8, 2.0 ** -15])
def test_gemm_few_tokens_keeps_the_minima_sums(hip, scale):
    """Below 8 tokens the sums that the Q4_K minima multiply are FP32 sums, all of whose 24 bits count:
    weights that are minima alone (quants 0, minima 1), and sub-blocks of activations whose sums
    32006 + 2^-9 and -32006 leave the last one. Exact in FP32 in any order, so the result is, too."""
    rows, in_dim, n = 16384, 4096, 3  # 37.7 MB: the few-token kernels, not the GEMV, from 2 tokens
    block = np.zeros(144, np.uint8)
    block[2:4] = np.frombuffer(np.float16(1.0).tobytes(), np.uint8)  # d = 0, dmin = 1
    block[8:12] = 1    # minima of sub-blocks 0-3
    block[12:16] = 16  # and 4-7 (high nibbles)
    w = np.tile(block, rows * (in_dim // 256))
    assert (O.dequant(F.FMT_Q4_K, w[:144], 1, 256) == -1.0).all()
    x = np.zeros((n, in_dim), np.float32)
    for t in range(n):
        s0, s1 = 32 * (5 * t), 32 * (5 * t + 3)  # in one block and across two
        x[t, s0:s0 + 16], x[t, s0 + 20], x[t, s0 + 31] = 2000.0, 6.0, 2.0 ** -9
        x[t, s1:s1 + 16], x[t, s1 + 20] = -2000.0, -6.0
    x *= scale
    a16 = O.f16(x.reshape(-1))
    assert np.array_equal(O.f32(a16), x.reshape(-1))
    wb, ab, ob = hip.load_weight(F.FMT_Q4_K, w, in_dim, rows), hip.from_host(a16), hip.alloc_buffer(n * rows * 2)
    hip.matmul_batched(ob, ab, wb, in_dim, rows, n)
    got = O.f32(hip.download(ob, np.uint16, n * rows))
    assert (got == -scale * 2.0 ** -9).all(), np.unique(got)
    for b in (wb, ab, ob):
        hip.free_buffer(b)


def _lcg(count, seed=0x9E3779B9):
    """The reference test generator, seed = seed * 1664525 + 1013904223 (mod 2^32), as the
    array of its first `count` outputs (blocks of M steps advanced with the M-step map)."""
    a, c, m, M = 1664525, 1013904223, 0xFFFFFFFF, 65536
    first = np.empty(M, np.uint64)
    for i in range(M):
        seed = (seed * a + c) & m
        first[i] = seed
    am, cm = 1, 0  # s -> am·s + cm is M steps
    for _ in range(M):
        am, cm = (am * a) & m, (cm * a + c) & m
    out = np.empty(((count + M - 1) // M) * M, np.uint64)
    blk = first
    for b in range(len(out) // M):
        out[b * M:(b + 1) * M] = blk
        blk = (blk * np.uint64(am) + np.uint64(cm)) & np.uint64(m)
    return out[:count]


def _reference_q4k_case(in_dim, out_dim, n):
    """q4k_cpu_oracle inputs (prefill/mod.rs:190-215): LCG bytes, d = 0.03, dmin = 0.01,
    activations (rng >> 8) / u32::MAX - 0.5 in FP32, narrowed to FP16 for the device."""
    nbytes = out_dim * (in_dim // 256) * 144
    stream = _lcg(nbytes + n * in_dim)
    q = ((stream[:nbytes] >> np.uint64(16)) & np.uint64(0xFF)).astype(np.uint8)
    blocks = q.reshape(-1, 144)
    blocks[:, 0:2] = np.frombuffer(np.float16(0.03).tobytes(), np.uint8)
    blocks[:, 2:4] = np.frombuffer(np.float16(0.01).tobytes(), np.uint8)
    vals = (stream[nbytes:] >> np.uint64(8)).astype(np.float32)
    act = vals / np.float32(4294967295.0) - np.float32(0.5)
    return q, O.f16(act.astype(np.float32))


def _reference_q6k_case(in_dim, out_dim, n):
    """q6k_cpu_oracle inputs (prefill/mod.rs:360-385): byte i of block b = 17 i + b (mod 256),
    scales i % 7 + 1, d = 0.01; activations (i % 31) / 32 - 0.5."""
    nblk = out_dim * (in_dim // 256)
    q = np.zeros((nblk, 210), np.uint8)
    idx = np.arange(192, dtype=np.uint32)
    for b in range(nblk):
        q[b, :192] = ((idx * 17) + (b & 0xFF)) & 0xFF
    q[:, 192:208] = (np.arange(16) % 7 + 1).astype(np.uint8)
    q[:, 208:210] = np.frombuffer(np.float16(0.01).tobytes(), np.uint8)
    act = (np.arange(n * in_dim) % 31).astype(np.float32) / np.float32(32.0) - np.float32(0.5)
    return q.reshape(-1), O.f16(act)


@pytest.mark.parametrize("fmt,in_dim,out_dim,n", [
    (F.FMT_Q4_K, 4096, 70, 37),       # batched_q4k_small_output_matches_cpu_oracle
    (F.FMT_Q4_K, 14336, 4096, 16),    # batched_q4k_large_k (more tokens than the reference's 3)
    (F.FMT_Q4_K, 5120, 16384, 8),     # batched_q4k_14b gate/up
    (F.FMT_Q4_K, 16384, 5120, 8),     # batched_q4k_14b down
    (F.FMT_Q6_K, 3072, 70, 16),       # batched_q6k_matches_cpu_oracle
    (F.FMT_Q6_K, 3072, 3072, 8),      # batched_q6k_matrix2
    (F.FMT_Q6_K, 5120, 1024, 8),      # batched_q6k_14b V
    (F.FMT_Q6_K, 16384, 5120, 8),     # batched_q6k_14b down
])
def test_gemm_reference_prefill_vectors(hip, fmt, in_dim, out_dim, n):
    make = _reference_q4k_case if fmt == F.FMT_Q4_K else _reference_q6k_case
    w, a16 = make(in_dim, out_dim, n)
    wb, ab = hip.load_weight(fmt, w, in_dim, out_dim), hip.from_host(a16)
    ob = hip.alloc_buffer(n * out_dim * 2)
    hip.matmul_batched(ob, ab, wb, in_dim, out_dim, n)
    got = O.f32(hip.download(ob, np.uint16, n * out_dim)).reshape(n, out_dim).astype(np.float64)
    want = O.f32(O.matmul_batched(fmt, a16, w, in_dim, out_dim, n)).reshape(n, out_dim)
    assert np.isfinite(got).all()
    _reference_bar(got, want.astype(np.float64), f"{fmt} {in_dim}->{out_dim} n={n}")
    for b in (wb, ab, ob):
        hip.free_buffer(b)

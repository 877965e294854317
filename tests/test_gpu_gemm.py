"""GPU parity of the prefill GEMM paths against the CPU oracle.

EXACT_I8: same arithmetic as aion's CPU kernels (int8 activations, exact block dots): held to
max|err| <= 1e-5 rms(ref) and the 2e-3 elementwise bound. BF16_MFMA: weights dequantized to
bf16, activations rounded to bf16, f32 accumulate: normalised error <= 1e-2 against the
f32-activation dequant oracle and NMSE <= 1e-4 against the int8-activation CPU oracle (the
activation-quantization noise floor is ~3e-5). Rows of A never interact, so at the full
config-3 sizes the oracle is evaluated on a sample of rows.
"""
import sys

import numpy as np
import pytest
import torch

from aion_amd import backend as be
from conftest import norm_err, rms_err

pytestmark = pytest.mark.gpu


def say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


def bf16_round(a):
    """f32 -> nearest-even bf16, returned as f32 (config 3: activations are cast to bf16 for the MFMA path)"""
    u = np.ascontiguousarray(a, np.float32).view(np.uint32).astype(np.uint64)
    return (((u + 0x7FFF + ((u >> 16) & 1)) >> 16).astype(np.uint32) << 16).view(np.float32)


CASES = [(be.Q8_0, be.ROWS_NK), (be.Q8_0, be.KMAJOR_KN), (be.Q4_0, be.KMAJOR_KN)]


def make_weight(gpu, dtype, layout, n, k, seed):
    rng = np.random.default_rng(seed)
    shape = (n, k) if layout == be.ROWS_NK else (k, n)
    w = (rng.standard_normal(shape) * 0.02).astype(np.float32)
    blocks = be.quantize_blocks(dtype, w, 1 if layout == be.ROWS_NK else 0)
    return blocks, gpu.upload_weight(dtype, layout, n, k, blocks)


def oracle_i8(orc, dtype, layout, a, blocks, n, **kw):
    if layout == be.ROWS_NK:
        return orc.matmul_nt_q8(a, blocks, n, threads=8, **kw)
    return orc.matmul_q_packed(dtype, a, blocks, n, threads=8, **kw)


@pytest.mark.parametrize("dtype,layout", CASES)
@pytest.mark.parametrize("m,n,k", [(9, 64, 64), (17, 100, 96), (33, 300, 256), (70, 257, 512), (130, 1000, 1024)])
def test_exact_gemm_ragged_shapes(gpu, orc, dtype, layout, m, n, k):
    say("exact", dtype, layout, m, n, k)
    gpu.set_gemm_mode(be.GEMM_EXACT_I8)
    blocks, w = make_weight(gpu, dtype, layout, n, k, seed=m + n + k)
    a = np.random.default_rng(m).standard_normal((m, k)).astype(np.float32)
    a[0, :32] = 0
    got = gpu.matmul(w, a)
    assert gpu.last_kernel() == ("gemm_i8_q8" if dtype == be.Q8_0 else "gemm_i8_q4")
    want = oracle_i8(orc, dtype, layout, a, blocks, n)
    assert norm_err(got, want) < 2e-3 and rms_err(got, want) < 1e-5, (norm_err(got, want), rms_err(got, want))
    # alpha / beta
    c0 = np.random.default_rng(1).standard_normal((m, n)).astype(np.float32)
    got2 = gpu.matmul(w, a, alpha=0.5, beta=2.0, c=c0)
    want2 = oracle_i8(orc, dtype, layout, a, blocks, n, alpha=0.5, beta=2.0, c=c0)
    assert rms_err(got2, want2) < 1e-5
    w.free()


@pytest.mark.parametrize("dtype,layout", CASES)
def test_exact_gemm_rows_match_decode_path(gpu, orc, dtype, layout):
    # the GEMM and the GEMV compute the same formula: per-row results agree to f32 summation order
    gpu.set_gemm_mode(be.GEMM_EXACT_I8)
    blocks, w = make_weight(gpu, dtype, layout, 512, 1024, seed=3)
    a = np.random.default_rng(4).standard_normal((40, 1024)).astype(np.float32)
    full = gpu.matmul(w, a)
    one = gpu.matmul(w, a[7:8])
    assert rms_err(full[7:8], one) < 1e-5
    w.free()


# every (M, N) pair of config 3 (each picks its own tile and launch shape) in every weight format and layout
@pytest.mark.parametrize("dtype,layout", CASES)
@pytest.mark.parametrize("m,n", [(512, 4096), (512, 14336), (2048, 4096), (2048, 14336)])
def test_config3_exact_full_size_on_row_sample(gpu, orc, dtype, layout, m, n):
    k = 4096
    say("config3 exact", dtype, m, n)
    gpu.set_gemm_mode(be.GEMM_EXACT_I8)
    blocks, w = make_weight(gpu, dtype, layout, n, k, seed=n)
    a = np.random.default_rng(m).standard_normal((m, k)).astype(np.float32)
    got = gpu.matmul(w, a)
    rows = np.array([0, 1, 15, 16, 63, 64, m // 2 + 3, m - 2, m - 1])
    want = oracle_i8(orc, dtype, layout, np.ascontiguousarray(a[rows]), blocks, n)
    assert norm_err(got[rows], want) < 2e-3 and rms_err(got[rows], want) < 1e-5
    w.free()


@pytest.mark.parametrize("dtype,layout", CASES)
@pytest.mark.parametrize("m,n,k", [(9, 64, 64), (100, 130, 256), (300, 520, 1024)])
def test_bf16_gemm_ragged_shapes(gpu, orc, dtype, layout, m, n, k):
    say("bf16", dtype, layout, m, n, k)
    gpu.set_gemm_mode(be.GEMM_BF16_MFMA_ALWAYS)         # shapes this small run on the exact kernel in the plain bf16 mode
    try:
        blocks, w = make_weight(gpu, dtype, layout, n, k, seed=m * n)
        a = bf16_round(np.random.default_rng(k).standard_normal((m, k)).astype(np.float32))
        got = gpu.matmul(w, a)
        assert gpu.last_kernel() == "gemm_bf16"
        f32a = orc.matmul_q_f32a(dtype, layout == be.ROWS_NK, a, blocks, n, threads=8)
        e = norm_err(got, f32a)
        say("  norm err vs f32-A", e)
        # the dequantized weight is rounded to bf16 (relative error <= 2^-8 per product, random sign):
        # the output error is ~1.6e-3 of rms(ref) at 1 sigma, independent of k
        assert rms_err(got, f32a) < 1e-2
        i8 = oracle_i8(orc, dtype, layout, a, blocks, n)
        nmse = float(((got - i8) ** 2).sum() / (i8 ** 2).sum())
        assert nmse < 1e-4
        c0 = np.random.default_rng(2).standard_normal((m, n)).astype(np.float32)
        got2 = gpu.matmul(w, a, alpha=0.5, beta=2.0, c=c0)
        assert np.allclose(got2, 0.5 * got + 2.0 * c0, rtol=1e-5, atol=1e-5)
        w.free()
    finally:
        gpu.set_gemm_mode(be.GEMM_EXACT_I8)


# (2048, 14336): 32 column tiles of 256 and 32 of 192 interleaved in one launch (wide, wide, narrow, narrow, ...);
# (2048, 13000): 32 of 256 and 26 of 192 - thirteen whole blocks of that pattern, then the rest of the wide tiles; the last
# narrow tile hangs over the last column. (2048, 9092): 48 tiles of 192 only (two rounds of 3/4 beat one wide round plus a
# narrow one), the last one hanging over; (2048, 5120): 27 tiles of 192 in one round instead of two rounds of 128-row tiles.
# (1300, 11008): 258 tiles of 256 rows would need a second round, so 473 tiles of 128 rows run in two half-time rounds.
# Rows from every 256-row tile, all columns.
@pytest.mark.parametrize("dtype,layout", CASES)
@pytest.mark.parametrize("m,n", [(512, 4096), (512, 14336), (2048, 4096), (2048, 14336), (2048, 9092), (2048, 13000), (2048, 5120), (1300, 11008)])
def test_config3_bf16_full_size_on_row_sample(gpu, orc, dtype, layout, m, n):
    k = 4096
    say("config3 bf16", dtype, m, n)
    gpu.set_gemm_mode(be.GEMM_BF16_MFMA_ALWAYS)
    try:
        blocks, w = make_weight(gpu, dtype, layout, n, k, seed=n + 1)
        a = bf16_round(np.random.default_rng(m + 1).standard_normal((m, k)).astype(np.float32))
        got = gpu.matmul(w, a)
        rows = np.unique(np.array([0, 17, 255, 256, m // 2, m - 1] + [t * 256 + 29 * (t + 1) for t in range(m // 256)]))
        f32a = orc.matmul_q_f32a(dtype, layout == be.ROWS_NK, np.ascontiguousarray(a[rows]), blocks, n, threads=8)
        r = rms_err(got[rows], f32a)
        say("  max|err|/rms vs f32-A dequant", r)
        assert r < 1e-2
        i8 = oracle_i8(orc, dtype, layout, np.ascontiguousarray(a[rows]), blocks, n)
        assert float(((got[rows] - i8) ** 2).sum() / (i8 ** 2).sum()) < 1e-4
        w.free()
    finally:
        gpu.set_gemm_mode(be.GEMM_EXACT_I8)


@pytest.mark.parametrize("dtype,layout", CASES)
def test_exact_gemm_k_slices(gpu, orc, dtype, layout):
    """Few workgroups against a long K: the exact kernel cuts the K steps into slices across workgroups (grid z) and a
    second launch adds the slices in order. Parity as for every exact kernel, alpha / beta / row pitch through the second
    launch, the same bits on a second run (nothing depends on which slice finishes first), and sibling weights that share
    the launch."""
    say("k slices", dtype, layout)
    m, n, k = 24, 520, 8192
    gpu.set_gemm_mode(be.GEMM_EXACT_I8)
    blocks, w = make_weight(gpu, dtype, layout, n, k, seed=41)
    blocks2, w2 = make_weight(gpu, dtype, layout, 200, k, seed=42)
    rng = np.random.default_rng(43)
    a = rng.standard_normal((m, k)).astype(np.float32)
    a_buf = gpu.upload(a)
    ldc = 524
    c0 = rng.standard_normal((m, ldc)).astype(np.float32)
    c_buf = gpu.upload(c0)
    gpu.profile_start()
    gpu.step_matmul(w, a_buf, m, c_buf, ldc=ldc, alpha=0.5, beta=2.0)
    prof = gpu.profile_stop()
    assert [nm for nm, _ in prof if nm.startswith("gemm_i8")] == [prof[-1][0]] * 2        # the sliced kernel and the fold
    got = gpu.download(c_buf, np.float32, (m, ldc))
    want = oracle_i8(orc, dtype, layout, a, blocks, n, alpha=0.5, beta=2.0, c=np.ascontiguousarray(c0[:, :n]))
    assert norm_err(got[:, :n], want) < 2e-3 and rms_err(got[:, :n], want) < 1e-5
    assert np.array_equal(got[:, n:], c0[:, n:])
    first = gpu.matmul(w, a)
    assert np.array_equal(first.view(np.uint32), gpu.matmul(w, a).view(np.uint32))
    c1, c2 = gpu.alloc(m * n * 4), gpu.alloc(m * 200 * 4)
    gpu.step_matmul_batch([w, w2], a_buf, m, [c1, c2])
    got1, got2 = gpu.download(c1, np.float32, (m, n)), gpu.download(c2, np.float32, (m, 200))
    assert rms_err(got1, oracle_i8(orc, dtype, layout, a, blocks, n)) < 1e-5
    assert rms_err(got2, oracle_i8(orc, dtype, layout, a, blocks2, 200)) < 1e-5
    for t in (a_buf, c_buf, c1, c2):
        t.free()
    w.free(); w2.free()


# The exact GEMM's row tiles of 32 (the last one partial, alone and behind full ones), columns that end inside a tile, K of one block, of
# less than a group of four, and of a group and one block; each division of K (2, 4 and 8 wavefronts per tile, 4 slices).
# Tolerance: the dots are exact, so both sides are f32 sums of K / 32 terms, within K / 32 * 2^-24 * sum|terms| of the exact value;
# the terms are of both signs and sum|terms| < 4 sqrt(K / 32) rms here: 3e-5 at 8192, 1e-6 seen.
@pytest.mark.parametrize("dtype,layout", CASES)
@pytest.mark.parametrize("m,n,k", [(9, 31, 32), (31, 33, 64), (32, 32, 96), (33, 65, 160), (97, 64, 2080), (129, 1000, 2048), (64, 4099, 544),
                                   (10, 2050, 8192), (1025, 4097, 64)])
def test_exact_gemm_tiles_and_k_divisions(gpu, orc, dtype, layout, m, n, k):
    say("exact gemm tiles", dtype, layout, m, n, k)
    gpu.set_gemm_mode(be.GEMM_EXACT_I8)
    blocks, w = make_weight(gpu, dtype, layout, n, k, seed=m + k)
    blocks2, w2 = make_weight(gpu, dtype, layout, 40, k, seed=m + k + 1)
    a = np.random.default_rng(m * k).standard_normal((m, k)).astype(np.float32)
    got, got2 = gpu.matmul(w, a), gpu.matmul(w2, a)
    assert rms_err(got, oracle_i8(orc, dtype, layout, a, blocks, n)) < 3e-5
    assert rms_err(got2, oracle_i8(orc, dtype, layout, a, blocks2, 40)) < 3e-5
    # a weight gives the same bits beside a sibling, whether the two share their division of K (and a launch) or not
    a_buf, c, c2 = gpu.upload(a), gpu.alloc(m * n * 4), gpu.alloc(m * 40 * 4)
    gpu.step_matmul_batch([w, w2], a_buf, m, [c, c2])
    assert np.array_equal(gpu.download(c, np.uint32, (m, n)), got.view(np.uint32))
    assert np.array_equal(gpu.download(c2, np.uint32, (m, 40)), got2.view(np.uint32))
    for t in (a_buf, c, c2):
        t.free()
    w.free(); w2.free()


@pytest.mark.parametrize("dtype,layout", CASES)
@pytest.mark.parametrize("m,n,k", [(2048, 14336, 4096), (512, 4096, 4096), (300, 520, 1056), (1300, 11008, 4096), (70, 200, 96)])
def test_bf16_gemm_without_weight_copies_gives_the_same_bits(gpu, orc, dtype, layout, m, n, k):
    """The bf16 kernel's two weight operands: the bf16 copy the context keeps of a weight, and the weight's quant blocks
    converted while the kernel stages them (aionhip_set_bf16_weight_copies(0): nothing resident, nothing allocated).
    Both round code * scale to bf16 once and multiply in the same order: the same bits, every tile shape (256 x 256 and
    256 x 192 mixed, 128-row, 64-row and 64 x 128 tiles, ragged edges, a K that is not a multiple of four blocks)."""
    say("bf16 without copies", dtype, layout, m, n, k)
    gpu.set_gemm_mode(be.GEMM_BF16_MFMA_ALWAYS)
    try:
        blocks, w = make_weight(gpu, dtype, layout, n, k, seed=m + n)
        a = bf16_round(np.random.default_rng(k).standard_normal((m, k)).astype(np.float32))
        copies0 = gpu.bf16_copy_stats()
        with_copy = gpu.matmul(w, a)
        assert gpu.last_kernel() == "gemm_bf16" and gpu.bf16_copy_stats()[0] == copies0[0] + 1
        w.drop_bf16()
        assert gpu.bf16_copy_stats() == copies0
        gpu.set_bf16_weight_copies(False)
        streamed = gpu.matmul(w, a)
        assert gpu.last_kernel() == "gemm_bf16" and gpu.bf16_copy_stats() == copies0      # no copy was built
        assert np.array_equal(with_copy.view(np.uint32), streamed.view(np.uint32))
        rows = np.unique(np.array([0, m // 3, m - 1]))
        f32a = orc.matmul_q_f32a(dtype, layout == be.ROWS_NK, np.ascontiguousarray(a[rows]), blocks, n, threads=8)
        assert rms_err(streamed[rows], f32a) < 1e-2
        c0 = np.random.default_rng(2).standard_normal((m, n)).astype(np.float32)
        got2 = gpu.matmul(w, a, alpha=0.5, beta=2.0, c=c0)
        assert np.allclose(got2, 0.5 * streamed + 2.0 * c0, rtol=1e-5, atol=1e-5)
        w.free()
    finally:
        gpu.set_bf16_weight_copies(True)
        gpu.set_gemm_mode(be.GEMM_EXACT_I8)


@pytest.mark.parametrize("ldc,c_offset", [(520, 0), (524, 0), (521, 0), (528, 3)])
def test_bf16_gemm_alpha_beta_and_output_strides(gpu, orc, ldc, c_offset):
    """The bf16 kernel's epilogue: 16-byte stores where the output rows allow them (row pitch and base 16-byte aligned),
    single floats otherwise (odd pitch, a base that is only 4-byte aligned), alpha and beta in both, the columns between
    n and the pitch untouched. Checked against the same kernel's plain product: C' = alpha * (A W^T) + beta * C."""
    say("bf16 alpha/beta", ldc, c_offset)
    m, n, k = 300, 520, 1024
    gpu.set_gemm_mode(be.GEMM_BF16_MFMA_ALWAYS)
    try:
        blocks, w = make_weight(gpu, be.Q4_0, be.KMAJOR_KN, n, k, seed=31)
        rng = np.random.default_rng(32)
        a = rng.standard_normal((m, k)).astype(np.float32)
        c0 = rng.standard_normal(m * ldc + c_offset).astype(np.float32)
        plain = gpu.matmul(w, a)
        assert gpu.last_kernel() == "gemm_bf16"
        a_buf, c_buf = gpu.upload(a), gpu.upload(c0)
        gpu.step_matmul(w, a_buf, m, c_buf, ldc=ldc, alpha=0.5, beta=2.0, c_offset=c_offset * 4)
        got = gpu.download(c_buf, np.float32, (m * ldc + c_offset,))
        assert np.array_equal(got[:c_offset], c0[:c_offset])
        got2, old2 = got[c_offset:].reshape(m, ldc), c0[c_offset:].reshape(m, ldc)
        want = 0.5 * plain + 2.0 * old2[:, :n]
        assert float(np.abs(got2[:, :n] - want).max()) <= 1e-5 * float(np.abs(want).max())
        assert np.array_equal(got2[:, n:], old2[:, n:])
        a_buf.free(); c_buf.free(); w.free()
    finally:
        gpu.set_gemm_mode(be.GEMM_EXACT_I8)


def test_bf16_mode_runs_the_bf16_kernel_only_where_it_pays(gpu, orc):
    """In bf16 mode a shape the bf16 kernel is not expected to win (few rows: it streams a 2-byte copy of the weight
    through 256-column tiles) stays on the exact kernel - same numbers as the exact mode - and a large one moves."""
    blocks, w = make_weight(gpu, be.Q4_0, be.KMAJOR_KN, 4096, 4096, seed=5)
    rng = np.random.default_rng(6)
    small, large = rng.standard_normal((48, 4096)).astype(np.float32), rng.standard_normal((2048, 4096)).astype(np.float32)
    exact_small = gpu.matmul(w, small)
    gpu.set_gemm_mode(be.GEMM_BF16_MFMA)
    try:
        got = gpu.matmul(w, small)
        assert gpu.last_kernel() == "gemm_i8_q4" and np.array_equal(got, exact_small)
        gpu.matmul(w, large)
        assert gpu.last_kernel() == "gemm_bf16"
        gpu.set_gemm_mode(be.GEMM_BF16_MFMA_ALWAYS)
        gpu.matmul(w, small)
        assert gpu.last_kernel() == "gemm_bf16"
    finally:
        gpu.set_gemm_mode(be.GEMM_EXACT_I8)
    w.free()


# A row with an infinite element has one block of scale inf, whose codes are 0 but for -127 at that element (the clamp of 0 * inf): each sum
# is inf against the sign of the weight there, NaN where that weight is 0. Only what the block multiplies may leave the finite range:
# the rescale that starts a wavefront's pipeline, and the blocks a last group has past the end of K, must not meet it with a zero. The
# block is the first, the last and one in the middle; K ends inside a group of four blocks and at its end.
@pytest.mark.parametrize("dtype,layout", CASES)
@pytest.mark.parametrize("m,n,k", [(40, 100, 160), (33, 96, 2080), (9, 40, 8224), (8, 1056, 992), (150, 4128, 2048)])
def test_exact_gemm_infinite_activations(gpu, orc, dtype, layout, m, n, k):
    say("inf", dtype, layout, m, n, k)
    gpu.set_gemm_mode(be.GEMM_EXACT_I8)
    blocks, w = make_weight(gpu, dtype, layout, n, k, seed=m + k)
    a = np.random.default_rng(k).standard_normal((m, k)).astype(np.float32)
    a[0, 3], a[1, k - 5], a[m - 2, k // 64 * 32 + 7] = np.inf, np.inf, -np.inf
    got = gpu.matmul(w, a)
    assert "gemm_i8" in gpu.last_launch()["kernel"]
    for r, col in ((0, 3), (1, k - 5), (m - 2, k // 64 * 32 + 7)):
        one = np.zeros((1, k), np.float32)
        one[0, col] = 1
        sign = np.sign(gpu.matmul(w, one)[0])
        assert np.array_equal(got[r], np.where(sign == 0, np.nan, np.where(sign > 0, -np.inf, np.inf)), equal_nan=True), r
    rows = [r for r in range(m) if r not in (0, 1, m - 2)]
    assert rms_err(got[rows], oracle_i8(orc, dtype, layout, a[rows], blocks, n)) < 3e-5      # (bound: test_exact_gemm_tiles_and_k_divisions)
    w.free()


# The same with an infinite block in each place of K in turn, a row for each: whatever a wavefront's buffers held two groups earlier, the
# blocks that a last group has past the end of K (one to three here) multiply as zero.
@pytest.mark.parametrize("dtype,layout", CASES)
@pytest.mark.parametrize("n,k", [(64, 544), (96, 1120), (40, 2080), (4096, 992), (33, 4000)])
def test_exact_gemm_infinite_block_anywhere(gpu, dtype, layout, n, k):
    say("inf anywhere", dtype, layout, n, k)
    gpu.set_gemm_mode(be.GEMM_EXACT_I8)
    _, w = make_weight(gpu, dtype, layout, n, k, seed=n + k)
    m = k // 32
    one = np.zeros((m, k), np.float32)
    one[np.arange(m), np.arange(m) * 32 + 9] = 1
    a = np.random.default_rng(k).standard_normal((m, k)).astype(np.float32)
    a[one == 1] = np.inf
    for rows in (m, 12):                             # (the last rows: the last blocks of K)
        sign = np.sign(gpu.matmul(w, one[-rows:]))
        got = gpu.matmul(w, a[-rows:])
        assert "gemm_i8" in gpu.last_launch()["kernel"]
        assert np.array_equal(got, np.where(sign == 0, np.nan, np.where(sign > 0, -np.inf, np.inf)), equal_nan=True), rows
    w.free()


# Sums stay finite up to the f32 range: the lowest f32, as a mask leaves it, in four blocks of a row gives sums of 1e37 .. 1e38. Beside it
# rows of ordinary values. (test_gpu_prepare_act.py holds the other end: products of subnormal scales keep their bits.)
@pytest.mark.parametrize("dtype,layout", CASES)
@pytest.mark.parametrize("m,n,k", [(40, 100, 160), (33, 96, 2080), (9, 40, 8224), (8, 1056, 992), (150, 4128, 2048)])
def test_exact_gemm_lowest_activations(gpu, orc, dtype, layout, m, n, k):
    say("lowest", dtype, layout, m, n, k)
    gpu.set_gemm_mode(be.GEMM_EXACT_I8)
    blocks, w = make_weight(gpu, dtype, layout, n, k, seed=m + k)
    a = np.random.default_rng(k).standard_normal((m, k)).astype(np.float32)
    lowest = np.finfo(np.float32).min
    a[3, [0, 40, 70, k - 1]] = lowest
    a[m - 1, [5, 33, 100, k - 32]] = lowest
    got = gpu.matmul(w, a)
    assert "gemm_i8" in gpu.last_launch()["kernel"]
    want = oracle_i8(orc, dtype, layout, a, blocks, n)
    assert np.abs(want[[3, m - 1]]).max() > 2.2e37 and np.isfinite(want).all() and np.isfinite(got).all()
    assert max(rms_err(g, x) for g, x in zip(got, want)) < 3e-5          # (bound: test_exact_gemm_tiles_and_k_divisions)
    w.free()


# Division of a long K over workgroups: either side of the lines (K = 6144, half a 32 x 32 tile per CU; K = 11008, three quarters; q4 8192 and
# a quarter; up to 32 rows five quarters from K = 6528, q4 8192, and six from 11008), seen as the second launch that adds the slices. Tolerance as in test_exact_gemm_tiles_and_k_divisions: 3e-5 at K = 11008.
@pytest.mark.parametrize("m,n,k,q8_sliced,q4_sliced", [(9, 4096, 6144, True, False), (9, 4097, 6144, False, False), (16, 2048, 6112, False, False),
                                                       (33, 2050, 8192, False, False), (40, 1024, 8192, True, True), (10, 6144, 11008, True, False),
                                                       (10, 6145, 11008, False, False), (9, 9664, 11008, True, True), (9, 9665, 6528, True, False),
                                                       (32, 10240, 6496, False, False), (9, 12288, 11008, True, True), (9, 12289, 11008, False, False),
                                                       (33, 4900, 11008, False, False)])
def test_exact_gemm_k_slices(gpu, orc, m, n, k, q8_sliced, q4_sliced):
    for dtype, layout, sliced in ((be.Q8_0, be.ROWS_NK, q8_sliced), (be.Q4_0, be.KMAJOR_KN, q4_sliced)):
        say("slices", dtype, m, n, k)
        gpu.set_gemm_mode(be.GEMM_EXACT_I8)
        blocks, w = make_weight(gpu, dtype, layout, n, k, seed=m + k)
        a = np.random.default_rng(m * k).standard_normal((m, k)).astype(np.float32)
        got = gpu.matmul(w, a)
        assert ("slices" in gpu.last_launch()["kernel"]) == sliced
        assert rms_err(got, oracle_i8(orc, dtype, layout, a, blocks, n)) < 3e-5
        w.free()


# A short K against a wide grid: wide tiles whose wavefronts share K less (1 or 2 to a tile instead of 4), rows and columns that end inside a
# tile and inside a wavefront's part of it, K of one block, inside a group and of whole groups, both numbers of rows a tile keeps.
# Tolerance as in test_exact_gemm_tiles_and_k_divisions (K / 32 terms: far below its 3e-5).
@pytest.mark.parametrize("dtype,layout", CASES)
@pytest.mark.parametrize("m,n,k,most", [(257, 33000, 32, 2), (384, 32900, 96, 2), (300, 32900, 96, 2), (129, 131072, 128, 2), (1000, 16500, 160, 1), (9, 131100, 544, 2),
                                        (16, 131073, 512, 2), (17, 131110, 64, 2), (96, 33001, 512, 2), (5, 100000, 544, 2)])
def test_exact_gemm_short_k_wide_grid(gpu, orc, dtype, layout, m, n, k, most):
    say("short k", dtype, layout, m, n, k)
    gpu.set_gemm_mode(be.GEMM_EXACT_I8)
    blocks, w = make_weight(gpu, dtype, layout, n, k, seed=m + k)
    a = np.random.default_rng(m * k).standard_normal((m, k)).astype(np.float32)
    got = gpu.matmul(w, a)
    instance = [x.strip() for x in gpu.last_launch()["kernel"].split("<")[1].split(">")[0].split(",")]
    assert int(instance[3]) <= most, instance                      # wavefronts that share a tile's K
    rows = sorted({0, 1, 2, 15, 16, 31, 32, 63, 64, 127, 128, m - 2, m - 1} & set(range(m)))
    assert rms_err(got[rows], oracle_i8(orc, dtype, layout, a[rows], blocks, n)) < 3e-5
    again = gpu.matmul(w, a)
    assert np.array_equal(got.view(np.uint32), again.view(np.uint32))
    w.free()


# Wavefronts of more than one tile take the products of scales from the matrix pipe, calls of up to 16 rows multiply. With one block of a row's K
# that is not zero a sum is one rounded product, so every row has the bits that it has in a call of 12: row scales from 2^-100 to 2^40 beside
# each other, column tiles and row tiles with ends, every place of K.
@pytest.mark.parametrize("dtype,layout", CASES)
@pytest.mark.parametrize("m,n,k", [(512, 4096, 2048), (500, 4070, 2080), (1030, 8200, 1024), (77, 11008, 672), (300, 5000, 1056), (700, 14330, 544),
                                   (90, 2100, 4096), (24, 32800, 2048), (24, 32800, 4128)])
def test_exact_gemm_scale_products_keep_their_bits(gpu, orc, dtype, layout, m, n, k):
    say("scale products", dtype, layout, m, n, k)
    gpu.set_gemm_mode(be.GEMM_EXACT_I8)
    _, w = make_weight(gpu, dtype, layout, n, k, seed=m + k)
    rng = np.random.default_rng(k)
    a = np.zeros((m, k // 32, 32), np.float32)
    at = np.arange(m) * 7 % (k // 32)
    a[np.arange(m), at] = rng.standard_normal((m, 32)) * 2.0 ** rng.integers(-100, 41, (m, 1))
    a = a.reshape(m, k)
    got = gpu.matmul(w, a)
    assert "gemm_i8" in gpu.last_launch()["kernel"]
    for rows in ([0, 1, m // 2, m - 1, *rng.integers(0, m, 8)], rng.integers(0, m, 12)):
        assert np.array_equal(got[rows].view(np.uint32), gpu.matmul(w, a[rows]).view(np.uint32)), rows
        assert "gemm_i8" in gpu.last_launch()["kernel"]
    w.free()


# A GeGLU block of many rows with the gate and the preparation of its rows in the gate / up launch: the bits of the two calls it stands for, at
# the edges of the 32-, 64- and 128-row tiles and for widths and K that end inside a group of four blocks; a row of zeros among them.
@pytest.mark.parametrize("dtype,layout", CASES)
@pytest.mark.parametrize("rows,hidden,ffn", [(9, 256, 512), (16, 2048, 4128), (17, 2080, 8192), (32, 2048, 544), (33, 96, 8224), (64, 1056, 2048), (65, 2048, 8192),
                                             (100, 256, 11008), (5, 4128, 2080), (8, 4224, 12320), (16, 2624, 8224), (128, 2048, 8192), (129, 4096, 1056), (300, 672, 2080), (1100, 512, 16416), (2048, 2048, 8192)])
def test_geglu_block_of_many_rows_is_the_separate_calls(gpu, dtype, layout, rows, hidden, ffn):
    say("geglu rows", dtype, layout, rows, hidden, ffn)
    gpu.set_gemm_mode(be.GEMM_EXACT_I8)
    rng = np.random.default_rng(rows + ffn)
    wg, wu, wd = (make_weight(gpu, dtype, layout, n, k, seed=n + s)[1] for s, (n, k) in enumerate(((ffn, hidden), (ffn, hidden), (hidden, ffn))))
    x = rng.standard_normal((rows, hidden)).astype(np.float32)
    x[rows // 2] = 0
    gamma, beta = (gpu.upload(rng.standard_normal(hidden).astype(np.float32)) for _ in range(2))
    xb, gate, up = gpu.upload(x), gpu.alloc(4 * rows * ffn), gpu.alloc(4 * rows * ffn)
    for norm_beta, alpha, b in ((None, 1.0, 1.0), (beta, 0.5, 0.0)):
        c = [gpu.upload(np.full((rows, hidden), 0.25, np.float32)) for _ in range(2)]
        gpu.step_rmsnorm_matmul([wg, wu], xb, gamma, rows, [gate, up], 1e-6, beta_norm=norm_beta)
        gpu.step_gate_matmul(wd, gate, up, rows, c[0], alpha=alpha, beta=b)
        ran = gpu.step_rmsnorm_geglu_matmul_rows(wg, wu, wd, xb, gamma, rows, 1e-6, c[1], alpha=alpha, beta=b, beta_norm=norm_beta)
        if (rows, hidden) != (33, 96):                       # (may be refused there: one or two wavefronts to a K, and a row tile to spare)
            assert ran == (rows != 16 or hidden != 2624)     # (a nearly empty second round)
        want, got = (gpu.download(t, np.float32, (rows, hidden)) for t in c)
        if ran:
            assert np.isfinite(want).all() and np.array_equal(want.view(np.uint32), got.view(np.uint32))
        else:
            assert (got == 0.25).all()
        for t in c:
            t.free()
    for t in (wg, wu, wd, gamma, beta, xb, gate, up):
        t.free()
    say("ran" if ran else "refused")


# RMSNorm, q, k, v, the rotation and the cache appends of many tokens as two launches: the bits of the two calls they stand for, at the edges of
# the row tiles, over head sizes and layouts, divisions of K, for several sequences at their own write indices (one of them past the end of its cache: not
# written) and a partial rotation.
@pytest.mark.parametrize("dtype,layout", CASES)
@pytest.mark.parametrize("b,s,hidden,heads,kv_heads,d,t_cap,runs", [
    (1, 9, 512, 48, 48, 64, 40, True), (1, 128, 2048, 8, 1, 256, 256, True), (2, 33, 1056, 32, 4, 128, 100, True), (1, 33, 4096, 32, 8, 128, 40, True),
    (3, 50, 640, 4, 4, 192, 300, True), (3, 50, 640, 16, 16, 192, 300, True), (1, 9, 2080, 48, 48, 64, 30, True), (1, 17, 2080, 32, 32, 128, 17, True), (1, 16, 1056, 48, 48, 64, 40, True),
    (1, 300, 672, 8, 1, 256, 300, True), (1, 1100, 544, 16, 16, 128, 1100, True), (1, 700, 512, 32, 32, 128, 700, True), (1, 8, 4128, 40, 40, 128, 20, True), (5, 1, 4128, 48, 48, 64, 3, True),
    (1, 65, 4096, 32, 8, 128, 65, False), (1, 700, 512, 32, 8, 128, 1024, False),              # (the K of q and of k, v divided differently; q8: few rows)
    (1, 9, 512, 8, 1, 64, 40, False), (2, 33, 1056, 6, 2, 128, 100, False), (1, 32, 4096, 32, 8, 128, 40, False), (1, 48, 4096, 32, 32, 128, 48, False)])      # (the separate launches' tiles)
def test_qkv_rope_append_of_many_tokens_is_the_separate_calls(gpu, dtype, layout, b, s, hidden, heads, kv_heads, d, t_cap, runs):
    say("qkv rope rows", dtype, layout, b, s, hidden, heads, kv_heads, d)
    gpu.set_gemm_mode(be.GEMM_EXACT_I8)
    rng = np.random.default_rng(s + hidden)
    rows = b * s
    ws = [make_weight(gpu, dtype, layout, n * d, hidden, seed=n * d + i)[1] for i, n in enumerate((heads, kv_heads, kv_heads))]
    x, gamma = gpu.upload(rng.standard_normal((rows, hidden)).astype(np.float32)), gpu.upload(rng.standard_normal(hidden).astype(np.float32))
    at = np.minimum(np.arange(b) * 7, t_cap - s).astype(np.int32)
    if b > 1:
        at[-1] = t_cap - s + 2
    pos, widx = gpu.upload((at[:, None] + np.arange(s)).astype(np.int32)), gpu.upload(at)
    q, k, v = (gpu.alloc(4 * rows * n * d) for n in (heads, kv_heads, kv_heads))
    for proportion in (1.0, 0.4):
        outs = []
        for fused in (False, True):
            qr = gpu.zeros(4 * rows * heads * d)
            kc, vc = (gpu.upload(np.full((b, t_cap, kv_heads, d), 3.0, np.float16)) for _ in range(2))
            if fused:
                ran = gpu.step_rmsnorm_qkv_rope_append_rows(*ws, x, gamma, 1e-6, qr, kc, vc, pos, widx, b, s, t_cap, heads, kv_heads, d, proportion=proportion)
            else:
                gpu.step_rmsnorm_matmul(ws, x, gamma, rows, [q, k, v], 1e-6)
                gpu.step_rope_append(qr, q, k, v, kc, vc, pos, widx, b, s, t_cap, heads, kv_heads, d, proportion=proportion)
            outs.append([gpu.download(qr, np.uint32, (rows * heads * d,))] + [gpu.download(t, np.uint16, (b * t_cap * kv_heads * d,)) for t in (kc, vc)])
            for t in (qr, kc, vc):
                t.free()
        say("ran" if ran else "refused")
        for want, got in zip(*outs):
            assert np.array_equal(want, got) if ran else np.unique(got).size == 1
    assert ran == runs
    for t in ws + [x, gamma, pos, widx, q, k, v]:
        t.free()


# Attention whose rows leave as the exact GEMM reads them: the bits of the attention step and the matmul, at the edges of the 32-row tiles, over head
# sizes, layouts, types and windows, on both kernels of a prompt and for sequences of several lengths; refused, with nothing written, where the
# attention runs in segments or the rows are few.
@pytest.mark.parametrize("dtype,layout", CASES)
@pytest.mark.parametrize("b,s,t,heads,kv_heads,d,n,q_type,kv_type,window,runs", [
    (1, 9, 40, 8, 1, 64, 320, "f32", "f16", None, True), (1, 128, 256, 8, 1, 256, 2048, "f32", "f16", None, True), (2, 33, 100, 6, 2, 128, 500, "f16", "f16", None, True),
    (1, 65, 200, 32, 8, 128, 1024, "bf16", "bf16", (40, 0, 0), True), (3, 17, 64, 2, 2, 256, 96, "f32", "bf16", None, True), (1, 31, 31, 16, 4, 64, 33, "f32", "f16", (8, 3, 0), True),
    (1, 300, 2000, 8, 1, 128, 512, "f32", "f16", None, False), (1, 1000, 1000, 16, 4, 64, 512, "f32", "f16", None, False), (1, 64, 1500, 4, 1, 64, 512, "f32", "f16", None, False),
    (1, 4, 64, 8, 1, 64, 512, "f32", "f16", None, False), (1, 512, 512, 32, 8, 128, 2048, "f32", "f16", None, True), (2, 300, 300, 8, 2, 256, 320, "f32", "f16", None, True),
    (4, 200, 260, 32, 32, 128, 96, "f16", "f16", (70, 0, 0), True), (2, 500, 501, 16, 16, 64, 512, "f32", "bf16", None, True)])
def test_attention_and_its_matmul_is_the_separate_calls(gpu, dtype, layout, b, s, t, heads, kv_heads, d, n, q_type, kv_type, window, runs):
    say("attention matmul", dtype, layout, b, s, t, heads, kv_heads, d, n, q_type, kv_type, window)
    gpu.set_gemm_mode(be.GEMM_EXACT_I8)
    gen = torch.Generator().manual_seed(s + t)
    types = {"f32": (torch.float32, be.F32), "f16": (torch.float16, be.F16), "bf16": (torch.bfloat16, be.BF16)}

    def operand(kind, *shape):
        return gpu.upload(torch.randn(shape, generator=gen).to(types[kind][0]).contiguous().view(torch.uint8).numpy())

    q, k, v = operand(q_type, b, s, heads, d), operand(kv_type, b, t, kv_heads, d), operand(kv_type, b, t, kv_heads, d)
    lengths = np.array([max(s, t - 5 * i) for i in range(b)], np.int32)
    pos = gpu.upload((lengths[:, None] - s + np.arange(s)).astype(np.int32))
    if b == 4:
        lengths[-1] = 0                                      # (a sequence that sees no key: rows of zeros)
    lens = gpu.upload(lengths)
    w = make_weight(gpu, dtype, layout, n, heads * d, seed=n)[1]
    rows, shape = b * s, (b, s, t, heads, kv_heads, d, d)
    options = {"q_dtype": types[q_type][1], "kv_dtype": types[kv_type][1], "window": window or be.CAUSAL, "query_positions": pos, "kv_lengths": lens}
    out = gpu.alloc(4 * rows * heads * d)
    for alpha, beta in ((1.0, 1.0), (0.5, 0.0)):
        c = [gpu.upload(np.full((rows, n), 0.25, np.float32)) for _ in range(2)]
        gpu.step_attention(out, q, k, v, shape, d ** -0.5, **options)
        gpu.step_matmul(w, out, rows, c[0], alpha=alpha, beta=beta)
        assert gpu.step_attention_matmul(w, q, k, v, shape, d ** -0.5, c[1], alpha=alpha, beta=beta, **options) == runs
        want, got = (gpu.download(x, np.float32, (rows, n)) for x in c)
        if runs:
            assert np.isfinite(want).all() and np.array_equal(want.view(np.uint32), got.view(np.uint32))
        else:
            assert (got == 0.25).all()
        for x in c:
            x.free()
    for x in (q, k, v, pos, lens, w, out):
        x.free()


# What the row-preparing attention refuses has written nothing and says why: precise mode, a soft cap on the 128-row kernel, rolling caches, keys in
# segments, no keys, a head size of the generic kernel. A soft cap on the 16-row kernel runs, and so does a short prompt beside a sequence that
# sees no key (rows of zeros).
@pytest.mark.parametrize("b,s,t,heads,kv_heads,d,options,why", [
    (1, 33, 64, 8, 1, 64, {"precise": True}, "precise"), (1, 512, 512, 32, 8, 128, {"soft_cap": 20.0}, "soft cap"), (1, 20, 128, 8, 1, 64, {"rolling": True}, "rolling"),
    (1, 512, 512, 32, 8, 128, {"rolling": True}, "rolling"), (1, 64, 1500, 4, 1, 64, {}, "segments"), (1, 1000, 1000, 16, 4, 64, {}, "segments"), (1, 20, 0, 8, 1, 64, {}, "no keys"),
    (1, 20, 40, 8, 1, 96, {}, "generic"), (1, 20, 40, 8, 1, 64, {"soft_cap": 20.0}, None), (4, 17, 70, 8, 2, 128, {"unseen": True}, None),
    (3, 9, 40, 2, 2, 256, {"unseen": True}, None)])
def test_attention_matmul_refusals_and_unseen_rows(gpu, b, s, t, heads, kv_heads, d, options, why):
    say("attention matmul refusals", b, s, t, heads, kv_heads, d, options)
    gpu.set_gemm_mode(be.GEMM_EXACT_I8)
    rng = np.random.default_rng(s + t)
    n, rows, shape = 96, b * s, (b, s, t, heads, kv_heads, d, d)
    q = gpu.upload(rng.standard_normal((rows, heads, d)).astype(np.float32))
    k, v = (gpu.upload(rng.standard_normal((b, max(t, 1), kv_heads, d)).astype(np.float16)) for _ in range(2))
    lengths = np.full(b, t, np.int32)
    if options.get("unseen"):
        lengths[1] = 0
    pos, lens = gpu.upload((t - s + np.arange(rows) % s).astype(np.int32).reshape(b, s)), gpu.upload(lengths)
    w = make_weight(gpu, be.Q8_0, be.ROWS_NK, n, heads * d, seed=n)[1]
    kw = {"query_positions": pos, "kv_lengths": lens, "soft_cap": options.get("soft_cap", 0.0), "rolling": options.get("rolling", False)}
    c = [gpu.upload(np.full((rows, n), 0.25, np.float32)) for _ in range(2)]
    out = gpu.alloc(4 * rows * heads * d)
    gpu.set_attention_precise(options.get("precise", False))
    try:
        ran = gpu.step_attention_matmul(w, q, k, v, shape, d ** -0.5, c[1], beta=1.0, **kw)
        assert ran == (why is None)
        if not ran:
            said = gpu._lib.aionhip_last_error(gpu._ctx).decode()
            assert "attention_matmul" in said and why in said, said
            assert (gpu.download(c[1], np.float32, (rows, n)) == 0.25).all()
        else:
            gpu.step_attention(out, q, k, v, shape, d ** -0.5, **kw)
            gpu.step_matmul(w, out, rows, c[0], beta=1.0)
            want, got = (gpu.download(x, np.float32, (rows, n)) for x in c)
            assert np.array_equal(want.view(np.uint32), got.view(np.uint32))
            if options.get("unseen"):
                assert (got.reshape(b, s, n)[1] == 0.25).all() and (got.reshape(b, s, n)[0] != 0.25).any()
    finally:
        gpu.set_attention_precise(False)
    for x in (q, k, v, pos, lens, w, out, *c):
        x.free()


# A context whose scratch memory has grown for the two calls only: in a recording the GeGLU block of many rows, which needs both prepared forms at
# once, is refused as unsupported with nothing recorded, and the two calls are recorded in its place.
def test_geglu_block_in_a_recording_leaves_scratch_as_it_is(gpu):
    del gpu                                                     # (its scratch has long grown)
    own = be.HipBackend(0)
    try:
        rng = np.random.default_rng(3)
        rows, k = 64, 2048
        wg, wu, wd = (make_weight(own, be.Q8_0, be.ROWS_NK, k, k, seed=s)[1] for s in range(3))
        x, gamma = own.upload(rng.standard_normal((rows, k)).astype(np.float32)), own.upload(np.ones(k, np.float32))
        gate, up, c = (own.alloc(4 * rows * k) for _ in range(3))

        def two_calls():
            own.step_rmsnorm_matmul([wg, wu], x, gamma, rows, [gate, up], 1e-6)
            own.step_gate_matmul(wd, gate, up, rows, c)

        two_calls()
        want = own.download(c, np.uint32, (rows, k))
        ran = []

        def block():
            ran.append(own.step_rmsnorm_geglu_matmul_rows(wg, wu, wd, x, gamma, rows, 1e-6, c))
            if not ran[-1]:
                two_calls()

        for expected in (False, True):
            prog = own.record_program(block)
            assert ran == [expected]
            for _ in range(3):
                own.write(c, np.zeros((rows, k), np.float32))
                own.program_execute(prog)
                assert np.array_equal(own.download(c, np.uint32, (rows, k)), want)
            own.program_destroy(prog)
            assert own.step_rmsnorm_geglu_matmul_rows(wg, wu, wd, x, gamma, rows, 1e-6, c)      # eagerly: it grows the scratch
            ran.clear()
    finally:
        own.close()


# The same where products of scales are subnormal (weight scales of 2^-4 .. 2^-9 times row scales down to 2^-135) and where sums cross into them:
# the matrix pipe's products of scales are the multiply's there too.
@pytest.mark.parametrize("dtype,layout", CASES)
@pytest.mark.parametrize("m,n,k", [(512, 4096, 2048), (77, 11008, 672), (300, 5000, 1056), (90, 2100, 4096)])
def test_exact_gemm_scale_products_keep_their_bits_below_the_normal_range(gpu, orc, dtype, layout, m, n, k):
    say("subnormal scale products", dtype, layout, m, n, k)
    gpu.set_gemm_mode(be.GEMM_EXACT_I8)
    _, w = make_weight(gpu, dtype, layout, n, k, seed=m + k)
    rng = np.random.default_rng(k + 1)
    a = np.zeros((m, k // 32, 32), np.float32)
    at = np.arange(m) * 7 % (k // 32)
    a[np.arange(m), at] = rng.standard_normal((m, 32)) * 2.0 ** rng.integers(-135, -110, (m, 1))
    a = a.reshape(m, k)
    got = gpu.matmul(w, a)
    assert "gemm_i8" in gpu.last_launch()["kernel"]
    assert ((np.abs(got) < 2.0 ** -126) & (got != 0)).mean() > 0.05 and (np.abs(got) > 2.0 ** -126).mean() > 0.05
    for rows in ([0, 1, m // 2, m - 1, *rng.integers(0, m, 8)], rng.integers(0, m, 12)):
        assert np.array_equal(got[rows].view(np.uint32), gpu.matmul(w, a[rows]).view(np.uint32)), rows
        assert "gemm_i8" in gpu.last_launch()["kernel"]
    w.free()


# bf16 mode between the two kernels: the exact one is the faster of the two up to a few hundred rows (256 x 8192 x 2048 21 against 29 us), the bf16 one
# beyond (512 x 14336 x 4096 73 against 98)
@pytest.mark.parametrize("m,n,k,kernel", [(256, 8192, 2048, "gemm_i8_q4"), (512, 14336, 4096, "gemm_bf16")])
def test_bf16_mode_chooses_the_faster_kernel_at_a_few_hundred_rows(gpu, m, n, k, kernel):
    _, w = make_weight(gpu, be.Q4_0, be.KMAJOR_KN, n, k, seed=m)
    gpu.set_gemm_mode(be.GEMM_BF16_MFMA)
    try:
        gpu.matmul(w, np.random.default_rng(m).standard_normal((m, k)).astype(np.float32))
        assert gpu.last_kernel() == kernel
    finally:
        gpu.set_gemm_mode(be.GEMM_EXACT_I8)
        w.free()

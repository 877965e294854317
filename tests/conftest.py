import os
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs a real MI355X (run with -m gpu on the GPU box)")


@pytest.fixture(scope="session")
def orc():
    from oracle import oracle
    return oracle


@pytest.fixture(scope="session")
def gpu():
    """One device context for the whole GPU session (tests marked `gpu` only)."""
    from aion_amd.backend import HipBackend
    b = HipBackend(0)
    yield b
    b.close()


def norm_err(got, ref):
    """max |err| / max(|ref|, 1e-3 * rms(ref)): elementwise relative error with a floor, since an
    output that is a sum of +- terms can sit arbitrarily close to zero."""
    import numpy as np
    got = np.asarray(got, dtype=np.float64)
    ref = np.asarray(ref, dtype=np.float64)
    rms = float(np.sqrt((ref ** 2).mean())) if ref.size else 0.0
    den = np.maximum(np.abs(ref), 1e-3 * rms + 1e-30)
    return float((np.abs(got - ref) / den).max()) if ref.size else 0.0


def rms_err(got, ref):
    """max |err| / rms(ref)"""
    import numpy as np
    got = np.asarray(got, dtype=np.float64)
    ref = np.asarray(ref, dtype=np.float64)
    rms = float(np.sqrt((ref ** 2).mean())) if ref.size else 0.0
    return float(np.abs(got - ref).max() / (rms + 1e-30)) if ref.size else 0.0


def _row_err(got, ref, norm):
    import numpy as np
    got = np.asarray(got, dtype=np.float64)
    ref = np.asarray(ref, dtype=np.float64)
    if ref.size == 0:
        return 0.0
    den = norm(ref)
    err = np.abs(got - ref).max(axis=-1)
    rel = np.where(den > 0, err / np.where(den > 0, den, 1.0), np.where(err > 0, np.inf, 0.0))
    return float(rel.max())


def row_rel_err(got, ref):
    """Attention's gate: the max relative error of every output row (last axis = one head's values for one query) in
    the maximum norm, max |err| / max |ref row|, worst row. An attention output is an average of values, so its size
    shrinks with the number of visible keys; an absolute bound that fits a row seeing one key says nothing about a row
    seeing 16384. A row whose reference is all zeros (empty window) must be all zeros."""
    import numpy as np
    return _row_err(got, ref, lambda r: np.abs(r).max(axis=-1))


def row_rms_err(got, ref):
    """The same per row against the row's rms (2.5 to 3 times smaller than its largest element): max |err| / rms(ref row)"""
    import numpy as np
    return _row_err(got, ref, lambda r: np.sqrt((r ** 2).mean(axis=-1)))


def slim_rows(q8, m, n, k):
    """Whether gemv_slim_kernel takes 2..8 rows against an [n, k] weight of few rows (256 CUs)"""
    tiles = -(-n // 16)
    if k % 128 or not 512 <= k <= 1 << 26 or tiles > 768:
        return False
    return m > 2 or k > 4096 if m <= 4 else k <= 16384 and (q8 or not 256 < tiles <= 512)


def few_rows_on_gemm(q8, m, n, k):
    """Whether 2..8 rows against an [n, k] weight by itself run on the exact GEMM's kernel under the GEMV's name (256 CUs; not asked for five rows
    and more over a K past 4096, nor for what the matrix-pipe GEMV takes)"""
    if k < 256 or k > 1 << 26:
        return False
    if m >= 5:
        return n >= max(1024, k) and not (n > 8192 and k >= 2048 and slim_rows(q8, m, n, k))
    between = q8 and n > 8192 and (k <= 5120 or (2 if m == 2 else 4) * 40 * (k // 32) * 3 > 160 * 1024)
    upper = (16384 if m == 2 and k > 8192 else 32768) if q8 else (24576 if m >= 3 else 16384 if k >= 4096 else 0)
    return (7680 < n <= 8192 or n >= 12288 or between) and n <= upper and n * k <= 1 << 28


def rows_kernel(q8, m, n, k):
    """The kernel 2..8 activation rows against an [n, k] weight run on (what aionhip_last_kernel reports), for 256 CUs: for many weight rows and a
    K of 1024..4096 in whole 256-code stages (q4: from 14336 rows at 5..8 activation rows - 49152 below K = 2048 -, from 65536 at 3..4; q8:
    from 65536 rows, at 3..4 activation rows from K = 2048 on and up to 300 M weights) the matrix-pipe GEMV or, q4 up to 24576 rows from
    K = 2048 on, the slim one; for 5..8 rows over a K past 4096 the slim GEMV or the exact GEMM; else the exact GEMM's kernel under the
    vector-ALU rows kernel's name, the slim GEMV, or that rows kernel."""
    tag = "q8" if q8 else "q4"
    if 3 <= m <= 8 and 1024 <= k <= 4096 and k % 256 == 0:
        if not q8 and n >= (65536 if m < 5 else 49152 if k < 2048 else 14336):
            return "gemv_q4_slim" if m >= 5 and k >= 2048 and n <= 24576 else "gemv_q4_mfma"
        if q8 and n >= 65536 and (m >= 5 or (k >= 2048 and n * k <= 300_000_000)):
            return "gemv_q8_mfma"
    if m >= 5 and 4096 < k <= 1 << 26:
        return "gemv_%s_slim" % tag if slim_rows(q8, m, n, k) else "gemm_i8_" + tag
    return "gemv_%s_slim" % tag if slim_rows(q8, m, n, k) and not few_rows_on_gemm(q8, m, n, k) else "gemv_" + tag

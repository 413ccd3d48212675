"""Decode projections with a LoRA term (the GEMV kernels' LoRA forms) against the double oracle.

Every kernel form of one and two rows at both ends of its range of K (one and two lane slots, each K-split), ranks
1 to 64 on either side of a round of eight, columns that end inside a wavefront's run, fewer columns than one
run. The base sum is exact per group and T is fp32 over
at most 128 values, then double: the LoRA bar of the other kernels, 1e-5.
"""
from __future__ import annotations

import numpy as np
import pytest

from cases import lora_factors, make_case
from test_gpu_digit_tiles import note, run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,n,k,rank", [(1, 4096, 2048, 16), (1, 1, 1056, 8), (1, 70, 1056, 40), (1, 999, 2080, 5), (1, 14336, 4096, 16),
                                        (1, 1025, 4128, 7), (1, 333, 8192, 64), (1, 500, 8224, 9), (1, 77, 12288, 17),
                                        (1, 130, 16384, 8), (1, 65, 16416, 4), (1, 300, 32768, 16),
                                        (2, 5, 2048, 3), (2, 2049, 2080, 32), (2, 8200, 4096, 16), (2, 301, 4128, 8),
                                        (2, 90, 8224, 33), (2, 513, 12320, 16), (2, 40, 16384, 1)])
def test_shapes(session, oracle, gpu, m, n, k, rank):
    import torch

    note(f"gemv lora {m}x{n}x{k} r={rank}")
    c = make_case(m, n, k)
    la, lb = lora_factors(k, n, rank)
    got = run(session, torch, c, (la, lb), 2.0)
    rep = oracle.compare(got, oracle.q4gemm_lora(c.x, c.packed, c.scales, la, lb, 2.0, threads=8), 1e-5)
    note(f"max rel {rep['max_relative_error']:.2e}")
    assert rep["status"] == "pass", rep
    # a zero adapter leaves the plain call's bits
    assert np.array_equal(run(session, torch, c, (la, np.zeros_like(lb)), 2.0), run(session, torch, c))


@pytest.mark.parametrize("m,k", [(1, 4096), (1, 8192), (2, 2048), (2, 11008)])
def test_nonfinite_x_follows_ieee(session, oracle, gpu, m, k):
    import torch

    note(f"gemv lora non-finite {m}x{k}")
    c = make_case(m, 150, k)
    la, lb = lora_factors(k, 150, 8)
    for value, at in ((np.nan, 5), (np.inf, k - 1), (-np.inf, k // 2)):
        c.x[m - 1] = 0.5
        c.x[m - 1, at] = value
        got = run(session, torch, c, (la, lb), 2.0)
        with np.errstate(invalid="ignore"):
            ref = oracle.q4gemm_lora(c.x, c.packed, c.scales, la, lb, 2.0, threads=8)
        assert np.array_equal(np.isnan(got), np.isnan(ref)) and np.array_equal(np.isposinf(got), np.isposinf(ref)), value
        ok = np.isfinite(ref)
        assert np.array_equal(ok, np.isfinite(got)) and ok.sum() == 150 * (m - 1)
        assert np.all(np.abs(got[ok] - ref[ok]) <= 1e-5 * np.maximum(1, np.abs(ref[ok])))

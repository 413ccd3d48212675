"""The digit GEMM with several column tiles per workgroup (q4_gemm_tiles_kernel) at its edges.

Against the double oracle. The group sums are exact, x is held to 2^-30 of its group's largest
magnitude and y is rounded once, so the bar is that of the calls up to 32 rows, 2e-7 on x in [-1, 1)
and scales in [0.5, 1.5), also above 32 rows. The shapes cover each count of column tiles per
workgroup (1 to 6 and 8; 256 CUs), 1, 2 and 4 result rows per lane, ragged row blocks and tiles, one to
many chunks of four groups with a last chunk of one to four, odd and even chunks per wavefront, and
the 16- and 4-wavefront forms that keep a short K above 32 rows.
"""
from __future__ import annotations

import numpy as np
import pytest

from cases import lora_factors, make_case

pytestmark = pytest.mark.gpu

BAR = 2e-7

# m, n, k
SHAPES = [(5, 33, 544), (8, 8193, 544), (7, 8225, 1056), (2, 16400, 1120), (4, 24590, 640), (3, 16385, 2080),
          (9, 12300, 608), (24, 11001, 512), (13, 20481, 576), (32, 14336, 1504), (33, 97, 64), (40, 300, 1056),
          (77, 7001, 96), (100, 301, 4128), (129, 1030, 2048), (36, 100, 16416), (511, 65, 736), (1000, 100, 512)]


def note(msg: str) -> None:
    print(f"[gpu-case] {msg}", flush=True)


def run(session, torch, c, lora=None, scale=0.0):
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to("cuda:0")  # noqa: E731
    x, w, s = t(c.x), t(c.packed), t(c.scales)
    y = torch.full((c.m, c.n), float("nan"), dtype=torch.float32, device="cuda:0")
    st = torch.cuda.current_stream()
    if lora is None:
        session.q4gemm_device(x.data_ptr(), w.data_ptr(), s.data_ptr(), y.data_ptr(), c.m, c.n, c.k, st.cuda_stream)
    else:
        la, lb = t(lora[0]), t(lora[1])
        session.q4gemm_lora_device(x.data_ptr(), w.data_ptr(), s.data_ptr(), la.data_ptr(), lb.data_ptr(),
                                   y.data_ptr(), c.m, c.n, c.k, lora[0].shape[1], scale, st.cuda_stream)
    st.synchronize()
    return y.cpu().numpy()


@pytest.mark.parametrize("m,n,k", SHAPES)
def test_shapes(session, oracle, gpu, m, n, k):
    import torch

    note(f"digit tiles {m}x{n}x{k}")
    c = make_case(m, n, k, x_dist="uniform", x_range=(-1.0, 1.0), scale_range=(0.5, 1.5))
    rep = oracle.compare(run(session, torch, c), oracle.q4gemm_packed(c.x, c.packed, c.scales, threads=8), BAR)
    note(f"max_rel={rep['max_relative_error']:.3e}")
    assert rep["status"] == "pass", rep


@pytest.mark.parametrize("m,n,k,rank", [(40, 300, 1056, 5), (9, 9000, 544, 64), (128, 192, 64, 24), (100, 1030, 1024, 16),
                                        # T in the kernel: 16, 8 and 4 wavefronts, uneven slices, a slice past
                                        # the last run, one and 64 ranks, and the first K past it
                                        (3, 40, 32, 1), (61, 70, 224, 11), (128, 64, 64, 64), (70, 1500, 96, 3),
                                        (130, 3000, 64, 5), (17, 50, 416, 8), (17, 50, 544, 8)])
def test_lora(session, oracle, gpu, m, n, k, rank):
    import torch

    note(f"digit tiles lora {m}x{n}x{k} r={rank}")
    c = make_case(m, n, k)
    la, lb = lora_factors(k, n, rank)
    rep = oracle.compare(run(session, torch, c, (la, lb), 2.0),
                         oracle.q4gemm_lora(c.x, c.packed, c.scales, la, lb, 2.0, threads=8), 1e-5)
    assert rep["status"] == "pass", rep


def test_groups_past_k_and_nonfinite_rows(session, oracle, gpu):
    """K = 1056 leaves one live group in the last chunk, whose copies also bring the next row's values and
    the next column's scales: non-finite ones there must not reach this row or column. Rows with an
    infinity or a NaN follow IEEE arithmetic, as the oracle does; the others meet the bar. The column with
    the infinite scale itself is not compared (a group's sum meets its scale once, not term by term)."""
    import torch

    m, n, k = 60, 300, 1056
    note(f"digit tiles non-finite {m}x{n}x{k}")
    c = make_case(m, n, k, x_dist="uniform", x_range=(-1.0, 1.0), scale_range=(0.5, 1.5))
    c.x[3, 0] = np.inf       # read by row 2's last chunk
    c.x[17, 40] = np.nan
    c.x[40, 1055], c.x[40, 1] = -np.inf, np.inf
    c.scales[7, 0] = np.inf  # read by column 6's last chunk
    keep = np.delete(np.arange(n), 7)
    got = run(session, torch, c).astype(np.float64)[:, keep]
    with np.errstate(invalid="ignore"):
        ref = oracle.q4gemm_packed(c.x, c.packed, c.scales, threads=8)[:, keep]
    finite = np.isfinite(ref)
    assert np.array_equal(np.isfinite(got), finite)
    assert np.array_equal(np.isnan(got), np.isnan(ref)) and np.array_equal(np.isposinf(got), np.isposinf(ref))
    assert np.max(np.abs(got[finite] - ref[finite]) / np.maximum(1.0, np.abs(ref[finite]))) <= BAR
    assert np.all(finite[np.delete(np.arange(m), [3, 17, 40])])


@pytest.mark.parametrize("m,n,k", [(200, 1024, 14336), (128, 14336, 512), (256, 4096, 2048), (64, 14400, 1024)])
def test_limb_gemms_keep_their_shapes(session, oracle, gpu, m, n, k):
    """Shapes that stay on the limb GEMMs (K-split and single wide grids, the mid-size tiles), on two streams
    through the shared workspace: each stream's result against the oracle."""
    import torch

    note(f"limb GEMMs {m}x{n}x{k}")
    cs = [make_case(m, n, k, seed_a=0x500 + i) for i in range(2)]
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to("cuda:0")  # noqa: E731
    x, w, s = [t(c.x) for c in cs], t(cs[0].packed), t(cs[0].scales)
    ys = [torch.empty((m, n), dtype=torch.float32, device="cuda:0") for _ in range(2)]
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    torch.cuda.synchronize()
    for _ in range(3):
        for i in range(2):
            session.q4gemm_device(x[i].data_ptr(), w.data_ptr(), s.data_ptr(), ys[i].data_ptr(), m, n, k,
                                  streams[i].cuda_stream)
    torch.cuda.synchronize()
    for i in range(2):
        ref = oracle.q4gemm_packed(cs[i].x, cs[i].packed, cs[i].scales, threads=8)
        rep = oracle.compare(ys[i].cpu().numpy(), ref, 1e-5)
        assert rep["status"] == "pass", rep

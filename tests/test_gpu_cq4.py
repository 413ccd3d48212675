"""GPU parity of the CQ4 codebook matmul (spaceslug_cq4_matmul[_device]) against the CPU oracle.

Bar: every fp16 output within half an fp16 spacing of the exact (double) result plus
1e-5 * max(1, |ref|) for the fp32 arithmetic: |fp16(gpu) - ref| <= spacing(ref)/2 +
1e-5 max(1, |ref|). That is the fp16 rounding of the result and nothing more. The
reference's own test bar (|d| <= 2e-2 or <= 1e-2 |ref|, test_cq4.cpp:422) is checked
too, and where the reference's library is built (oracle/_ref) its outputs are compared
with the same bar. Cases: the reference test's five fixtures, rebuilt from its
generators, and random matrices of every bit width, layout and transform option.
"""
from __future__ import annotations

import numpy as np
import pytest

from oracle import cq4

pytestmark = pytest.mark.gpu

FIXTURES = ["cq4_interleaved", "cq4_hadamard_signs", "cq4_orthogonal", "cq4_interleaved_multigroup_m1",
            "cq4_interleaved_m1_n512"]


def note(msg: str) -> None:
    print(f"[gpu-case] {msg}", flush=True)


def within_fp16_rounding(got_bits: np.ndarray, ref: np.ndarray) -> tuple[bool, float]:
    g = np.asarray(got_bits, np.uint16).view(np.float16).astype(np.float64)
    _, e = np.frexp(np.maximum(np.abs(ref), 2.0 ** -14))
    spacing = np.ldexp(1.0, e - 11)
    excess = np.abs(g - ref) - (0.5 * spacing + 1e-5 * np.maximum(1.0, np.abs(ref)))
    return bool(np.all(excess <= 0)), float(np.max(np.abs(g - ref) / np.maximum(1.0, np.abs(ref))))


def run(session, W: cq4.CQ4Matrix, A: np.ndarray, M: int) -> np.ndarray:
    return session.cq4_matmul_values(bits=W.bits, K=W.K, N=W.N, group_size=W.group_size, num_groups=W.num_groups,
                                     flags=W.flags, codebook=W.codebook, norms=W.norms,
                                     packed_indices=W.packed_indices, a=A, m=M, input_scale=W.input_scale,
                                     input_scale_recip=W.input_scale_recip, left_signs=W.left_signs,
                                     right_signs=W.right_signs, permutation=W.permutation, rotation=W.rotation)


def check(session, W, A, M, label):
    got = run(session, W, A, M)
    ref = cq4.matmul(W, A, M)
    ok, rel = within_fp16_rounding(got, ref)
    note(f"{label}: max |d|/max(1,|ref|) = {rel:.3e}")
    assert ok, label
    g = got.view(np.float16).astype(np.float64)
    assert np.all((np.abs(g - ref) <= 2e-2) | (np.abs(g - ref) <= 1e-2 * np.abs(ref)))
    if cq4.reference_available():
        r16 = cq4.reference_matmul(W, A, M)
        # the reference rounds its own fp32 sum: the two fp16 results agree to within a spacing or two
        ok_ref, _ = within_fp16_rounding(r16, g)
        assert np.mean(r16 == got) >= 0.97 or ok_ref, label
    return got


@pytest.mark.parametrize("name", FIXTURES)
def test_reference_fixtures(session, gpu, name):
    W, A, M = cq4.reference_fixture(name)
    check(session, W, A, M, name)


CASES = [dict(bits=4, K=256, N=24, group_size=64, signs=True, perm=True, scale="scale", m=7),
         dict(bits=4, K=512, N=40, group_size=128, m=4),
         dict(bits=4, K=96, N=12, group_size=32, signs=True, m=3),
         dict(bits=3, K=256, N=20, group_size=128, signs=True, m=5),
         dict(bits=2, K=128, N=12, group_size=32, perm=True, m=9),
         dict(bits=1, K=64, N=8, group_size=64, scale="none", m=2),
         dict(bits=4, K=1024, N=64, group_size=256, signs=True, perm=True, m=1),
         dict(bits=4, K=512, N=36, group_size=128, interleaved=True, m=6),
         dict(bits=4, K=128, N=8, group_size=128, interleaved=True, orthogonal=True, m=4),
         dict(bits=4, K=96, N=8, group_size=96, orthogonal=True, m=2),
         dict(bits=3, K=64, N=8, group_size=64, orthogonal=True, scale="none", m=5),
         dict(bits=4, K=64, N=16, group_size=2, m=3),
         dict(bits=4, K=16, N=4, group_size=1, m=2),
         # M <= 4: transform and GEMV in one launch up to 4096 values of M x K, two launches beyond
         dict(bits=4, K=256, N=20, group_size=64, interleaved=True, signs=True, perm=True, scale="scale", m=2),
         dict(bits=4, K=2048, N=12, group_size=16, interleaved=True, m=2),
         dict(bits=4, K=4096, N=12, group_size=128, interleaved=True, m=1),
         dict(bits=4, K=2048, N=24, group_size=128, signs=True, perm=True, m=3)]


@pytest.mark.parametrize("case", range(len(CASES)))
def test_random_matrices(session, gpu, case):
    kw = dict(CASES[case])
    m = kw.pop("m")
    rng = np.random.default_rng(500 + case)
    W = cq4.random_matrix(rng, **kw)
    A = cq4.f16(rng.uniform(-1, 1, (m, W.K)))
    check(session, W, A, m, f"random {CASES[case]}")


# M >= 32 with 4-bit LSB-packed indices, group sizes that are multiples of 32 and K % 64 == 0 run
# on the MFMA kernel: ragged row and column tiles, one to several groups per row, signs,
# permutation, both input-scale forms, the orthogonal basis, and the reference benchmark's 1024^3
# shape; K = 96 (not a multiple of 64) at M = 48 stays on the other kernel. K = 768 and 320 end
# rows with a partial 512-value chunk of the vector transform. Up to 128 norm groups
# per column the pipelined MFMA kernel runs, beyond that the single-stage one.
MFMA_CASES = [dict(bits=4, K=512, N=200, group_size=128, m=70),
              dict(bits=4, K=96, N=50, group_size=32, m=48),
              dict(bits=4, K=1024, N=96, group_size=256, signs=True, perm=True, scale="scale", m=33),
              dict(bits=4, K=128, N=72, group_size=128, orthogonal=True, m=40),
              dict(bits=4, K=256, N=130, group_size=32, m=64),
              dict(bits=4, K=512, N=64, group_size=64, scale="none", m=129),
              dict(bits=4, K=1024, N=1024, group_size=128, m=1024),
              dict(bits=4, K=768, N=100, group_size=128, signs=True, perm=True, m=40),  # K % 512 != 0
              dict(bits=4, K=320, N=64, group_size=64, signs=True, scale="scale", m=35),
              dict(bits=4, K=320, N=70, group_size=64, signs=True, scale="scale", m=500),
              dict(bits=4, K=1024, N=96, group_size=256, signs=True, perm=True, scale="scale", m=512),
              dict(bits=4, K=4096, N=72, group_size=32, m=40),    # 128 norm groups: the most held in LDS
              dict(bits=4, K=8192, N=40, group_size=32, m=36),    # 256 groups: the single-stage kernel
              dict(bits=4, K=64, N=80, group_size=64, m=40),      # one 64-value stage: every copy clamped
              dict(bits=4, K=64, N=64, group_size=32, signs=True, scale="scale", m=64),
              dict(bits=4, K=128, N=136, group_size=128, perm=True, m=97)]  # two stages, one stage pair


@pytest.mark.parametrize("case", range(len(MFMA_CASES)))
def test_random_matrices_mfma(session, gpu, case):
    kw = dict(MFMA_CASES[case])
    m = kw.pop("m")
    rng = np.random.default_rng(900 + case)
    W = cq4.random_matrix(rng, **kw)
    A = cq4.f16(rng.uniform(-1, 1, (m, W.K)))
    check(session, W, A, m, f"mfma {MFMA_CASES[case]} m={m}")


def device_struct(W, keep: dict):
    """The matrix's arrays copied to cuda:0 (kept alive in `keep`) and its CQ4MatrixStruct."""
    import torch

    from spaceslug_amd.backend import CQ4MatrixStruct

    def d(name):
        a = getattr(W, name)
        if a is None:
            return None
        t = torch.from_numpy(np.ascontiguousarray(a).view(np.uint8).copy()).to("cuda:0")
        keep[name] = t
        return t.data_ptr()

    return CQ4MatrixStruct(W.bits, W.K, W.N, W.group_size, W.num_groups, W.flags, *(d(n) for n in cq4.ARRAYS),
                           None, None)


def run_device(session, s, a_ptr: int, M: int, N: int) -> np.ndarray:
    import torch

    c_t = torch.empty((M, N), dtype=torch.int16, device="cuda:0")
    st = torch.cuda.current_stream()
    session.cq4_matmul_device(s, a_ptr, M, c_t.data_ptr(), st.cuda_stream)
    st.synchronize()
    return c_t.cpu().numpy().view(np.uint16)


def test_device_entry_equals_host_entry(session, gpu):
    import torch

    note("cq4 device entry")
    W, A, M = cq4.reference_fixture("cq4_hadamard_signs")
    host = run(session, W, A, M)
    keep = {}
    s = device_struct(W, keep)
    a_t = torch.from_numpy(A.view(np.int16).copy()).to("cuda:0")
    assert np.array_equal(run_device(session, s, a_t.data_ptr(), M, W.N), host)


@pytest.mark.parametrize("gs,M", [(64, 40), (128, 40), (256, 40), (128, 500), (256, 1000)])
def test_transform_kernels_agree(session, gpu, gs, M):
    """On the MFMA path the Hadamard transform runs as 16-byte vector loads and limb stores when the
    activations are 16-byte aligned, and one wavefront per (row, group) otherwise (here: a pointer one
    element into an allocation). Both perform the same operations in the same order, so the products
    are bitwise equal."""
    import torch

    note(f"cq4 transform kernels agree gs={gs} M={M}")
    rng = np.random.default_rng(70 + gs + M)
    W = cq4.random_matrix(rng, bits=4, K=768, N=80, group_size=gs, signs=True, perm=True, scale="scale")
    A = cq4.f16(rng.uniform(-1, 1, (M, W.K)))
    keep = {}
    s = device_struct(W, keep)
    a_t = torch.from_numpy(A.view(np.int16).copy()).to("cuda:0")
    buf = torch.zeros(M * W.K + 1, dtype=torch.int16, device="cuda:0")
    buf[1:] = a_t.reshape(-1)
    aligned = run_device(session, s, a_t.data_ptr(), M, W.N)
    shifted = run_device(session, s, buf.data_ptr() + 2, M, W.N)
    assert np.array_equal(aligned, shifted)
    ok, _ = within_fp16_rounding(aligned, cq4.matmul(W, A, M))
    assert ok


def test_device_calls_in_a_row(session, gpu):
    """Three device calls in a row at 1024 x 1024 x 1024 on the shared workspace, with different
    activations: each matches the host entry bit for bit and the oracle to the fp16 bar (a call that
    read a stale part of the workspace would carry the previous call's activations)."""
    import torch

    note("cq4 device entry: three calls in a row")
    rng = np.random.default_rng(4242)
    W = cq4.random_matrix(rng, bits=4, K=1024, N=1024, group_size=128)
    M = 1024
    keep = {}
    s = device_struct(W, keep)
    for call in range(3):
        A = cq4.f16(rng.uniform(-1, 1, (M, W.K)))
        a_t = torch.from_numpy(A.view(np.int16).copy()).to("cuda:0")
        dev = run_device(session, s, a_t.data_ptr(), M, W.N)
        assert np.array_equal(dev, run(session, W, A, M)), call
        ok, _ = within_fp16_rounding(dev, cq4.matmul(W, A, M))
        assert ok, call


def test_decode_call_in_a_hip_graph(session, gpu):
    """A decode call (1 x 512 x 512, the reference benchmark's decode shape: one launch, no workspace)
    captured once in a HIP graph and replayed with new activations: every replay equals the eager call
    bit for bit and the oracle to the fp16 bar. A call that needs the workspace (M = 64) is refused
    under capture, and the capture still ends cleanly."""
    import ctypes

    import torch

    note("cq4 decode call in a HIP graph")
    rng = np.random.default_rng(777)
    W = cq4.random_matrix(rng, bits=4, K=512, N=512, group_size=128, signs=True, perm=True, scale="scale")
    keep = {}
    s = device_struct(W, keep)
    a_t = torch.zeros((1, W.K), dtype=torch.int16, device="cuda:0")
    c_t = torch.zeros((1, W.N), dtype=torch.int16, device="cuda:0")
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        session.cq4_matmul_device(s, a_t.data_ptr(), 1, c_t.data_ptr(), side.cuda_stream)  # warm-up
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        session.cq4_matmul_device(s, a_t.data_ptr(), 1, c_t.data_ptr(), torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    for rep in range(3):
        A = cq4.f16(rng.uniform(-1, 1, (1, W.K)))
        a_t.copy_(torch.from_numpy(A.view(np.int16).copy()).to("cuda:0"))
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        got = c_t.cpu().numpy().view(np.uint16).copy()
        eager = run_device(session, s, a_t.data_ptr(), 1, W.N)
        assert np.array_equal(got, eager), f"replay {rep} differs from the eager call"
        ok, _ = within_fp16_rounding(got, cq4.matmul(W, A, 1))
        assert ok, rep

    M = 64
    a64 = torch.zeros((M, W.K), dtype=torch.int16, device="cuda:0")
    c64 = torch.zeros((M, W.N), dtype=torch.int16, device="cuda:0")
    lib = session._native()
    g2 = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g2, stream=side):
        c64.add_(1)
        rc = lib.spaceslug_cq4_matmul_device(ctypes.addressof(s), ctypes.c_void_p(a64.data_ptr()), M,
                                             ctypes.c_void_p(c64.data_ptr()), ctypes.c_void_p(side.cuda_stream))
    assert rc == -4
    assert b"workspace" in lib.spaceslug_last_error()
    g2.replay()
    torch.cuda.synchronize()
    assert torch.all(c64 == 1)


# The batch kernel: steps of 32 values dealt in quads to 4, 8 or 16 wavefronts (odd quad counts, a
# last quad of one to three steps with groups of 32 and 64), one, two and four 16-row blocks with
# ragged rows, ragged 16-column tiles, panels, K % 64 != 0, and 1- to 3-bit indices expanded first.
BATCH_CASES = [dict(bits=4, K=8192, N=20, group_size=128, m=1),
               dict(bits=4, K=2176, N=33, group_size=128, signs=True, perm=True, scale="scale", m=16),
               dict(bits=4, K=320, N=17, group_size=64, perm=True, m=5),
               dict(bits=4, K=32, N=1, group_size=32, signs=True, m=6),
               dict(bits=4, K=1248, N=50, group_size=32, signs=True, scale="scale", m=17),
               dict(bits=4, K=96, N=40, group_size=32, m=70),
               dict(bits=4, K=2048, N=36, group_size=256, interleaved=True, signs=True, perm=True, m=31),
               dict(bits=4, K=1120, N=20, group_size=32, interleaved=True, m=8),
               dict(bits=4, K=384, N=68, group_size=128, interleaved=True, scale="none", m=129),
               dict(bits=4, K=160, N=24, group_size=160, interleaved=True, orthogonal=True, m=9),
               dict(bits=4, K=192, N=24, group_size=192, orthogonal=True, m=3),
               dict(bits=3, K=768, N=37, group_size=128, signs=True, m=40),
               dict(bits=2, K=512, N=18, group_size=64, m=4),
               dict(bits=1, K=96, N=21, group_size=32, m=33)]


@pytest.mark.parametrize("case", range(len(BATCH_CASES)))
def test_random_matrices_batch(session, gpu, case):
    kw = dict(BATCH_CASES[case])
    m = kw.pop("m")
    rng = np.random.default_rng(1300 + case)
    W = cq4.random_matrix(rng, **kw)
    A = cq4.f16(rng.uniform(-1, 1, (m, W.K)))
    check(session, W, A, m, f"batch {BATCH_CASES[case]} m={m}")


@pytest.mark.parametrize("interleaved,K,gs,m", [(False, 256, 64, 6), (True, 256, 128, 6), (False, 128, 128, 20)])
def test_batch_nonfinite_follows_ieee(session, gpu, interleaved, K, gs, m):
    """Infinities and NaNs in the activations, a norm or the codebook: the batch kernel's limb products
    cannot carry them, so every output's class (finite, +inf, -inf, NaN) is compared with double
    arithmetic on the code-basis activations, which the Hadamard transform spreads over a group."""
    rng = np.random.default_rng(41)
    W = cq4.random_matrix(rng, bits=4, K=K, N=20, group_size=gs, interleaved=interleaved, signs=True)
    W.codebook[3], W.codebook[9] = cq4.f16(np.array([0.0, -0.5]))  # a zero entry: inf * 0 is NaN
    A = cq4.f16(rng.uniform(-1, 1, (m, K)))
    A[1, 5] = 0x7C00            # +inf
    A[2, 70 % K] = 0xFC00       # -inf
    A[3, 1] = 0x7E00            # NaN
    A[4, 2], A[4, 3] = 0x7C00, 0xFC00
    for code in (None, 7):      # then also an infinite codebook entry
        if code is not None:
            W.codebook[code] = 0x7C00
        got = run(session, W, A, m).view(np.float16).astype(np.float64)
        with np.errstate(invalid="ignore"):
            ref = cq4.matmul(W, A, m)
        assert np.array_equal(np.isnan(got), np.isnan(ref)), code
        assert np.array_equal(np.isposinf(got), np.isposinf(ref)), code
        assert np.array_equal(np.isneginf(got), np.isneginf(ref)), code
        ok = np.isfinite(ref)
        assert ok.any() == (code is None)
        assert np.all(np.abs(got[ok] - ref[ok]) <= 2.0 ** -11 * np.abs(ref[ok]) + 1e-5 * np.maximum(1, np.abs(ref[ok])))


# The rotation on the matrix cores (K % 16 == 0): fewer steps than wavefronts, one and several passes, the
# last pass partly empty, column and row tiles that are ragged or exactly full, every limb layout, both scale
# forms; K = 100 on the other kernel.
@pytest.mark.parametrize("K,m,kw", [(16, 1, {}), (16, 17, dict(scale="none")), (48, 3, {}), (64, 16, dict(interleaved=True)),
                                    (100, 5, {}), (240, 33, dict(scale="scale")), (256, 4, dict(interleaved=True)),
                                    (272, 2, dict(bits=3)), (1008, 6, {}), (1024, 65, dict(interleaved=True)),
                                    (1040, 1, dict(scale="scale")), (2064, 31, {})])
def test_orthogonal_rotation(session, gpu, K, m, kw):
    rng = np.random.default_rng(77 + K)
    W = cq4.random_matrix(rng, **{**dict(bits=4, K=K, N=20, group_size=K, orthogonal=True), **kw})
    A = cq4.f16(rng.uniform(-1, 1, (m, K)))
    check(session, W, A, m, f"orthogonal K={K} m={m} {kw}")


# Decode calls with the transform in the launch: both workgroup sizes (the line at 2560 columns or 3072
# values), every group size, fewer values than one wavefront's 512, rows that end inside them, columns past
# one per wavefront of the grid, panels, permutations, signs; arrays as they are and shifted by one element.
@pytest.mark.parametrize("m,N,K,gs,kw", [(1, 3, 8, 8, dict(signs=True)), (3, 40, 16, 16, dict(signs=True, perm=True)),
                                         (4, 24, 1024, 32, dict(signs=True, interleaved=True)), (2, 2561, 96, 8, dict(scale="scale")),
                                         (1, 2560, 64, 64, dict(signs=True)), (3, 60, 1024, 256, dict(signs=True, perm=True)),
                                         (1, 4101, 520, 8, dict(signs=True)), (2, 8200, 256, 128, dict(signs=True, interleaved=True)),
                                         (3, 52, 1152, 128, dict(signs=True, scale="scale")), (1, 30, 4096, 16, dict(perm=True, scale="none")),
                                         (4, 9000, 128, 64, dict(perm=True, signs=True))])
def test_decode_transform_in_the_launch(session, gpu, m, N, K, gs, kw):
    import torch

    note(f"cq4 decode {m}x{K}->{N} gs={gs} {kw}")
    rng = np.random.default_rng(31 + N + K)
    W = cq4.random_matrix(rng, bits=4, K=K, N=N, group_size=gs, **kw)
    A = cq4.f16(rng.uniform(-1, 1, (m, K)))
    got = check(session, W, A, m, f"decode {m}x{K}->{N}")
    keep = {}
    s = device_struct(W, keep)
    a_t = torch.from_numpy(A.view(np.int16).copy()).to("cuda:0")
    assert np.array_equal(run_device(session, s, a_t.data_ptr(), m, N), got)
    buf = torch.zeros(m * K + 1, dtype=torch.int16, device="cuda:0")
    buf[1:] = a_t.reshape(-1)
    if W.left_signs is not None:
        signs = torch.zeros(gs + 1, dtype=torch.uint8, device="cuda:0")
        signs[1:] = keep["left_signs"]
        s.left_signs = signs.data_ptr() + 1
    assert np.array_equal(run_device(session, s, buf.data_ptr() + 2, m, N), got)

"""GEMV work splits: k ranges of unequal length on the matrix-core row kernel (2..16 rows, with
the hand-off and with the finish kernel), its packed MUL1 operands, and the unsplit single row of
a very wide matrix.  Against the CPU oracle's fp64 linear; bar max|y - ref| / max|ref| < 2e-3 (fp16
rounding of the rotated input and of the output, fp32 sums)."""
import numpy as np
import pytest

from ampstein_amd import synth

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch_cuda():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from ampstein_amd import ops
    ops.init(0)
    return torch


def gemm(torch, L, x):
    from ampstein_amd import ops
    t, s, v = L.torch()
    A = torch.from_numpy(x).cuda()
    C = torch.full((x.shape[0], L.n), float("nan"), dtype=torch.half, device="cuda")
    call = lambda: ops.exl3_gemm(A, t, C, s, torch.empty_like(A), v, 0, L.cb == 1, L.cb == 2)
    assert call() == 90
    return C, call


def check(C, ref, what):
    err = np.abs(C.cpu().numpy().astype(np.float64) - ref).max() / np.abs(ref).max()
    assert err < 2e-3, (what, err)


@pytest.mark.parametrize("m", [2, 3, 4, 5, 7, 8])
@pytest.mark.parametrize("k,n", [(128, 1024), (896, 1024), (1408, 384), (5248, 1024)])
@pytest.mark.parametrize("K,cb", [(4, 0), (3, 1), (5, 2), (2.5, 2)])
def test_rows_ranges(torch_cuda, orc, m, k, n, K, cb):
    """1, 7, 11 and 41 chunks of 128 rows: no divisor but one; odd numbers of (row, chunk) jobs."""
    L = synth.layer(k, n, K, cb, seed=9000 + k + m + int(10 * K))
    x = synth.activations(m, k, seed=9001 + k)
    C, call = gemm(torch_cuda, L, x)
    check(C, orc.linear_f64(x, L.trellis, L.suh, L.svh, int(K), half=K != int(K), cb=cb), (m, k, n, K, cb))
    first = C.clone()
    call()
    assert torch_cuda.equal(first, C)


@pytest.mark.parametrize("K,cb", [(6, 2), (4, 0), (1.5, 2)])
def test_single_row_whole_columns(torch_cuda, orc, K, cb):
    """768 and more column chunks: one workgroup per chunk takes all of k."""
    for n in (98304, 98432):
        L = synth.layer(512, n, K, cb, seed=9100 + int(10 * K))
        x = synth.activations(1, 512, seed=9101)
        C, _ = gemm(torch_cuda, L, x)
        check(C, orc.linear_f64(x, L.trellis, L.suh, L.svh, int(K), half=K != int(K), cb=cb), (n, K, cb))

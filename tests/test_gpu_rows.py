"""The row-tile trellis GEMM (exl3_rows.hip: exl3_gemm from 9 rows to a few hundred) against the
CPU oracle's fp64 linear.  Every test selects the row tiles by policy: at these small sizes exl3_gemm's
own choice for up to 16 rows is the GEMV.  Sizes sit at its edges: row groups of 16 (one row more or less), row
tiles (128 rows), the k split (one 128-k block, fewer blocks than ranges, ranges of unequal
length), the hand-off (n / 128 a multiple of the XCD count) and the finish kernel (not one).
Bar: max|y - ref| / max|ref| < 2e-3, the library's: the rotated input and the output round to
fp16 (2^-11 each, relative to values below the maximum), the sums are fp32."""
import numpy as np
import pytest

from ampstein_amd import _lib, synth

pytestmark = pytest.mark.gpu

TOL = 2e-3


@pytest.fixture(scope="module")
def torch_cuda():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from ampstein_amd import ops
    ops.init(0)
    return torch


@pytest.fixture(autouse=True)
def row_tiles(kernel_policy):
    kernel_policy(_lib.POLICY_GEMM_KERNEL, _lib.GEMM_KERNEL_ROWS)


def run(torch, L, x, fp32=False, suh=True, svh=True):
    from ampstein_amd import ops
    t, s, v = L.torch()
    A = torch.from_numpy(x).cuda()
    A_had = torch.empty_like(A)
    C = torch.full((x.shape[0], L.n), float("nan"), dtype=torch.float if fp32 else torch.half, device="cuda")
    call = lambda: ops.exl3_gemm(A, t, C, s if suh else None, A_had, v if svh else None, 0, L.cb == 1, L.cb == 2)
    tag = call()
    return tag, C, call


def check(C, ref, what):
    y = C.cpu().numpy().astype(np.float64)
    err = np.abs(y - ref).max() / np.abs(ref).max()
    assert err < TOL, (what, err)


@pytest.mark.parametrize("m", [9, 15, 16, 17, 32, 33, 48, 49, 64, 65, 80, 81, 96, 97, 112, 113, 128, 129, 200, 257])
@pytest.mark.parametrize("k,n", [(256, 1024), (640, 384)])
def test_rows_row_counts(torch_cuda, orc, m, k, n):
    L = synth.layer(k, n, 4, 0, seed=7000 + m + n)
    x = synth.activations(m, k, seed=7001 + m)
    tag, C, call = run(torch_cuda, L, x)
    assert tag == (90 if m <= 16 else 91)
    check(C, orc.linear_f64(x, L.trellis, L.suh, L.svh, 4, cb=0), (m, k, n))
    first = C.clone()
    call()                                                # re-armed counters, the same order of sums
    assert torch_cuda.equal(first, C)


@pytest.mark.parametrize("K,cb", [(K, cb) for K in range(1, 9) for cb in range(3)] + [(1.5, 2), (2.5, 2), (3.5, 2)])
@pytest.mark.parametrize("m", [9, 16, 24, 120])
def test_rows_bitrates(torch_cuda, orc, K, cb, m):
    L = synth.layer(384, 1024, K, cb, seed=7100 + int(10 * K) + cb)
    x = synth.activations(m, 384, seed=7101 + m)
    _, C, _ = run(torch_cuda, L, x)
    check(C, orc.linear_f64(x, L.trellis, L.suh, L.svh, int(K), half=K != int(K), cb=cb), (K, cb, m))


@pytest.mark.parametrize("m,k,n", [(33, 128, 128), (20, 128, 1024), (70, 4096, 1024), (33, 4096, 1152), (100, 1664, 256),
                                   (40, 8192, 2048), (9, 128, 128), (9, 1664, 1152), (16, 4096, 1024), (16, 1664, 384)])
@pytest.mark.parametrize("fp32,suh,svh", [(False, True, True), (True, True, True), (False, False, True), (True, True, False)])
def test_rows_splits_and_forms(torch_cuda, orc, m, k, n, fp32, suh, svh):
    """One block, many ranges, ranges of unequal length, with the hand-off and the finish kernel, at one row
    group and more; fp32 output; without either rotation."""
    L = synth.layer(k, n, 3, 2, seed=7200 + m + n)
    x = synth.activations(m, k, seed=7201 + k)
    _, C, _ = run(torch_cuda, L, x, fp32, suh, svh)
    W = orc.reconstruct(L.trellis, 3, cb=2).astype(np.float64)
    xr = orc.had128(x, pre=L.suh).astype(np.float64) if suh else x.astype(np.float64)
    y = xr @ W
    if svh:
        H = np.array([[(-1.0) ** bin(i & j).count("1") for j in range(128)] for i in range(128)]) / np.sqrt(128.0)
        y = (y.reshape(m, n // 128, 128) @ H).reshape(m, n) * L.svh.astype(np.float64)
    check(C, y, (m, k, n, fp32, suh, svh))


@pytest.mark.parametrize("m", [12, 33])
@pytest.mark.parametrize("n", [1024, 1152])
def test_rows_is_the_kernel(torch_cuda, kernel_policy, m, n):
    """The policy selects a kernel of its own: fp32 sums in another order than the GEMV's and the tiled GEMM's."""
    from ampstein_amd import ops
    torch = torch_cuda
    L = synth.layer(1664, n, 4, 0, seed=7300)
    x = synth.activations(m, 1664, seed=7301)
    _, C, _ = run(torch, L, x, True)
    t, s, v = L.torch()
    A = torch.from_numpy(x).cuda()
    for force in (1, 2):
        D = torch.empty_like(C)
        ops.exl3_gemm(A, t, D, s, torch.empty_like(A), v, force)
        assert not torch.equal(C, D), force
        # fp32 sums; the others take 3INST's two halves apart, here each weight is rounded: at most 2^-11 of it
        assert ((C - D).abs().max() / D.abs().max()).item() < 2.0 ** -11


def test_rows_captured(torch_cuda, orc):
    """Graph replays, with eager calls between them, give the eager call's bits."""
    torch = torch_cuda
    L = synth.layer(2048, 1024, 5, 1, seed=7400)
    x = synth.activations(37, 2048, seed=7401)
    _, C, call = run(torch, L, x)
    first = C.clone()
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        call()
    for _ in range(3):
        C.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(first, C)
        call()
        torch.cuda.synchronize()

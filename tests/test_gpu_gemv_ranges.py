"""GEMV work splits: k ranges of unequal length on the matrix-core row kernel (2..16 rows, with
the hand-off and with the finish kernel), its packed MUL1 operands, and the unsplit single row of
a very wide matrix.  Against the CPU oracle's fp64 linear; bar max|y - ref| / max|ref| < 2e-3 (fp16
rounding of the rotated input and of the output, fp32 sums)."""
import numpy as np
import pytest

from ampstein_amd import _lib, synth

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch_cuda():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from ampstein_amd import ops
    ops.init(0)
    return torch


def gemm(torch, L, x, force=0):
    from ampstein_amd import ops
    t, s, v = L.torch()
    A = torch.from_numpy(x).cuda()
    C = torch.full((x.shape[0], L.n), float("nan"), dtype=torch.half, device="cuda")
    call = lambda: ops.exl3_gemm(A, t, C, s, torch.empty_like(A), v, force, L.cb == 1, L.cb == 2)
    assert call() == 90
    return C, call


def _device_cus():
    import ctypes
    cus, xcd = ctypes.c_int(), ctypes.c_int()
    _lib.check(_lib.lib().exl3_amd_device_info(0, ctypes.byref(cus), ctypes.byref(xcd)))
    return cus.value


def check(C, ref, what):
    err = np.abs(C.cpu().numpy().astype(np.float64) - ref).max() / np.abs(ref).max()
    assert err < 2e-3, (what, err)


@pytest.mark.parametrize("m", [2, 3, 4, 5, 7, 8])
@pytest.mark.parametrize("k,n", [(128, 1024), (896, 1024), (1408, 384), (5248, 1024)])
@pytest.mark.parametrize("K,cb", [(4, 0), (3, 1), (5, 2), (2.5, 2)])
def test_rows_ranges(torch_cuda, orc, m, k, n, K, cb):
    """1, 7, 11 and 41 chunks of 128 rows: no divisor but one; odd numbers of (row, chunk) jobs.  On 256 CUs
    the planner takes 1, 7 and 11 ranges of one chunk each, and 21 or 22 unequal ones of 41 chunks."""
    ranges(torch_cuda, orc, m, k, n, K, cb, 0)


@pytest.mark.parametrize("m,k,n", [(m, 5248, n) for m in (3, 4, 8) for n in (384, 1152)]
                         + [(m, k, n) for m in (9, 12, 16) for k, n in ((5248, 384), (5248, 1024), (1408, 384))])
@pytest.mark.parametrize("K,cb", [(4, 0), (3, 1), (5, 2), (2.5, 2)])
def test_rows_unequal_ranges(torch_cuda, orc, m, k, n, K, cb):
    """Unequal ranges (256 CUs: 21 of 41 chunks at 3..8 rows; 14 of 41, and 6 of 11 at 16 rows, at 9..16
    rows) with the finish kernel (n / 128 = 3, 9) and the hand-off; the 9..16-row instance, which exl3_gemm
    takes under force_shape_idx 1 at any size."""
    ranges(torch_cuda, orc, m, k, n, K, cb, 1)


def ranges(torch_cuda, orc, m, k, n, K, cb, force):
    L = synth.layer(k, n, K, cb, seed=9000 + k + m + int(10 * K))
    x = synth.activations(m, k, seed=9001 + k)
    C, call = gemm(torch_cuda, L, x, force)
    check(C, orc.linear_f64(x, L.trellis, L.suh, L.svh, int(K), half=K != int(K), cb=cb), (m, k, n, K, cb))
    first = C.clone()
    call()
    assert torch_cuda.equal(first, C)


@pytest.mark.parametrize("K,cb", [(6, 2), (4, 0), (1.5, 2)])
def test_single_row_whole_columns(torch_cuda, orc, K, cb):
    """768 column chunks (three full rounds of workgroups): one per chunk takes all of k.  769: split."""
    for n in (98304, 98432):
        L = synth.layer(512, n, K, cb, seed=9100 + int(10 * K))
        x = synth.activations(1, 512, seed=9101)
        C, _ = gemm(torch_cuda, L, x)
        check(C, orc.linear_f64(x, L.trellis, L.suh, L.svh, int(K), half=K != int(K), cb=cb), (n, K, cb))


def same_as_split(torch, kernel_policy, call, slices):
    """Which of two forced splits (k-slices per workgroup) the planner's own call gives the bits of: the
    fp32 sums of another split differ."""
    outs = []
    for forced in (0, *slices):
        kernel_policy(_lib.POLICY_GEMV_SLICES, forced)
        outs.append(call())
    assert not torch.equal(outs[1], outs[2])
    return [torch.equal(outs[0], o) for o in outs[1:]]


@pytest.mark.parametrize("n,whole", [(98304, True), (102400, False), (65536, False)])
def test_single_row_split_rule(torch_cuda, kernel_policy, n, whole):
    """3 workgroups per CU of whole columns stay unsplit; 800 (a fourth, nearly empty round) and 512 do not."""
    from ampstein_amd import ops
    torch = torch_cuda
    if _device_cus() != 256:
        pytest.skip("the sizes are for 256 CUs")
    t, s, v = synth.layer(512, n, 4, 0, seed=9200).torch()
    A = torch.from_numpy(synth.activations(1, 512, seed=9201)).cuda()

    def call():
        C = torch.empty((1, n), dtype=torch.float, device="cuda")
        ops.exl3_gemm(A, t, C, s, torch.empty_like(A), v)
        return C
    assert same_as_split(torch, kernel_policy, call, (16, 32)) == [not whole, whole]


@pytest.mark.parametrize("form", ["indices", "filter", "widths"])
def test_bundle_split_with_idle_slots(torch_cuda, kernel_policy, form):
    """64 slots of 12 column chunks, 2 of them in use: workgroups without work do not count, k is split."""
    from ampstein_amd import ops
    torch = torch_cuda
    k, n, slots = 512, 1536, 64
    mats = [synth.layer(k, n, 4, 0, seed=9300 + i).torch() for i in range(2)]
    P = lambda i, num: ops.ptr_array([mats[j % 2][i] for j in range(num)])
    A = torch.from_numpy(synth.activations(1, k, seed=9301)).cuda()[None]
    A_had = torch.empty((slots, 1, k), dtype=torch.half, device="cuda")

    def call():
        C = torch.zeros((slots, 1, n), dtype=torch.float, device="cuda")
        if form == "widths":
            widths = torch.tensor([n] + [128] * (slots - 1), dtype=torch.int32, device="cuda")
            c_ptrs = ops.ptr_array([C.data_ptr() + j * n * 4 for j in range(slots)])
            ops.exl3_mgemm(A, P(0, slots), C, P(1, slots), A_had, P(2, slots), None, None, 4, size_n_list=widths,
                           c_ptrs=c_ptrs)
            return C[:1].clone()
        idx = torch.full((1, slots), -1 if form == "indices" else 1000, dtype=torch.long, device="cuda")
        idx[0, 0], idx[0, 1] = 0, 1
        lo, hi = (-1, -1) if form == "indices" else (0, 2)
        ops.exl3_mgemm(A, P(0, 2), C, P(1, 2), A_had, P(2, 2), idx, None, 4, min_index=lo, max_index=hi)
        return C[:2].clone()
    assert same_as_split(torch, kernel_policy, call, (16, 32)) == [True, False]


@pytest.mark.parametrize("form", ["indices", "filter", "widths", "full"])
@pytest.mark.parametrize("m", [2, 4])
def test_rows_split_with_idle_slots(torch_cuda, orc, form, m):
    """The same for 2 to 4 rows, where a range holds at most 8 chunks of 128 rows with lists: 9 chunks are split
    (partial sums in the workspace), which 64 slots in use are not."""
    from ampstein_amd import ops
    torch = torch_cuda
    if _device_cus() != 256:
        pytest.skip("the sizes are for 256 CUs")
    k, n, slots = 1152, 1536, 64
    layers = [synth.layer(k, n, 4, 0, seed=9400 + i) for i in range(2)]
    mats = [L.torch() for L in layers]
    P = lambda i, num: ops.ptr_array([mats[j % 2][i] for j in range(num)])
    x = synth.activations(m, k, seed=9401)
    A = torch.from_numpy(x).cuda()[None]
    A_had = torch.empty((slots, m, k), dtype=torch.half, device="cuda")
    C = torch.zeros((slots, m, n), dtype=torch.float, device="cuda")
    dev = torch.cuda.current_device()
    _lib.check(_lib.lib().exl3_amd_debug_fill_workspace(dev, 0xFF))
    if form == "widths":
        widths = torch.tensor([n] + [128] * (slots - 1), dtype=torch.int32, device="cuda")
        c_ptrs = ops.ptr_array([C.data_ptr() + j * m * n * 4 for j in range(slots)])
        ops.exl3_mgemm(A, P(0, slots), C, P(1, slots), A_had, P(2, slots), None, None, 4, size_n_list=widths, c_ptrs=c_ptrs)
    elif form == "full":
        ops.exl3_mgemm(A, P(0, slots), C, P(1, slots), A_had, P(2, slots), None, None, 4)
    else:
        idx = torch.full((1, slots), -1 if form == "indices" else 1000, dtype=torch.long, device="cuda")
        idx[0, 0], idx[0, 1] = 0, 1
        lo, hi = (-1, -1) if form == "indices" else (0, 2)
        ops.exl3_mgemm(A, P(0, 2), C, P(1, 2), A_had, P(2, 2), idx, None, 4, min_index=lo, max_index=hi)
    torch.cuda.synchronize()
    L = layers[0]
    check(C[0], orc.linear_f64(x, L.trellis, L.suh, L.svh, 4, cb=0), (form, m))
    head = np.empty(m * n, np.uint32)
    _lib.check(_lib.lib().exl3_amd_debug_read_workspace(dev, 0, head.nbytes, head.ctypes.data))
    assert bool((head != 0xFFFFFFFF).any()) == (form != "full")

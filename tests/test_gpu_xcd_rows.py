"""The row-tile GEMM under the hand-off check's alarm (exl3_xcd.cuh).  A file of its own, ordered
after test_gpu_xcd_guard.py, whose first test wants no alarm raised before it."""
import pytest

from ampstein_amd import synth
from tests.test_gpu_rows import check, run, torch_cuda  # noqa: F401

pytestmark = pytest.mark.gpu


def test_rows_finish_kernel(torch_cuda, orc):
    """The hand-off's alarm path: one workgroup reports another XCC, the next call sums its ranges
    in rows_finish; the sums are taken in the same order, so both give the same bits."""
    from ampstein_amd import _lib
    torch = torch_cuda
    L = synth.layer(4096, 1024, 4, 0, seed=7300)
    x = synth.activations(50, 4096, seed=7301)
    _, C, call = run(torch, L, x)
    ref = orc.linear_f64(x, L.trellis, L.suh, L.svh, 4, cb=0)
    check(C, ref, "hand-off")
    first = C.clone()
    lib = _lib.lib()
    try:
        lib.exl3_amd_set_policy(_lib.POLICY_XCD_FAKE, 1)
        call()
        torch.cuda.synchronize()
        lib.exl3_amd_set_policy(_lib.POLICY_XCD_FAKE, 0)
        C.zero_()
        call()
        torch.cuda.synchronize()
        check(C, ref, "finish kernel")
        assert torch.equal(first, C)
    finally:
        lib.exl3_amd_set_policy(_lib.POLICY_XCD_FAKE, 0)
        lib.exl3_amd_xcd_rearm(0)

"""Rows at addresses that the LDS DMA (global_load_lds_dwordx4, 16 bytes a lane) cannot take: the calls
that run on it otherwise take a kernel with plain loads.  Buffers sit 8 bytes past an aligned start;
the results are those of the same kernel on aligned rows, bit for bit."""
import numpy as np
import pytest

from ampstein_amd import _lib, synth
from tests.moe_ref import ExpertSet, routing

pytestmark = pytest.mark.gpu

OFF = 4          # fp16 elements


@pytest.fixture(scope="module")
def torch_cuda():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from ampstein_amd import ops
    ops.init(0)
    return torch


def off_by(torch, shape, offset, fill=None):
    t = torch.empty(int(np.prod(shape)) + offset, dtype=torch.half, device="cuda")[offset:].view(shape)
    assert t.data_ptr() % 16 == (2 * offset) % 16
    if fill is not None: t.copy_(fill)
    return t


@pytest.mark.parametrize("m,groups", [(12, True), (24, True), (100, False)])
@pytest.mark.parametrize("rotate", [False, True])
def test_gemm_rows(torch_cuda, kernel_policy, m, groups, rotate):
    """The GEMV's 16-row groups up to some 30 rows, register-staged tiles above; the rows read are A's, or
    A_had's with the input rotation."""
    from ampstein_amd import ops
    torch = torch_cuda
    k, n = 256, 1024
    t, s, v = synth.layer(k, n, 4, 0, seed=9500).torch()
    x = torch.from_numpy(synth.activations(m, k, seed=9501)).cuda()

    def call(offset, force):
        A = off_by(torch, (m, k), 0 if rotate else offset, x)
        A_had = off_by(torch, (m, k), offset)
        C = torch.full((m, n), float("nan"), dtype=torch.float, device="cuda")
        ops.exl3_gemm(A, t, C, s if rotate else None, A_had, v, force)
        return C
    y = call(OFF, 0)
    if not groups: kernel_policy(_lib.POLICY_GEMM_STAGING, _lib.GEMM_STAGING_REGS)
    assert torch.equal(y, call(0, 1 if groups else 2))


@pytest.mark.parametrize("Ks", [[4] * 4, [2, 3, 4, 5]], ids=["one-rate", "rates"])
def test_moe_row_buffers(torch_cuda, orc, kernel_policy, Ks):
    from tests.test_gpu_moe_sorted import run_moe
    torch = torch_cuda
    es = ExpertSet(torch, orc, 4, 256, 384, 256, Ks, 2, seed=71)
    x = np.random.default_rng(6).standard_normal((40, 256)).astype(np.float16)
    rt = routing(40, 4, 2, seed=9)
    args = (es, x, rt, 64, 2, 0, 1 << 30, 0, 0.0, Ks)
    y = run_moe(*args, offset=OFF)[0]
    kernel_policy(_lib.POLICY_MOE_GEMM, _lib.MOE_GEMM_LDS)
    assert torch.equal(y, run_moe(*args)[0])

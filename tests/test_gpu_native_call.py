"""The native launch path of ops.exl3_gemm, ops.mgemm and LinearEXL3.forward
(adapter/exl3_amd_torch.cpp): every form the operators accept gives the same bits as the Python
statement of the operator (the same C-ABI call), and what they refuse is refused as before."""
import pytest

from ampstein_amd import synth

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch_cuda():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return torch


class _Decline:
    """The native module with every call declined: the Python statement runs."""

    def __init__(self, mod):
        self.DECLINED = mod.DECLINED
        self.gemm_call = self.mgemm_call = lambda *a: mod.DECLINED
        self.linear_call = lambda *a: None


def both(monkeypatch, fn):
    """fn() on the native path and on the Python statement: two results, or two Exl3Errors."""
    from ampstein_amd import _lib, ops
    res = []
    mod = ops._native()
    for calls in (mod, _Decline(mod)):
        monkeypatch.setattr(ops, "_calls", calls)
        try:
            res.append(fn())
        except _lib.Exl3Error as e:
            res.append((type(e), e.code))
    monkeypatch.setattr(ops, "_calls", mod)
    return res


FORMS = ["plain", "3d", "fp32", "no_suh", "no_svh", "uint16", "one_row", "zero_rows", "int_flags",
         "bad_dtype", "strided", "short_suh", "wrong_k", "wrong_rows", "half_no_mul1", "both_books", "cpu"]


@pytest.mark.parametrize("form", FORMS)
def test_gemm_forms(torch_cuda, monkeypatch, form):
    torch = torch_cuda
    from ampstein_amd import ops
    L = synth.layer(256, 384, 2.5 if form == "half_no_mul1" else 3, 2, seed=77)
    t, s, v = L.torch()
    rows = {"one_row": 1, "zero_rows": 0}.get(form, 6)
    A = torch.randn(rows, 256, device="cuda").half()
    if form == "3d": A = A.view(2, 3, 256)
    if form == "bad_dtype": A = A.float()
    if form == "strided": A = torch.cat([A, A], 1)[:, :256]
    if form == "wrong_k": A = torch.randn(6, 128, device="cuda").half()
    if form == "cpu": A = A.cpu()
    if form == "uint16": t = t.view(torch.uint16)
    if form == "short_suh": s = s[:128]
    mcg, mul1 = form == "both_books", form != "half_no_mul1"
    if form == "int_flags": mcg, mul1 = 0, 1

    def call():
        C = torch.full((*A.shape[:-1], 384), float("nan"), dtype=torch.float if form == "fp32" else torch.half, device="cuda")
        if form == "wrong_rows": C = C[:5].contiguous()
        tag = ops.exl3_gemm(A, t, C, None if form == "no_suh" else s, torch.empty_like(A), None if form == "no_svh" else v,
                            0, mcg, mul1)
        return tag, C
    a, b = both(monkeypatch, call)
    assert a[0] == b[0]
    if isinstance(a[0], int):
        assert torch.equal(a[1], b[1])
    else:
        assert a == b


@pytest.mark.parametrize("form", ["stacked", "sliced", "missing_list", "missing_src", "rank", "rows"])
def test_mgemm_forms(torch_cuda, monkeypatch, form):
    torch = torch_cuda
    from ampstein_amd import bundles, ops
    lins = []
    for i, n in enumerate((512, 256, 256) if form != "stacked" else (256, 256)):
        t, s, v = synth.layer(384, n, 4, 0, seed=80 + i).torch()
        lins.append(bundles.Linear(t, s, v, 4.0))
    x = torch.randn(1, 3, 384, device="cuda").half()

    def call():
        if form == "stacked":
            out = torch.zeros((2, 3, 256), dtype=torch.half, device="cuda")
            return 0, bundles.Multi(lins, out).run(x)
        outs = [torch.zeros((1, 3, w.out_features), dtype=torch.half, device="cuda") for w in lins]
        b = bundles.Sliced(lins, outs)
        if form == "missing_list": b.opts["c_ptrs"] = None
        if form == "missing_src": del b.opts["num_had_src"]
        b.run(x[0] if form == "rank" else x[:, :2].contiguous() if form == "rows" else x)
        return 0, torch.cat([o.view(-1) for o in outs])
    a, b = both(monkeypatch, call)
    assert a[0] == b[0]
    if a[0] == 0:
        assert torch.equal(a[1], b[1])
    else:
        assert a == b


@pytest.mark.parametrize("rows", [1, 8, 9, 144, 200, 513])
@pytest.mark.parametrize("bias", [False, True])
def test_linear_forms(torch_cuda, monkeypatch, rows, bias):
    torch = torch_cuda
    from ampstein_amd.linear import LinearEXL3
    t, s, v = synth.layer(256, 384, 4, 1, seed=90).torch()
    W = {"w.trellis": t, "w.suh": s, "w.svh": v, "w.mcg": t}
    if bias: W["w.bias"] = torch.randn(384, device="cuda").half()

    class Store:
        has = staticmethod(lambda key: key in W)
        info = staticmethod(lambda key: {"shape": list(W[key].shape)})
        gpu = gpu16 = staticmethod(lambda key, dev=None: W[key])
    lin = LinearEXL3(Store, "w")
    x = torch.randn(rows, 256, device="cuda").half()
    for form in (x, torch.cat([x, x], 1)[:, :256], x.float(), x[:, :128].contiguous()):
        a, b = both(monkeypatch, lambda: (0, lin(form)))
        assert a[0] == b[0]
        if a[0] == 0:
            assert torch.equal(a[1], b[1]) and a[1].stride() == b[1].stride()
        else:
            assert a == b

"""The token-sorted MoE's grouped GEMM over experts of every integer bitrate at once (one launch per
phase), with row counts at the edges of its 16-row groups and row tiles, and k of a few 64-row units
(2 units: no full turn of the four row buffers; 6: one turn and a remainder).  Same model and bar as
tests/test_gpu_moe_sorted.py: max |y - ref| / max |ref| < 2e-3 for the fp16 rounding of the staged
rows, the GEMM outputs and the activation."""
import numpy as np
import pytest
import torch

from ampstein_amd import _lib
from tests.moe_ref import ExpertSet, routing
from tests.test_gpu_moe_sorted import model, run_moe

pytestmark = pytest.mark.gpu

# rows of each expert: 0 (no list entry), group edges, a tile and one row
COUNTS = [16, 1, 65, 0, 33, 49, 17, 64]


@pytest.mark.parametrize("tile_rows", [32, 64, 96, 128])
@pytest.mark.parametrize("cb,H,I,Ks", [(2, 384, 128, [1, 2, 3, 4, 5, 6, 7, 8]), (2, 128, 384, [4, 4, 1, 1, 8, 8, 2, 2]),
                                       (2, 384, 128, [3.5] * 8), (2, 128, 384, [1.5] * 8), (2, 128, 384, [2.5] * 8),
                                       (1, 384, 128, [1] * 8), (1, 128, 384, [5] * 8),
                                       (1, 384, 128, [8] * 8)],
                         ids=["mul1-all", "mul1-shared", "mul1-k3.5", "mul1-k1.5", "mul1-k2.5", "mcg-k1", "mcg-k5", "mcg-k8"])
def test_all_rates_in_one_launch(orc, kernel_policy, cb, H, I, Ks, tile_rows):
    kernel_policy(_lib.POLICY_MOE_TILE_ROWS, tile_rows)
    E, T = len(Ks), 65
    es = ExpertSet(torch, orc, E, H, I, H, Ks, cb, seed=11 + cb)
    rng = np.random.default_rng(tile_rows)
    x = rng.standard_normal((T, H)).astype(np.float16)
    spare = 4 * T - sum(COUNTS)                    # the list holds 4 a token; the last count is ignored
    count = np.array(COUNTS + [spare], np.int64)
    start = np.concatenate([[0], np.cumsum(count)[:-1]]).astype(np.int64)
    token_sorted = np.concatenate([rng.permutation(T)[:c] for c in COUNTS + [spare]]).astype(np.int64)
    weight_sorted = rng.uniform(0.1, 1.0, token_sorted.size).astype(np.float16)
    rt = (None, None, None, token_sorted, weight_sorted, count, start)
    print(f"rates cb {cb} {H}x{I} tile {tile_rows}", flush=True)
    out, _, _, _ = run_moe(es, x, rt, 65, 4, 0, 1 << 30, 0, 0.0, Ks)
    ref, _ = model(es, x, None, token_sorted, weight_sorted, count, start, 65, 0, 1 << 30, 0, 0.0)
    y = out.cpu().numpy().astype(np.float64)
    err = np.abs(y - ref).max() / np.abs(ref).max()
    print(f"  rel err {err:.2e}", flush=True)
    assert err < 2e-3


@pytest.mark.parametrize("tile_rows", [32, 64, 96, 128])
@pytest.mark.parametrize("cb,Ks", [(2, [1, 2, 3, 4, 5, 6, 7, 8]), (2, [2.5] * 4), (1, [3] * 4)], ids=["mul1-all", "mul1-k2.5", "mcg-k3"])
def test_long_k(orc, kernel_policy, cb, Ks, tile_rows):
    """Many turns of the row buffers (32 and 12 units), more items than workgroups: the LDS-tiled kernel's
    results, and the same bits on every call (rows read before they land would differ between calls).
    Both round the same points; each GEMM's fp32 sums may round to the neighbouring fp16 (2^-11)."""
    kernel_policy(_lib.POLICY_MOE_TILE_ROWS, tile_rows)
    E, T, H, I = len(Ks), 200, 2048, 768
    es = ExpertSet(torch, orc, E, H, I, H, Ks, cb, seed=21 + cb)
    # (small rows: the synthetic weights' products leave the fp16 range at this k)
    x = (np.random.default_rng(8).standard_normal((T, H)) / 64).astype(np.float16)
    rt = routing(T, E, 3, seed=tile_rows)
    print(f"long k cb {cb} K {Ks[0]} tile {tile_rows}", flush=True)
    outs = [run_moe(es, x, rt, T, 3, 0, 1 << 30, 0, 0.0, Ks)[0].clone() for _ in range(4)]
    for o in outs[1:]:
        assert torch.equal(outs[0], o)
    kernel_policy(_lib.POLICY_MOE_GEMM, _lib.MOE_GEMM_LDS)
    kernel_policy(_lib.POLICY_MOE_TILE_ROWS, 0)
    ref = run_moe(es, x, rt, T, 3, 0, 1 << 30, 0, 0.0, Ks)[0]
    assert torch.isfinite(ref).all()
    err = ((outs[0] - ref).abs().max() / ref.abs().max()).item()
    print(f"  rel err {err:.2e}", flush=True)
    assert err < 2e-3

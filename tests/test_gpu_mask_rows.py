"""GPU: the shared-pool block mask against the generic kernel (which reads a strided copy of the key pool), bit for bit:
scores, lists and counts at the edges of its chunks of 64 blocks, its register sizes and its groups of four rows."""
import pytest
import torch

from li_sparse import _core, _lib

pytestmark = pytest.mark.gpu


def _pools(B, NH, nq, nk, D, dtype, dev, seed):
    gen = torch.Generator().manual_seed(seed)
    q, k = ((torch.randn(B, NH, n, D, generator=gen) * 0.3).to(dtype).to(dev) for n in (nq, nk))
    if nk > 4:
        k[:, :, nk // 2] = 0            # a zero row: the cosine normaliser's floor
        k[:, :, nk // 3] = k[:, :, 0]   # equal scores
    return q, k


@pytest.mark.parametrize("nk", [1, 3, 63, 64, 65, 255, 256, 257, 511, 513, 1023, 1024, 1025, 1791, 1792, 1793])
@pytest.mark.parametrize("D,dtype", [(128, torch.bfloat16), (64, torch.float16)])
def test_equals_generic_kernel(dev, nk, D, dtype):
    B, NH, nh, nw = 1, 3, 3, 7
    print(f"[gpu] block mask nk={nk} D={D} {dtype}", flush=True)
    for nq, metric in ((1, "cosine"), (4, "scaled_dot_product"), (5, "dot"), (11, "cosine")):
        q, k = _pools(B, NH, nq, nk, D, dtype, dev, nk + nq)
        strided = torch.stack([k, k], -1)[..., 0]          # d stride 2: the generic kernel
        for kw in (dict(budget_mode=_lib.LI_BUDGET_HISTORY, ratio=0.3, n_recent=2, force_diag=True, force_sink=True),
                   dict(budget_mode=_lib.LI_BUDGET_TOTAL, ratio=0.21, force_neighbors=True),
                   dict(budget_mode=_lib.LI_BUDGET_TOTAL, ratio=0.0, min_budget=0,
                        row_budget=[(5 * i) % (nk + 1) for i in range(nq)])):
            kw.update(metric=metric, nh=nh, nw=nw, num_txt_blk=2, return_scores=True)
            a, b = _core.block_mask(q, k, **kw), _core.block_mask(q, strided, **kw)
            torch.cuda.synchronize()
            for x, y in zip(a, b):
                assert torch.equal(x.view(torch.int16) if x.dtype != torch.int32 else x,
                                   y.view(torch.int16) if y.dtype != torch.int32 else y), (nq, metric, kw)


@pytest.mark.parametrize("nk", [257, 320, 700, 1024])
@pytest.mark.parametrize("D,dtype", [(128, torch.float16), (64, torch.bfloat16)])
def test_many_row_groups_equal_generic_kernel(dev, nk, D, dtype):
    """More row groups than CUs: four scoring waves a workgroup."""
    NH, nq = 8, 4 * (torch.cuda.get_device_properties(dev).multi_processor_count // 8) + 3
    print(f"[gpu] block mask, many rows: {NH} x {nq} x {nk} D={D} {dtype}", flush=True)
    q, k = _pools(1, NH, nq, nk, D, dtype, dev, nk)
    strided = torch.stack([k, k], -1)[..., 0]
    for metric in ("cosine", "scaled_dot_product"):
        kw = dict(metric=metric, nh=3, nw=7, num_txt_blk=1, return_scores=True, budget_mode=_lib.LI_BUDGET_HISTORY,
                  ratio=0.3, n_recent=2, force_diag=True)
        a, b = _core.block_mask(q, k, **kw), _core.block_mask(q, strided, **kw)
        torch.cuda.synchronize()
        for x, y in zip(a, b):
            assert torch.equal(x.view(torch.int16) if x.dtype != torch.int32 else x,
                               y.view(torch.int16) if y.dtype != torch.int32 else y), metric


def test_special_values_and_strided_pools(dev):
    """Infinities, NaN and the smallest numbers in the pools; pools that are views of longer buffers."""
    B, NH, nq, nk, D = 2, 2, 6, 130, 128
    q, k = _pools(B, NH, nq, nk, D, torch.bfloat16, dev, 3)
    q[0, 0, 1, 5], k[0, 0, 7, 9], k[0, 1, 64, 0] = float("inf"), float("-inf"), float("nan")
    q[1, 0, 2] = 1e-38
    k[1, 0, 100] = -1e-20
    wide = torch.zeros(B, NH, nk + 6, D + 8, dtype=torch.bfloat16, device=dev)
    wide[:, :, 3:3 + nk, 8:] = k
    view = wide[:, :, 3:3 + nk, 8:]
    for metric in ("cosine", "scaled_dot_product", "dot"):
        kw = dict(metric=metric, budget_mode=_lib.LI_BUDGET_HISTORY, ratio=0.3, nh=2, nw=5, return_scores=True)
        ref = _core.block_mask(q, torch.stack([k, k], -1)[..., 0], **kw)
        for pool in (k, view):
            got = _core.block_mask(q, pool, **kw)
            torch.cuda.synchronize()
            nan = torch.isnan(ref[2].float())
            assert torch.equal(torch.isnan(got[2].float()), nan)
            assert torch.equal(got[2].view(torch.int16)[~nan], ref[2].view(torch.int16)[~nan]), metric
            keep = ~nan.any(-1)
            assert torch.equal(got[0][keep], ref[0][keep]) and torch.equal(got[1], ref[1])

"""GPU: the range check of block ids (li_check_block_ids) against the host's own, and when its result is read."""
import pytest
import torch

from li_sparse import _core
from li_sparse.hy.longcat_kernel import longcat_flash_attn

pytestmark = pytest.mark.gpu


# around the 4-id vectors, the 1024 ids of a pass of a workgroup, its 4096-id share, and the 512 workgroups' 2 M ids
@pytest.mark.parametrize("n", [1, 3, 4, 7, 1023, 4096, 4097, 70001, (1 << 21) + 4099])
def test_finds_one_bad_id_anywhere(dev, n):
    print(f"[gpu] check_block_ids n={n}", flush=True)
    nkb = 1000
    ids = torch.randint(0, nkb, (n,), dtype=torch.int32, device=dev)
    ids[-1] = nkb - 1
    assert _core.check_block_ids(ids, nkb)()
    for at in sorted({0, n // 3, n // 2, max(n - 5, 0), n - 1}):
        for bad in (nkb, -1, 2 ** 31 - 1, -2 ** 31):
            x = ids.clone()
            x[at] = bad
            assert not _core.check_block_ids(x, nkb)(), (at, bad)
    assert not _core.check_block_ids(ids, nkb - 1)()
    assert not _core.check_block_ids(ids, 0)()
    wide = torch.zeros(n + 1, dtype=torch.int32, device=dev)
    wide[0] = nkb               # before the list: not part of it
    assert _core.check_block_ids(wide[1:], 1)()
    assert _core.check_block_ids(ids[:0], 0)()


def test_results_of_calls_in_flight_are_their_own(dev):
    good = torch.zeros(50000, dtype=torch.int32, device=dev)
    bad = torch.full_like(good, 7)
    checks = [_core.check_block_ids(x, 7) for x in (good, bad, good, bad)]
    assert [c() for c in checks] == [True, False, True, False]


def test_wrapper_errors_and_capture(dev):
    q = torch.randn(1, 2, 256, 128, device=dev).to(torch.bfloat16)
    ind = torch.tensor([0, 1], dtype=torch.int32, device=dev).expand(1, 2, 2, 2)
    cnt = torch.full((1, 2, 2), 2, dtype=torch.int32, device=dev)
    longcat_flash_attn(q, q, q, ind, cnt)
    for bad in (ind + 1, ind - 1):
        with pytest.raises(ValueError, match="Sparse indices out of bounds."):
            longcat_flash_attn(q, q, q, bad, cnt)
    with pytest.raises(ValueError, match="Sparse indices out of bounds."):   # no key block: every id is out of range
        longcat_flash_attn(q, q[:, :, :0], q[:, :, :0], ind, cnt)
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    graph = torch.cuda.CUDAGraph()
    with pytest.raises(RuntimeError), torch.cuda.graph(graph, stream=stream):
        longcat_flash_attn(q, q, q, ind, cnt)
    torch.cuda.synchronize()
    longcat_flash_attn(q, q, q, ind, cnt)
    torch.cuda.synchronize()

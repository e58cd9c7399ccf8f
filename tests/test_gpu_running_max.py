"""GPU: later blocks whose scores lie far above the first one's, where the running max is kept or raised.

The kernels take exponentials against a running max that they raise only when a partial sum passes a bound, so
probabilities up to that bound are rounded to the element type.  Blocks between 9 and 21 log2 units above the earlier
ones are on both sides of the bounds (2^20 in bf16, 2^15 in half precision) and of a half's largest value (2^16).

Tolerance for |V| <= 1 and unit roundoff u (2^-8 in bf16, 2^-11 in half precision): rounding the probabilities moves the
weighted mean by at most u, rounding the output by u, the fp32 arithmetic by far less: 2.5 u.  LSE (fp32): 1e-3.
"""
import math

import numpy as np
import pytest
import torch

from li_sparse import _core
from oracle import attention as oatt

pytestmark = pytest.mark.gpu

JUMPS = (9.0, 13.0, 14.9, 15.5, 16.5, 17.0, 19.0, 21.0)
COLS = 9
DENSE_KEYS = COLS * 128 - 100
U = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}


def _case(D, bs, H, nq, dtype, jump, at, many, gen):
    """Tiles in list order: scores near 0 but for one key (or every key) of the blocks in ``at``, n jumps above it for the
    n-th of them in a third of the rows, half of that in another third and as far below it in the last."""
    scale = 1.0 / math.sqrt(D)
    q = torch.randn(1, H, nq * bs, D, generator=gen) * 0.05
    k = torch.randn(1, H, COLS * bs, D, generator=gen) * 0.05
    v = torch.rand(1, H, COLS * bs, D, generator=gen) * 2 - 1
    row = torch.arange(nq * bs) % 3
    q[..., 0] = torch.tensor([8.0, 4.0, -8.0])[row]
    for n, b in enumerate(at):
        rows = slice(b * bs, (b + 1) * bs) if many else slice(b * bs + 37, b * bs + 38)
        k[:, :, rows, 0] = (n + 1) * jump / (8.0 * scale * math.log2(math.e))
    return q.to(dtype), k.to(dtype), v.to(dtype), scale


def _run(kind, D, bs, q, k, v, ind, cnt, scale, split, dev):
    """(out, lse).  The token-order calls take a grid of one tile per slab of frames, whose tile order is the token order."""
    if kind == "dense":
        txt, n = 2 * bs - 4, DENSE_KEYS      # the first keys as text, its last block a partial one
        return _core.attn_dense(q.to(dev), k[:, :, txt:n].to(dev), v[:, :, txt:n].to(dev), k[:, :, :txt].to(dev),
                                v[:, :, :txt].to(dev), return_lse=True, split=split)
    q, k, v, ind, cnt = (t.to(dev) for t in (q, k, v, ind, cnt))
    if kind == "tiled":
        return _core.bsa_forward(q, k, v, ind, cnt, scale, bs, return_lse=True, split=split)
    tile = (2, 8, 8) if bs == 128 else (4, 4, 4)
    grid = (tile[1], tile[2], *tile, 1, 1)
    fq, fk = q.shape[2] // (tile[1] * tile[2]), k.shape[2] // (tile[1] * tile[2])
    out = torch.empty_like(q)
    if kind == "token":
        return _core.bsa_forward_gather(q, k, v, None, None, 0, fq, fk, *grid, ind, cnt, scale, out, return_lse=True,
                                        split=split)
    return _core.bsa_forward_qo(q, k.unflatten(2, (COLS, bs)), v.unflatten(2, (COLS, bs)), (fq, *grid), ind, cnt, scale,
                                out, return_lse=True, split=split)


def _reference(kind, bs, q, k, v, ind, cnt, scale):
    f64 = [t.double().numpy() for t in (q, k, v)]
    if kind != "dense":
        return oatt.bsa_forward(*f64, ind.numpy(), cnt.numpy(), scale, bs)
    s = (f64[0] @ f64[1][:, :, :DENSE_KEYS].swapaxes(-1, -2)) * scale
    mx = s.max(axis=-1, keepdims=True)
    p = np.exp(s - mx)
    l = p.sum(axis=-1, keepdims=True)
    return p @ f64[2][:, :, :DENSE_KEYS] / l, (mx[..., 0] + np.log(l[..., 0])) / math.log(2.0)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "f16"])
@pytest.mark.parametrize("kind,D,bs,H,nq", [
    ("tiled", 64, 64, 2, 3), ("tiled", 64, 64, 20, 16), ("rows", 64, 64, 2, 3),    # four interleaves, two, Q / O as tokens
    ("tiled", 64, 128, 2, 3), ("tiled", 128, 64, 2, 3), ("rows", 128, 128, 2, 3),
    ("tiled", 128, 128, 2, 3), ("token", 128, 128, 2, 3), ("dense", 128, 128, 2, 3)])
def test_blocks_far_above_the_running_max(dev, kind, D, bs, H, nq, dtype):
    print(f"[gpu] running max {kind} D={D} bs={bs} tiles={H * nq} {dtype}", flush=True)
    rng = np.random.default_rng(D + bs)
    gen = torch.Generator().manual_seed(D)
    worst = 0.0
    for jump in JUMPS:
        for at, many in (((1,), False), ((4, 7), False), ((5,), True), ((8,), False)):
            q, k, v, scale = _case(D, bs, H, nq, dtype, jump, at, many, gen)
            ind = torch.arange(COLS, dtype=torch.int32).repeat(1, H, nq, 1)
            ind = torch.nn.functional.pad(ind, (0, 3), value=-1)   # wide enough for four interleaves; never read
            cnt = torch.full((1, H, nq), COLS, dtype=torch.int32)
            if kind != "dense":  # shorter lists too: the raised block the last one, or absent
                cnt[0, 0] = torch.from_numpy(rng.integers(at[0], COLS + 1, nq).astype(np.int32))
            some = sorted({0, 1, H - 1})
            ref, lse_ref = _reference(kind, bs, *(t[:, some] for t in (q, k, v, ind, cnt)), scale)
            for split in ((False, True) if D == bs == 128 else (False,)):   # only these tiles are ever split
                o, lse = _run(kind, D, bs, q, k, v, ind, cnt, scale, split, dev)
                torch.cuda.synchronize()
                got, lse = (t[:, some].double().cpu().numpy() for t in (o, lse[:, :, :q.shape[2]]))
                what = (jump, at, many, split)
                assert np.isfinite(got).all(), what
                err = np.abs(got - ref).max()
                worst = max(worst, err)
                assert err <= 2.5 * U[dtype], (what, err)
                assert np.abs(lse - lse_ref).max() <= 1e-3, what
    print(f"[gpu]   largest error {worst:.2e} (bound {2.5 * U[dtype]:.2e})", flush=True)

"""GPU: query tiles split into several pieces of their block lists (launches that fill the CUs unevenly).

Each split call is compared with whole tiles and, on the tiled kernel, with the float64 oracle.  Piece results are
combined in fp32, so a split output differs from the whole tile's by at most one bf16 ulp (7.8e-3 for |out| < 2;
1e-2 asserted), its LSE by fp32 rounding (1e-4).
"""
import math

import numpy as np
import pytest
import torch

from helpers import bits
from li_sparse import _core, _lib
from oracle import attention as oatt
from oracle.bf16 import bf16_to_f32

pytestmark = pytest.mark.gpu


def _bf16(seed, shape, scale=1.0):
    return (torch.randn(shape, generator=torch.Generator().manual_seed(seed)) * scale).to(torch.bfloat16)


def _pieces(H, rows, cols, dev):
    with torch.cuda.device(dev):
        ws = _lib.lib.li_bsa_fwd_workspace_size_cols(1, H, rows, 128, 128, cols)
    return ws // (128 * 130 * 4)


# tiles below, at and above a multiple of 8 and of the CU count; lists shorter than, equal to and longer than the pieces
@pytest.mark.parametrize("H,nq,cols", [(1, 1, 60), (1, 8, 40), (3, 5, 33), (1, 13, 21), (3, 17, 24), (2, 52, 40),
                                       (5, 53, 16), (8, 33, 30), (8, 44, 24)])
def test_pieces_match_whole_tiles_and_oracle(dev, H, nq, cols):
    bs, D, nkb = 128, 128, max(cols, 4) + 3
    Lq, Lk = nq * bs - 40, nkb * bs
    n = _pieces(H, Lq, cols, dev)
    print(f"[gpu] split H={H} nq={nq} cols={cols}: room for {n} pieces", flush=True)
    assert n >= 2 * ((H * nq) % 256)
    rng = np.random.default_rng(nq)
    q, k, v = _bf16(1, (1, H, Lq, D), 0.3), _bf16(2, (1, H, Lk, D)), _bf16(3, (1, H, Lk, D))
    ind = np.argsort(rng.random((1, H, nq, nkb)), axis=-1)[..., :cols].astype(np.int32)
    cnt = rng.integers(max(cols - 3, 0), cols + 1, size=(1, H, nq)).astype(np.int32)
    flat = cnt.reshape(-1)  # short and empty lists too: pieces without a block
    for j, c in enumerate([0, 1, 2, 3]):
        flat[-1 - (j % flat.size)] = c
    dv = [t.to(dev) for t in (q, k, v)] + [torch.from_numpy(ind).to(dev), torch.from_numpy(cnt).to(dev)]
    scale = 1.0 / math.sqrt(D)
    out_s, lse_s = _core.bsa_forward(*dv, scale, bs, return_lse=True, split=True)
    out_w, lse_w = _core.bsa_forward(*dv, scale, bs, return_lse=True, split=False)
    torch.cuda.synchronize()
    fin = torch.isfinite(lse_w)
    assert torch.equal(torch.isneginf(lse_s), ~fin)
    d_out, d_lse = (out_s.float() - out_w.float()).abs().max().item(), (lse_s[fin] - lse_w[fin]).abs().max().item()
    print(f"[gpu]   split vs whole: out {d_out:.3e} lse {d_lse:.3e}", flush=True)
    assert d_out <= 1e-2 and d_lse <= 1e-4
    f64 = lambda t: bf16_to_f32(bits(t)).astype(np.float64)  # noqa: E731
    tiles = [(0, H - 1, nq - 1), (0, 0, 0), (0, H // 2, nq // 2)]
    o_ref, _ = oatt.bsa_forward(f64(q), f64(k), f64(v), ind, cnt, scale, bs, heads=tiles)
    got = out_s.float().cpu().numpy()
    for b, h, m in tiles:
        rows = slice(m * bs, min((m + 1) * bs, Lq))
        assert np.abs(got[b, h, rows] - o_ref[b, h, rows]).max() <= 2e-2


@pytest.mark.parametrize("H,nq,cols,parts", [(16, 22, 24, 2), (16, 24, 36, 2), (16, 56, 36, 2), (16, 56, 51, 2),
                                             (2, 26, 24, 3), (2, 26, 16, 2), (2, 14, 10, 0), (2, 52, 16, 0), (2, 26, 8, 0), (16, 28, 36, 0)])
def test_pieces_of_the_faster_choice(dev, H, nq, cols, parts):
    """Lists of 12 to 36 blocks behind a last round at most half full run as two pieces (the first three were whole, 3-9%
    slower), a small launch with short lists as two or three (not four: 3-8% slower) or whole, as do fuller last rounds."""
    if torch.cuda.get_device_properties(dev).multi_processor_count != 256:
        pytest.skip("the sizes are those of 256 CUs")
    n = -(-H * nq // 8)
    assert _pieces(H, nq * 128, cols, dev) == 8 * (n % 32) * parts


@pytest.mark.parametrize("H,Lq,Lk,txt", [(1, 300, 1500, 0), (2, 640, 2052, 300), (16, 6240, 3072, 77)])
def test_dense_pieces_match_whole_tiles(dev, H, Lq, Lk, txt):
    q, k, v = (_bf16(s, (1, H, n, 128)).to(dev) for s, n in ((4, Lq), (5, Lk), (6, Lk)))
    kt, vt = (_bf16(s, (1, H, txt, 128)).to(dev) for s in (7, 8))
    n = _pieces(H, -(-Lq // 128) * 128, -(-txt // 128) - (-Lk // 128), dev)
    print(f"[gpu] dense split H={H} Lq={Lq} Lk={Lk} text={txt}: room for {n} pieces", flush=True)
    assert n >= 2
    out_s, lse_s = _core.attn_dense(q, k, v, kt, vt, return_lse=True, split=True)
    out_w, lse_w = _core.attn_dense(q, k, v, kt, vt, return_lse=True, split=False)
    torch.cuda.synchronize()
    assert (out_s.float() - out_w.float()).abs().max().item() <= 1e-2
    assert (lse_s - lse_w)[:, :, :Lq].abs().max().item() <= 1e-4


def test_token_order_pieces_equal_tiled_pieces(dev):
    """A small fused call with text blocks, split: the same bits as the tiled sequence, also in e4m3."""
    from li_sparse import _pipeline
    from li_sparse.hy.ar_sparse_operation import fast_generate_indices

    H, hw, tile, dtype = 2, (18, 28), (4, 8, 4), torch.bfloat16
    tok = hw[0] * hw[1]
    q, k, v = (_bf16(s, (1, H, f * tok, 128)).to(dev) for s, f in ((1, 3), (2, 10), (3, 10)))
    kt, vt = _bf16(4, (1, H, 300, 128)).to(dev), _bf16(5, (1, H, 300, 128)).to(dev)
    params = {"tile_size": tile, "topk_ratio": 0.5, "sim_metric": "scaled_dot_product"}

    def select(qp, kp, tl, gq, gk):
        ind, cnt = fast_generate_indices(qp, kp, tl, gq, gk, params, dev)
        rows = qp.shape[2] * 128
        print(f"[gpu]   {H * qp.shape[2]} tiles x {ind.shape[3]} blocks: {_pieces(H, rows, ind.shape[3], dev)} pieces")
        assert _pieces(H, rows, ind.shape[3], dev) >= 2
        return ind, cnt

    for fp8 in (False, True):
        a, b = (_pipeline.sparse_attention(q, kt, vt, k, v, hw, tile, select, fused=f, qk_fp8=fp8, sorted_lists=True)
                for f in (True, False))
        torch.cuda.synchronize()
        assert a.dtype == dtype and torch.equal(a.view(torch.int16), b.view(torch.int16))


def test_nan_rows_stay_nan_when_split(dev):
    """A NaN in a query row (every score NaN) or in a key gives NaN outputs from split tiles as from whole ones."""
    bs, D, H, nq, cols = 128, 128, 2, 4, 40
    print(f"[gpu] NaN rows: room for {_pieces(H, nq * bs, cols, dev)} pieces", flush=True)
    assert _pieces(H, nq * bs, cols, dev) >= 16
    q, k, v = _bf16(1, (1, H, nq * bs, D), 0.3), _bf16(2, (1, H, cols * bs, D)), _bf16(3, (1, H, cols * bs, D))
    q[0, 0, 5, 7] = q[0, 1, 200] = float("nan")
    k[0, 1, 9 * bs + 3, 2] = float("nan")
    ind = torch.arange(cols, dtype=torch.int32, device=dev).repeat(1, H, nq, 1)
    cnt = torch.full((1, H, nq), cols, dtype=torch.int32, device=dev)
    cnt[0, 1, 2:] = 9            # lists that end before the key with the NaN
    scale = 1.0 / math.sqrt(D)
    got = [_core.bsa_forward(q.to(dev), k.to(dev), v.to(dev), ind, cnt, scale, bs, return_lse=True, split=s)
           for s in (True, False)]
    torch.cuda.synchronize()
    (out_s, _), (out_w, _) = got
    want = torch.zeros(1, H, nq * bs, dtype=torch.bool, device=dev)
    want[0, 0, 5] = want[0, 1, :2 * bs] = True
    for out in (out_s, out_w):
        assert torch.equal(torch.isnan(out).any(-1), want) and torch.equal(torch.isnan(out).all(-1), want)
    assert (out_s.float() - out_w.float())[~want].abs().max().item() <= 1e-2
